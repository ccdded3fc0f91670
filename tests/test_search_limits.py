"""Sizes of the split search's LDS arrays against a host model of what they
must hold (tests/cpp/search_limits.cc over csrc/dte_limits.h)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def _build(tmp_path):
    exe = str(tmp_path / "search_limits")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(HERE, "cpp", "search_limits.cc")], check=True)
    return exe


def test_in_bag_bits_of_a_workgroup_take_whole_words(tmp_path):
    """Every row count's bits fit, in no more words than they need."""
    assert subprocess.run([_build(tmp_path), "bag"], timeout=60).returncode == 0


def test_ranges_of_the_workgroup_tier_fit_their_stack(tmp_path):
    exe = _build(tmp_path)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout
    # a bootstrapped node alone holds more ranges than its entries suggest
    # (2048 entries: 33 ranges of more than 64)
    bootstrap = max(int(line.split()[1]) for line in p.stdout.splitlines() if line.startswith("bootstrap"))
    assert bootstrap > 2048 // 64 + 1


def test_buffers_of_the_side_stream_outlive_it():
    """A fit's buffers go back to the pool in the reverse order of their
    declarations: those that kernels of the side stream read come before it."""
    src = open(os.path.join(HERE, "..", "datamininglibs_amd", "csrc", "dte_build.hip")).read()
    side = src.index("struct SideStream {")
    for buffer in ("key_rows, draw_keys", "rowA, auxA", "res_score, res_thr", "BigState bigst", "tier_list[kMaxTiers]"):
        at = src.index(buffer)
        assert src.rindex("Forest* fit_batch(", 0, side) < at < side, buffer
