"""HIP kernels at the sizes where their tiers, tiles and staging change, bit
for bit against the CPU oracle (or a plain walk of the model)."""
import ctypes
import threading

import numpy as np
import pytest

from datamininglibs_amd import capi, synth
import pyoracle
from parity import assert_same_forest, fit_both

pytestmark = pytest.mark.gpu

RF, ERT = capi.RANDOM_FOREST, capi.EXTRA_TREES


def _targets(kind, X, rng):
    n = X.shape[1]
    if kind == "reg":
        return dict(task=capi.REGRESSION), (np.sin(4 * X[0]) + X[1] * X[2] + 0.1 * rng.standard_normal(n))
    c = int(kind)
    s = X[:3].sum(0) + 0.4 * rng.standard_normal(n)
    return dict(n_classes=c), np.clip(np.argsort(np.argsort(s)) * c // n, 0, c - 1)


@pytest.mark.parametrize("kind", ["2", "9", "16", "32", "reg"])
@pytest.mark.parametrize("n", [26, 51, 101, 811, 3241])
def test_rf_tiers_around_their_limits(kind, n):
    """Bootstraps of these row counts hold about 16, 32, 64, 512 and 2048
    distinct rows, on both sides of each tier's limit over 12 trees; the last
    one has nodes above the workgroup tier inside the level graphs."""
    rng = np.random.default_rng(n)
    X = rng.random((9, n)).astype(np.float32)
    X[6:] = np.floor(X[6:] * [[3], [8], [40]])  # ties
    kw, y = _targets(kind, X, rng)
    g, o = fit_both(X, y.astype(np.float32), algorithm=RF, n_trees=12, k=4, min_node_size=1, seed=n, **kw)
    assert_same_forest(g, o)


@pytest.mark.parametrize("kind", ["3", "reg"])
def test_rf_keys_in_clusters(kind):
    """Features that follow one another: below the first splits a node's keys
    fill a sliver of the feature's range, or two ends of it."""
    rng = np.random.default_rng(5)
    n = 2600
    X = np.empty((6, n), np.float32)
    X[0] = rng.random(n)
    X[1] = X[0] + 1e-4 * rng.random(n)
    X[2] = X[0] ** 9
    X[3] = np.where(rng.random(n) < 0.5, X[0], 100 - X[0])
    X[4] = np.floor(X[0] * 30)
    X[5] = np.where(rng.random(n) < 0.97, 0, rng.random(n))
    kw, y = _targets(kind, X, rng)
    g, o = fit_both(X, y.astype(np.float32), algorithm=RF, n_trees=10, k=3, min_node_size=1, **kw)
    assert_same_forest(g, o)


@pytest.mark.parametrize("target", ["constant", "zero_one", "offset", "spike"])
def test_rf_regression_targets_of_little_variance(target):
    """Gains of exactly or nearly nothing: rounding decides, and retries run."""
    rng = np.random.default_rng(8)
    n = 5000
    X = rng.random((6, n)).astype(np.float32)
    X[3:] = X[3:] < 0.1
    y = {"constant": np.full(n, 5.25), "zero_one": rng.integers(0, 2, n),
         "offset": 1e6 + 1e-2 * rng.standard_normal(n), "spike": (np.arange(n) == 7) * 1e3}[target]
    g, o = fit_both(X, y.astype(np.float32), algorithm=RF, task=capi.REGRESSION, n_trees=4, k=2)
    assert_same_forest(g, o)


def test_rf_retries_on_sparse_features():
    rng = np.random.default_rng(9)
    X = (rng.random((40, 3000)) < 0.004).astype(np.float32)
    X[0] = rng.random(3000)
    y = (rng.random(3000) < 0.02).astype(np.float32)
    g, o = fit_both(X, y, algorithm=RF, n_trees=6, k=2, min_node_size=1)
    assert_same_forest(g, o)


@pytest.mark.parametrize("kind", ["4", "24", "reg"])
def test_rf_chunk_pipeline_tiles_and_single_key_buckets(kind):
    """Roots of two tiles; features of fewer values than buckets (a bucket a
    key) beside continuous ones."""
    rng = np.random.default_rng(13)
    n = 45_000
    X = rng.random((6, n)).astype(np.float32)
    X[3] = np.floor(X[3] * 2)
    X[4] = np.floor(X[4] * 300)
    X[5] = np.floor(X[5] ** 4 * 3000)
    kw, y = _targets(kind, X, rng)
    g, o = fit_both(X, y.astype(np.float32), algorithm=RF, n_trees=2, k=3, max_depth=9, **kw)
    assert_same_forest(g, o)


@pytest.mark.parametrize("kind,n,f,k", [("5", 2_100_011, 16, 6), ("reg", 1_770_001, 19, 10)])
def test_rf_keys_gathered_by_row(kind, n, f, k):
    """Large enough for the row-major keys; deep enough for every tier that
    reads the gathered keys."""
    rng = np.random.default_rng(17)
    X = rng.random((f, n), dtype=np.float32)
    X[3] = np.floor(X[3] * 7)
    kw, y = _targets(kind, X, rng)
    g, o = fit_both(X, y.astype(np.float32), algorithm=RF, n_trees=1, k=k, max_depth=15, **kw)
    assert_same_forest(g, o)


@pytest.mark.parametrize("task", [capi.CLASSIFICATION, capi.REGRESSION])
@pytest.mark.parametrize("n", [255, 2049, 65_536, 65_537, 140_001])
def test_ert_nodes_around_the_walk_and_side_words(task, n):
    """Extra trees' roots hold every row: one step of a wave's or workgroup's
    walk more or less, and one or several spans of the partition's side words."""
    if task == capi.REGRESSION:
        X, y = synth.sine_regression(seed=n, n=n, f=6)
    else:
        X, y = synth.gaussian_classes(seed=n, n=n, f=6, n_informative=4, n_classes=3)
    g, o = fit_both(X, y, algorithm=ERT, task=task, n_trees=2, k=3, max_depth=6, n_classes=3)
    assert_same_forest(g, o)


@pytest.mark.parametrize("task", [capi.CLASSIFICATION, capi.REGRESSION])
@pytest.mark.parametrize("depth", [1, 2, 12])
def test_export_equals_the_canonical_arrays(task, depth):
    """Roots first, then each tree's other nodes in order; leaves' payloads in
    node order.  Depth 1: trees of a single node."""
    if task == capi.REGRESSION:
        X, y = synth.sine_regression(seed=3, n=900, f=5)
    else:
        X, y = synth.gaussian_classes(seed=3, n=900, f=5, n_informative=4, n_classes=3)
    p = capi.default_params(RF, task=task, n_trees=7, n_features_per_node=2, max_depth=depth,
                            n_classes=0 if task else 3, seed=2)
    g = capi.fit(X, y, p)
    c = g.canonical()
    nodes, probs = g.export()
    ts = c["tree_start"]
    order = np.concatenate([ts[:-1]] + [np.arange(a + 1, b) for a, b in zip(ts[:-1], ts[1:])])
    where = np.empty(g.n_nodes, np.int64)
    where[order] = np.arange(g.n_nodes)
    inner = c["feature"][order] >= 0
    assert np.array_equal(nodes["attribute"][inner], c["feature"][order][inner])
    assert np.array_equal(nodes["split_point"][inner], c["threshold"][order][inner])
    assert np.array_equal(nodes["child_start"][inner], where[c["left"][order][inner]])
    assert np.array_equal(nodes["child_count"], np.where(inner, 2, 0))
    leaf = order[~inner]
    width = 1 if task else 3
    assert np.array_equal(nodes["probability_start"][~inner], width * np.arange(leaf.size))
    if task:
        assert np.array_equal(probs, c["value"][leaf])
    else:
        assert np.array_equal(probs, c["class_counts"].reshape(-1, 3)[leaf].ravel().astype(np.float32))


@pytest.mark.parametrize("task", [capi.CLASSIFICATION, capi.REGRESSION])
@pytest.mark.parametrize("rows", [1, 2, 3, 16, 17, 64, 128, 129, 1001])
def test_predict_row_counts(task, rows):
    """Both sides of every change of rows per block, and a ragged last block;
    the call without allocations takes the same kernels."""
    if task == capi.REGRESSION:
        X, y = synth.sine_regression(seed=4, n=1500, f=7)
        Xp, _ = synth.sine_regression(seed=5, n=rows, f=7)
    else:
        X, y = synth.gaussian_classes(seed=4, n=1500, f=7, n_informative=4, n_classes=5)
        Xp, _ = synth.gaussian_classes(seed=5, n=rows, f=7, n_informative=4, n_classes=5)
    g, o = fit_both(X, y, algorithm=RF, task=task, n_trees=70, k=2, max_depth=14, min_node_size=1, n_classes=5)
    want = o.predict(Xp)
    got = g.predict(Xp), g.predict_noalloc(Xp)
    for v in got:
        assert np.array_equal(np.asarray(v, np.float64), np.asarray(want, np.float64))


@pytest.mark.parametrize("shape", ["full", "chain", "mixed"])
@pytest.mark.parametrize("depth", [0, 1, 8, 9, 10, 12, 13, 17])
def test_predict_over_the_top_levels_and_clusters(shape, depth):
    """Trees that end above, at and below the level where clusters begin, with
    full, one-sided and random subtrees."""
    if shape == "full" and depth > 13:
        depth = 14
    rng = np.random.default_rng(depth)
    trees, f, rows = 3, 5, 200
    nodes, front, base = [], trees, 0
    for level in range(depth + 1):
        if level == depth:
            split = np.zeros(front, bool)
        elif shape == "full":
            split = np.ones(front, bool)
        elif shape == "chain":
            split = np.arange(front) % 2 == level % 2 if level else np.ones(front, bool)
        else:
            split = rng.random(front) < (0.95 if level < 5 else 0.6)
        lv = np.zeros(front, capi.NODE_DTYPE)
        lv["child_start"] = np.where(split, base + front + 2 * (np.cumsum(split) - 1), -1)
        lv["child_count"] = np.where(split, 2, 0)
        lv["attribute"] = np.where(split, rng.integers(0, f, front), -1)
        lv["split_point"] = np.where(split, rng.uniform(0.2, 0.8, front), -1).astype(np.float32)
        nodes.append(lv)
        base += front
        front = 2 * int(split.sum())
        if not front:
            break
    nodes = np.concatenate(nodes)
    leaf = nodes["child_count"] == 0
    nodes["probability_start"] = np.where(leaf, np.cumsum(leaf) - 1, -1)
    value = rng.integers(-9, 10, int(leaf.sum())).astype(np.float32)  # sums are exact
    g = capi.import_forest(nodes, value, trees, 1, f, capi.REGRESSION)
    X = rng.random((f, rows), dtype=np.float32)
    want = np.zeros(rows)
    for t in range(trees):
        at = np.full(rows, t)
        while not leaf[at].all():
            n = nodes[at]
            right = X[np.maximum(n["attribute"], 0), np.arange(rows)] >= n["split_point"]
            at = np.where(leaf[at], at, n["child_start"] + right)
        want += value[nodes["probability_start"][at]]
    assert np.array_equal(g.predict(X), want.astype(np.float32))


def test_predict_with_wide_records():
    """A feature number and a pair number that do not fit 32 bits together."""
    rng = np.random.default_rng(6)
    f, depth, rows = 1 << 22, 9, 5
    n = 2 ** (depth + 1) - 1
    nodes = np.zeros(n, capi.NODE_DTYPE)
    inner = np.arange(n) < n // 2
    nodes["child_start"] = np.where(inner, 2 * np.arange(n) + 1, -1)
    nodes["child_count"] = np.where(inner, 2, 0)
    nodes["attribute"] = np.where(inner, rng.integers(0, f, n), -1)
    nodes["attribute"][0] = f - 1
    nodes["split_point"] = np.where(inner, 0.5, -1).astype(np.float32)
    nodes["probability_start"] = np.where(inner, -1, np.arange(n) - n // 2)
    value = rng.standard_normal(n - n // 2).astype(np.float32)
    g = capi.import_forest(nodes, value, 1, 1, f, capi.REGRESSION)
    X = rng.random((f, rows), dtype=np.float32)
    got = g.predict(X)
    for r in range(rows):
        i = 0
        while inner[i]:
            i = 2 * i + 1 + int(X[nodes["attribute"][i], r] >= 0.5)
        assert got[r] == value[i - n // 2]


@pytest.mark.parametrize("n,trees", [(40, 3), (1000, 64), (1000, 130)])
def test_out_of_bag_lists_over_tree_chunks(n, trees):
    """Fewer rows than a block, one chunk of trees and several."""
    X, y = synth.gaussian_classes(seed=n, n=n, f=6, n_informative=4, n_classes=3)
    p = capi.default_params(RF, n_trees=trees, n_features_per_node=2, max_depth=8, n_classes=3, seed=4)
    Xd = capi.DeviceArray.from_numpy(X)
    g = capi.fit_device(Xd.ptr, n, 6, y, p)
    o = pyoracle.fit(X, y, algorithm=RF, n_trees=trees, k=2, max_depth=8, n_classes=3, seed=4)
    for perm in (-1, 1):
        assert capi.oob_evaluate(g, Xd.ptr, y, n, perm) == pyoracle.oob_evaluate(o, X, y, seed=4, permuted_feature=perm)
    bad = y.copy()
    bad[n // 2] = 3
    with pytest.raises(Exception):
        capi.oob_evaluate(g, Xd.ptr, bad, n)
    bad[n // 2] = 0.5
    with pytest.raises(Exception):
        capi.oob_evaluate(g, Xd.ptr, bad, n)
    g.close()
    Xd.free()


def test_predict_of_a_file_out_of_level_order(tmp_path):
    """A forest file may hold a level's sibling pairs in another order than
    their parents': it loads, and predicts the same."""
    rng = np.random.default_rng(3)
    n = 31
    nodes = np.zeros(n, capi.NODE_DTYPE)
    inner = np.arange(n) < 15
    nodes["child_start"] = np.where(inner, 2 * np.arange(n) + 1, -1)
    nodes["child_count"] = np.where(inner, 2, 0)
    nodes["attribute"] = np.where(inner, rng.integers(0, 4, n), -1)
    nodes["split_point"] = np.where(inner, rng.uniform(0.2, 0.8, n), -1).astype(np.float32)
    nodes["probability_start"] = np.where(inner, -1, np.arange(n) - 15)
    value = np.arange(16, dtype=np.float32)
    g = capi.import_forest(nodes, value, 1, 1, 4, capi.REGRESSION)
    path = tmp_path / "forest"
    g.save(path)
    raw = bytearray(path.read_bytes())
    head = 8 + 4 + 8 * 4 + 3 * 8 + 16  # header, tree table of one tree
    order = np.arange(n)
    order[3:7] = [5, 6, 3, 4]
    cols = np.frombuffer(bytes(raw[head:head + 20 * n]), np.int32).reshape(5, n).copy()
    left = cols[2]  # feature, threshold, left, depth, value
    left[1], left[2] = left[2], left[1]
    raw[head:head + 20 * n] = cols[:, order].tobytes()
    h = 0xCBF29CE484222325
    for b in raw[:-8]:
        h = (h ^ b) * 0x100000001B3 & (2 ** 64 - 1)
    raw[-8:] = h.to_bytes(8, "little")
    path.write_bytes(bytes(raw))
    X = rng.random((4, 300), dtype=np.float32)
    assert np.array_equal(capi.load_forest(path).predict(X), g.predict(X))


@pytest.mark.parametrize("kind", ["2", "10", "reg"])
def test_rf_many_heavy_buckets(kind):
    """Roots of about 2,000 rows whose features have 35 or 36 common values
    among some 300 rare ones, and labels of noise: most common values weigh
    more than a wave's list, share their bucket with rare keys, and survive
    the bound, so many ranges wait to be split again (test_search_limits.py)."""
    rng = np.random.default_rng(21)
    n, f = 3150, 8
    X = np.empty((f, n), np.float32)
    for j in range(f):
        c = 35 + j % 2
        X[j] = np.where(rng.random(n) < 0.92, rng.integers(0, c, n) + 0.5, c * rng.random(n))
    kw = dict(task=capi.REGRESSION) if kind == "reg" else dict(n_classes=int(kind))
    y = rng.standard_normal(n) if kind == "reg" else rng.integers(0, int(kind), n)
    g, o = fit_both(X, y.astype(np.float32), algorithm=RF, n_trees=60, k=6, max_depth=4, **kw)
    assert_same_forest(g, o)


@pytest.mark.parametrize("n,trees,depth", [(1500, 800, 4), (40_000, 4, 5)])
@pytest.mark.parametrize("target", ["1e17", "3e18", "1e19", "1e25", "constant 1e-5", "constant 3e-7"])
def test_rf_regression_scores_at_the_ends_of_fp32(target, n, trees, depth):
    """Variances around and above the largest fp32 number: draws of different
    gains have the score infinity there, and the lowest feature wins.
    Variances of rounding alone, near the smallest.  Enough nodes for a
    node's draws to be searched one after the other."""
    rng = np.random.default_rng(n)
    X = rng.random((6, n)).astype(np.float32)
    X[4:] = np.floor(X[4:] * 5)
    if target.startswith("constant"):
        y = np.full(n, float(target.split()[1]))
    else:
        y = float(target) * (rng.standard_normal(n) + X[1])
    g, o = fit_both(X, y.astype(np.float32), algorithm=RF, task=capi.REGRESSION, n_trees=trees, k=3, max_depth=depth)
    assert_same_forest(g, o)


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("n,trees,depth", [(1500, 800, 4), (40_000, 4, 6)])
def test_rf_regression_with_a_target_that_is_not_finite(bad, n, trees, depth):
    """Such a target's fixed-point value is the least integer and sums wrap:
    no bound of a gain holds, the scores are those of the oracle's sums."""
    rng = np.random.default_rng(n)
    X = rng.random((6, n)).astype(np.float32)
    y = (rng.standard_normal(n) + X[1]).astype(np.float32)
    y[n // 3] = bad
    g, o = fit_both(X, y, algorithm=RF, task=capi.REGRESSION, n_trees=trees, k=3, max_depth=depth)
    assert_same_forest(g, o)


def test_import_of_a_root_that_is_another_trees_child():
    """Roots 1 and 2, leaves, are the children of root 0: they lie side by
    side, so the model stands, and exports as it came.  A root and another
    node as children cannot lie side by side: refused."""
    nodes = np.zeros(3, capi.NODE_DTYPE)
    nodes["attribute"] = [0, -1, -1]
    nodes["child_count"] = [2, 0, 0]
    nodes["child_start"] = [1, -1, -1]
    nodes["split_point"] = np.array([0.5, -1, -1], np.float32)
    nodes["probability_start"] = [-1, 0, 1]
    value = np.array([1, 10], np.float32)
    g = capi.import_forest(nodes, value, 3, 1, 2, capi.REGRESSION)
    X = np.random.default_rng(1).random((2, 500), dtype=np.float32)
    assert np.array_equal(g.predict(X), np.where(X[0] < 0.5, 12, 21).astype(np.float32))
    out, probs = g.export()
    assert out["child_start"][0] == 1 and out["child_count"][:3].tolist() == [2, 0, 0]
    assert probs[out["probability_start"][1]] == 1 and probs[out["probability_start"][2]] == 10
    g.close()
    with pytest.raises(Exception):  # roots 0 and 1, child 2 of root 0
        capi.import_forest(nodes, value, 2, 1, 2, capi.REGRESSION)


def _stumps(task):
    """Three trees of one split each, at 0.25, 0.5 and 0.75 of the only feature."""
    nodes = np.zeros(9, capi.NODE_DTYPE)
    inner = np.arange(9) < 3
    nodes["attribute"] = np.where(inner, 0, -1)
    nodes["child_count"] = np.where(inner, 2, 0)
    nodes["child_start"] = np.where(inner, 3 + 2 * np.arange(9), -1)
    nodes["split_point"] = np.where(inner, 0.25 * (1 + np.arange(9)), -1).astype(np.float32)
    width = 1 if task else 2
    nodes["probability_start"] = np.where(inner, -1, width * (np.arange(9) - 3))
    probs = np.array([1, 10] * 3 if task else [1, 0, 0, 1] * 3, np.float32)
    return capi.import_forest(nodes, probs, 3, width, 1, task)


def _repeated(values, n):
    """values, a prime number of them, over and over: no two blocks alike."""
    return np.resize(values, n)


@pytest.mark.parametrize("task,row_major", [(capi.CLASSIFICATION, 0), (capi.REGRESSION, 1)])
def test_predict_of_more_rows_than_a_launch_holds(task, row_major):
    """2^32 threads are 537 M rows at 64 a block of 512."""
    n = (1 << 29) + 777
    x = np.random.default_rng(1).random(1_000_003, dtype=np.float32)
    right = (x >= 0.25).astype(np.int32) + (x >= 0.5) + (x >= 0.75)
    g = _stumps(task)
    X = capi.DeviceArray.from_numpy(_repeated(x, n))
    width = 1 if task else 2
    out = np.full((n, width), -1, np.float32 if task else np.int32)
    D = capi.DeviceArray.from_numpy(out)
    p = ctypes.c_void_p
    capi._check(capi.lib().dte_predict_device(g.handle, p(X.ptr), n, 1 if row_major else n, row_major,
                                              None if task else p(D.ptr), p(D.ptr) if task else None, None))
    capi._check(capi.lib().dte_memcpy_to_host(0, p(out.ctypes.data), p(D.ptr), out.nbytes))
    if task:
        assert np.array_equal(out[:, 0], _repeated((3 + 9 * right).astype(np.float32), n))
    else:
        want = np.stack([3 - right, right], 1)
        assert np.array_equal(out.reshape(-1), _repeated(want, 2 * n))
    g.close()
    X.free()
    D.free()


def test_out_of_bag_of_more_rows_than_a_launch_holds(tmp_path):
    """Every row's label is what its tree says, so all pairs are right; a
    bootstrap leaves a row out with probability 1 / e."""
    n = (1 << 29) + 777
    Xf = np.linspace(0, 1, 64, dtype=np.float32).reshape(1, -1)
    g = capi.fit(Xf, (Xf[0] >= 0.5).astype(np.float32), capi.default_params(RF, n_trees=1, n_classes=2, max_depth=2))
    thr = float(g.canonical()["threshold"][0])
    path = tmp_path / "forest"
    g.save(path)
    g.close()
    raw = bytearray(path.read_bytes())
    at = 8 + 4 + 8 * 4 + 8  # fit_rows
    assert int.from_bytes(raw[at:at + 8], "little") == 64
    raw[at:at + 8] = n.to_bytes(8, "little")
    h = 0xCBF29CE484222325
    for b in raw[:-8]:
        h = (h ^ b) * 0x100000001B3 & (2 ** 64 - 1)
    raw[-8:] = h.to_bytes(8, "little")
    path.write_bytes(bytes(raw))
    g = capi.load_forest(path)
    x = np.random.default_rng(1).random(1_000_003, dtype=np.float32)
    y = _repeated((x >= thr).astype(np.float32), n)
    X = capi.DeviceArray.from_numpy(_repeated(x, n))
    pairs, good = capi.oob_evaluate(g, X.ptr, y, n)
    assert good == pairs
    # the count of rows left out has variance N (1 / e - 2 / e^2)
    assert abs(pairs - n / np.e) < 6 * np.sqrt(0.0973 * n)
    y[-1] = 1 - y[-1]
    y[0] = 1 - y[0]
    pairs2, good2 = capi.oob_evaluate(g, X.ptr, y, n)
    assert pairs2 == pairs and pairs - 2 <= good2 <= pairs
    g.close()
    X.free()


def _leave_free(left):
    """Allocations that leave about `left` bytes of the device free.  (What is
    left after a large one may be more than was free beside it: twice.)"""
    hip = ctypes.CDLL("libamdhip64.so.7")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    fill = []
    for _ in range(2):
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        if free.value > left + (20 << 20):
            fill.append(capi.DeviceArray(free.value - left))
    return fill


def test_a_second_fit_takes_the_row_major_keys_like_the_first():
    """The scratch that a fit leaves cached is free to the next one: with
    little other memory it must not turn the row-major keys away."""
    n, f, k = 2_100_011, 16, 6
    rng = np.random.default_rng(17)
    X = capi.DeviceArray.from_numpy(rng.random((f, n), dtype=np.float32))
    y = rng.integers(0, 5, n).astype(np.float32)
    p = capi.default_params(RF, n_trees=1, n_features_per_node=k, max_depth=6, n_classes=5)

    def gathers():
        capi.profile_reset()
        capi.profiling(True)
        g = capi.fit_device(X.ptr, n, f, y, p)
        capi.profiling(False)
        g.close()
        return capi.profile_stats().get("gather_draws", {"launches": 0})["launches"]

    capi.release_cached_memory()
    first = gathers()
    assert first > 0
    scratch = capi.release_cached_memory()
    fill = _leave_free(scratch + (600 << 20))
    try:
        assert gathers() == first
        assert gathers() == first
    finally:
        for b in fill:
            b.free()
        X.free()
        capi.release_cached_memory()


def test_cached_scratch_gives_way_to_allocations_of_the_library():
    """What an out-of-bag pass and a fit leave cached is no loss to a caller
    of the library who needs the memory."""
    n, f = 1_000_003, 32
    rng = np.random.default_rng(2)
    X = capi.DeviceArray.from_numpy(rng.random((f, n), dtype=np.float32))
    y = rng.integers(0, 3, n).astype(np.float32)
    g = capi.fit_device(X.ptr, n, f, y, capi.default_params(RF, n_trees=4, max_depth=4, n_classes=3))
    capi.release_cached_memory()
    fill = _leave_free(1 << 30)
    try:
        capi.oob_evaluate(g, X.ptr, y, n)
        h = capi.fit_device(X.ptr, n, f, y, capi.default_params(RF, n_trees=1, max_depth=2, n_classes=3))
        h.close()
        held = capi.DeviceArray(900 << 20)  # more than is left beside the scratch
        held.free()
    finally:
        for b in fill:
            b.free()
        X.free()
        g.close()
        capi.release_cached_memory()


@pytest.mark.parametrize("f", [9, 200, 600])
@pytest.mark.parametrize("task", [capi.CLASSIFICATION, capi.REGRESSION])
def test_predict_of_many_rows_by_a_big_model(task, f):
    """Models of more than 6 Mi nodes under 4,096 row blocks and more walk in
    blocks of fewer threads, with 64, 32 and no rows in LDS; the same rows, a
    few at a time, take the others."""
    trees, depth = 97, 15
    per = 2 ** (depth + 1) - 1
    rng = np.random.default_rng(f)
    n = trees * per
    assert n >= 6 << 20
    k = np.arange(per)
    inner = k < per // 2
    where = lambda t, i: np.where(i == 0, t, trees + t * (per - 1) + i - 1)
    nodes = np.zeros(n, capi.NODE_DTYPE)
    for t in range(trees):
        at = where(t, k)
        nodes["child_start"][at] = np.where(inner, where(t, 2 * k + 1), -1)
        nodes["child_count"][at] = np.where(inner, 2, 0)
        nodes["attribute"][at] = np.where(inner, rng.integers(0, f, per), -1)
        nodes["split_point"][at] = np.where(inner, 0.5, -1)
    leaf = nodes["child_count"] == 0
    width = 1 if task else 3
    nodes["probability_start"] = np.where(leaf, width * (np.cumsum(leaf) - 1), -1)
    probs = rng.integers(0, 9, width * int(leaf.sum())).astype(np.float32)  # sums are exact
    g = capi.import_forest(nodes, probs, trees, width, f, task)
    rows = 64 * 4096 + 33
    X = rng.random((f, 2048), dtype=np.float32)
    few = g.predict(X)
    got = g.predict(_repeated(X.T, rows * f).reshape(rows, f).T.copy()).reshape(rows, -1)
    assert np.array_equal(got, _repeated(few.reshape(2048, -1), got.size).reshape(got.shape))
    x, total = X[:, :40], np.zeros(40)
    for t in range(trees):
        at = np.full(40, t)
        for _ in range(depth):
            d = nodes[at]
            at = d["child_start"] + (x[d["attribute"], np.arange(40)] >= 0.5)
        p = nodes["probability_start"][at]
        if task:
            total += probs[p]
        else:
            total += probs[p[:, None] + np.arange(3)].argmax(1) == 1
    assert np.array_equal(few.reshape(2048, -1)[:40, 0 if task else 1], total.astype(np.float32))
    g.close()


def test_calls_of_other_threads_while_a_fit_records_its_level_steps():
    """Fits of small data record graphs; predictions, exports and other fits
    of the same device run beside them and share the library's stream."""
    X, y = synth.gaussian_classes(seed=3, n=3000, f=8, n_informative=5, n_classes=3)
    params = {a: capi.default_params(a, n_trees=6, n_classes=3, seed=4) for a in (RF, ERT)}
    want = {a: capi.fit(X, y, params[a]) for a in (RF, ERT)}
    canon = {a: want[a].canonical() for a in want}
    votes = {a: want[a].predict(X) for a in want}
    nodes = {a: want[a].export()[0].tobytes() for a in want}
    errors = []

    def fits(a):
        for _ in range(40):
            g = capi.fit(X, y, params[a])
            c = g.canonical()
            g.close()
            if not all(np.array_equal(c[k], canon[a][k]) for k in ("feature", "threshold", "left", "rowhash")):
                errors.append("fit")

    def uses(a):
        for _ in range(150):
            if not np.array_equal(want[a].predict(X), votes[a]):
                errors.append("predict")
            if want[a].export()[0].tobytes() != nodes[a]:
                errors.append("export")

    def run(fn, a):
        try:
            fn(a)
        except Exception as e:  # noqa: BLE001
            errors.append(repr(e))

    threads = [threading.Thread(target=run, args=(fn, a)) for fn in (fits, uses) for a in (RF, ERT)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[:3]
