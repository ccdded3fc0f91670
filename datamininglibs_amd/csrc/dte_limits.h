// Limits that LDS arrays are sized by: the bounded split search and the
// out-of-bag pass.  Plain C++: host code can check them without the kernels.
#pragma once

#include <cstdint>

namespace dte {

constexpr int kBoundRun = 64;          // entries that one wave ranks and scores at a time
constexpr int kBoundWeight = 65535;    // largest weight of a bounded node: class counts are 16 bits

// The workgroup tier counts a bucket's weight (bootstrap multiplicities), not
// its entries, so it splits a bucket again once its weight passes a run.  The
// ranges on its stack are disjoint, and a range popped makes room for its own
// parts: a node's weight bounds them, however few entries it has (2,048
// bootstrapped entries weigh about 3,240: 49 ranges).
constexpr bool team_splits_again(unsigned weight, int shift) { return weight > (unsigned)kBoundRun && shift > 0; }
constexpr int kTeamStack = kBoundWeight / (kBoundRun + 1);

// The wave tier decides by entries, and a node's entries bound its ranges.
constexpr int wave_stack(int entries) { return entries / (kBoundRun + 1); }

// Rows whose in-bag bits a workgroup of the out-of-bag pass holds, and their
// words: at most 64 KB, what any launch may have.
constexpr int64_t kBagRange = (int64_t)1 << 19;
constexpr int64_t bag_lds_bytes(int64_t rows) { return ((rows < kBagRange ? rows : kBagRange) + 31) / 32 * 4; }
static_assert(bag_lds_bytes(kBagRange) == 65536, "");

}  // namespace dte
