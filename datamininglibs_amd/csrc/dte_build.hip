// Level-wise tree-ensemble build for MI355X (gfx950).
//
// Replaces the device side of the reference's build (lib_ensembles/source/
// gpudte_algorithm.cc:14-267 driving gpurf.cu / gpuert.cu / gpudte.cu):
//
//   reference                               here
//   kSetupKernel (cuRAND states)            counter-based Philox, no state
//   kInitTreeBatch (bootstrap, 1 blk/tree)  k_boot_count + k_boot_compact
//   kFindSplit (1 64-lane block per node)   k_search_rf / k_search_ert over
//                                           (node, feature draw) items of all
//                                           trees of a level
//   kPerformSplit (atomic slots)            k_partition: stable compaction
//   host node cache + frame swapping        level arrays resident in HBM
//
// Layout in HBM during a fit:
//   X     fp32 [F][N]    feature-major samples (canonical: -0 -> +0)
//   K     u32  [F][N]    dense rank of X[f][row] among the distinct values of
//                        feature f (random forest only)
//   SV    fp32 [sum S_f] distinct sorted values of each feature
//   rows  u32  [E]       entries: in-bag rows of every tree, ascending row id
//                        inside every node (E = sum over trees of distinct
//                        bootstrap rows), ping-pong A/B between levels
//   aux   u32  [E]       label << 16 | bootstrap multiplicity
//   ey    i64  [E]       fixed-point target of the entry (regression)
//   nodes: level-major SoA (tree, id, depth, count, m, stats, hash, split)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <numeric>
#include <thread>
#include <type_traits>
#include <cstdlib>
#include <chrono>
#include <memory>
#include <utility>

#include "dte_block.h"
#include "dte_internal.h"
#include "dte_limits.h"

namespace dte {

__device__ LnTable g_ln_table;
const LnTable& host_ln_table();

namespace {

constexpr int kIpt = 8;                 // elements per thread in the LDS sort
constexpr int kCap = kBlock * kIpt;     // LDS chunk capacity (2048)
constexpr int kHistWords = 8192;        // LDS histogram words (32 KB)
constexpr int kMaxBuckets = 2048;       // bucket table of the big-item path
constexpr uint32_t kNone = 0xFFFFFFFFu;

__device__ __forceinline__ void load_ln_table(double* s_inv, double* s_logc) {
  const int t = threadIdx.x;
  if (t < 128) s_inv[t] = g_ln_table.inv[t];
  else s_logc[t - 128] = g_ln_table.logc[t - 128];
}

// ------------------------------------------------------------- args -----
constexpr int kMaxTiers = 7;
constexpr int kTfMax = 4096;  // entries of the fp32 x ln x table
struct DataArgs {
  const float* X;
  const uint32_t* K;
  const float* SV;
  const int64_t* SVoff;
  const uint32_t* S;
  int64_t N;
  int F;
  int C;
  int shift;
  uint64_t seed;
  int min_node;
  int max_depth;
  int igF;           // fixed-point shift of the x ln x terms (per fit)
  const int64_t* T;  // T[x] = xlnx_fixed(x, igF) for x <= Tmax (classification)
  int64_t Tmax;
  const float* Tf;   // x ln x in fp32 for x < kTfMax (bounds of the random-forest search)
  int no_bound;      // regression: a target is not finite, so sums wrap and only exact scores count
  // Joint build of several extra-trees forests in one set of level steps:
  // the data of batch tree t is forests[forest_of_tree[t]], whose D0 / R
  // are its mandatory and retry draws; C is the joint class width in every
  // forest's entry (classes past a forest's own count hold zero counts,
  // which add nothing to the entropy sums).  NULL for a fit of one forest.
  const struct DataArgs* forests;
  const int32_t* forest_of_tree;
  int D0, R;
};

__device__ __forceinline__ DataArgs forest_data(const DataArgs& d, int tree) {
  return d.forests ? d.forests[d.forest_of_tree[tree]] : d;
}

// Counts and offsets of the level being built, in device memory, for the
// level steps that run without a host round trip (captured in a hipGraph and
// replayed level after level): the kernels read them at entry instead of
// taking them as launch arguments.
struct alignas(128) DevLevel {
  int64_t off;                    // level-major offset of the level
  int64_t n;                      // nodes of the level
  int64_t depth;
  unsigned int n_open;            // open nodes (total of the open-flag scan)
  unsigned int n_next;            // nodes of the next level
  unsigned int tier[kMaxTiers];   // split-search tier sizes, first phase
  unsigned int ptier[kMaxTiers];  // partition tier sizes
  unsigned int rtier[kMaxTiers];  // split-search tier sizes, retry phase
};

struct LevelArgs {
  // level node slice (level-local index i)
  const int32_t* tree;   // batch tree index
  const uint32_t* id;    // tree-local level-order id
  const int32_t* count;  // sum of weights
  const int32_t* m;      // entries
  const uint32_t* cls;   // class counts [i * C]
  const int64_t* sum;    // regression fixed-point sum
  const int64_t* start;  // entry start (current buffer)
  const uint32_t* open_idx;  // open position -> level index
  const int32_t* tree_global;
  const uint32_t* row;   // current entry buffer
  const uint32_t* aux;
  const int64_t* ey;
  // device-described level: the slice pointers above are the level-major
  // bases and *off_dev the level's offset (NULL: already offset)
  const int64_t* off_dev;
};

struct ItemArgs {
  const uint32_t* list;  // optional: item group -> open position
  int64_t n_groups;
  int per_group;         // draws per group in this phase
  int j0;                // first draw index of this phase
  int D;                 // result stride per open node
  float* res_score;
  float* res_thr;
  int32_t* res_feat;
  unsigned long long* bytes;  // algorithmic bytes counter (NULL unless the profile is on)
  int node_major;        // 1: a grid of n_groups teams, each team walks its own group's draws in order
  uint32_t* scr_key;     // big-item scratch, one slab per block
  uint32_t* scr_aux;
  int64_t* scr_y;
  int64_t scr_stride;
  const unsigned int* n_dev;  // device-described level: n_groups = *n_dev
  int spread;            // waves to keep busy (node_split)
  const uint32_t* gk;    // keys of the phase's draws by entry: draw q of entry e at gk[q * gk_stride + e]
  int64_t gk_stride;     // (NULL: gathered from K; see k_gather_draws)
};

// Parts that a node's draws are dealt to, so that `units` teams have work: a
// level of few nodes is bound by the latency of one node's draws in a row
// (about 8 us a draw), and its chip is idle.  With enough nodes a team takes
// all draws of its node: later draws then profit from what earlier ones found.
__device__ __forceinline__ int node_split(const ItemArgs& it, int64_t units, int64_t nodes) {
  const int64_t s = nodes > 0 ? units / nodes : 1;
  return (int)(s < 1 ? 1 : (s < it.per_group ? s : it.per_group));
}

// Counts a wave's algorithmic bytes for the profile.  Atomics on one address
// pass at one in about 15 ns: a grid's 16 k waves on one counter took 250 us
// of every tier, so a counter is kByteSlots words, one line each, and there
// is none outside a profile.
constexpr int kByteSlots = 64;
constexpr int kByteStride = 16;
constexpr int kByteWords = kByteSlots * kByteStride;  // of one counter
__device__ __forceinline__ void add_bytes(unsigned long long* counter, unsigned long long v) {
  atomicAdd(counter + (blockIdx.x & (kByteSlots - 1)) * kByteStride, v);
}

// Level slice and item count of a device-described level (a no-op for
// launches whose arguments carry them).
__device__ __forceinline__ void resolve_level(LevelArgs& lv, int C) {
  if (lv.off_dev) {
    const int64_t off = *lv.off_dev;
    lv.tree += off;
    lv.id += off;
    lv.count += off;
    lv.m += off;
    if (lv.cls) lv.cls += off * C;
    if (lv.sum) lv.sum += off;
    lv.off_dev = nullptr;
  }
}
__device__ __forceinline__ void resolve_items(ItemArgs& it) {
  if (it.n_dev) it.n_groups = *it.n_dev;
}

// Draw index of item position q of a node whose forest data is dd: j0 + q
// for a fit of one forest.  A joint build pads every node to the widest
// forest's draws: the first phase covers draws 0 .. D0-1 of the node's own
// forest, the retry phase (j0 > 0) its draws D0 .. D0+R-1; -1 marks a
// position past them.
__device__ __forceinline__ int item_draw(const DataArgs& d, const DataArgs& dd, const ItemArgs& it, int q) {
  if (!d.forests) return it.j0 + q;
  if (it.j0 == 0) return q < dd.D0 ? q : -1;
  return q < dd.R ? dd.D0 + q : -1;
}

// ------------------------------------------------- per-node context -----
// Fixed-point x ln x with the fit-wide shift F.  Counts never exceed the
// root's total weight, so a per-fit table T[x] = xlnx_fixed(x, F) for
// x <= Tmax (built by k_build_T with the same function) answers every
// lookup with one cached load; counts above a capped table fall back to the
// computation -- the same bits either way.
__device__ __attribute__((noinline)) int64_t xlnx_fixed_slow(uint64_t x, int F, const double* inv,
                                                           const double* logc) {
  return xlnx_fixed(x, F, inv, logc);
}

struct LnCtx {
  const double* inv;
  const double* logc;
  const int64_t* T;
  int64_t Tmax;
  int F;
  __device__ __forceinline__ int64_t t(uint64_t x) const {
    return x <= (uint64_t)Tmax ? T[x] : xlnx_fixed_slow(x, F, inv, logc);
  }
};

// The same with a copy of T[0, nTL) in LDS, for kernels whose nodes are
// small (their lookups mostly fall below nTL).
struct LnCtxL {
  const double* inv;
  const double* logc;
  const int64_t* T;
  int64_t Tmax;
  int F;
  const int64_t* TL;
  int64_t nTL;
  __device__ __forceinline__ int64_t t(uint64_t x) const {
    if (x < (uint64_t)nTL) return TL[x];
    return x <= (uint64_t)Tmax ? T[x] : xlnx_fixed_slow(x, F, inv, logc);
  }
};

// Stages T[0, min(n, Tmax + 1)) into LDS; returns the staged length (0 when
// the fit has no table: regression).
template <int NT>
__device__ __forceinline__ int64_t load_t_prefix(int64_t* s_T, const int64_t* T, int64_t Tmax) {
  if (!T) return 0;
  const int64_t n = Tmax + 1 < NT ? Tmax + 1 : NT;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) s_T[i] = T[i];
  return n;
}

struct NodeCtx {
  int64_t n;        // sum of weights
  int64_t ssum;     // regression: fixed-point target sum
  int64_t P;        // classification: T(n) - sum_c T(n_c)
  double inv;       // 1 / (n ln 2)
  int C;
};

template <int MAXC, int TASK>
struct Carry {
  uint32_t run[MAXC];  // classification: class counts before the chunk
  int64_t run_n;       // weights before the chunk
  int64_t run_s;       // regression: target sum before the chunk
  uint32_t last_key;   // last key before the chunk (valid if run_n > 0)
  double best_g;
  uint32_t best_key;
  uint32_t best_prev;
};

// Per-team LDS of the sorted-chunk evaluator.
template <int MAXC, int TASK, int TEAM, int IPT>
struct TeamLds {
  static constexpr int CAP = TEAM * IPT;
  // 16-bit counters: 16 radix digits per thread, or the packed counters of a
  // counting sort over a key span of up to SPAN.
  static constexpr int SPAN = 16 * TEAM > (4 * CAP < 2048 ? 4 * CAP : 2048) ? 16 * TEAM
                                                                           : (4 * CAP < 2048 ? 4 * CAP : 2048);
  union {
    struct {
      uint32_t k[2][CAP];
      uint16_t v[2][CAP];
      uint16_t cnt[SPAN];
    } srt;
    uint32_t hist[TEAM == 256 ? kHistWords : 1];
    uint32_t bpos[TEAM == 256 ? kMaxBuckets : 1];
  } u;
  uint32_t aux[CAP];
  int64_t y[TASK == 1 ? CAP : 1];
  // Per-lane class columns [c * TEAM + t] of the walk; a wave team of up to
  // 16 classes keeps them in the sort counters, free once the chunk is sorted.
  static constexpr bool kColsInCnt = TEAM == kWave && MAXC * TEAM * 4 <= SPAN * 2;
  uint32_t pre[TASK == 0 && !kColsInCnt ? MAXC * TEAM : 1];
  uint32_t ncls[MAXC];
  uint32_t ctot[MAXC];
  uint32_t last[TEAM == kWave ? 1 : TEAM];  // histogram walk of whole-workgroup teams
  __device__ __forceinline__ uint32_t* cols() {
    if constexpr (kColsInCnt) {
      return reinterpret_cast<uint32_t*>(u.srt.cnt);
    } else {
      return pre;
    }
  }
  __device__ __forceinline__ const uint32_t* cols() const { return const_cast<TeamLds*>(this)->cols(); }
  uint32_t w[8 * kWaves + kWaves];
  int64_t w64[kWaves];
  int64_t w64v[4 * kWaves];
  double bg[kWaves];
  uint32_t bk[kWaves];
  uint32_t bp[kWaves];
  Carry<MAXC, TASK> cr;
};

// Exclusive scan of the per-lane class columns pre[c][t] across the team,
// plus the carry; chunk totals go to ctot[c].
template <int G, int MAXC, int TASK, int TEAM, int IPT>
__device__ __forceinline__ void scan_class_group(TeamLds<MAXC, TASK, TEAM, IPT>& L, int c0, int C) {
  const int t = team_tid<TEAM>();
  uint32_t v[G], tot[G];
#pragma unroll
  for (int q = 0; q < G; ++q) v[q] = (c0 + q < C) ? L.cols()[(c0 + q) * TEAM + t] : 0u;
  team_excl_scan_vec<TEAM, G>(v, L.w, tot);
#pragma unroll
  for (int q = 0; q < G; ++q)
    if (c0 + q < C) {
      L.cols()[(c0 + q) * TEAM + t] = v[q] + L.cr.run[c0 + q];
      if (t == 0) L.ctot[c0 + q] = tot[q];
    }
}

// Groups of 8 columns, then one group of 4, 2 or 1 for the rest, so that C
// classes take C scans.
template <int MAXC, int TASK, int TEAM, int IPT>
__device__ void scan_class_columns(TeamLds<MAXC, TASK, TEAM, IPT>& L, int C) {
  int c0 = 0;
  if constexpr (MAXC >= 8)
    for (; c0 + 8 <= C; c0 += 8) scan_class_group<8>(L, c0, C);
  while (c0 < C) {
    const int r = C - c0;
    if (MAXC >= 4 && r > 2) {
      scan_class_group<4>(L, c0, C);
      c0 += 4;
    } else if (r == 2) {
      scan_class_group<2>(L, c0, C);
      c0 += 2;
    } else {
      scan_class_group<1>(L, c0, C);
      c0 += 1;
    }
  }
}

// Incremental state of one lane's walk: exact fixed-point sums of the left
// and right x ln x terms.
struct WalkState {
  int64_t sl, sr;
  int64_t nl;
};

template <int MAXC, int TASK, int TEAM, int IPT, class LX>
__device__ __forceinline__ WalkState walk_init(const TeamLds<MAXC, TASK, TEAM, IPT>& L, const NodeCtx& nc,
                                               const LX& lx) {
  const int t = team_tid<TEAM>();
  WalkState w{0, 0, 0};
  for (int c = 0; c < nc.C; ++c) {
    const uint32_t l = L.cols()[c * TEAM + t];
    w.nl += l;
    w.sl += lx.t(l);
    w.sr += lx.t(L.ncls[c] - l);
  }
  return w;
}

template <class LX>
__device__ __forceinline__ double walk_gain(const WalkState& w, const NodeCtx& nc, const LX& lx) {
  const int64_t q = (w.sl - lx.t((uint64_t)w.nl)) + (w.sr - lx.t((uint64_t)(nc.n - w.nl)));
  return ig_from_fixed(nc.P + q, lx.F, nc.inv);
}

template <int MAXC, int TASK, int TEAM, int IPT, class LX>
__device__ __forceinline__ void walk_add(WalkState& w, TeamLds<MAXC, TASK, TEAM, IPT>& L, int lab, uint32_t add,
                                         const LX& lx) {
  const int t = team_tid<TEAM>();
  const uint32_t lo = L.cols()[lab * TEAM + t];
  const uint32_t ln = lo + add;
  L.cols()[lab * TEAM + t] = ln;
  const uint32_t tot = L.ncls[lab];
  w.sl += lx.t(ln) - lx.t(lo);
  w.sr += lx.t(tot - ln) - lx.t(tot - lo);
  w.nl += add;
}

template <int MAXC, int TASK>
__device__ __forceinline__ void carry_best(Carry<MAXC, TASK>& cr, const BestCand& b) {
  if (b.key != kNone && cand_better(b.g, b.key, cr.best_g, cr.best_key)) {
    cr.best_g = b.g;
    cr.best_key = b.key;
    cr.best_prev = b.prev;
  }
}

// Classification walk of a key-sorted chunk on a one-wave team.  The class
// counts before each position come from the per-lane class columns (lane t
// owns a run of consecutive positions) and go to LDS; the x ln x reads and
// the running sums then go row by row, lane t on position 64 * i + t, so
// that the 64 reads of one instruction are at neighbouring counts (a few
// cache lines) instead of 64 runs ipt positions apart.  The candidates and
// their order are those of the run-per-lane walk: positions ascend within a
// lane, and the best candidate is a maximum under a total order.
template <int MAXC, int TASK, int IPT, class LX>
__device__ void eval_sorted_wave(const uint32_t* keys, const uint16_t* vals, int n, uint32_t kbase,
                                 const NodeCtx& nc, TeamLds<MAXC, TASK, kWave, IPT>& L, const LX& lx) {
  const int t = threadIdx.x & (kWave - 1);
  const int ipt = lane_span<kWave>(n);
  const int lo = t * ipt;
  const int hi = min(lo + ipt, n);
  // Counts before each position, in the key buffer the sort left free.
  uint32_t* lbp = keys == L.u.srt.k[0] ? L.u.srt.k[1] : L.u.srt.k[0];
  for (int c = 0; c < nc.C; ++c) L.cols()[c * kWave + t] = 0;
  for (int p = lo; p < hi; ++p) {
    const uint32_t a = L.aux[vals[p]];
    L.cols()[(a >> 16) * kWave + t] += a & 0xFFFFu;
  }
  scan_class_columns<MAXC, TASK, kWave, IPT>(L, nc.C);
  for (int p = lo; p < hi; ++p) {
    const uint32_t a = L.aux[vals[p]];
    const int c = (int)(a >> 16);
    const uint32_t l = L.cols()[c * kWave + t];
    lbp[p] = l;
    L.cols()[c * kWave + t] = l + (a & 0xFFFFu);
  }
  // Left and right sums and the weight before the chunk (one class per lane).
  int64_t s0 = 0;
  uint32_t n0 = 0;
  if (t < nc.C) {
    n0 = L.cr.run[t];
    s0 = lx.t(n0) + lx.t(L.ncls[t] - n0);
  }
  s0 = wave_last_i64(wave_incl_scan_i64(s0));
  n0 = wave_last(wave_incl_scan(n0));
  team_sync<kWave>();
  // Row pass 1: every x ln x read of the chunk, independent of each other.
  const int rows = (n + kWave - 1) / kWave;
  int64_t dd[IPT], tq[IPT];
  uint32_t nrun = n0;
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    dd[i] = 0;
    tq[i] = 0;
    if (i < rows) {
      const int p = i * kWave + t;
      uint32_t w = 0, lb = 0, tc = 0;
      if (p < n) {
        const uint32_t a = L.aux[vals[p]];
        w = a & 0xFFFFu;
        lb = lbp[p];
        tc = L.ncls[a >> 16];
      }
      const uint32_t inc = wave_incl_scan(w);
      const uint32_t nlb = nrun + inc - w;
      nrun += wave_last(inc);
      if (p < n) {
        dd[i] = (lx.t(lb + w) - lx.t(lb)) + (lx.t(tc - lb - w) - lx.t(tc - lb));
        tq[i] = nlb > 0 ? lx.t((uint64_t)nlb) + lx.t((uint64_t)(nc.n - nlb)) : -1;
      }
    }
  }
  // Row pass 2: running sums, the gain at each boundary between distinct keys.
  BestCand tb{0.0, kNone, kNone};
  int64_t best_pq = 0;
  int64_t srun = s0;
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    if (i < rows) {
      const int p = i * kWave + t;
      const int64_t inc = wave_incl_scan_i64(dd[i]);
      const int64_t before = srun + inc - dd[i];
      srun += wave_last_i64(inc);
      if (p < n && tq[i] >= 0) {
        const uint32_t k = keys[p] + kbase;
        const uint32_t prevk = p > 0 ? keys[p - 1] + kbase : L.cr.last_key;
        if (prevk < k) {
          const int64_t pq = nc.P + before - tq[i];
          if (pq > best_pq) {
            const double g = ig_from_fixed(pq, lx.F, nc.inv);
            if (g > tb.g) {
              tb = BestCand{g, k, prevk};
              best_pq = pq;
            }
          }
        }
      }
    }
  }
  const BestCand b = team_best<kWave>(tb, L.bg, L.bk, L.bp);
  if (t == 0) {
    carry_best(L.cr, b);
    for (int c = 0; c < nc.C; ++c) {
      L.cr.run[c] += L.ctot[c];
      L.cr.run_n += L.ctot[c];
    }
    if (n > 0) L.cr.last_key = keys[n - 1] + kbase;
  }
  team_sync<kWave>();
}

// Evaluate every boundary of a key-sorted chunk (keys relative to kbase,
// vals index the chunk's payload in L.aux / L.y).
template <int MAXC, int TASK, int TEAM, int IPT, class LX>
__device__ void eval_sorted_chunk(const uint32_t* keys, const uint16_t* vals, int n, uint32_t kbase,
                                  const NodeCtx& nc, TeamLds<MAXC, TASK, TEAM, IPT>& L, const LX& lx) {
  const int t = team_tid<TEAM>();
  const int ipt = lane_span<TEAM>(n);
  const int lo = t * ipt;
  const int hi = min(lo + ipt, n);
  BestCand tb{0.0, kNone, kNone};
  if constexpr (TASK == 0 && TEAM == kWave) {
    eval_sorted_wave<MAXC, TASK, IPT>(keys, vals, n, kbase, nc, L, lx);
  } else if constexpr (TASK == 0) {
    for (int c = 0; c < nc.C; ++c) L.cols()[c * TEAM + t] = 0;
    for (int p = lo; p < hi; ++p) {
      const uint32_t a = L.aux[vals[p]];
      L.cols()[(a >> 16) * TEAM + t] += a & 0xFFFFu;
    }
    scan_class_columns<MAXC, TASK, TEAM, IPT>(L, nc.C);
    // Three passes so that the x ln x lookups of all positions are
    // independent: (1) counts before each position, (2) the lane's deltas of
    // the left / right sums (plus one exclusive scan that gives every lane
    // its starting sums), (3) running sums and the gain at each boundary.
    uint32_t lb[IPT], tc[IPT], wv[IPT];
    int64_t nlb[IPT];
    if (lo < hi) {
      int64_t nl = 0;
      for (int c = 0; c < nc.C; ++c) nl += L.cols()[c * TEAM + t];
#pragma unroll
      for (int i = 0; i < IPT; ++i) {
        const int p = lo + i;
        if (p < hi) {
          const uint32_t a = L.aux[vals[p]];
          const int c = (int)(a >> 16);
          const uint32_t wt = a & 0xFFFFu;
          lb[i] = L.cols()[c * TEAM + t];
          L.cols()[c * TEAM + t] = lb[i] + wt;
          tc[i] = L.ncls[c];
          wv[i] = wt;
          nlb[i] = nl;
          nl += wt;
        }
      }
    }
    int64_t sc[4] = {0, 0, 0, 0};  // lane deltas of sl, sr; sums at the chunk start
    int64_t dl[IPT], dr[IPT];
    int64_t tq[IPT];  // T(nl) + T(n - nl) before each position, read with the deltas
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
      if (lo + i < hi) {
        dl[i] = lx.t(lb[i] + wv[i]) - lx.t(lb[i]);
        dr[i] = lx.t(tc[i] - lb[i] - wv[i]) - lx.t(tc[i] - lb[i]);
        tq[i] = nlb[i] > 0 ? lx.t((uint64_t)nlb[i]) + lx.t((uint64_t)(nc.n - nlb[i])) : 0;
        sc[0] += dl[i];
        sc[1] += dr[i];
      }
    }
    if (t < nc.C) {  // one class per lane
      sc[2] = lx.t(L.cr.run[t]);
      sc[3] = lx.t(L.ncls[t] - L.cr.run[t]);
    }
    int64_t tot[4];
    team_excl_scan_i64_vec<TEAM, 4>(sc, L.w64v, tot);
    if (lo < hi) {
      int64_t sl = tot[2] + sc[0], sr = tot[3] + sc[1];
      uint32_t prevk = (lo > 0) ? keys[lo - 1] + kbase : L.cr.last_key;
      // The gain is a non-decreasing function of the exact sum P + q, and a
      // later boundary only wins with a strictly larger gain: a sum below
      // the lane's best sum cannot win.
      int64_t best_pq = 0;
#pragma unroll
      for (int i = 0; i < IPT; ++i) {
        const int p = lo + i;
        if (p < hi) {
          const uint32_t k = keys[p] + kbase;
          if (nlb[i] > 0 && prevk < k) {
            const int64_t pq = nc.P + sl + sr - tq[i];
            if (pq > best_pq) {
              const double g = ig_from_fixed(pq, lx.F, nc.inv);
              if (g > tb.g) {
                tb = BestCand{g, k, prevk};
                best_pq = pq;
              }
            }
          }
          sl += dl[i];
          sr += dr[i];
          prevk = k;
        }
      }
    }
    const BestCand b = team_best<TEAM>(tb, L.bg, L.bk, L.bp);
    if (t == 0) {
      carry_best(L.cr, b);
      for (int c = 0; c < nc.C; ++c) {
        L.cr.run[c] += L.ctot[c];
        L.cr.run_n += L.ctot[c];
      }
      if (n > 0) L.cr.last_key = keys[n - 1] + kbase;
    }
    team_sync<TEAM>();
  } else {
    int64_t ln = 0, ls = 0;
    for (int p = lo; p < hi; ++p) {
      const uint16_t v = vals[p];
      const int64_t w = (int64_t)(L.aux[v] & 0xFFFFu);
      ln += w;
      ls += w * L.y[v];
    }
    int64_t tot_n, tot_s;
    int64_t pn = team_excl_scan_i64<TEAM>(ln, L.w64, &tot_n);
    int64_t ps = team_excl_scan_i64<TEAM>(ls, L.w64, &tot_s);
    pn += L.cr.run_n;
    ps += L.cr.run_s;
    if (lo < hi) {
      uint32_t prevk = (lo > 0) ? keys[lo - 1] + kbase : L.cr.last_key;
      for (int p = lo; p < hi; ++p) {
        const uint32_t k = keys[p] + kbase;
        if (pn > 0 && prevk < k) {
          const double g = variance_gain(pn, ps, nc.n - pn, nc.ssum - ps, 0);
          if (g > tb.g) tb = BestCand{g, k, prevk};
        }
        const uint16_t v = vals[p];
        const int64_t w = (int64_t)(L.aux[v] & 0xFFFFu);
        pn += w;
        ps += w * L.y[v];
        prevk = k;
      }
    }
    const BestCand b = team_best<TEAM>(tb, L.bg, L.bk, L.bp);
    if (t == 0) {
      carry_best(L.cr, b);
      L.cr.run_n += tot_n;
      L.cr.run_s += tot_s;
      if (n > 0) L.cr.last_key = keys[n - 1] + kbase;
    }
    team_sync<TEAM>();
  }
}

// One bucket of W key slots through an LDS histogram (bucket holds more
// elements than the sort capacity: heavy ties).  Classification:
// hist[slot * C + class]; regression: counts in words [0, W), 64-bit sums
// from word W on.  Whole-workgroup teams only.
template <int MAXC, int TASK, int IPT>
__device__ void eval_hist_bucket(const uint32_t* skey, const uint32_t* saux, const int64_t* sy, int64_t n_el,
                                 uint32_t kbase, int W, const NodeCtx& nc, TeamLds<MAXC, TASK, 256, IPT>& L,
                                 const LnCtx& lx) {
  const int t = threadIdx.x;
  const int C = nc.C;
  uint32_t* s_hist = L.u.hist;
  const int zero_words = (TASK == 0) ? W * C : 3 * W;
  for (int i = t; i < zero_words; i += 256) s_hist[i] = 0;
  __syncthreads();
  unsigned long long* hsum = (unsigned long long*)(s_hist + W);
  for (int64_t e = t; e < n_el; e += 256) {
    const uint32_t slot = skey[e] - kbase;
    const uint32_t a = saux[e];
    const uint32_t w = a & 0xFFFFu;
    if (TASK == 0) {
      atomicAdd(&s_hist[slot * C + (a >> 16)], w);
    } else {
      atomicAdd(&s_hist[slot], w);
      atomicAdd(&hsum[slot], (unsigned long long)((int64_t)w * sy[e]));
    }
  }
  __syncthreads();
  const int spt = (W + 255) / 256;
  const int s0 = t * spt, s1 = min(s0 + spt, W);
  uint32_t my_last = 0;  // last non-empty slot key + 1 in my range, 0 = none
  BestCand tb{0.0, kNone, kNone};
  if constexpr (TASK == 0) {
    for (int c = 0; c < C; ++c) L.cols()[c * 256 + t] = 0;
    for (int sl = s0; sl < s1; ++sl) {
      uint32_t any = 0;
      for (int c = 0; c < C; ++c) {
        const uint32_t h = s_hist[sl * C + c];
        L.cols()[c * 256 + t] += h;
        any |= h;
      }
      if (any) my_last = kbase + sl + 1;
    }
    L.last[t] = my_last;
    scan_class_columns<MAXC, TASK, 256, IPT>(L, C);
    uint32_t prev_last = 0;
    for (int i = 0; i < t; ++i) prev_last = max(prev_last, L.last[i]);
    if (s0 < s1) {
      WalkState w = walk_init<MAXC, TASK, 256, IPT>(L, nc, lx);
      uint32_t prevk = prev_last ? prev_last - 1 : L.cr.last_key;
      for (int sl = s0; sl < s1; ++sl) {
        uint32_t any = 0;
        for (int c = 0; c < C; ++c) any |= s_hist[sl * C + c];
        if (!any) continue;
        const uint32_t k = kbase + sl;
        if (w.nl > 0 && prevk < k) {
          const double g = walk_gain(w, nc, lx);
          if (g > tb.g) tb = BestCand{g, k, prevk};
        }
        for (int c = 0; c < C; ++c) {
          const uint32_t h = s_hist[sl * C + c];
          if (h) walk_add<MAXC, TASK, 256, IPT>(w, L, c, h, lx);
        }
        prevk = k;
      }
    }
    const BestCand b = team_best<256>(tb, L.bg, L.bk, L.bp);
    if (t == 0) {
      carry_best(L.cr, b);
      uint32_t last = 0;
      for (int i = 0; i < 256; ++i) last = max(last, L.last[i]);
      for (int c = 0; c < C; ++c) {
        L.cr.run[c] += L.ctot[c];
        L.cr.run_n += L.ctot[c];
      }
      if (last) L.cr.last_key = last - 1;
    }
    __syncthreads();
  } else {
    int64_t ln = 0, ls = 0;
    for (int sl = s0; sl < s1; ++sl) {
      const uint32_t hc = s_hist[sl];
      if (hc) {
        ln += hc;
        ls += (int64_t)hsum[sl];
        my_last = kbase + sl + 1;
      }
    }
    L.last[t] = my_last;
    int64_t tot_n, tot_s;
    int64_t pn = team_excl_scan_i64<256>(ln, L.w64, &tot_n);
    int64_t ps = team_excl_scan_i64<256>(ls, L.w64, &tot_s);
    uint32_t prev_last = 0;
    for (int i = 0; i < t; ++i) prev_last = max(prev_last, L.last[i]);
    pn += L.cr.run_n;
    ps += L.cr.run_s;
    uint32_t prevk = prev_last ? prev_last - 1 : L.cr.last_key;
    for (int sl = s0; sl < s1; ++sl) {
      const uint32_t hc = s_hist[sl];
      if (!hc) continue;
      const uint32_t k = kbase + sl;
      if (pn > 0 && prevk < k) {
        const double g = variance_gain(pn, ps, nc.n - pn, nc.ssum - ps, 0);
        if (g > tb.g) tb = BestCand{g, k, prevk};
      }
      pn += hc;
      ps += (int64_t)hsum[sl];
      prevk = k;
    }
    const BestCand b = team_best<256>(tb, L.bg, L.bk, L.bp);
    if (t == 0) {
      carry_best(L.cr, b);
      uint32_t last = 0;
      for (int i = 0; i < 256; ++i) last = max(last, L.last[i]);
      L.cr.run_n += tot_n;
      L.cr.run_s += tot_s;
      if (last) L.cr.last_key = last - 1;
    }
    __syncthreads();
  }
}

// Sort a chunk (keys relative to kbase, span < 2^bits) held in LDS buffer 0
// and evaluate it.
template <int MAXC, int TASK, int TEAM, int IPT, class LX = LnCtx>
__device__ void sort_and_eval(int n, int bits, uint32_t kbase, const NodeCtx& nc,
                              TeamLds<MAXC, TASK, TEAM, IPT>& L, const LX& lx) {
  constexpr int kSpan = TeamLds<MAXC, TASK, TEAM, IPT>::SPAN;
  if (bits > 4 && (1 << bits) <= kSpan) {
    lds_count_sort<IPT, TEAM>(L.u.srt.k[0], L.u.srt.v[0], L.u.srt.k[1], L.u.srt.v[1], n, 1 << bits,
                              reinterpret_cast<uint32_t*>(L.u.srt.cnt), L.w);
    eval_sorted_chunk<MAXC, TASK, TEAM, IPT>(L.u.srt.k[1], L.u.srt.v[1], n, kbase, nc, L, lx);
    return;
  }
  int cur = 0;
  for (int sh = 0; sh < bits; sh += 4) {
    lds_sort_pass<IPT, TEAM>(L.u.srt.k[cur], L.u.srt.v[cur], L.u.srt.k[cur ^ 1], L.u.srt.v[cur ^ 1], n, sh,
                             L.u.srt.cnt, L.w);
    cur ^= 1;
  }
  eval_sorted_chunk<MAXC, TASK, TEAM, IPT>(L.u.srt.k[cur], L.u.srt.v[cur], n, kbase, nc, L, lx);
}

__device__ __forceinline__ int bit_length(uint32_t v) { return v ? 32 - __clz((int)v) : 0; }

__device__ __forceinline__ void load_tables(double* s_inv, double* s_logc) {
  for (int i = threadIdx.x; i < 128; i += blockDim.x) {
    s_inv[i] = g_ln_table.inv[i];
    s_logc[i] = g_ln_table.logc[i];
  }
}

// Node statistics of one item, computed by the whole workgroup.
template <int MAXC, int TASK>
__device__ __forceinline__ bool node_context(const DataArgs& d, const LevelArgs& lv, uint32_t i, NodeCtx& nc,
                                             TeamLds<MAXC, TASK, kBlock, kIpt>& L, const LnCtx& lx) {
  const int t = threadIdx.x;
  nc.C = d.C;
  nc.n = lv.count[i];
  nc.ssum = 0;
  nc.P = 0;
  nc.inv = 0.0;
  if constexpr (TASK == 0) {
    const uint32_t my = t < d.C ? lv.cls[(int64_t)i * d.C + t] : 0u;
    if (t < d.C) L.ncls[t] = my;
    const uint32_t mx = team_reduce_max<kBlock>(my, L.w);
    const int64_t tn = t < d.C ? lx.t(my) : 0;
    int64_t tsum = 0;  // sum of T(n_c) over the classes (lanes < C)
    (void)team_excl_scan_i64<kBlock>(tn, L.w64, &tsum);
    nc.P = lx.t((uint64_t)nc.n) - tsum;
    nc.inv = 1.0 / ((double)nc.n * kLn2);
    return (int64_t)mx == nc.n;  // pure node
  } else {
    nc.ssum = lv.sum[i];
    return false;
  }
}

// Evaluate one RF item on a workgroup; returns through L.cr.  An item above
// the LDS capacity is bucketed through the workgroup's scratch slab.
template <int MAXC, int TASK>
__device__ void rf_item(const DataArgs& d, const LevelArgs& lv, const ItemArgs& it, int f, uint32_t i, const NodeCtx& nc,
                        TeamLds<MAXC, TASK, kBlock, kIpt>& L, const LnCtx& lx, uint32_t* s_boff, int slab) {
  constexpr int IPT = kIpt;
  constexpr int CAP = kCap;
  const int t = threadIdx.x;
  const int m = lv.m[i];
  const int64_t st = lv.start[i];
  const uint32_t* Kf = d.K + (int64_t)f * d.N;
  if (t == 0) {
    for (int c = 0; c < MAXC; ++c) L.cr.run[c] = 0;
    L.cr.run_n = 0;
    L.cr.run_s = 0;
    L.cr.last_key = 0;
    L.cr.best_g = 0.0;
    L.cr.best_key = kNone;
    L.cr.best_prev = kNone;
  }
  if (m <= CAP) {
    // Gather: independent loads first (rows, payloads), then the keys.
    uint32_t kmin = kNone, kmax = 0;
    uint32_t rows[IPT];
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
      const int e = t + q * kBlock;
      if (e < m) {
        rows[q] = lv.row[st + e];
        L.aux[e] = lv.aux[st + e];
        if (TASK == 1) L.y[e] = lv.ey[st + e];
      }
    }
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
      const int e = t + q * kBlock;
      if (e < m) {
        const uint32_t key = Kf[rows[q]];
        L.u.srt.k[0][e] = key;
        L.u.srt.v[0][e] = (uint16_t)e;
        kmin = min(kmin, key);
        kmax = max(kmax, key);
      }
    }
    kmin = team_reduce_min<kBlock>(kmin, L.w);
    kmax = team_reduce_max<kBlock>(kmax, L.w);
    for (int e = t; e < m; e += kBlock) L.u.srt.k[0][e] -= kmin;
    __syncthreads();
    sort_and_eval<MAXC, TASK, kBlock, IPT>(m, bit_length(kmax - kmin), kmin, nc, L, lx);
    return;
  }
  // Big node: bucket by dense key into this block's scratch slab, then
  // pack consecutive buckets into LDS-sized chunks.
  const uint32_t S = d.S[f];
  const int words = (TASK == 0) ? d.C : 3;
  int wbits = 0;
  while ((1 << (wbits + 1)) * words <= kHistWords) ++wbits;
  while (((S + (1u << wbits) - 1) >> wbits) > (uint32_t)kMaxBuckets) ++wbits;
  const int W = 1 << wbits;
  const int NB = (int)((S + (uint32_t)W - 1) >> wbits);
  uint32_t* skey = it.scr_key + (int64_t)slab * it.scr_stride;
  uint32_t* saux = it.scr_aux + (int64_t)slab * it.scr_stride;
  int64_t* sy = TASK == 1 ? it.scr_y + (int64_t)slab * it.scr_stride : nullptr;
  for (int b = t; b <= NB; b += 256) s_boff[b] = 0;
  __syncthreads();
  constexpr int U = 8;
  for (int e0 = 0; e0 < m; e0 += 256 * U) {
    uint32_t rows[U];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int e = e0 + t + q * 256;
      rows[q] = e < m ? lv.row[st + e] : 0u;
    }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int e = e0 + t + q * 256;
      if (e < m) atomicAdd(&s_boff[Kf[rows[q]] >> wbits], 1u);
    }
  }
  __syncthreads();
  {
    const int per = (NB + 255) / 256;
    const int b0 = t * per, b1 = min(b0 + per, NB);
    uint32_t loc = 0;
    for (int b = b0; b < b1; ++b) loc += s_boff[b];
    uint32_t base = team_excl_scan<256>(loc, L.w, nullptr);
    for (int b = b0; b < b1; ++b) {
      const uint32_t c = s_boff[b];
      s_boff[b] = base;
      base += c;
    }
    if (t == 0) s_boff[NB] = (uint32_t)m;
    __syncthreads();
    for (int b = t; b < NB; b += 256) L.u.bpos[b] = s_boff[b];
    __syncthreads();
  }
  for (int e0 = 0; e0 < m; e0 += 256 * U) {
    uint32_t rows[U], auxv[U], keys[U];
    int64_t yv[U];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int e = e0 + t + q * 256;
      if (e < m) {
        rows[q] = lv.row[st + e];
        auxv[q] = lv.aux[st + e];
        if (TASK == 1) yv[q] = lv.ey[st + e];
      }
    }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int e = e0 + t + q * 256;
      if (e < m) keys[q] = Kf[rows[q]];
    }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int e = e0 + t + q * 256;
      if (e < m) {
        const uint32_t pos = atomicAdd(&L.u.bpos[keys[q] >> wbits], 1u);
        skey[pos] = keys[q];
        saux[pos] = auxv[q];
        if (TASK == 1) sy[pos] = yv[q];
      }
    }
  }
  __syncthreads();
  int b = 0;
  while (b < NB) {
    const uint32_t cb = s_boff[b + 1] - s_boff[b];
    if (cb == 0) {
      ++b;
      continue;
    }
    if (cb > (uint32_t)CAP) {
      eval_hist_bucket<MAXC, TASK, IPT>(skey + s_boff[b], saux + s_boff[b], TASK == 1 ? sy + s_boff[b] : nullptr,
                                        cb, (uint32_t)b << wbits, W, nc, L, lx);
      ++b;
      continue;
    }
    int be = b;
    uint32_t tot = 0;
    while (be < NB) {
      const uint32_t c = s_boff[be + 1] - s_boff[be];
      if (c > (uint32_t)CAP || tot + c > (uint32_t)CAP) break;
      tot += c;
      ++be;
    }
    const uint32_t e0 = s_boff[b];
    const uint32_t kbase = (uint32_t)b << wbits;
    for (int e = t; e < (int)tot; e += 256) {
      L.u.srt.k[0][e] = skey[e0 + e] - kbase;
      L.u.srt.v[0][e] = (uint16_t)e;
      L.aux[e] = saux[e0 + e];
      if (TASK == 1) L.y[e] = sy[e0 + e];
    }
    __syncthreads();
    sort_and_eval<MAXC, TASK, 256, IPT>((int)tot, bit_length((uint32_t)(be - b) * (uint32_t)W - 1u), kbase, nc,
                                        L, lx);
    b = be;
  }
}

template <int MAXC, int TASK>
__device__ __forceinline__ void rf_write_result(const DataArgs& d, const ItemArgs& it, int64_t ridx, int f,
                                                const Carry<MAXC, TASK>& cr) {
  float score = 0.0f, thr = 0.0f;
  if (cr.best_key != kNone) {
    const float* sv = d.SV + d.SVoff[f];
    score = (float)(TASK == 0 ? cr.best_g : ldexp_d(cr.best_g, -2 * d.shift));
    thr = midpoint(sv[cr.best_prev], sv[cr.best_key]);
  }
  it.res_score[ridx] = score;
  it.res_thr[ridx] = thr;
  it.res_feat[ridx] = f;
}

// ------------------------------------------------- RF split search ------
// One workgroup per (node, feature draw) item, grid-stride over items: the
// plain driver's nodes of any size, and the few nodes above cut_block of the
// level graphs.  Nodes of up to 2048 entries are sorted in LDS, larger ones
// are bucketed by dense key into a scratch slab first.  Every boundary between
// distinct values is scored.  Its speed hangs on what the compiler is told:
// 32-bit block numbers (64-bit ones cost 4 to 8 registers) and 16-byte aligned
// LDS (the digit counters are read 16 bytes at a time); 1M x 128, 12 trees in
// the plain driver 2.07 s, without the first 2.21, without the second 2.10.
template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock) k_search_rf(DataArgs d, LevelArgs lv, ItemArgs it) {
  resolve_level(lv, d.C);
  resolve_items(it);
  const int64_t n_items = it.n_groups * it.per_group;
  if ((int64_t)blockIdx.x >= n_items) return;
  __shared__ double s_inv[128], s_logc[128];
  __shared__ alignas(16) TeamLds<MAXC, TASK, kBlock, kIpt> L;
  __shared__ uint32_t s_boff[kMaxBuckets + 1];
  load_tables(s_inv, s_logc);
  __syncthreads();
  const LnCtx lx{s_inv, s_logc, d.T, d.Tmax, d.igF};
  const int t = threadIdx.x;
  unsigned long long my_bytes = 0;
  for (int64_t item = (int)blockIdx.x; item < n_items; item += (int64_t)gridDim.x) {
    const int64_t grp = it.node_major ? item % it.n_groups : item / it.per_group;
    const int j = it.j0 + (int)(it.node_major ? item / it.n_groups : item % it.per_group);
    const uint32_t o = it.list ? it.list[grp] : (uint32_t)grp;
    const uint32_t i = lv.open_idx[o];
    const int f = (int)(rand_u32(d.seed, kStreamFeat, (uint32_t)lv.tree_global[lv.tree[i]], lv.id[i], (uint64_t)j) %
                        (uint32_t)d.F);
    const int64_t ridx = (int64_t)o * it.D + j;
    NodeCtx nc;
    const bool pure = node_context<MAXC, TASK>(d, lv, i, nc, L, lx);
    if (pure) {
      // Every boundary of a pure node has gain exactly 0: no positive split.
      if (t == 0) {
        it.res_score[ridx] = 0.0f;
        it.res_thr[ridx] = 0.0f;
        it.res_feat[ridx] = f;
      }
      __syncthreads();
      continue;
    }
    if (t == 0) my_bytes += (unsigned long long)lv.m[i] * (TASK == 0 ? 12ull : 20ull);
    rf_item<MAXC, TASK>(d, lv, it, f, i, nc, L, lx, s_boff, (int)blockIdx.x);
    __syncthreads();
    if (t == 0) rf_write_result<MAXC, TASK>(d, it, ridx, f, L.cr);
    __syncthreads();
  }
  if (t == 0 && my_bytes && it.bytes) add_bytes(it.bytes, my_bytes);
}

// ------------------------------------- chunk-parallel big-node search ---
// Items (node, feature draw) above the workgroup's LDS capacity.  The keys of
// an item (dense ranks of the drawn feature) are split into nb buckets of
// consecutive keys, bucket = key / width, of about 64 entries each.  The gain
// is a convex function of what lies left of a boundary, so a bucket's class
// counts (regression: weights and target sums) bound the gain of every
// boundary inside it; only buckets whose bound reaches the best bucket edge
// of the node's draws are sorted and walked:
//   1. k_v2_hist     per (item, tile): class counts (weight, target sums) of
//                    every bucket; the gathered keys are kept in entry order
//   2. k_v2_bound    per item: totals before each bucket, the gain at each
//                    bucket's lower edge, the bound of the bucket; the best
//                    edge over a node's draws
//   3. k_v2_select   per item: the buckets that can still hold the node's
//                    best split, with a scratch slot each
//   4. k_v2_collect  per (item, tile): entries of selected buckets into their
//                    slots, last key before each selected bucket
//   5. k_v2_eval     per selected bucket, one wave each: LDS sort + scored
//                    walk from the totals before it
//   6. k_v2_spill    per selected bucket above a wave's capacity (clustered
//                    keys, capped bucket counts): fine sub-buckets walked in
//                    order by one workgroup
//   7. k_v2_reduce   per item: best bucket -> (score, threshold)
// A draw whose best candidate is pruned reports a lower score (or none), and
// never one of the node's best score: every bucket that could reach it, ties
// in fp32 included, is walked.  Entry order inside a bucket does not matter:
// the walk sorts by key and scores only boundaries between distinct keys from
// integer prefix sums.
// Entries per tile: a tile of a larger node adds its whole bucket table to the
// item's, so its size is what the merging of tables costs against the number
// of workgroups (big_pipeline: at least kV2TileRounds a slot of the chip).
// 8 trees of 4M rows, 21 draws, a level of few nodes: 1.62 ms at 16,384
// entries, 1.35 at 65,536.
constexpr int kV2Tile = 16384;
constexpr int kV2TileMax = 65536;  // entry numbers of a tile in 16 bits (k_v2_collect)
constexpr int kV2TileRounds = 6;
constexpr int kXcds = 8;          // XCDs of an MI355X, one L2 each
constexpr int kV2MaxB = 4096;    // buckets per item
constexpr int kV2Ipt = kIpt;     // entries per lane of the bucket evaluator
constexpr int kV2WaveCap = kWave * kV2Ipt;  // bucket capacity of a wave (512)
// LDS words of a tile's bucket table: three workgroups per CU.  A bucket
// takes a word per class (regression: a weight and two 64-bit sums).
constexpr int kV2HistWords = 12288;
constexpr int kV2RegWords = 5;

struct V2Item {
  int32_t f;
  int32_t m;
  int64_t start;  // first entry of the node
  int64_t soff;   // first slot of the item's gathered keys
  int32_t boff;   // first bucket slot of the item
  int32_t nb;     // buckets
  uint32_t width;  // bucket = key / width (v2_bucket)
  uint32_t magic;  // floor(2^32 / width)
  uint32_t node;  // level node index
  int32_t grp;    // node of the phase (its best bucket edge: nbest[grp])
  int64_t ridx;   // result slot (open position * D + draw)
  // node context (as node_context computes it)
  int64_t n_w;    // sum of weights
  int64_t P;      // classification: T(n) - sum_c T(n_c)
  int64_t ssum;   // regression: fixed-point target sum
  double inv;     // 1 / (n ln 2)
};

// key / width from the high word of key * floor(2^32 / width), which is the
// quotient or one below it, and one exact correction.
__device__ __forceinline__ uint32_t v2_bucket(uint32_t key, const V2Item& it) {
  uint32_t q = __umulhi(key, it.magic);
  if ((uint64_t)(q + 1u) * it.width <= key) ++q;
  return q;
}

// Fixed-point mean of a regression node: its targets are centred on it, which
// makes the bounds tight (the gain does not depend on the centre).
__device__ __forceinline__ int64_t v2_centre(const V2Item& it) {
  return d2ll_rn((double)it.ssum / (double)it.n_w);
}

struct V2Tile {
  uint32_t item;
  uint32_t e0;
};

struct V2Task {
  uint32_t item;
  uint32_t b;
};

struct V2Args {
  const V2Item* items;
  int tile;         // entries per tile
  int64_t n_items;
  const V2Tile* tiles;
  // per bucket: k_v2_hist's counts, overwritten by k_v2_bound with the totals
  // before the bucket
  uint32_t* bcls;   // classification [boff * C + c * nb + b]
  uint32_t* bn;     // weights
  int64_t* bpos;    // regression: sums of the targets above / below the node's
  int64_t* bneg;    // centre; then bpos: target sum before the bucket
  float* bub;       // bound of the scores inside the bucket (-1: empty)
  uint32_t* nbest;  // per node of the phase: best edge score (float bits)
  float best_cap;   // edges above this count as this (retry phase)
  double max_dev;   // regression: largest |fixed target|
  uint32_t* bslot;  // scratch slot of a selected bucket (kNone: not selected)
  uint32_t* bnext;  // selected bucket whose lower neighbour this is (kNone: none)
  uint32_t* bcur;   // entries collected
  uint32_t* carry_last;  // last key before the bucket
  uint32_t* isel;   // per item: selected buckets
  double* res_g;
  uint32_t* res_key;
  uint32_t* res_prev;
  uint32_t* gkey;   // keys in entry order, item-major, or (gathered) the phase's keys by draw
  // scratch slots of the selected buckets
  uint32_t* skey;
  uint32_t* saux;
  int64_t* sy;
  uint32_t* skey2;  // k_v2_spill: fine sub-bucket order (skey2 aliases gkey)
  uint32_t* saux2;
  int64_t* sy2;
  // task lists
  V2Task* tasks;
  V2Task* spill;
  unsigned int* counters;  // [0] tasks, [1] spill, [2] scratch slots
};

// Tiles are issued feature-major and split in eighths across the XCDs (see
// big_pipeline).  The bucket table lives in dynamic LDS: [c * nb + b] class
// counts, or nb sums above, nb sums below, nb weights.
template <int TASK, bool GATHERED>  // GATHERED: gkey holds the keys already (k_gather_draws)
__global__ void __launch_bounds__(kBlock) k_v2_hist(DataArgs d, LevelArgs lv, V2Args a) {
  extern __shared__ uint64_t s_tab[];
  const V2Tile tl = a.tiles[blockIdx.x];
  const V2Item it = a.items[tl.item];
  const int t = threadIdx.x;
  const int nb = it.nb;
  uint32_t* s_cls = reinterpret_cast<uint32_t*>(s_tab);
  unsigned long long* s_pos = reinterpret_cast<unsigned long long*>(s_tab);
  unsigned long long* s_neg = s_pos + nb;
  uint32_t* s_n = reinterpret_cast<uint32_t*>(s_neg + nb);
  const int words = TASK == 0 ? nb * d.C : nb * kV2RegWords;
  for (int b = t; b < words; b += kBlock) s_cls[b] = 0;
  const int64_t mu = TASK == 1 ? v2_centre(it) : 0;
  __syncthreads();
  const uint32_t* Kf = d.K + (int64_t)it.f * d.N;
  const int n = min(a.tile, it.m - (int)tl.e0);
  const int64_t e0 = it.start + tl.e0;
  uint32_t* gkey = a.gkey + it.soff + tl.e0;
  // Two stages ahead of the counting: the next step's payloads (and rows) are
  // in flight, and its keys once their rows are there.  The table leaves a CU
  // three workgroups, too few to cover a step's loads from outside the wave.
  constexpr int U = 8;
  struct Step {
    uint32_t rows[GATHERED ? 1 : U], aux[U], keys[U];
    int64_t y[TASK == 1 ? U : 1];
  };
  auto fetch = [&](int base, Step& st) {
    if (base >= n) return;  // workgroup-uniform
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int e = min(base + t + q * kBlock, n - 1);
      if (GATHERED) st.keys[q] = gkey[e];
      else st.rows[q] = lv.row[e0 + e];
      st.aux[q] = lv.aux[e0 + e];
      if (TASK == 1) st.y[q] = lv.ey[e0 + e];
    }
  };
  auto gather = [&](int base, Step& st) {
    if (GATHERED || base >= n) return;
#pragma unroll
    for (int q = 0; q < U; ++q) st.keys[q] = Kf[st.rows[GATHERED ? 0 : q]];
  };
  auto count = [&](int base, const Step& st) {
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int e = base + t + q * kBlock;
      if (e < n) {
        if (!GATHERED) gkey[e] = st.keys[q];
        const uint32_t b = v2_bucket(st.keys[q], it);
        const uint32_t w = st.aux[q] & 0xFFFFu;
        if (TASK == 0) {
          atomicAdd(&s_cls[(st.aux[q] >> 16) * (uint32_t)nb + b], w);
        } else {
          const int64_t dy = st.y[q] - mu;
          atomicAdd(&s_n[b], w);
          atomicAdd(dy < 0 ? &s_neg[b] : &s_pos[b], (unsigned long long)((int64_t)w * dy));
        }
      }
    }
  };
  constexpr int kStep = kBlock * U;
  Step s0, s1;
  fetch(0, s0);
  gather(0, s0);
  fetch(kStep, s1);
  for (int base = 0; base < n; base += 2 * kStep) {
    gather(base + kStep, s1);
    count(base, s0);
    fetch(base + 2 * kStep, s0);
    if (base + kStep >= n) break;
    gather(base + 2 * kStep, s0);
    count(base + kStep, s1);
    fetch(base + 3 * kStep, s1);
  }
  __syncthreads();
  const bool only = it.m <= a.tile;  // the item's only tile: plain stores
  if (TASK == 0) {
    uint32_t* g = a.bcls + (int64_t)it.boff * d.C;
    for (int i = t; i < words; i += kBlock) {
      const uint32_t v = s_cls[i];
      if (only) g[i] = v;
      else if (v) atomicAdd(&g[i], v);
    }
  } else {
    for (int b = t; b < nb; b += kBlock) {
      const int64_t gb = (int64_t)it.boff + b;
      const uint32_t w = s_n[b];
      if (only) {
        a.bn[gb] = w;
        a.bpos[gb] = (int64_t)s_pos[b];
        a.bneg[gb] = (int64_t)s_neg[b];
      } else if (w) {
        atomicAdd(&a.bn[gb], w);
        atomicAdd(reinterpret_cast<unsigned long long*>(&a.bpos[gb]), s_pos[b]);
        atomicAdd(reinterpret_cast<unsigned long long*>(&a.bneg[gb]), s_neg[b]);
      }
    }
  }
}

// Largest distance (in units of x) between x ln x and its chord over an
// interval of s that starts at a: at most s / e (a = 0), and s^2 / 8 times the
// largest curvature 1 / a.
__device__ __forceinline__ double chord_gap(double a, double s) {
  const double e = s * 0.36787944117144233;
  return a > 0.0 ? fmin(e, s * s / (8.0 * a)) : e;
}

// Units of the fixed-point entropy sums that cover the difference between the
// fixed-point terms and the double arithmetic of the bounds: each term is at
// most 2^62 / (2C + 2) units and off by 7e-16 of that (its series) and half a
// unit, a few tens of terms and roundings of 1.1e-16 each.
constexpr double kBoundUnits = 131072.0;

// Value of the lane below (lane 0: `first`), and of the last lane.
__device__ __forceinline__ double lane_below(double v, double first) {
  const double y = __shfl_up(v, 1, kWave);
  return (threadIdx.x & (kWave - 1)) == 0 ? first : y;
}
__device__ __forceinline__ double wave_last_f64(double v) {
  return __builtin_bit_cast(double, wave_last_i64(__builtin_bit_cast(int64_t, v)));
}

// variance_gain takes the difference of two rounded means: it is off by up to
// 2^-50 of their size, so a computed gain g and the real one f, both sums over
// the node, satisfy |sqrt g - sqrt f| <= e = sqrt(N) / 2 * 2^-50 max|y|, hence
// g <= f (1 + t) + e^2 (1 + 1 / t), and the same with f and g exchanged.  The
// bounds take t = 1e-6; this is the second term.
__device__ __forceinline__ double reg_gain_error(double N, double y_max) {
  const double e = y_max * 8.8817841970012523e-16;
  return 0.25 * N * e * e * 1.1e6;
}

// fp32 score of a variance gain that must not pass for none: a positive gain's
// score may round to 0, and its threshold still decides among draws of score 0.
__device__ __forceinline__ float reg_score_bound(double gain, int shift) {
  return gain > 0.0 ? fmaxf((float)ldexp_d(gain, -2 * shift), FLT_TRUE_MIN) : 0.0f;
}

// Upper bound of the variance criterion over left weights [n0, n1] and left
// target sums [lo, hi], for a node of weight N, target sum S and largest
// deviation M: f(n, s) = s^2 / n + (S - s)^2 / (N - n) is convex, so its
// maximum over the box is at a corner; a side that may be empty has a mean of
// at most M, so its term is at most |sum| M.
__device__ __forceinline__ double reg_box_bound(double n0, double n1, double lo, double hi, double N, double S,
                                                double M) {
  const double a = lo * lo, b = hi * hi, c = (S - lo) * (S - lo), e = (S - hi) * (S - hi);
  if (n0 > 0.0 && n1 < N) {
    const double l0 = 1.0 / n0, l1 = 1.0 / n1, r0 = 1.0 / (N - n0), r1 = 1.0 / (N - n1);
    const double f0 = fmax(a * l0 + c * r0, b * l0 + e * r0);
    const double f1 = fmax(a * l1 + c * r1, b * l1 + e * r1);
    return fmax(f0, f1) - S * S / N;
  }
  const double left = n0 > 0.0 ? fmax(a, b) / n0 : fmax(fabs(lo), fabs(hi)) * M;
  const double right = n1 < N ? fmax(c, e) / (N - n1) : fmax(fabs(S - lo), fabs(S - hi)) * M;
  return left + right;
}

// One wave per item, 64 buckets at a time.  Per bucket: totals before it (in
// place of the counts), the gain at its lower edge, and a bound of every gain
// inside it.  Classification: with phi_c(x) = T(x) + T(n_c - x) and
// psi(x) = T(x) + T(n - x), both convex, the gain sum is
// P + sum_c phi_c(l_c) - psi(sum_c l_c).  Between the bucket's ends each phi_c
// tilted by the chord slope of psi stays below the larger of its ends, and psi
// less its own chord stays above -chord_gap, so
//   gain <= edge + sum_c max(0, phi_c(end) - phi_c(start) - slope s_c) + gap.
template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock) k_v2_bound(DataArgs d, LevelArgs lv, V2Args a) {
  __shared__ double s_inv[128], s_logc[128];
  load_tables(s_inv, s_logc);
  __syncthreads();
  const int64_t k = (int64_t)blockIdx.x * kWaves + threadIdx.x / kWave;
  if (k >= a.n_items) return;  // wave-uniform; no workgroup barrier follows
  const V2Item it = a.items[k];
  const int lane = threadIdx.x & (kWave - 1);
  const int nb = it.nb;
  float best = 0.0f;
  if constexpr (TASK == 0) {
    // x ln x in double from the reduction table in LDS: the counts of a big
    // node spread over an 8 MB table of terms, and 4 reads per class and
    // bucket of it took 0.45 ms per phase of a 32-tree 1M-row level.
    auto xl = [&](uint32_t x) { return xlnx(x, s_inv, s_logc); };
    const int C = d.C;
    uint32_t* cls = a.bcls + (int64_t)it.boff * C;
    uint32_t run[MAXC], ncl[MAXC];
    double phi_row[MAXC];  // phi_c before the row
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
      run[c] = 0;
      ncl[c] = c < C ? lv.cls[(int64_t)it.node * C + c] : 0u;
      phi_row[c] = c < C ? xl(ncl[c]) : 0.0;
    }
    const uint32_t n_w = (uint32_t)it.n_w;
    const double P = ldexp_d((double)it.P, -d.igF);
    const double margin = ldexp_d(kBoundUnits, -d.igF);
    uint32_t run_n = 0;
    double psi_row = xl(n_w);  // psi before the row
    for (int b0 = 0; b0 < nb; b0 += kWave) {
      const int b = b0 + lane;
      const bool ok = b < nb;
      uint32_t v[MAXC], sw = 0;
#pragma unroll
      for (int c = 0; c < MAXC; ++c) {
        v[c] = c < C && ok ? cls[c * nb + b] : 0u;
        sw += v[c];
      }
      // values at the bucket's end; its start is the end of the lane below
      const uint32_t lb = run_n + wave_incl_scan(sw), la = lb - sw;
      run_n = wave_last(lb);
      const double psb = xl(lb) + xl(n_w - lb);
      const double psa = lane_below(psb, psi_row);
      psi_row = wave_last_f64(psb);
      const double slope = sw ? (psb - psa) / (double)sw : 0.0;
      double phi = 0.0, slack = 0.0;
#pragma unroll
      for (int c = 0; c < MAXC; ++c) {
        if (c < C) {
          const uint32_t l = run[c] + wave_incl_scan(v[c]);
          run[c] = wave_last(l);
          const double pb = xl(l) + xl(ncl[c] - l);
          const double pa = lane_below(pb, phi_row[c]);
          phi_row[c] = wave_last_f64(pb);
          phi += pa;
          slack += fmax(0.0, (pb - pa) - slope * (double)v[c]);
          if (ok) cls[c * nb + b] = l - v[c];
        }
      }
      slack += chord_gap((double)la, (double)sw) + chord_gap((double)(n_w - lb), (double)sw);
      const double edge = P + phi - psa;
      float ub = -1.0f;
      if (sw) {
        // nats to bits per unit weight, as ig_from_fixed
        ub = (float)((edge + slack * (1.0 + 1e-9) + margin) * it.inv * (1.0 + 1e-12));
        if (la > 0) best = fmaxf(best, (float)((edge - margin) * it.inv * (1.0 - 1e-12)));
        if (it.width == 1) {  // one key: no boundary but the lower edge
          const LnCtx lx{s_inv, s_logc, d.T, d.Tmax, d.igF};
          int64_t e = it.P - lx.t(la) - lx.t(n_w - la);
#pragma unroll
          for (int c = 0; c < MAXC; ++c)
            if (c < C) {
              const uint32_t l = cls[c * nb + b];  // stored above by this lane
              e += lx.t(l) + lx.t(ncl[c] - l);
            }
          const double g = la > 0 ? ig_from_fixed(e, d.igF, it.inv) : 0.0;
          a.res_g[(int64_t)it.boff + b] = g;
          ub = fmaxf((float)g, 0.0f);
        }
      }
      if (ok) {
        a.bn[(int64_t)it.boff + b] = la;
        a.bub[(int64_t)it.boff + b] = it.P > 0 ? ub : -1.0f;  // P = 0: pure node, every gain is 0
      }
    }
  } else {
    const int64_t mu = v2_centre(it);
    const double M = a.max_dev + fabs((double)mu), E = reg_gain_error((double)it.n_w, a.max_dev);
    const double N = (double)it.n_w, S = (double)(it.ssum - mu * it.n_w);
    uint32_t run_n = 0;
    int64_t run_s = 0;  // centred sum before the row
    for (int b0 = 0; b0 < nb; b0 += kWave) {
      const int b = b0 + lane;
      const bool ok = b < nb;
      const int64_t gb = (int64_t)it.boff + b;
      const uint32_t w = ok ? a.bn[gb] : 0u;
      const int64_t sp = ok ? a.bpos[gb] : 0, sn = ok ? a.bneg[gb] : 0;
      const uint32_t inc = wave_incl_scan(w);
      const uint32_t la = run_n + inc - w;
      run_n += wave_last(inc);
      const int64_t is = wave_incl_scan_i64(sp + sn);
      const int64_t sa = run_s + is - (sp + sn);
      run_s += wave_last_i64(is);
      const int64_t su = sa + mu * (int64_t)la;  // uncentred target sum before the bucket
      float ub = -1.0f;
      if (w) {
        const double u = reg_box_bound((double)la, (double)(la + w), (double)(sa + sn), (double)(sa + sp), N, S, M);
        ub = d.no_bound ? __builtin_inff() : reg_score_bound(u * (1.0 + 2e-6) + E, d.shift);
        if (la > 0) {
          const double g = variance_gain(la, su, it.n_w - la, it.ssum - su, 0);
          best = fmaxf(best, (float)ldexp_d(g, -2 * d.shift));
          if (it.width == 1) {
            a.res_g[gb] = g;
            ub = reg_score_bound(g, d.shift);
          }
        } else if (it.width == 1) {
          ub = 0.0f;
        }
      }
      if (ok) {
        a.bn[gb] = la;
        a.bpos[gb] = su;
        a.bub[gb] = ub;
      }
    }
  }
  // scores are at least 0: their bits order as unsigned words
  const uint32_t bits = wave_max_u32(__float_as_uint(best));
  if (lane == 0 && bits) atomicMax(&a.nbest[it.grp], bits);
}

// One wave per item: selects the buckets whose bound reaches the node's best
// edge, from the last bucket down (a bucket that precedes a selected one keeps
// its largest key).  A selected bucket of one key (width 1) is its lower edge:
// its result is complete here and its entries are not collected (kDone).
constexpr uint32_t kDone = kNone - 1u;
// The slots and list places of a workgroup's items are taken by two atomics:
// with one per item and row, the waves queued on those words (1.1 ms of a
// phase of 172,000 items; 4M x 64 regression).
constexpr int kSelectWaves = 16;
template <int TASK>
__global__ void __launch_bounds__(kSelectWaves * kWave) k_v2_select(DataArgs d, V2Args a) {
  __shared__ unsigned int s_cnt[kSelectWaves][3];
  __shared__ unsigned int s_base[3];
  const int wv = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t k = (int64_t)blockIdx.x * kSelectWaves + wv;
  const bool live = k < a.n_items;
  V2Item it{};
  if (live) it = a.items[k];
  const int nb = live ? it.nb : 0;
  const int64_t g0 = it.boff;
  const float thr = live ? fminf(__uint_as_float(a.nbest[it.grp]), a.best_cap) : 0.0f;
  auto weight = [&](int b) {
    return (b + 1 < nb ? a.bn[g0 + b + 1] : (uint32_t)it.n_w) - a.bn[g0 + b];
  };
  unsigned int n_small = 0, n_big = 0, n_slot = 0;
  for (int b0 = 0; b0 < nb; b0 += kWave) {
    const int b = b0 + lane;
    const float u = b < nb ? a.bub[g0 + b] : -1.0f;
    const bool sel = u > 0.0f && u >= thr;
    if (!__ballot(sel)) continue;
    const uint32_t w = sel ? weight(b) : 0u;
    n_small += (unsigned int)__popcll(__ballot(sel && w <= (uint32_t)kV2WaveCap));
    n_big += (unsigned int)__popcll(__ballot(w > (uint32_t)kV2WaveCap));
    n_slot += wave_last(wave_incl_scan(w));
  }
  const unsigned int n_sel = n_small + n_big;
  if (live && lane == 0) a.isel[k] = n_sel;
  const bool one_key = it.width == 1;
  if (lane == 0) {
    s_cnt[wv][0] = one_key ? 0u : n_small;
    s_cnt[wv][1] = one_key ? 0u : n_big;
    s_cnt[wv][2] = one_key ? 0u : n_slot;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    unsigned int sum = 0;
    for (int i = 0; i < kSelectWaves; ++i) {
      const unsigned int c = s_cnt[i][threadIdx.x];
      s_cnt[i][threadIdx.x] = sum;
      sum += c;
    }
    s_base[threadIdx.x] = sum ? atomicAdd(&a.counters[threadIdx.x], sum) : 0u;
  }
  __syncthreads();
  if (!n_sel) return;
  uint32_t at_small = s_base[0] + s_cnt[wv][0], at_big = s_base[1] + s_cnt[wv][1], at_slot = s_base[2] + s_cnt[wv][2];
  uint32_t next = kNone;  // the selected bucket next above the row, if it is the next non-empty one
  for (int b0 = (nb - 1) / kWave * kWave; b0 >= 0; b0 -= kWave) {
    const int b = b0 + lane;
    const bool ok = b < nb;
    const int64_t gb = g0 + b;
    const float u = ok ? a.bub[gb] : -1.0f;
    const bool full = u >= 0.0f;
    const bool sel = u > 0.0f && u >= thr;
    if (one_key) {
      if (sel) {
        const uint32_t lo = a.bn[gb];
        int p = b - 1;  // the key before: the bucket in which the weight before b ends
        while (a.bn[g0 + p] == lo) --p;
        a.res_key[gb] = (uint32_t)b;
        a.res_prev[gb] = (uint32_t)p;
      }
      if (ok) {
        a.bslot[gb] = sel ? kDone : kNone;
        a.bnext[gb] = kNone;
      }
      continue;
    }
    const uint64_t m_full = __ballot(full), m_sel = __ballot(sel);
    // next non-empty bucket above this one
    const uint64_t above = lane == 63 ? 0ull : m_full >> (lane + 1);
    uint32_t nx = next;
    if (above) {
      const int l = lane + 1 + (int)__ffsll((unsigned long long)above) - 1;
      nx = (m_sel >> l) & 1ull ? (uint32_t)(g0 + b0 + l) : kNone;
    }
    uint32_t slot = kNone;
    if (m_sel) {
      const uint32_t w = sel ? weight(b) : 0u;
      const bool big = w > (uint32_t)kV2WaveCap;
      const uint64_t m_big = __ballot(big), m_small = m_sel & ~m_big;
      const uint32_t winc = wave_incl_scan(w);
      const uint64_t below = (1ull << lane) - 1ull;
      if (sel) {
        const V2Task tk{(uint32_t)k, (uint32_t)b};
        if (big) a.spill[at_big + (uint32_t)__popcll(m_big & below)] = tk;
        else a.tasks[at_small + (uint32_t)__popcll(m_small & below)] = tk;
        a.bcur[gb] = 0;
        a.carry_last[gb] = 0;
        slot = at_slot + winc - w;
      }
      at_small += (uint32_t)__popcll(m_small);
      at_big += (uint32_t)__popcll(m_big);
      at_slot += wave_last(winc);
    }
    if (ok) {
      a.bslot[gb] = slot;
      a.bnext[gb] = full ? nx : kNone;
    }
    if (m_full) {
      const int l = (int)__ffsll((unsigned long long)m_full) - 1;
      next = (m_sel >> l) & 1ull ? (uint32_t)(g0 + b0 + l) : kNone;
    }
  }
}

// Entries of the selected buckets into their scratch slots (the tiles of
// k_v2_hist; a tile of an item without a selected bucket ends at once).  A
// pass over the tile's keys appends the few selected entries to a list in LDS;
// the list then takes ranks per bucket in LDS and one run per bucket in the
// slots, so that a bucket's cursor sees one atomic per tile.  Bound by reading
// the keys (4 B per entry).
constexpr int kCollectCap = 4096;
template <int TASK>
__global__ void __launch_bounds__(kBlock) k_v2_collect(DataArgs d, LevelArgs lv, V2Args a) {
  extern __shared__ uint64_t s_tab[];
  __shared__ uint16_t s_list[kCollectCap];
  __shared__ unsigned int s_n;
  const V2Tile tl = a.tiles[blockIdx.x];
  if (!a.isel[tl.item]) return;
  const V2Item it = a.items[tl.item];
  if (it.width == 1) return;
  const int t = threadIdx.x;
  uint32_t* s_cnt = reinterpret_cast<uint32_t*>(s_tab);  // entries taken, then first position
  uint32_t* s_max = s_cnt + it.nb;                       // largest key (buckets below a selected one)
  uint8_t* s_flag = reinterpret_cast<uint8_t*>(s_max + it.nb);  // 1: selected, 2: below a selected one
  for (int b = t; b < it.nb; b += kBlock) {
    s_cnt[b] = 0;
    s_max[b] = 0;
    s_flag[b] = (uint8_t)((a.bslot[(int64_t)it.boff + b] != kNone ? 1 : 0) |
                          (a.bnext[(int64_t)it.boff + b] != kNone ? 2 : 0));
  }
  if (t == 0) s_n = 0;
  __syncthreads();
  const int n = min(a.tile, it.m - (int)tl.e0);
  const int64_t e0 = it.start + tl.e0;
  const uint32_t* gkey = a.gkey + it.soff + tl.e0;
  const int lane = t & (kWave - 1);
  auto flush = [&]() {
    __syncthreads();
    const int m = (int)s_n;
    constexpr int R = kCollectCap / kBlock;
    uint32_t key[R], rank[R], bk[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = t + r * kBlock;
      if (i < m) {
        key[r] = gkey[s_list[i]];
        bk[r] = v2_bucket(key[r], it);
        rank[r] = atomicAdd(&s_cnt[bk[r]], 1u);
      }
    }
    __syncthreads();
    for (int b = t; b < it.nb; b += kBlock) {
      const uint32_t c = s_cnt[b];
      if (c) s_cnt[b] = a.bslot[(int64_t)it.boff + b] + atomicAdd(&a.bcur[(int64_t)it.boff + b], c);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = t + r * kBlock;
      if (i < m) {
        const int64_t e = e0 + s_list[i];
        const uint32_t pos = s_cnt[bk[r]] + rank[r];
        a.skey[pos] = key[r];
        a.saux[pos] = lv.aux[e];
        if (TASK == 1) a.sy[pos] = lv.ey[e];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (t + r * kBlock < m) s_cnt[bk[r]] = 0;
    if (t == 0) s_n = 0;
    __syncthreads();
  };
  constexpr int U = 8;
  for (int base = 0; base < n; base += kBlock * U) {
    uint32_t keys[U];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int e = base + t + q * kBlock;
      keys[q] = e < n ? gkey[e] : 0u;
    }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int e = base + t + q * kBlock;
      uint32_t fl = 0;
      if (e < n) {
        const uint32_t b = v2_bucket(keys[q], it);
        fl = s_flag[b];
        if (fl & 2u) atomicMax(&s_max[b], keys[q]);
      }
      const uint64_t sel = __ballot(fl & 1u);
      if (sel) {
        unsigned int at = 0;
        if (lane == 0) at = atomicAdd(&s_n, (unsigned int)__popcll(sel));
        at = __builtin_amdgcn_readfirstlane(at);
        if (fl & 1u) s_list[at + (unsigned int)__popcll(sel & ((1ull << lane) - 1ull))] = (uint16_t)e;
      }
    }
    __syncthreads();
    const bool full = s_n > (unsigned int)(kCollectCap - kBlock * U);
    if (full) flush();  // workgroup-uniform
    else __syncthreads();
  }
  flush();
  for (int b = t; b < it.nb; b += kBlock)
    if (s_flag[b] & 2u) atomicMax(&a.carry_last[a.bnext[(int64_t)it.boff + b]], s_max[b]);
}

template <int MAXC, int TASK, int IPT>
__device__ __forceinline__ void v2_carry(const DataArgs& d, const V2Args& a, const V2Item& it, int64_t gb,
                                         TeamLds<MAXC, TASK, 256, IPT>& L) {
  if (threadIdx.x == 0) {
    for (int c = 0; c < MAXC; ++c)
      L.cr.run[c] = (TASK == 0 && c < d.C) ? a.bcls[(int64_t)it.boff * d.C + (int64_t)c * it.nb + (gb - it.boff)] : 0u;
    L.cr.run_n = a.bn[gb];
    L.cr.run_s = TASK == 1 ? a.bpos[gb] : 0;
    L.cr.last_key = a.carry_last[gb];
    L.cr.best_g = 0.0;
    L.cr.best_key = kNone;
    L.cr.best_prev = kNone;
  }
}

// Node context of an item from its precomputed fields; class totals to LDS
// (visible after the caller's next barrier).
template <int MAXC, int TASK, int IPT>
__device__ __forceinline__ NodeCtx v2_node(const DataArgs& d, const LevelArgs& lv, const V2Item& it,
                                           TeamLds<MAXC, TASK, 256, IPT>& L) {
  NodeCtx nc;
  nc.C = d.C;
  nc.n = it.n_w;
  nc.P = it.P;
  nc.ssum = it.ssum;
  nc.inv = it.inv;
  if (TASK == 0 && (int)threadIdx.x < d.C) L.ncls[threadIdx.x] = lv.cls[(int64_t)it.node * d.C + threadIdx.x];
  return nc;
}

// One wave per bucket of at most kV2WaveCap entries (four independent
// buckets per workgroup), grid-stride over the task list.  The loads of a
// wave's next bucket (task, item and bucket fields, carries, entries) are
// issued before its current bucket is sorted and walked.  Classification:
// k_v2_eval, three workgroups per CU (up to 16 classes: about 53 KB of LDS
// each, at most 168 VGPRs), bound by the latency of its x ln x reads;
// regression: k_v2_eval_reg.
template <int TASK, int IPT>
struct V2Pre {
  int64_t gb, e0;
  uint32_t node, kbase, width;
  int n;
  int64_t n_w, P, ssum;
  double inv;
  uint32_t carry_c;  // class carry of class `lane` (lanes < C)
  int64_t carry_n, carry_s;
  uint32_t carry_last;
  uint32_t ncls;     // node class total of class `lane`
  uint32_t key[IPT], aux[IPT];
  int64_t y[TASK == 1 ? IPT : 1];
};

template <int TASK, int IPT>
__device__ __forceinline__ void v2_prefetch(const DataArgs& d, const LevelArgs& lv, const V2Args& a, int64_t q,
                                            V2Pre<TASK, IPT>& P) {
  const int lane = threadIdx.x & (kWave - 1);
  const V2Task tk = a.tasks[q];
  const V2Item& it = a.items[tk.item];
  P.gb = (int64_t)it.boff + tk.b;
  P.kbase = tk.b * it.width;
  P.node = it.node;
  P.n_w = it.n_w;
  P.P = it.P;
  P.ssum = it.ssum;
  P.inv = it.inv;
  P.width = it.width;
  P.n = (int)a.bcur[P.gb];
  P.e0 = a.bslot[P.gb];
  P.carry_n = a.bn[P.gb];
  P.carry_s = TASK == 1 ? a.bpos[P.gb] : 0;
  P.carry_last = a.carry_last[P.gb];
  P.carry_c = (TASK == 0 && lane < d.C) ? a.bcls[(int64_t)it.boff * d.C + (int64_t)lane * it.nb + tk.b] : 0u;
  P.ncls = (TASK == 0 && lane < d.C) ? lv.cls[(int64_t)P.node * d.C + lane] : 0u;
#pragma unroll
  for (int k = 0; k < IPT; ++k) {
    const int e = lane + k * kWave;
    if (e < P.n) {
      P.key[k] = a.skey[P.e0 + e];
      P.aux[k] = a.saux[P.e0 + e];
      if (TASK == 1) P.y[k] = a.sy[P.e0 + e];
    }
  }
}

template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock, MAXC <= 16 ? 3 : 1) k_v2_eval(DataArgs d, LevelArgs lv, V2Args a) {
  const int64_t n_tasks = a.counters[0];
  static_assert(TASK == 0, "regression buckets go through k_v2_eval_reg");
  constexpr int IPT = kV2Ipt;
  __shared__ double s_inv[128], s_logc[128];
  __shared__ TeamLds<MAXC, TASK, kWave, IPT> s_team[kWaves];
  load_tables(s_inv, s_logc);
  __syncthreads();
  const LnCtx lx{s_inv, s_logc, d.T, d.Tmax, d.igF};
  const int t = threadIdx.x & (kWave - 1);
  TeamLds<MAXC, TASK, kWave, IPT>& L = s_team[threadIdx.x / kWave];
  const int64_t stride = (int64_t)gridDim.x * kWaves;
  int64_t q = (int64_t)blockIdx.x * kWaves + threadIdx.x / kWave;
  if (q >= n_tasks) return;  // wave-uniform; no workgroup barrier follows
  V2Pre<TASK, IPT> cur;
  v2_prefetch<TASK, IPT>(d, lv, a, q, cur);
  while (q < n_tasks) {
    NodeCtx nc;
    nc.C = d.C;
    nc.n = cur.n_w;
    nc.P = cur.P;
    nc.ssum = cur.ssum;
    nc.inv = cur.inv;
    if (t < d.C) {
      L.ncls[t] = cur.ncls;
      L.cr.run[t] = cur.carry_c;
    }
    if (t == 0) {
      for (int c = d.C; c < MAXC; ++c) L.cr.run[c] = 0u;
      L.cr.run_n = cur.carry_n;
      L.cr.run_s = cur.carry_s;
      L.cr.last_key = cur.carry_last;
      L.cr.best_g = 0.0;
      L.cr.best_key = kNone;
      L.cr.best_prev = kNone;
    }
    const int n = cur.n;
#pragma unroll
    for (int k = 0; k < IPT; ++k) {
      const int e = t + k * kWave;
      if (e < n) {
        L.u.srt.k[0][e] = cur.key[k] - cur.kbase;
        L.u.srt.v[0][e] = (uint16_t)e;
        L.aux[e] = cur.aux[k];
      }
    }
    const int64_t gb = cur.gb;
    const uint32_t kbase = cur.kbase;
    const int bits = bit_length(cur.width - 1u);
    team_sync<kWave>();
    const int64_t qn = q + stride;
    if (qn < n_tasks) v2_prefetch<TASK, IPT>(d, lv, a, qn, cur);
    sort_and_eval<MAXC, TASK, kWave, IPT>(n, bits, kbase, nc, L, lx);
    team_sync<kWave>();
    if (t == 0) {
      a.res_g[gb] = L.cr.best_g;
      a.res_key[gb] = L.cr.best_key;
      a.res_prev[gb] = L.cr.best_prev;
    }
    team_sync<kWave>();
    q = qn;
  }
}

// LDS of one wave of the regression bucket evaluator.  The payloads
// (weights, fixed-point targets) stay in registers through the sort and then
// go into the sort counters (targets) and the key buffer the sort left free
// (weights): about 10 KB per wave, three workgroups per CU.
template <int IPT>
struct RegWaveLds {
  static constexpr int CAP = kWave * IPT;
  static constexpr int SPAN = TeamLds<1, 1, kWave, IPT>::SPAN;
  uint32_t k[2][CAP];
  uint16_t v[2][CAP];
  union {
    uint16_t cnt[SPAN];
    int64_t y[CAP];
  } u;
  uint32_t w[8 * kWaves + kWaves];
  Carry<1, 1> cr;
  static_assert(sizeof(uint16_t) * SPAN >= sizeof(int64_t) * CAP, "targets fit the sort counters");
};

// Regression walk of a key-sorted bucket on one wave (the regression branch
// of eval_sorted_chunk with the payloads at wts / ys).
template <int IPT>
__device__ void eval_sorted_reg_wave(const uint32_t* keys, const uint16_t* vals, const uint32_t* wts,
                                     const int64_t* ys, int n, uint32_t kbase, const NodeCtx& nc, Carry<1, 1>& cr) {
  const int t = threadIdx.x & (kWave - 1);
  const int ipt = lane_span<kWave>(n);
  const int lo = t * ipt;
  const int hi = min(lo + ipt, n);
  BestCand tb{0.0, kNone, kNone};
  int64_t ln = 0, ls = 0;
  for (int p = lo; p < hi; ++p) {
    const uint16_t v = vals[p];
    const int64_t w = (int64_t)wts[v];
    ln += w;
    ls += w * ys[v];
  }
  int64_t tot_n, tot_s;
  int64_t pn = team_excl_scan_i64<kWave>(ln, nullptr, &tot_n);
  int64_t ps = team_excl_scan_i64<kWave>(ls, nullptr, &tot_s);
  pn += cr.run_n;
  ps += cr.run_s;
  if (lo < hi) {
    uint32_t prevk = (lo > 0) ? keys[lo - 1] + kbase : cr.last_key;
    for (int p = lo; p < hi; ++p) {
      const uint32_t k = keys[p] + kbase;
      if (pn > 0 && prevk < k) {
        const double g = variance_gain(pn, ps, nc.n - pn, nc.ssum - ps, 0);
        if (g > tb.g) tb = BestCand{g, k, prevk};
      }
      const uint16_t v = vals[p];
      const int64_t w = (int64_t)wts[v];
      pn += w;
      ps += w * ys[v];
      prevk = k;
    }
  }
  const BestCand b = wave_best(tb);
  if (t == 0) {
    carry_best(cr, b);
    cr.run_n += tot_n;
    cr.run_s += tot_s;
    if (n > 0) cr.last_key = keys[n - 1] + kbase;
  }
  team_sync<kWave>();
}

// k_v2_eval for regression: one wave per bucket, the same task order, sorts
// and walk, with the payloads written to LDS only once the bucket is sorted.
template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock, 3) k_v2_eval_reg(DataArgs d, LevelArgs lv, V2Args a) {
  const int64_t n_tasks = a.counters[0];
  static_assert(TASK == 1, "regression only");
  constexpr int IPT = kV2Ipt;
  constexpr int kSpan = RegWaveLds<IPT>::SPAN;
  __shared__ RegWaveLds<IPT> s_wave[kWaves];
  const int t = threadIdx.x & (kWave - 1);
  RegWaveLds<IPT>& L = s_wave[threadIdx.x / kWave];
  const int64_t stride = (int64_t)gridDim.x * kWaves;
  int64_t q = (int64_t)blockIdx.x * kWaves + threadIdx.x / kWave;
  if (q >= n_tasks) return;  // wave-uniform; no workgroup barrier follows
  V2Pre<TASK, IPT> cur;
  v2_prefetch<TASK, IPT>(d, lv, a, q, cur);
  while (q < n_tasks) {
    NodeCtx nc;
    nc.C = d.C;
    nc.n = cur.n_w;
    nc.P = cur.P;
    nc.ssum = cur.ssum;
    nc.inv = cur.inv;
    if (t == 0) {
      L.cr.run[0] = 0u;
      L.cr.run_n = cur.carry_n;
      L.cr.run_s = cur.carry_s;
      L.cr.last_key = cur.carry_last;
      L.cr.best_g = 0.0;
      L.cr.best_key = kNone;
      L.cr.best_prev = kNone;
    }
    const int n = cur.n;
    uint32_t pw[IPT];
    int64_t py[IPT];
#pragma unroll
    for (int k = 0; k < IPT; ++k) {
      const int e = t + k * kWave;
      if (e < n) {
        L.k[0][e] = cur.key[k] - cur.kbase;
        L.v[0][e] = (uint16_t)e;
        pw[k] = cur.aux[k] & 0xFFFFu;
        py[k] = cur.y[k];
      }
    }
    const int64_t gb = cur.gb;
    const uint32_t kbase = cur.kbase;
    const int bits = bit_length(cur.width - 1u);
    team_sync<kWave>();
    const int64_t qn = q + stride;
    if (qn < n_tasks) v2_prefetch<TASK, IPT>(d, lv, a, qn, cur);
    int sorted = 0;  // buffer holding the sorted bucket
    if (bits > 4 && (1 << bits) <= kSpan) {
      lds_count_sort<IPT, kWave>(L.k[0], L.v[0], L.k[1], L.v[1], n, 1 << bits, reinterpret_cast<uint32_t*>(L.u.cnt),
                                 L.w);
      sorted = 1;
    } else {
      for (int sh = 0; sh < bits; sh += 4) {
        lds_sort_pass<IPT, kWave>(L.k[sorted], L.v[sorted], L.k[sorted ^ 1], L.v[sorted ^ 1], n, sh, L.u.cnt, L.w);
        sorted ^= 1;
      }
    }
    uint32_t* wts = L.k[sorted ^ 1];
#pragma unroll
    for (int k = 0; k < IPT; ++k) {
      const int e = t + k * kWave;
      if (e < n) {
        wts[e] = pw[k];
        L.u.y[e] = py[k];
      }
    }
    team_sync<kWave>();
    eval_sorted_reg_wave<IPT>(L.k[sorted], L.v[sorted], wts, L.u.y, n, kbase, nc, L.cr);
    if (t == 0) {
      a.res_g[gb] = L.cr.best_g;
      a.res_key[gb] = L.cr.best_key;
      a.res_prev[gb] = L.cr.best_prev;
    }
    team_sync<kWave>();
    q = qn;
  }
}

// One workgroup per overfull bucket: fine sub-buckets of the bucket's key
// range, packed into LDS-sized chunks or read through an LDS histogram
// (a single sub-bucket above the capacity: heavy ties), walked in order.
template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock) k_v2_spill(DataArgs d, LevelArgs lv, V2Args a) {
  const int64_t n_spill = a.counters[1];
  if ((int64_t)blockIdx.x >= n_spill) return;
  constexpr int IPT = kIpt;
  constexpr int CAP = kCap;
  __shared__ double s_inv[128], s_logc[128];
  __shared__ TeamLds<MAXC, TASK, 256, IPT> L;
  __shared__ uint32_t s_boff[kMaxBuckets + 1];
  load_tables(s_inv, s_logc);
  __syncthreads();
  const LnCtx lx{s_inv, s_logc, d.T, d.Tmax, d.igF};
  const int t = threadIdx.x;
  for (int64_t q = blockIdx.x; q < n_spill; q += gridDim.x) {
    const V2Task tk = a.spill[q];
    const V2Item it = a.items[tk.item];
    const int64_t gb = (int64_t)it.boff + tk.b;
    const int n = (int)a.bcur[gb];
    const int64_t e0 = a.bslot[gb];
    const uint32_t klo = tk.b * it.width;
    const uint32_t span = min(it.width, d.S[it.f] - klo);
    const NodeCtx nc = v2_node(d, lv, it, L);
    v2_carry<MAXC, TASK, IPT>(d, a, it, gb, L);
    __syncthreads();
    if (n <= CAP) {
      // within the workgroup's LDS chunk: one sort and walk
      for (int e = t; e < n; e += 256) {
        L.u.srt.k[0][e] = a.skey[e0 + e] - klo;
        L.u.srt.v[0][e] = (uint16_t)e;
        L.aux[e] = a.saux[e0 + e];
        if (TASK == 1) L.y[e] = a.sy[e0 + e];
      }
      __syncthreads();
      sort_and_eval<MAXC, TASK, 256, IPT>(n, bit_length(span - 1u), klo, nc, L, lx);
      __syncthreads();
      if (t == 0) {
        a.res_g[gb] = L.cr.best_g;
        a.res_key[gb] = L.cr.best_key;
        a.res_prev[gb] = L.cr.best_prev;
      }
      __syncthreads();
      continue;
    }
    const int words = (TASK == 0) ? d.C : 3;
    int wbits = 0;
    while ((1 << (wbits + 1)) * words <= kHistWords) ++wbits;
    while (((span + (1u << wbits) - 1) >> wbits) > (uint32_t)kMaxBuckets) ++wbits;
    const int W = 1 << wbits;
    const int NB = (int)((span + (uint32_t)W - 1) >> wbits);
    const uint32_t* skey = a.skey + e0;
    const uint32_t* saux = a.saux + e0;
    const int64_t* sy = TASK == 1 ? a.sy + e0 : nullptr;
    uint32_t* dkey = a.skey2 + e0;
    uint32_t* daux = a.saux2 + e0;
    int64_t* dy = TASK == 1 ? a.sy2 + e0 : nullptr;
    for (int b = t; b <= NB; b += 256) s_boff[b] = 0;
    __syncthreads();
    for (int e = t; e < n; e += 256) atomicAdd(&s_boff[(skey[e] - klo) >> wbits], 1u);
    __syncthreads();
    {
      const int per = (NB + 255) / 256;
      const int b0 = t * per, b1 = min(b0 + per, NB);
      uint32_t loc = 0;
      for (int b = b0; b < b1; ++b) loc += s_boff[b];
      uint32_t base = team_excl_scan<256>(loc, L.w, nullptr);
      for (int b = b0; b < b1; ++b) {
        const uint32_t c = s_boff[b];
        s_boff[b] = base;
        base += c;
      }
      if (t == 0) s_boff[NB] = (uint32_t)n;
      __syncthreads();
      for (int b = t; b < NB; b += 256) L.u.bpos[b] = s_boff[b];
      __syncthreads();
    }
    for (int e = t; e < n; e += 256) {
      const uint32_t k = skey[e];
      const uint32_t pos = atomicAdd(&L.u.bpos[(k - klo) >> wbits], 1u);
      dkey[pos] = k;
      daux[pos] = saux[e];
      if (TASK == 1) dy[pos] = sy[e];
    }
    __syncthreads();
    int b = 0;
    while (b < NB) {
      const uint32_t cb = s_boff[b + 1] - s_boff[b];
      if (cb == 0) {
        ++b;
        continue;
      }
      if (cb > (uint32_t)CAP) {
        eval_hist_bucket<MAXC, TASK, IPT>(dkey + s_boff[b], daux + s_boff[b], TASK == 1 ? dy + s_boff[b] : nullptr,
                                          cb, klo + ((uint32_t)b << wbits), W, nc, L, lx);
        ++b;
        continue;
      }
      int be = b;
      uint32_t tot = 0;
      while (be < NB) {
        const uint32_t c = s_boff[be + 1] - s_boff[be];
        if (c > (uint32_t)CAP || tot + c > (uint32_t)CAP) break;
        tot += c;
        ++be;
      }
      const uint32_t c0 = s_boff[b];
      const uint32_t kbase = klo + ((uint32_t)b << wbits);
      for (int e = t; e < (int)tot; e += 256) {
        L.u.srt.k[0][e] = dkey[c0 + e] - kbase;
        L.u.srt.v[0][e] = (uint16_t)e;
        L.aux[e] = daux[c0 + e];
        if (TASK == 1) L.y[e] = dy[c0 + e];
      }
      __syncthreads();
      sort_and_eval<MAXC, TASK, 256, IPT>((int)tot, bit_length((uint32_t)(be - b) * (uint32_t)W - 1u), kbase, nc, L,
                                          lx);
      b = be;
    }
    __syncthreads();
    if (t == 0) {
      a.res_g[gb] = L.cr.best_g;
      a.res_key[gb] = L.cr.best_key;
      a.res_prev[gb] = L.cr.best_prev;
    }
    __syncthreads();
  }
}

// One wave per item: the best bucket (ties to the lower key).
template <int TASK>
__global__ void __launch_bounds__(kBlock) k_v2_reduce(DataArgs d, V2Args a, ItemArgs it) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t k = (int64_t)blockIdx.x * kWaves + threadIdx.x / kWave;
  if (k >= a.n_items) return;
  const V2Item bi = a.items[k];
  BestCand b{0.0, kNone, kNone};
  const int nb = a.isel[k] ? bi.nb : 0;
  for (int q = lane; q < nb; q += kWave) {
    const int64_t gb = (int64_t)bi.boff + q;
    if (a.bslot[gb] == kNone) continue;
    const uint32_t key = a.res_key[gb];
    if (key != kNone && cand_better(a.res_g[gb], key, b.g, b.key)) b = BestCand{a.res_g[gb], key, a.res_prev[gb]};
  }
  b = wave_best(b);
  if (lane == 0) {
    float score = 0.0f, thr = 0.0f;
    if (b.key != kNone) {
      const float* sv = d.SV + d.SVoff[bi.f];
      score = (float)(TASK == 0 ? b.g : ldexp_d(b.g, -2 * d.shift));
      thr = midpoint(sv[b.prev], sv[b.key]);
    }
    it.res_score[bi.ridx] = score;
    it.res_thr[bi.ridx] = thr;
    it.res_feat[bi.ridx] = bi.f;
  }
}

// Item table of a phase: one item per (big group, draw).
__global__ void k_v2_items(DataArgs d, LevelArgs lv, const uint32_t* groups, int64_t n_groups, int per_group, int j0,
                           int D, int nb_cap, int target, const float* res_score, uint32_t* nbest, V2Item* items) {
  const int64_t n = n_groups * per_group;
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t o = groups[k / per_group];
    const int j = j0 + (int)(k % per_group);
    const uint32_t i = lv.open_idx[o];
    V2Item b;
    b.f = (int)(rand_u32(d.seed, kStreamFeat, (uint32_t)lv.tree_global[lv.tree[i]], lv.id[i], (uint64_t)j) %
                (uint32_t)d.F);
    b.m = lv.m[i];
    b.start = lv.start[i];
    // Buckets of `width` consecutive keys of the feature's dense range
    // [0, S), so that a bucket holds about `target` of the node's m entries
    // (m * width / S), and at most nb_cap buckets.
    const uint32_t S = max(d.S[b.f], 1u);
    const uint64_t w_target = (uint64_t)S * (uint64_t)target / (uint64_t)max(b.m, 1);
    const uint32_t w_min = (uint32_t)(((uint64_t)S + nb_cap - 1) / nb_cap);
    b.width = (uint32_t)max<uint64_t>(max<uint64_t>(w_target, (uint64_t)w_min), 1);
    b.magic = b.width == 1 ? 0xFFFFFFFFu : (uint32_t)(0x100000000ull / b.width);
    b.nb = (int)((S + b.width - 1) / b.width);
    b.soff = 0;
    b.boff = 0;
    b.node = i;
    b.grp = (int)(k / per_group);
    if (j == j0) {  // the node's best score so far: the draws before this phase
      float best = 0.0f;
      for (int q = 0; q < j0; ++q) best = fmaxf(best, res_score[(int64_t)o * D + q]);
      nbest[b.grp] = __float_as_uint(best);
    }
    b.ridx = (int64_t)o * D + j;
    b.n_w = lv.count[i];
    b.P = 0;
    b.ssum = 0;
    b.inv = 0.0;
    if (d.C > 0) {
      const LnCtx lx{g_ln_table.inv, g_ln_table.logc, d.T, d.Tmax, d.igF};
      int64_t tsum = 0;
      for (int c = 0; c < d.C; ++c) tsum += lx.t(lv.cls[(int64_t)i * d.C + c]);
      b.P = lx.t((uint64_t)b.n_w) - tsum;
      b.inv = 1.0 / ((double)b.n_w * kLn2);
    } else {
      b.ssum = lv.sum[i];
    }
    items[k] = b;
  }
}

// Loads in flight for a walk over a node's entries by a team of TEAM threads:
// f(e, in, row, aux, value, target) for e = t, t + TEAM, ... < m, in order, kWalk
// steps' loads issued together.  One step at a time was bound by the latency
// of its chain (row, then the value it points at, then the payload of a left
// entry): about 1.8 us a step of a workgroup, 1.4 ms for the roots of 20
// forests of up to 200,000 rows; 0.39 ms with eight.
// Steps of a team that ends past m read the last entry again and come with
// `in` false, so that f may use ballots over the whole wave.
constexpr int kWalk = 8;
template <int TASK, int TEAM, class F>
__device__ __forceinline__ void walk_entries(const LevelArgs& lv, int64_t st, int m, const float* Xf, F&& f) {
  const int t = TEAM == kWave ? (int)(threadIdx.x & (kWave - 1)) : (int)threadIdx.x;
  const uint32_t* row = lv.row + st;
  const uint32_t* aux = lv.aux + st;
  const int64_t* ey = TASK == 1 ? lv.ey + st : nullptr;
  for (int e0 = 0; e0 < m; e0 += TEAM * kWalk) {
    uint32_t r[kWalk], a[kWalk];
    float x[kWalk];
    int64_t y[TASK == 1 ? kWalk : 1];
#pragma unroll
    for (int q = 0; q < kWalk; ++q)
      if (e0 + q * TEAM < m) {
        const uint32_t e = (uint32_t)min(e0 + q * TEAM + t, m - 1);
        r[q] = row[e];
        a[q] = aux[e];
        if constexpr (TASK == 1) y[q] = ey[e];
      }
#pragma unroll
    for (int q = 0; q < kWalk; ++q)
      if (e0 + q * TEAM < m) x[q] = Xf[r[q]];
#pragma unroll
    for (int q = 0; q < kWalk; ++q)
      if (e0 + q * TEAM < m) {
        const int e = e0 + q * TEAM + t;
        int64_t yq = 0;
        if constexpr (TASK == 1) yq = y[q];
        f(e, e < m, r[q], a[q], x[q], yq);
      }
  }
}

// ------------------------------------------------ ERT split search ------
// One block per item: threshold = fp32 mean of 10 node values drawn with
// replacement (gpuert.cu:167-183, summed in draw order), then a 2 x C
// histogram (gpuert.cu:287-301) or per-side target sums (gpuert.cu:348-361).
template <int MAXC, int TASK>
__device__ __forceinline__ void ert_block_body(DataArgs d, LevelArgs lv, ItemArgs it, int64_t bid, int64_t nblk,
                                               double* s_inv, double* s_logc) {
  resolve_level(lv, d.C);
  resolve_items(it);
  if ((int64_t)bid >= it.n_groups * it.per_group) return;
  __shared__ uint32_t s_left[MAXC];
  __shared__ unsigned long long s_nl;
  __shared__ unsigned long long s_sl;
  __shared__ float s_thr;
  load_ln_table(s_inv, s_logc);
  __syncthreads();
  const int t = threadIdx.x;
  unsigned long long my_bytes = 0;
  const int64_t n_items = it.n_groups * it.per_group;
  for (int64_t item = bid; item < n_items; item += nblk) {
    const int64_t grp = it.node_major ? item % it.n_groups : item / it.per_group;
    const int q = (int)(it.node_major ? item / it.n_groups : item % it.per_group);
    const uint32_t o = it.list ? it.list[grp] : (uint32_t)grp;
    const uint32_t i = lv.open_idx[o];
    const int tr = lv.tree[i];
    const DataArgs dd = forest_data(d, tr);
    const int j = item_draw(d, dd, it, q);
    if (j < 0) continue;  // past this forest's draws (joint build); block-uniform
    const uint32_t tg = (uint32_t)lv.tree_global[tr];
    const uint32_t nid = lv.id[i];
    const int f = (int)(rand_u32(dd.seed, kStreamFeat, tg, nid, (uint64_t)j) % (uint32_t)dd.F);
    const int m = lv.m[i];
    const int64_t st = lv.start[i];
    const float* Xf = dd.X + (int64_t)f * dd.N;
    if (t < MAXC) s_left[t] = 0;
    if (t == 0) {
      s_nl = 0;
      s_sl = 0;
      float acc = 0.0f;
      for (int s = 0; s < 10; ++s) {
        const uint32_t pos = rand_u32(dd.seed, kStreamThr, tg, nid, (uint64_t)j * 10 + s) % (uint32_t)m;
        acc = acc + Xf[lv.row[st + pos]];
      }
      s_thr = acc / 10.0f;
      my_bytes += (unsigned long long)m * (TASK == 0 ? 12ull : 20ull);
    }
    __syncthreads();
    const float thr = s_thr;
    uint32_t loc[MAXC];
#pragma unroll
    for (int c = 0; c < MAXC; ++c) loc[c] = 0;
    uint64_t nl = 0;
    int64_t sl = 0;
    walk_entries<TASK, kBlock>(lv, st, m, Xf, [&](int, bool in, uint32_t, uint32_t a, float x, int64_t y) {
      const uint32_t w = in && side_of(x, thr) == 0 ? a & 0xFFFFu : 0u;
      nl += w;
      if (TASK == 0) {
        const int lab = (int)(a >> 16);
#pragma unroll
        for (int c = 0; c < MAXC; ++c) loc[c] += (c == lab) ? w : 0u;
      } else {
        sl += (int64_t)w * y;
      }
    });
    if (TASK == 0) {
#pragma unroll
      for (int c = 0; c < MAXC; ++c) {
        uint32_t v = loc[c];
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
        if ((t & (kWave - 1)) == 0 && v) atomicAdd(&s_left[c], v);
      }
    }
    {
      uint64_t v = nl;
      int64_t sm = sl;
#pragma unroll
      for (int off = kWave / 2; off > 0; off >>= 1) {
        v += __shfl_xor(v, off, kWave);
        sm += __shfl_xor(sm, off, kWave);
      }
      if ((t & (kWave - 1)) == 0) {
        atomicAdd(&s_nl, (unsigned long long)v);
        if (TASK == 1) atomicAdd(&s_sl, (unsigned long long)sm);
      }
    }
    __syncthreads();
    if (t == 0) {
      const int64_t n = lv.count[i];
      const int64_t nlt = (int64_t)s_nl;
      float score;
      if (nlt == 0 || nlt == n) {
        score = -FLT_MAX;
      } else if (TASK == 0) {
        const uint32_t* nclsp = lv.cls + (int64_t)i * d.C;
        const int F = dd.igF;
        const double inv = 1.0 / ((double)n * kLn2);
        int64_t P = xlnx_fixed((uint64_t)n, F, s_inv, s_logc);
        int64_t sls = 0, srs = 0;
        for (int c = 0; c < d.C; ++c) {
          P -= xlnx_fixed(nclsp[c], F, s_inv, s_logc);
          sls += xlnx_fixed(s_left[c], F, s_inv, s_logc);
          srs += xlnx_fixed(nclsp[c] - s_left[c], F, s_inv, s_logc);
        }
        const int64_t Q = (sls - xlnx_fixed((uint64_t)nlt, F, s_inv, s_logc)) +
                          (srs - xlnx_fixed((uint64_t)(n - nlt), F, s_inv, s_logc));
        score = (float)ig_from_fixed(P + Q, F, inv);
      } else {
        const int64_t slt = (int64_t)s_sl;
        score = (float)variance_gain(nlt, slt, n - nlt, lv.sum[i] - slt, dd.shift);
      }
      const int64_t ridx = (int64_t)o * it.D + j;
      it.res_score[ridx] = score;
      it.res_thr[ridx] = thr;
      it.res_feat[ridx] = f;
    }
    __syncthreads();
  }
  if (t == 0 && my_bytes && it.bytes) add_bytes(it.bytes, my_bytes);
}
template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock) k_search_ert(DataArgs d, LevelArgs lv, ItemArgs it) {
  __shared__ double s_inv[128], s_logc[128];
  ert_block_body<MAXC, TASK>(d, lv, it, blockIdx.x, gridDim.x, s_inv, s_logc);
}

// ------------------------------------------------ wave and segment moves --
__device__ __forceinline__ uint32_t ds_permute_u32(uint32_t dst_lane, uint32_t v) {
  return (uint32_t)__builtin_amdgcn_ds_permute((int)(dst_lane << 2), (int)v);
}

// All lanes active.
__device__ __forceinline__ int64_t wave_sum_i64(int64_t v) { return wave_last_i64(wave_incl_scan_i64(v)); }

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = max(v, dpp_u32<0x111>(v, 0u));
  v = max(v, dpp_u32<0x112>(v, 0u));
  v = max(v, dpp_u32<0x114>(v, 0u));
  v = max(v, dpp_u32<0x118>(v, 0u));
  v = max(v, dpp_u32<0x142, 0xa>(v, 0u));
  v = max(v, dpp_u32<0x143, 0xc>(v, 0u));
  return wave_last(v);
}

// Scans and sums of a 16- or 32-lane segment in DPP moves (a shuffle goes
// through the LDS pipe).  All lanes of a segment are active together.
template <int SEG>
__device__ __forceinline__ uint32_t seg_incl_u32(uint32_t x) {
  static_assert(SEG == 16 || SEG == 32, "");
  x += dpp_u32<0x111>(x, 0u);
  x += dpp_u32<0x112>(x, 0u);
  x += dpp_u32<0x114>(x, 0u);
  x += dpp_u32<0x118>(x, 0u);
  if constexpr (SEG == 32) x += dpp_u32<0x142, 0xa>(x, 0u);
  return x;
}
template <int SEG>
__device__ __forceinline__ int64_t seg_incl_i64(int64_t x) {
  static_assert(SEG == 16 || SEG == 32, "");
  x += dpp_i64<0x111>(x);
  x += dpp_i64<0x112>(x);
  x += dpp_i64<0x114>(x);
  x += dpp_i64<0x118>(x);
  if constexpr (SEG == 32) x += dpp_i64<0x142, 0xa>(x);
  return x;
}

template <int SEG>
__device__ __forceinline__ int64_t seg_sum_i64(int64_t v) {
  if constexpr (SEG == kWave) {
    return wave_sum_i64(v);
  } else {
    v += dpp_i64<0x128>(v);  // row_ror: every lane gets the row's sum
    v += dpp_i64<0x124>(v);
    v += dpp_i64<0x122>(v);
    v += dpp_i64<0x121>(v);
    if constexpr (SEG == 32) v += __shfl_xor(v, 16, 32);
    return v;
  }
}

// f(r, value of lane r of this lane's row of 16), r = 0 .. 15.
template <class F, int... R>
__device__ __forceinline__ void row_lanes_impl(uint32_t v, F&& f, std::integer_sequence<int, R...>) {
  (f(R, dpp_u32<0x150 + R>(v, 0u)), ...);
}
template <class F>
__device__ __forceinline__ void row_lanes(uint32_t v, F&& f) {
  row_lanes_impl(v, f, std::make_integer_sequence<int, 16>{});
}

// Rank of a lane's key among its segment's, ties by lane.
template <int SEG>
__device__ __forceinline__ uint32_t seg_rank(uint32_t key) {
  const int rl = threadIdx.x & 15;
  uint32_t cnt = 0;
  const uint32_t next = key + 1u;
  row_lanes(key, [&](int r, uint32_t k) { cnt += k < (r < rl ? next : key) ? 1u : 0u; });
  if constexpr (SEG == 32) {  // the other row's lanes all come before or after
    const uint32_t other = (uint32_t)__shfl_xor((int)key, 16, 32);
    const uint32_t lim = (threadIdx.x & 16) ? next : key;
    row_lanes(other, [&](int, uint32_t k) { cnt += k < lim ? 1u : 0u; });
  }
  return cnt;
}

template <int SEG>
__device__ __forceinline__ uint32_t seg_max_u32(uint32_t v) {
#pragma unroll
  for (int off = SEG / 2; off > 0; off >>= 1) v = max(v, (uint32_t)__shfl_xor(v, off, SEG));
  return v;
}

// Largest positive gain of a segment whose lanes are in key order, the lowest
// key among equals (positive doubles order as their bits).
template <int SEG>
__device__ __forceinline__ BestCand seg_best(double gain, uint32_t key, uint32_t prev) {
  const int64_t g = __builtin_bit_cast(int64_t, gain > 0.0 ? gain : 0.0);
  int64_t b = g;
  auto take = [&](int64_t o) { b = o > b ? o : b; };
  take(dpp_i64<0x128>(b));
  take(dpp_i64<0x124>(b));
  take(dpp_i64<0x122>(b));
  take(dpp_i64<0x121>(b));
  if constexpr (SEG == 32) take(__shfl_xor(b, 16, 32));
  const int base = threadIdx.x & (kWave - 1) & ~(SEG - 1);
  const uint64_t win = (__ballot(b > 0 && g == b) >> base) & ((1ull << SEG) - 1ull);
  const int w = win ? (int)__ffsll((unsigned long long)win) - 1 : 0;
  const uint32_t k = (uint32_t)__shfl((int)key, w, SEG), p = (uint32_t)__shfl((int)prev, w, SEG);
  return win ? BestCand{__builtin_bit_cast(double, b), k, p} : BestCand{0.0, kNone, kNone};
}

template <int TASK>
struct SegLds {
  static constexpr int kTL = 2048;  // LDS copy of T's head
  double inv[128], logc[128];
  int64_t T[TASK == 0 ? kTL : 1];
};

// Segment-per-node RF search for tiny nodes: a wave holds 64 / SEG nodes, one
// per SEG-lane segment (one entry per lane, m <= SEG, C <= SEG), and loops
// over the node's draws (its unit's, in a level of few nodes), so node
// statistics and entry loads are shared by the draws.
template <int MAXC, int TASK, int SEG>
__device__ __forceinline__ void rf_seg_body(DataArgs d, LevelArgs lv, ItemArgs it, int64_t bid, int64_t nblk,
                                            SegLds<TASK>& S) {
  constexpr int NPW = kWave / SEG;  // segments per wave
  resolve_level(lv, d.C);
  resolve_items(it);
  const int split = node_split(it, (int64_t)it.spread * NPW, it.n_groups);
  const int64_t n_units = it.n_groups * split;
  if (bid * kWaves * NPW >= n_units) return;
  load_tables(S.inv, S.logc);
  const int64_t nTL = TASK == 0 ? load_t_prefix<SegLds<TASK>::kTL>(S.T, d.T, d.Tmax) : 0;
  __syncthreads();
  const LnCtxL lx{S.inv, S.logc, d.T, d.Tmax, d.igF, S.T, nTL};
  const int sl = threadIdx.x & (SEG - 1);
  const int seg = (threadIdx.x & (kWave - 1)) / SEG;
  unsigned long long my_bytes = 0;
  const int64_t wave_id = bid * kWaves + threadIdx.x / kWave;
  const int64_t n_waves = nblk * kWaves;
  for (int64_t u0 = wave_id * NPW; u0 < n_units; u0 += n_waves * NPW) {
    const int64_t u = u0 + seg;
    const bool node_ok = u < n_units;
    const int64_t g = split > 1 ? (int64_t)((uint32_t)u / (uint32_t)split) : u;
    const int j1 = split > 1 ? (int)((uint32_t)u % (uint32_t)split) : 0;  // the unit's first draw
    uint32_t o = 0, i = 0, tg = 0, nid = 0;
    int m = 0;
    int64_t st = 0, n = 0, ssum = 0;
    if (node_ok) {
      o = it.list ? it.list[g] : (uint32_t)g;
      i = lv.open_idx[o];
      tg = (uint32_t)lv.tree_global[lv.tree[i]];
      nid = lv.id[i];
      m = lv.m[i];
      st = lv.start[i];
      n = lv.count[i];
      if (TASK == 1) ssum = lv.sum[i];
    }
    // node statistics (shared by all draws)
    uint32_t ncls_lane = 0;
    int64_t P = 0, SR0 = 0;
    double inv = 0.0;
    bool pure = false;
    if (TASK == 0) {
      ncls_lane = (node_ok && sl < d.C) ? lv.cls[(int64_t)i * d.C + sl] : 0u;
      pure = (int64_t)seg_max_u32<SEG>(ncls_lane) == n;
      SR0 = seg_sum_i64<SEG>(sl < d.C ? lx.t(ncls_lane) : 0);
      P = lx.t((uint64_t)n) - SR0;
      inv = 1.0 / ((double)n * kLn2);
    }
    const bool valid = node_ok && sl < m;
    uint32_t row = 0, pay0 = 0;
    int64_t y0 = 0;
    if (valid) {
      row = lv.row[st + sl];
      pay0 = lv.aux[st + sl];
      if (TASK == 1) y0 = lv.ey[st + sl];
    }
    if (sl == 0 && node_ok && !pure && j1 == 0) my_bytes += (unsigned long long)m * it.per_group * (TASK == 0 ? 12ull : 20ull);
    // Draw pipeline: the key gather (and value offset) of draw jj + 1 and the
    // threshold values of draw jj - 1 are in flight while draw jj is ranked
    // and scored.
    int f_nx = 0;
    uint32_t key_nx = kNone;
    int64_t svo_nx = 0;
    if (!pure && it.per_group > 0) {
      f_nx = (int)(rand_u32(d.seed, kStreamFeat, tg, nid, (uint64_t)(it.j0 + j1)) % (uint32_t)d.F);
      key_nx = valid ? d.K[(int64_t)f_nx * d.N + row] : kNone;
      svo_nx = d.SVoff[f_nx];
    }
    bool pend = false, p_has = false;
    int64_t p_ridx = 0;
    int p_f = 0;
    float p_score = 0.0f, p_lo = 0.0f, p_hi = 0.0f;
    for (int jj = j1; jj < it.per_group; jj += split) {
      const int j = it.j0 + jj;
      const int64_t ridx = (int64_t)o * it.D + j;
      if (pure) {
        if (sl == 0 && node_ok) {
          it.res_score[ridx] = 0.0f;
          it.res_thr[ridx] = 0.0f;
          it.res_feat[ridx] = (int)(rand_u32(d.seed, kStreamFeat, tg, nid, (uint64_t)j) % (uint32_t)d.F);
        }
        continue;
      }
      const int f = f_nx;
      const int64_t svo = svo_nx;
      uint32_t key = key_nx;
      if (jj + split < it.per_group) {
        f_nx = (int)(rand_u32(d.seed, kStreamFeat, tg, nid, (uint64_t)(j + split)) % (uint32_t)d.F);
        key_nx = valid ? d.K[(int64_t)f_nx * d.N + row] : kNone;
        svo_nx = d.SVoff[f_nx];
      }
      // rank inside the segment (ties by lane; lanes past m hold kNone), then
      // move entries into key order
      const uint32_t cnt = seg_rank<SEG>(key);
      const uint32_t rank = valid ? cnt : (uint32_t)sl;
      const uint32_t dst = (uint32_t)(threadIdx.x & (kWave - 1) & ~(SEG - 1)) + rank;
      key = ds_permute_u32(dst, key);
      const uint32_t pay = ds_permute_u32(dst, pay0);
      int64_t yv = 0;
      if (TASK == 1) {
        const uint32_t lo = ds_permute_u32(dst, (uint32_t)(uint64_t)y0);
        const uint32_t hi = ds_permute_u32(dst, (uint32_t)((uint64_t)y0 >> 32));
        yv = (int64_t)(((uint64_t)hi << 32) | lo);
      }
      const uint32_t w = valid ? (pay & 0xFFFFu) : 0u;
      const uint32_t prevk = (uint32_t)__shfl_up((int)key, 1, SEG);
      const bool cand = valid && sl >= 1 && prevk < key;
      double gval = 0.0;
      const uint32_t nl = seg_incl_u32<SEG>(w) - w;
      if (TASK == 0) {
        // class weights before the entry: two classes to a word, each word
        // scanned, and the entry's half picked
        const uint32_t lab = pay >> 16;
        const uint32_t wv2 = (lab & 1u) ? w << 16 : w;
        uint32_t mine = 0;
        constexpr int PAIRS = (MAXC + 1) / 2;
#pragma unroll
        for (int p = 0; p < PAIRS; ++p)
          if (2 * p < d.C) {
            const bool own = (lab >> 1) == (uint32_t)p;
            const uint32_t x = seg_incl_u32<SEG>(own ? wv2 : 0u);
            if (own) mine = x;
          }
        const uint32_t pre = ((lab & 1u) ? mine >> 16 : mine & 0xFFFFu) - w;
        const uint32_t ncl = (uint32_t)__shfl((int)ncls_lane, (int)lab, SEG);
        int64_t dt = 0;  // left and right terms move together
        if (valid) dt = (S.T[pre + w] - S.T[pre]) + (S.T[ncl - pre - w] - S.T[ncl - pre]);
        const int64_t q = SR0 + (seg_incl_i64<SEG>(dt) - dt);
        if (cand) gval = ig_from_fixed(P + (q - S.T[nl] - S.T[(uint32_t)n - nl]), lx.F, inv);
      } else {
        const int64_t wy = (int64_t)w * yv;
        const int64_t ps = seg_incl_i64<SEG>(wy) - wy;
        if (cand) gval = variance_gain((int64_t)nl, ps, n - (int64_t)nl, ssum - ps, 0);
      }
      const BestCand b = seg_best<SEG>(cand ? gval : 0.0, key, prevk);
      if (pend) {
        it.res_score[p_ridx] = p_score;
        it.res_thr[p_ridx] = p_has ? midpoint(p_lo, p_hi) : 0.0f;
        it.res_feat[p_ridx] = p_f;
        pend = false;
      }
      if (sl == 0 && node_ok) {
        pend = true;
        p_ridx = ridx;
        p_f = f;
        p_has = b.key != kNone;
        p_score = 0.0f;
        if (p_has) {
          const float* sv = d.SV + svo;
          p_score = (float)(TASK == 0 ? b.g : ldexp_d(b.g, -2 * d.shift));
          p_lo = sv[b.prev];
          p_hi = sv[b.key];
        }
      }
    }
    if (pend) {
      it.res_score[p_ridx] = p_score;
      it.res_thr[p_ridx] = p_has ? midpoint(p_lo, p_hi) : 0.0f;
      it.res_feat[p_ridx] = p_f;
    }
  }
  if (sl == 0 && my_bytes && it.bytes) add_bytes(it.bytes, my_bytes);
}
template <int MAXC, int TASK, int SEG>
__global__ void __launch_bounds__(kBlock) k_search_rf_seg(DataArgs d, LevelArgs lv, ItemArgs it) {
  __shared__ SegLds<TASK> S;
  rf_seg_body<MAXC, TASK, SEG>(d, lv, it, blockIdx.x, gridDim.x, S);
}

// ------------------------------------ RF split search by bucket bounds ---
// Nodes of 33 .. 2048 entries.  A wave takes one (node, draw) at a time with
// the node's keys in registers, spreads them over power-of-two wide key
// buckets, counts classes (regression: weights and centred target sums) per
// bucket in LDS, and bounds the gain of every boundary inside a bucket from
// the counts on both sides of it (k_v2_bound has the inequality).  Only
// buckets whose bound reaches the node's best candidate so far -- over the
// bucket edges of this draw and everything earlier draws found -- are ordered
// and scored exactly; with about 8 entries a bucket that is one bucket in a
// hundred, so the sort and the scored walk of all entries (310 wave
// instructions per 64 entries at 10 classes) are replaced by a histogram (14)
// and a fixed 400 or so per draw.  The bounds are in fp32 with a margin for
// their rounding; scored candidates use the exact fixed-point sums, and a
// candidate whose fp32 score could equal the node's best is always scored.
// A surviving bucket above 64 entries is split again over its own key range
// (entries below it are counted as the totals before it); one of a single key
// has no boundary but its lower edge.
//
// Bound by VALU issue, so the register budget decides (a first version with
// 184 VGPRs ran two waves per SIMD).  Node weights stay within 16 bits (fit_batch's cuts), so that two classes
// share a word and the table of terms answers every lookup.
constexpr uint32_t kEdge = 0xFFFFFFFEu;  // previous key not in the list (lower edge of a bucket)

// Best candidate of a draw: exact gain, key, key before it.
struct DrawBest {
  double g;
  uint32_t key, prev;
};

// Entries of a run of surviving buckets, for one wave.
struct BoundList {
  uint32_t key[kWave], aux[kWave];
  int64_t y[kWave];
};

template <int MAXC, int TASK, int LOGB, int IPT>
struct BoundLds {
  static constexpr int NB = 1 << LOGB;
  static constexpr int PAIRS = (MAXC + 1) / 2;
  static constexpr int TAB = kTfMax / 2;  // staged x ln x terms
  // classification: [p * NB + b], classes 2p and 2p + 1 in the halves of a
  // word; regression: weights.  Counts, then totals before the bucket.
  uint32_t hist[TASK == 0 ? NB * PAIRS : NB];
  int64_t pos[TASK == 1 ? NB : 1], neg[TASK == 1 ? NB : 1];
  uint16_t wgt[NB];  // bucket weights
  uint32_t below[TASK == 0 ? PAIRS : 1];
  int64_t below_s[1];
  uint32_t ncls[TASK == 0 ? MAXC : 1];
  BoundList list;
  uint32_t stk_k[IPT + 1];  // from 1 on
  uint32_t stk_b[IPT + 1];
  static_assert(wave_stack(kWave * IPT) <= IPT, "ranges of the wave tier");
};

// Value of the lane below (lane 0: `first`) through DPP wave_shr:1.
__device__ __forceinline__ float lane_below_f32(float v, float first) {
  return __uint_as_float(dpp_u32<0x138>(__float_as_uint(v), __float_as_uint(first)));
}

// fp32 chord_gap.
__device__ __forceinline__ float chord_gap_f32(float a, float s) {
  const float e = s * 0.36788f;
  return a > 0.0f ? fminf(e, s * s * 0.125001f * __builtin_amdgcn_rcpf(a) * 1.00001f) : e;
}

// A node as one wave works on it.
struct BoundNode {
  int m;
  int64_t n;
  int64_t start;  // first entry
  const uint32_t* row;  // the node's entries (wave-uniform bases: the loads
  const uint32_t* aux;  // take a scalar base and a 32-bit lane offset)
  const int64_t* ey;
  int64_t P;      // classification
  int64_t ssum;   // regression
  double inv;     // classification: 1 / (n ln 2)
  float Pn, margin;  // classification: P and the rounding margin, nats
  int64_t mu;     // regression: centre
  double M;       // regression: largest |target - centre|
  double E;       // regression: reg_gain_error
};

// f(q, e) for the steps q of a team of TEAM lanes over a node's m entries, q
// unrolled behind a wave-uniform test; e = lane + TEAM q, clamped to the last
// entry (no lane is masked off: loads of several steps stay in flight
// together).  Keys of lanes past m are kNone and fall in no range.
template <int IPT, int TEAM, class F>
__device__ __forceinline__ void for_entries(int m, F&& f) {
  const uint32_t t = TEAM == kWave ? threadIdx.x & (kWave - 1) : threadIdx.x;
#pragma unroll
  for (int q = 0; q < IPT; ++q)
    if (q * TEAM < m) f(q, min(t + (uint32_t)(q * TEAM), (uint32_t)(m - 1)));
}

// Keys of a draw; kNone past the node's entries.  Kf: the feature's keys by
// row, or the draw's keys of the node by entry with rows = the entry numbers
// (draw_base).
template <int IPT, int TEAM>
__device__ __forceinline__ void gather_keys(const uint32_t* Kf, int m, const uint32_t (&rows)[IPT],
                                            uint32_t (&key)[IPT]) {
  for_entries<IPT, TEAM>(m, [&](int q, uint32_t) {
    uint32_t r = rows[q];
    asm volatile("" : "+v"(r));  // 32-bit here: else every row is kept as a 64-bit pair
    key[q] = Kf[r];
  });
}
__device__ __forceinline__ const uint32_t* draw_base(const DataArgs& d, const ItemArgs& it, int f, int q,
                                                     int64_t start) {
  return it.gk ? it.gk + q * it.gk_stride + start : d.K + (int64_t)f * d.N;
}
template <int IPT, int TEAM>
__device__ __forceinline__ void mask_keys(int m, uint32_t (&key)[IPT]) {
  const uint32_t t = TEAM == kWave ? threadIdx.x & (kWave - 1) : threadIdx.x;
  for_entries<IPT, TEAM>(m, [&](int q, uint32_t) {
    if (t + (uint32_t)(q * TEAM) >= (uint32_t)m) key[q] = kNone;
  });
}

// A node's payloads.
template <int TASK, int IPT>
struct BoundPay {
  uint32_t a[IPT];
  int64_t t[TASK == 1 ? IPT : 1];
};

// Payloads of a list whose aux words hold entry numbers.
template <int TASK>
__device__ __forceinline__ void bound_list_payload(const BoundNode& nd, BoundList& W, int cnt) {
  const int lane = threadIdx.x & (kWave - 1);
  if (lane < cnt) {
    const uint32_t x = W.aux[lane];
    W.aux[lane] = nd.aux[x];
    if constexpr (TASK == 1) W.y[lane] = nd.ey[x];
  }
  team_sync<kWave>();
}

// Exact scores of the boundaries of a run of buckets holding cnt <= 64
// entries (in L.lkey / laux / ly), with the totals before bucket b of the
// bucket table.
template <int TASK, int LOGB, class LdsT>
__device__ __forceinline__ void bound_run(const DataArgs& d, const BoundNode& nd, const LdsT& L, const BoundList& W,
                                          int cnt, int b, DrawBest& best) {
  constexpr int NB = 1 << LOGB;
  const int lane = threadIdx.x & (kWave - 1);
  const bool valid = lane < cnt;
  const uint32_t key = valid ? W.key[lane] : kNone;
  const uint32_t pay = valid ? W.aux[lane] : 0u;
  const uint32_t w = pay & 0xFFFFu;
  BestCand c{0.0, kNone, kNone};
  if constexpr (TASK == 0) {
    const int64_t* T = d.T;
    const uint32_t lab = pay >> 16;
    auto before = [&](uint32_t cl) -> uint32_t { return (L.hist[(cl >> 1) * NB + b] >> ((cl & 1u) << 4)) & 0xFFFFu; };
    // totals before the run, one class per lane
    const uint32_t rc = lane < d.C ? before((uint32_t)lane) : 0u;
    int64_t s0 = lane < d.C ? T[rc] + T[L.ncls[lane] - rc] : 0;
    s0 = wave_last_i64(wave_incl_scan_i64(s0));
    const uint32_t n0 = wave_last(wave_incl_scan(rc));
    uint32_t rank = 0, pre = 0, nw = 0;
    for (int x = 0; x < cnt; ++x) {
      const uint32_t kx = (uint32_t)__builtin_amdgcn_readlane((int)key, x);
      const uint32_t px = (uint32_t)__builtin_amdgcn_readlane((int)pay, x);
      const uint32_t lt = kx < key || (kx == key && x < lane) ? 1u : 0u;
      const uint32_t wx = lt ? px & 0xFFFFu : 0u;
      rank += lt;
      nw += wx;
      pre += (px >> 16) == lab ? wx : 0u;
    }
    if (!valid) rank = (uint32_t)lane;
    int64_t dd = 0, tq = 0;
    const uint32_t nl = n0 + nw;
    if (valid) {
      const uint32_t l = before(lab) + pre, tc = L.ncls[lab];
      dd = (T[l + w] - T[l]) + (T[tc - l - w] - T[tc - l]);
      tq = T[nl] + T[(uint32_t)nd.n - nl];
    }
    // running sums in key order, then back to the entry's lane
    const uint32_t ks = ds_permute_u32(rank, key);
    const uint32_t dlo = ds_permute_u32(rank, (uint32_t)(uint64_t)dd);
    const uint32_t dhi = ds_permute_u32(rank, (uint32_t)((uint64_t)dd >> 32));
    const int64_t ds = (int64_t)(((uint64_t)dhi << 32) | dlo);
    const int64_t ex = wave_incl_scan_i64(ds) - ds;
    const int64_t sum = __shfl(ex, (int)rank, kWave);
    const uint32_t pk = __shfl(ks, (int)rank > 0 ? (int)rank - 1 : 0, kWave);
    if (valid && nl > 0 && (rank == 0 || pk < key)) {
      const int64_t pq = nd.P + s0 + sum - tq;
      if (pq > 0) {
        const double g = ig_from_fixed(pq, d.igF, nd.inv);
        if (cand_better(g, key, best.g, best.key)) c = BestCand{g, key, rank == 0 ? kEdge : pk};
      }
    }
  } else {
    const int64_t y = valid ? W.y[lane] : 0;
    uint32_t rank = 0;
    for (int x = 0; x < cnt; ++x) {
      const uint32_t kx = (uint32_t)__builtin_amdgcn_readlane((int)key, x);
      rank += kx < key || (kx == key && x < lane) ? 1u : 0u;
    }
    if (!valid) rank = (uint32_t)lane;
    const uint32_t ks = ds_permute_u32(rank, key);
    const uint32_t ws = ds_permute_u32(rank, w);
    const int64_t wy = (int64_t)w * y;
    const uint32_t ylo = ds_permute_u32(rank, (uint32_t)(uint64_t)wy);
    const uint32_t yhi = ds_permute_u32(rank, (uint32_t)((uint64_t)wy >> 32));
    const int64_t ys = (int64_t)(((uint64_t)yhi << 32) | ylo);
    const int64_t pn = (int64_t)(L.hist[b] + wave_incl_scan(ws) - ws);
    const int64_t ps = L.pos[b] + wave_incl_scan_i64(ys) - ys;
    const uint32_t pk = dpp_u32<0x138>(ks, 0u);
    if (lane < cnt && pn > 0 && (lane == 0 || pk < ks)) {
      const double g = variance_gain(pn, ps, nd.n - pn, nd.ssum - ps, 0);
      if (g > 0.0 && cand_better(g, ks, best.g, best.key)) c = BestCand{g, ks, lane == 0 ? kEdge : pk};
    }
  }
  if (__ballot(c.key != kNone)) {
    c = wave_best(c);
    best = DrawBest{c.g, c.key, c.prev};
  }
}

// The lower edge of bucket b (a single key, `key`) alone.
template <int TASK, int LOGB, class LdsT>
__device__ __forceinline__ void bound_edge(const DataArgs& d, const BoundNode& nd, const LdsT& L, uint32_t key, int b, DrawBest& best) {
  constexpr int NB = 1 << LOGB;
  const int lane = threadIdx.x & (kWave - 1);
  double g = 0.0;
  if constexpr (TASK == 0) {
    const int64_t* T = d.T;
    const uint32_t rc = lane < d.C ? (L.hist[(lane >> 1) * NB + b] >> ((lane & 1) << 4)) & 0xFFFFu : 0u;
    int64_t s0 = lane < d.C ? T[rc] + T[L.ncls[lane] - rc] : 0;
    s0 = wave_last_i64(wave_incl_scan_i64(s0));
    const uint32_t n0 = wave_last(wave_incl_scan(rc));
    if (n0 == 0) return;
    const int64_t pq = nd.P + s0 - (T[n0] + T[(uint32_t)nd.n - n0]);
    if (pq > 0) g = ig_from_fixed(pq, d.igF, nd.inv);
  } else {
    const int64_t pn = (int64_t)L.hist[b], ps = L.pos[b];
    if (pn == 0) return;
    g = variance_gain(pn, ps, nd.n - pn, nd.ssum - ps, 0);
  }
  if (g > 0.0 && cand_better(g, key, best.g, best.key)) best = DrawBest{g, key, kEdge};
}

// Least gain whose fp32 score can equal the score of gain thr.  Variances have
// no scale: above the largest fp32 number all scores are infinity, below the
// normal ones they are 2^-149 apart.
template <int TASK>
__device__ __forceinline__ double bound_cut(const DataArgs& d, double thr) {
  if (TASK == 0) return thr * (1.0 - 1e-6);
  return fmin(thr, ldexp_d((double)FLT_MAX, 2 * d.shift)) * (1.0 - 1e-6) - ldexp_d(1.0, 2 * d.shift - 148);
}

// One draw of a node.  thr: lower bound of the node's best gain that matters
// here (nats, or fixed-point units squared); returns the draw's best in
// `best` (none when no candidate of it can be the node's best) and raises thr
// by what it found.
template <int MAXC, int TASK, int LOGB, int IPT>
__device__ __forceinline__ void bound_draw(const DataArgs& d, const BoundNode& nd,
                                           const float* s_tf, BoundLds<MAXC, TASK, LOGB, IPT>& L,
                                           const uint32_t (&key)[IPT], const BoundPay<TASK, IPT>& pay, double& thr,
                                           DrawBest& best) {
  using LdsT = BoundLds<MAXC, TASK, LOGB, IPT>;
  constexpr int NB = LdsT::NB;
  constexpr int NR = NB / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int m = nd.m;
  uint32_t kmin = kNone, kmax = 0;
  for_entries<IPT, kWave>(m, [&](int q, uint32_t) {
    kmin = min(kmin, key[q]);
    kmax = max(kmax, key[q] + 1u);  // kNone wraps to 0
  });
  kmin = wave_min_u32(kmin);
  kmax = wave_max_u32(kmax) - 1u;
  best = DrawBest{0.0, kNone, kNone};
  if (kmin == kmax) return;  // one value: no boundary
  int sp = 1;
  uint32_t k0 = kmin;
  int sb = bit_length(kmax - kmin);
  for (;;) {
    const int shift = max(0, sb - LOGB);
    const uint32_t nbk = 1u << (sb - shift);  // buckets of the range
    // ---- bucket table
    if constexpr (TASK == 0) {
      const int words = (d.C + 1) / 2;
      for (int i = lane; i < words * NB; i += kWave) L.hist[i] = 0;
      if (lane < LdsT::PAIRS) L.below[lane] = 0;
    } else {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        L.hist[r * kWave + lane] = 0;
        L.pos[r * kWave + lane] = 0;
        L.neg[r * kWave + lane] = 0;
      }
      if (lane == 0) {
        L.below[0] = 0;
        L.below_s[0] = 0;
      }
    }
    team_sync<kWave>();
    for_entries<IPT, kWave>(m, [&](int q, uint32_t e) {
      const uint32_t b = (key[q] - k0) >> shift;
      const bool in = key[q] >= k0 && b < nbk, lower = key[q] < k0;
      const uint32_t a = pay.a[q];
      const uint32_t w = a & 0xFFFFu;
      if constexpr (TASK == 0) {
        const uint32_t p = a >> 17;                 // class / 2
        const uint32_t v = w << ((a >> 12) & 16u);  // odd class: high half
        if (in) atomicAdd(&L.hist[p * (uint32_t)NB + b], v);
        else if (lower) atomicAdd(&L.below[p], v);
      } else {
        const int64_t dy = pay.t[q] - nd.mu;
        const unsigned long long wy = (unsigned long long)((int64_t)w * dy);
        if (in) {
          atomicAdd(&L.hist[b], w);
          atomicAdd(reinterpret_cast<unsigned long long*>(dy < 0 ? &L.neg[b] : &L.pos[b]), wy);
        } else if (lower) {
          atomicAdd(&L.below[0], w);
          atomicAdd(reinterpret_cast<unsigned long long*>(&L.below_s[0]), wy);
        }
      }
    });
    team_sync<kWave>();
    // ---- edges and bounds, 64 buckets at a time
    uint64_t mask[NR];
    if constexpr (TASK == 0) {
      const bool big_n = nd.n >= LdsT::TAB;
      auto tf = [&](uint32_t x) -> float {
        if (big_n) return x > 1 ? (float)x * __logf((float)x) : 0.0f;
        return s_tf[x];
      };
      constexpr int PAIRS = LdsT::PAIRS;
      const uint32_t n = (uint32_t)nd.n;
      const int words = (d.C + 1) / 2;
      float eb = 0.0f;
      float ub[NR];
      uint32_t run[PAIRS];
      uint32_t run_n = 0;
#pragma unroll
      for (int p = 0; p < PAIRS; ++p) {
        run[p] = p < words ? __builtin_amdgcn_readfirstlane(L.below[p]) : 0u;
        run_n += (run[p] & 0xFFFFu) + (run[p] >> 16);
      }
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        ub[r] = -1.0f;
        if ((uint32_t)(r * kWave) >= nbk) break;
        const int b = r * kWave + lane;
        uint32_t sw = 0;
#pragma unroll
        for (int p = 0; p < PAIRS; ++p)
          if (p < words) {
            const uint32_t v = L.hist[p * NB + b];
            sw += (v & 0xFFFFu) + (v >> 16);
          }
        const uint32_t lb = run_n + wave_incl_scan(sw), la = lb - sw;
        const float psb = tf(lb) + tf(n - lb);
        const float psa = lane_below_f32(psb, tf(run_n) + tf(n - run_n));
        run_n = wave_last(lb);
        const float slope = sw ? (psb - psa) / (float)sw : 0.0f;
        float phi = 0.0f, slack = 0.0f;
#pragma unroll
        for (int p = 0; p < PAIRS; ++p) {
          if (p < words) {
            const uint32_t v = L.hist[p * NB + b];
            const uint32_t inc = run[p] + wave_incl_scan(v);
            const uint32_t n0 = L.ncls[2 * p], n1 = PAIRS > 1 || MAXC > 1 ? L.ncls[2 * p + 1] : 0u;
            const uint32_t l0 = inc & 0xFFFFu, l1 = inc >> 16;
            const float b0 = tf(l0) + tf(n0 - l0), b1 = tf(l1) + tf(n1 - l1);
            const uint32_t r0 = run[p] & 0xFFFFu, r1 = run[p] >> 16;
            const float a0 = lane_below_f32(b0, tf(r0) + tf(n0 - r0));
            const float a1 = lane_below_f32(b1, tf(r1) + tf(n1 - r1));
            run[p] = wave_last(inc);
            phi += a0 + a1;
            slack += fmaxf(0.0f, (b0 - a0) - slope * (float)(v & 0xFFFFu)) +
                     fmaxf(0.0f, (b1 - a1) - slope * (float)(v >> 16));
            L.hist[p * NB + b] = inc - v;
          }
        }
        slack += chord_gap_f32((float)la, (float)sw) + chord_gap_f32((float)(n - lb), (float)sw);
        const float edge = nd.Pn + phi - psa;
        if (sw) {
          ub[r] = edge + (shift ? slack : 0.0f) + nd.margin;  // shift 0: one key, only the edge
          if (la > 0) eb = fmaxf(eb, edge - nd.margin);
          else if (!shift) ub[r] = -1.0f;
        }
        L.wgt[b] = (uint16_t)sw;
      }
      eb = __uint_as_float(wave_max_u32(__float_as_uint(eb)));
      thr = fmax(thr, (double)eb);
      const float thr_f = (float)bound_cut<TASK>(d, thr);
#pragma unroll
      for (int r = 0; r < NR; ++r) mask[r] = __ballot(ub[r] >= thr_f && ub[r] > 0.0f);
    } else {
      const double N = (double)nd.n, S = (double)(nd.ssum - nd.mu * nd.n);
      uint32_t run_n = __builtin_amdgcn_readfirstlane(L.below[0]);
      int64_t run_s = L.below_s[0];
      double eb = 0.0;
      double ub[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        ub[r] = -1.0;
        if ((uint32_t)(r * kWave) >= nbk) break;
        const int b = r * kWave + lane;
        const uint32_t w = L.hist[b];
        const int64_t sp_ = L.pos[b], sn_ = L.neg[b];
        const uint32_t lb = run_n + wave_incl_scan(w), la = lb - w;
        run_n = wave_last(lb);
        const int64_t se = run_s + wave_incl_scan_i64(sp_ + sn_), sa = se - (sp_ + sn_);
        run_s = wave_last_i64(se);
        L.hist[b] = la;
        L.pos[b] = sa + nd.mu * (int64_t)la;  // uncentred target sum before the bucket
        if (w) {
          double edge = 0.0;
          if (la > 0) {
            const double s = (double)sa, t = S - s;
            edge = s * s / (double)la + t * t / (N - (double)la) - S * S / N;
            eb = fmax(eb, edge * (1.0 - 2e-6) - nd.E);
          }
          if (shift)
            ub[r] = reg_box_bound((double)la, (double)lb, (double)(sa + sn_), (double)(sa + sp_), N, S, nd.M) *
                        (1.0 + 2e-6) + nd.E;
          else if (la > 0)
            ub[r] = edge * (1.0 + 2e-6) + nd.E;
        }
        L.wgt[b] = (uint16_t)w;
      }
#pragma unroll
      for (int off = kWave / 2; off > 0; off >>= 1) eb = fmax(eb, __shfl_xor(eb, off, kWave));
      thr = fmax(thr, eb);
      const double thr_d = bound_cut<TASK>(d, thr);
#pragma unroll
      for (int r = 0; r < NR; ++r) mask[r] = __ballot(ub[r] >= thr_d && ub[r] > 0.0);
    }
    team_sync<kWave>();
    // ---- surviving buckets
    for (int r = 0; r < NR; ++r) {
      uint64_t mk = mask[0];
#pragma unroll
      for (int x = 1; x < NR; ++x) mk = r == x ? mask[x] : mk;
      while (mk) {
        const int i = (int)__ffsll((unsigned long long)mk) - 1;
        int e = i;  // last bucket of the run
        const int b = r * kWave + i;
        uint32_t wsum = __builtin_amdgcn_readfirstlane((uint32_t)L.wgt[b]);
        mk &= mk - 1;
        while (e + 1 < kWave && ((mk >> (e + 1)) & 1ull)) {
          const uint32_t wn = __builtin_amdgcn_readfirstlane((uint32_t)L.wgt[b + (e - i) + 1]);
          if (wsum + wn > (uint32_t)kWave) break;
          wsum += wn;
          ++e;
          mk &= mk - 1;
        }
        const uint32_t klo = k0 + ((uint32_t)b << shift);
        const uint32_t kspan = (uint32_t)(e - i + 1) << shift;
        if (!shift && wsum > (uint32_t)kWave) {
          bound_edge<TASK, LOGB>(d, nd, L, klo, b, best);
          continue;
        }
        int cnt = 0;
        for_entries<IPT, kWave>(m, [&](int q, uint32_t x) {
          const bool in = key[q] >= klo && key[q] - klo < kspan;
          const uint64_t bal = __ballot(in);
          const int at = cnt + (int)__popcll(bal & ((1ull << lane) - 1ull));
          if (in && at < kWave) {
            L.list.key[at] = key[q];
            L.list.aux[at] = x;  // entry, its payload below
          }
          cnt += (int)__popcll(bal);
        });
        team_sync<kWave>();
        if (cnt > kWave) {
          // one bucket above 64 entries (runs are merged by weight): split it
          // again; fewer than IPT disjoint ranges of more than 64 entries exist
          if (lane == 0) {
            L.stk_k[sp] = klo;
            L.stk_b[sp] = (uint32_t)shift;
          }
          ++sp;
        } else {
          bound_list_payload<TASK>(nd, L.list, cnt);
          bound_run<TASK, LOGB>(d, nd, L, L.list, cnt, b, best);
        }
        team_sync<kWave>();
      }
    }
    if (best.key != kNone)
      thr = fmax(thr, (TASK == 0 ? best.g * (double)nd.n * kLn2 : best.g) * (1.0 - 1e-6));
    if (sp <= 1) break;
    --sp;
    team_sync<kWave>();
    k0 = __builtin_amdgcn_readfirstlane(L.stk_k[sp]);
    sb = (int)__builtin_amdgcn_readfirstlane(L.stk_b[sp]);
  }
  if (best.prev == kEdge) {  // largest key below the best candidate's
    uint32_t p = 0;
    for_entries<IPT, kWave>(m, [&](int q, uint32_t) {
      if (key[q] < best.key) p = max(p, key[q]);
    });
    best.prev = wave_max_u32(p);
  }
}

// Node context of a bounded search; returns whether the node is pure.  ncls:
// class totals (LDS).  WG: entries of the node spread over the workgroup
// (256 per step), else over a wave.
template <int MAXC, int TASK>
__device__ __forceinline__ bool bound_node(const DataArgs& d, const LevelArgs& lv, uint32_t i, uint32_t* ncls,
                                           BoundNode& nd) {
  const int lane = threadIdx.x & (kWave - 1);
  nd.m = __builtin_amdgcn_readfirstlane(lv.m[i]);
  nd.n = __builtin_amdgcn_readfirstlane(lv.count[i]);
  const int64_t st = lv.start[i];
  nd.start = st;
  nd.row = lv.row + st;
  nd.aux = lv.aux + st;
  nd.ey = TASK == 1 ? lv.ey + st : nullptr;
  nd.P = 0;
  nd.ssum = 0;
  nd.mu = 0;
  nd.M = 0.0;
  nd.E = 0.0;
  if constexpr (TASK == 0) {
    const uint32_t my = lane < d.C ? lv.cls[(int64_t)i * d.C + lane] : 0u;
    if (lane < MAXC) ncls[lane] = my;
    const int64_t tn_fixed = d.T[nd.n];
    nd.P = tn_fixed - wave_last_i64(wave_incl_scan_i64(lane < d.C ? d.T[my] : 0));
    nd.inv = 1.0 / ((double)nd.n * kLn2);
    nd.Pn = (float)ldexp_d((double)nd.P, -d.igF);
    // fp32 terms of at most T(n) nats: (4 C + 16) roundings of 2^-24 of
    // twice that, doubled
    const float tn = (float)ldexp_d((double)tn_fixed, -d.igF);
    nd.margin = tn * (float)(4 * d.C + 16) * 2.4e-7f + 1e-6f;
    return (int64_t)wave_max_u32(my) == nd.n;
  } else {
    nd.ssum = lv.sum[i];
    nd.mu = d2ll_rn((double)nd.ssum / (double)nd.n);
    return false;
  }
}

// A score in the units of the bounds, rounded down.
template <int TASK>
__device__ __forceinline__ double bound_units(const DataArgs& d, const BoundNode& nd, float s) {
  return (TASK == 0 ? (double)s * (double)nd.n * kLn2 : ldexp_d((double)s, 2 * d.shift)) * (1.0 - 1e-6);
}

template <int TASK>
__device__ __forceinline__ void bound_write(const DataArgs& d, const ItemArgs& it, int64_t ridx, int f,
                                            const DrawBest& best, float score) {
  const float* sv = d.SV + d.SVoff[f];
  it.res_score[ridx] = score;
  it.res_thr[ridx] = best.key != kNone ? midpoint(sv[best.prev], sv[best.key]) : 0.0f;
  it.res_feat[ridx] = f;
}

// Every boundary of a pure node has gain exactly 0: no positive split.
__device__ __forceinline__ void bound_pure(const DataArgs& d, const ItemArgs& it, uint32_t o, uint32_t tg,
                                           uint32_t nid) {
  for (int jj = 0; jj < it.per_group; ++jj) {
    const int j = it.j0 + jj;
    const int64_t ridx = (int64_t)o * it.D + j;
    it.res_score[ridx] = 0.0f;
    it.res_thr[ridx] = 0.0f;
    it.res_feat[ridx] = (int)(rand_u32(d.seed, kStreamFeat, tg, nid, (uint64_t)j) % (uint32_t)d.F);
  }
}

// ------------------------------------------- all draws' keys of a level ---
// A draw's key costs the fabric a 64-byte half of a line per entry (rows of a
// node lie anywhere), so a level with many draws moves 64 D bytes an entry.
// With the keys of a row side by side (KR, rows of FS words), the entry's row
// comes over once, whole, and its D keys are written in entry order, where
// every search kernel reads them back streaming: 4 FS + 8 D bytes.  Taken
// where that is at most a third, with more keys than the caches hold
// (key_rows_pay).  Fits of 64 features in ms, without and with: 4M rows, 21
// draws, 8 trees 175 and 141; 1M, 21, 16 trees 75 and 69; 250 k, 21 26.9 and
// 27.5; 1M, 11 draws 51 and 50 (regression), 43 and 44 (8 classes).
// A wave takes 64 entries of a node at a time through LDS: rows in, 16 bytes a
// lane, and a column out per draw (an odd row stride: no bank conflicts).
// 20 M entries, 64 features, 21 draws: 1.7 ms a level, 7 GB at 4.1 TB/s (a copy
// runs at 4.7); the searches it feeds fell from 7.3 to 3.4 ms a level.
constexpr int kGatherWaves = 2;
constexpr int kGatherRun = 8;        // tiles a wave takes in a row
constexpr int kGatherMaxFS = 112;    // 2 waves' rows in 64 KB of LDS
constexpr int64_t kGatherMinKeys = (int64_t)32 << 20;

inline bool key_rows_pay(int64_t N, int F, int draws) {
  const int FS = (F + 15) / 16 * 16;
  return FS <= kGatherMaxFS && draws <= kWave && N * F >= kGatherMinKeys && 64 * draws >= 3 * (4 * FS + 8 * draws);
}

// KR[row * FS + f] = K[f][row], zero above F; 64 rows a workgroup.
__global__ void __launch_bounds__(kBlock) k_key_rows(const uint32_t* __restrict__ K, int64_t N, int F, int FS,
                                                     uint32_t* __restrict__ KR) {
  extern __shared__ uint32_t s_rows[];
  const int64_t row0 = blockIdx.x * (int64_t)kWave;
  const int nr = (int)min<int64_t>(kWave, N - row0);
  const int lane = threadIdx.x & (kWave - 1);
  for (int f = threadIdx.x / kWave; f < FS; f += kWaves)
    s_rows[lane * (FS + 1) + f] = f < F && lane < nr ? K[(int64_t)f * N + row0 + lane] : 0u;
  __syncthreads();
  for (int x = threadIdx.x; x < nr * FS; x += kBlock) KR[row0 * FS + x] = s_rows[x / FS * (FS + 1) + x % FS];
}

// Nodes whose draws are gathered: the lists of search tiers 2 .. 5, one after
// the other.
struct DrawNodes {
  const uint32_t* list[4];
  int64_t first[5];
};
__device__ __forceinline__ uint32_t draw_node(const DrawNodes& dn, int64_t q) {
  int k = 0;
  while (k < 3 && q >= dn.first[k + 1]) ++k;
  return dn.list[k][q - dn.first[k]];
}

__global__ void k_draw_tiles(LevelArgs lv, DrawNodes dn, uint32_t* tiles) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < dn.first[4]; q += (int64_t)gridDim.x * blockDim.x)
    tiles[q] = (uint32_t)((lv.m[lv.open_idx[draw_node(dn, q)]] + kWave - 1) / kWave);
}

__global__ void __launch_bounds__(kGatherWaves * kWave)
    k_gather_draws(DataArgs d, LevelArgs lv, const uint32_t* __restrict__ KR, int FS, DrawNodes dn,
                   const uint32_t* __restrict__ toff, int draws, uint32_t* __restrict__ gk, int64_t stride) {
  extern __shared__ uint32_t s_rows[];
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  uint32_t* S = s_rows + wv * kWave * (FS + 1);
  const int64_t n = dn.first[4];
  const int64_t total = toff[n];
  const int lpr = FS / 4;  // 16-byte pieces of a row
  const int sub = lane >> 4, c = lane & 15;
  for (int64_t run = (int64_t)blockIdx.x * kGatherWaves + wv; run * kGatherRun < total;
       run += (int64_t)gridDim.x * kGatherWaves) {
    int64_t tile = run * kGatherRun;
    const int64_t t1 = min(tile + kGatherRun, total);
    int64_t q = 0, hi = n - 1;  // the last node whose first tile is at most `tile`
    while (q < hi) {
      const int64_t mid = (q + hi + 1) >> 1;
      if ((int64_t)toff[mid] <= tile) q = mid;
      else hi = mid - 1;
    }
    for (; tile < t1; ++q) {
      const uint32_t o = __builtin_amdgcn_readfirstlane(draw_node(dn, q));
      const uint32_t i = __builtin_amdgcn_readfirstlane(lv.open_idx[o]);
      const int m = __builtin_amdgcn_readfirstlane(lv.m[i]);
      const int64_t st = lv.start[i];
      const uint32_t tg = (uint32_t)lv.tree_global[lv.tree[i]], nid = lv.id[i];
      const int fl = lane < draws ? (int)(rand_u32(d.seed, kStreamFeat, tg, nid, (uint64_t)lane) % (uint32_t)d.F) : 0;
      const int64_t first = toff[q], last = min(t1, (int64_t)toff[q + 1]);
      for (; tile < last; ++tile) {
        const int e0 = (int)(tile - first) * kWave;
        const int cnt = min(kWave, m - e0);
        const int64_t at = st + e0 + min(lane, cnt - 1);
        const uint32_t row = lv.row[at];
        for (int c0 = 0; c0 < lpr; c0 += 16)
          for (int i0 = 0; i0 < cnt; i0 += 32) {
            uint4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              const uint32_t r = (uint32_t)__shfl((int)row, i0 + u * 4 + sub, kWave);
              if (c0 + c < lpr) v[u] = *reinterpret_cast<const uint4*>(KR + (int64_t)r * FS + 4 * (c0 + c));
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
              if (c0 + c < lpr) {
                uint32_t* w = S + (i0 + u * 4 + sub) * (FS + 1) + 4 * (c0 + c);
                w[0] = v[u].x;
                w[1] = v[u].y;
                w[2] = v[u].z;
                w[3] = v[u].w;
              }
          }
        team_sync<kWave>();
        uint32_t* out = gk + at;
        for (int j = 0; j < draws; ++j) {
          const uint32_t key = S[lane * (FS + 1) + __builtin_amdgcn_readlane(fl, j)];
          if (lane < cnt) out[j * stride] = key;
        }
        team_sync<kWave>();
      }
    }
  }
}

// Nodes of up to 64 IPT entries, one wave per node: the draws in order, the
// next draw's key gather in flight.
constexpr int kBoundLogB = 6;

template <int MAXC, int TASK, int IPT>
struct BoundWgLds {
  using Wave = BoundLds<MAXC, TASK, kBoundLogB, IPT>;
  float tf[TASK == 0 ? Wave::TAB : 1];
  Wave l[kWaves];
};

template <int MAXC, int TASK, int IPT>
__device__ __forceinline__ void rf_bound_body(DataArgs d, LevelArgs lv, ItemArgs it, int64_t bid, int64_t nblk,
                                              BoundWgLds<MAXC, TASK, IPT>& S) {
  constexpr int LOGB = kBoundLogB;
  using LdsT = BoundLds<MAXC, TASK, LOGB, IPT>;
  resolve_level(lv, d.C);
  resolve_items(it);
  const int split = node_split(it, it.spread, it.n_groups);
  const int64_t n_units = it.n_groups * split;
  if (bid * kWaves >= n_units) return;  // no node for this workgroup
  float* s_tf = S.tf;
  if (TASK == 0)
    for (int i = threadIdx.x; i < LdsT::TAB; i += kBlock) s_tf[i] = d.Tf[i];
  __syncthreads();
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  LdsT& L = S.l[wv];
  const int lane = threadIdx.x & (kWave - 1);
  unsigned long long my_bytes = 0;
  for (int64_t u = bid * kWaves + wv; u < n_units; u += nblk * kWaves) {
    const int64_t grp = split > 1 ? (int64_t)((uint32_t)u / (uint32_t)split) : u;
    const int j1 = split > 1 ? (int)((uint32_t)u % (uint32_t)split) : 0;  // the unit's first draw
    const uint32_t o = __builtin_amdgcn_readfirstlane(it.list ? it.list[grp] : (uint32_t)grp);
    const uint32_t i = __builtin_amdgcn_readfirstlane(lv.open_idx[o]);
    const uint32_t tg = (uint32_t)__builtin_amdgcn_readfirstlane(lv.tree_global[lv.tree[i]]);
    const uint32_t nid = __builtin_amdgcn_readfirstlane(lv.id[i]);
    BoundNode nd;
    if (bound_node<MAXC, TASK>(d, lv, i, L.ncls, nd)) {
      if (lane == 0 && j1 == 0) bound_pure(d, it, o, tg, nid);
      continue;
    }
    const int m = nd.m;
    uint32_t rows[IPT], kn[IPT];
    BoundPay<TASK, IPT> pay;
    const bool by_row = !it.gk;
    for_entries<IPT, kWave>(m, [&](int q, uint32_t e) {
      rows[q] = by_row ? nd.row[e] : e;
      pay.a[q] = nd.aux[e];
      if constexpr (TASK == 1) pay.t[q] = nd.ey[e];
    });
    if constexpr (TASK == 1) {
      double M = 0.0;
      for_entries<IPT, kWave>(m, [&](int q, uint32_t) { M = fmax(M, fabs((double)(pay.t[q] - nd.mu))); });
#pragma unroll
      for (int off = kWave / 2; off > 0; off >>= 1) M = fmax(M, __shfl_xor(M, off, kWave));
      nd.M = M * (1.0 + 1e-12);
      nd.E = d.no_bound ? __builtin_inf() : reg_gain_error((double)nd.n, fabs((double)nd.mu) + nd.M);
    }
    // the node's best score so far: the draws before this phase
    float best_score = 0.0f;
    for (int q = 0; q < it.j0; ++q) best_score = fmaxf(best_score, it.res_score[(int64_t)o * it.D + q]);
    double thr = bound_units<TASK>(d, nd, best_score);
    int f_nx = (int)(rand_u32(d.seed, kStreamFeat, tg, nid, (uint64_t)(it.j0 + j1)) % (uint32_t)d.F);
    gather_keys<IPT, kWave>(draw_base(d, it, f_nx, j1, nd.start), m, rows, kn);
    for (int jj = j1; jj < it.per_group; jj += split) {
      const int j = it.j0 + jj;
      // once a retry draw passed 1e-3 the later ones are not looked at (k_decide2)
      if (it.j0 > 0 && (double)best_score > 1e-3) break;
      const int f = f_nx;
      uint32_t key[IPT];
#pragma unroll
      for (int q = 0; q < IPT; ++q) key[q] = kn[q];
      mask_keys<IPT, kWave>(m, key);
      if (jj + split < it.per_group) {
        f_nx = (int)(rand_u32(d.seed, kStreamFeat, tg, nid, (uint64_t)(j + split)) % (uint32_t)d.F);
        gather_keys<IPT, kWave>(draw_base(d, it, f_nx, jj + split, nd.start), m, rows, kn);
      }
      DrawBest best;
      bound_draw<MAXC, TASK, LOGB, IPT>(d, nd, s_tf, L, key, pay, thr, best);
      float score = 0.0f;
      if (best.key != kNone) score = (float)(TASK == 0 ? best.g : ldexp_d(best.g, -2 * d.shift));
      best_score = fmaxf(best_score, score);
      if (lane == 0) bound_write<TASK>(d, it, (int64_t)o * it.D + j, f, best, score);
    }
    if (lane == 0 && j1 == 0) my_bytes += (unsigned long long)m * it.per_group * (TASK == 0 ? 12ull : 20ull);
  }
  if (lane == 0 && my_bytes && it.bytes) add_bytes(it.bytes, my_bytes);
}
template <int MAXC, int TASK, int IPT>
__global__ void __launch_bounds__(kBlock, IPT == 1 ? 5 : 4 - TASK) k_search_rf_bound(DataArgs d, LevelArgs lv, ItemArgs it) {
  __shared__ BoundWgLds<MAXC, TASK, IPT> S;
  rf_bound_body<MAXC, TASK, IPT>(d, lv, it, blockIdx.x, gridDim.x, S);
}

// Nodes of up to 2048 entries, one workgroup per node and draw at a time: 256
// buckets (128 above 16 classes), bounded 64 to a wave; every wave scores the
// surviving buckets of its own 64.  The entries of those buckets come from
// all waves through a list per wave, in rounds of at most kTeamList of them.
constexpr int kTeamIpt2 = kCap / kBlock;  // entries per thread
constexpr int kTeamList = 128;
static_assert(kBoundRun == kWave, "a run is an entry per lane");

template <int MAXC, int TASK, int LOGB>
struct BoundTeamLds {
  static constexpr int NB = 1 << LOGB;
  static constexpr int PAIRS = (MAXC + 1) / 2;
  uint32_t hist[TASK == 0 ? NB * PAIRS : NB];
  int64_t pos[TASK == 1 ? NB : 1], neg[TASK == 1 ? NB : 1];
  uint16_t wgt[NB];
  uint32_t below[TASK == 0 ? PAIRS : 1];
  int64_t below_s[1];
  uint32_t ncls[TASK == 0 ? MAXC : 1];
  uint32_t tot[kWaves][TASK == 0 ? PAIRS : 1];  // of a wave's buckets
  uint32_t tot_n[kWaves];
  int64_t tot_s[kWaves];
  uint32_t w[kWaves], w2[kWaves];
  double eb[kWaves];
  unsigned long long mask[kWaves];
  unsigned int cnt[kWaves];
  uint32_t lkey[kWaves][kTeamList];
  uint16_t lidx[kWaves][kTeamList];
  BoundList list[kWaves];
  DrawBest best[kWaves];
  uint32_t stk_k[kTeamStack];  // first keys and widths (log2) of ranges to split again
  uint8_t stk_b[kTeamStack];
  int sp;
};

template <int MAXC, int TASK>
struct BoundTeamWgLds {
  static constexpr int LOGB = MAXC <= 16 ? 8 : 7;
  float tf[TASK == 0 ? kTfMax : 1];
  BoundTeamLds<MAXC, TASK, LOGB> l;
};

template <int MAXC, int TASK>
__device__ __forceinline__ void rf_bound_team_body(DataArgs d, LevelArgs lv, ItemArgs it, int64_t bid, int64_t nblk,
                                                   BoundTeamWgLds<MAXC, TASK>& S) {
  constexpr int LOGB = BoundTeamWgLds<MAXC, TASK>::LOGB;
  using LdsT = BoundTeamLds<MAXC, TASK, LOGB>;
  constexpr int IPT = kTeamIpt2;
  constexpr int NB = LdsT::NB, PAIRS = LdsT::PAIRS;
  constexpr int NW = NB / kWave;  // waves with buckets
  resolve_level(lv, d.C);
  resolve_items(it);
  const int split = node_split(it, it.spread / kWaves, it.n_groups);
  const int64_t n_units = it.n_groups * split;
  if (bid >= n_units) return;  // no node for this workgroup
  float* s_tf = S.tf;
  LdsT& L = S.l;
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(t / kWave);
  if (TASK == 0)
    for (int i = t; i < kTfMax; i += kBlock) s_tf[i] = d.Tf[i];
  unsigned long long my_bytes = 0;
  for (int64_t u = bid; u < n_units; u += nblk) {
    const int64_t grp = split > 1 ? (int64_t)((uint32_t)u / (uint32_t)split) : u;
    const int j1 = split > 1 ? (int)((uint32_t)u % (uint32_t)split) : 0;  // the unit's first draw
    const uint32_t o = __builtin_amdgcn_readfirstlane(it.list ? it.list[grp] : (uint32_t)grp);
    const uint32_t i = __builtin_amdgcn_readfirstlane(lv.open_idx[o]);
    const uint32_t tg = (uint32_t)__builtin_amdgcn_readfirstlane(lv.tree_global[lv.tree[i]]);
    const uint32_t nid = __builtin_amdgcn_readfirstlane(lv.id[i]);
    BoundNode nd;
    __syncthreads();  // the previous node's class totals are read no more
    if (bound_node<MAXC, TASK>(d, lv, i, L.ncls, nd)) {  // workgroup-uniform
      if (t == 0 && j1 == 0) bound_pure(d, it, o, tg, nid);
      continue;
    }
    const int m = nd.m;
    uint32_t rows[IPT], kn[IPT];
    BoundPay<TASK, IPT> pay;
    const bool by_row = !it.gk;
    auto entries = [&](auto&& f) { for_entries<IPT, kBlock>(m, f); };
    entries([&](int q, uint32_t e) {
      rows[q] = by_row ? nd.row[e] : e;
      pay.a[q] = nd.aux[e];
      if constexpr (TASK == 1) pay.t[q] = nd.ey[e];
    });
    if constexpr (TASK == 1) {
      double M = 0.0;
      entries([&](int q, uint32_t) { M = fmax(M, fabs((double)(pay.t[q] - nd.mu))); });
#pragma unroll
      for (int off = kWave / 2; off > 0; off >>= 1) M = fmax(M, __shfl_xor(M, off, kWave));
      if (lane == 0) L.eb[wv] = M;
      __syncthreads();
      for (int x = 0; x < kWaves; ++x) M = fmax(M, L.eb[x]);
      nd.M = M * (1.0 + 1e-12);
      nd.E = d.no_bound ? __builtin_inf() : reg_gain_error((double)nd.n, fabs((double)nd.mu) + nd.M);
    }
    float best_score = 0.0f;
    for (int q = 0; q < it.j0; ++q) best_score = fmaxf(best_score, it.res_score[(int64_t)o * it.D + q]);
    double thr = bound_units<TASK>(d, nd, best_score);
    int f_nx = (int)(rand_u32(d.seed, kStreamFeat, tg, nid, (uint64_t)(it.j0 + j1)) % (uint32_t)d.F);
    gather_keys<IPT, kBlock>(draw_base(d, it, f_nx, j1, nd.start), m, rows, kn);
    for (int jj = j1; jj < it.per_group; jj += split) {
      const int j = it.j0 + jj;
      if (it.j0 > 0 && (double)best_score > 1e-3) break;
      const int f = f_nx;
      uint32_t key[IPT];
#pragma unroll
      for (int q = 0; q < IPT; ++q) key[q] = kn[q];
      mask_keys<IPT, kBlock>(m, key);
      if (jj + split < it.per_group) {
        f_nx = (int)(rand_u32(d.seed, kStreamFeat, tg, nid, (uint64_t)(j + split)) % (uint32_t)d.F);
        gather_keys<IPT, kBlock>(draw_base(d, it, f_nx, jj + split, nd.start), m, rows, kn);
      }
      uint32_t kmin = kNone, kmax = 0;
      entries([&](int q, uint32_t) {
        kmin = min(kmin, key[q]);
        kmax = max(kmax, key[q] + 1u);  // kNone wraps to 0
      });
      kmin = wave_min_u32(kmin);
      kmax = wave_max_u32(kmax);
      if (lane == 0) {
        L.w[wv] = kmin;
        L.w2[wv] = kmax;
      }
      if (t == 0) L.sp = 0;
      __syncthreads();
#pragma unroll
      for (int x = 0; x < kWaves; ++x) {
        kmin = min(kmin, L.w[x]);
        kmax = max(kmax, L.w2[x]);
      }
      kmin = __builtin_amdgcn_readfirstlane(kmin);
      kmax = __builtin_amdgcn_readfirstlane(kmax) - 1u;
      DrawBest best{0.0, kNone, kNone};
      uint32_t k0 = kmin;
      int sb = bit_length(kmax - kmin);
      bool more = kmin != kmax;  // one value: no boundary
      while (more) {
        const int shift = max(0, sb - LOGB);
        const uint32_t nbk = 1u << (sb - shift);  // buckets of the range
        // ---- bucket table
        if constexpr (TASK == 0) {
          const int words = (d.C + 1) / 2;
          for (int x = t; x < words * NB; x += kBlock) L.hist[x] = 0;
          if (t < PAIRS) L.below[t] = 0;
        } else {
          for (int x = t; x < NB; x += kBlock) {
            L.hist[x] = 0;
            L.pos[x] = 0;
            L.neg[x] = 0;
          }
          if (t == 0) {
            L.below[0] = 0;
            L.below_s[0] = 0;
          }
        }
        __syncthreads();
        entries([&](int q, uint32_t) {
          const uint32_t b = (key[q] - k0) >> shift;
          const bool in = key[q] >= k0 && b < nbk, lower = key[q] < k0;
          const uint32_t a = pay.a[q];
          const uint32_t w = a & 0xFFFFu;
          if constexpr (TASK == 0) {
            const uint32_t p = a >> 17;                 // class / 2
            const uint32_t v = w << ((a >> 12) & 16u);  // odd class: high half
            if (in) atomicAdd(&L.hist[p * (uint32_t)NB + b], v);
            else if (lower) atomicAdd(&L.below[p], v);
          } else {
            const int64_t dy = pay.t[q] - nd.mu;
            const unsigned long long wy = (unsigned long long)((int64_t)w * dy);
            if (in) {
              atomicAdd(&L.hist[b], w);
              atomicAdd(reinterpret_cast<unsigned long long*>(dy < 0 ? &L.neg[b] : &L.pos[b]), wy);
            } else if (lower) {
              atomicAdd(&L.below[0], w);
              atomicAdd(reinterpret_cast<unsigned long long*>(&L.below_s[0]), wy);
            }
          }
        });
        __syncthreads();
        // ---- edges and bounds of the wave's 64 buckets
        const int b = wv * kWave + lane;
        const bool mine = wv < NW && (uint32_t)(wv * kWave) < nbk;
        double ub = -1.0, eb = 0.0;
        if constexpr (TASK == 0) {
          const bool big_n = nd.n >= kTfMax;
          auto tf = [&](uint32_t x) -> float {
            if (big_n) return x > 1 ? (float)x * __logf((float)x) : 0.0f;
            return s_tf[x];
          };
          const uint32_t n = (uint32_t)nd.n;
          const int words = (d.C + 1) / 2;
          uint32_t inc[PAIRS], sw = 0;
          if (mine) {
#pragma unroll
            for (int p = 0; p < PAIRS; ++p) {
              inc[p] = 0;
              if (p < words) {
                const uint32_t v = L.hist[p * NB + b];
                sw += (v & 0xFFFFu) + (v >> 16);
                inc[p] = wave_incl_scan(v);
                if (lane == kWave - 1) L.tot[wv][p] = inc[p];
              }
            }
            const uint32_t si = wave_incl_scan(sw);
            if (lane == kWave - 1) L.tot_n[wv] = si;
          }
          __syncthreads();
          if (mine) {
            uint32_t run_n = 0;
#pragma unroll
            for (int p = 0; p < PAIRS; ++p)
              if (p < words) {
                const uint32_t bl = L.below[p];
                run_n += (bl & 0xFFFFu) + (bl >> 16);
              }
            for (int x = 0; x < wv; ++x) run_n += L.tot_n[x];
            const uint32_t lb = run_n + wave_incl_scan(sw), la = lb - sw;
            const float psb = tf(lb) + tf(n - lb);
            const float psa = lane_below_f32(psb, tf(run_n) + tf(n - run_n));
            const float slope = sw ? (psb - psa) / (float)sw : 0.0f;
            float phi = 0.0f, slack = 0.0f;
#pragma unroll
            for (int p = 0; p < PAIRS; ++p) {
              if (p < words) {
                uint32_t run = L.below[p];
                for (int x = 0; x < wv; ++x) run += L.tot[x][p];
                const uint32_t v = L.hist[p * NB + b];
                const uint32_t e = run + inc[p];
                const uint32_t n0 = L.ncls[2 * p], n1 = MAXC > 1 ? L.ncls[2 * p + 1] : 0u;
                const uint32_t l0 = e & 0xFFFFu, l1 = e >> 16;
                const float b0 = tf(l0) + tf(n0 - l0), b1 = tf(l1) + tf(n1 - l1);
                const uint32_t r0 = run & 0xFFFFu, r1 = run >> 16;
                const float a0 = lane_below_f32(b0, tf(r0) + tf(n0 - r0));
                const float a1 = lane_below_f32(b1, tf(r1) + tf(n1 - r1));
                phi += a0 + a1;
                slack += fmaxf(0.0f, (b0 - a0) - slope * (float)(v & 0xFFFFu)) +
                         fmaxf(0.0f, (b1 - a1) - slope * (float)(v >> 16));
                L.hist[p * NB + b] = e - v;
              }
            }
            slack += chord_gap_f32((float)la, (float)sw) + chord_gap_f32((float)(n - lb), (float)sw);
            const float edge = nd.Pn + phi - psa;
            float ebf = 0.0f;
            if (sw) {
              if (shift || la > 0) ub = (double)(edge + (shift ? slack : 0.0f) + nd.margin);
              if (la > 0) ebf = fmaxf(0.0f, edge - nd.margin);
            }
            L.wgt[b] = (uint16_t)sw;
            eb = (double)__uint_as_float(wave_max_u32(__float_as_uint(ebf)));
          }
        } else {
          uint32_t w = 0;
          int64_t sp_ = 0, sn_ = 0, si = 0;
          uint32_t wi = 0;
          if (mine) {
            w = L.hist[b];
            sp_ = L.pos[b];
            sn_ = L.neg[b];
            wi = wave_incl_scan(w);
            si = wave_incl_scan_i64(sp_ + sn_);
            if (lane == kWave - 1) {
              L.tot_n[wv] = wi;
              L.tot_s[wv] = si;
            }
          }
          __syncthreads();
          if (mine) {
            uint32_t run_n = L.below[0];
            int64_t run_s = L.below_s[0];
            for (int x = 0; x < wv; ++x) {
              run_n += L.tot_n[x];
              run_s += L.tot_s[x];
            }
            const double N = (double)nd.n, S = (double)(nd.ssum - nd.mu * nd.n);
            const uint32_t lb = run_n + wi, la = lb - w;
            const int64_t sa = run_s + si - (sp_ + sn_);
            L.hist[b] = la;
            L.pos[b] = sa + nd.mu * (int64_t)la;  // uncentred target sum before the bucket
            L.wgt[b] = (uint16_t)w;
            if (w) {
              double edge = 0.0;
              if (la > 0) {
                const double s = (double)sa, q = S - s;
                edge = s * s / (double)la + q * q / (N - (double)la) - S * S / N;
                eb = fmax(0.0, edge * (1.0 - 2e-6) - nd.E);
              }
              if (shift)
                ub = reg_box_bound((double)la, (double)lb, (double)(sa + sn_), (double)(sa + sp_), N, S, nd.M) *
                         (1.0 + 2e-6) + nd.E;
              else if (la > 0)
                ub = edge * (1.0 + 2e-6) + nd.E;
            }
#pragma unroll
            for (int off = kWave / 2; off > 0; off >>= 1) eb = fmax(eb, __shfl_xor(eb, off, kWave));
          }
        }
        if (lane == 0) L.eb[wv] = eb;
        __syncthreads();
#pragma unroll
        for (int x = 0; x < kWaves; ++x) thr = fmax(thr, L.eb[x]);
        const double thr_d = bound_cut<TASK>(d, thr);
        uint64_t mk = __ballot(ub >= thr_d && ub > 0.0);
        // ---- surviving buckets, in rounds of at most kTeamList entries a wave
        for (;;) {
          uint64_t sel = 0;
          uint32_t wsel = 0;
          while (mk) {
            const int x = (int)__ffsll((unsigned long long)mk) - 1;
            const int bx = wv * kWave + x;
            const uint32_t w = __builtin_amdgcn_readfirstlane((uint32_t)L.wgt[bx]);
            if (w > (uint32_t)kBoundRun) {
              // more than a list: a single key has only its edge, a wider
              // bucket is split again
              const uint32_t klo = k0 + ((uint32_t)bx << shift);
              if (!team_splits_again(w, shift)) {
                bound_edge<TASK, LOGB>(d, nd, L, klo, bx, best);
              } else if (lane == 0) {
                const int at = atomicAdd(&L.sp, 1);  // below kTeamStack
                L.stk_k[at] = klo;
                L.stk_b[at] = (uint8_t)shift;
              }
            } else {
              if (wsel + w > (uint32_t)kTeamList) break;
              wsel += w;
              sel |= 1ull << x;
            }
            mk &= mk - 1;
          }
          if (lane == 0) {
            L.mask[wv] = sel;
            L.cnt[wv] = 0;
            L.w[wv] = mk != 0;
          }
          __syncthreads();
          uint64_t any = 0;
          bool left = false;
#pragma unroll
          for (int x = 0; x < NW; ++x) {
            any |= L.mask[x];
            left = left || L.w[x];
          }
          if (any) {  // workgroup-uniform
            entries([&](int q, uint32_t e) {
              const uint32_t bx = (key[q] - k0) >> shift;
              if (key[q] >= k0 && bx < nbk && ((L.mask[bx / kWave] >> (bx & (kWave - 1))) & 1ull)) {
                const unsigned int at = atomicAdd(&L.cnt[bx / kWave], 1u);
                L.lkey[bx / kWave][at] = key[q];
                L.lidx[bx / kWave][at] = (uint16_t)e;
              }
            });
          }
          __syncthreads();
          if (sel) {
            const int nl = (int)L.cnt[wv];
            uint32_t lk[kTeamList / kWave], lx[kTeamList / kWave];
#pragma unroll
            for (int x = 0; x < kTeamList / kWave; ++x) {
              const bool in = lane + x * kWave < nl;
              lk[x] = in ? L.lkey[wv][lane + x * kWave] : 0u;
              lx[x] = in ? L.lidx[wv][lane + x * kWave] : 0u;
            }
            BoundList& W = L.list[wv];
            while (sel) {
              const int x0 = (int)__ffsll((unsigned long long)sel) - 1;
              int x1 = x0;  // last bucket of the run
              const int bx = wv * kWave + x0;
              uint32_t wsum = __builtin_amdgcn_readfirstlane((uint32_t)L.wgt[bx]);
              sel &= sel - 1;
              while (x1 + 1 < kWave && ((sel >> (x1 + 1)) & 1ull)) {
                const uint32_t wn = __builtin_amdgcn_readfirstlane((uint32_t)L.wgt[wv * kWave + x1 + 1]);
                if (wsum + wn > (uint32_t)kWave) break;
                wsum += wn;
                ++x1;
                sel &= sel - 1;
              }
              const uint32_t klo = k0 + ((uint32_t)bx << shift);
              const uint32_t kspan = (uint32_t)(x1 - x0 + 1) << shift;
              int cnt = 0;
#pragma unroll
              for (int x = 0; x < kTeamList / kWave; ++x) {
                const bool in = lane + x * kWave < nl && lk[x] >= klo && lk[x] - klo < kspan;
                const uint64_t bal = __ballot(in);
                const int at = cnt + (int)__popcll(bal & ((1ull << lane) - 1ull));
                if (in) {
                  W.key[at] = lk[x];
                  W.aux[at] = lx[x];
                }
                cnt += (int)__popcll(bal);
              }
              team_sync<kWave>();
              bound_list_payload<TASK>(nd, W, cnt);
              bound_run<TASK, LOGB>(d, nd, L, W, cnt, bx, best);
              team_sync<kWave>();
            }
          }
          __syncthreads();
          if (!left) break;  // workgroup-uniform
        }
        if (best.key != kNone)
          thr = fmax(thr, (TASK == 0 ? best.g * (double)nd.n * kLn2 : best.g) * (1.0 - 1e-6));
        // ---- next range (every thread takes the same one)
        const int sp = L.sp;
        more = sp > 0;
        if (more) {
          k0 = __builtin_amdgcn_readfirstlane(L.stk_k[sp - 1]);
          sb = (int)__builtin_amdgcn_readfirstlane((uint32_t)L.stk_b[sp - 1]);
        }
        __syncthreads();
        if (more && t == 0) L.sp = sp - 1;
      }
      // ---- the draw's best over the waves
      if (lane == 0) L.best[wv] = best;
      __syncthreads();
#pragma unroll
      for (int x = 0; x < kWaves; ++x)
        if (L.best[x].key != kNone && cand_better(L.best[x].g, L.best[x].key, best.g, best.key)) best = L.best[x];
      if (best.prev == kEdge) {  // largest key below the best candidate's
        uint32_t p = 0;
        entries([&](int q, uint32_t) {
          if (key[q] < best.key) p = max(p, key[q]);
        });
        p = wave_max_u32(p);
        if (lane == 0) L.w[wv] = p;
        __syncthreads();
#pragma unroll
        for (int x = 0; x < kWaves; ++x) p = max(p, L.w[x]);
        best.prev = p;
      }
      float score = 0.0f;
      if (best.key != kNone) {
        score = (float)(TASK == 0 ? best.g : ldexp_d(best.g, -2 * d.shift));
        thr = fmax(thr, (TASK == 0 ? best.g * (double)nd.n * kLn2 : best.g) * (1.0 - 1e-6));
      }
      best_score = fmaxf(best_score, score);
      if (t == 0) bound_write<TASK>(d, it, (int64_t)o * it.D + j, f, best, score);
      __syncthreads();  // L.best, L.w are rewritten by the next draw
    }
    if (t == 0 && j1 == 0) my_bytes += (unsigned long long)m * it.per_group * (TASK == 0 ? 12ull : 20ull);
  }
  if (t == 0 && my_bytes && it.bytes) add_bytes(it.bytes, my_bytes);
}
template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock, 3 - TASK) k_search_rf_bound_team(DataArgs d, LevelArgs lv, ItemArgs it) {
  __shared__ BoundTeamWgLds<MAXC, TASK> S;
  rf_bound_team_body<MAXC, TASK>(d, lv, it, blockIdx.x, gridDim.x, S);
}

// Random-forest tiers 0..4 of a phase in one launch.  A small level is bound
// by the latency of its tiers, one launch after the other (35 to 100 us each
// at 4,601 x 57, 100 trees); side by side the level takes as long as its
// slowest tier.  Workgroups go to the tiers by their device counts, the
// largest nodes first, at most cap[k] to a tier (they loop over its nodes);
// the rest of the grid returns at once, which costs 1.5 ns a workgroup: with
// the single tiers' caps, 17 k of them, a level without nodes took 26 us.
struct RfTiers {
  const uint32_t* list[5];
  const unsigned int* n_dev[5];  // counts on the device, or NULL:
  int64_t n[5];
  unsigned long long* bytes[5];
  int cap[5];                    // most blocks of a tier
};

// Blocks that a random-forest tier's units fill: 4 / 2 / 1 / 1 nodes per wave,
// then a node per workgroup.
__host__ __device__ __forceinline__ int64_t rf_tier_blocks(int tier, int64_t nodes, int per_group, int spread) {
  const int per_wg = tier == 0 ? 4 * kWaves : (tier == 1 ? 2 * kWaves : (tier <= 3 ? kWaves : 1));
  const int64_t target = (int64_t)spread / kWaves * per_wg;  // units of node_split
  const int64_t all = nodes * per_group;
  const int64_t units = nodes >= target ? nodes : (all < target ? all : target);
  return (units + per_wg - 1) / per_wg;
}

template <size_t A, size_t B>
constexpr size_t max_size() { return A > B ? A : B; }

template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock, 3 - TASK) k_search_rf_all(DataArgs d, LevelArgs lv, ItemArgs it, RfTiers ts) {
  using Seg = SegLds<TASK>;
  using B1 = BoundWgLds<MAXC, TASK, 1>;
  using B8 = BoundWgLds<MAXC, TASK, 8>;
  using Tm = BoundTeamWgLds<MAXC, TASK>;
  __shared__ __align__(16) unsigned char
      s_raw[max_size<max_size<sizeof(Seg), sizeof(B1)>(), max_size<sizeof(B8), sizeof(Tm)>()>()];
  int64_t bid = blockIdx.x, nblk = 0;
  int tier = 4;
  for (;; --tier) {
    const int64_t n = ts.n_dev[tier] ? (int64_t)*ts.n_dev[tier] : ts.n[tier];
    nblk = rf_tier_blocks(tier, n, it.per_group, it.spread);
    nblk = nblk < ts.cap[tier] ? nblk : ts.cap[tier];
    if (bid < nblk) break;
    bid -= nblk;
    if (tier == 0) return;
  }
  it.list = ts.list[tier];
  it.n_groups = ts.n[tier];
  it.n_dev = ts.n_dev[tier];
  it.bytes = ts.bytes[tier];
  switch (tier) {
    case 0: rf_seg_body<MAXC, TASK, 16>(d, lv, it, bid, nblk, *reinterpret_cast<Seg*>(s_raw)); break;
    case 1: rf_seg_body<MAXC, TASK, 32>(d, lv, it, bid, nblk, *reinterpret_cast<Seg*>(s_raw)); break;
    case 2: rf_bound_body<MAXC, TASK, 1>(d, lv, it, bid, nblk, *reinterpret_cast<B1*>(s_raw)); break;
    case 3: rf_bound_body<MAXC, TASK, 8>(d, lv, it, bid, nblk, *reinterpret_cast<B8*>(s_raw)); break;
    default: rf_bound_team_body<MAXC, TASK>(d, lv, it, bid, nblk, *reinterpret_cast<Tm*>(s_raw)); break;
  }
}

template <int MAXC, int TASK>
void launch_search_rf_all(int64_t grid, hipStream_t s, const DataArgs& d, const LevelArgs& lv, const ItemArgs& it,
                          const RfTiers& ts) {
  hipLaunchKernelGGL((k_search_rf_all<MAXC, TASK>), dim3((unsigned)grid), dim3(kBlock), 0, s, d, lv, it, ts);
}
using RfAllFn = void (*)(int64_t, hipStream_t, const DataArgs&, const LevelArgs&, const ItemArgs&, const RfTiers&);
RfAllFn pick_rf_all(int task, int C) {
  if (task == 1) return launch_search_rf_all<1, 1>;
  if (C <= 2) return launch_search_rf_all<2, 0>;
  if (C <= 4) return launch_search_rf_all<4, 0>;
  if (C <= 8) return launch_search_rf_all<8, 0>;
  if (C <= 16) return launch_search_rf_all<16, 0>;
  return launch_search_rf_all<32, 0>;
}

// ERT, one wave per item (any node size; lanes stride over the entries).
template <int MAXC, int TASK>
__device__ __forceinline__ void ert_wave_body(DataArgs d, LevelArgs lv, ItemArgs it, int64_t bid, int64_t nblk,
                                              double* s_inv, double* s_logc) {
  resolve_level(lv, d.C);
  resolve_items(it);
  if ((int64_t)bid * kWaves >= it.n_groups * it.per_group) return;
  load_ln_table(s_inv, s_logc);
  __syncthreads();
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x / kWave;
  unsigned long long my_bytes = 0;
  const int64_t n_items = it.n_groups * it.per_group;
  for (int64_t item = (int64_t)bid * kWaves + wv; item < n_items; item += (int64_t)nblk * kWaves) {
    const int64_t grp = item / it.per_group;
    const uint32_t o = it.list ? it.list[grp] : (uint32_t)grp;
    const uint32_t i = lv.open_idx[o];
    const int tri = lv.tree[i];
    const DataArgs dd = forest_data(d, tri);
    const int j = item_draw(d, dd, it, (int)(item % it.per_group));
    if (j < 0) continue;  // past this forest's draws (joint build); wave-uniform
    const uint32_t tg = (uint32_t)lv.tree_global[tri];
    const uint32_t nid = lv.id[i];
    const int f = (int)(rand_u32(dd.seed, kStreamFeat, tg, nid, (uint64_t)j) % (uint32_t)dd.F);
    const int m = lv.m[i];
    const int64_t st = lv.start[i];
    const int64_t n = lv.count[i];
    const float* Xf = dd.X + (int64_t)f * dd.N;
    float xs = 0.0f;
    if (lane < 10) {
      const uint32_t pos = rand_u32(dd.seed, kStreamThr, tg, nid, (uint64_t)j * 10 + lane) % (uint32_t)m;
      xs = Xf[lv.row[st + pos]];
    }
    float acc = 0.0f;
    for (int s = 0; s < 10; ++s) acc = acc + __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(xs), s));
    const float thr = acc / 10.0f;
    // Left-side counts.  Extra-trees entries weigh 1 (every row once), so a
    // chunk's class counts are popcounts of ballots: lane c accumulates
    // class c in lc, the left total is wave-uniform in nl_u.  A chunk with
    // another weight takes per-lane accumulators reduced at the end.
    uint32_t loc[MAXC];
#pragma unroll
    for (int c = 0; c < MAXC; ++c) loc[c] = 0;
    uint32_t lc = 0;
    int64_t nl_u = 0, nl_l = 0, sl = 0;
    bool any_loc = false;  // wave-uniform
    walk_entries<TASK, kWave>(lv, st, m, Xf, [&](int, bool in, uint32_t, uint32_t a, float x, int64_t y) {
      const bool left = in && side_of(x, thr) == 0;
      const uint32_t w = a & 0xFFFFu;
      if (TASK == 0) {
        const int lab = (int)(a >> 16);
        if (__ballot(left && w != 1u) == 0) {
          nl_u += __popcll(__ballot(left));
#pragma unroll
          for (int c = 0; c < MAXC; ++c)
            if (c < d.C) {
              const uint32_t cnt = (uint32_t)__popcll(__ballot(left && lab == c));
              if (lane == c) lc += cnt;
            }
        } else {
          any_loc = true;
          if (left) {
            nl_l += w;
#pragma unroll
            for (int c = 0; c < MAXC; ++c) loc[c] += (c == lab) ? w : 0u;
          }
        }
      } else if (left) {
        nl_l += w;
        sl += (int64_t)w * y;
      }
    });
    const int64_t nl = nl_u + ((TASK == 1 || any_loc) ? wave_sum_i64(nl_l) : 0);
    if (lane == 0) my_bytes += (unsigned long long)m * (TASK == 0 ? 12ull : 20ull);
    float score;
    if (nl == 0 || nl == n) {
      score = -FLT_MAX;
    } else if (TASK == 0) {
      // lane c keeps class c's left count
      if (any_loc) {
#pragma unroll
        for (int c = 0; c < MAXC; ++c) {
          uint32_t v = loc[c];
#pragma unroll
          for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
          lc += (lane == c) ? v : 0u;
        }
      }
      const int F = dd.igF;
      const double inv = 1.0 / ((double)n * kLn2);
      int64_t tn = 0, tl = 0, tr = 0;
      if (lane < d.C) {
        const uint32_t nc = lv.cls[(int64_t)i * d.C + lane];
        tn = xlnx_fixed(nc, F, s_inv, s_logc);
        tl = xlnx_fixed(lc, F, s_inv, s_logc);
        tr = xlnx_fixed(nc - lc, F, s_inv, s_logc);
      }
      const int64_t P = xlnx_fixed((uint64_t)n, F, s_inv, s_logc) - wave_sum_i64(tn);
      const int64_t Q = wave_sum_i64(tl + tr) - xlnx_fixed((uint64_t)nl, F, s_inv, s_logc) -
                        xlnx_fixed((uint64_t)(n - nl), F, s_inv, s_logc);
      score = (float)ig_from_fixed(P + Q, F, inv);
    } else {
      sl = wave_sum_i64(sl);
      score = (float)variance_gain(nl, sl, n - nl, lv.sum[i] - sl, dd.shift);
    }
    if (lane == 0) {
      const int64_t ridx = (int64_t)o * it.D + j;
      it.res_score[ridx] = score;
      it.res_thr[ridx] = thr;
      it.res_feat[ridx] = f;
    }
  }
  if (lane == 0 && my_bytes && it.bytes) add_bytes(it.bytes, my_bytes);
}
template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock) k_search_ert_wave(DataArgs d, LevelArgs lv, ItemArgs it) {
  __shared__ double s_inv[128], s_logc[128];
  ert_wave_body<MAXC, TASK>(d, lv, it, blockIdx.x, gridDim.x, s_inv, s_logc);
}

// ERT, one node per SEG-lane segment (nodes of at most SEG entries and at
// most SEG classes; kWave / SEG nodes per wave).  A node's entries sit one
// per lane and stay in registers across its draws: a draw takes its ten
// threshold samples from those lanes by shuffles, so its two gathers (the
// samples and the entries' values of the drawn feature) are independent,
// and the gathers of draw q + 1 are issued before draw q is counted and
// scored.  The draw-independent entropy term of the node is computed once.
// Every draw's (score, threshold, feature) equals k_search_ert_wave's bit
// for bit: the same Philox draws, the same sequential fp32 threshold sum
// (gpuert.cu:167-183), exact integer side counts (gpuert.cu:287-301) or
// target sums (gpuert.cu:348-361) and the same fixed-point entropy sums.
template <int MAXC, int TASK, int SEG>
__device__ __forceinline__ void ert_seg_body(DataArgs d, LevelArgs lv, ItemArgs it, int64_t bid, int64_t nblk,
                                             double* s_inv, double* s_logc) {
  constexpr int NPW = kWave / SEG;  // nodes per wave
  resolve_level(lv, d.C);
  resolve_items(it);
  if ((int64_t)bid * kWaves * NPW >= it.n_groups) return;
  load_ln_table(s_inv, s_logc);
  __syncthreads();
  const int lane = threadIdx.x & (kWave - 1);
  const int sl = lane & (SEG - 1);
  const int base = lane & ~(SEG - 1);
  const unsigned long long segmask = SEG == kWave ? ~0ull : (((1ull << (SEG & 63)) - 1ull) << base);
  unsigned long long my_bytes = 0;
  const int64_t wave_id = (int64_t)bid * kWaves + threadIdx.x / kWave;
  const int64_t n_waves = (int64_t)nblk * kWaves;
  for (int64_t g0 = wave_id * NPW; g0 < it.n_groups; g0 += n_waves * NPW) {
    const int64_t g = g0 + lane / SEG;
    const bool node_ok = g < it.n_groups;
    uint32_t o = 0, i = 0, tg = 0, nid = 0;
    int m = 0;
    int64_t st = 0, n = 0, ssum = 0;
    int tri = 0;
    if (node_ok) {
      o = it.list ? it.list[g] : (uint32_t)g;
      i = lv.open_idx[o];
      tri = lv.tree[i];
      tg = (uint32_t)lv.tree_global[tri];
      nid = lv.id[i];
      m = lv.m[i];
      st = lv.start[i];
      n = lv.count[i];
      if (TASK == 1) ssum = lv.sum[i];
    }
    const DataArgs dd = forest_data(d, tri);
    const bool valid = node_ok && sl < m;
    uint32_t row = 0, a = 0;
    int64_t ey = 0;
    if (valid) {
      row = lv.row[st + sl];
      a = lv.aux[st + sl];
      if (TASK == 1) ey = lv.ey[st + sl];
    }
    const uint32_t w = a & 0xFFFFu;
    const int lab = (int)(a >> 16);
    // Extra-trees entries weigh 1 (every row once): counts are popcounts of
    // ballots.  A wave holding another weight sums weights by shuffles.
    const bool unit_w = __ballot(valid && w != 1u) == 0;  // wave-uniform
    const int F = dd.igF;
    uint32_t nc = 0;
    int64_t P = 0;
    double inv = 0.0;
    if (TASK == 0) {
      if (node_ok && sl < d.C) nc = lv.cls[(int64_t)i * d.C + sl];
      P = xlnx_fixed((uint64_t)n, F, s_inv, s_logc) -
          seg_sum_i64<SEG>(sl < d.C ? xlnx_fixed(nc, F, s_inv, s_logc) : 0);
      inv = 1.0 / ((double)n * kLn2);
    }
    const uint32_t mm = m > 0 ? (uint32_t)m : 1u;
    // The gathers of draw j (< 0: none): the drawn feature, this lane's
    // threshold sample (the first 10 lanes of every row of 16, so that the rows
    // of a segment each sum them) and its entry's value.
    const int rl = lane & 15;
    auto gather = [&](int j, int& f, float& xs, float& xe) {
      const uint32_t jj = j >= 0 ? (uint32_t)j : 0u;
      f = (int)(rand_u32(dd.seed, kStreamFeat, tg, nid, (uint64_t)jj) % (uint32_t)dd.F);
      const uint32_t pos =
          rand_u32(dd.seed, kStreamThr, tg, nid, (uint64_t)jj * 10 + (uint32_t)(rl < 10 ? rl : 0)) % mm;
      const uint32_t rp = (uint32_t)__shfl((int)row, base + (int)pos, kWave);
      const float* Xf = dd.X + (int64_t)f * dd.N;
      xs = (j >= 0 && node_ok && rl < 10) ? Xf[rp] : 0.0f;
      xe = (j >= 0 && valid) ? Xf[row] : 0.0f;
    };
    auto draw_of = [&](int q) { return (node_ok && q < it.per_group) ? item_draw(d, dd, it, q) : -1; };
    int j_c = draw_of(0), f_c = 0;
    float xs_c = 0.0f, xe_c = 0.0f;
    gather(j_c, f_c, xs_c, xe_c);
    for (int q = 0; q < it.per_group; ++q) {
      const int j_n = draw_of(q + 1);
      int f_n = 0;
      float xs_n = 0.0f, xe_n = 0.0f;
      if (q + 1 < it.per_group) gather(j_n, f_n, xs_n, xe_n);
      float acc = 0.0f;
      row_lanes(__float_as_uint(xs_c), [&](int s, uint32_t x) {
        if (s < 10) acc = acc + __uint_as_float(x);
      });
      const float thr = acc / 10.0f;
      const bool left = valid && j_c >= 0 && side_of(xe_c, thr) == 0;
      int64_t nl, sls = 0;
      uint32_t lc = 0;
      if (unit_w) {
        nl = __popcll(__ballot(left) & segmask);
      } else {
        nl = seg_sum_i64<SEG>(left ? (int64_t)w : 0);
      }
      if (TASK == 0) {
#pragma unroll
        for (int c = 0; c < MAXC; ++c)
          if (c < d.C) {
            uint32_t cnt;
            if (unit_w)
              cnt = (uint32_t)__popcll(__ballot(left && lab == c) & segmask);
            else
              cnt = (uint32_t)seg_sum_i64<SEG>((left && lab == c) ? (int64_t)w : 0);
            if (sl == c) lc = cnt;
          }
      } else {
        sls = seg_sum_i64<SEG>(left ? (int64_t)w * ey : 0);
      }
      float score;
      if (TASK == 0) {
        int64_t tl = 0, tr = 0;
        if (sl < d.C) {
          tl = xlnx_fixed(lc, F, s_inv, s_logc);
          tr = xlnx_fixed(nc - lc, F, s_inv, s_logc);
        }
        const int64_t Q = seg_sum_i64<SEG>(tl + tr) - xlnx_fixed((uint64_t)nl, F, s_inv, s_logc) -
                          xlnx_fixed((uint64_t)(n - nl), F, s_inv, s_logc);
        score = (float)ig_from_fixed(P + Q, F, inv);
      } else {
        score = (float)variance_gain(nl, sls, n - nl, ssum - sls, dd.shift);
      }
      if (nl == 0 || nl == n) score = -FLT_MAX;
      if (sl == 0 && j_c >= 0) {
        const int64_t ridx = (int64_t)o * it.D + j_c;
        it.res_score[ridx] = score;
        it.res_thr[ridx] = thr;
        it.res_feat[ridx] = f_c;
        my_bytes += (unsigned long long)m * (TASK == 0 ? 12ull : 20ull);
      }
      j_c = j_n;
      f_c = f_n;
      xs_c = xs_n;
      xe_c = xe_n;
    }
  }
  if (my_bytes && it.bytes) add_bytes(it.bytes, my_bytes);
}
// Four waves per SIMD (128 VGPRs, no spills; three at the unbounded 131).
template <int MAXC, int TASK, int SEG>
__global__ void __launch_bounds__(kBlock, 4) k_search_ert_seg(DataArgs d, LevelArgs lv, ItemArgs it) {
  __shared__ double s_inv[128], s_logc[128];
  ert_seg_body<MAXC, TASK, SEG>(d, lv, it, blockIdx.x, gridDim.x, s_inv, s_logc);
}

// ERT, one wave per node of at most kErtTeamIpt * 64 entries, all draws in
// order.  The node's rows and payloads are read once into registers (slot
// q of lane l holds entry l + 64 q); a draw gathers its feature's values
// of all entries at once, and the next draw's feature, threshold samples
// and gathers are in flight while the current draw is counted and scored.
// Results equal k_search_ert_wave's bit for bit (the same draws, the same
// sequential fp32 threshold sum, exact integer counts and fixed-point
// entropy sums; gpuert.cu:144-230, 287-301, 348-361).
constexpr int kErtTeamIpt = 8;

template <int MAXC, int TASK>
__device__ __forceinline__ void ert_team_body(DataArgs d, LevelArgs lv, ItemArgs it, int64_t bid, int64_t nblk,
                                              double* s_inv, double* s_logc) {
  constexpr int IPT = kErtTeamIpt;
  resolve_level(lv, d.C);
  resolve_items(it);
  if ((int64_t)bid * kWaves >= it.n_groups) return;
  load_ln_table(s_inv, s_logc);
  __syncthreads();
  const int lane = threadIdx.x & (kWave - 1);
  unsigned long long my_bytes = 0;
  const int64_t wave_id = (int64_t)bid * kWaves + threadIdx.x / kWave;
  const int64_t n_waves = (int64_t)nblk * kWaves;
  for (int64_t g = wave_id; g < it.n_groups; g += n_waves) {
    const uint32_t o = it.list ? it.list[g] : (uint32_t)g;
    const uint32_t i = lv.open_idx[o];
    const int tri = lv.tree[i];
    const DataArgs dd = forest_data(d, tri);
    const uint32_t tg = (uint32_t)lv.tree_global[tri];
    const uint32_t nid = lv.id[i];
    const int m = lv.m[i];
    const int64_t st = lv.start[i];
    const int64_t n = lv.count[i];
    const int64_t ssum = TASK == 1 ? lv.sum[i] : 0;
    uint32_t rows[IPT], aux[IPT];
    int64_t eys[IPT];
    bool anyw = false;
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
      const int e = lane + q * kWave;
      rows[q] = 0;
      aux[q] = 0;
      eys[q] = 0;
      if (e < m) {
        rows[q] = lv.row[st + e];
        aux[q] = lv.aux[st + e];
        if (TASK == 1) eys[q] = lv.ey[st + e];
        anyw |= (aux[q] & 0xFFFFu) != 1u;
      }
    }
    // Extra-trees entries weigh 1 (every row once): counts are popcounts of
    // ballots.  A node holding another weight sums weights by shuffles.
    const bool unit_w = __ballot(anyw) == 0;  // wave-uniform
    const int F = dd.igF;
    uint32_t nc = 0;
    int64_t P = 0;
    double inv = 0.0;
    if (TASK == 0) {
      if (lane < d.C) nc = lv.cls[(int64_t)i * d.C + lane];
      P = xlnx_fixed((uint64_t)n, F, s_inv, s_logc) - wave_sum_i64(lane < d.C ? xlnx_fixed(nc, F, s_inv, s_logc) : 0);
      inv = 1.0 / ((double)n * kLn2);
    }
    // Gathers of draw j: the drawn feature, this lane's threshold sample
    // (lanes < 10) and every entry's value.
    auto gather = [&](int j, int& f, float& xs, float* xe) {
      const uint32_t jj = j >= 0 ? (uint32_t)j : 0u;
      f = (int)(rand_u32(dd.seed, kStreamFeat, tg, nid, (uint64_t)jj) % (uint32_t)dd.F);
      const float* Xf = dd.X + (int64_t)f * dd.N;
      xs = 0.0f;
      if (j >= 0 && lane < 10) {
        const uint32_t pos = rand_u32(dd.seed, kStreamThr, tg, nid, (uint64_t)jj * 10 + lane) % (uint32_t)m;
        xs = Xf[lv.row[st + pos]];
      }
#pragma unroll
      for (int q = 0; q < IPT; ++q) xe[q] = (j >= 0 && lane + q * kWave < m) ? Xf[rows[q]] : 0.0f;
    };
    int j_c = item_draw(d, dd, it, 0), f_c = 0;
    float xs_c = 0.0f, xe_c[IPT];
    gather(j_c, f_c, xs_c, xe_c);
    for (int qd = 0; qd < it.per_group; ++qd) {
      const int j_n = qd + 1 < it.per_group ? item_draw(d, dd, it, qd + 1) : -1;
      int f_n = 0;
      float xs_n = 0.0f, xe_n[IPT];
      if (qd + 1 < it.per_group) gather(j_n, f_n, xs_n, xe_n);
      if (j_c >= 0) {  // wave-uniform
        float acc = 0.0f;
        for (int s2 = 0; s2 < 10; ++s2) acc = acc + __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(xs_c), s2));
        const float thr = acc / 10.0f;
        bool left[IPT];
#pragma unroll
        for (int q = 0; q < IPT; ++q) left[q] = lane + q * kWave < m && side_of(xe_c[q], thr) == 0;
        int64_t nl = 0, sls = 0;
        uint32_t lc = 0;
        if (unit_w) {
#pragma unroll
          for (int q = 0; q < IPT; ++q) nl += __popcll(__ballot(left[q]));
        } else {
          int64_t v = 0;
#pragma unroll
          for (int q = 0; q < IPT; ++q) v += left[q] ? (int64_t)(aux[q] & 0xFFFFu) : 0;
          nl = wave_sum_i64(v);
        }
        if (TASK == 0) {
          // one class at a time (lane c keeps class c's left count)
#pragma unroll 1
          for (int c = 0; c < d.C; ++c) {
            uint32_t cnt = 0;
            if (unit_w) {
#pragma unroll
              for (int q = 0; q < IPT; ++q) cnt += (uint32_t)__popcll(__ballot(left[q] && (int)(aux[q] >> 16) == c));
            } else {
              int64_t v = 0;
#pragma unroll
              for (int q = 0; q < IPT; ++q)
                v += (left[q] && (int)(aux[q] >> 16) == c) ? (int64_t)(aux[q] & 0xFFFFu) : 0;
              cnt = (uint32_t)wave_sum_i64(v);
            }
            if (lane == c) lc = cnt;
          }
        } else {
          int64_t v = 0;
#pragma unroll
          for (int q = 0; q < IPT; ++q) v += left[q] ? (int64_t)(aux[q] & 0xFFFFu) * eys[q] : 0;
          sls = wave_sum_i64(v);
        }
        float score;
        if (nl == 0 || nl == n) {
          score = -FLT_MAX;
        } else if (TASK == 0) {
          int64_t tl = 0, tr = 0;
          if (lane < d.C) {
            tl = xlnx_fixed(lc, F, s_inv, s_logc);
            tr = xlnx_fixed(nc - lc, F, s_inv, s_logc);
          }
          const int64_t Q = wave_sum_i64(tl + tr) - xlnx_fixed((uint64_t)nl, F, s_inv, s_logc) -
                            xlnx_fixed((uint64_t)(n - nl), F, s_inv, s_logc);
          score = (float)ig_from_fixed(P + Q, F, inv);
        } else {
          score = (float)variance_gain(nl, sls, n - nl, ssum - sls, dd.shift);
        }
        if (lane == 0) {
          const int64_t ridx = (int64_t)o * it.D + j_c;
          it.res_score[ridx] = score;
          it.res_thr[ridx] = thr;
          it.res_feat[ridx] = f_c;
          my_bytes += (unsigned long long)m * (TASK == 0 ? 12ull : 20ull);
        }
      }
      j_c = j_n;
      f_c = f_n;
      xs_c = xs_n;
#pragma unroll
      for (int q = 0; q < IPT; ++q) xe_c[q] = xe_n[q];
    }
  }
  if (lane == 0 && my_bytes && it.bytes) add_bytes(it.bytes, my_bytes);
}
template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock) k_search_ert_team(DataArgs d, LevelArgs lv, ItemArgs it) {
  __shared__ double s_inv[128], s_logc[128];
  ert_team_body<MAXC, TASK>(d, lv, it, blockIdx.x, gridDim.x, s_inv, s_logc);
}

// All extra-trees tiers of a phase in one launch (each tier exactly as its own
// kernel would run, with its share of the grid; see RfTiers).
constexpr int64_t kMergeEntries = (int64_t)8 << 20;

struct ErtTiers {
  int cap[6];  // most blocks of a tier
  const uint32_t* list[6];
  const unsigned int* n_dev[6];
  unsigned long long* bytes[6];
};

// Three waves per SIMD (168 VGPRs, no spills; two at the unbounded 171).
template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock, 3) k_search_ert_all(DataArgs d, LevelArgs lv, ItemArgs it, ErtTiers ts) {
  __shared__ double s_inv[128], s_logc[128];
  int64_t bid = blockIdx.x, nblk = 0;
  int k = 5;
  for (;; --k) {
    // nodes per block: 16 / 8 / 4 / 4; items per block: 4, 1
    const int64_t n = (int64_t)*ts.n_dev[k] * (k >= 4 ? it.per_group : 1);
    const int per_wg = k == 0 ? 4 * kWaves : (k == 1 ? 2 * kWaves : (k <= 4 ? kWaves : 1));
    nblk = (n + per_wg - 1) / per_wg;
    nblk = nblk < ts.cap[k] ? nblk : ts.cap[k];
    if (bid < nblk) break;
    bid -= nblk;
    if (k == 0) return;
  }
  ItemArgs a = it;
  a.list = ts.list[k];
  a.n_groups = 0;
  a.n_dev = ts.n_dev[k];
  a.bytes = ts.bytes[k];
  switch (k) {
    case 0: ert_seg_body<MAXC, TASK, 16>(d, lv, a, bid, nblk, s_inv, s_logc); break;
    case 1: ert_seg_body<MAXC, TASK, 32>(d, lv, a, bid, nblk, s_inv, s_logc); break;
    case 2: ert_seg_body<MAXC, TASK, 64>(d, lv, a, bid, nblk, s_inv, s_logc); break;
    case 3: ert_team_body<MAXC, TASK>(d, lv, a, bid, nblk, s_inv, s_logc); break;
    case 4: ert_wave_body<MAXC, TASK>(d, lv, a, bid, nblk, s_inv, s_logc); break;
    default: ert_block_body<MAXC, TASK>(d, lv, a, bid, nblk, s_inv, s_logc); break;
  }
}

template <int MAXC, int TASK>
void launch_search_ert_all(int64_t grid, hipStream_t s, const DataArgs& d, const LevelArgs& lv, const ItemArgs& it,
                           const ErtTiers& ts) {
  hipLaunchKernelGGL((k_search_ert_all<MAXC, TASK>), dim3((unsigned)grid), dim3(kBlock), 0, s, d, lv, it, ts);
}
using ErtAllFn = void (*)(int64_t, hipStream_t, const DataArgs&, const LevelArgs&, const ItemArgs&, const ErtTiers&);
ErtAllFn pick_ert_all(int task, int C) {
  if (task == 1) return launch_search_ert_all<1, 1>;
  if (C <= 2) return launch_search_ert_all<2, 0>;
  if (C <= 4) return launch_search_ert_all<4, 0>;
  if (C <= 8) return launch_search_ert_all<8, 0>;
  if (C <= 16) return launch_search_ert_all<16, 0>;
  return launch_search_ert_all<32, 0>;
}

// Split a list of open positions (or all of them) by node size into the
// wave tier and the block tier.  Order inside a tier is irrelevant: every
// item writes its own result slot.
// Tier k holds the groups with cuts[k-1] < m <= cuts[k].
struct Cuts {
  int c[kMaxTiers];  // ascending; the last tier takes everything above
  int n;             // number of tiers
};
struct TierLists {
  uint32_t* l[kMaxTiers];
};

__device__ __forceinline__ int tier_of(int m, const Cuts& cuts) {
  int tier = cuts.n - 1;
#pragma unroll
  for (int k = 0; k < kMaxTiers - 1; ++k)
    if (k < cuts.n - 1 && m <= cuts.c[k]) {
      tier = k;
      break;
    }
  return tier;
}

// Each wave owns a contiguous range of the list: it counts its tiers, the
// workgroup takes one slot range per tier with a single atomic instruction
// (all tiers' counters lie in one line), then the waves write their entries.
// Bound by those atomics, which pass one at a time per line: 1,024 waves with
// an atomic per tier took 85 us for 150 k nodes, 64 workgroups of 16 waves take
// about 10 us.
constexpr int kTierGrid = 64;
constexpr int kTierBlock = 1024;
__global__ void __launch_bounds__(kTierBlock) k_tier_split(const uint32_t* list, int64_t n, const uint32_t* open_idx,
                                                           const int32_t* node_m, Cuts cuts, TierLists out,
                                                           unsigned int* counts) {
  constexpr int NW = kTierBlock / kWave;
  __shared__ unsigned int s_cnt[NW][kMaxTiers], s_base[NW][kMaxTiers];
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x / kWave;
  const int64_t wave = (int64_t)blockIdx.x * NW + wv;
  const int64_t n_waves = (int64_t)gridDim.x * NW;
  const int64_t per = (((n + n_waves - 1) / n_waves) + kWave - 1) & ~(int64_t)(kWave - 1);
  const int64_t lo = wave * per, hi = min(lo + per, n);
  if ((int64_t)blockIdx.x * NW * per >= n) return;  // workgroup-uniform
  unsigned int cnt[kMaxTiers];
#pragma unroll
  for (int k = 0; k < kMaxTiers; ++k) cnt[k] = 0;
  for (int64_t b = lo; b < hi; b += kWave) {
    const int64_t g = b + lane;
    const int tier = g < hi ? tier_of(node_m[open_idx[list ? list[g] : (uint32_t)g]], cuts) : -1;
#pragma unroll
    for (int k = 0; k < kMaxTiers; ++k)
      if (k < cuts.n) cnt[k] += (unsigned int)__popcll(__ballot(tier == k));
  }
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < kMaxTiers; ++k) s_cnt[wv][k] = cnt[k];
  }
  __syncthreads();
  if (threadIdx.x < kMaxTiers) {
    unsigned int sum = 0;
    for (int x = 0; x < NW; ++x) sum += s_cnt[x][threadIdx.x];
    unsigned int base = sum ? atomicAdd(&counts[threadIdx.x], sum) : 0u;
    for (int x = 0; x < NW; ++x) {
      s_base[x][threadIdx.x] = base;
      base += s_cnt[x][threadIdx.x];
    }
  }
  __syncthreads();
  unsigned int base[kMaxTiers];
#pragma unroll
  for (int k = 0; k < kMaxTiers; ++k) base[k] = s_base[wv][k];
  const uint64_t below = (1ull << lane) - 1ull;
  for (int64_t b = lo; b < hi; b += kWave) {
    const int64_t g = b + lane;
    uint32_t o = 0;
    int tier = -1;
    if (g < hi) {
      o = list ? list[g] : (uint32_t)g;
      tier = tier_of(node_m[open_idx[o]], cuts);
    }
#pragma unroll
    for (int k = 0; k < kMaxTiers; ++k) {
      if (k >= cuts.n) break;
      const uint64_t mask = __ballot(tier == k);
      if (tier == k) out.l[k][base[k] + (unsigned int)__popcll(mask & below)] = o;
      base[k] += (unsigned int)__popcll(mask);
    }
  }
}

// ------------------------------------------------------ decide ----------
__device__ __forceinline__ bool split_better(float sa, int fa, float ta, float sb, int fb, float tb) {
  if (sa != sb) return sa > sb;
  if (fa != fb) return fa < fb;
  return ta < tb;
}

// Phase 1: best of the mandatory draws (T1 ties); decide whether the
// retry draws (gpurf.cu:177-182, 242) are needed.  Pure classification
// nodes score 0 on every draw, so their result is the lowest feature index
// among all draws, without evaluating the retries.
struct DecideArgs {
  int64_t n_open;
  int D0, R, D;
  const float* res_score;
  const float* res_thr;
  const int32_t* res_feat;
  float* ch_score;
  float* ch_thr;
  int32_t* ch_feat;
  uint32_t* retry_flag;
  const uint32_t* retry_list;
  int64_t n_retry;
  const unsigned int* n_open_dev;   // device-described level
};

// The best of a node's first draws into ch_*; returns whether it draws retries.
__device__ __forceinline__ bool decide_first(const DataArgs& d, const LevelArgs& lv, const DecideArgs& a, int64_t o,
                                             int algorithm) {
  const float* rs = a.res_score + o * a.D;
  const float* rt = a.res_thr + o * a.D;
  const int32_t* rf = a.res_feat + o * a.D;
  int D0 = a.D0, R = a.R;
  if (d.forests) {  // joint build: the node's own forest's draws
    const DataArgs dd = forest_data(d, lv.tree[lv.open_idx[o]]);
    D0 = dd.D0;
    R = dd.R;
  }
  float bs = rs[0], bt = rt[0];
  int bf = rf[0];
  for (int j = 1; j < D0; ++j)
    if (split_better(rs[j], rf[j], rt[j], bs, bf, bt)) {
      bs = rs[j];
      bf = rf[j];
      bt = rt[j];
    }
  uint32_t need = 0;
  if (R > 0 && (double)bs <= 1e-3) {
    const uint32_t i = lv.open_idx[o];
    bool pure = false;
    if (algorithm == 0 && d.C > 0 && lv.cls) {
      uint32_t mx = 0;
      for (int c = 0; c < d.C; ++c) mx = max(mx, lv.cls[(int64_t)i * d.C + c]);
      pure = (int64_t)mx == (int64_t)lv.count[i];
    }
    if (pure) {
      const uint32_t tg = (uint32_t)lv.tree_global[lv.tree[i]];
      for (int r = 0; r < R; ++r) {
        const int f = (int)(rand_u32(d.seed, kStreamFeat, tg, lv.id[i], (uint64_t)(D0 + r)) % (uint32_t)d.F);
        if (split_better(0.0f, f, 0.0f, bs, bf, bt)) {
          bs = 0.0f;
          bf = f;
          bt = 0.0f;
        }
      }
    } else {
      need = 1;
    }
  }
  a.ch_score[o] = bs;
  a.ch_thr[o] = bt;
  a.ch_feat[o] = bf;
  return need != 0;
}

__global__ void k_decide1(DataArgs d, LevelArgs lv, DecideArgs a, int algorithm) {
  for (int64_t o = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; o < a.n_open;
       o += (int64_t)gridDim.x * blockDim.x)
    a.retry_flag[o] = decide_first(d, lv, a, o, algorithm) ? 1u : 0u;
}

// Phase 2: continue the sequential retry rule on the nodes that needed it.
__device__ __forceinline__ void decide_retry(const DataArgs& d, const LevelArgs& lv, const DecideArgs& a, int64_t o) {
  float bs = a.ch_score[o], bt = a.ch_thr[o];
  int bf = a.ch_feat[o];
  const float* rs = a.res_score + (int64_t)o * a.D;
  const float* rt = a.res_thr + (int64_t)o * a.D;
  const int32_t* rf = a.res_feat + (int64_t)o * a.D;
  int D0 = a.D0, R = a.R;
  if (d.forests) {  // joint build: the node's own forest's draws
    const DataArgs dd = forest_data(d, lv.tree[lv.open_idx[o]]);
    D0 = dd.D0;
    R = dd.R;
  }
  for (int r = 0; r < R; ++r) {
    if ((double)bs > 1e-3) break;
    const int j = D0 + r;
    if (split_better(rs[j], rf[j], rt[j], bs, bf, bt)) {
      bs = rs[j];
      bf = rf[j];
      bt = rt[j];
    }
  }
  a.ch_score[o] = bs;
  a.ch_thr[o] = bt;
  a.ch_feat[o] = bf;
}

__global__ void k_decide2(DataArgs d, LevelArgs lv, DecideArgs a) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < a.n_retry; q += (int64_t)gridDim.x * blockDim.x)
    decide_retry(d, lv, a, a.retry_list[q]);
}

// The same of a device-described level, over the retry flags.
__global__ void k_decide2_dev(DataArgs d, LevelArgs lv, DecideArgs a) {
  resolve_level(lv, d.C);
  const int64_t n = *a.n_open_dev;
  for (int64_t o = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; o < n; o += (int64_t)gridDim.x * blockDim.x)
    if (a.retry_flag[o]) decide_retry(d, lv, a, o);
}

// ------------------------------------------------------ partition -------
// One block per open node: count the left side of the chosen split, then a
// stable two-way compaction into the next entry buffer (FIX of the
// reference's atomic slot order, gpudte.cu:205-232).  Children occupy the
// parent's range: left [start, start+mL), right [start+mL, start+m).
struct PartArgs {
  int64_t n_open;
  const int32_t* ch_feat;
  const float* ch_thr;
  uint32_t* nrow;
  uint32_t* naux;
  int64_t* ney;
  // left child statistics per open node
  int32_t* l_m;
  int32_t* l_count;
  uint32_t* l_cls;
  int64_t* l_sum;
  uint64_t* l_hash;
  uint8_t* split_ok;
  unsigned long long* bytes;
  const uint32_t* list;  // optional: which open positions to process
  const unsigned int* n_dev;  // device-described level: the launch's node count
};

// Side bits of the first pass kept for the scatter pass (nodes of up to
// 64 Ki entries), which then reads no X; with the left entries before each
// word of 64 the scatter needs no scan, no barrier and no order of its own.
// Larger nodes are scattered 64 Ki entries at a time, their sides taken again.
constexpr int kSideWords = 1024;
constexpr int kSideEntries = kSideWords * kWave;

template <int MAXC, int TASK>
__device__ __forceinline__ void part_block_body(DataArgs d, LevelArgs lv, PartArgs pa, int64_t bid, int64_t nblk) {
  resolve_level(lv, d.C);
  if (pa.n_dev) pa.n_open = *pa.n_dev;
  if ((int64_t)bid >= pa.n_open) return;
  __shared__ unsigned long long s_side[kSideWords];
  __shared__ uint32_t s_pre[kSideWords];
  __shared__ uint32_t s_w[kWaves];
  __shared__ uint32_t s_cls[MAXC];
  __shared__ unsigned long long s_cnt, s_sum, s_hash;
  __shared__ uint32_t s_ml;
  const int t = threadIdx.x;
  unsigned long long my_bytes = 0;
  for (int64_t q = bid; q < pa.n_open; q += nblk) {
    const int64_t o = pa.list ? pa.list[q] : q;
    const uint32_t i = lv.open_idx[o];
    const int m = lv.m[i];
    const int64_t st = lv.start[i];
    const int f = pa.ch_feat[o];
    const float thr = pa.ch_thr[o];
    const DataArgs dd = forest_data(d, lv.tree[i]);
    const float* Xf = dd.X + (int64_t)f * dd.N;
    if (t < MAXC) s_cls[t] = 0;
    if (t == 0) {
      s_cnt = 0;
      s_sum = 0;
      s_hash = 0;
      s_ml = 0;
    }
    __syncthreads();
    uint32_t loc[MAXC];
#pragma unroll
    for (int c = 0; c < MAXC; ++c) loc[c] = 0;
    uint64_t cnt = 0, hsh = 0;
    int64_t sm = 0;
    uint32_t ml = 0;
    const bool keep = m <= kSideEntries;
    walk_entries<TASK, kBlock>(lv, st, m, Xf, [&](int e, bool in, uint32_t row, uint32_t a, float x, int64_t y) {
      const bool isl = in && side_of(x, thr) == 0;
      if (keep) {
        const unsigned long long bits = __ballot(isl);
        if ((t & (kWave - 1)) == 0 && in) s_side[e / kWave] = bits;
      }
      const uint32_t w = isl ? a & 0xFFFFu : 0u;
      ml += isl ? 1u : 0u;
      cnt += w;
      hsh += (uint64_t)w * mix64(row);
      if (TASK == 0) {
        const int lab = (int)(a >> 16);
#pragma unroll
        for (int c = 0; c < MAXC; ++c) loc[c] += (c == lab) ? w : 0u;
      } else {
        sm += (int64_t)w * y;
      }
    });
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
      cnt += __shfl_xor(cnt, off, kWave);
      hsh += __shfl_xor(hsh, off, kWave);
      sm += __shfl_xor(sm, off, kWave);
      ml += __shfl_xor(ml, off, kWave);
    }
    if (TASK == 0) {
#pragma unroll
      for (int c = 0; c < MAXC; ++c) {
        uint32_t v = loc[c];
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
        if ((t & (kWave - 1)) == 0 && v) atomicAdd(&s_cls[c], v);
      }
    }
    if ((t & (kWave - 1)) == 0) {
      atomicAdd(&s_cnt, (unsigned long long)cnt);
      atomicAdd(&s_hash, (unsigned long long)hsh);
      atomicAdd(&s_sum, (unsigned long long)sm);
      atomicAdd(&s_ml, ml);
    }
    __syncthreads();
    const int mL = (int)s_ml;
    const bool ok = mL > 0 && mL < m;
    if (t == 0) {
      my_bytes += (unsigned long long)m * (TASK == 0 ? 12ull : 20ull);
      pa.split_ok[o] = ok ? 1 : 0;
      pa.l_m[o] = mL;
      pa.l_count[o] = (int32_t)s_cnt;
      pa.l_hash[o] = (uint64_t)s_hash;
      if (TASK == 1) pa.l_sum[o] = (int64_t)s_sum;
    }
    if (TASK == 0 && t < d.C) pa.l_cls[o * d.C + t] = s_cls[t];
    if (ok) {
      uint32_t lbase = 0;  // left entries before the segment
      for (int s0 = 0; s0 < m; s0 += kSideEntries) {
        const int sm_ = min(m - s0, kSideEntries);
        if (!keep) {
          walk_entries<0, kBlock>(lv, st + s0, sm_, Xf, [&](int e, bool in, uint32_t, uint32_t, float x, int64_t) {
            const unsigned long long bits = __ballot(in && side_of(x, thr) == 0);
            if ((t & (kWave - 1)) == 0 && in) s_side[e / kWave] = bits;
          });
          __syncthreads();
        }
        const int words = (sm_ + kWave - 1) / kWave;
        constexpr int WPT = kSideWords / kBlock;
        uint32_t pc[WPT], mine = 0;
#pragma unroll
        for (int q = 0; q < WPT; ++q) {
          const int x = t * WPT + q;
          pc[q] = x < words ? (uint32_t)__popcll(s_side[x]) : 0u;
          mine += pc[q];
        }
        uint32_t tot;
        uint32_t before = block_excl_scan(mine, s_w, &tot);
#pragma unroll
        for (int q = 0; q < WPT; ++q) {
          s_pre[t * WPT + q] = before;
          before += pc[q];
        }
        __syncthreads();
        const uint32_t rbase = (uint32_t)mL + (uint32_t)s0 - lbase;  // rights before the segment follow every left
        for (int e0 = 0; e0 < sm_; e0 += kBlock * kWalk) {
          uint32_t row[kWalk], aux[kWalk];
          int64_t y[TASK == 1 ? kWalk : 1];
#pragma unroll
          for (int q = 0; q < kWalk; ++q)
            if (e0 + q * kBlock < sm_) {
              const int64_t g = st + s0 + min(e0 + q * kBlock + t, sm_ - 1);
              row[q] = lv.row[g];
              aux[q] = lv.aux[g];
              if constexpr (TASK == 1) y[q] = lv.ey[g];
            }
#pragma unroll
          for (int q = 0; q < kWalk; ++q) {
            const int e = e0 + q * kBlock + t;
            if (e < sm_) {
              const unsigned long long bits = s_side[e / kWave];
              const uint32_t pl = s_pre[e / kWave] + (uint32_t)__popcll(bits & ((1ull << (e & (kWave - 1))) - 1ull));
              const bool isl = (bits >> (e & (kWave - 1))) & 1ull;
              const uint32_t pos = isl ? lbase + pl : rbase + (uint32_t)e - pl;
              pa.nrow[st + pos] = row[q];
              pa.naux[st + pos] = aux[q];
              if constexpr (TASK == 1) pa.ney[st + pos] = y[q];
            }
          }
        }
        lbase += tot;
        __syncthreads();  // s_side, s_pre and s_w are rewritten
      }
    }
    __syncthreads();
  }
  if (t == 0 && my_bytes && pa.bytes) add_bytes(pa.bytes, my_bytes);
}
template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock, 4 - TASK) k_partition(DataArgs d, LevelArgs lv, PartArgs pa) {
  part_block_body<MAXC, TASK>(d, lv, pa, blockIdx.x, gridDim.x);
}

// Nodes above kPartBig entries (the top levels, where a workgroup per node
// leaves most CUs idle): the same stable partition over chunks of
// kPartChunk entries, each chunk a workgroup.
//   1. k_part_chunk_stats    per chunk: left count, left statistics
//                            (atomics into the node's accumulators)
//   2. k_part_chunk_finish   per node: the node's results, left offset of
//                            every chunk (exclusive scan of the chunks'
//                            left counts)
//   3. k_part_chunk_scatter  per chunk: stable two-way compaction at the
//                            chunk's offsets (lefts before it on the left,
//                            rights before it after the node's mL lefts)
// Sums of integers, so the statistics equal k_partition's bit for bit, and
// entries land where k_partition puts them (a stable compaction in place of
// the reference's atomic slot order, gpudte.cu:205-232).
constexpr int kPartBig = 32768;
constexpr int kPartChunk = 8192;

struct PartChunks {
  const uint32_t* list;  // big-node open positions
  int64_t n_nodes;
  const uint32_t* coff;  // first chunk of each big node (n_nodes + 1)
  uint32_t* chunk_ml;    // left entries of each chunk, then their exclusive scan per node
  uint32_t* acc_ml;      // per big node
  unsigned long long* acc_cnt;
  unsigned long long* acc_hash;
  unsigned long long* acc_sum;
  uint32_t* acc_cls;     // [node * C + c]
};

__global__ void k_part_nchunks(const uint32_t* list, int64_t n, const uint32_t* open_idx, const int32_t* node_m,
                               uint32_t* nch) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x)
    nch[q] = (uint32_t)((node_m[open_idx[list[q]]] + kPartChunk - 1) / kPartChunk);
}

// Big node of chunk k: the last q with coff[q] <= k.
__device__ __forceinline__ int64_t part_chunk_node(const PartChunks& pc, int64_t k) {
  int64_t lo = 0, hi = pc.n_nodes - 1;
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) >> 1;
    if ((int64_t)pc.coff[mid] <= k) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock) k_part_chunk_stats(DataArgs d, LevelArgs lv, PartArgs pa, PartChunks pc) {
  __shared__ uint32_t s_cls[MAXC];
  __shared__ unsigned long long s_cnt, s_sum, s_hash;
  __shared__ uint32_t s_ml;
  const int t = threadIdx.x;
  const int64_t k = blockIdx.x;
  const int64_t q = part_chunk_node(pc, k);
  const uint32_t o = pc.list[q];
  const uint32_t i = lv.open_idx[o];
  const int m = lv.m[i];
  const int e0 = (int)(k - pc.coff[q]) * kPartChunk;
  const int e1 = min(m, e0 + kPartChunk);
  const int64_t st = lv.start[i];
  const DataArgs dd = forest_data(d, lv.tree[i]);
  const float* Xf = dd.X + (int64_t)pa.ch_feat[o] * dd.N;
  const float thr = pa.ch_thr[o];
  if (t < MAXC) s_cls[t] = 0;
  if (t == 0) {
    s_cnt = 0;
    s_sum = 0;
    s_hash = 0;
    s_ml = 0;
  }
  __syncthreads();
  uint32_t loc[MAXC];
#pragma unroll
  for (int c = 0; c < MAXC; ++c) loc[c] = 0;
  uint64_t cnt = 0, hsh = 0;
  int64_t sm = 0;
  uint32_t ml = 0;
  for (int e = e0 + t; e < e1; e += kBlock) {
    const uint32_t row = lv.row[st + e];
    const uint32_t a = lv.aux[st + e];
    if (side_of(Xf[row], thr) == 0) {
      const uint32_t w = a & 0xFFFFu;
      ++ml;
      cnt += w;
      hsh += (uint64_t)w * mix64(row);
      if (TASK == 0) {
        const int lab = (int)(a >> 16);
#pragma unroll
        for (int c = 0; c < MAXC; ++c) loc[c] += (c == lab) ? w : 0u;
      } else {
        sm += (int64_t)w * lv.ey[st + e];
      }
    }
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    cnt += __shfl_xor(cnt, off, kWave);
    hsh += __shfl_xor(hsh, off, kWave);
    sm += __shfl_xor(sm, off, kWave);
    ml += __shfl_xor(ml, off, kWave);
  }
  if (TASK == 0) {
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
      uint32_t v = loc[c];
#pragma unroll
      for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
      if ((t & (kWave - 1)) == 0 && v) atomicAdd(&s_cls[c], v);
    }
  }
  if ((t & (kWave - 1)) == 0) {
    atomicAdd(&s_cnt, (unsigned long long)cnt);
    atomicAdd(&s_hash, (unsigned long long)hsh);
    atomicAdd(&s_sum, (unsigned long long)sm);
    atomicAdd(&s_ml, ml);
  }
  __syncthreads();
  if (t == 0) {
    pc.chunk_ml[k] = s_ml;
    if (s_ml) atomicAdd(&pc.acc_ml[q], s_ml);
    if (s_cnt) atomicAdd(&pc.acc_cnt[q], s_cnt);
    if (s_hash) atomicAdd(&pc.acc_hash[q], s_hash);
    if (TASK == 1 && s_sum) atomicAdd(&pc.acc_sum[q], s_sum);
  }
  if (TASK == 0 && t < d.C && s_cls[t]) atomicAdd(&pc.acc_cls[q * d.C + t], s_cls[t]);
}

// One workgroup per big node.
template <int TASK>
__global__ void __launch_bounds__(kBlock) k_part_chunk_finish(DataArgs d, LevelArgs lv, PartArgs pa, PartChunks pc) {
  __shared__ uint32_t s_w[kWaves];
  const int64_t q = blockIdx.x;
  const int t = threadIdx.x;
  const uint32_t o = pc.list[q];
  const uint32_t i = lv.open_idx[o];
  const int m = lv.m[i];
  const int mL = (int)pc.acc_ml[q];
  const bool ok = mL > 0 && mL < m;
  if (t == 0) {
    pa.split_ok[o] = ok ? 1 : 0;
    pa.l_m[o] = mL;
    pa.l_count[o] = (int32_t)pc.acc_cnt[q];
    pa.l_hash[o] = (uint64_t)pc.acc_hash[q];
    if (TASK == 1) pa.l_sum[o] = (int64_t)pc.acc_sum[q];
  }
  if (TASK == 0 && t < d.C) pa.l_cls[(int64_t)o * d.C + t] = pc.acc_cls[q * d.C + t];
  // exclusive scan of the chunks' left counts, in place
  const uint32_t c0 = pc.coff[q], c1 = pc.coff[q + 1];
  uint32_t base = 0;
  for (uint32_t k0 = c0; k0 < c1; k0 += kBlock) {
    const uint32_t k = k0 + t;
    const uint32_t v = k < c1 ? pc.chunk_ml[k] : 0u;
    uint32_t tot;
    const uint32_t ex = block_excl_scan(v, s_w, &tot);
    if (k < c1) pc.chunk_ml[k] = base + ex;
    base += tot;
    __syncthreads();
  }
  if (t == 0 && pa.bytes) add_bytes(pa.bytes, (unsigned long long)m * (TASK == 0 ? 12ull : 20ull));
}

template <int TASK>
__global__ void __launch_bounds__(kBlock) k_part_chunk_scatter(DataArgs d, LevelArgs lv, PartArgs pa, PartChunks pc) {
  __shared__ uint32_t s_w[kWaves];
  const int t = threadIdx.x;
  const int64_t k = blockIdx.x;
  const int64_t q = part_chunk_node(pc, k);
  const uint32_t o = pc.list[q];
  if (!pa.split_ok[o]) return;  // workgroup-uniform
  const uint32_t i = lv.open_idx[o];
  const int m = lv.m[i];
  const int mL = (int)pc.acc_ml[q];
  const int e0 = (int)(k - pc.coff[q]) * kPartChunk;
  const int e1 = min(m, e0 + kPartChunk);
  const int64_t st = lv.start[i];
  const DataArgs dd = forest_data(d, lv.tree[i]);
  const float* Xf = dd.X + (int64_t)pa.ch_feat[o] * dd.N;
  const float thr = pa.ch_thr[o];
  uint32_t lbase = pc.chunk_ml[k];                           // lefts before this chunk
  uint32_t rbase = (uint32_t)mL + (uint32_t)e0 - lbase;      // rights before it follow every left
  for (int b = e0; b < e1; b += kBlock) {
    const int e = b + t;
    uint32_t row = 0, isl = 0;
    if (e < e1) {
      row = lv.row[st + e];
      isl = side_of(Xf[row], thr) == 0 ? 1u : 0u;
    }
    uint32_t tot;
    const uint32_t pl = block_excl_scan(isl, s_w, &tot);
    if (e < e1) {
      const uint32_t pos = isl ? lbase + pl : rbase + (uint32_t)(e - b) - pl;
      pa.nrow[st + pos] = row;
      pa.naux[st + pos] = lv.aux[st + e];
      if (TASK == 1) pa.ney[st + pos] = lv.ey[st + e];
    }
    lbase += tot;
    rbase += (uint32_t)min(kBlock, e1 - b) - tot;
  }
}

// Small nodes: one wave per node; stable compaction with ballots, tile by
// tile (64 entries), statistics reduced across the wave.
template <int MAXC, int TASK>
__device__ __forceinline__ void part_wave_body(DataArgs d, LevelArgs lv, PartArgs pa, const uint32_t* list,
                                               int64_t n_list, int64_t bid, int64_t nblk) {
  resolve_level(lv, d.C);
  if (pa.n_dev) n_list = *pa.n_dev;
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t lt_mask = (1ull << lane) - 1ull;
  unsigned long long my_bytes = 0;
  for (int64_t q = (int64_t)bid * kWaves + threadIdx.x / kWave; q < n_list;
       q += (int64_t)nblk * kWaves) {
    const uint32_t o = list[q];
    const uint32_t i = lv.open_idx[o];
    const int m = lv.m[i];
    const int64_t st = lv.start[i];
    const float thr = pa.ch_thr[o];
    const DataArgs dd = forest_data(d, lv.tree[i]);
    const float* Xf = dd.X + (int64_t)pa.ch_feat[o] * dd.N;
    uint32_t loc[MAXC];
#pragma unroll
    for (int c = 0; c < MAXC; ++c) loc[c] = 0;
    uint64_t cnt = 0, hsh = 0;
    int64_t sm = 0;
    uint32_t ml = 0;
    uint32_t side = 0;  // bit k: entry k * 64 + lane goes left (nodes of up to 2048 entries)
    const bool keep = m <= 32 * kWave;
    walk_entries<TASK, kWave>(lv, st, m, Xf, [&](int e, bool in, uint32_t row, uint32_t a, float x, int64_t y) {
      const bool isl = in && side_of(x, thr) == 0;
      if (isl && keep) side |= 1u << (e / kWave);
      const uint32_t w = isl ? a & 0xFFFFu : 0u;
      cnt += w;
      hsh += (uint64_t)w * mix64(row);
      if (TASK == 0) {
        const int lab = (int)(a >> 16);
#pragma unroll
        for (int c = 0; c < MAXC; ++c) loc[c] += (c == lab) ? w : 0u;
      } else {
        sm += (int64_t)w * y;
      }
      ml += (uint32_t)__popcll(__ballot(isl));
    });
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
      cnt += __shfl_xor(cnt, off, kWave);
      hsh += __shfl_xor(hsh, off, kWave);
      sm += __shfl_xor(sm, off, kWave);
    }
    const int mL = (int)ml;
    const bool ok = mL > 0 && mL < m;
    if (TASK == 0) {
#pragma unroll
      for (int c = 0; c < MAXC; ++c) {
        uint32_t v = loc[c];
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
        if (lane == c && c < d.C) pa.l_cls[(int64_t)o * d.C + c] = v;
      }
    }
    if (lane == 0) {
      my_bytes += (unsigned long long)m * (TASK == 0 ? 12ull : 20ull);
      pa.split_ok[o] = ok ? 1 : 0;
      pa.l_m[o] = mL;
      pa.l_count[o] = (int32_t)cnt;
      pa.l_hash[o] = hsh;
      if (TASK == 1) pa.l_sum[o] = sm;
    }
    if (ok) {
      uint32_t lbase = 0, rbase = (uint32_t)mL;
      for (int e0 = 0; e0 < m; e0 += kWave * kWalk) {
        uint32_t row[kWalk], aux[kWalk];
        int64_t y[TASK == 1 ? kWalk : 1];
#pragma unroll
        for (int q = 0; q < kWalk; ++q)
          if (e0 + q * kWave < m) {
            const int64_t g = st + min(e0 + q * kWave + lane, m - 1);
            row[q] = lv.row[g];
            aux[q] = lv.aux[g];
            if constexpr (TASK == 1) y[q] = lv.ey[g];
          }
#pragma unroll
        for (int q = 0; q < kWalk; ++q)
          if (e0 + q * kWave < m) {
            const int e = e0 + q * kWave + lane;
            bool isl = false;
            if (e < m) isl = keep ? ((side >> (e / kWave)) & 1u) != 0 : side_of(Xf[row[q]], thr) == 0;
            const uint64_t bl = __ballot(isl);
            const uint64_t br = __ballot(e < m && !isl);
            if (e < m) {
              const uint32_t pos =
                  isl ? lbase + (uint32_t)__popcll(bl & lt_mask) : rbase + (uint32_t)__popcll(br & lt_mask);
              pa.nrow[st + pos] = row[q];
              pa.naux[st + pos] = aux[q];
              if constexpr (TASK == 1) pa.ney[st + pos] = y[q];
            }
            lbase += (uint32_t)__popcll(bl);
            rbase += (uint32_t)__popcll(br);
          }
      }
    }
  }
  if (lane == 0 && my_bytes && pa.bytes) add_bytes(pa.bytes, my_bytes);
}
template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock, 5 - TASK) k_partition_wave(DataArgs d, LevelArgs lv, PartArgs pa,
                                                           const uint32_t* list, int64_t n_list) {
  part_wave_body<MAXC, TASK>(d, lv, pa, list, n_list, blockIdx.x, gridDim.x);
}

// Nodes of at most SEG entries: one SEG-lane segment per node, one entry
// per lane, a single pass (side, left statistics, stable positions from the
// segment's ballots).  Same outputs as k_partition_wave.
template <int MAXC, int TASK, int SEG>
__device__ __forceinline__ void part_seg_body(DataArgs d, LevelArgs lv, PartArgs pa, const uint32_t* list,
                                              int64_t n_list, int64_t bid, int64_t nblk) {
  constexpr int NPW = kWave / SEG;
  resolve_level(lv, d.C);
  if (pa.n_dev) n_list = *pa.n_dev;
  __shared__ uint32_t s_cls[kWaves][NPW][TASK == 0 ? MAXC : 1];
  const int lane = threadIdx.x & (kWave - 1);
  const int sl = lane & (SEG - 1);
  const int seg = lane / SEG;
  const int wv = threadIdx.x / kWave;
  const uint64_t seg_mask = (SEG == kWave ? ~0ull : ((1ull << SEG) - 1ull)) << (seg * SEG);
  const uint64_t below = (1ull << lane) - 1ull;
  unsigned long long my_bytes = 0;
  const int64_t wave_id = (int64_t)bid * kWaves + wv;
  const int64_t n_waves = (int64_t)nblk * kWaves;
  for (int64_t q0 = wave_id * NPW; q0 < n_list; q0 += n_waves * NPW) {
    const int64_t q = q0 + seg;
    const bool node_ok = q < n_list;
    uint32_t o = 0;
    int m = 0;
    int64_t st = 0;
    float thr = 0.0f;
    const float* Xf = d.X;
    if (node_ok) {
      o = list[q];
      const uint32_t i = lv.open_idx[o];
      m = lv.m[i];
      st = lv.start[i];
      thr = pa.ch_thr[o];
      if (d.forests) {
        const DataArgs dd = forest_data(d, lv.tree[i]);
        Xf = dd.X + (int64_t)pa.ch_feat[o] * dd.N;
      } else {
        Xf = d.X + (int64_t)pa.ch_feat[o] * d.N;
      }
    }
    const bool valid = node_ok && sl < m;
    uint32_t row = 0, a = 0;
    int64_t ey = 0;
    bool isl = false;
    if (valid) {
      row = lv.row[st + sl];
      a = lv.aux[st + sl];
      if (TASK == 1) ey = lv.ey[st + sl];
      isl = side_of(Xf[row], thr) == 0;
    }
    const uint64_t bl = __ballot(isl) & seg_mask;
    const uint64_t bv = __ballot(valid) & seg_mask;
    const int mL = __popcll(bl);
    const bool ok = mL > 0 && mL < m;
    const uint32_t w = isl ? (a & 0xFFFFu) : 0u;
    const int64_t cnt = seg_sum_i64<SEG>((int64_t)w);
    const int64_t hsh = seg_sum_i64<SEG>(isl ? (int64_t)((uint64_t)w * mix64(row)) : 0);
    const int64_t sm = TASK == 1 ? seg_sum_i64<SEG>(isl ? (int64_t)w * ey : 0) : 0;
    if constexpr (TASK == 0) {
      uint32_t* sc = s_cls[wv][seg];
      for (int c = sl; c < MAXC; c += SEG) sc[c] = 0u;
      team_sync<kWave>();
      if (isl) atomicAdd(&sc[a >> 16], w);
      team_sync<kWave>();
      if (node_ok)
        for (int c = sl; c < d.C; c += SEG) pa.l_cls[(int64_t)o * d.C + c] = sc[c];
      team_sync<kWave>();
    }
    if (node_ok && sl == 0) {
      my_bytes += (unsigned long long)m * (TASK == 0 ? 12ull : 20ull);
      pa.split_ok[o] = ok ? 1 : 0;
      pa.l_m[o] = mL;
      pa.l_count[o] = (int32_t)cnt;
      pa.l_hash[o] = (uint64_t)hsh;
      if (TASK == 1) pa.l_sum[o] = sm;
    }
    if (ok && valid) {
      const uint32_t pos = isl ? (uint32_t)__popcll(bl & below)
                               : (uint32_t)mL + (uint32_t)__popcll(bv & ~bl & below);
      pa.nrow[st + pos] = row;
      pa.naux[st + pos] = a;
      if (TASK == 1) pa.ney[st + pos] = ey;
    }
  }
  if (sl == 0 && my_bytes && pa.bytes) add_bytes(pa.bytes, my_bytes);
}
template <int MAXC, int TASK, int SEG>
__global__ void __launch_bounds__(kBlock) k_partition_seg(DataArgs d, LevelArgs lv, PartArgs pa,
                                                          const uint32_t* list, int64_t n_list) {
  part_seg_body<MAXC, TASK, SEG>(d, lv, pa, list, n_list, blockIdx.x, gridDim.x);
}

// All partition tiers of a level step in one launch (small data, see
// RfTiers): 16-lane segments, 32-lane segments, a wave, a workgroup per node.
struct PartTiers {
  int cap[4];  // most blocks of a tier
  const uint32_t* list[4];
  const unsigned int* n_dev[4];
  int64_t n_bound;  // list capacity (the device counts hold the sizes)
};

template <int MAXC, int TASK>
__global__ void __launch_bounds__(kBlock, 4 - TASK) k_partition_all(DataArgs d, LevelArgs lv, PartArgs pa, PartTiers pt) {
  int64_t bid = blockIdx.x, nblk = 0;
  int k = 3;
  for (;; --k) {
    const int per_wg = k == 0 ? 4 * kWaves : (k == 1 ? 2 * kWaves : (k == 2 ? kWaves : 1));
    nblk = ((int64_t)*pt.n_dev[k] + per_wg - 1) / per_wg;
    nblk = nblk < pt.cap[k] ? nblk : pt.cap[k];
    if (bid < nblk) break;
    bid -= nblk;
    if (k == 0) return;
  }
  pa.n_dev = pt.n_dev[k];
  switch (k) {
    case 0: part_seg_body<MAXC, TASK, 16>(d, lv, pa, pt.list[0], pt.n_bound, bid, nblk); break;
    case 1: part_seg_body<MAXC, TASK, 32>(d, lv, pa, pt.list[1], pt.n_bound, bid, nblk); break;
    case 2: part_wave_body<MAXC, TASK>(d, lv, pa, pt.list[2], pt.n_bound, bid, nblk); break;
    default:
      pa.list = pt.list[3];
      part_block_body<MAXC, TASK>(d, lv, pa, bid, nblk);
      break;
  }
}

template <int MAXC, int TASK>
void launch_partition_all(int64_t grid, hipStream_t s, const DataArgs& d, const LevelArgs& lv, const PartArgs& pa,
                          const PartTiers& pt) {
  hipLaunchKernelGGL((k_partition_all<MAXC, TASK>), dim3((unsigned)grid), dim3(kBlock), 0, s, d, lv, pa, pt);
}
using PartAllFn = void (*)(int64_t, hipStream_t, const DataArgs&, const LevelArgs&, const PartArgs&, const PartTiers&);
PartAllFn pick_part_all(int task, int C) {
  if (task == 1) return launch_partition_all<1, 1>;
  if (C <= 2) return launch_partition_all<2, 0>;
  if (C <= 4) return launch_partition_all<4, 0>;
  if (C <= 8) return launch_partition_all<8, 0>;
  if (C <= 16) return launch_partition_all<16, 0>;
  return launch_partition_all<32, 0>;
}

// ------------------------------------------------------ children --------
struct ChildArgs {
  int64_t n_level;         // nodes at this level
  int64_t off_level;       // level-major offset of this level
  int64_t off_next;        // level-major offset of the next level
  int depth;
  const uint8_t* open;     // per level node
  const uint32_t* open_pos;  // level index -> open position (valid if open)
  const uint8_t* split_ok;   // per open position
  const int32_t* ch_feat;
  const float* ch_thr;
  const float* ch_score;
  const int32_t* l_m;
  const int32_t* l_count;
  const uint32_t* l_cls;
  const int64_t* l_sum;
  const uint64_t* l_hash;
  uint32_t* nchild;        // per level node (scan input)
  const uint32_t* cpos;    // exclusive scan of nchild (n_level + 1)
  const uint32_t* lf;      // first level index of each tree (n_trees + 1)
  const uint32_t* base;    // tree-local id of each tree's first node at this level
  // output arrays (level-major)
  int32_t* o_tree;
  uint32_t* o_id;
  int32_t* o_depth;
  int32_t* o_count;
  int32_t* o_m;
  uint32_t* o_cls;
  int64_t* o_sum;
  uint64_t* o_hash;
  float* o_value;
  int32_t* o_feature;
  float* o_thr;
  float* o_score;
  int64_t* o_left;
  // next level working arrays
  int64_t* n_start;
  uint8_t* n_open;
  const int64_t* start;    // current level starts
  const DevLevel* lvl;     // device-described level: n_level, offsets, depth
};

__device__ __forceinline__ void resolve_children(ChildArgs& a) {
  if (a.lvl) {
    a.n_level = a.lvl->n;
    a.off_level = a.lvl->off;
    a.off_next = a.off_level + a.n_level;
    a.depth = (int)a.lvl->depth;
  }
}

__device__ __forceinline__ uint32_t child_count(const ChildArgs& a, int64_t i) {
  return a.open[i] && a.split_ok[a.open_pos[i]] ? 2u : 0u;
}

__global__ void k_children_count(ChildArgs a) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < a.n_level;
       i += (int64_t)gridDim.x * blockDim.x)
    a.nchild[i] = child_count(a, i);
}

__device__ __forceinline__ void child_write(const DataArgs& d, const ChildArgs& a, int64_t i) {
  const int64_t gi = a.off_level + i;
  if (a.nchild[i] == 0) {
    a.o_feature[gi] = -1;
    a.o_thr[gi] = -1.0f;
    a.o_score[gi] = 0.0f;
    a.o_left[gi] = -1;
    return;
  }
  const uint32_t o = a.open_pos[i];
  const int tr = a.o_tree[gi];
  const DataArgs dd = forest_data(d, tr);
  a.o_feature[gi] = a.ch_feat[o];
  a.o_thr[gi] = a.ch_thr[o];
  a.o_score[gi] = a.ch_score[o];
  const uint32_t p = a.cpos[i];
  const int64_t gl = a.off_next + p;
  a.o_left[gi] = gl;
  const uint32_t first = a.cpos[a.lf[tr]];
  const uint32_t idl = a.base[tr] + (a.lf[tr + 1] - a.lf[tr]) + (p - first);
  const int m = a.o_m[gi];
  const int mL = a.l_m[o];
  const int cnt = a.o_count[gi];
  const int cL = a.l_count[o];
  const int64_t st = a.start[i];
  for (int s = 0; s < 2; ++s) {
    const int64_t g = gl + s;
    a.o_tree[g] = tr;
    a.o_id[g] = idl + s;
    a.o_depth[g] = a.depth + 1;
    const int cm = s == 0 ? mL : m - mL;
    const int cc = s == 0 ? cL : cnt - cL;
    a.o_m[g] = cm;
    a.o_count[g] = cc;
    a.o_hash[g] = s == 0 ? a.l_hash[o] : a.o_hash[gi] - a.l_hash[o];
    if (d.C > 0 && a.o_cls) {
      for (int c = 0; c < d.C; ++c) {
        const uint32_t lc = a.l_cls[(int64_t)o * d.C + c];
        a.o_cls[g * d.C + c] = s == 0 ? lc : a.o_cls[gi * d.C + c] - lc;
      }
      a.o_value[g] = 0.0f;
    } else {
      const int64_t sm = s == 0 ? a.l_sum[o] : a.o_sum[gi] - a.l_sum[o];
      a.o_sum[g] = sm;
      a.o_value[g] = (float)ldexp_d((double)sm / (double)cc, -dd.shift);
    }
    a.n_start[p + s] = s == 0 ? st : st + mL;
    a.n_open[p + s] = (cc > dd.min_node && a.depth + 1 < dd.max_depth) ? 1 : 0;
  }
}

__global__ void k_children_write(DataArgs d, ChildArgs a) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < a.n_level;
       i += (int64_t)gridDim.x * blockDim.x)
    child_write(d, a, i);
}

// Per-tree bookkeeping for the next level: first index and base id.
__global__ void k_tree_update(int n_trees, const uint32_t* cpos, const uint32_t* lf, const uint32_t* base,
                              uint32_t* lf_next, uint32_t* base_next) {
  const int tr = blockIdx.x * blockDim.x + threadIdx.x;
  if (tr > n_trees) return;
  lf_next[tr] = cpos[lf[tr]];
  if (tr < n_trees) base_next[tr] = base[tr] + (lf[tr + 1] - lf[tr]);
}

// ------------------------------------------------------ scans -----------
constexpr int kScanTile = kBlock * 16;

__global__ void k_scan_tiles(const uint32_t* in, int64_t n, uint32_t* tile_sums) {
  __shared__ uint32_t s_w[kWaves];
  const int64_t t0 = (int64_t)blockIdx.x * kScanTile;
  uint32_t s = 0;
  for (int k = 0; k < 16; ++k) {
    const int64_t idx = t0 + (int64_t)threadIdx.x * 16 + k;
    if (idx < n) s += in[idx];
  }
  uint32_t tot;
  block_excl_scan(s, s_w, &tot);
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = tot;
}

__global__ void k_scan_apply(const uint32_t* in, int64_t n, const uint32_t* tile_off, uint32_t* out) {
  __shared__ uint32_t s_w[kWaves];
  const int64_t t0 = (int64_t)blockIdx.x * kScanTile;
  uint32_t v[16];
  uint32_t s = 0;
  for (int k = 0; k < 16; ++k) {
    const int64_t idx = t0 + (int64_t)threadIdx.x * 16 + k;
    v[k] = idx < n ? in[idx] : 0u;
    s += v[k];
  }
  uint32_t base = block_excl_scan(s, s_w, nullptr) + tile_off[blockIdx.x];
  for (int k = 0; k < 16; ++k) {
    const int64_t idx = t0 + (int64_t)threadIdx.x * 16 + k;
    if (idx < n) out[idx] = base;
    base += v[k];
  }
  const int64_t last = (int64_t)gridDim.x * kScanTile;
  (void)last;
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == kBlock - 1) out[n] = base;
}

// ---------------------------------------------------- bootstrap ---------
// Multiplicity of every row in the bootstrap of every tree: draw i of tree t
// is rand(seed, BOOT, t, 0, i) % N (gpurf.cu:101-113 keyed by (tree, i)).
__global__ void k_boot_count(uint32_t* mult, int64_t N, int n_trees, const int32_t* tree_global,
                             uint64_t seed) {
  const int tr = blockIdx.y;
  const uint32_t tg = (uint32_t)tree_global[tr];
  uint32_t* mt = mult + (int64_t)tr * N;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < N; i += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t r = rand_u32(seed, kStreamBoot, tg, 0, (uint64_t)i) % (uint32_t)N;
    atomicAdd(&mt[r], 1u);
  }
  (void)n_trees;
}

__global__ void k_nonzero(const uint32_t* mult, int64_t n, uint32_t* flag) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    flag[i] = mult[i] ? 1u : 0u;
}

// Compact in-bag rows into entries (ascending within each tree) and
// accumulate each root's statistics.  A few workgroups per tree (grid-stride
// over its rows), class counts in per-thread LDS columns: the root's
// counters then take a handful of global atomics per workgroup instead of
// one per row range, and no two lanes add into one LDS word.
constexpr int kBootCompactBlocks = 32;  // workgroups per tree
__global__ void __launch_bounds__(kBlock) k_boot_compact(const uint32_t* mult, const uint32_t* pos, int64_t N,
                                                         const uint32_t* label, const int64_t* yfix, int C,
                                                         uint32_t* row, uint32_t* aux, int64_t* ey,
                                                         uint32_t* root_cls, int64_t* root_sum, uint64_t* root_hash,
                                                         uint32_t* w_max) {
  __shared__ uint32_t s_cls[32 * kBlock];  // [class * kBlock + thread]
  const int tr = blockIdx.y;
  const uint32_t* mt = mult + (int64_t)tr * N;
  const uint32_t* pt = pos + (int64_t)tr * N;
  const int t = threadIdx.x;
  if (!yfix)
    for (int c = 0; c < C; ++c) s_cls[c * kBlock + t] = 0;
  uint64_t hsh = 0;
  int64_t sm = 0;
  uint32_t wm = 0;
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < N; r += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t w = mt[r];
    if (!w) continue;
    wm = max(wm, w);
    const uint32_t p = pt[r];
    const uint32_t lab = label ? label[r] : 0u;
    row[p] = (uint32_t)r;
    aux[p] = (lab << 16) | (w & 0xFFFFu);
    if (yfix) {
      ey[p] = yfix[r];
      sm += (int64_t)w * yfix[r];
    } else {
      s_cls[lab * kBlock + t] += w;
    }
    hsh += (uint64_t)w * mix64((uint64_t)r);
  }
  __syncthreads();
  if (!yfix && t < C) {
    uint32_t v = 0;
    for (int i = 0; i < kBlock; ++i) v += s_cls[t * kBlock + i];
    if (v) atomicAdd(&root_cls[(int64_t)tr * C + t], v);
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    hsh += __shfl_xor(hsh, off, kWave);
    sm += __shfl_xor(sm, off, kWave);
  }
  wm = wave_max_u32(wm);
  if ((threadIdx.x & (kWave - 1)) == 0) {
    // one word for all waves: an atomic each, one after the other, was most of
    // 87 us for 100 trees of 4,601 rows; few raise the maximum
    if (wm > __hip_atomic_load(w_max, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(w_max, wm);
    atomicAdd((unsigned long long*)&root_hash[tr], (unsigned long long)hsh);
    if (yfix) atomicAdd((unsigned long long*)&root_sum[tr], (unsigned long long)sm);
  }
}

// Extra trees: every tree starts from all rows with weight 1 (gpuert.cu:97-102).
__global__ void k_identity_entries(int64_t N, int n_trees, const uint32_t* label, const int64_t* yfix,
                                   uint32_t* row, uint32_t* aux, int64_t* ey) {
  const int tr = blockIdx.y;
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < N; r += (int64_t)gridDim.x * blockDim.x) {
    const int64_t p = (int64_t)tr * N + r;
    row[p] = (uint32_t)r;
    aux[p] = ((label ? label[r] : 0u) << 16) | 1u;
    if (yfix) ey[p] = yfix[r];
  }
  (void)n_trees;
}

__global__ void k_root_stats_identity(int64_t N, const uint32_t* label, const int64_t* yfix, int C,
                                      uint32_t* cls1, int64_t* sum1, uint64_t* hash1) {
  __shared__ uint32_t s_cls[32];  // C <= 32: counted in LDS, one global atomic per class and block
  if (threadIdx.x < 32) s_cls[threadIdx.x] = 0u;
  __syncthreads();
  uint64_t hsh = 0;
  int64_t sm = 0;
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < N; r += (int64_t)gridDim.x * blockDim.x) {
    hsh += mix64((uint64_t)r);
    if (yfix) sm += yfix[r];
    else atomicAdd(&s_cls[label[r]], 1u);
  }
  __syncthreads();
  if (!yfix && (int)threadIdx.x < C && s_cls[threadIdx.x]) atomicAdd(&cls1[threadIdx.x], s_cls[threadIdx.x]);
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    hsh += __shfl_xor(hsh, off, kWave);
    sm += __shfl_xor(sm, off, kWave);
  }
  if ((threadIdx.x & (kWave - 1)) == 0) {
    atomicAdd((unsigned long long*)hash1, (unsigned long long)hsh);
    if (yfix) atomicAdd((unsigned long long*)sum1, (unsigned long long)sm);
  }
}

__global__ void k_canon(float* X, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    if (X[i] == 0.0f) X[i] = 0.0f;
}

// ------------------------------------------------------ finalize --------
struct FinalArgs {
  int64_t n_nodes;
  int C;
  const int32_t* tree;
  const uint32_t* id;
  const int64_t* tree_start;
  const int32_t* feature;
  const float* thr;
  const float* score;
  const int64_t* left;
  const int32_t* depth;
  const int32_t* count;
  const int32_t* m;
  const uint64_t* hash;
  const uint32_t* cls;
  const int64_t* sum;
  const float* value;
  int32_t* f_feature;
  float* f_thr;
  float* f_score;
  int32_t* f_left;
  int32_t* f_depth;
  int32_t* f_count;
  int32_t* f_m;
  uint64_t* f_hash;
  uint32_t* f_cls;
  int64_t* f_sum;
  float* f_value;
};

__global__ void k_finalize(FinalArgs a) {
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < a.n_nodes;
       g += (int64_t)gridDim.x * blockDim.x) {
    const int64_t pos = a.tree_start[a.tree[g]] + a.id[g];
    a.f_feature[pos] = a.feature[g];
    a.f_thr[pos] = a.thr[g];
    a.f_score[pos] = a.score[g];
    const int64_t l = a.left[g];
    a.f_left[pos] = l < 0 ? -1 : (int32_t)(a.tree_start[a.tree[l]] + a.id[l]);
    a.f_depth[pos] = a.depth[g];
    a.f_count[pos] = a.count[g];
    a.f_m[pos] = a.m[g];
    a.f_hash[pos] = a.hash[g];
    if (a.cls)
      for (int c = 0; c < a.C; ++c) a.f_cls[pos * a.C + c] = a.cls[g * a.C + c];
    a.f_sum[pos] = a.sum ? a.sum[g] : 0;
    a.f_value[pos] = a.value[g];
  }
}

// ---------------------------------------- device-described level step --
// Partition tiers: 16- and 32-lane segments, a wave, a workgroup per node.
constexpr Cuts kPartCuts{{16, 32, 512, 0x7FFFFFFF, 0, 0}, 4};

// Exclusive scan of n u32 (n read from the device) into out[0..n], out[n] =
// total, also stored to *total: kDScanBlocks workgroups each own a
// contiguous range (per-range sums; then every range sums the sums before
// it for its offset and is rescanned in tiles of kScanTile).  Two kernels:
// a level step is a chain of short launches, each a fixed latency.
constexpr int kDScanBlocks = 256;

// Sums of a level's open flags.
__global__ void __launch_bounds__(kBlock) k_open_sums(const uint8_t* in, const DevLevel* L, uint32_t* sums) {
  __shared__ uint32_t s_w[kWaves];
  const int64_t n = L->n;
  const int64_t per = (n + kDScanBlocks - 1) / kDScanBlocks;
  const int64_t lo = blockIdx.x * per, hi = min(lo + per, n);
  uint32_t acc = 0;
  for (int64_t i = lo + threadIdx.x; i < hi; i += kBlock) acc += in[i];
  uint32_t tot;
  block_excl_scan(acc, s_w, &tot);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// Children of the level's nodes (2 or 0, kept for the scan) and their sums.
__global__ void __launch_bounds__(kBlock) k_child_sums(ChildArgs a, uint32_t* sums) {
  __shared__ uint32_t s_w[kWaves];
  resolve_children(a);
  const int64_t n = a.n_level;
  const int64_t per = (n + kDScanBlocks - 1) / kDScanBlocks;
  const int64_t lo = blockIdx.x * per, hi = min(lo + per, n);
  uint32_t acc = 0;
  for (int64_t i = lo + threadIdx.x; i < hi; i += kBlock) {
    const uint32_t nc = child_count(a, i);
    a.nchild[i] = nc;
    acc += nc;
  }
  uint32_t tot;
  block_excl_scan(acc, s_w, &tot);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// Sum of the ranges before the workgroup's; the last one stores the total.
__device__ __forceinline__ uint32_t dscan_carry(const uint32_t* sums, uint32_t* s_w, uint32_t* total, uint32_t* out_n) {
  uint32_t part = 0;
  for (int i = threadIdx.x; i < (int)blockIdx.x; i += kBlock) part += sums[i];
  uint32_t carry;
  (void)block_excl_scan(part, s_w, &carry);
  if (blockIdx.x == kDScanBlocks - 1 && threadIdx.x == 0) {
    const uint32_t tot = carry + sums[blockIdx.x];
    if (out_n) *out_n = tot;
    *total = tot;
  }
  return carry;
}

// Exclusive scan of in[lo, hi) from carry, handed over as f(i, in[i], prefix).
template <class In, class F>
__device__ __forceinline__ void dscan_range(const In* in, int64_t lo, int64_t hi, uint32_t carry, uint32_t* s_w, F&& f) {
  for (int64_t t0 = lo; t0 < hi; t0 += kScanTile) {
    uint32_t v[16];
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int64_t idx = t0 + (int64_t)threadIdx.x * 16 + k;
      v[k] = idx < hi ? (uint32_t)in[idx] : 0u;
      sum += v[k];
    }
    uint32_t tile_tot;
    uint32_t base = block_excl_scan(sum, s_w, &tile_tot) + carry;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int64_t idx = t0 + (int64_t)threadIdx.x * 16 + k;
      if (idx < hi) f(idx, v[k], base);
      base += v[k];
    }
    carry += tile_tot;
    __syncthreads();  // s_w is reused by the next tile's scan
  }
}

__global__ void __launch_bounds__(kBlock) k_child_scan(const uint32_t* in, DevLevel* L, const uint32_t* sums,
                                                       uint32_t* out) {
  __shared__ uint32_t s_w[kWaves];
  const int64_t n = L->n;
  const int64_t per = (n + kDScanBlocks - 1) / kDScanBlocks;
  const int64_t lo = blockIdx.x * per, hi = min(lo + per, n);
  const uint32_t carry = dscan_carry(sums, s_w, &L->n_next, out + n);
  __syncthreads();
  dscan_range(in, lo, hi, carry, s_w, [&](int64_t i, uint32_t, uint32_t at) { out[i] = at; });
}

// A level's open nodes: their positions, their list, and the lists of the
// search's and the partition's tiers, in one pass (four launches before, each
// 3 to 12 us however small the level).  A workgroup takes its tiers' slots
// with one atomic instruction (k_tier_split has the reason).
__global__ void __launch_bounds__(kBlock) k_level_lists(const uint8_t* open, DevLevel* L, const uint32_t* sums,
                                                        const int32_t* node_m, uint32_t* open_pos, uint32_t* open_idx,
                                                        Cuts cuts, TierLists out, Cuts pcuts, TierLists pout) {
  __shared__ uint32_t s_w[kWaves];
  __shared__ unsigned int s_tier[2 * kMaxTiers];
  const int t = threadIdx.x;
  const int64_t n = L->n;
  const int64_t per = (n + kDScanBlocks - 1) / kDScanBlocks;
  const int64_t lo = blockIdx.x * per, hi = min(lo + per, n);
  node_m += L->off;
  if (t < 2 * kMaxTiers) s_tier[t] = 0;
  const uint32_t carry = dscan_carry(sums, s_w, &L->n_open, nullptr);
  __syncthreads();
  for (int64_t i = lo + t; i < hi; i += kBlock)
    if (open[i]) {
      const int m = node_m[i];
      atomicAdd(&s_tier[tier_of(m, cuts)], 1u);
      atomicAdd(&s_tier[kMaxTiers + tier_of(m, pcuts)], 1u);
    }
  __syncthreads();
  if (t < 2 * kMaxTiers) {
    const unsigned int c = s_tier[t];
    if (c) s_tier[t] = atomicAdd(t < kMaxTiers ? &L->tier[t] : &L->ptier[t - kMaxTiers], c);
  }
  __syncthreads();
  dscan_range(open, lo, hi, carry, s_w, [&](int64_t i, uint32_t v, uint32_t at) {
    open_pos[i] = at;
    if (v) {
      open_idx[at] = (uint32_t)i;
      const int m = node_m[i];
      const int k = tier_of(m, cuts), pk = tier_of(m, pcuts);
      const unsigned int o = atomicAdd(&s_tier[k], 1u), po = atomicAdd(&s_tier[kMaxTiers + pk], 1u);
      out.l[k][o] = at;
      pout.l[pk][po] = at;
    }
  });
}

// k_decide1 of a device-described level, which also lists the nodes that
// draw retries by search tier.
constexpr int kDecideGrid = 256;
__global__ void __launch_bounds__(kTierBlock) k_decide1_dev(DataArgs d, LevelArgs lv, DecideArgs a, int algorithm,
                                                            Cuts cuts, TierLists out, unsigned int* counts) {
  __shared__ unsigned int s_tier[kMaxTiers];
  resolve_level(lv, d.C);
  const int t = threadIdx.x;
  const int64_t n = *a.n_open_dev;
  const int64_t first = blockIdx.x * (int64_t)kTierBlock + t, step = (int64_t)gridDim.x * kTierBlock;
  if (blockIdx.x * (int64_t)kTierBlock >= n) return;  // workgroup-uniform
  if (t < kMaxTiers) s_tier[t] = 0;
  __syncthreads();
  for (int64_t o = first; o < n; o += step) {
    const bool need = decide_first(d, lv, a, o, algorithm);
    a.retry_flag[o] = need ? 1u : 0u;
    if (need) atomicAdd(&s_tier[tier_of(lv.m[lv.open_idx[o]], cuts)], 1u);
  }
  __syncthreads();
  if (t < kMaxTiers) {
    const unsigned int c = s_tier[t];
    if (c) s_tier[t] = atomicAdd(&counts[t], c);
  }
  __syncthreads();
  for (int64_t o = first; o < n; o += step)
    if (a.retry_flag[o]) {  // this thread's own store
      const int k = tier_of(lv.m[lv.open_idx[o]], cuts);
      out.l[k][atomicAdd(&s_tier[k], 1u)] = (uint32_t)o;
    }
}


// Last kernel of a device level step: the children, the per-tree cursors of
// the next level (k_tree_update's work), and by one thread the next level's
// description with its counters at zero -- a second DevLevel, since every
// workgroup reads the current one.
__global__ void k_children_write_dev(DataArgs d, ChildArgs a, int n_trees, uint32_t* lf_next, uint32_t* base_next,
                                     DevLevel* next) {
  resolve_children(a);
  const int64_t first = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
  if (first == 0) {
    DevLevel n{};
    n.off = a.off_next;
    n.n = a.lvl->n_next;
    n.depth = a.depth + 1;
    *next = n;
  }
  for (int64_t tr = first; tr <= n_trees; tr += step) {
    lf_next[tr] = a.cpos[a.lf[tr]];
    if (tr < n_trees) base_next[tr] = a.base[tr] + (a.lf[tr + 1] - a.lf[tr]);
  }
  for (int64_t i = first; i < a.n_level; i += step) child_write(d, a, i);
}

// ------------------------------------------------------ small helpers ---
__global__ void k_open_flags(const uint8_t* open, int64_t n, uint32_t* flag) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    flag[i] = open[i] ? 1u : 0u;
}

__global__ void k_open_list(const uint8_t* open, const uint32_t* pos, int64_t n, uint32_t* list) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    if (open[i]) list[pos[i]] = (uint32_t)i;
}

__global__ void k_compact_list(const uint32_t* flag, const uint32_t* pos, int64_t n, uint32_t* list) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    if (flag[i]) list[pos[i]] = (uint32_t)i;
}

__global__ void k_add_u64(unsigned long long* p, unsigned long long v) { *p += v; }

__global__ void k_iota(uint32_t* out, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = (uint32_t)i;
}

// Appends one tree batch to the merged canonical arrays: child links and
// tree starts shift by the batch's node offset.
__global__ void k_offset_links(const int32_t* left, int64_t n, int32_t off, int32_t* out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t l = left[i];
    out[i] = l < 0 ? l : l + off;
  }
}
__global__ void k_offset_i64(const int64_t* in, int64_t n, int64_t off, int64_t* out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = in[i] + off;
}

__global__ void k_strided_gather(const uint32_t* in, int64_t stride, int n, uint32_t* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = in[(int64_t)i * stride];
}

// Largest node of a level (out[0]) and the entries of its nodes above
// `cut` entries (out[1]).
__global__ void k_level_sizes(const int32_t* m, int64_t n, int cut, unsigned long long* out) {
  unsigned long long v = 0, big = 0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const unsigned long long x = (unsigned long long)m[i];
    v = max(v, x);
    big += x > (unsigned long long)cut ? x : 0ull;
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    v = max(v, (unsigned long long)__shfl_xor(v, off, kWave));
    big += __shfl_xor(big, off, kWave);
  }
  if ((threadIdx.x & (kWave - 1)) == 0) {
    atomicMax(&out[0], v);
    if (big) atomicAdd(&out[1], big);
  }
}

// ------------------------------------------------------ host side -------
int grid_for(int64_t n, int per_block = kBlock, int cap = 65535 * 4) {
  int64_t g = (n + per_block - 1) / per_block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (int)g;
}

// Exclusive scan of n u32 into out[0..n] (out[n] = total).
void scan_u32(const uint32_t* in, int64_t n, uint32_t* out, hipStream_t s, std::vector<DevBuf<uint32_t>>& tmp,
              int depth = 0) {
  const int64_t tiles = (n + kScanTile - 1) / kScanTile;
  // Sized once: a resize during the recursion would move the buffers that
  // outer levels still reference.
  if (tmp.size() < 16) tmp.resize(16);
  if (depth >= 7) fail(DTE_ERR_INTERNAL, "scan too deep");
  DevBuf<uint32_t>& sums = tmp[2 * depth];
  DevBuf<uint32_t>& offs = tmp[2 * depth + 1];
  sums.reserve((size_t)tiles + 1);
  offs.reserve((size_t)tiles + 1);
  if (n == 0) {
    DTE_HIP(hipMemsetAsync(out, 0, sizeof(uint32_t), s));
    return;
  }
  hipLaunchKernelGGL(k_scan_tiles, dim3((unsigned)tiles), dim3(kBlock), 0, s, in, n, sums.p);
  if (tiles == 1) {
    DTE_HIP(hipMemsetAsync(offs.p, 0, sizeof(uint32_t), s));
  } else {
    scan_u32(sums.p, tiles, offs.p, s, tmp, depth + 1);
  }
  hipLaunchKernelGGL(k_scan_apply, dim3((unsigned)tiles), dim3(kBlock), 0, s, in, n, offs.p, out);
}

template <typename T>
T read_one(const T* p, hipStream_t s) {
  T v;
  DTE_HIP(hipMemcpyAsync(&v, p, sizeof(T), hipMemcpyDeviceToHost, s));
  DTE_HIP(hipStreamSynchronize(s));
  return v;
}


// Profile family of a split-search tier (one kernel per family).
const char* search_family(int algorithm, int tier) {
  static const char* rf[] = {"search_seg16", "search_seg32", "search_seg64", "search_team64", "search_block",
                             "search_chunked", "search_block"};
  static const char* ert[] = {"search_ert_seg16", "search_ert_seg32", "search_ert_seg64", "search_ert_team",
                              "search_ert_wave", "search_ert_block"};
  return algorithm == DTE_RANDOM_FOREST ? rf[tier] : ert[tier];
}

// RF tiers: 0/1 = one 16/32-lane segment per node (one entry per lane, draws
// looped in the kernel); 2/3 = a wave per node, bounded search (1 / 8 entries
// per lane); 4 = a workgroup per node, bounded search; 5 = the chunk pipeline
// (big_pipeline); 6 = a workgroup per item of any size (the plain driver, few
// nodes above cut_block).  ERT tiers: 0/1/2 = one 16/32/64-lane segment per
// node (draws looped in the kernel), 3 = one wave per node (entries in
// registers), 4 = one wave per item, 5 = workgroup per item.
template <int MAXC, int TASK>
void launch_search(int algorithm, int tier, int grid, hipStream_t s, const DataArgs& d, const LevelArgs& lv,
                   const ItemArgs& it) {
  if (algorithm == DTE_RANDOM_FOREST) {
    switch (tier) {
      case 0: hipLaunchKernelGGL((k_search_rf_seg<MAXC, TASK, 16>), dim3(grid), dim3(kBlock), 0, s, d, lv, it); break;
      case 1: hipLaunchKernelGGL((k_search_rf_seg<MAXC, TASK, 32>), dim3(grid), dim3(kBlock), 0, s, d, lv, it); break;
      case 2: hipLaunchKernelGGL((k_search_rf_bound<MAXC, TASK, 1>), dim3(grid), dim3(kBlock), 0, s, d, lv, it); break;
      case 3: hipLaunchKernelGGL((k_search_rf_bound<MAXC, TASK, 8>), dim3(grid), dim3(kBlock), 0, s, d, lv, it); break;
      case 4: hipLaunchKernelGGL((k_search_rf_bound_team<MAXC, TASK>), dim3(grid), dim3(kBlock), 0, s, d, lv, it); break;
      default: hipLaunchKernelGGL((k_search_rf<MAXC, TASK>), dim3(grid), dim3(kBlock), 0, s, d, lv, it); break;
    }
  } else {
    switch (tier) {
      case 0: hipLaunchKernelGGL((k_search_ert_seg<MAXC, TASK, 16>), dim3(grid), dim3(kBlock), 0, s, d, lv, it); break;
      case 1: hipLaunchKernelGGL((k_search_ert_seg<MAXC, TASK, 32>), dim3(grid), dim3(kBlock), 0, s, d, lv, it); break;
      case 2: hipLaunchKernelGGL((k_search_ert_seg<MAXC, TASK, 64>), dim3(grid), dim3(kBlock), 0, s, d, lv, it); break;
      case 3: hipLaunchKernelGGL((k_search_ert_team<MAXC, TASK>), dim3(grid), dim3(kBlock), 0, s, d, lv, it); break;
      case 4: hipLaunchKernelGGL((k_search_ert_wave<MAXC, TASK>), dim3(grid), dim3(kBlock), 0, s, d, lv, it); break;
      default: hipLaunchKernelGGL((k_search_ert<MAXC, TASK>), dim3(grid), dim3(kBlock), 0, s, d, lv, it); break;
    }
  }
}

template <int MAXC, int TASK>
void launch_partition(int grid, hipStream_t s, const DataArgs& d, const LevelArgs& lv, const PartArgs& pa) {
  hipLaunchKernelGGL((k_partition<MAXC, TASK>), dim3(grid), dim3(kBlock), 0, s, d, lv, pa);
}

template <int MAXC, int TASK>
void launch_partition_wave(int grid, hipStream_t s, const DataArgs& d, const LevelArgs& lv, const PartArgs& pa,
                           const uint32_t* list, int64_t n) {
  hipLaunchKernelGGL((k_partition_wave<MAXC, TASK>), dim3(grid), dim3(kBlock), 0, s, d, lv, pa, list, n);
}

// Nodes of at most 16 (32) entries, 4 (2) per wave; the grid covers n nodes.
template <int MAXC, int TASK, int SEG>
void launch_partition_seg(int grid_cap, hipStream_t s, const DataArgs& d, const LevelArgs& lv, const PartArgs& pa,
                          const uint32_t* list, int64_t n) {
  constexpr int per_block = kWaves * (kWave / SEG);
  const int grid = (int)std::min<int64_t>((n + per_block - 1) / per_block, grid_cap);
  hipLaunchKernelGGL((k_partition_seg<MAXC, TASK, SEG>), dim3(grid), dim3(kBlock), 0, s, d, lv, pa, list, n);
}


template <int MAXC, int TASK>
void launch_partition_chunks(hipStream_t s, const DataArgs& d, const LevelArgs& lv, const PartArgs& pa,
                             const PartChunks& pc, int64_t n_chunks) {
  hipLaunchKernelGGL((k_part_chunk_stats<MAXC, TASK>), dim3((unsigned)n_chunks), dim3(kBlock), 0, s, d, lv, pa, pc);
  hipLaunchKernelGGL((k_part_chunk_finish<TASK>), dim3((unsigned)pc.n_nodes), dim3(kBlock), 0, s, d, lv, pa, pc);
  hipLaunchKernelGGL((k_part_chunk_scatter<TASK>), dim3((unsigned)n_chunks), dim3(kBlock), 0, s, d, lv, pa, pc);
}

// Scratch and bookkeeping of the big-node pipeline, reused across levels.
struct BigState {
  DevBuf<V2Item> items;
  DevBuf<V2Tile> htiles;
  DevBuf<uint32_t> bcls, bn, bslot, bnext, bcur, carry_last, res_key, res_prev, isel, nbest;
  DevBuf<int64_t> bpos, bneg;
  DevBuf<float> bub;
  DevBuf<double> res_g;
  DevBuf<uint32_t> skey, saux, skey2, saux2;
  DevBuf<int64_t> sy, sy2;
  DevBuf<V2Task> tasks, spill;
  DevBuf<unsigned int> ctr;
  std::vector<V2Item> host_items;
  std::vector<V2Tile> host_htiles;
  std::vector<int64_t> host_fcount;   // tiles: items per feature
  std::vector<uint32_t> host_forder;  // batch items in feature order
  std::vector<V2Tile> host_forder_tiles;
  int target = kDefBucketTarget;  // bucket_target of the fit
  double max_dev = 0.0;           // regression: largest |fixed target|
};

// Entries per bucket aimed at: a sixth of bucket_target (64 by default).
// Finer buckets give tighter bounds (fewer entries to sort) and larger tables.
constexpr int kV2TargetDiv = 6;

// Chunk-parallel search of the big items of one phase (see k_v2_*): items in
// batches of at most kV2Batch scratch slots (a slot per unit of bootstrap
// weight, the bound of a bucket's entries).  A batch's scratch is four words a
// slot, and two targets for regression, so 1.5 Gi slots (24 or 48 GB) hold most
// of a level of a 200-tree 1M-row fit in one batch.
constexpr int64_t kV2Batch = (int64_t)1536 << 20;
constexpr size_t v2_slot_bytes(int task) { return 4 * sizeof(uint32_t) + (task == 1 ? 2 * sizeof(int64_t) : 0); }

template <int MAXC, int TASK>
void big_pipeline(BigState& B, const DataArgs& d, const LevelArgs& lv, const ItemArgs& it, const uint32_t* groups,
                  int64_t n_groups, hipStream_t s, int num_cu) {
  const int64_t n_all = n_groups * it.per_group;
  if (n_all == 0) return;
  const int C = d.C;
  const int bucket_words = TASK == 0 ? C : kV2RegWords;
  const int nb_cap = std::min(kV2MaxB, kV2HistWords / bucket_words);
  B.items.reserve(n_all);
  B.nbest.reserve(n_groups);
  hipLaunchKernelGGL(k_v2_items, dim3(grid_for(n_all)), dim3(kBlock), 0, s, d, lv, groups, n_groups, it.per_group,
                     it.j0, it.D, nb_cap, std::max(1, B.target / kV2TargetDiv), (const float*)it.res_score, B.nbest.p,
                     B.items.p);
  B.host_items.resize(n_all);
  DTE_HIP(hipMemcpyAsync(B.host_items.data(), B.items.p, sizeof(V2Item) * n_all, hipMemcpyDeviceToHost, s));
  DTE_HIP(hipStreamSynchronize(s));
  int64_t k0 = 0;
  while (k0 < n_all) {
    int64_t k1 = k0, el = 0, slots = 0, nb = 0;
    int nb_max = 0;
    B.host_htiles.clear();
    while (k1 < n_all && (k1 == k0 || slots + B.host_items[k1].n_w <= kV2Batch)) {
      V2Item& bi = B.host_items[k1];
      bi.boff = (int32_t)nb;
      bi.soff = it.gk ? (k1 % it.per_group) * it.gk_stride + bi.start : el;
      el += bi.m;
      slots += bi.n_w;
      nb += bi.nb;
      nb_max = std::max(nb_max, (int)bi.nb);
      ++k1;
    }
    const int64_t n_items = k1 - k0;
    const int tile = (int)std::min<int64_t>(
        kV2TileMax, std::max<int64_t>(kV2Tile, el / ((int64_t)num_cu * 3 * kV2TileRounds) / kBlock * kBlock));
    // Tiles feature-major: the tiles in flight gather from a few feature
    // columns of K at a time instead of from all of them, so the columns stay
    // in the caches.  The results do not depend on the tile order (counts,
    // keys stored per entry).
    B.host_fcount.assign((size_t)d.F + 1, 0);
    for (int64_t k = k0; k < k1; ++k) ++B.host_fcount[(size_t)B.host_items[k].f + 1];
    for (int f = 0; f < d.F; ++f) B.host_fcount[(size_t)f + 1] += B.host_fcount[(size_t)f];
    B.host_forder.resize((size_t)n_items);
    for (int64_t k = k0; k < k1; ++k) B.host_forder[B.host_fcount[(size_t)B.host_items[k].f]++] = (uint32_t)(k - k0);
    if (it.gk) {
      // keys gathered already: a node's draws side by side, which read the
      // same payloads
      for (int64_t g0 = k0, g1; g0 < k1; g0 = g1) {
        for (g1 = g0 + 1; g1 < k1 && B.host_items[g1].grp == B.host_items[g0].grp;) ++g1;
        for (int e0 = 0; e0 < B.host_items[g0].m; e0 += tile)
          for (int64_t k = g0; k < g1; ++k) B.host_forder_tiles.push_back(V2Tile{(uint32_t)(k - k0), (uint32_t)e0});
      }
    } else {
      for (const uint32_t li : B.host_forder)
        for (int e0 = 0; e0 < B.host_items[k0 + li].m; e0 += tile)
          B.host_forder_tiles.push_back(V2Tile{li, (uint32_t)e0});
    }
    {
      // Workgroups go to the 8 XCDs round robin (workgroup w to XCD w % 8),
      // each XCD with its own L2: XCD x takes the x-th eighth of the
      // feature-ordered tiles, so each L2 holds its own few columns.
      const int64_t nt = (int64_t)B.host_forder_tiles.size();
      const int64_t q = (nt + kXcds - 1) / kXcds;
      B.host_htiles.reserve((size_t)nt);
      for (int64_t j = 0; j < q; ++j)
        for (int x = 0; x < kXcds; ++x) {
          const int64_t src = x * q + j;
          if (src < std::min<int64_t>((int64_t)(x + 1) * q, nt)) B.host_htiles.push_back(B.host_forder_tiles[src]);
        }
      B.host_forder_tiles.clear();
    }
    DTE_HIP(hipMemcpyAsync(B.items.p, B.host_items.data() + k0, sizeof(V2Item) * n_items, hipMemcpyHostToDevice, s));
    B.htiles.reserve(B.host_htiles.size());
    DTE_HIP(hipMemcpyAsync(B.htiles.p, B.host_htiles.data(), sizeof(V2Tile) * B.host_htiles.size(),
                           hipMemcpyHostToDevice, s));
    B.bn.reserve(nb);
    B.bub.reserve(nb);
    B.bslot.reserve(nb);
    B.bnext.reserve(nb);
    B.bcur.reserve(nb);
    B.carry_last.reserve(nb);
    B.res_g.reserve(nb);
    B.res_key.reserve(nb);
    B.res_prev.reserve(nb);
    B.tasks.reserve(nb);
    B.spill.reserve(nb);
    B.isel.reserve(n_items);
    B.ctr.reserve(3);
    if (TASK == 0) {
      B.bcls.reserve((size_t)nb * C);
    } else {
      B.bpos.reserve(nb);
      B.bneg.reserve(nb);
    }
    B.skey.reserve(slots);
    B.saux.reserve(slots);
    B.skey2.reserve(slots);
    B.saux2.reserve(slots);
    if (TASK == 1) {
      B.sy.reserve(slots);
      B.sy2.reserve(slots);
    }
    if (TASK == 0) {
      DTE_HIP(hipMemsetAsync(B.bcls.p, 0, 4 * (size_t)nb * C, s));
    } else {
      DTE_HIP(hipMemsetAsync(B.bn.p, 0, 4 * nb, s));
      DTE_HIP(hipMemsetAsync(B.bpos.p, 0, 8 * nb, s));
      DTE_HIP(hipMemsetAsync(B.bneg.p, 0, 8 * nb, s));
    }
    DTE_HIP(hipMemsetAsync(B.ctr.p, 0, 12, s));
    V2Args a{};
    a.items = B.items.p;
    a.n_items = n_items;
    a.tile = tile;
    a.tiles = B.htiles.p;
    a.bcls = B.bcls.p;
    a.bn = B.bn.p;
    a.bpos = B.bpos.p;
    a.bneg = B.bneg.p;
    a.bub = B.bub.p;
    a.nbest = B.nbest.p;
    // Retry draws are taken in order until one scores above 1e-3 (k_decide2):
    // a draw may be dropped for a later one only while it scores at most that.
    a.best_cap = it.j0 > 0 ? 1e-3f : __builtin_inff();
    a.max_dev = B.max_dev;
    a.bslot = B.bslot.p;
    a.bnext = B.bnext.p;
    a.bcur = B.bcur.p;
    a.carry_last = B.carry_last.p;
    a.isel = B.isel.p;
    a.res_g = B.res_g.p;
    a.res_key = B.res_key.p;
    a.res_prev = B.res_prev.p;
    a.gkey = it.gk ? const_cast<uint32_t*>(it.gk) : B.skey2.p;
    a.skey = B.skey.p;
    a.saux = B.saux.p;
    a.sy = B.sy.p;
    a.skey2 = B.skey2.p;
    a.saux2 = B.saux2.p;
    a.sy2 = B.sy2.p;
    a.tasks = B.tasks.p;
    a.spill = B.spill.p;
    a.counters = B.ctr.p;
    const dim3 tiles((unsigned)B.host_htiles.size());
    const dim3 waves((unsigned)((n_items + kWaves - 1) / kWaves));
    {
      // Algorithmic bytes of the batch's items (12 B per entry, 20 B for
      // regression) belong to the kernel that reads every entry.
      Timer tm("chunk_hist", profiling_enabled() ? (double)el * (TASK == 0 ? 12.0 : 20.0) : 0.0, s);
      hipLaunchKernelGGL((it.gk ? k_v2_hist<TASK, true> : k_v2_hist<TASK, false>), tiles, dim3(kBlock), (unsigned)(4 * bucket_words * nb_max), s, d, lv, a);
    }
    {
      Timer tm("chunk_bound", 0.0, s);
      hipLaunchKernelGGL((k_v2_bound<MAXC, TASK>), waves, dim3(kBlock), 0, s, d, lv, a);
      hipLaunchKernelGGL(k_v2_select<TASK>, dim3((unsigned)((n_items + kSelectWaves - 1) / kSelectWaves)),
                         dim3(kSelectWaves * kWave), 0, s, d, a);
    }
    {
      Timer tm("chunk_collect", 0.0, s);
      hipLaunchKernelGGL(k_v2_collect<TASK>, tiles, dim3(kBlock), (unsigned)(9 * nb_max), s, d, lv, a);
    }
    {
      Timer tm("chunk_eval", 0.0, s);
      // at most two full rounds of the three workgroups a CU holds,
      // grid-stride over similar buckets (no partial last round)
      const dim3 grid((unsigned)std::min<int64_t>((nb + kWaves - 1) / kWaves, (int64_t)num_cu * 6));
      if constexpr (TASK == 1)
        hipLaunchKernelGGL((k_v2_eval_reg<MAXC, TASK>), grid, dim3(kBlock), 0, s, d, lv, a);
      else
        hipLaunchKernelGGL((k_v2_eval<MAXC, TASK>), grid, dim3(kBlock), 0, s, d, lv, a);
    }
    {
      Timer tm("chunk_spill", 0.0, s);
      hipLaunchKernelGGL((k_v2_spill<MAXC, TASK>), dim3((unsigned)std::min<int64_t>(nb, (int64_t)num_cu * 4)),
                         dim3(kBlock), 0, s, d, lv, a);
    }
    hipLaunchKernelGGL(k_v2_reduce<TASK>, waves, dim3(kBlock), 0, s, d, a, it);
    if (it.bytes) {
      // algorithmic bytes of the batch: 12 (20) bytes per entry
      const unsigned long long by = (unsigned long long)el * (TASK == 0 ? 12ull : 20ull);
      hipLaunchKernelGGL(k_add_u64, dim3(1), dim3(1), 0, s, it.bytes, by);
    }
    k0 = k1;
    // the host tables are refilled for the next batch
    if (k0 < n_all) DTE_HIP(hipStreamSynchronize(s));
  }
}

using BigFn = void (*)(BigState&, const DataArgs&, const LevelArgs&, const ItemArgs&, const uint32_t*, int64_t,
                       hipStream_t, int);
BigFn pick_big(int task, int C) {
  if (task == 1) return big_pipeline<1, 1>;
  if (C <= 2) return big_pipeline<2, 0>;
  if (C <= 4) return big_pipeline<4, 0>;
  if (C <= 8) return big_pipeline<8, 0>;
  if (C <= 16) return big_pipeline<16, 0>;
  return big_pipeline<32, 0>;
}

using SearchFn = void (*)(int, int, int, hipStream_t, const DataArgs&, const LevelArgs&, const ItemArgs&);
using PartFn = void (*)(int, hipStream_t, const DataArgs&, const LevelArgs&, const PartArgs&);
using PartWaveFn = void (*)(int, hipStream_t, const DataArgs&, const LevelArgs&, const PartArgs&, const uint32_t*,
                            int64_t);

SearchFn pick_search(int task, int C) {
  if (task == 1) return launch_search<1, 1>;
  if (C <= 2) return launch_search<2, 0>;
  if (C <= 4) return launch_search<4, 0>;
  if (C <= 8) return launch_search<8, 0>;
  if (C <= 16) return launch_search<16, 0>;
  return launch_search<32, 0>;
}
template <int SEG>
PartWaveFn pick_part_seg(int task, int C) {
  if (task == 1) return launch_partition_seg<1, 1, SEG>;
  if (C <= 2) return launch_partition_seg<2, 0, SEG>;
  if (C <= 4) return launch_partition_seg<4, 0, SEG>;
  if (C <= 8) return launch_partition_seg<8, 0, SEG>;
  if (C <= 16) return launch_partition_seg<16, 0, SEG>;
  return launch_partition_seg<32, 0, SEG>;
}
using PartChunkFn = void (*)(hipStream_t, const DataArgs&, const LevelArgs&, const PartArgs&, const PartChunks&,
                             int64_t);
PartChunkFn pick_part_chunks(int task, int C) {
  if (task == 1) return launch_partition_chunks<1, 1>;
  if (C <= 2) return launch_partition_chunks<2, 0>;
  if (C <= 4) return launch_partition_chunks<4, 0>;
  if (C <= 8) return launch_partition_chunks<8, 0>;
  if (C <= 16) return launch_partition_chunks<16, 0>;
  return launch_partition_chunks<32, 0>;
}
PartWaveFn pick_part_wave(int task, int C) {
  if (task == 1) return launch_partition_wave<1, 1>;
  if (C <= 2) return launch_partition_wave<2, 0>;
  if (C <= 4) return launch_partition_wave<4, 0>;
  if (C <= 8) return launch_partition_wave<8, 0>;
  if (C <= 16) return launch_partition_wave<16, 0>;
  return launch_partition_wave<32, 0>;
}

PartFn pick_part(int task, int C) {
  if (task == 1) return launch_partition<1, 1>;
  if (C <= 2) return launch_partition<2, 0>;
  if (C <= 4) return launch_partition<4, 0>;
  if (C <= 8) return launch_partition<8, 0>;
  if (C <= 16) return launch_partition<16, 0>;
  return launch_partition<32, 0>;
}

}  // namespace

void scan_u32_ext(const uint32_t* in, int64_t n, uint32_t* out, hipStream_t s,
                  std::vector<DevBuf<uint32_t>>& tmp) {
  scan_u32(in, n, out, s, tmp);
}

void dense_ranks_device(const float* X, int64_t N, int F, DevBuf<uint32_t>& K, DevBuf<float>& SV,
                        DevBuf<int64_t>& SVoff, DevBuf<uint32_t>& S, hipStream_t s,
                        std::vector<DevBuf<uint32_t>>& scan_tmp);

const LnTable& host_ln_table() {
  static LnTable t = [] {
    LnTable x;
    build_ln_table(&x);
    return x;
  }();
  return t;
}

void upload_ln_table(int device) {
  (void)device;
  const LnTable& t = host_ln_table();
  DTE_HIP(hipMemcpyToSymbol(HIP_SYMBOL(g_ln_table), &t, sizeof(LnTable), 0, hipMemcpyHostToDevice));
}

// ------------------------------------------------------------ Builder ---
// Plain launch structure of the reference: at most 100 trees per batch
// (gpudte_algorithm.cc:116-118), at most 512 open nodes per launch chunk
// (gpudte_algorithm.cc:149-151).
constexpr int kPlainTrees = 100;
constexpr int64_t kPlainChunk = 512;

// Largest count with a precomputed x ln x term (512 MB of table).
constexpr int64_t kTMaxCap = (int64_t)1 << 26;

// Largest node a level graph takes (entries): its workgroup-per-item kernel
// needs a scratch slab of this many entries per workgroup.
constexpr int64_t kGraphMaxM = 65536;
constexpr int64_t kGraphSmallM = 8192;
constexpr int64_t kGraphBigWork = (int64_t)2 << 20;

__global__ void k_build_T(int64_t* T, int64_t tmax, int F, float* Tf) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < kTfMax) Tf[t] = (float)xlnx((uint64_t)t, g_ln_table.inv, g_ln_table.logc);
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x <= tmax; x += (int64_t)gridDim.x * blockDim.x)
    T[x] = xlnx_fixed((uint64_t)x, F, g_ln_table.inv, g_ln_table.logc);
}

// Device-resident inputs of one fit, shared by every tree batch.
struct FitData {
  DevBuf<float> X;         // canonical copy (-0 -> +0), feature-major
  DevBuf<uint32_t> label;  // classification
  DevBuf<int64_t> yfix;    // regression: fixed-point targets
  int shift = 0;
  double max_fixed = 0.0;  // regression: largest |fixed-point target|
  DevBuf<uint32_t> K;      // dense ranks (random forest)
  DevBuf<float> SV;
  DevBuf<int64_t> SVoff;
  DevBuf<uint32_t> Sdev;
  DevBuf<int64_t> Ttab;    // fixed-point x ln x terms T[0..Tmax]
  DevBuf<float> Tf;        // x ln x in fp32, x < kTfMax
  DataArgs d{};
};

void prepare_data(FitData& fd, const float* X_dev_in, const float* y_host, int64_t N, int32_t F,
                  const dte_params& p, hipStream_t s) {
  const int task = p.task;
  const int algorithm = p.algorithm;
  const int C = task == 0 ? p.n_classes : 1;
  if (C > 32) fail(DTE_ERR_INVALID_ARGUMENT, "at most 32 classes are supported");
  if (N > (int64_t)0x7FFFFFFF) fail(DTE_ERR_INVALID_ARGUMENT, "too many rows");
  DevBuf<float>& X = fd.X;
  DevBuf<uint32_t>& label = fd.label;
  DevBuf<int64_t>& yfix = fd.yfix;
  int& shift = fd.shift;
  int no_bound = 0;
  DevBuf<uint32_t>& K = fd.K;
  DevBuf<float>& SV = fd.SV;
  DevBuf<int64_t>& SVoff = fd.SVoff;
  DevBuf<uint32_t>& Sdev = fd.Sdev;
  DevBuf<int64_t>& Ttab = fd.Ttab;
  DataArgs& d = fd.d;
  // ---- dataset: canonical copy of X, labels / fixed-point targets.
  X.alloc((size_t)N * F);
  DTE_HIP(hipMemcpyAsync(X.p, X_dev_in, sizeof(float) * N * F, hipMemcpyDeviceToDevice, s));
  hipLaunchKernelGGL(k_canon, dim3(grid_for((int64_t)N * F)), dim3(kBlock), 0, s, X.p, (int64_t)N * F);
  if (task == 0) {
    std::vector<uint32_t> lab(N);
    for (int64_t i = 0; i < N; ++i) {
      const int c = (int)y_host[i];
      if (c < 0 || c >= C || (float)c != y_host[i]) fail(DTE_ERR_INVALID_ARGUMENT, "class label out of range");
      lab[i] = (uint32_t)c;
    }
    label.alloc(N);
    DTE_HIP(hipMemcpyAsync(label.p, lab.data(), 4 * N, hipMemcpyHostToDevice, s));
    DTE_HIP(hipStreamSynchronize(s));
  } else {
    double mx = 0;
    bool finite = true;
    for (int64_t i = 0; i < N; ++i) {
      mx = std::max(mx, std::fabs((double)y_host[i]));
      finite = finite && std::isfinite(y_host[i]);
    }
    no_bound = finite ? 0 : 1;
    shift = fixed_shift(mx, N);
    fd.max_fixed = std::ldexp(mx, shift) + 1.0;
    std::vector<int64_t> yf(N);
    for (int64_t i = 0; i < N; ++i) yf[i] = std::llrint(std::ldexp((double)y_host[i], shift));
    yfix.alloc(N);
    DTE_HIP(hipMemcpyAsync(yfix.p, yf.data(), 8 * N, hipMemcpyHostToDevice, s));
    DTE_HIP(hipStreamSynchronize(s));
  }
  std::vector<DevBuf<uint32_t>> scan_tmp;
  if (algorithm == DTE_RANDOM_FOREST) {
    {
      Timer tm("dense_ranks", 0.0, s);
      dense_ranks_device(X.p, N, F, K, SV, SVoff, Sdev, s, scan_tmp);
    }
    std::vector<uint32_t> Sh(F);
    DTE_HIP(hipMemcpyAsync(Sh.data(), Sdev.p, 4 * F, hipMemcpyDeviceToHost, s));
    DTE_HIP(hipStreamSynchronize(s));
    for (int f = 0; f < F; ++f) {
      int words = task == 0 ? C : 3;
      int wbits = 0;
      while ((1 << (wbits + 1)) * words <= kHistWords) ++wbits;
      while (((Sh[f] + (1u << wbits) - 1) >> wbits) > (uint32_t)kMaxBuckets) ++wbits;
      if ((1 << wbits) * words > kHistWords)
        fail(DTE_ERR_INVALID_ARGUMENT, "too many distinct values in a feature for the split-search buckets");
    }
  }
  d = DataArgs{};
  d.X = X.p;
  d.K = K.p;
  d.SV = SV.p;
  d.SVoff = SVoff.p;
  d.S = Sdev.p;
  d.N = N;
  d.F = F;
  d.C = task == 0 ? C : 0;
  d.shift = shift;
  d.no_bound = no_bound;
  d.seed = p.seed;
  d.min_node = p.min_node_size;
  d.max_depth = p.max_depth;
  {
    const LnTable& lt = host_ln_table();
    d.igF = ig_shift((uint64_t)N, task == 0 ? C : 1, lt.inv, lt.logc);
    // Counts of a fit never exceed the root's total weight N.
    d.Tmax = task == 0 ? std::min<int64_t>(N, kTMaxCap) : 0;
    Ttab.alloc(d.Tmax + 1);
    fd.Tf.alloc(kTfMax);
    hipLaunchKernelGGL(k_build_T, dim3(grid_for(std::max<int64_t>(d.Tmax + 1, kTfMax))), dim3(kBlock), 0, s, Ttab.p,
                       d.Tmax, d.igF, fd.Tf.p);
    d.T = Ttab.p;
    d.Tf = fd.Tf.p;
  }
}

// The arrays of a forest of n_nodes nodes in one allocation, with room for its
// predict records if max_tree, the nodes of its largest tree, is given.
void take_forest(Forest& f, int64_t max_tree) {
  const size_t n = (size_t)f.n_nodes, trees = (size_t)f.n_trees + 1;
  const size_t cls = f.task == 0 ? n * f.n_classes : 1;
  f.slab.alloc(Forest::slab_bytes(8 * trees) + 8 * Forest::slab_bytes(4 * n) + 2 * Forest::slab_bytes(8 * n) +
               Forest::slab_bytes(4 * cls) + (max_tree ? predict_slab_bytes(f, max_tree) : 0));
  f.take(f.tree_start, trees);
  f.take(f.feature, n);
  f.take(f.left, n);
  f.take(f.depth, n);
  f.take(f.count, n);
  f.take(f.n_entries, n);
  f.take(f.threshold, n);
  f.take(f.score, n);
  f.take(f.value, n);
  f.take(f.rowhash, n);
  f.take(f.sum_fixed, n);
  f.take(f.class_counts, cls);
}

// A joint build of several extra-trees forests (dte_fit_many): the trees of
// forest f are batch trees [t0, t0 + T) of one build whose level steps serve
// every forest at once.
struct JointForest {
  FitData* fd;
  int64_t N;
  int32_t F;
  int T;
  int t0;
  dte_params p;
};
struct JointSpec {
  std::vector<JointForest> f;
  DataArgs d;  // joint data: forests / forest_of_tree set, C = joint class width
  int C;       // joint class width (the widest forest's)
  int D0, R;   // the widest mandatory and retry draw counts
  int F;       // the widest feature count
};

// Builds trees [t0, t0 + T) of the fit level by level.  plain = 1 is the
// per-node launch structure of the reference (gpudte_algorithm.cc:116-217):
// open nodes in chunks of at most 512, one workgroup per node walking its
// feature draws in order, a host round trip after every chunk; the same
// device functions compute every result, so both modes give the same bits.
// whole: the trees are a forest of their own (else part of one, without
// predict records).
Forest* fit_batch(FitData& fd, int t0, int T, int64_t N, int32_t F, const dte_params& p, hipStream_t s,
                  bool plain, const JointSpec* J = nullptr, bool whole = true) {
  const auto fit_t0 = std::chrono::steady_clock::now();
  const int task = p.task;
  const int algorithm = p.algorithm;
  const int C = J ? J->C : (task == 0 ? p.n_classes : 1);
  const int k = p.n_features_per_node > 0 ? p.n_features_per_node
                                          : (int)std::round(std::log((double)F)) + 1;
  const int D0 = J ? J->D0 : std::min(k, F);
  const int R = J ? J->R : (k < F ? std::min(10, F - k) : 0);
  const int D = D0 + R;
  const DataArgs d = J ? J->d : fd.d;
  const uint32_t* label = fd.label.p;
  const int64_t* yfix = fd.yfix.p;
  const int shift = fd.shift;
  std::vector<DevBuf<uint32_t>> scan_tmp;
  // per batch tree: rows at its root, forest (joint build), global tree id
  std::vector<int64_t> tN(T, N);
  std::vector<int32_t> tf(T, 0);
  std::vector<int32_t> tg_h(T);
  std::iota(tg_h.begin(), tg_h.end(), t0);
  if (J) {
    for (size_t f = 0; f < J->f.size(); ++f)
      for (int q = 0; q < J->f[f].T; ++q) {
        const int t = J->f[f].t0 + q;
        tN[t] = J->f[f].N;
        tf[t] = (int32_t)f;
        tg_h[t] = J->f[f].p.tree_offset + q;
      }
  }
  auto tree_min_node = [&](int t) { return J ? J->f[tf[t]].p.min_node_size : p.min_node_size; };
  auto tree_max_depth = [&](int t) { return J ? J->f[tf[t]].p.max_depth : p.max_depth; };
  DevBuf<int32_t> tree_global(T);
  DTE_HIP(hipMemcpyAsync(tree_global.p, tg_h.data(), 4 * T, hipMemcpyHostToDevice, s));

  // profile: algorithmic bytes, search (one counter per tier) and partition
  const bool count_bytes = profiling_enabled();
  DevBuf<unsigned long long> byte_counts(count_bytes ? (kMaxTiers + 1) * kByteWords : 1);
  auto tier_bytes = [&](int tier) { return count_bytes ? byte_counts.p + (size_t)tier * kByteWords : nullptr; };
  unsigned long long* const part_bytes = tier_bytes(kMaxTiers);
  if (count_bytes) DTE_HIP(hipMemsetAsync(byte_counts.p, 0, byte_counts.bytes(), s));

  // ---- root entries.
  int64_t E = 0;
  uint32_t w_max = 1;  // largest entry weight
  std::vector<int64_t> root_start(T), root_m(T);
  DevBuf<uint32_t> rowA, auxA, rowB, auxB;
  DevBuf<int64_t> eyA, eyB;
  DevBuf<uint32_t> root_cls((size_t)T * std::max(C, 1));
  DevBuf<int64_t> root_sum(T);
  DevBuf<uint64_t> root_hash(T);
  DTE_HIP(hipMemsetAsync(root_cls.p, 0, root_cls.bytes(), s));
  DTE_HIP(hipMemsetAsync(root_sum.p, 0, root_sum.bytes(), s));
  DTE_HIP(hipMemsetAsync(root_hash.p, 0, root_hash.bytes(), s));
  if (algorithm == DTE_RANDOM_FOREST) {
    const int64_t TN = (int64_t)T * N;
    DevBuf<uint32_t> mult(TN), flag(TN), pos(TN + 1);
    DTE_HIP(hipMemsetAsync(mult.p, 0, mult.bytes(), s));
    {
      Timer tm("bootstrap", 4.0 * TN, s);
      hipLaunchKernelGGL(k_boot_count, dim3(grid_for(N, kBlock, 4096), T), dim3(kBlock), 0, s, mult.p, N, T,
                         tree_global.p, p.seed);
    }
    hipLaunchKernelGGL(k_nonzero, dim3(grid_for(TN)), dim3(kBlock), 0, s, mult.p, TN, flag.p);
    scan_u32(flag.p, TN, pos.p, s, scan_tmp);
    std::vector<uint32_t> starts(T + 1);
    {
      DevBuf<uint32_t> st(T + 1);
      hipLaunchKernelGGL(k_strided_gather, dim3(grid_for(T + 1)), dim3(kBlock), 0, s, pos.p, N, T + 1, st.p);
      DTE_HIP(hipMemcpyAsync(starts.data(), st.p, 4 * (T + 1), hipMemcpyDeviceToHost, s));
      DTE_HIP(hipStreamSynchronize(s));
    }
    E = starts[T];
    for (int t = 0; t < T; ++t) {
      root_start[t] = starts[t];
      root_m[t] = starts[t + 1] - starts[t];
    }
    rowA.alloc(E);
    auxA.alloc(E);
    rowB.alloc(E);
    auxB.alloc(E);
    if (task == 1) {
      eyA.alloc(E);
      eyB.alloc(E);
    }
    DevBuf<uint32_t> w_max_dev(1);
    DTE_HIP(hipMemsetAsync(w_max_dev.p, 0, 4, s));
    hipLaunchKernelGGL(k_boot_compact, dim3(grid_for(N, kBlock, kBootCompactBlocks), T), dim3(kBlock), 0, s, mult.p,
                       pos.p, N,
                       label, yfix, C, rowA.p, auxA.p, eyA.p, root_cls.p, root_sum.p, root_hash.p,
                       w_max_dev.p);
    w_max = read_one(w_max_dev.p, s);
    if (w_max > 0xFFFFu) fail(DTE_ERR_INTERNAL, "bootstrap multiplicity above 65535");
  } else {
    E = 0;
    for (int t = 0; t < T; ++t) {
      root_start[t] = E;
      root_m[t] = tN[t];
      E += tN[t];
    }
    rowA.alloc(E);
    auxA.alloc(E);
    rowB.alloc(E);
    auxB.alloc(E);
    if (task == 1) {
      eyA.alloc(E);
      eyB.alloc(E);
    }
    if (J) {
      // joint build: each forest's trees hold its own rows, entries of the
      // forests one after another
      std::vector<uint32_t> rc((size_t)T * std::max(C, 1), 0u);
      std::vector<int64_t> rs(T, 0);
      std::vector<uint64_t> rh(T, 0);
      DevBuf<uint32_t> c1(std::max(C, 1));
      DevBuf<int64_t> s1(1);
      DevBuf<uint64_t> h1(1);
      for (const JointForest& jf : J->f) {
        const int64_t off = root_start[jf.t0];
        const uint32_t* lab = jf.fd->label.p;
        const int64_t* yf = jf.fd->yfix.p;
        hipLaunchKernelGGL(k_identity_entries, dim3(grid_for(jf.N, kBlock, 4096), jf.T), dim3(kBlock), 0, s, jf.N,
                           jf.T, lab, yf, rowA.p + off, auxA.p + off, task == 1 ? eyA.p + off : nullptr);
        DTE_HIP(hipMemsetAsync(c1.p, 0, c1.bytes(), s));
        DTE_HIP(hipMemsetAsync(s1.p, 0, 8, s));
        DTE_HIP(hipMemsetAsync(h1.p, 0, 8, s));
        hipLaunchKernelGGL(k_root_stats_identity, dim3(grid_for(jf.N, kBlock, 4096)), dim3(kBlock), 0, s, jf.N, lab,
                           yf, C, c1.p, s1.p, h1.p);
        std::vector<uint32_t> c1h(std::max(C, 1));
        int64_t s1h;
        uint64_t h1h;
        DTE_HIP(hipMemcpyAsync(c1h.data(), c1.p, c1.bytes(), hipMemcpyDeviceToHost, s));
        DTE_HIP(hipMemcpyAsync(&s1h, s1.p, 8, hipMemcpyDeviceToHost, s));
        DTE_HIP(hipMemcpyAsync(&h1h, h1.p, 8, hipMemcpyDeviceToHost, s));
        DTE_HIP(hipStreamSynchronize(s));
        for (int q = 0; q < jf.T; ++q) {
          const int t = jf.t0 + q;
          rs[t] = s1h;
          rh[t] = h1h;
          for (int c = 0; c < std::max(C, 1); ++c) rc[(size_t)t * std::max(C, 1) + c] = c1h[c];
        }
      }
      DTE_HIP(hipMemcpyAsync(root_cls.p, rc.data(), 4 * rc.size(), hipMemcpyHostToDevice, s));
      DTE_HIP(hipMemcpyAsync(root_sum.p, rs.data(), 8 * T, hipMemcpyHostToDevice, s));
      DTE_HIP(hipMemcpyAsync(root_hash.p, rh.data(), 8 * T, hipMemcpyHostToDevice, s));
      DTE_HIP(hipStreamSynchronize(s));  // the host vectors above go out of scope
    } else {
    hipLaunchKernelGGL(k_identity_entries, dim3(grid_for(N, kBlock, 4096), T), dim3(kBlock), 0, s, N, T, label,
                       yfix, rowA.p, auxA.p, eyA.p);
    DevBuf<uint32_t> c1(std::max(C, 1));
    DevBuf<int64_t> s1(1);
    DevBuf<uint64_t> h1(1);
    DTE_HIP(hipMemsetAsync(c1.p, 0, c1.bytes(), s));
    DTE_HIP(hipMemsetAsync(s1.p, 0, 8, s));
    DTE_HIP(hipMemsetAsync(h1.p, 0, 8, s));
    hipLaunchKernelGGL(k_root_stats_identity, dim3(grid_for(N, kBlock, 4096)), dim3(kBlock), 0, s, N, label,
                       yfix, C, c1.p, s1.p, h1.p);
    std::vector<uint32_t> c1h(std::max(C, 1));
    int64_t s1h;
    uint64_t h1h;
    DTE_HIP(hipMemcpyAsync(c1h.data(), c1.p, c1.bytes(), hipMemcpyDeviceToHost, s));
    DTE_HIP(hipMemcpyAsync(&s1h, s1.p, 8, hipMemcpyDeviceToHost, s));
    DTE_HIP(hipMemcpyAsync(&h1h, h1.p, 8, hipMemcpyDeviceToHost, s));
    DTE_HIP(hipStreamSynchronize(s));
    std::vector<uint32_t> rc((size_t)T * std::max(C, 1));
    std::vector<int64_t> rs(T, s1h);
    std::vector<uint64_t> rh(T, h1h);
    for (int t = 0; t < T; ++t)
      for (int c = 0; c < std::max(C, 1); ++c) rc[(size_t)t * std::max(C, 1) + c] = c1h[c];
    DTE_HIP(hipMemcpyAsync(root_cls.p, rc.data(), 4 * rc.size(), hipMemcpyHostToDevice, s));
    DTE_HIP(hipMemcpyAsync(root_sum.p, rs.data(), 8 * T, hipMemcpyHostToDevice, s));
    DTE_HIP(hipMemcpyAsync(root_hash.p, rh.data(), 8 * T, hipMemcpyHostToDevice, s));
    }
  }

  // ---- level-major node arrays (capacity: a tree has at most 2m-1 nodes).
  const int64_t cap = 2 * E + T;
  DevBuf<int32_t> o_tree(cap), o_depth(cap), o_count(cap), o_m(cap), o_feature(cap);
  DevBuf<uint32_t> o_id(cap);
  DevBuf<uint32_t> o_cls(task == 0 ? (size_t)cap * C : 1);
  DevBuf<int64_t> o_sum(task == 1 ? cap : 1);
  DevBuf<uint64_t> o_hash(cap);
  DevBuf<float> o_value(cap), o_thr(cap), o_score(cap);
  DevBuf<int64_t> o_left(cap);

  // roots
  {
    std::vector<int32_t> tr(T), dep(T, 0), cnt(T), mm(T);
    std::vector<uint32_t> idv(T, 0);
    std::vector<int64_t> st(T);
    std::vector<uint8_t> op(T);
    for (int t = 0; t < T; ++t) {
      tr[t] = t;
      cnt[t] = (int32_t)tN[t];
      mm[t] = (int32_t)root_m[t];
      st[t] = root_start[t];
      op[t] = (tN[t] > tree_min_node(t) && 0 < tree_max_depth(t)) ? 1 : 0;
    }
    DTE_HIP(hipMemcpyAsync(o_tree.p, tr.data(), 4 * T, hipMemcpyHostToDevice, s));
    DTE_HIP(hipMemcpyAsync(o_depth.p, dep.data(), 4 * T, hipMemcpyHostToDevice, s));
    DTE_HIP(hipMemcpyAsync(o_count.p, cnt.data(), 4 * T, hipMemcpyHostToDevice, s));
    DTE_HIP(hipMemcpyAsync(o_m.p, mm.data(), 4 * T, hipMemcpyHostToDevice, s));
    DTE_HIP(hipMemcpyAsync(o_id.p, idv.data(), 4 * T, hipMemcpyHostToDevice, s));
    if (task == 0)
      DTE_HIP(hipMemcpyAsync(o_cls.p, root_cls.p, 4 * (size_t)T * C, hipMemcpyDeviceToDevice, s));
    else
      DTE_HIP(hipMemcpyAsync(o_sum.p, root_sum.p, 8 * (size_t)T, hipMemcpyDeviceToDevice, s));
    DTE_HIP(hipMemcpyAsync(o_hash.p, root_hash.p, 8 * (size_t)T, hipMemcpyDeviceToDevice, s));
    // root value (regression mean)
    if (task == 1) {
      std::vector<int64_t> rs(T);
      DTE_HIP(hipMemcpyAsync(rs.data(), root_sum.p, 8 * T, hipMemcpyDeviceToHost, s));
      DTE_HIP(hipStreamSynchronize(s));
      std::vector<float> rv(T);
      for (int t = 0; t < T; ++t)
        rv[t] = (float)std::ldexp((double)rs[t] / (double)tN[t], -(J ? J->f[tf[t]].fd->shift : shift));
      DTE_HIP(hipMemcpyAsync(o_value.p, rv.data(), 4 * T, hipMemcpyHostToDevice, s));
    } else {
      DTE_HIP(hipMemsetAsync(o_value.p, 0, 4 * T, s));
    }
    // working arrays of level 0
  }
  DevBuf<int64_t> w_start(T), w_start_next;
  DevBuf<uint8_t> w_open(T), w_open_next;
  {
    std::vector<int64_t> st(root_start);
    std::vector<uint8_t> op(T);
    for (int t = 0; t < T; ++t) op[t] = (tN[t] > tree_min_node(t) && 0 < tree_max_depth(t)) ? 1 : 0;
    DTE_HIP(hipMemcpyAsync(w_start.p, st.data(), 8 * T, hipMemcpyHostToDevice, s));
    DTE_HIP(hipMemcpyAsync(w_open.p, op.data(), T, hipMemcpyHostToDevice, s));
  }
  DevBuf<uint32_t> lf(T + 1), base(T), lf_next(T + 1), base_next(T);
  {
    std::vector<uint32_t> l(T + 1), b(T, 0);
    for (int t = 0; t <= T; ++t) l[t] = t;
    DTE_HIP(hipMemcpyAsync(lf.p, l.data(), 4 * (T + 1), hipMemcpyHostToDevice, s));
    DTE_HIP(hipMemcpyAsync(base.p, b.data(), 4 * T, hipMemcpyHostToDevice, s));
  }

  // per-level scratch
  DevBuf<uint32_t> flag32, open_pos, open_idx, nchild, cpos, retry_flag, retry_pos, retry_list;
  DevBuf<float> res_score, res_thr, ch_score, ch_thr;
  DevBuf<int32_t> res_feat, ch_feat, l_m, l_count;
  DevBuf<uint32_t> l_cls;
  DevBuf<int64_t> l_sum;
  DevBuf<uint64_t> l_hash;
  DevBuf<uint8_t> split_ok;
  DevBuf<uint32_t> scr_key, scr_aux;
  DevBuf<int64_t> scr_y;
  int64_t scr_stride = 0;

  int num_cu = 256;
  {
    int dev;
    DTE_HIP(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    DTE_HIP(hipGetDeviceProperties(&prop, dev));
    num_cu = prop.multiProcessorCount;
  }
  const int search_grid_cap = num_cu * 4;

  SearchFn search = pick_search(task, C);
  BigFn big = pick_big(task, C);
  BigState bigst;
  PartFn partition = pick_part(task, C);
  PartWaveFn partition_wave = pick_part_wave(task, C);
  PartWaveFn partition_seg16 = pick_part_seg<16>(task, C);
  PartWaveFn partition_seg32 = pick_part_seg<32>(task, C);
  PartChunkFn partition_chunks = pick_part_chunks(task, C);
  // host-sized levels: nodes above kPartBig entries partition by chunks
  constexpr Cuts kPartCutsHost{{16, 32, 512, kPartBig, 0x7FFFFFFF, 0}, 5};
  DevBuf<uint32_t> pch_n, pch_off, pch_ml, pch_acc_ml, pch_acc_cls;
  DevBuf<unsigned long long> pch_acc64;

  // Size tiers of the split search: wave per item up to wave_cutoff entries,
  // block per item above (the block kernel itself switches to the bucketed
  // path above its LDS capacity).
  // Nodes above the workgroup's LDS capacity go through the chunk-parallel
  // pipeline (the plain driver keeps one workgroup per node throughout).
  // k_search_rf_bound counts two classes in a word: its nodes weigh at most
  // 65535 (a bootstrap's multiplicities hardly ever pass 15, so this bites at
  // no node size; the pipeline takes any weight).
  const int m_packed = (int)std::max<int64_t>(1, kBoundWeight / (int64_t)std::max<uint32_t>(w_max, 1));
  const int cut_team = std::min(m_packed, p.cut_team ? p.cut_team : kDefCutTeam);
  const int cut_block =
      std::min(m_packed, std::max(cut_team, std::min(kCap, p.cut_block ? p.cut_block : kDefCutBlock)));
  bigst.target = p.bucket_target ? p.bucket_target : kDefBucketTarget;
  bigst.max_dev = fd.max_fixed;
  Cuts cuts{};
  if (algorithm == DTE_RANDOM_FOREST) {
    // the segment tiers take x ln x terms from the table's head in LDS: a node
    // of 32 entries must weigh less than it (a multiplicity of 64 hardly ever
    // occurs in a bootstrap; such a fit starts at the wave tier)
    const bool light = task == 1 || 32 * (int64_t)w_max < SegLds<0>::kTL;
    const int c16 = light && (task == 1 || C <= 16) ? 16 : 0;
    const int c32 = light ? 32 : 0;
    cuts = Cuts{{c16, std::max(c16, c32), std::min(64, cut_team), cut_team, cut_block, 0x7FFFFFFF}, 6};
  } else {
    // segment tiers need a lane per class
    const int c16 = (task == 1 || C <= 16) ? 16 : 0;
    const int c32 = (task == 1 || C <= 32) ? 32 : 0;
    const int ce = p.cut_ert ? p.cut_ert : kDefCutErt;
    cuts = Cuts{{c16, std::max(c16, c32), 64, std::min(ce, kErtTeamIpt * kWave), ce, 0x7FFFFFFF}, 6};
  }
  DevBuf<uint32_t> tier_list[kMaxTiers];
  DevBuf<unsigned int> tier_cnt(kMaxTiers);
  auto tier_grid = [](int64_t n) { return (unsigned)std::min<int64_t>((n + kTierBlock - 1) / kTierBlock, kTierGrid); };
  auto tier_lists = [&]() {
    TierLists tl{};
    for (int k = 0; k < kMaxTiers; ++k) tl.l[k] = tier_list[k].p;
    return tl;
  };
  const int wave_grid_cap = num_cu * 16;
  const int spread_waves = num_cu * 12;  // three waves per SIMD, the least the bounded tiers run at
  // a little over the merged kernel's three workgroups a CU
  auto merged_cap = [num_cu](int tier) { return tier <= 3 ? num_cu * 4 : num_cu * 3; };
  const bool small_data = E <= kMergeEntries;
  const RfAllFn rf_all = pick_rf_all(task, C);
  LevelArgs lv{};
  int64_t trace_tier[3] = {0, 0, 0};
  // Keys of a level's first draws by entry (k_gather_draws), read on the side
  // stream: declared before it, so that a fit that fails gives them up after
  // the stream's last wait.
  DevBuf<uint32_t> key_rows, draw_keys, draw_tiles, draw_toff;
  // Side stream of the split search's tiers beside the chunk pipeline
  // (created on first use; default priority).
  struct SideStream {
    hipStream_t st = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
    hipStream_t get() {
      if (!st) {
        DTE_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
        DTE_HIP(hipEventCreateWithFlags(&fork, hipEventDisableTiming));
        DTE_HIP(hipEventCreateWithFlags(&join, hipEventDisableTiming));
      }
      return st;
    }
    ~SideStream() {
      if (st) {
        (void)hipStreamSynchronize(st);
        (void)hipEventDestroy(fork);
        (void)hipEventDestroy(join);
        (void)hipStreamDestroy(st);
      }
    }
  } side;
  // The draws' keys are gathered if they pay and, with the scratch of the chunk
  // pipeline's largest batch, leave half of the free memory; without them the
  // searches gather from K.
  const int FS = (d.F + 15) / 16 * 16;
  bool use_rows = algorithm == DTE_RANDOM_FOREST && !plain && key_rows_pay(d.N, d.F, D0);
  if (use_rows) {
    size_t free_b = 0, total_b = 0;
    int dev;
    DTE_HIP(hipGetDevice(&dev));
    DTE_HIP(hipMemGetInfo(&free_b, &total_b));
    free_b += pool_cached(dev);  // what an earlier fit left counts as free
    const int64_t slots = std::min<int64_t>(kV2Batch, (int64_t)T * N * D0) + N;
    const size_t batch = (size_t)(slots + slots / 4) * v2_slot_bytes(task);  // reserve() adds a quarter
    use_rows = 4 * ((size_t)d.N * FS + (size_t)E * D0) + batch <= free_b / 2;
  }
  if (use_rows) {
    try {
      key_rows.alloc((size_t)d.N * FS);
      draw_keys.alloc((size_t)E * D0);
    } catch (const std::exception&) {  // another thread's fit took the memory
      (void)hipGetLastError();
      key_rows.release();
      draw_keys.release();
      use_rows = false;
    }
  }
  if (use_rows) {
    hipLaunchKernelGGL(k_key_rows, dim3((unsigned)((d.N + kWave - 1) / kWave)), dim3(kBlock),
                       (unsigned)(4 * kWave * (FS + 1)), s, d.K, d.N, d.F, FS, key_rows.p);
  }
  auto run_phase = [&](ItemArgs it) {
    for (auto& tl : tier_list) tl.reserve(it.n_groups);
    DTE_HIP(hipMemsetAsync(tier_cnt.p, 0, 4 * kMaxTiers, s));
    hipLaunchKernelGGL(k_tier_split, dim3(tier_grid(it.n_groups)), dim3(kTierBlock), 0, s, it.list, it.n_groups,
                       lv.open_idx, lv.m, cuts, tier_lists(), tier_cnt.p);
    unsigned int cnt[kMaxTiers];
    DTE_HIP(hipMemcpyAsync(cnt, tier_cnt.p, 4 * kMaxTiers, hipMemcpyDeviceToHost, s));
    DTE_HIP(hipStreamSynchronize(s));
    Timer tm("split_search", 0.0, s);
    const bool rf = algorithm == DTE_RANDOM_FOREST;
    // The chunk pipeline (random-forest nodes above cut_block) runs on the
    // library stream with host round trips between its batches; the other
    // tiers touch other nodes and run beside it on a side stream.
    bool others = false;
    for (int tier = 0; tier < 5; ++tier) others = others || cnt[tier] > 0;
    if (use_rows && it.j0 == 0 && cnt[2] + cnt[3] + cnt[4] + cnt[5] > 0) {
      Timer tk("gather_draws", 0.0, s);
      DrawNodes dn{};
      for (int k = 0; k < 4; ++k) {
        dn.list[k] = tier_list[2 + k].p;
        dn.first[k + 1] = dn.first[k] + cnt[2 + k];
      }
      const int64_t n = dn.first[4];
      draw_tiles.reserve(n + 1);
      draw_toff.reserve(n + 1);
      hipLaunchKernelGGL(k_draw_tiles, dim3(grid_for(n)), dim3(kBlock), 0, s, lv, dn, draw_tiles.p);
      scan_u32(draw_tiles.p, n, draw_toff.p, s, scan_tmp);
      hipLaunchKernelGGL(k_gather_draws, dim3((unsigned)num_cu * 16), dim3(kGatherWaves * kWave),
                         (unsigned)(4 * kGatherWaves * kWave * (FS + 1)), s, d, lv, (const uint32_t*)key_rows.p, FS, dn,
                         (const uint32_t*)draw_toff.p, it.per_group, draw_keys.p, E);
      it.gk = draw_keys.p;
      it.gk_stride = E;
    }
    const bool overlap = rf && cnt[5] > 0 && others;
    hipStream_t ts = s;
    if (overlap) {
      ts = side.get();
      DTE_HIP(hipEventRecord(side.fork, s));
      DTE_HIP(hipStreamWaitEvent(ts, side.fork, 0));
    }
    const bool merged = rf && small_data && others;
    if (merged) {
      RfTiers rt{};
      int64_t blocks = 0;
      for (int tier = 0; tier < 5; ++tier) {
        rt.cap[tier] = merged_cap(tier);
        blocks += std::min<int64_t>(rf_tier_blocks(tier, cnt[tier], it.per_group, it.spread), rt.cap[tier]);
        rt.list[tier] = tier_list[tier].p;
        rt.n[tier] = cnt[tier];
        rt.bytes[tier] = it.bytes ? it.bytes + (size_t)tier * kByteWords : nullptr;
        trace_tier[tier <= 2 ? 0 : (tier == 3 ? 1 : 2)] += cnt[tier];
      }
      Timer tk("search_merged", 0.0, ts);
      rf_all(blocks, ts, d, lv, it, rt);
    }
    for (int tier = merged ? 5 : 0; tier < cuts.n; ++tier) {
      if (!cnt[tier]) continue;
      ItemArgs a = it;
      a.list = tier_list[tier].p;
      a.n_groups = cnt[tier];
      a.bytes = it.bytes ? it.bytes + (size_t)tier * kByteWords : nullptr;
      trace_tier[rf ? (tier <= 2 ? 0 : (tier == 3 ? 1 : 2)) : (tier <= 2 ? 0 : (tier <= 4 ? 1 : 2))] += cnt[tier];
      if (rf && tier == 5) continue;  // below, after the side launches
      int grid;
      if (rf) {
        grid = (int)std::min<int64_t>(rf_tier_blocks(tier, cnt[tier], it.per_group, it.spread),
                                      tier <= 3 ? wave_grid_cap : search_grid_cap);
      } else if (tier <= 3) {
        // node-major tiers: 4 / 2 / 1 / 1 nodes per wave
        const int npw = tier == 0 ? 4 : (tier == 1 ? 2 : 1);
        grid = (int)std::min<int64_t>((cnt[tier] + npw * kWaves - 1) / (npw * kWaves), wave_grid_cap);
      } else {
        const int64_t items = (int64_t)cnt[tier] * it.per_group;
        const bool whole = tier == 5;
        const int per_block = whole ? 1 : kWaves;
        const int cap = whole ? search_grid_cap : wave_grid_cap;
        grid = (int)std::min<int64_t>((items + per_block - 1) / per_block, cap);
      }
      Timer tk(search_family(algorithm, tier), 0.0, ts);
      search(algorithm, tier, grid, ts, d, lv, a);
    }
    if (rf && cnt[5]) {
      ItemArgs a = it;
      a.list = tier_list[5].p;
      a.n_groups = cnt[5];
      a.bytes = it.bytes ? it.bytes + (size_t)5 * kByteWords : nullptr;
      Timer tk(search_family(algorithm, 5), 0.0, s);
      big(bigst, d, lv, a, tier_list[5].p, cnt[5], s, num_cu);
    }
    if (overlap) {
      DTE_HIP(hipEventRecord(side.join, ts));
      DTE_HIP(hipStreamWaitEvent(s, side.join, 0));
    }
  };
  // Plain launch structure: chunks of at most kPlainChunk open nodes, one
  // workgroup per node, a host round trip after every chunk.
  DevBuf<uint32_t> iota_list;
  auto identity_list = [&](int64_t n) {
    iota_list.reserve(n);
    hipLaunchKernelGGL(k_iota, dim3(grid_for(n)), dim3(kBlock), 0, s, iota_list.p, n);
    return (const uint32_t*)iota_list.p;
  };
  auto plain_phase = [&](ItemArgs it) {
    const uint32_t* lst = it.list ? it.list : identity_list(it.n_groups);
    const int tier = algorithm == DTE_RANDOM_FOREST ? 6 : 5;  // workgroup per node, any size
    Timer tm("split_search", 0.0, s);
    for (int64_t c0 = 0; c0 < it.n_groups; c0 += kPlainChunk) {
      ItemArgs a = it;
      a.list = lst + c0;
      a.n_groups = std::min<int64_t>(kPlainChunk, it.n_groups - c0);
      a.node_major = 1;
      a.bytes = it.bytes ? it.bytes + (size_t)tier * kByteWords : nullptr;
      Timer tk(search_family(algorithm, tier), 0.0, s);
      search(algorithm, tier, (int)a.n_groups, s, d, lv, a);
      DTE_HIP(hipStreamSynchronize(s));
    }
  };
  const bool trace = std::getenv("DTE_TRACE") != nullptr;

  int64_t off_level = 0;
  int64_t n_level = T;
  int64_t max_m = 0;
  for (int t = 0; t < T; ++t) max_m = std::max(max_m, root_m[t]);
  int64_t big_entries = max_m > cut_block ? E : 0;  // entries in nodes above cut_block

  uint32_t* cur_row = rowA.p;
  uint32_t* cur_aux = auxA.p;
  int64_t* cur_ey = eyA.p;
  uint32_t* nxt_row = rowB.p;
  uint32_t* nxt_aux = auxB.p;
  int64_t* nxt_ey = eyB.p;

  // ---- device-described level steps.  Once every open node of a level
  // fits the device-sized tiers, all further levels run from two captured
  // hipGraphs (even / odd: the ping-pong buffers swap every level) whose
  // kernels read the level's offset and counts from a DevLevel in device
  // memory and run on capped grids; counters are cleared by a kernel.  The
  // buffers are sized once for the largest level possible: a level has at
  // most one node per entry, and at most T * N / (min_node + 1) open nodes.
  DevBuf<unsigned long long> graph_bytes(count_bytes ? (kMaxTiers + 1) * kByteWords : 1);  // search tiers, partition
  auto graph_counter = [&](int tier) { return count_bytes ? graph_bytes.p + (size_t)tier * kByteWords : nullptr; };
  int64_t graph_replays = 0;
  auto device_levels = [&](int depth0) {
    int64_t min1 = (int64_t)std::max(p.min_node_size, 0) + 1, W = 0;
    for (int t = 0; t < T; ++t) {
      W += tN[t];
      min1 = std::min<int64_t>(min1, (int64_t)std::max(tree_min_node(t), 0) + 1);
    }
    const int64_t NO = std::max<int64_t>(1, std::min<int64_t>(E, W / min1));
    const int64_t NL = std::max<int64_t>(n_level, std::min<int64_t>(E, 2 * NO));
    auto fit_to = [](auto& b, int64_t n) {
      if ((int64_t)b.n < n) b.alloc((size_t)n);
    };
    {  // the current level's working arrays keep their contents
      DevBuf<int64_t> st((size_t)NL + 1);
      DevBuf<uint8_t> op((size_t)NL + 1);
      DTE_HIP(hipMemcpyAsync(st.p, w_start.p, 8 * n_level, hipMemcpyDeviceToDevice, s));
      DTE_HIP(hipMemcpyAsync(op.p, w_open.p, n_level, hipMemcpyDeviceToDevice, s));
      w_start = std::move(st);
      w_open = std::move(op);
    }
    fit_to(w_start_next, NL + 1);
    fit_to(w_open_next, NL + 1);
    fit_to(open_pos, NL + 1);
    fit_to(open_idx, NO + 1);
    fit_to(res_score, NO * D);
    fit_to(res_thr, NO * D);
    fit_to(res_feat, NO * D);
    fit_to(ch_score, NO);
    fit_to(ch_thr, NO);
    fit_to(ch_feat, NO);
    fit_to(retry_flag, NO);
    fit_to(l_m, NO);
    fit_to(l_count, NO);
    fit_to(l_cls, task == 0 ? NO * C : 1);
    fit_to(l_sum, NO);
    fit_to(l_hash, NO);
    fit_to(split_ok, NO);
    for (auto& tl : tier_list) fit_to(tl, NO);
    fit_to(nchild, NL);
    fit_to(cpos, NL + 1);
    // scratch slabs of the workgroup-per-item kernel for nodes above
    // cut_block (random forest), one per workgroup of its grid
    const bool big_tier = algorithm == DTE_RANDOM_FOREST && max_m > cut_block;
    if (big_tier && scr_stride < max_m) {
      scr_key.alloc((size_t)search_grid_cap * max_m);
      scr_aux.alloc((size_t)search_grid_cap * max_m);
      if (task == 1) scr_y.alloc((size_t)search_grid_cap * max_m);
      scr_stride = max_m;
    }
    DevBuf<uint32_t> dsums(kDScanBlocks);
    DevBuf<DevLevel> dlv(2);  // even and odd levels
    constexpr int kPartLists = 4;
    DevBuf<uint32_t> part_list[kPartLists];
    TierLists part_lists{};
    for (int k = 0; k < kPartLists; ++k) {
      part_list[k].alloc(NO);
      part_lists.l[k] = part_list[k].p;
    }
    DevLevel h{};
    h.off = off_level;
    h.n = n_level;
    h.depth = depth0;
    DTE_HIP(hipMemcpyAsync(dlv.p, &h, sizeof(h), hipMemcpyHostToDevice, s));
    if (count_bytes) DTE_HIP(hipMemsetAsync(graph_bytes.p, 0, graph_bytes.bytes(), s));
    const bool rf = algorithm == DTE_RANDOM_FOREST;
    constexpr int kElemGrid = 1024;
    // Small data (at most kMergeEntries entries over all trees): one launch
    // for all search tiers of a phase.  Its levels are small and
    // latency-bound, and side by side the tiers finish sooner (4,601 x 57, 100
    // extra trees: 12.3k -> 15.9k trees/s; random forest of 3.2 M entries, a
    // level of its deepest: 0.92 -> 0.77 ms); on large data the merged
    // kernel's register budget (the largest tier's) costs more occupancy than
    // the overlap gains (64 extra-trees forests: 8.2k -> 6.9k).
    const bool ert_merged = !rf && small_data;
    const ErtAllFn ert_all = pick_ert_all(task, C);
    // likewise the partition tiers of a step (both algorithms)
    const PartAllFn partition_all = pick_part_all(task, C);

    // One level step on stream s; par = 1 swaps the ping-pong buffers.
    auto enqueue = [&](int par, hipStream_t s) {
      DevLevel* const L = dlv.p + par;
      DevLevel* const L_next = dlv.p + (par ^ 1);
      int64_t* cs = par ? w_start_next.p : w_start.p;
      int64_t* ns = par ? w_start.p : w_start_next.p;
      uint8_t* co = par ? w_open_next.p : w_open.p;
      uint8_t* no = par ? w_open.p : w_open_next.p;
      uint32_t* clf = par ? lf_next.p : lf.p;
      uint32_t* nlf = par ? lf.p : lf_next.p;
      uint32_t* cbase = par ? base_next.p : base.p;
      uint32_t* nbase = par ? base.p : base_next.p;
      uint32_t* crow = par ? nxt_row : cur_row;
      uint32_t* nrw = par ? cur_row : nxt_row;
      uint32_t* caux = par ? nxt_aux : cur_aux;
      uint32_t* nax = par ? cur_aux : nxt_aux;
      int64_t* cey = par ? nxt_ey : cur_ey;
      int64_t* ney = par ? cur_ey : nxt_ey;
      // open nodes, by search and partition tier
      hipLaunchKernelGGL(k_open_sums, dim3(kDScanBlocks), dim3(kBlock), 0, s, (const uint8_t*)co, (const DevLevel*)L,
                         dsums.p);
      hipLaunchKernelGGL(k_level_lists, dim3(kDScanBlocks), dim3(kBlock), 0, s, (const uint8_t*)co, L,
                         (const uint32_t*)dsums.p, (const int32_t*)o_m.p, open_pos.p, open_idx.p, cuts, tier_lists(),
                         kPartCuts, part_lists);
      LevelArgs lvd{};
      lvd.tree = o_tree.p;
      lvd.id = o_id.p;
      lvd.count = o_count.p;
      lvd.m = o_m.p;
      lvd.cls = task == 0 ? o_cls.p : nullptr;
      lvd.sum = task == 1 ? o_sum.p : nullptr;
      lvd.start = cs;
      lvd.open_idx = open_idx.p;
      lvd.tree_global = tree_global.p;
      lvd.row = crow;
      lvd.aux = caux;
      lvd.ey = cey;
      lvd.off_dev = &L->off;
      ItemArgs it{};
      it.D = D;
      it.res_score = res_score.p;
      it.res_thr = res_thr.p;
      it.res_feat = res_feat.p;
      it.scr_key = scr_key.p;
      it.scr_aux = scr_aux.p;
      it.scr_y = scr_y.p;
      it.scr_stride = scr_stride;
      it.spread = spread_waves;
      // split search of one phase over the tiers; nodes above cut_block
      // (tier 5) take one workgroup per item through its scratch slab
      auto phase = [&](unsigned int* cnt, int per_group, int j0) {
        if (ert_merged) {
          ErtTiers ts{};
          int64_t acc = 0;
          for (int k = 0; k < 6; ++k) {
            ts.cap[k] = k <= 4 ? num_cu * 6 : search_grid_cap;
            acc += ts.cap[k];
            ts.list[k] = tier_list[k].p;
            ts.n_dev[k] = cnt + k;
            ts.bytes[k] = graph_counter(k);
          }
          ItemArgs a = it;
          a.per_group = per_group;
          a.j0 = j0;
          ert_all(acc, s, d, lvd, a, ts);
          return;
        }
        if (rf && small_data) {
          RfTiers ts{};
          for (int tier = 0; tier < 5; ++tier) {
            ts.cap[tier] = merged_cap(tier);
            ts.list[tier] = tier_list[tier].p;
            ts.n_dev[tier] = cnt + tier;
            ts.bytes[tier] = graph_counter(tier);
          }
          ItemArgs a = it;
          a.per_group = per_group;
          a.j0 = j0;
          int64_t blocks = 0;
          for (int c : ts.cap) blocks += c;
          rf_all(blocks, s, d, lvd, a, ts);
        }
        for (int tier = rf && small_data ? 5 : 0; tier < cuts.n; ++tier) {
          if (rf && tier == 5 && !big_tier) continue;  // no node above cut_block in these levels
          ItemArgs a = it;
          a.list = tier_list[tier].p;
          a.n_groups = 0;
          a.n_dev = cnt + tier;
          a.per_group = per_group;
          a.j0 = j0;
          a.bytes = graph_counter(tier);
          const int grid = tier <= (rf ? 3 : 4) ? wave_grid_cap : search_grid_cap;
          search(algorithm, rf && tier == 5 ? 6 : tier, grid, s, d, lvd, a);
        }
      };
      phase(L->tier, D0, 0);
      DecideArgs da{};
      da.D0 = D0;
      da.R = R;
      da.D = D;
      da.res_score = res_score.p;
      da.res_thr = res_thr.p;
      da.res_feat = res_feat.p;
      da.ch_score = ch_score.p;
      da.ch_thr = ch_thr.p;
      da.ch_feat = ch_feat.p;
      da.retry_flag = retry_flag.p;
      da.n_open_dev = &L->n_open;
      // the retry phase's tier lists take the place of the first phase's
      hipLaunchKernelGGL(k_decide1_dev, dim3(kDecideGrid), dim3(kTierBlock), 0, s, d, lvd, da, algorithm, cuts,
                         tier_lists(), L->rtier);
      if (R > 0) {
        phase(L->rtier, R, D0);
        hipLaunchKernelGGL(k_decide2_dev, dim3(kElemGrid), dim3(kBlock), 0, s, d, lvd, da);
      }
      // partition
      PartArgs pa{};
      pa.ch_feat = ch_feat.p;
      pa.ch_thr = ch_thr.p;
      pa.nrow = nrw;
      pa.naux = nax;
      pa.ney = ney;
      pa.l_m = l_m.p;
      pa.l_count = l_count.p;
      pa.l_cls = l_cls.p;
      pa.l_sum = l_sum.p;
      pa.l_hash = l_hash.p;
      pa.split_ok = split_ok.p;
      pa.bytes = graph_counter(kMaxTiers);
      PartArgs p0 = pa, p1 = pa, p2 = pa, p3 = pa;
      p0.n_dev = L->ptier + 0;
      p1.n_dev = L->ptier + 1;
      p2.n_dev = L->ptier + 2;
      p3.n_dev = L->ptier + 3;
      p3.list = part_list[3].p;
      if (small_data) {
        PartTiers pt{};
        int64_t acc = 0;
        for (int k = 0; k < 4; ++k) {
          pt.cap[k] = k <= 2 ? num_cu * 8 : search_grid_cap;
          acc += pt.cap[k];
          pt.list[k] = part_list[k].p;
          pt.n_dev[k] = L->ptier + k;
        }
        pt.n_bound = NO;
        partition_all(acc, s, d, lvd, pa, pt);
      } else {
        partition_seg16(wave_grid_cap, s, d, lvd, p0, part_list[0].p, NO);  // grid from the bound; count from p0.n_dev
        partition_seg32(wave_grid_cap, s, d, lvd, p1, part_list[1].p, NO);
        partition_wave(wave_grid_cap, s, d, lvd, p2, part_list[2].p, NO);
        partition(search_grid_cap, s, d, lvd, p3);
      }
      // children
      ChildArgs ca{};
      ca.lvl = L;
      ca.open = co;
      ca.open_pos = open_pos.p;
      ca.split_ok = split_ok.p;
      ca.ch_feat = ch_feat.p;
      ca.ch_thr = ch_thr.p;
      ca.ch_score = ch_score.p;
      ca.l_m = l_m.p;
      ca.l_count = l_count.p;
      ca.l_cls = l_cls.p;
      ca.l_sum = l_sum.p;
      ca.l_hash = l_hash.p;
      ca.nchild = nchild.p;
      ca.cpos = cpos.p;
      ca.lf = clf;
      ca.base = cbase;
      ca.o_tree = o_tree.p;
      ca.o_id = o_id.p;
      ca.o_depth = o_depth.p;
      ca.o_count = o_count.p;
      ca.o_m = o_m.p;
      ca.o_cls = task == 0 ? o_cls.p : nullptr;
      ca.o_sum = o_sum.p;
      ca.o_hash = o_hash.p;
      ca.o_value = o_value.p;
      ca.o_feature = o_feature.p;
      ca.o_thr = o_thr.p;
      ca.o_score = o_score.p;
      ca.o_left = o_left.p;
      ca.start = cs;
      ca.n_start = ns;
      ca.n_open = no;
      hipLaunchKernelGGL(k_child_sums, dim3(kDScanBlocks), dim3(kBlock), 0, s, ca, dsums.p);
      hipLaunchKernelGGL(k_child_scan, dim3(kDScanBlocks), dim3(kBlock), 0, s, (const uint32_t*)nchild.p, L,
                         (const uint32_t*)dsums.p, cpos.p);
      hipLaunchKernelGGL(k_children_write_dev, dim3(kElemGrid), dim3(kBlock), 0, s, d, ca, T, nlf, nbase, L_next);
      DTE_HIP(hipGetLastError());
    };

    struct Graphs {
      hipGraphExec_t e[2] = {nullptr, nullptr};
      ~Graphs() {
        for (auto x : e)
          if (x) (void)hipGraphExecDestroy(x);
      }
    } gr;
    const auto cap_t0 = std::chrono::steady_clock::now();
    for (int par = 0; par < 2; ++par) {
      hipGraph_t g = nullptr;
      {
        const RecordStream rec(s);
        DTE_HIP(hipStreamBeginCapture(rec.stream, hipStreamCaptureModeThreadLocal));
        try {
          enqueue(par, rec.stream);
        } catch (...) {
          (void)hipStreamEndCapture(rec.stream, &g);
          if (g) (void)hipGraphDestroy(g);
          throw;
        }
        DTE_HIP(hipStreamEndCapture(rec.stream, &g));
      }
      const hipError_t e = hipGraphInstantiate(&gr.e[par], g, nullptr, nullptr, 0);
      (void)hipGraphDestroy(g);
      DTE_HIP(e);
    }
    if (profiling_enabled())
      profile_host("graph_capture_host",
                   std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - cap_t0).count());
    int par = 0;
    auto replay = [&](int64_t k) {
      for (int64_t i = 0; i < k; ++i) {
        DTE_HIP(hipGraphLaunch(gr.e[par], s));
        par ^= 1;
        ++graph_replays;
      }
    };
    {
      Timer tm("level_graph", 0.0, s);
      int max_depth = p.max_depth;
      for (int t = 0; t < T; ++t) max_depth = std::max(max_depth, tree_max_depth(t));
      const int64_t steps = (int64_t)max_depth - depth0 + 1;  // levels depth0 .. max_depth
      if (steps <= 64) {
        replay(std::max<int64_t>(steps, 1));
      } else {
        // deep trees: batches of 8 steps; the next batch is queued before the
        // previous one's node count is looked at, so the device never waits
        constexpr int kStepBatch = 8;
        int64_t* pin = nullptr;
        DTE_HIP(hipHostMalloc((void**)&pin, 2 * sizeof(int64_t), hipHostMallocDefault));
        hipEvent_t ev[2] = {nullptr, nullptr};
        try {
          DTE_HIP(hipEventCreateWithFlags(&ev[0], hipEventDisableTiming));
          DTE_HIP(hipEventCreateWithFlags(&ev[1], hipEventDisableTiming));
          for (int64_t b = 0;; ++b) {
            replay(kStepBatch);
            DTE_HIP(hipMemcpyAsync(pin + (b & 1), &dlv.p[par].n, sizeof(int64_t), hipMemcpyDeviceToHost, s));
            DTE_HIP(hipEventRecord(ev[b & 1], s));
            if (b > 0) {
              DTE_HIP(hipEventSynchronize(ev[(b - 1) & 1]));
              if (pin[(b - 1) & 1] == 0) break;
            }
          }
        } catch (...) {
          (void)hipStreamSynchronize(s);
          for (auto e : ev)
            if (e) (void)hipEventDestroy(e);
          (void)hipHostFree(pin);
          throw;
        }
        DTE_HIP(hipStreamSynchronize(s));
        for (auto e : ev) (void)hipEventDestroy(e);
        (void)hipHostFree(pin);
      }
    }
    int64_t fin[2];  // DevLevel.off, DevLevel.n
    DTE_HIP(hipMemcpyAsync(fin, dlv.p + par, sizeof(fin), hipMemcpyDeviceToHost, s));
    DTE_HIP(hipStreamSynchronize(s));
    if (fin[1] != 0) fail(DTE_ERR_INTERNAL, "level graph: nodes left after the last level step");
    off_level = fin[0];
    n_level = 0;
    if (par) {  // the final per-tree counts are in the other ping-pong buffer
      std::swap(lf, lf_next);
      std::swap(base, base_next);
      std::swap(w_start, w_start_next);
      std::swap(w_open, w_open_next);
      std::swap(cur_row, nxt_row);
      std::swap(cur_aux, nxt_aux);
      std::swap(cur_ey, nxt_ey);
    }
  };
  const bool level_graphs = !plain && p.build_mode == DTE_BUILD_BATCHED;
  if (profiling_enabled()) {
    DTE_HIP(hipStreamSynchronize(s));
    profile_host("fit_setup_host", std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - fit_t0).count());
  }

  for (int depth = 0; n_level > 0; ++depth) {
    // Random forests switch to the level graphs once the nodes above
    // cut_block hold at most 1/64 of the entries and none exceeds
    // kGraphMaxM: inside a graph such nodes take one workgroup per
    // (node, draw) with a scratch slab each (the plain driver's kernel).
    // They also do where these nodes are few and small enough for that kernel
    // to take less than the pipeline's launches and host round trips, 0.3 ms
    // and more a level: 4,601 x 57, 100 trees 7.3 ms without this, 6.3 at 1M
    // entry draws, 6.0 from 2M to 16M; 60,013 x 19 regression 16.8, 16.2, 15.9.
    if (level_graphs && (algorithm != DTE_RANDOM_FOREST ||
                         (max_m <= kGraphMaxM && big_entries * 64 <= E) ||
                         (max_m <= kGraphSmallM && big_entries * D0 <= kGraphBigWork))) {
      device_levels(depth);
      break;
    }
    double t_level0 = 0;
    if (trace) {
      DTE_HIP(hipStreamSynchronize(s));
      t_level0 = std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
      trace_tier[0] = trace_tier[1] = trace_tier[2] = 0;
    }
    // ---- open list
    flag32.reserve(n_level);
    open_pos.reserve(n_level + 1);
    hipLaunchKernelGGL(k_open_flags, dim3(grid_for(n_level)), dim3(kBlock), 0, s, w_open.p,
                       n_level, flag32.p);
    scan_u32(flag32.p, n_level, open_pos.p, s, scan_tmp);
    const int64_t n_open = read_one(open_pos.p + n_level, s);
    open_idx.reserve(n_open + 1);
    if (n_open > 0)
      hipLaunchKernelGGL(k_open_list, dim3(grid_for(n_level)), dim3(kBlock), 0, s, w_open.p,
                         open_pos.p, n_level, open_idx.p);

    lv = LevelArgs{};
    lv.tree = o_tree.p + off_level;
    lv.id = o_id.p + off_level;
    lv.count = o_count.p + off_level;
    lv.m = o_m.p + off_level;
    lv.cls = task == 0 ? o_cls.p + off_level * C : nullptr;
    lv.sum = task == 1 ? o_sum.p + off_level : nullptr;
    lv.start = w_start.p;
    lv.open_idx = open_idx.p;
    lv.tree_global = tree_global.p;
    lv.row = cur_row;
    lv.aux = cur_aux;
    lv.ey = cur_ey;

    if (n_open > 0) {
      res_score.reserve(n_open * D);
      res_thr.reserve(n_open * D);
      res_feat.reserve(n_open * D);
      ch_score.reserve(n_open);
      ch_thr.reserve(n_open);
      ch_feat.reserve(n_open);
      retry_flag.reserve(n_open);
      retry_pos.reserve(n_open + 1);
      retry_list.reserve(n_open + 1);
      // scratch slabs of the in-kernel bucketed path (nodes above kCap that
      // do not go through the chunk pipeline)
      if (algorithm == DTE_RANDOM_FOREST && max_m > kCap && plain) {
        const int64_t need = (int64_t)search_grid_cap * max_m;
        if (scr_stride < max_m) {
          scr_key.alloc(need);
          scr_aux.alloc(need);
          if (task == 1) scr_y.alloc(need);
          scr_stride = max_m;
        }
      }
      ItemArgs it{};
      it.list = nullptr;
      it.n_groups = n_open;
      it.per_group = D0;
      it.j0 = 0;
      it.D = D;
      it.res_score = res_score.p;
      it.res_thr = res_thr.p;
      it.res_feat = res_feat.p;
      it.bytes = tier_bytes(0);
      it.scr_key = scr_key.p;
      it.scr_aux = scr_aux.p;
      it.scr_y = scr_y.p;
      it.scr_stride = scr_stride;
      it.spread = spread_waves;
      if (plain) plain_phase(it); else run_phase(it);
      DecideArgs da{};
      da.n_open = n_open;
      da.D0 = D0;
      da.R = R;
      da.D = D;
      da.res_score = res_score.p;
      da.res_thr = res_thr.p;
      da.res_feat = res_feat.p;
      da.ch_score = ch_score.p;
      da.ch_thr = ch_thr.p;
      da.ch_feat = ch_feat.p;
      da.retry_flag = retry_flag.p;
      hipLaunchKernelGGL(k_decide1, dim3(grid_for(n_open)), dim3(kBlock), 0, s, d, lv, da, algorithm);
      if (R > 0) {
        scan_u32(retry_flag.p, n_open, retry_pos.p, s, scan_tmp);
        const int64_t n_retry = read_one(retry_pos.p + n_open, s);
        if (n_retry > 0) {
          hipLaunchKernelGGL(k_compact_list, dim3(grid_for(n_open)), dim3(kBlock), 0, s,
                             retry_flag.p, retry_pos.p, n_open, retry_list.p);
          it.list = retry_list.p;
          it.n_groups = n_retry;
          it.per_group = R;
          it.j0 = D0;
          if (plain) plain_phase(it); else run_phase(it);
          da.retry_list = retry_list.p;
          da.n_retry = n_retry;
          hipLaunchKernelGGL(k_decide2, dim3(grid_for(n_retry)), dim3(kBlock), 0, s, d, lv, da);
        }
      }
      // ---- partition
      l_m.reserve(n_open);
      l_count.reserve(n_open);
      l_cls.reserve(task == 0 ? n_open * C : 1);
      l_sum.reserve(n_open);
      l_hash.reserve(n_open);
      split_ok.reserve(n_open);
      PartArgs pa{};
      pa.n_open = n_open;
      pa.ch_feat = ch_feat.p;
      pa.ch_thr = ch_thr.p;
      pa.nrow = nxt_row;
      pa.naux = nxt_aux;
      pa.ney = nxt_ey;
      pa.l_m = l_m.p;
      pa.l_count = l_count.p;
      pa.l_cls = l_cls.p;
      pa.l_sum = l_sum.p;
      pa.l_hash = l_hash.p;
      pa.split_ok = split_ok.p;
      pa.bytes = part_bytes;
      if (plain) {
        const uint32_t* lst = identity_list(n_open);
        Timer tm("partition", 0.0, s);
        for (int64_t c0 = 0; c0 < n_open; c0 += kPlainChunk) {
          pa.list = lst + c0;
          pa.n_open = std::min<int64_t>(kPlainChunk, n_open - c0);
          partition((int)pa.n_open, s, d, lv, pa);
          DTE_HIP(hipStreamSynchronize(s));
        }
      } else {
        for (auto& tl : tier_list) tl.reserve(n_open);
        DTE_HIP(hipMemsetAsync(tier_cnt.p, 0, 4 * kMaxTiers, s));
        hipLaunchKernelGGL(k_tier_split, dim3(tier_grid(n_open)), dim3(kTierBlock), 0, s, (const uint32_t*)nullptr,
                           n_open, lv.open_idx, lv.m, kPartCutsHost, tier_lists(), tier_cnt.p);
        unsigned int pc[kMaxTiers];
        DTE_HIP(hipMemcpyAsync(pc, tier_cnt.p, 4 * kMaxTiers, hipMemcpyDeviceToHost, s));
        DTE_HIP(hipStreamSynchronize(s));
        Timer tm("partition", 0.0, s);
        if (pc[0]) partition_seg16(wave_grid_cap, s, d, lv, pa, tier_list[0].p, pc[0]);
        if (pc[1]) partition_seg32(wave_grid_cap, s, d, lv, pa, tier_list[1].p, pc[1]);
        if (pc[2])
          partition_wave((int)std::min<int64_t>((pc[2] + kWaves - 1) / kWaves, wave_grid_cap), s, d, lv, pa,
                         tier_list[2].p, pc[2]);
        if (pc[3]) {
          // workgroup partition over the remaining open positions
          pa.list = tier_list[3].p;
          pa.n_open = pc[3];
          partition((int)std::min<int64_t>(pc[3], search_grid_cap), s, d, lv, pa);
        }
        if (pc[4]) {
          // big nodes: chunks of kPartChunk entries, a workgroup each
          const int64_t nb = pc[4];
          pch_n.reserve(nb + 1);
          pch_off.reserve(nb + 1);
          hipLaunchKernelGGL(k_part_nchunks, dim3(std::min(grid_for(nb), 1024)), dim3(kBlock), 0, s,
                             (const uint32_t*)tier_list[4].p, nb, lv.open_idx, lv.m, pch_n.p);
          scan_u32(pch_n.p, nb, pch_off.p, s, scan_tmp);
          const int64_t n_chunks = (int64_t)read_one(pch_off.p + nb, s);
          pch_ml.reserve(n_chunks);
          pch_acc_ml.reserve(nb);
          pch_acc64.reserve(3 * nb);
          pch_acc_cls.reserve(task == 0 ? nb * C : 1);
          DTE_HIP(hipMemsetAsync(pch_acc_ml.p, 0, 4 * nb, s));
          DTE_HIP(hipMemsetAsync(pch_acc64.p, 0, 8 * 3 * nb, s));
          if (task == 0) DTE_HIP(hipMemsetAsync(pch_acc_cls.p, 0, 4 * nb * C, s));
          PartChunks pcs{tier_list[4].p, nb, pch_off.p, pch_ml.p, pch_acc_ml.p,
                         pch_acc64.p, pch_acc64.p + nb, pch_acc64.p + 2 * nb, pch_acc_cls.p};
          pa.list = nullptr;
          pa.n_open = n_open;
          partition_chunks(s, d, lv, pa, pcs, n_chunks);
        }
      }
    }

    // ---- children
    nchild.reserve(n_level);
    cpos.reserve(n_level + 1);
    ChildArgs ca{};
    ca.n_level = n_level;
    ca.off_level = off_level;
    ca.off_next = off_level + n_level;
    ca.depth = depth;
    ca.open = w_open.p;
    ca.open_pos = open_pos.p;
    ca.split_ok = split_ok.p;
    ca.ch_feat = ch_feat.p;
    ca.ch_thr = ch_thr.p;
    ca.ch_score = ch_score.p;
    ca.l_m = l_m.p;
    ca.l_count = l_count.p;
    ca.l_cls = l_cls.p;
    ca.l_sum = l_sum.p;
    ca.l_hash = l_hash.p;
    ca.nchild = nchild.p;
    ca.cpos = cpos.p;
    ca.lf = lf.p;
    ca.base = base.p;
    ca.o_tree = o_tree.p;
    ca.o_id = o_id.p;
    ca.o_depth = o_depth.p;
    ca.o_count = o_count.p;
    ca.o_m = o_m.p;
    ca.o_cls = task == 0 ? o_cls.p : nullptr;
    ca.o_sum = o_sum.p;
    ca.o_hash = o_hash.p;
    ca.o_value = o_value.p;
    ca.o_feature = o_feature.p;
    ca.o_thr = o_thr.p;
    ca.o_score = o_score.p;
    ca.o_left = o_left.p;
    ca.start = w_start.p;
    if (n_open == 0) {
      DTE_HIP(hipMemsetAsync(nchild.p, 0, 4 * n_level, s));
    } else {
      hipLaunchKernelGGL(k_children_count, dim3(grid_for(n_level)), dim3(kBlock), 0, s, ca);
    }
    scan_u32(nchild.p, n_level, cpos.p, s, scan_tmp);
    const int64_t n_next = read_one(cpos.p + n_level, s);
    w_start_next.reserve(n_next + 1);
    w_open_next.reserve(n_next + 1);
    ca.n_start = w_start_next.p;
    ca.n_open = w_open_next.p;
    hipLaunchKernelGGL(k_children_write, dim3(grid_for(n_level)), dim3(kBlock), 0, s, d, ca);
    hipLaunchKernelGGL(k_tree_update, dim3(grid_for(T + 1)), dim3(kBlock), 0, s, T, cpos.p, lf.p, base.p,
                       lf_next.p, base_next.p);
    std::swap(lf, lf_next);
    std::swap(base, base_next);
    std::swap(w_start, w_start_next);
    std::swap(w_open, w_open_next);
    std::swap(cur_row, nxt_row);
    std::swap(cur_aux, nxt_aux);
    std::swap(cur_ey, nxt_ey);
    if (trace) {
      DTE_HIP(hipStreamSynchronize(s));
      fprintf(stderr, "[dte] depth %d nodes %lld open %lld tiers %lld/%lld/%lld : %.3f ms\n", depth,
              (long long)n_level, (long long)n_open, (long long)trace_tier[0], (long long)trace_tier[1],
              (long long)trace_tier[2],
              1000.0 * (std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count() - t_level0));
    }
    off_level += n_level;
    n_level = n_next;
    // largest node of the next level (for scratch sizing) and the entries
    // in nodes above cut_block (whether the level graphs can take over)
    if (n_level > 0 && algorithm == DTE_RANDOM_FOREST) {
      DevBuf<unsigned long long> mx(2);
      DTE_HIP(hipMemsetAsync(mx.p, 0, 16, s));
      hipLaunchKernelGGL(k_level_sizes, dim3(std::min(grid_for(n_level), 1024)), dim3(kBlock), 0, s,
                         o_m.p + off_level, n_level, cut_block, mx.p);
      unsigned long long hm[2];
      DTE_HIP(hipMemcpyAsync(hm, mx.p, 16, hipMemcpyDeviceToHost, s));
      DTE_HIP(hipStreamSynchronize(s));
      max_m = (int64_t)hm[0];
      big_entries = (int64_t)hm[1];
    }
  }
  const int64_t n_nodes = off_level;
  if (count_bytes) {
    auto totals = [&](const DevBuf<unsigned long long>& counters) {
      std::vector<unsigned long long> w((kMaxTiers + 1) * kByteWords);
      DTE_HIP(hipMemcpyAsync(w.data(), counters.p, w.size() * 8, hipMemcpyDeviceToHost, s));
      DTE_HIP(hipStreamSynchronize(s));
      std::vector<unsigned long long> t(kMaxTiers + 1, 0);
      for (size_t x = 0; x < w.size(); x += kByteStride) t[x / kByteWords] += w[x];
      return t;
    };
    const std::vector<unsigned long long> sb = totals(byte_counts);
    double total = 0;
    for (int tier = 0; tier < kMaxTiers; ++tier) {
      if (!sb[tier]) continue;
      profile_add_bytes(search_family(algorithm, tier), (double)sb[tier]);
      total += (double)sb[tier];
    }
    profile_add_bytes("split_search", total);
    profile_add_bytes("partition", (double)sb[kMaxTiers]);
    if (graph_replays) {
      const std::vector<unsigned long long> gb = totals(graph_bytes);
      double g_search = 0;
      for (int tier = 0; tier < kMaxTiers; ++tier) g_search += (double)gb[tier];
      // level steps of the graphs: their split-search bytes (partition bytes
      // beside them) over the whole step time
      profile_add_bytes("level_graph", g_search);
      profile_add_bytes("level_graph_partition", (double)gb[kMaxTiers]);
    }
    profile_count("level_graph_replays", graph_replays);
  }

  // ---- canonical tree-major arrays
  std::vector<uint32_t> per_tree(T);
  DTE_HIP(hipMemcpyAsync(per_tree.data(), base.p, 4 * T, hipMemcpyDeviceToHost, s));
  DTE_HIP(hipStreamSynchronize(s));
  std::vector<int64_t> ts(T + 1, 0);
  for (int t = 0; t < T; ++t) ts[t + 1] = ts[t] + per_tree[t];
  if (ts[T] != n_nodes) fail(DTE_ERR_INTERNAL, "node count mismatch after build");

  auto* fo = new Forest();
  int dev;
  DTE_HIP(hipGetDevice(&dev));
  fo->device = dev;
  fo->task = task;
  fo->algorithm = algorithm;
  fo->n_classes = C;
  fo->n_features = J ? J->F : F;
  fo->n_trees = T;
  fo->fixed_shift = shift;
  fo->seed = p.seed;
  fo->tree_offset = t0;
  fo->fit_rows = algorithm == DTE_RANDOM_FOREST ? N : 0;
  fo->n_nodes = n_nodes;
  fo->n_leaves = (n_nodes + T) / 2;  // per tree: nodes = 2 splits + 1, leaves = splits + 1
  fo->has_stats = true;
  std::unique_ptr<PoolSuspend> own;  // the forest outlives the fit, unless it is merged or sliced
  if (whole) own = std::make_unique<PoolSuspend>();
  take_forest(*fo, whole ? *std::max_element(per_tree.begin(), per_tree.end()) : 0);
  DTE_HIP(hipMemcpyAsync(fo->tree_start.p, ts.data(), 8 * (T + 1), hipMemcpyHostToDevice, s));
  FinalArgs fa{};
  fa.n_nodes = n_nodes;
  fa.C = C;
  fa.tree = o_tree.p;
  fa.id = o_id.p;
  fa.tree_start = fo->tree_start.p;
  fa.feature = o_feature.p;
  fa.thr = o_thr.p;
  fa.score = o_score.p;
  fa.left = o_left.p;
  fa.depth = o_depth.p;
  fa.count = o_count.p;
  fa.m = o_m.p;
  fa.hash = o_hash.p;
  fa.cls = task == 0 ? o_cls.p : nullptr;
  fa.sum = task == 1 ? o_sum.p : nullptr;
  fa.value = o_value.p;
  fa.f_feature = fo->feature.p;
  fa.f_thr = fo->threshold.p;
  fa.f_score = fo->score.p;
  fa.f_left = fo->left.p;
  fa.f_depth = fo->depth.p;
  fa.f_count = fo->count.p;
  fa.f_m = fo->n_entries.p;
  fa.f_hash = fo->rowhash.p;
  fa.f_cls = fo->class_counts.p;
  fa.f_sum = fo->sum_fixed.p;
  fa.f_value = fo->value.p;
  hipLaunchKernelGGL(k_finalize, dim3(grid_for(n_nodes)), dim3(kBlock), 0, s, fa);
  if (whole) build_predict_nodes(*fo, *std::max_element(per_tree.begin(), per_tree.end()), s);
  DTE_HIP(hipStreamSynchronize(s));
  return fo;
}

// Concatenates tree batches into one forest (the reference's
// AggregateModels, gpudte_algorithm.cc:333-397, on canonical arrays).
Forest* merge_forests(std::vector<std::unique_ptr<Forest>>& parts, hipStream_t s) {
  auto* fo = new Forest();
  std::unique_ptr<Forest> guard(fo);
  const Forest& p0 = *parts[0];
  fo->device = p0.device;
  fo->task = p0.task;
  fo->algorithm = p0.algorithm;
  fo->n_classes = p0.n_classes;
  fo->n_features = p0.n_features;
  fo->fixed_shift = p0.fixed_shift;
  fo->seed = p0.seed;
  fo->tree_offset = p0.tree_offset;
  fo->fit_rows = p0.fit_rows;
  fo->has_stats = true;
  int64_t n = 0;
  int T = 0;
  int64_t leaves = 0;
  for (auto& q : parts) {
    n += q->n_nodes;
    T += q->n_trees;
    leaves = (leaves < 0 || q->n_leaves < 0) ? -1 : leaves + q->n_leaves;
  }
  fo->n_nodes = n;
  fo->n_leaves = leaves;
  fo->n_trees = T;
  const int C = fo->n_classes;
  const size_t W = fo->task == 0 ? (size_t)C : 1;
  PoolSuspend own;  // the forest outlives the fit
  int64_t largest = 1;  // a bound of its largest tree
  for (auto& q : parts) largest = std::max(largest, q->n_nodes);
  take_forest(*fo, largest);
  int64_t off = 0;
  int t_off = 0;
  for (auto& q : parts) {
    const int64_t m = q->n_nodes;
    auto cp = [&](auto* dst, const auto* src, size_t count) {
      DTE_HIP(hipMemcpyAsync(dst, src, sizeof(*src) * count, hipMemcpyDeviceToDevice, s));
    };
    cp(fo->feature.p + off, q->feature.p, m);
    cp(fo->depth.p + off, q->depth.p, m);
    cp(fo->count.p + off, q->count.p, m);
    cp(fo->n_entries.p + off, q->n_entries.p, m);
    cp(fo->threshold.p + off, q->threshold.p, m);
    cp(fo->score.p + off, q->score.p, m);
    cp(fo->value.p + off, q->value.p, m);
    cp(fo->rowhash.p + off, q->rowhash.p, m);
    cp(fo->sum_fixed.p + off, q->sum_fixed.p, m);
    if (fo->task == 0) cp(fo->class_counts.p + off * W, q->class_counts.p, m * W);
    hipLaunchKernelGGL(k_offset_links, dim3(grid_for(m)), dim3(kBlock), 0, s, q->left.p, m, (int32_t)off,
                       fo->left.p + off);
    hipLaunchKernelGGL(k_offset_i64, dim3(grid_for(q->n_trees + 1)), dim3(kBlock), 0, s, q->tree_start.p,
                       (int64_t)q->n_trees + 1, off, fo->tree_start.p + t_off);
    off += m;
    t_off += q->n_trees;
  }
  std::vector<int64_t> ts(T + 1);
  DTE_HIP(hipMemcpyAsync(ts.data(), fo->tree_start.p, 8 * ts.size(), hipMemcpyDeviceToHost, s));
  DTE_HIP(hipStreamSynchronize(s));
  int64_t max_tree = 1;
  for (int t = 0; t < T; ++t) max_tree = std::max(max_tree, ts[t + 1] - ts[t]);
  build_predict_nodes(*fo, max_tree, s);
  DTE_HIP(hipStreamSynchronize(s));
  return guard.release();
}

Forest* fit_forest(const float* X_dev_in, const float* y_host, int64_t N, int32_t F, const dte_params& p,
                   hipStream_t s) {
  PoolScope pool(s);  // the fit's temporaries come from the stream's scratch pool
  FitData fd;
  prepare_data(fd, X_dev_in, y_host, N, F, p, s);
  if (p.build_mode != DTE_BUILD_PLAIN) return fit_batch(fd, p.tree_offset, p.n_trees, N, F, p, s, false);
  std::vector<std::unique_ptr<Forest>> parts;
  for (int t0 = 0; t0 < p.n_trees; t0 += kPlainTrees)
    parts.emplace_back(
        fit_batch(fd, p.tree_offset + t0, std::min(kPlainTrees, p.n_trees - t0), N, F, p, s, true, nullptr,
                  p.n_trees <= kPlainTrees));
  if (parts.size() == 1) return parts[0].release();
  return merge_forests(parts, s);
}

// Node range [off, off + n) of a joint build's forest, as a forest of its
// own: child links relative to the range, class counts narrowed from the
// joint width Cs to the forest's C.
struct SliceArgs {
  int64_t off, n;
  int Cs, C;
  const int32_t *feature, *left, *depth, *count, *m;
  const float *thr, *score, *value;
  const uint64_t* hash;
  const uint32_t* cls;
  const int64_t* sum;
  int32_t *o_feature, *o_left, *o_depth, *o_count, *o_m;
  float *o_thr, *o_score, *o_value;
  uint64_t* o_hash;
  uint32_t* o_cls;
  int64_t* o_sum;
};

__global__ void k_slice_nodes(SliceArgs a) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t g = a.off + i;
    a.o_feature[i] = a.feature[g];
    const int32_t l = a.left[g];
    a.o_left[i] = l < 0 ? -1 : (int32_t)(l - a.off);
    a.o_depth[i] = a.depth[g];
    a.o_count[i] = a.count[g];
    a.o_m[i] = a.m[g];
    a.o_thr[i] = a.thr[g];
    a.o_score[i] = a.score[g];
    a.o_value[i] = a.value[g];
    a.o_hash[i] = a.hash[g];
    a.o_sum[i] = a.sum[g];
    if (a.cls)
      for (int c = 0; c < a.C; ++c) a.o_cls[i * a.C + c] = a.cls[g * a.Cs + c];
  }
}

std::vector<Forest*> fit_joint(const float* const* X, const float* const* y, const int64_t* N, const int32_t* F,
                               const dte_params* ps, int n, hipStream_t s) {
  PoolScope pool(s);
  const bool prof = profiling_enabled();
  auto now = [] { return std::chrono::steady_clock::now(); };
  auto ms = [](std::chrono::steady_clock::time_point a, std::chrono::steady_clock::time_point b) {
    return std::chrono::duration<double, std::milli>(b - a).count();
  };
  const auto h0 = now();
  const int task = ps[0].task;
  std::vector<std::unique_ptr<FitData>> fds(n);
  std::vector<DataArgs> da(n);
  JointSpec J;
  J.C = 1;
  J.D0 = J.R = J.F = 0;
  int T = 0;
  for (int f = 0; f < n; ++f) {
    fds[f] = std::make_unique<FitData>();
    prepare_data(*fds[f], X[f], y[f], N[f], F[f], ps[f], s);
    const int k = ps[f].n_features_per_node > 0 ? ps[f].n_features_per_node
                                                : (int)std::round(std::log((double)F[f])) + 1;
    da[f] = fds[f]->d;
    da[f].D0 = std::min(k, F[f]);
    da[f].R = k < F[f] ? std::min(10, F[f] - k) : 0;
    J.f.push_back(JointForest{fds[f].get(), N[f], F[f], ps[f].n_trees, T, ps[f]});
    T += ps[f].n_trees;
    if (task == 0) J.C = std::max(J.C, ps[f].n_classes);
    J.D0 = std::max(J.D0, da[f].D0);
    J.R = std::max(J.R, da[f].R);
    J.F = std::max(J.F, F[f]);
  }
  for (auto& a : da) a.C = task == 0 ? J.C : 0;  // joint class width in every forest's data
  DevBuf<DataArgs> dforests(n);
  std::vector<int32_t> fot(T);
  for (const JointForest& jf : J.f)
    for (int q = 0; q < jf.T; ++q) fot[jf.t0 + q] = (int32_t)(&jf - J.f.data());
  DevBuf<int32_t> dfot(T);
  DTE_HIP(hipMemcpyAsync(dforests.p, da.data(), sizeof(DataArgs) * n, hipMemcpyHostToDevice, s));
  DTE_HIP(hipMemcpyAsync(dfot.p, fot.data(), 4 * (size_t)T, hipMemcpyHostToDevice, s));
  J.d = da[0];
  J.d.forests = dforests.p;
  J.d.forest_of_tree = dfot.p;
  dte_params pj = ps[0];
  pj.n_trees = T;
  pj.n_classes = task == 0 ? J.C : 0;
  if (prof) {
    DTE_HIP(hipStreamSynchronize(s));
    profile_host("joint_prepare_host", ms(h0, now()));
  }
  const auto h1 = now();
  std::unique_ptr<Forest> all(fit_batch(*fds[0], 0, T, N[0], F[0], pj, s, false, &J, false));
  const auto h2 = now();
  if (prof) profile_host("joint_build_host", ms(h1, h2));
  // one forest per input, from its trees' node range
  std::vector<int64_t> ts(T + 1);
  DTE_HIP(hipMemcpyAsync(ts.data(), all->tree_start.p, 8 * (size_t)(T + 1), hipMemcpyDeviceToHost, s));
  DTE_HIP(hipStreamSynchronize(s));
  std::vector<std::unique_ptr<Forest>> out;
  PoolSuspend own;  // the forests outlive the fit
  for (const JointForest& jf : J.f) {
    const int64_t off = ts[jf.t0], nn = ts[jf.t0 + jf.T] - off;
    const int Cf = task == 0 ? jf.p.n_classes : 1;
    auto fo = std::make_unique<Forest>();
    fo->device = all->device;
    fo->task = task;
    fo->algorithm = all->algorithm;
    fo->n_classes = Cf;
    fo->n_features = jf.F;
    fo->n_trees = jf.T;
    fo->fixed_shift = jf.fd->shift;
    fo->seed = jf.p.seed;
    fo->tree_offset = jf.p.tree_offset;
    fo->fit_rows = 0;  // extra trees: no bootstrap record
    fo->n_nodes = nn;
    fo->n_leaves = (nn + jf.T) / 2;
    fo->has_stats = true;
    std::vector<int64_t> tsf(jf.T + 1);
    int64_t max_tree = 1;
    for (int q = 0; q <= jf.T; ++q) {
      tsf[q] = ts[jf.t0 + q] - off;
      if (q) max_tree = std::max(max_tree, tsf[q] - tsf[q - 1]);
    }
    take_forest(*fo, max_tree);
    DTE_HIP(hipMemcpyAsync(fo->tree_start.p, tsf.data(), 8 * (size_t)(jf.T + 1), hipMemcpyHostToDevice, s));
    SliceArgs sa{off, nn, all->n_classes, task == 0 ? Cf : 0,
                 all->feature.p, all->left.p, all->depth.p, all->count.p, all->n_entries.p,
                 all->threshold.p, all->score.p, all->value.p, all->rowhash.p,
                 task == 0 ? all->class_counts.p : nullptr, all->sum_fixed.p,
                 fo->feature.p, fo->left.p, fo->depth.p, fo->count.p, fo->n_entries.p,
                 fo->threshold.p, fo->score.p, fo->value.p, fo->rowhash.p, fo->class_counts.p, fo->sum_fixed.p};
    hipLaunchKernelGGL(k_slice_nodes, dim3(grid_for(nn)), dim3(kBlock), 0, s, sa);
    build_predict_nodes(*fo, max_tree, s);
    DTE_HIP(hipStreamSynchronize(s));  // tsf goes out of scope
    out.push_back(std::move(fo));
  }
  all.reset();
  if (prof) profile_host("joint_split_host", ms(h2, now()));
  std::vector<Forest*> res;
  for (auto& f : out) res.push_back(f.release());
  return res;
}

}  // namespace dte
