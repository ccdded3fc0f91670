// Forest traversal for MI355X.  Replaces gpudte_predict (lib_ensembles/
// source/gpudte.cu:311-359) and the host launch loop of
// GpuDteAlgorithm<T>::Predict (gpudte_algorithm.cc:292-311):
//
//  * nodes are 8-byte records, siblings side by side, a tree's top levels in
//    level order and below them three levels of a subtree in one cache line
//    (build_predict_nodes);
//  * classification: every (row, tree) pair is walked exactly once (FIX of
//    the truncated grid, gpudte_algorithm.cc:297-305) and votes are integer
//    sums, so the result is order-free;
//  * regression: every row's trees are summed in tree order (fixed fp32
//    order instead of float atomics, gpudte.cu:354-357).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "dte_internal.h"
#include "dte_limits.h"

namespace dte {
namespace {

constexpr int kWave = 64;
// Threads of a walk block.  Eight waves a block's rows in LDS keep the CU full
// where a block's LDS holds it to four; but a block walks as many trees at once
// as a row has lanes, and what its CU's neighbours miss grows with them.  Models
// past the caches (kBigModel) under many row blocks (kManyBlocks, where blocks
// start at different times and drift over all trees) take four: 1M x 128, 64
// trees of 300,000 nodes 4.65 ms at 512 threads, 3.8 at 256; 200 trees 17.1 and
// 12.9; 400 trees 37.8 and 28.5.  The other side of the line: 300,000 x 128, 64
// trees of 83,000 nodes 0.86 and 0.88; 100,000 x 128, 64 trees of 230,000 nodes
// 0.39 and 0.40; 300,000 x 128, 200 trees of 1,700 nodes 0.82 and 1.27.
constexpr int kWalkThreads = 512;
constexpr int kBigWalkThreads = 256;
constexpr int64_t kBigModel = (int64_t)6 << 20;  // nodes
constexpr int64_t kManyBlocks = 4096;
// Row blocks of a launch: it holds fewer than 2^32 threads in a direction.
// More rows (537 M at 64 a block) take several launches.
constexpr int64_t kMaxRowBlocks = 0xFFFFFFFFll / kWalkThreads;

// ------------------------------------------------------ node layout ----
// Bound by read requests of the deep levels: a scattered read that misses the
// L2 brings a 64-byte half of a line, and the fabric passes 45 to 55 G of them
// a second (single words at random, one a line or one a half line: 48 G/s).
// Below kTopLevels a tree's pairs are grouped by clusters of three levels --
// the pair below a node at depth 9, 12, .. and up to six pairs below it, 16 B
// each -- in slots of 1, 2, 4 or 8 pairs aligned to their size, so that a
// cluster never straddles a 128-byte line and a walk takes one or two half
// lines per three levels.  1M x 128, trees of 300,000 nodes: 2.7 requests a
// walk with 64 trees and 2.9 with 200, at 45 G/s (16-byte records in level
// order 4.5 and 3.1, at 51 and 39 G/s).  The top levels stay in the caches
// whatever their order; there the lines that the 64 rows of a wave touch in
// one step count, fewest in level order.  600,000 rows x 6, 64 trees of 8,000
// nodes: 0.69 ms with 16-byte records, 0.81 clustered from the root, 0.64 like
// this; 1M x 128, 64 trees of 300,000 nodes: 5.2, 4.1, 4.1 ms at 512 threads
// a block, 3.7 like this at 256.
constexpr int kClusterLevels = 3;
constexpr int kTopLevels = 9;  // a multiple of kClusterLevels

// Pair of the children of a node above kTopLevels: the tree's pairs in level
// order behind the root's (canonical order is level order, so the children of
// the tree's k-th internal node are its nodes 2k - 1 and 2k).
__device__ __forceinline__ uint32_t top_pair(int64_t first, int64_t tree_start) {
  return 1u + (uint32_t)((first - tree_start - 1) >> 1);
}

// Slot class of a cluster of s pairs: 2^class slots of a pair.
__device__ __forceinline__ int slot_class(int s) { return s <= 1 ? 0 : s <= 2 ? 1 : s <= 4 ? 2 : 3; }

// Tree of canonical node g.
__device__ __forceinline__ int tree_of(int64_t g, int T, const int64_t* __restrict__ ts) {
  int lo = 0, hi = T - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (ts[mid] <= g) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// The pairs of a cluster, by their first nodes (-1: not there): the head pair,
// the pairs below its two nodes, and the pairs below those.
struct Cluster {
  int32_t head, mid[2], low[4];
  int n;  // pairs
};
__device__ __forceinline__ Cluster cluster_at(int32_t head, const int32_t* __restrict__ feature,
                                              const int32_t* __restrict__ left) {
  Cluster c;
  c.head = head;
  c.n = 1;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    c.mid[k] = feature[head + k] >= 0 ? left[head + k] : -1;
    c.n += c.mid[k] >= 0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      c.low[2 * k + j] = c.mid[k] >= 0 && feature[c.mid[k] + j] >= 0 ? left[c.mid[k] + j] : -1;
      c.n += c.low[2 * k + j] >= 0;
    }
  }
  return c;
}

// From kTopLevels on, every internal node at a depth divisible by three heads
// the cluster of its children: its slot class and number among the tree's
// clusters of that class.
__global__ void __launch_bounds__(kBlock) k_cluster_count(int64_t n, int T, const int64_t* __restrict__ ts,
                                                          const int32_t* __restrict__ feature,
                                                          const int32_t* __restrict__ left,
                                                          const int32_t* __restrict__ depth, uint32_t* code,
                                                          unsigned int* cnt) {
  // Slots are taken kCountPer nodes a thread at a time, with one atomic
  // instruction for the workgroup's first tree: an atomic per wave and class
  // took 0.2 ms for 50 trees of 2.6 M nodes, whose counters share seven lines
  // before).
  constexpr int kCountPer = 8;
  __shared__ unsigned int s_cnt[4], s_base[4];
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1);
  const uint64_t below = (1ull << lane) - 1ull;
  for (int64_t c0 = blockIdx.x * (int64_t)(kBlock * kCountPer); c0 < n; c0 += (int64_t)gridDim.x * (kBlock * kCountPer)) {
    const int tree0 = tree_of(c0, T, ts);
    const int64_t end0 = ts[tree0 + 1];
    if (t < 4) s_cnt[t] = 0;
    __syncthreads();
    int cls[kCountPer];
    int32_t first[kCountPer];
    unsigned int at[kCountPer], run[4] = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < kCountPer; ++q) {
      const int64_t g = c0 + q * kBlock + t;
      cls[q] = -1;
      first[q] = 0;
      if (g < n && feature[g] >= 0 && depth[g] >= kTopLevels && depth[g] % kClusterLevels == 0) {
        first[q] = left[g];
        cls[q] = slot_class(cluster_at(first[q], feature, left).n);
        if (cls[q] >= 0 && g >= end0) {  // a later tree's
          code[first[q]] = atomicAdd(&cnt[4 * (int64_t)tree_of(g, T, ts) + cls[q]], 1u) * 4u + (unsigned)cls[q];
          cls[q] = -1;
        }
      }
      at[q] = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint64_t same = __ballot(cls[q] == k);
        if (cls[q] == k) at[q] = run[k] + (unsigned int)__popcll(same & below);
        run[k] += (unsigned int)__popcll(same);
      }
    }
    unsigned int wave0[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      unsigned int b = 0;
      if (lane == 0 && run[k]) b = atomicAdd(&s_cnt[k], run[k]);
      wave0[k] = (unsigned int)__shfl((int)b, 0, kWave);
    }
    __syncthreads();
    if (t < 4) s_base[t] = s_cnt[t] ? atomicAdd(&cnt[4 * (int64_t)tree0 + t], s_cnt[t]) : 0u;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kCountPer; ++q)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (cls[q] == k) code[first[q]] = (s_base[k] + wave0[k] + at[q]) * 4u + (unsigned)k;
    __syncthreads();  // s_cnt is cleared, s_base rewritten
  }
}
__global__ void __launch_bounds__(kBlock) k_cluster_bases(int T, const int64_t* __restrict__ ts,
                                                          const int32_t* __restrict__ depth,
                                                          const unsigned int* __restrict__ cnt,
                                                          int64_t* __restrict__ tbase,
                                                          uint32_t* __restrict__ cbase) {
  __shared__ int64_t s_sum[kBlock];
  const int t = threadIdx.x;
  int64_t run = 0;
  for (int t0 = 0; t0 < T; t0 += kBlock) {
    const int i = t0 + t;
    int64_t size = 0;
    if (i < T) {
      const unsigned int* c = cnt + 4 * (int64_t)i;
      // nodes of the top levels: a prefix of the tree
      int64_t lo = ts[i], hi = ts[i + 1];
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (depth[mid] <= kTopLevels) lo = mid + 1;
        else hi = mid;
      }
      uint32_t at = (1u + (uint32_t)((lo - ts[i]) >> 1) + 7u) & ~7u;
      cbase[4 * (int64_t)i + 3] = at;
      at += 8u * c[3];
      cbase[4 * (int64_t)i + 2] = at;
      at += 4u * c[2];
      cbase[4 * (int64_t)i + 1] = at;
      at += 2u * c[1];
      cbase[4 * (int64_t)i] = at;
      at += c[0];
      size = (at + 7u) & ~7u;
    }
    s_sum[t] = size;
    __syncthreads();
    for (int off = 1; off < kBlock; off <<= 1) {
      const int64_t v = t >= off ? s_sum[t - off] : 0;
      __syncthreads();
      s_sum[t] += v;
      __syncthreads();
    }
    if (i < T) tbase[i] = run + s_sum[t] - size;
    run += s_sum[kBlock - 1];
    __syncthreads();
  }
}

// vote = argmax, strict > from 0: lowest class on ties (gpudte.cu:341-351)
__device__ __forceinline__ int vote_of(const uint32_t* __restrict__ cls, int C) {
  int best = 0;
  uint32_t bv = 0;
  for (int c = 0; c < C; ++c)
    if (cls[c] > bv) {
      bv = cls[c];
      best = c;
    }
  return best;
}

// Record of node g: (threshold, link) or, for a leaf, (payload, 0); link =
// pair of the children << fbits | feature + 1.
__device__ __forceinline__ uint2 leaf_record(int64_t g, int C, int task, const uint32_t* __restrict__ cls,
                                             const float* __restrict__ value) {
  return make_uint2(task == 0 ? (uint32_t)vote_of(cls + g * C, C) : __float_as_uint(value[g]), 0u);
}

__global__ void __launch_bounds__(kBlock) k_cluster_write(int64_t n, int T, const int64_t* __restrict__ ts,
                                                          const int32_t* __restrict__ feature,
                                                          const int32_t* __restrict__ left,
                                                          const int32_t* __restrict__ depth,
                                                          const float* __restrict__ thr,
                                                          const uint32_t* __restrict__ cls,
                                                          const float* __restrict__ value, int C, int task, int fbits,
                                                          const uint32_t* __restrict__ code,
                                                          const int64_t* __restrict__ tbase,
                                                          const uint32_t* __restrict__ cbase, uint4* __restrict__ out) {
  for (int64_t g = blockIdx.x * (int64_t)kBlock + threadIdx.x; g < n; g += (int64_t)gridDim.x * kBlock) {
    const int32_t dg = depth[g];
    if (dg >= kTopLevels && dg % kClusterLevels != 0) continue;
    const int32_t f = feature[g];
    const bool root = dg == 0;
    if (f < 0 && !root) continue;
    const int t = tree_of(g, T, ts);
    const uint32_t* cb = cbase + 4 * (int64_t)t;
    uint4* tree = out + tbase[t];
    if (root) {
      const uint2 r = f < 0 ? leaf_record(g, C, task, cls, value)
                            : make_uint2(__float_as_uint(thr[g]), 1u << fbits | (uint32_t)(f + 1));
      tree[0] = make_uint4(r.x, r.y, 0u, 0u);
      if (f < 0) continue;
    }
    auto slot = [&](int32_t first) { return cb[code[first] & 3u] + ((code[first] >> 2) << (code[first] & 3u)); };
    auto record = [&](int32_t i, uint32_t child) {
      const int32_t cf = feature[i];
      return cf < 0 ? leaf_record(i, C, task, cls, value)
                    : make_uint2(__float_as_uint(thr[i]), child << fbits | (uint32_t)(cf + 1));
    };
    auto put = [&](uint32_t where, uint2 l, uint2 r) { tree[where] = make_uint4(l.x, l.y, r.x, r.y); };
    if (dg < kTopLevels) {
      const int32_t h = left[g];
      auto below = [&](int32_t i) -> uint32_t {  // pair of a child's children
        if (feature[i] < 0) return 0u;
        return dg + 1 < kTopLevels ? top_pair(left[i], ts[t]) : slot(left[i]);
      };
      put(top_pair(h, ts[t]), record(h, below(h)), record(h + 1, below(h + 1)));
      continue;
    }
    const Cluster c = cluster_at(left[g], feature, left);
    const uint32_t at = slot(c.head);
    // breadth-first places of the pairs in the cluster's slots
    uint32_t next = at + 1u, mid[2], low[4];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      mid[k] = next;
      next += c.mid[k] >= 0;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      low[k] = next;
      next += c.low[k] >= 0;
    }
    put(at, record(c.head, mid[0]), record(c.head + 1, mid[1]));
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (c.mid[k] >= 0) put(mid[k], record(c.mid[k], low[2 * k]), record(c.mid[k] + 1, low[2 * k + 1]));
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (c.low[k] >= 0) {  // below it: heads of other clusters
        const int32_t i = c.low[k];
        put(low[k], record(i, feature[i] >= 0 ? slot(left[i]) : 0u),
            record(i + 1, feature[i + 1] >= 0 ? slot(left[i + 1]) : 0u));
      }
  }
}

// Canonical order, 16-byte records: trees too large for a link of 32 bits.
__global__ void __launch_bounds__(kBlock) k_wide_nodes(int64_t n, int C, int task, const int32_t* feature,
                                                       const float* thr, const int32_t* left, const uint32_t* cls,
                                                       const float* value, PNode* out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    PNode p;
    p.feature = feature[i];
    p.pad = 0;
    if (p.feature >= 0) {
      p.thr = __float_as_uint(thr[i]);
      p.left = left[i];
    } else {
      p.thr = leaf_record(i, C, task, cls, value).x;
      p.left = 0;
    }
    out[i] = p;
  }
}

// ------------------------------------------------------------- walks ----
struct Trees {
  const uint4* pairs;        // packed: sibling pairs
  const int64_t* tbase;      // packed: first pair of each tree
  int fbits;
  const PNode* wide;         // wide: canonical records
  const int64_t* tree_start;
  int T;
};

// Leaf payload of a row in tree t: its values at xr[feature * xs].  visit(f,
// depth, &x) may replace the value read.
template <bool PACKED, class Visit>
__device__ __forceinline__ uint32_t walk(const Trees& tr, int t, const float* xr, int64_t xs, Visit&& visit) {
  uint32_t depth = 0;
  if constexpr (PACKED) {
    const uint4* tree = tr.pairs + tr.tbase[t];
    const uint32_t fmask = (1u << tr.fbits) - 1u;
    uint2 nd = *reinterpret_cast<const uint2*>(tree);
    while (nd.y & fmask) {
      const int f = (int)(nd.y & fmask) - 1;
      float x = xr[f * xs];
      visit(f, depth, x);
      // the child alone: the pair in flight beside the feature value takes
      // twice the lanes' share of the L1 (regression 600,000 x 6, 64 trees:
      // 0.36 ms with the pair, 0.33 with the child)
      const uint2* kids = reinterpret_cast<const uint2*>(tree + (nd.y >> tr.fbits));
      nd = kids[side_of(x, __uint_as_float(nd.x))];
      ++depth;
    }
    return nd.x;
  } else {
    PNode nd = tr.wide[tr.tree_start[t]];
    while (nd.feature >= 0) {
      float x = xr[nd.feature * xs];
      visit(nd.feature, depth, x);
      nd = tr.wide[(int64_t)nd.left + side_of(x, __uint_as_float(nd.thr))];
      ++depth;
    }
    return nd.thr;
  }
}

// Stages a block's R rows of F features in LDS, F + 1 floats apart.
template <int R, int NT>
__device__ __forceinline__ void stage_rows(const float* __restrict__ X, int64_t row0, int nr, int64_t ld,
                                           int row_major, int F, float* s_x) {
  const int FP = F + 1;
  if (row_major) {
    for (int i = threadIdx.x; i < nr * F; i += NT) {
      const int r = i / F, f = i - r * F;
      s_x[r * FP + f] = X[(row0 + r) * ld + f];
    }
  } else {
    for (int i = threadIdx.x; i < R * F; i += NT) {
      const int f = i / R, r = i - f * R;
      if (r < nr) s_x[r * FP + f] = X[(int64_t)f * ld + row0 + r];
    }
  }
}

// What a block does with its votes: it adds them to others' (several tree
// chunks), or it alone covers its rows' trees and stores them.
enum VoteMode { kVoteAdd = 0, kVoteInt = 1, kVoteFloat = 2 };

// A block's R rows x (NT / R) tree lanes; R = 0: rows read from X, 64 rows
// x NT / 64 tree lanes.
template <int R, bool PACKED, int NT>
__global__ void __launch_bounds__(NT) k_predict_cls(Trees tr, const float* __restrict__ X, int64_t n_rows,
                                                              int64_t ld, int row_major, int C, int F,
                                                              int trees_per_block, int mode, void* __restrict__ out) {
  extern __shared__ uint32_t s_mem[];
  constexpr int RB = R ? R : 64;
  uint32_t* s_votes = s_mem;                              // RB * C
  float* s_x = reinterpret_cast<float*>(s_mem + RB * C);  // R rows of F + 1 floats
  const int lane = threadIdx.x % RB;
  const int group = threadIdx.x / RB;
  const int64_t row0 = (int64_t)blockIdx.x * RB;
  const int nr = (int)min<int64_t>(RB, n_rows - row0);
  const int t0 = blockIdx.y * trees_per_block;
  const int t1 = min(tr.T, t0 + trees_per_block);
  for (int i = threadIdx.x; i < RB * C; i += NT) s_votes[i] = 0;
  if (R) stage_rows<RB, NT>(X, row0, nr, ld, row_major, F, s_x);
  __syncthreads();
  if (lane < nr) {
    const float* xr = R ? s_x + lane * (F + 1) : row_major ? X + (row0 + lane) * ld : X + row0 + lane;
    const int64_t xs = R || row_major ? 1 : ld;
    for (int t = t0 + group; t < t1; t += NT / RB)
      atomicAdd(&s_votes[lane * C + walk<PACKED>(tr, t, xr, xs, [](int, uint32_t, float&) {})], 1u);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nr * C; i += NT) {
    const uint32_t v = s_votes[i];
    const int64_t o = row0 * C + i;
    if (mode == kVoteFloat) {
      static_cast<float*>(out)[o] = (float)v;
    } else if (mode == kVoteInt) {
      static_cast<int32_t*>(out)[o] = (int32_t)v;
    } else if (v) {
      atomicAdd(static_cast<int32_t*>(out) + o, (int32_t)v);
    }
  }
}

// Regression: trees go in chunks of as many as the block has tree lanes (at
// least 32); the lanes of a row write the chunk's leaf values to LDS, then
// one lane per row adds them in tree order, so every row's sum is formed in
// that order whatever R is.
constexpr int reg_chunk(int R) { return kWalkThreads / (R ? R : 64) > 32 ? kWalkThreads / (R ? R : 64) : 32; }

template <int R, bool PACKED, int NT>
__global__ void __launch_bounds__(NT) k_predict_reg(Trees tr, const float* __restrict__ X, int64_t n_rows,
                                                              int64_t ld, int row_major, int F,
                                                              float* __restrict__ sums) {
  extern __shared__ float s_mem_f[];
  constexpr int RB = R ? R : 64;
  constexpr int CH = reg_chunk(R);
  float* s_val = s_mem_f;              // RB x CH leaf values, CH + 1 apart
  float* s_x = s_mem_f + RB * (CH + 1);  // R rows of F + 1 floats
  const int lane = threadIdx.x % RB;
  const int group = threadIdx.x / RB;
  const int64_t row0 = (int64_t)blockIdx.x * RB;
  const int nr = (int)min<int64_t>(RB, n_rows - row0);
  if (R) stage_rows<RB, NT>(X, row0, nr, ld, row_major, F, s_x);
  __syncthreads();
  const float* xr = R ? s_x + lane * (F + 1) : row_major ? X + (row0 + lane) * ld : X + row0 + lane;
  const int64_t xs = R || row_major ? 1 : ld;
  float acc = 0.0f;
  for (int c0 = 0; c0 < tr.T; c0 += CH) {
    const int c1 = min(tr.T, c0 + CH);
    if (lane < nr)
      for (int t = c0 + group; t < c1; t += NT / RB)
        s_val[lane * (CH + 1) + (t - c0)] = __uint_as_float(walk<PACKED>(tr, t, xr, xs, [](int, uint32_t, float&) {}));
    __syncthreads();
    if (group == 0 && lane < nr)
      for (int t = c0; t < c1; ++t) acc = acc + s_val[lane * (CH + 1) + (t - c0)];
    __syncthreads();
  }
  if (group == 0 && lane < nr) sums[row0 + lane] = acc;
}

// ---------------------------------------------------- out-of-bag pass --
// Stream of the per-visit row draws of the permutation pass.
constexpr uint32_t kStreamImp = 0x00706d69u;

// In-bag bits: bit r of tree t is set iff tree t's bootstrap drew row r
// (the draws of the fit's bootstrap, k_boot_count).  One workgroup per
// (tree, range of kBagRange rows): every draw of the tree is generated, the
// range's bits are set in LDS and written out once.
constexpr int kBagThreads = 1024;
// Workgroups beside each other on a tree's draws, so that few trees fill the
// chip (100 trees of 200,003 rows: 0.115 ms at one workgroup a tree, 0.05 ms at five);
// with several, each adds its bits to words that start at zero.
__global__ void __launch_bounds__(kBagThreads) k_inbag_bits_lds(uint32_t* bits, int64_t N, int64_t words,
                                                                int32_t tree0, uint64_t seed) {
  extern __shared__ uint32_t s_bits[];
  const int t = blockIdx.x;
  const int64_t r0 = (int64_t)blockIdx.y * kBagRange;
  const int64_t nw = (min(kBagRange, N - r0) + 31) / 32;  // words of this range
  const int64_t per = (N + gridDim.z - 1) / gridDim.z;
  const int64_t i0 = blockIdx.z * per, i1 = min(N, i0 + per);
  for (int64_t w = threadIdx.x; w < nw; w += kBagThreads) s_bits[w] = 0;
  __syncthreads();
  const uint32_t tg = (uint32_t)(tree0 + t);
  for (int64_t i = i0 + threadIdx.x; i < i1; i += kBagThreads) {
    const int64_t r = (int64_t)(rand_u32(seed, kStreamBoot, tg, 0, (uint64_t)i) % (uint32_t)N) - r0;
    if (r >= 0 && r < kBagRange) atomicOr(&s_bits[r >> 5], 1u << (r & 31));
  }
  __syncthreads();
  uint32_t* bt = bits + (int64_t)t * words + r0 / 32;
  for (int64_t w = threadIdx.x; w < nw; w += kBagThreads) {
    const uint32_t v = s_bits[w];
    if (gridDim.z == 1) bt[w] = v;
    else if (v) atomicOr(&bt[w], v);
  }
}

// Every (tree, row) pair whose row is out of the tree's bag is routed
// through the tree (gpurf.cu:290-353); with perm >= 0, nodes that split on
// feature perm read the value of row draw % N instead, one counter-based
// draw per visit keyed by (tree, row, depth) (gpurf.cu:356-438).
// Classification counts the pairs whose tree vote equals the label;
// regression sums the squared errors of the leaf values.
//
// A block's R rows are staged in LDS (R = 0: 64 rows read from X); the
// permuted feature always reads its drawn row from X.  The block lists the
// pairs of its rows and kOobChunk trees that are out of the bag and deals them
// to its threads: with a row and a share of the trees to each lane, 63 % of the
// lanes stood idle.  Every block adds its counts once, to one of kOobSlots
// lines: a wave's atomics on one line pass at one in about 15 ns, and 50,000 of
// them were most of the 0.88 ms that 200,003 rows x 96 and 100 trees took
// before; 0.51 ms now).
constexpr int kOobChunk = 64;
constexpr int kOobSlots = 64;
struct alignas(128) OobSlot {
  unsigned long long pairs, right, bad;  // bad: labels that are no class
  double sse;
};

template <int TASK, int R, bool PACKED>
__global__ void __launch_bounds__(kWalkThreads) k_oob(Trees tr, const float* __restrict__ X, int64_t N, int F,
                                                      const uint32_t* __restrict__ bits, int64_t words,
                                                      const float* __restrict__ y, int n_classes, int32_t tree0,
                                                      uint64_t seed, int perm, int trees_per_block,
                                                      int64_t block0, OobSlot* slots) {
  extern __shared__ float s_x[];  // R rows of F + 1 floats
  constexpr int RB = R ? R : 64;
  constexpr int NW = kWalkThreads / kWave;
  __shared__ uint16_t s_pair[RB * kOobChunk];  // row | tree of the chunk << 6
  __shared__ float s_y[RB];
  __shared__ unsigned int s_n;
  __shared__ unsigned long long s_right[NW], s_bad;
  __shared__ double s_sse[NW];
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1);
  const int64_t row0 = (block0 + blockIdx.x) * RB;
  const int nr = (int)min<int64_t>(RB, N - row0);
  const int t0 = blockIdx.y * trees_per_block;
  const int t1 = min(tr.T, t0 + trees_per_block);
  if (R) stage_rows<RB, kWalkThreads>(X, row0, nr, N, 0, F, s_x);
  if (t < kWave) {
    const float yr = t < nr ? y[row0 + t] : 0.0f;
    if (t < RB) s_y[t] = yr;
    const bool bad = TASK == 0 && t < nr && !(yr >= 0.0f && yr < (float)n_classes && truncf(yr) == yr);
    const uint64_t b = __ballot(bad);
    if (t == 0) s_bad = blockIdx.y == 0 ? __popcll(b) : 0;
  }
  unsigned long long n_pairs = 0, n_ok = 0;
  double e2 = 0.0;
  for (int c0 = t0; c0 < t1; c0 += kOobChunk) {
    __syncthreads();  // the last chunk's list is read no more
    if (t == 0) s_n = 0;
    __syncthreads();
    const int want = min(kOobChunk, t1 - c0) * RB;
    for (int x0 = 0; x0 < want; x0 += kWalkThreads) {
      const int x = x0 + t, row = x % RB, tc = x / RB;
      const int64_t r = row0 + row;
      const bool out = x < want && row < nr &&
                       !((bits[(int64_t)(c0 + tc) * words + (r >> 5)] >> (r & 31)) & 1u);
      const uint64_t b = __ballot(out);
      unsigned int at = 0;
      if (lane == 0 && b) at = atomicAdd(&s_n, (unsigned int)__popcll(b));
      at = (unsigned int)__shfl((int)at, 0, kWave);
      if (out) s_pair[at + (unsigned int)__popcll(b & ((1ull << lane) - 1ull))] = (uint16_t)(row | tc << 6);
    }
    __syncthreads();
    const int n = (int)s_n;
    n_pairs += (unsigned long long)n;
    for (int p = t; p < n; p += kWalkThreads) {
      const int row = s_pair[p] & 63, tree = c0 + (s_pair[p] >> 6);
      const int64_t r = row0 + row;
      const float* xr = R ? s_x + row * (F + 1) : X + r;
      const uint32_t tg = (uint32_t)(tree0 + tree);
      const uint32_t leaf = walk<PACKED>(tr, tree, xr, R ? 1 : N, [&](int f, uint32_t depth, float& x) {
        if (f == perm)
          x = X[(int64_t)perm * N + rand_u32(seed, kStreamImp, tg, (uint32_t)r, depth) % (uint32_t)N];
      });
      if (TASK == 0) {
        n_ok += (float)leaf == s_y[row] ? 1ull : 0ull;
      } else {
        const double e = (double)__uint_as_float(leaf) - (double)s_y[row];
        e2 += e * e;
      }
    }
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    n_ok += __shfl_xor(n_ok, off, kWave);
    if (TASK == 1) e2 += __shfl_xor(e2, off, kWave);
  }
  if (lane == 0) {
    s_right[t / kWave] = n_ok;
    s_sse[t / kWave] = e2;
  }
  __syncthreads();
  if (t == 0) {
    for (int w = 1; w < NW; ++w) {
      n_ok += s_right[w];
      e2 += s_sse[w];
    }
    OobSlot& o = slots[blockIdx.x % kOobSlots];
    if (n_pairs) atomicAdd(&o.pairs, n_pairs);
    if (n_ok) atomicAdd(&o.right, n_ok);
    if (s_bad) atomicAdd(&o.bad, s_bad);
    if (TASK == 1 && n_pairs) atomicAdd(&o.sse, e2);
  }
}

__global__ void __launch_bounds__(kBlock) k_zero_u32(uint32_t* __restrict__ p, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) p[i] = 0u;
}

__global__ void __launch_bounds__(kBlock) k_votes_to_float(int32_t* __restrict__ p, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
    const float v = (float)p[i];
    reinterpret_cast<float*>(p)[i] = v;
  }
}

// ------------------------------------------------------------ export --
// Export order: the roots, then every tree's other nodes in level order
// (gpudte_algorithm.cc:349-357).  Canonical node g of tree t, not its root,
// is export node T + g - t - 1.
__device__ __forceinline__ int64_t export_to_canonical(int64_t e, int T, const int64_t* __restrict__ ts, int* tree) {
  if (e < T) {
    *tree = (int)e;
    return ts[e];
  }
  // the last tree whose first non-root export node, T + ts[t] - t, is at most e
  int lo = 0, hi = T - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (T + ts[mid] - mid <= e) lo = mid;
    else hi = mid - 1;
  }
  *tree = lo;
  return e - T + lo + 1;
}

__global__ void __launch_bounds__(kBlock) k_export_leaves(int64_t n, int T, const int64_t* __restrict__ ts,
                                                          const int32_t* __restrict__ feature, uint32_t* flag) {
  for (int64_t e = blockIdx.x * (int64_t)kBlock + threadIdx.x; e < n; e += (int64_t)gridDim.x * kBlock) {
    int t;
    flag[e] = feature[export_to_canonical(e, T, ts, &t)] < 0 ? 1u : 0u;
  }
}

// Records and leaf payloads of export nodes [e0, e1); pos[e] = leaves before e.
// level_order: children lie in their parents' trees (else a tree's root may be
// another tree's child).
__global__ void __launch_bounds__(kBlock) k_export(int64_t e0, int64_t e1, int T, const int64_t* __restrict__ ts,
                                                   const int32_t* __restrict__ feature,
                                                   const int32_t* __restrict__ left, const float* __restrict__ thr,
                                                   const float* __restrict__ value,
                                                   const uint32_t* __restrict__ cls, int P, bool level_order,
                                                   const uint32_t* __restrict__ pos, dte_node* __restrict__ nodes,
                                                   float* __restrict__ probs) {
  const uint32_t p0 = pos[e0];
  for (int64_t e = e0 + blockIdx.x * (int64_t)kBlock + threadIdx.x; e < e1; e += (int64_t)gridDim.x * kBlock) {
    int t;
    const int64_t g = export_to_canonical(e, T, ts, &t);
    dte_node d;
    const int32_t f = feature[g];
    if (f >= 0) {
      const int64_t l = left[g];
      const int lt = level_order ? t : tree_of(l, T, ts);
      d.child_start = !level_order && l == ts[lt] ? lt : (int32_t)(T + l - lt - 1);
      d.child_count = 2;
      d.probability_start = -1;
      d.attribute = f;
      d.split_point = thr[g];
    } else {
      const int64_t at = (int64_t)pos[e] * P;
      d.child_start = -1;
      d.child_count = 0;
      d.probability_start = (int32_t)at;
      d.attribute = -1;
      d.split_point = -1.0f;
      float* o = probs + (at - (int64_t)p0 * P);
      if (cls)
        for (int c = 0; c < P; ++c) o[c] = (float)cls[g * P + c];
      else
        o[0] = value[g];
    }
    nodes[e - e0] = d;
  }
}

unsigned elementwise_grid(int64_t n) { return (unsigned)std::min<int64_t>((n + kBlock - 1) / kBlock, 4096); }

// Rows per block of the walk kernels: 64 (32, 16) while the block's rows and
// `per_row` more words each fit 48 KB of LDS, else 0 (rows read from HBM).
// Few rows take fewer per block, so that a wave's lanes spread over trees.
int staged_rows(int F, int per_row, int64_t n_rows) {
  auto fits = [&](int r) { return (int64_t)4 * r * ((int64_t)F + 1 + per_row) <= 48 * 1024; };
  if (n_rows <= 2 && fits(1)) return 1;
  if (n_rows <= 16 && fits(4)) return 4;
  if (n_rows <= 128 && fits(16)) return 16;
  return fits(64) ? 64 : fits(32) ? 32 : 0;
}

// Tree chunks so that row blocks x chunks fill the chip even for few rows: a
// chunk keeps at least two trees per tree lane.
int tree_chunks(int64_t row_blocks, int n_trees, int lanes) {
  int chunks = 1;
  while (row_blocks * chunks < 1024 && (int64_t)chunks * 4 * lanes <= n_trees) chunks *= 2;
  return chunks;
}

Trees trees_of(const Forest& f) {
  return Trees{reinterpret_cast<const uint4*>(f.pairs.p), f.pair_base.p, f.pair_fbits, f.pnodes.p, f.tree_start.p,
               f.n_trees};
}

// fn(integral_constant R, integral_constant PACKED) for the rows per block r.
template <class Fn>
void with_rows(int r, bool packed, Fn&& fn) {
  auto go = [&](auto R) {
    if (packed) fn(R, std::true_type());
    else fn(R, std::false_type());
  };
  switch (r) {
    case 64: go(std::integral_constant<int, 64>()); break;
    case 32: go(std::integral_constant<int, 32>()); break;
    case 16: go(std::integral_constant<int, 16>()); break;
    case 4: go(std::integral_constant<int, 4>()); break;
    case 1: go(std::integral_constant<int, 1>()); break;
    default: go(std::integral_constant<int, 0>()); break;
  }
}

// The same with integral_constant NT for a prediction of row_blocks blocks of r
// rows (fewer than 32: few blocks).
template <class Fn>
void with_walk(const Forest& f, int r, int64_t row_blocks, Fn&& fn) {
  const bool big = f.n_nodes >= kBigModel && row_blocks >= kManyBlocks;
  with_rows(r, f.pairs.p != nullptr, [&](auto R, auto packed) {
    constexpr int kR = decltype(R)::value;
    if constexpr (kR == 0 || kR >= 32) {
      if (big) {
        fn(R, packed, std::integral_constant<int, kBigWalkThreads>());
        return;
      }
    }
    fn(R, packed, std::integral_constant<int, kWalkThreads>());
  });
}

}  // namespace

void oob_evaluate(const Forest& f, const float* X, const float* targets, int64_t N, int perm, double out[2],
                  hipStream_t s) {
  const int T = f.n_trees;
  if (T > 65535) fail(DTE_ERR_INVALID_ARGUMENT, "the out-of-bag pass handles at most 65535 trees");
  PoolScope pool(s);
  const int64_t words = (N + 31) / 32;
  const int64_t ranges = (N + kBagRange - 1) / kBagRange;
  DevBuf<uint32_t> bits((size_t)words * T);
  const unsigned parts = (unsigned)std::max<int64_t>(1, std::min<int64_t>(8, 512 / (T * ranges)));
  if (parts > 1)
    hipLaunchKernelGGL(k_zero_u32, dim3(elementwise_grid(words * T)), dim3(kBlock), 0, s, bits.p, words * T);
  hipLaunchKernelGGL(k_inbag_bits_lds, dim3((unsigned)T, (unsigned)ranges, parts), dim3(kBagThreads),
                     (unsigned)bag_lds_bytes(N), s, bits.p, N, words, f.tree_offset, f.seed);
  DevBuf<float> yv(N);
  DTE_HIP(hipMemcpyAsync(yv.p, targets, 4 * N, hipMemcpyHostToDevice, s));
  DevBuf<OobSlot> slots(kOobSlots);
  DTE_HIP(hipMemsetAsync(slots.p, 0, slots.bytes(), s));
  const int R = staged_rows(f.n_features, 0, N), RB = R ? R : 64;
  const int64_t row_blocks = (N + RB - 1) / RB;
  const int chunks = tree_chunks(row_blocks, T, kWalkThreads / RB);
  const int tpb = (T + chunks - 1) / chunks;
  const size_t lds = R ? sizeof(float) * (size_t)R * (f.n_features + 1) : 0;
  with_rows(R, f.pairs.p != nullptr, [&](auto r, auto packed) {
    constexpr int kR = decltype(r)::value;
    constexpr bool kP = decltype(packed)::value;
    auto kernel = f.task == 0 ? k_oob<0, kR, kP> : k_oob<1, kR, kP>;
    for (int64_t b0 = 0; b0 < row_blocks; b0 += kMaxRowBlocks) {
      const dim3 grid((unsigned)std::min(row_blocks - b0, kMaxRowBlocks), (unsigned)((T + tpb - 1) / tpb));
      hipLaunchKernelGGL(kernel, grid, dim3(kWalkThreads), lds, s, trees_of(f), X, N, f.n_features,
                         (const uint32_t*)bits.p, words, (const float*)yv.p, f.n_classes, f.tree_offset, f.seed, perm,
                         tpb, b0, slots.p);
    }
  });
  DTE_HIP(hipGetLastError());
  std::vector<OobSlot> h(kOobSlots);
  DTE_HIP(hipMemcpyAsync(h.data(), slots.p, sizeof(OobSlot) * kOobSlots, hipMemcpyDeviceToHost, s));
  DTE_HIP(hipStreamSynchronize(s));
  unsigned long long pairs = 0, right = 0;
  double sse = 0.0;
  for (const OobSlot& o : h) {
    if (o.bad) fail(DTE_ERR_INVALID_ARGUMENT, "class label out of range");
    pairs += o.pairs;
    right += o.right;
    sse += o.sse;
  }
  out[0] = (double)pairs;
  out[1] = f.task == 0 ? (double)right : sse;
}

// The records are made on the GPU, in the order the caller gets them, and
// copied straight into the caller's arrays, kExportChunk nodes at a time
// (at most 160 MB of records and their leaves' payloads).  9.8 M nodes, 10
// classes (394 MB out): 207 ms when the canonical arrays (840 MB, class counts
// of inner nodes included) came over and one host thread rebuilt them.
constexpr int64_t kExportChunk = (int64_t)8 << 20;

void export_forest(const Forest& f, dte_node* nodes, int64_t nodes_cap, float* probs, int64_t probs_cap,
                   hipStream_t s) {
  const int64_t n = f.n_nodes;
  const int T = f.n_trees;
  const int P = f.task == 0 ? f.n_classes : 1;
  if (nodes_cap < n) fail(DTE_ERR_INVALID_ARGUMENT, "nodes_cap too small");
  PoolScope pool(s);
  std::vector<DevBuf<uint32_t>> tmp;
  DevBuf<uint32_t> flag(n), pos(n + 1);
  hipLaunchKernelGGL(k_export_leaves, dim3(elementwise_grid(n)), dim3(kBlock), 0, s, n, T, f.tree_start.p,
                     f.feature.p, flag.p);
  scan_u32_ext(flag.p, n, pos.p, s, tmp);
  const int64_t n_chunks = (n + kExportChunk - 1) / kExportChunk;
  std::vector<uint32_t> first(n_chunks + 1);  // leaves before each chunk
  first[n_chunks] = (uint32_t)std::max<int64_t>(f.n_leaves, 0);
  for (int64_t c = 1; c < n_chunks; ++c)
    DTE_HIP(hipMemcpyAsync(&first[c], pos.p + c * kExportChunk, 4, hipMemcpyDeviceToHost, s));
  if (f.n_leaves < 0) DTE_HIP(hipMemcpyAsync(&first[n_chunks], pos.p + n, 4, hipMemcpyDeviceToHost, s));
  if (n_chunks > 1 || f.n_leaves < 0) DTE_HIP(hipStreamSynchronize(s));
  if (probs_cap < (int64_t)first[n_chunks] * P) fail(DTE_ERR_INVALID_ARGUMENT, "probs_cap too small");
  uint32_t most = 0;
  for (int64_t c = 0; c < n_chunks; ++c) most = std::max(most, first[c + 1] - first[c]);
  DevBuf<dte_node> d_nodes(std::min(n, kExportChunk));
  DevBuf<float> d_probs((size_t)most * P);
  for (int64_t c = 0; c < n_chunks; ++c) {
    const int64_t e0 = c * kExportChunk, e1 = std::min(n, e0 + kExportChunk);
    hipLaunchKernelGGL(k_export, dim3(elementwise_grid(e1 - e0)), dim3(kBlock), 0, s, e0, e1, T, f.tree_start.p,
                       f.feature.p, f.left.p, f.threshold.p, f.value.p,
                       f.task == 0 ? f.class_counts.p : (const uint32_t*)nullptr, P, f.level_order, pos.p, d_nodes.p, d_probs.p);
    DTE_HIP(hipGetLastError());
    DTE_HIP(hipMemcpyAsync(nodes + e0, d_nodes.p, sizeof(dte_node) * (e1 - e0), hipMemcpyDeviceToHost, s));
    if (first[c + 1] > first[c])
      DTE_HIP(hipMemcpyAsync(probs + (int64_t)first[c] * P, d_probs.p,
                             sizeof(float) * (int64_t)(first[c + 1] - first[c]) * P, hipMemcpyDeviceToHost, s));
  }
  DTE_HIP(hipStreamSynchronize(s));
}

void predict_forest(const Forest& f, const float* X, int64_t n_rows, int64_t ld, int row_major,
                    int32_t* votes, float* sums, hipStream_t s, bool float_votes) {
  if (n_rows <= 0) return;
  const int F = f.n_features, C = f.n_classes;
  Timer tm("predict", 0.0, s);
  if (f.task == 0) {
    const int R = staged_rows(F, C, n_rows), RB = R ? R : 64;
    const int64_t row_blocks = (n_rows + RB - 1) / RB;
    const int chunks = tree_chunks(row_blocks, f.n_trees, kWalkThreads / RB);
    const int tpb = (f.n_trees + chunks - 1) / chunks;
    const unsigned tree_blocks = (unsigned)((f.n_trees + tpb - 1) / tpb);
    const size_t lds = sizeof(uint32_t) * (size_t)RB * (C + (R ? F + 1 : 0));
    const int64_t nv = n_rows * C;
    const int mode = tree_blocks > 1 ? kVoteAdd : float_votes ? kVoteFloat : kVoteInt;
    // votes cleared by a kernel (no memset node if the caller captures)
    if (mode == kVoteAdd)
      hipLaunchKernelGGL(k_zero_u32, dim3(elementwise_grid(nv)), dim3(kBlock), 0, s, reinterpret_cast<uint32_t*>(votes),
                         nv);
    with_walk(f, R, row_blocks, [&](auto r, auto packed, auto nt) {
      constexpr int kThreads = decltype(nt)::value;
      for (int64_t r0 = 0; r0 < n_rows; r0 += kMaxRowBlocks * RB) {
        const int64_t rows = std::min(n_rows - r0, kMaxRowBlocks * RB);
        hipLaunchKernelGGL((k_predict_cls<decltype(r)::value, decltype(packed)::value, kThreads>),
                           dim3((unsigned)((rows + RB - 1) / RB), tree_blocks), dim3(kThreads), lds, s,
                           trees_of(f), row_major ? X + r0 * ld : X + r0, rows, ld, row_major, C, F, tpb, mode,
                           (void*)(votes + r0 * C));
      }
    });
    if (mode == kVoteAdd && float_votes)
      hipLaunchKernelGGL(k_votes_to_float, dim3(elementwise_grid(nv)), dim3(kBlock), 0, s, votes, nv);
  } else {
    // the chunk's leaf values are staged beside the rows
    const int want = staged_rows(F, reg_chunk(64) + 1, n_rows);
    const int R = want && staged_rows(F, reg_chunk(want) + 1, n_rows) == want ? want : 0;
    const int RB = R ? R : 64;
    const size_t lds = sizeof(float) * (size_t)RB * (reg_chunk(R) + 1 + (R ? F + 1 : 0));
    with_walk(f, R, (n_rows + RB - 1) / RB, [&](auto r, auto packed, auto nt) {
      constexpr int kThreads = decltype(nt)::value;
      for (int64_t r0 = 0; r0 < n_rows; r0 += kMaxRowBlocks * RB) {
        const int64_t rows = std::min(n_rows - r0, kMaxRowBlocks * RB);
        hipLaunchKernelGGL((k_predict_reg<decltype(r)::value, decltype(packed)::value, kThreads>),
                           dim3((unsigned)((rows + RB - 1) / RB)), dim3(kThreads), lds, s, trees_of(f),
                           row_major ? X + r0 * ld : X + r0, rows, ld, row_major, F, sums + r0);
      }
    });
  }
  DTE_HIP(hipGetLastError());
}

// Predict records of a forest (its canonical arrays are complete on stream
// s).  max_tree: nodes of its largest tree.
namespace {
// Feature bits of the packed records' links, or 0: wide records.
int packed_feature_bits(const Forest& f, int64_t max_tree) {
  if (!f.level_order) return 0;
  int fbits = 1;
  while (((int64_t)1 << fbits) <= (int64_t)f.n_features) ++fbits;  // feature + 1, 0 for a leaf
  // slots of a tree: a cluster of s pairs takes at most 1.6 s of them
  const int64_t slots = 8 + (max_tree / 2) * 8 / 5 + 8;
  int pbits = 1;
  while (((int64_t)1 << pbits) <= slots) ++pbits;
  return fbits + pbits > 32 ? 0 : fbits;
}
size_t packed_pairs(const Forest& f) { return (size_t)16 * f.n_trees + (size_t)((f.n_nodes + 1) / 2) * 8 / 5; }
}  // namespace

size_t predict_slab_bytes(const Forest& f, int64_t max_tree) {
  if (!packed_feature_bits(f, max_tree)) return Forest::slab_bytes(sizeof(PNode) * (size_t)f.n_nodes);
  return Forest::slab_bytes(sizeof(PPair) * packed_pairs(f)) + Forest::slab_bytes(sizeof(int64_t) * (size_t)f.n_trees);
}

void build_predict_nodes(Forest& f, int64_t max_tree, hipStream_t s) {
  const int64_t n = f.n_nodes;
  const int T = f.n_trees;
  const uint32_t* cls = f.task == 0 ? f.class_counts.p : nullptr;
  const unsigned grid = (unsigned)std::min<int64_t>((n + kBlock - 1) / kBlock, 16384);
  const int fbits = packed_feature_bits(f, max_tree);
  if (!fbits) {
    {
      PoolSuspend own;  // kept with the forest
      f.take(f.pnodes, n);
    }
    hipLaunchKernelGGL(k_wide_nodes, dim3(grid), dim3(kBlock), 0, s, n, f.n_classes, f.task, f.feature.p,
                       f.threshold.p, f.left.p, cls, f.value.p, f.pnodes.p);
    DTE_HIP(hipGetLastError());
    return;
  }
  {
    PoolSuspend own;  // kept with the forest
    f.take(f.pairs, packed_pairs(f));
    f.take(f.pair_base, T);
  }
  f.pair_fbits = fbits;
  PoolScope pool(s);
  DevBuf<uint32_t> code(n), cbase(4 * (size_t)T);
  DevBuf<unsigned int> cnt(4 * (size_t)T);
  hipLaunchKernelGGL(k_zero_u32, dim3(elementwise_grid(4 * (int64_t)T)), dim3(kBlock), 0, s, cnt.p, 4 * (int64_t)T);
  hipLaunchKernelGGL(k_cluster_count, dim3(grid), dim3(kBlock), 0, s, n, T, f.tree_start.p, f.feature.p, f.left.p,
                     f.depth.p, code.p, cnt.p);
  hipLaunchKernelGGL(k_cluster_bases, dim3(1), dim3(kBlock), 0, s, T, f.tree_start.p, f.depth.p,
                     (const unsigned int*)cnt.p, f.pair_base.p,
                     cbase.p);
  hipLaunchKernelGGL(k_cluster_write, dim3(grid), dim3(kBlock), 0, s, n, T, f.tree_start.p, f.feature.p, f.left.p,
                     f.depth.p, f.threshold.p, cls, f.value.p, f.n_classes, f.task, fbits, (const uint32_t*)code.p,
                     (const int64_t*)f.pair_base.p, (const uint32_t*)cbase.p, reinterpret_cast<uint4*>(f.pairs.p));
  DTE_HIP(hipGetLastError());
}

}  // namespace dte
