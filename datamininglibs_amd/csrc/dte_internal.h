// Internal declarations shared by the build, predict, serve and C-ABI units
// of libdte.  Not part of the public ABI (include/dte.h is).
#pragma once
#include <algorithm>
#include <hip/hip_runtime.h>

#include <cstdint>
#include <functional>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/dte.h"
#include "dte_numerics.h"

namespace dte {

// ------------------------------------------------------------- errors ----
struct Error {
  int code;
  std::string msg;
};
void set_error(int code, const std::string& msg);
// Runs fn, turning exceptions into a status code and the thread's last error.
int run_guarded(const std::function<void()>& fn);
// hipSetDevice + one-time library initialisation of that device.
void select_device(int device);
[[noreturn]] void fail(int code, const std::string& msg);

#define DTE_HIP(expr)                                                                  \
  do {                                                                                 \
    hipError_t _e = (expr);                                                            \
    if (_e != hipSuccess)                                                              \
      ::dte::fail(_e == hipErrorOutOfMemory ? DTE_ERR_OUT_OF_MEMORY : DTE_ERR_HIP,      \
                  std::string(#expr) + ": " + hipGetErrorString(_e));                  \
  } while (0)

// ------------------------------------------------------- scratch pool --
// Device blocks of the temporaries of a fit, an export, an out-of-bag pass and
// a forest's predict records are cached per (device, stream) when
// released and handed back to later requests on the same stream, so that the
// growing per-level buffers and repeated fits do not call hipMalloc / hipFree
// (which synchronise the device) inside the level loop.  Reuse on the same
// stream is ordered by the stream.  Pooling is on for the allocations of a
// thread inside a PoolScope; forests handed to the caller are allocated
// outside the pool (PoolSuspend).
struct PoolBlock {
  void* p;
  size_t bytes;
};
// Takes a block of at least `bytes` for the thread's pool stream (granted
// size in *got, owning device and stream in *dev, *owner).
void* pool_alloc(size_t bytes, size_t* got, int* dev, hipStream_t* owner);
void pool_free(void* p, size_t bytes, int dev, hipStream_t owner);
// Frees every cached block (all devices); returns the bytes released.
size_t pool_trim();
// hipMalloc; without memory once more after pool_trim.
void* device_malloc(size_t bytes);
// Bytes of the cached blocks of a device: free to a fit as hipMemGetInfo's are,
// since an allocation that finds no memory trims the pool.
size_t pool_cached(int dev);
bool pool_on();  // inside a PoolScope (and not suspended) on this thread

struct PoolScope {
  bool prev_on;
  hipStream_t prev_s;
  explicit PoolScope(hipStream_t s);
  ~PoolScope();
};
struct PoolSuspend {
  bool prev_on;
  PoolSuspend();
  ~PoolSuspend();
};

// Device buffer owned by RAII (the reference frees by hand in
// GpuParams::finalize, gpudte_algorithm_shared.cc:30-52, and leaks on throw).
template <typename T>
struct DevBuf {
  T* p = nullptr;
  size_t n = 0;           // elements requested
  size_t block = 0;       // bytes of the pool block (pooled buffers)
  bool pooled = false;
  bool view = false;      // part of another buffer, which frees it
  int dev = 0;
  hipStream_t owner = nullptr;
  DevBuf() = default;
  explicit DevBuf(size_t count) { alloc(count); }
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  DevBuf(DevBuf&& o) noexcept : p(o.p), n(o.n), block(o.block), pooled(o.pooled), view(o.view), dev(o.dev), owner(o.owner) {
    o.p = nullptr;
    o.n = 0;
  }
  DevBuf& operator=(DevBuf&& o) noexcept {
    if (this != &o) {
      release();
      p = o.p;
      n = o.n;
      block = o.block;
      pooled = o.pooled;
      view = o.view;
      dev = o.dev;
      owner = o.owner;
      o.p = nullptr;
      o.n = 0;
    }
    return *this;
  }
  ~DevBuf() { release(); }
  void alloc(size_t count) {
    release();
    if (count == 0) count = 1;
    if (pool_on()) {
      p = (T*)pool_alloc(count * sizeof(T), &block, &dev, &owner);
      pooled = true;
      n = count;
    } else {
      p = (T*)device_malloc(count * sizeof(T));
      pooled = false;
      n = count;
    }
  }
  // Grow to at least `count` elements; contents are not preserved.
  void reserve(size_t count) {
    if (count > n) alloc(count + count / 4);
  }
  void release() {
    if (p && !view) {
      if (pooled)
        pool_free(p, block, dev, owner);
      else
        (void)hipFree(p);
    }
    p = nullptr;
    n = 0;
    block = 0;
    pooled = false;
    view = false;
  }
  size_t bytes() const { return n * sizeof(T); }
};

// Kernel timing of one named kernel family, collected with HIP events on the
// library's stream when profiling is on.
struct KernelStat {
  std::string name;
  int64_t launches = 0;
  double total_ms = 0.0;
  double bytes = 0.0;  // algorithmic bytes
};

void profile_record(const char* name, hipEvent_t a, hipEvent_t b, double bytes);
void profile_add_bytes(const char* name, double bytes);
void profile_count(const char* name, int64_t n);
void profile_host(const char* name, double ms);
bool profiling_enabled();

// HIP events around the launches of one kernel family on stream s (only
// while profiling is on); recorded under `name` with `bytes` algorithmic bytes.
struct Timer {
  hipEvent_t a = nullptr, b = nullptr;
  const char* name;
  double bytes;
  hipStream_t s;
  Timer(const char* nm, double by, hipStream_t st) : name(nm), bytes(by), s(st) {
    if (profiling_enabled()) {
      DTE_HIP(hipEventCreate(&a));
      DTE_HIP(hipEventCreate(&b));
      DTE_HIP(hipEventRecord(a, s));
    }
  }
  ~Timer() {
    if (a) {
      (void)hipEventRecord(b, s);
      profile_record(name, a, b, bytes);
    }
  }
};

// Predict-side records.  Packed (dte_predict.hip: build_predict_nodes): 8
// bytes a node, (threshold bits, pair of the children << fbits | feature + 1)
// or (leaf payload, 0), siblings side by side in a 16-byte pair; the payload is
// the vote class or the bits of the regression value.  Wide, for trees whose
// pairs and features do not fit a link of 32 bits: 16 bytes a node in
// canonical order,
//   internal: feature >= 0, thr bits, left child index (right = left + 1)
//   leaf:     feature = -1, thr = payload
struct PPair {
  uint32_t w[4];
};
struct PNode {
  int32_t feature;
  uint32_t thr;
  int32_t left;
  int32_t pad;
};

// A fitted forest resident in HBM.  Node arrays are canonical: tree-major,
// level order inside each tree, children adjacent.
struct Forest {
  int device = 0;
  int task = 0;
  int n_classes = 1;
  int n_features = 0;
  int n_trees = 0;
  int fixed_shift = 0;
  int algorithm = 0;
  int64_t n_nodes = 0;
  // Leaves; -1 until known.  A built tree has one more leaf than splits
  // (every split makes two children), so a fit knows it without a pass.
  int64_t n_leaves = -1;
  // Bootstrap record of a fit (random forest): tree t drew its rows with
  // seed and global tree id tree_offset + t from fit_rows rows; fit_rows = 0
  // when unknown (imported forests).
  uint64_t seed = 0;
  int32_t tree_offset = 0;
  int64_t fit_rows = 0;
  // One allocation for all arrays of a fitted forest: a fit made 13 of them and
  // a destroy freed 13, at 50 to 200 us each (13 ms for 20 forests, 2.7 of a
  // 28 ms fit of 2.6 M nodes).
  DevBuf<unsigned char> slab;
  size_t slab_used = 0;
  static size_t slab_bytes(size_t bytes) { return (std::max<size_t>(bytes, 1) + 255) & ~(size_t)255; }
  // `count` elements from the slab, or memory of their own where it has no room.
  template <typename T>
  void take(DevBuf<T>& b, size_t count) {
    const size_t bytes = slab_bytes(count * sizeof(T));
    if (slab_used + bytes > slab.n) {
      b.alloc(count);
      return;
    }
    b.release();
    b.p = reinterpret_cast<T*>(slab.p + slab_used);
    b.n = std::max<size_t>(count, 1);
    b.view = true;
    slab_used += bytes;
  }
  DevBuf<int64_t> tree_start;  // n_trees + 1
  DevBuf<PPair> pairs;         // packed predict records (empty: wide ones)
  DevBuf<int64_t> pair_base;   // packed: first pair of each tree
  int pair_fbits = 0;          // packed: feature bits of a link
  DevBuf<PNode> pnodes;        // wide predict records (n_nodes), or empty
  // Build diagnostics (absent for imported forests).
  bool has_stats = false;
  // Every tree's nodes in level order, children in their parents' order and
  // tree (a file from elsewhere may hold another order, an imported model's
  // root be another tree's child; they take the wide predict records).
  bool level_order = true;
  DevBuf<int32_t> feature, left, depth, count, n_entries;
  DevBuf<float> threshold, score, value;
  DevBuf<uint64_t> rowhash;
  DevBuf<uint32_t> class_counts;  // n_nodes * n_classes (classification)
  DevBuf<int64_t> sum_fixed;
};

struct FitInput {
  const float* X;  // device, feature-major, canonical (-0 -> +0)
  const float* y;  // device or host targets (see caller)
  int64_t n_rows;
  int32_t n_features;
};

// Entry points implemented in dte_build.hip / dte_predict.hip.
Forest* fit_forest(const float* X_dev, const float* y_host, int64_t n_rows, int32_t n_features,
                   const dte_params& p, hipStream_t stream);
void build_predict_nodes(Forest& f, int64_t max_tree, hipStream_t stream);
size_t predict_slab_bytes(const Forest& f, int64_t max_tree);  // what it takes from the slab
// Several extra-trees forests of one task in one build: every level step
// serves the open nodes of all forests (see dte_fit_many).
std::vector<Forest*> fit_joint(const float* const* X_dev, const float* const* y_host, const int64_t* n_rows,
                               const int32_t* n_features, const dte_params* params, int n, hipStream_t stream);
// float_votes: the vote counts as floats in votes_dev's words.
void predict_forest(const Forest& f, const float* X_dev, int64_t n_rows, int64_t ld,
                    int row_major, int32_t* votes_dev, float* sums_dev, hipStream_t stream,
                    bool float_votes = false);
// Reference model layout (dte_forest_export) into host arrays.
void export_forest(const Forest& f, dte_node* nodes, int64_t nodes_cap, float* probs, int64_t probs_cap,
                   hipStream_t stream);
// Exclusive scan of n words into out[0 .. n] (out[n] = total).
void scan_u32_ext(const uint32_t* in, int64_t n, uint32_t* out, hipStream_t s, std::vector<DevBuf<uint32_t>>& tmp);
// Out-of-bag evaluation (dte_oob_evaluate): pairs evaluated, correct pairs
// (classification) or the sum of squared errors (regression).
void oob_evaluate(const Forest& f, const float* X_dev, const float* targets, int64_t n_rows, int perm_feature,
                  double out[2], hipStream_t stream);
void device_init(int device);
hipStream_t library_stream(int device);
// The stream to record a graph on whose replays go to stream s, held until the
// object ends.  A stream takes part in a recording with whatever any thread
// sends to it, so the library stream, which all callers share, never records.
struct RecordStream {
  std::unique_lock<std::mutex> lock;
  hipStream_t stream;
  explicit RecordStream(hipStream_t s);
};
const LnTable& host_ln_table();

constexpr int kBlock = 256;

// Defaults of the split-search tuning fields of dte_params (0 selects them).
constexpr int kDefCutTeam = 512;
constexpr int kMaxCutTeam = 512;  // capacity of the wave-per-item tier (64 lanes x 8)
constexpr int kDefCutBlock = 2048;
constexpr int kDefBucketTarget = 384;
constexpr int kDefCutErt = 4096;

}  // namespace dte

// Opaque handle of the C ABI.
struct dte_forest {
  dte::Forest f;
};
