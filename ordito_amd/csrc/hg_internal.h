// Internal declarations of libheatgeo: mesh state, the Cholesky plan and error plumbing.
// Everything here is private to the library; the public C ABI is include/heatgeo.h.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cstdint>
#include <future>
#include <memory>
#include <string>
#include <thread>
#include <vector>

#include "../../include/heatgeo.h"

namespace hg {

// ------------------------------------------------------------------------------------------------
// Errors: every entry point returns an hg_status and leaves a message for hg_last_error().
// ------------------------------------------------------------------------------------------------

void set_error(const std::string& message);

struct Error {
  int status;
  std::string message;
};

#define HG_HIP(call)                                                                          \
  do {                                                                                        \
    hipError_t hg_err_ = (call);                                                              \
    if (hg_err_ != hipSuccess) {                                                              \
      throw ::hg::Error{HG_ERR_RUNTIME, std::string(#call) + ": " + hipGetErrorString(hg_err_)}; \
    }                                                                                         \
  } while (0)

#define HG_REQUIRE(cond, status, message)          \
  do {                                             \
    if (!(cond)) throw ::hg::Error{(status), (message)}; \
  } while (0)

// A device allocation owned by the library.
template <typename T>
struct DeviceArray {
  T* ptr = nullptr;
  int64_t size = 0;
  DeviceArray() = default;
  explicit DeviceArray(int64_t n) { allocate(n); }
  DeviceArray(const DeviceArray&) = delete;
  DeviceArray& operator=(const DeviceArray&) = delete;
  DeviceArray(DeviceArray&& o) noexcept : ptr(o.ptr), size(o.size) { o.ptr = nullptr; o.size = 0; }
  DeviceArray& operator=(DeviceArray&& o) noexcept {
    if (this != &o) { reset(); ptr = o.ptr; size = o.size; o.ptr = nullptr; o.size = 0; }
    return *this;
  }
  ~DeviceArray() { reset(); }
  // An allocation that fails leaves the array empty: callers grow it by its size.
  void allocate(int64_t n) {
    reset();
    if (n > 0) HG_HIP(hipMalloc(&ptr, sizeof(T) * static_cast<size_t>(n)));
    size = n;
  }
  void reset() {
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    size = 0;
  }
  int64_t bytes() const { return size * static_cast<int64_t>(sizeof(T)); }
  void upload(const T* host, int64_t n, hipStream_t stream) {
    if (n > 0) HG_HIP(hipMemcpyAsync(ptr, host, sizeof(T) * n, hipMemcpyHostToDevice, stream));
  }
  void upload(const std::vector<T>& host, hipStream_t stream) {
    allocate(static_cast<int64_t>(host.size()));
    upload(host.data(), size, stream);
  }
  // Copies host into the array, reallocating only to grow: per-call arrays (sources, offsets)
  // keep their memory, so a solve allocates nothing once warm (hipMalloc and hipFree synchronize
  // the device, which would serialize solves on other streams).
  void assign(const std::vector<T>& host, hipStream_t stream) {
    const int64_t count = static_cast<int64_t>(host.size());
    if (size < std::max<int64_t>(count, 1)) allocate(std::max<int64_t>(count, 1));
    upload(host.data(), count, stream);
  }
};

// A pinned host allocation (hipHostMalloc): device-to-host copies into it stay asynchronous.
template <typename T>
struct PinnedArray {
  T* ptr = nullptr;
  int64_t size = 0;
  PinnedArray() = default;
  PinnedArray(const PinnedArray&) = delete;
  PinnedArray& operator=(const PinnedArray&) = delete;
  ~PinnedArray() { reset(); }
  void allocate(int64_t n) {
    reset();
    HG_HIP(hipHostMalloc(reinterpret_cast<void**>(&ptr), sizeof(T) * static_cast<size_t>(n),
                         hipHostMallocDefault));
    size = n;
  }
  void reset() {
    if (ptr) (void)hipHostFree(ptr);
    ptr = nullptr;
    size = 0;
  }
};

// ------------------------------------------------------------------------------------------------
// Host analysis (pattern.cpp, analysis.cpp)
// ------------------------------------------------------------------------------------------------

// The cotangent operator's sparsity: every face edge in both directions plus a diagonal per
// referenced vertex, rows sorted by column, and for each stored entry its run of contributing
// corner slots 3f+e (corner e opposite the edge) in ascending order.
struct HostPattern {
  int64_t n = 0;
  std::vector<int32_t> offsets;       // n+1
  std::vector<int32_t> columns;       // nnz
  std::vector<int32_t> corner_ptr;    // nnz+1
  std::vector<int32_t> corner_slots;  // <= 6F
  std::vector<int32_t> vertex_ptr;    // n+1: each vertex's corners, ascending
  std::vector<int32_t> vertex_corners;
  std::vector<int32_t> diagonal;      // n: slot of the diagonal entry, -1 for an empty row
};

// The pattern's device arrays (the HostPattern fields but the diagonal).
struct PatternArrays {
  DeviceArray<int32_t>& offsets;
  DeviceArray<int32_t>& columns;
  DeviceArray<int32_t>& corner_ptr;
  DeviceArray<int32_t>& corner_slots;
  DeviceArray<int32_t>& vertex_ptr;
  DeviceArray<int32_t>& vertex_corners;
};

// Builds the pattern on the device from the device faces (range-checked there) and, when host is
// not null, downloads it there for the host-side work.
void build_pattern_device(int64_t n_vertices, const int32_t* d_faces, int64_t n_faces,
                          hipStream_t stream, PatternArrays out, HostPattern* host);

// Connected components of the pattern's graph.
std::vector<int32_t> component_labels(const HostPattern& pattern, int32_t* n_components);

// A supernodal Cholesky plan: nested-dissection order, supernode tree, level schedule, the maps
// the numeric factorization and the multifrontal solves use.
struct Plan {
  int64_t n = 0;
  int32_t n_super = 0;
  int32_t n_levels = 0;
  std::vector<int32_t> perm;        // new -> old
  std::vector<int32_t> iperm;       // old -> new
  std::vector<int32_t> col_begin;   // per supernode, new index of its first column
  std::vector<int32_t> ncol;
  std::vector<int32_t> nrow;
  std::vector<int32_t> parent;
  std::vector<int32_t> level;
  std::vector<int32_t> row_ptr;     // CSR over supernodes: the structure rows (new indices)
  std::vector<int32_t> rows;
  std::vector<int32_t> child_ptr;   // CSR over supernodes: children, ascending
  std::vector<int32_t> children;
  std::vector<int32_t> rel;         // per supernode s, nrow[s] positions of rows(s) in parent's front
  std::vector<int32_t> rel_ptr;     // = row_ptr
  std::vector<int32_t> level_ptr;   // CSR over levels: supernodes at each level (bottom-up)
  std::vector<int32_t> level_nodes;
  std::vector<int64_t> front_off;   // arena offset (doubles) of each m x m front
  std::vector<int64_t> w_off;       // offset of each m x ncol solve block
  std::vector<int64_t> vec_off;     // offset (per column) of each front's m-vector in solve scratch
  int64_t arena_size = 0;
  int64_t w_size = 0;
  int64_t vec_size = 0;
  // Lower-triangle entries of the operator in front coordinates: value slot -> arena offset.
  std::vector<int32_t> entry_src;
  std::vector<int64_t> entry_dst;
  std::vector<int32_t> entry_row;   // new row index of the entry
  std::vector<int32_t> entry_col;   // new column index
  double flops = 0.0;               // dense partial-factorization flops
  int64_t nnz_w = 0;                // stored solve-block entries
  int32_t max_front = 0;
  bool merged = false;  // separators were merged upwards
};

// Leaf 128: on the 1024 x 512 torus with 64 right-hand sides, leaves of 96-192 rows serve fastest
// (fewer, fuller levels), 128 by a small margin over 48 (3%) and 512 (16%).
struct AnalysisOptions {
  int32_t leaf_rows = 128;
  int32_t top_rows = 512;
  int32_t merge_rows = -1;  // small separators merged upwards (0: none; -1: by the rows, analyse)
};

Plan analyse(const HostPattern& pattern, const float* coordinates, const AnalysisOptions& options);

// The triangular sweeps' product tasks of one direction (cholesky.hip): per level, every 64-wide
// tile of every front and its inner range [k0, k1); slot >= 0 names a partial that the level's
// reduction groups (rs, rtile, rfirst, rcount) add in slot order.
struct HostSweep {
  std::vector<int32_t> level_ptr, reduce_ptr, slots;
  std::vector<int32_t> s, tile, k0, k1, slot;
  std::vector<int32_t> rs, rtile, rfirst, rcount;
  int32_t max_slots = 0;
};
// A level whose tiles are fewer than `target_tasks` has its products split along the inner
// dimension until it has about that many tasks (a few per compute unit by default).
constexpr int32_t kDefaultSplitTarget = 1024;
HostSweep sweep_tasks(const Plan& plan, bool forward, int32_t target_tasks = kDefaultSplitTarget);
// The targets of a plan's two task lists (DevicePlan): for up to 16 columns, and for more.
inline std::array<int32_t, 2> sweep_targets(int32_t target_tasks) {
  return {target_tasks, std::max(1, target_tasks / 4)};
}

// The forward sweep's gather lists: for each front-vector row (vec_off[s] + position) the rows of
// the children's update vectors that add into it, and the first two of them inline per position
// (pair[2v], pair[2v+1]; -1 none, -2 in the second: more than two, the rest in the lists).
struct HostGather {
  std::vector<int32_t> ptr, src, pair;
};
HostGather gather_lists(const Plan& plan);

// A whole sweep of a few right-hand sides as one launch's tasks (flow.hip), in an order in which
// each follows everything it waits for: the forward tasks by level upwards, then the backward ones
// downwards. Twelve int32 a task: {shape, tile, inner, gathers, ncol, col_begin, ncol + nrow,
// front, w_off (two words), vec_off (forward) or row_ptr (backward) as two words}. A forward task
// is rows [tile, tile + 256 / shape) over columns [0, inner), shape 1, 4 or 16 threads a row; a
// backward task columns [tile, tile + 16 shape), shape 1 or 4.
struct HostFlow {
  int32_t n_forward = 0;
  std::vector<int32_t> desc;
};
// The most right-hand sides such a sweep takes. Its products are on the vector units, a multiply a
// column; level by level they are on the matrix cores, sixteen columns for the price of one. A sweep
// of 4 columns takes 196 us against 407 on icosphere(7), 491 against 899 on the 524,288-row torus
// and 2.14 ms against 3.58 on icosphere(9); of 8, 360 against 411, 927 against 900 and 4.22 ms
// against 3.62.
constexpr int32_t kFlowColumns = 4;
// The most stored entries of FP32 blocks such a sweep takes. Its loads bring half the bytes then, and the
// level sweeps' tiles catch up where the blocks outgrow the last-level cache: refined diffusions of one
// column and of four took 671 and 777 us in one launch a sweep and 821 and 829 level by level with 27.5
// million entries (a grid of 160,000), 953 and 1,067 against 907 and 932 with 38.3 (a torus of 160,000),
// 2,377 and 2,606 against 1,721 and 1,789 with 108 (the 524,288-row torus).
constexpr int64_t kFlowFp32Entries = int64_t{1} << 25;
// A level of this many 64-wide tiles keeps them (icosphere(7): 160 us a sweep; from 128 on 164, from
// 2,048 on 161, never 187).
constexpr int64_t kFlowWideTiles = 512;
constexpr int32_t kFlowAborted = 2;      // the pending word's bit of a launch that gave up waiting
HostFlow flow_tasks(const Plan& plan);

// Checks every index the device sweeps form from the plan against its buffer; throws on the first
// violation.
void validate_sweeps(const Plan& plan, int32_t target_tasks = kDefaultSplitTarget);

// The numeric factorization as launches of 64 x 64 tile tasks (cholesky.hip), in execution order.
// A front's inverse factor Z is the first ncol columns of the inverse of its unit-extended lower
// factor [L11 0; L21 I], i.e. [L11^-1; -L21 L11^-1] (m x ncol, column-major, leading dimension
// m); it is what the sweeps multiply by. Task fields (4 int32 each):
//   kFactorExtend (parent s, child c, i0, k0): the child's Schur-complement tile rows
//       [i0, i0+64) x columns [k0, k0+64), i0 >= k0, added into the parent through the child's
//       relative map. One launch per child rank, so siblings add in ascending order.
//   kFactorPanel (s, j0, kind, t0): the diagonal block at j0 (width b = min(64, ncol - j0)) is
//       eliminated in LDS together with its inverse; kind 0 solves the panel rows [t0, t0+64)
//       below it, kind 1 applies the inverse to Z's block rows at columns [t0, t0+64) (t0 < j0),
//       kind 2 stores the inverse as Z's diagonal block.
//   kFactorUpdate (s, j0, i0, c0): rows [i0, i0+64) minus the panel's rows [i0, i0+64) times
//       the panel rows [c0, c0+64) transposed (the trailing matrix, c0 >= j0 + b, c0 <= i0) or
//       times Z's block rows at columns [c0, c0+64) (c0 < j0 + b).
enum FactorKind : int32_t { kFactorExtend = 0, kFactorPanel = 1, kFactorUpdate = 2 };
struct FactorLaunch {
  int32_t kind, level, first, count;
};
struct HostFactorTasks {
  std::vector<FactorLaunch> launches;
  std::vector<int32_t> tasks;  // 4 per task
};
constexpr int32_t kFactorTile = 64;
HostFactorTasks factor_tasks(const Plan& plan);

// Checks every factorization task against the plan (fronts, children, tile ranges, the step
// order); throws on the first violation.
void validate_factor_tasks(const Plan& plan, const HostFactorTasks& tasks);

// Runs body(begin, end, worker) over [0, count) in contiguous chunks, one a worker thread (the
// caller's thread takes the first); waits for all, rethrowing the first failure.
template <typename F>
void parallel_chunks(int64_t count, int64_t grain, F&& body) {
  const int64_t hw = std::max<int64_t>(1, std::thread::hardware_concurrency());
  const int64_t workers = std::max<int64_t>(1, std::min<int64_t>(hw, (count + grain - 1) / grain));
  const int64_t chunk = (count + workers - 1) / std::max<int64_t>(workers, 1);
  std::vector<std::future<void>> pool;
  for (int64_t w = 1; w < workers; ++w) {
    const int64_t b = w * chunk, e = std::min(count, b + chunk);
    if (b >= e) break;
    pool.push_back(std::async(std::launch::async, [&body, b, e, w] { body(b, e, w); }));
  }
  body(0, std::min(count, chunk), 0);
  for (std::future<void>& f : pool) f.get();
}

}  // namespace hg
