// Refined multi-column solves through the partitioned-inverse factor, level by level.
//
// The whole refinement (ordito kernels/cholesky.py:1357-1463, cholesky.py:1606-1902) runs in the
// elimination order with the k right-hand sides of a chunk interleaved ([row][k]): the operator is
// held permuted (P A P^T), so a right-hand side in the caller's layout is permuted in once and the
// solution out once (fields stored by rows are already in that order), and every round is forward
// sweep, backward sweep, residual -- no per-round permutation. Each level of
// a sweep is a batch of dense tile products over every front of the level:
//   forward : y(cols) = Z11 f(cols) and the front's update vector u = f(rows) + Z21 f(cols), where
//             f = [r(cols); 0] + the children's update vectors, gathered as the tile loads it
//             (children in ascending order);
//   backward: d(cols) = Z11^T y(cols) + Z21^T d(rows), and the next iterate x + d beside it;
// Z = [L11^-1; -L21 L11^-1] is the front's inverse factor (cholesky.hip).
// A product task is one 64-wide tile of one front and a range of the inner dimension; a level with
// too few tiles to fill the device splits the inner dimension into partial slots, added in slot
// order by a reduction, so every sum keeps one fixed order. Tiles stage the solve block and the
// right-hand sides through LDS and accumulate in FP64 (FP32 solve blocks widen as they load).
#include "cholesky.h"

namespace hg {
namespace {

constexpr int kTile = 64;   // rows (forward) or columns (backward) of W per tile
constexpr int kCols = 64;   // right-hand sides per solve chunk
static_assert(kCols == kFieldChunk, "a row-layout field chunk is one solve chunk");
constexpr int kReduceSplit = 4;  // blocks a reduction group is spread over (16 rows each)

template <typename T>
__device__ __forceinline__ double widen(T v) {
  return static_cast<double>(v);
}

// b (user layout, column q at q*n) -> bp[i*kk + q] in elimination order through an LDS transpose
// of 64 rows; a pinned row's equation is dropped (zero).
__global__ __launch_bounds__(256) void perm_in_kernel(const double* __restrict__ b,
                                                      const int32_t* __restrict__ perm,
                                                      const int32_t* __restrict__ pinned,
                                                      int64_t n, int32_t kk,
                                                      double* __restrict__ bp) {
  __shared__ double tile[kTile][kCols + 1];
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kTile;
  const int ii = threadIdx.x % kTile, qq = threadIdx.x / kTile;
  const int64_t i = i0 + ii;
  const bool live = i < n;
  const int64_t src = live ? perm[i] : 0;
  const bool drop = !live || (pinned && pinned[i]);
  for (int q = qq; q < kk; q += 4) tile[ii][q] = drop ? 0.0 : b[q * n + src];
  __syncthreads();
  const int32_t rows = static_cast<int32_t>(min<int64_t>(kTile, n - i0));
  for (int e = threadIdx.x; e < rows * kk; e += 256) {
    const int r_ = e / kk, q = e % kk;
    bp[(i0 + r_) * kk + q] = tile[r_][q];
  }
}

// out (user layout) [q*n + perm[i]] = x[i*kk + q], through the same transpose.
__global__ __launch_bounds__(256) void perm_out_kernel(const double* __restrict__ x,
                                                       const int32_t* __restrict__ perm,
                                                       int64_t n, int32_t kk,
                                                       double* __restrict__ out) {
  __shared__ double tile[kTile][kCols + 1];
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kTile;
  const int32_t rows = static_cast<int32_t>(min<int64_t>(kTile, n - i0));
  for (int e = threadIdx.x; e < rows * kk; e += 256) tile[e / kk][e % kk] = x[i0 * kk + e];
  __syncthreads();
  const int ii = threadIdx.x % kTile, qq = threadIdx.x / kTile;
  if (ii >= rows) return;
  const int64_t dst = perm[i0 + ii];
  for (int q = qq; q < kk; q += 4) out[q * n + dst] = tile[ii][q];
}

// Pinned rows of a right-hand side stored by rows: zero, the pins' values (a component's last
// row, an unreferenced vertex) held there by the identity rows of the factor.
__global__ __launch_bounds__(256) void zero_pinned_rows_kernel(const int32_t* __restrict__ pinned,
                                                               int64_t n, int32_t kk,
                                                               double* __restrict__ b) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n || !pinned[i]) return;
  for (int32_t q = 0; q < kk; ++q) b[i * kk + q] = 0.0;
}

struct SweepArgs {
  const int32_t* col_begin;
  const int32_t* ncol;
  const int32_t* nrow;
  const int32_t* row_ptr;
  const int32_t* rows;
  const int64_t* w_off;
  const int64_t* vec_off;
  const int32_t* gather_pair;
  const int32_t* gather_ptr;
  const int32_t* gather_src;
  const double* r;   // residual, the sweep's right-hand side
  double* fvec;      // update vectors (rows part of each front's vector)
  double* y;         // forward result
  double* d;         // backward result (the correction)
  const double* x;   // current iterate; null on the first round (x = 0: d is the next iterate)
  double* x_next;    // x + d; null on the first round
  double* partials;
  int32_t kk;
  int32_t gathers;   // the level's fronts have children (forward sweep): f gathers their updates
  const int32_t* live;  // null, or the fronts the forward sweep reaches (LiveFronts)
  const int32_t* vec_front;
};

// The children's update rows that add into front-vector rows, in three steps so that a caller can
// issue other loads, and products, between them. gather_pairs: each row's first two sources (inline
// in gather_pair; -1: none; -2 in the second: more than two, the rest in the lists after the first;
// live[u] false: none). gather_issue: the two update rows' entries of column q[u] (an absent source
// reads row 0). gather_add: the sum, in ascending child order. Nothing waits before gather_add.
// q may run up to 63 past the chunk's columns: the update vectors end in as much padding.
template <int N>
__device__ __forceinline__ void gather_pairs(const SweepArgs& a, const int64_t (&row)[N],
                                             const bool (&live)[N], int2 (&p)[N]) {
  const int2* pairs = reinterpret_cast<const int2*>(a.gather_pair);
#pragma unroll
  for (int u = 0; u < N; ++u) p[u] = live[u] ? pairs[row[u]] : make_int2(-1, -1);
}

__device__ __forceinline__ const double* update_row(const SweepArgs& a, int32_t row) {
  return a.fvec + static_cast<int64_t>(max(row, 0)) * a.kk;
}

template <int N>
__device__ __forceinline__ void gather_issue(const SweepArgs& a, const int2 (&p)[N],
                                             const int (&q)[N], double (&first)[N],
                                             double (&second)[N]) {
#pragma unroll
  for (int u = 0; u < N; ++u) {
    first[u] = update_row(a, p[u].x)[q[u]];
    second[u] = update_row(a, p[u].y)[q[u]];
  }
}

// v plus row `row`'s gathered entries of column q, the first two already loaded.
__device__ __forceinline__ double gather_add(const SweepArgs& a, int64_t row, int q, int2 p,
                                             double first, double second, double v) {
  if (p.x >= 0) v += first;
  if (p.y >= 0) {
    v += second;
  } else if (p.y == -2) {
    for (int32_t g = a.gather_ptr[row] + 1; g < a.gather_ptr[row + 1]; ++g)
      if (!a.live || a.live[a.vec_front[a.gather_src[g]]])
        v += a.fvec[static_cast<int64_t>(a.gather_src[g]) * a.kk + q];
  }
  return v;
}

// The tile products run on the FP64 matrix cores: v_mfma_f64_16x16x4 takes a 16 x 4 block of A
// (lane l holds A[l % 16][l / 16]) and a 4 x 16 block of B (lane l holds B[l / 16][l % 16]) and
// accumulates the 16 x 16 product, lane l holding rows l / 16 + 4v (v < 4) of column l % 16. A
// tile's four waves each own 16 of its 64 rows and accumulate NB blocks of 16 right-hand sides. The
// vectors are staged through LDS, shared by the waves, kDepth inner indices at a time; a wave's
// part of the inverse factor is its own, so its lanes load it straight into the operand's layout.
// The next stage's global loads are issued before the current stage's products, so they overlap.
typedef double f64x4 __attribute__((ext_vector_type(4)));
// A stage is 16 inner indices of 32 or 64 right-hand sides, 32 of 16: a block of few columns waits on
// its loads' round trips (16 columns on icosphere(7): 303 us a heat sweep 16 deep, 285 at 32; 64
// deep 298, and on icosphere(9) 1.60 ms against 1.36).
template <int NB>
constexpr int kStages = NB == 1 ? 2 : 1;
// Staged rows are kPad doubles more than their columns apart, which puts the two inner rows that half a
// wave's operand read spans (neighbours forward, four apart backward) 32 banks apart.

__device__ __forceinline__ f64x4 mfma16x16x4(double a, double b, f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// The entry `bytes` past a wave-uniform base: one address register a lane for a run of loads.
template <typename T>
__device__ __forceinline__ T load_at(const T* base, uint32_t bytes) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + bytes);
}

// A task's descriptor: {s, tile, k0, k1}, {slot, ncol, col_begin, m}, {a 64-bit offset of the
// front's solve block, a 64-bit second offset}, read together.
struct Task {
  int32_t s, tile, k0, k1, slot, nc, c0, m;
  int64_t w_off, other;
};

__device__ __forceinline__ Task load_task(const int4* __restrict__ desc, int32_t task) {
  const int4* d = desc + 3 * static_cast<int64_t>(task);
  const int4 d0 = d[0], d1 = d[1], d2 = d[2];
  Task t;
  t.s = d0.x;
  t.tile = d0.y;
  t.k0 = d0.z;
  t.k1 = d0.w;
  t.slot = d1.x;
  t.nc = d1.y;
  t.c0 = d1.z;
  t.m = d1.w;
  t.w_off = static_cast<int64_t>(static_cast<uint32_t>(d2.x)) | (static_cast<int64_t>(d2.y) << 32);
  t.other = static_cast<int64_t>(static_cast<uint32_t>(d2.z)) | (static_cast<int64_t>(d2.w) << 32);
  return t;
}

// Forward tile product for up to 16 NB right-hand sides: rows [r0, r0+64) of the front's inverse
// factor times f over the inner range [k0, k1), f gathered as it is staged. slot < 0 applies the
// product; otherwise it is stored as a partial for the reduction.
// kGathers: the level's fronts have children whose update vectors f gathers (a.gathers); the
// leaves' instance carries none of that code.
template <typename TW, int NB, bool kGathers>
__global__ __launch_bounds__(256, kGathers ? 4 : (NB == 4 ? 5 : 6)) void fwd_tile_kernel(
    const int4* __restrict__ desc, int32_t parts, const TW* __restrict__ w, SweepArgs a) {
  constexpr int D = kStages<NB>, kN = 16 * NB, kDepth = 16 * D, U = NB * D;
  constexpr int kPad = NB == 1 ? 0 : 16;
  __shared__ double Fs[2][kDepth][kN + kPad];  // [stage][inner][right-hand side]
  const int32_t block = xcd_block();
  const Task tk = load_task(desc, block / parts);
  const int32_t q0 = block % parts * kN;  // the block's first right-hand side
  if (a.live && !a.live[tk.s]) return;
  const int32_t r0 = tk.tile;
  const int32_t k0 = tk.k0, k1 = tk.k1;
  const int32_t slot = tk.slot;
  const int32_t nc = tk.nc, c0 = tk.c0;
  const int32_t m = tk.m;
  const int32_t kk = a.kk;
  const TW* W = w + tk.w_off;
  const int64_t vbase = tk.other;
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t / 64), lane = t % 64;
  const int li = lane % 16, lk = lane / 16;
  const bool rows_live = r0 + 16 * wave < m;  // wave-uniform
  // The wave's inner range: its rows of the leading block are zero past the diagonal.
  const int32_t wave_k1 = !rows_live ? 0 : min(k1, r0 + 16 * wave + 16 <= nc ? r0 + 16 * wave + 16 : nc);
  const bool applies = kGathers && slot < 0;  // the epilogue gathers too
  // The epilogue's gather pairs (this lane's update rows lane / 16 + 4v), loaded before the stages.
  int2 epair[4];
  int64_t erow[4];
  {
    bool elive[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int32_t i = r0 + 16 * wave + lk + 4 * v;
      erow[v] = vbase + i;
      elive[v] = applies && i >= nc && i < m;
    }
    gather_pairs<4>(a, erow, elive, epair);
  }
  // Operand step h of a stage: W row r0 + 16 wave + li at inner j0 + 4 h + lk (a row past the front
  // reads its last, whose product nothing stores).
  const uint32_t lane_w = (static_cast<uint32_t>(lk) * static_cast<uint32_t>(m) +
                           static_cast<uint32_t>(min(r0 + 16 * wave + li, m - 1))) * sizeof(TW);
  double wreg[4 * D];
  auto load_w = [&](int32_t j0) {
    if (j0 >= wave_k1) return;
    if (j0 + kDepth <= k1) {
#pragma unroll
      for (int h = 0; h < 4 * D; ++h)
        wreg[h] = widen(load_at(W + static_cast<int64_t>(j0 + 4 * h) * m, lane_w));
    } else {
#pragma unroll
      for (int h = 0; h < 4 * D; ++h)
        wreg[h] = j0 + 4 * h + lk < k1
                      ? widen(load_at(W + static_cast<int64_t>(j0 + 4 * h) * m, lane_w))
                      : 0.0;
    }
  };
  // f = r(cols) plus the children's updates: entry e = t + 256u of a stage is f column e % kN at
  // inner e / kN (past the range, its last row again, which W multiplies by zero). A stage's gather
  // pairs are loaded two stages ahead of its products, its entries one, and they are added and
  // staged after the products in between: nothing waits for a load it has just issued.
  int2 pair[U];
  double rreg[U], first[U], second[U];
  const int qe = q0 + t % kN, ql = min(qe, a.kk - 1);
  auto inner_of = [&](int32_t j0, int u) { return min(j0 + (t + 256 * u) / kN, k1 - 1); };
  auto load_pairs = [&](int32_t j0) {
    if (!kGathers) return;
    int64_t grow[U];
    bool glive[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      grow[u] = vbase + inner_of(j0, u);
      glive[u] = true;
    }
    gather_pairs<U>(a, grow, glive, pair);
  };
  int2 used[U];  // the pairs of the entries in flight
  auto load_f = [&](int32_t j0) {
    int q[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      q[u] = qe;
      rreg[u] = a.r[static_cast<int64_t>(c0 + inner_of(j0, u)) * kk + ql];
    }
    if constexpr (kGathers) {
#pragma unroll
      for (int u = 0; u < U; ++u) used[u] = pair[u];
      gather_issue<U>(a, used, q, first, second);
    }
  };
  auto stage = [&](int32_t j0, double (*F)[kN + kPad]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      double v = rreg[u];
      if constexpr (kGathers)
        v = gather_add(a, vbase + inner_of(j0, u), ql, used[u], first[u], second[u], v);
      F[(t + 256 * u) / kN][t % kN] = v;
    }
  };
  f64x4 acc[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) acc[n] = f64x4{0.0, 0.0, 0.0, 0.0};
  load_pairs(k0);
  load_w(k0);
  load_f(k0);
  if (k0 + kDepth < k1) load_pairs(k0 + kDepth);
  stage(k0, Fs[0]);
  __syncthreads();
  int p = 0;
  for (int32_t j0 = k0; j0 < k1; j0 += kDepth, p ^= 1) {
    double av[4 * D];
#pragma unroll
    for (int h = 0; h < 4 * D; ++h) av[h] = wreg[h];
    const bool more = j0 + kDepth < k1;
    if (more) {
      load_w(j0 + kDepth);
      load_f(j0 + kDepth);
      if (j0 + 2 * kDepth < k1) load_pairs(j0 + 2 * kDepth);
    }
    if (j0 < wave_k1)
#pragma unroll
      for (int h = 0; h < 4 * D; ++h) {
        double bv[NB];
#pragma unroll
        for (int n = 0; n < NB; ++n) bv[n] = Fs[p][4 * h + lk][16 * n + li];
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[n] = mfma16x16x4(av[h], bv[n], acc[n]);
      }
    if (more) {
      stage(j0 + kDepth, Fs[p ^ 1]);
      __syncthreads();
    }
  }
  if (!rows_live) return;
  // Epilogue: every load (the children's update rows that add into this tile's update rows) before
  // any is added or stored. A lane's outputs are rows lane / 16 + 4v of its wave's block; the sums
  // keep the gather's order (0, then each child in ascending order, then the product).
  double efirst[NB][4], esecond[NB][4];
  if (applies) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const double* one = update_row(a, epair[v].x) + q0 + li;
      const double* two = update_row(a, epair[v].y) + q0 + li;
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        efirst[n][v] = one[16 * n];
        esecond[n][v] = two[16 * n];
      }
    }
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int32_t ii = 16 * wave + lk + 4 * v;
    const int32_t i = r0 + ii;
    if (i >= m) continue;
    double* out = slot >= 0 ? a.partials + (static_cast<int64_t>(slot) * kTile + ii) * kk
                  : i < nc  ? a.y + static_cast<int64_t>(c0 + i) * kk
                            : a.fvec + (vbase + i) * kk;
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      const int q = q0 + 16 * n + li;
      if (q >= kk) continue;
      double value = acc[n][v];
      if (applies && i >= nc)
        value += gather_add(a, erow[v], q, epair[v], efirst[n][v], esecond[n][v], 0.0);
      out[q] = value;
    }
  }
}

// Adds the reduction partials of entries off[u] (offsets inside a slot of `stride` doubles) over
// slots [first, first + count) in slot order into sum[u]; four slots' loads are issued before
// their adds, so the loads overlap while each sum keeps its order.
__device__ __forceinline__ void add_partials(const double* __restrict__ partials, int64_t stride,
                                             int32_t first, int32_t count, const int64_t off[4],
                                             double sum[4]) {
  const double* p = partials + static_cast<int64_t>(first) * stride;
  int32_t c = 0;
  for (; c + 4 <= count; c += 4) {
    double v[4][4];
#pragma unroll
    for (int cc = 0; cc < 4; ++cc)
#pragma unroll
      for (int u = 0; u < 4; ++u) v[cc][u] = p[(c + cc) * stride + off[u]];
#pragma unroll
    for (int cc = 0; cc < 4; ++cc)
#pragma unroll
      for (int u = 0; u < 4; ++u) sum[u] += v[cc][u];
  }
  for (; c < count; ++c)
#pragma unroll
    for (int u = 0; u < 4; ++u) sum[u] += p[c * stride + off[u]];
}

// Adds a split forward tile's partials in slot order and applies the sum; blockIdx.y picks 16 of
// the tile's 64 rows.
__global__ __launch_bounds__(256) void fwd_reduce_kernel(const int4* __restrict__ rdesc,
                                                         SweepArgs a) {
  const Task g = load_task(rdesc, xcd_block());
  if (a.live && !a.live[g.s]) return;
  const int32_t r0 = g.tile;
  const int32_t first = g.k0, count = g.k1;
  const int32_t nc = g.nc, m = g.m, c0 = g.c0;
  const int32_t kk = a.kk;
  const int64_t vbase = g.other;
  constexpr int kRows = kTile / kReduceSplit;
  const int32_t lo = blockIdx.y * kRows;
  const int32_t rows = min(kRows, m - r0 - lo);
  // At most kRows * kCols = 4 x 256 entries: each thread's four, every load before any store.
  // Entries past the group's rows read slot offset 0 and store nothing.
  double sum[4] = {}, base[4] = {};
  int64_t off[4], grow[4];
  int gq[4];
  bool glive[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int32_t e = threadIdx.x + 256 * u;
    const bool live = e < rows * kk;
    const int32_t ii = live ? lo + e / kk : 0;
    off[u] = live ? static_cast<int64_t>(ii) * kk + e % kk : 0;
    grow[u] = vbase + r0 + ii;
    gq[u] = live ? e % kk : 0;
    glive[u] = live && r0 + ii >= nc;
  }
  int2 pair[4];
  double first_row[4], second_row[4];
  if (a.gathers) {
    gather_pairs<4>(a, grow, glive, pair);
    gather_issue<4>(a, pair, gq, first_row, second_row);
  }
  add_partials(a.partials, static_cast<int64_t>(kTile) * kk, first, count, off, sum);
  if (a.gathers)
#pragma unroll
    for (int u = 0; u < 4; ++u)
      base[u] = gather_add(a, grow[u], gq[u], pair[u], first_row[u], second_row[u], 0.0);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int32_t e = threadIdx.x + 256 * u;
    if (e >= rows * kk) continue;
    const int32_t ii = lo + e / kk, q = e % kk;
    const int32_t i = r0 + ii;
    if (i < nc) a.y[static_cast<int64_t>(c0 + i) * kk + q] = sum[u];
    else a.fvec[(vbase + i) * kk + q] = base[u] + sum[u];
  }
}

// Four consecutive entries of an inverse-factor column, widened (8-byte aligned: two loads of two
// doubles, or one of four floats).
__device__ __forceinline__ void load_four(const double* p, double (&v)[4]) {
  typedef double pair_t __attribute__((ext_vector_type(2), aligned(8)));
  const pair_t a = *reinterpret_cast<const pair_t*>(p);
  const pair_t b = *reinterpret_cast<const pair_t*>(p + 2);
  v[0] = a.x;
  v[1] = a.y;
  v[2] = b.x;
  v[3] = b.y;
}

__device__ __forceinline__ void load_four(const float* p, double (&v)[4]) {
  typedef float quad_t __attribute__((ext_vector_type(4), aligned(4)));
  const quad_t a = *reinterpret_cast<const quad_t*>(p);
  v[0] = a.x;
  v[1] = a.y;
  v[2] = a.z;
  v[3] = a.w;
}

// Backward tile product: inverse-factor columns [j0, j0+64) transposed, times
// g = [y(cols); d(rows)] over the inner range [k0, k1); each wave owns 16 of the columns. Applied
// results also give x_next = x + d when kIterate (a later round; the first round's d is the
// iterate itself, and its instance holds no iterate registers).
// A lane loads four consecutive rows 4 lk .. 4 lk + 3 of its column a stage: its column's sixteen
// rows of a stage are one 128-byte run, and operand step h contracts rows {4 g + h}, of both
// operands alike.
template <typename TW, int NB, bool kIterate>
__global__ __launch_bounds__(256, NB == 4 ? 5 : 6) void bwd_tile_kernel(
    const int4* __restrict__ desc, int32_t parts, const TW* __restrict__ w, SweepArgs a) {
  constexpr int D = kStages<NB>, kN = 16 * NB, kDepth = 16 * D, U = NB * D;
  constexpr int kPad = 4;
  __shared__ double Gs[2][kDepth][kN + kPad];  // [stage][inner][right-hand side]
  const int32_t block = xcd_block();
  const Task tk = load_task(desc, block / parts);
  const int32_t q0 = block % parts * kN;  // the block's first right-hand side
  const int32_t j0 = tk.tile;
  const int32_t slot = tk.slot;
  const int32_t nc = tk.nc, c0 = tk.c0;
  // A front the forward sweep did not reach has y = 0: its range starts past the leading block.
  const int32_t k0 = a.live && !a.live[tk.s] ? max(tk.k0, nc) : tk.k0, k1 = tk.k1;
  const int32_t m = tk.m;
  const int32_t kk = a.kk;
  const int32_t* srows = a.rows + tk.other;
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t / 64), lane = t % 64;
  const int li = lane % 16, lk = lane / 16;
  const bool cols_live = j0 + 16 * wave < nc;  // wave-uniform
  // The wave's inner range: its columns are zero above the diagonal.
  const int32_t wave_k0 = cols_live ? j0 + 16 * wave : k1;
  // A column past the front's reads its last, whose product nothing stores.
  const TW* W = w + tk.w_off;
  const uint32_t column = static_cast<uint32_t>(min(j0 + 16 * wave + li, nc - 1)) *
                              static_cast<uint32_t>(m) + 4 * lk;
  double wreg[D][4], greg[U];
  // A stage's structure-row indices are loaded a stage ahead (load_rows), so its W and g loads
  // issue together. Entry e = t + 256u of a stage is g's right-hand side e % kN at inner e / kN.
  int32_t srow[U];
  auto load_rows = [&](int32_t i0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int32_t ig = i0 + (t + 256 * u) / kN;
      srow[u] = (ig >= nc && ig < k1) ? srows[ig - nc] : 0;
    }
  };
  auto load = [&](int32_t i0) {
    if (i0 + kDepth > wave_k0) {
      if (i0 + kDepth <= k1) {  // uniform: the whole stage is inside the range
#pragma unroll
        for (int g = 0; g < D; ++g) load_four(W + column + i0 + 16 * g, wreg[g]);
      } else {
#pragma unroll
        for (int g = 0; g < D; ++g)
#pragma unroll
          for (int h = 0; h < 4; ++h)
            wreg[g][h] =
                i0 + 16 * g + 4 * lk + h < k1 ? widen(W[column + i0 + 16 * g + h]) : 0.0;
      }
    }
    // 32-bit element offsets from wave-uniform bases (a field stays under 2^31 entries), one
    // register an address.
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = t + 256 * u;
      const int q = q0 + e % kN;
      const int32_t ig = i0 + e / kN;
      double g = 0.0;
      if (q < kk && ig < k1) {
        if (ig < nc) g = a.y[static_cast<uint32_t>(c0 + ig) * static_cast<uint32_t>(kk) + q];
        else g = a.d[static_cast<uint32_t>(srow[u]) * static_cast<uint32_t>(kk) + q];
      }
      greg[u] = g;
    }
  };
  f64x4 acc[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) acc[n] = f64x4{0.0, 0.0, 0.0, 0.0};
  auto stage = [&](double (*G)[kN + kPad]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = t + 256 * u;
      G[e / kN][e % kN] = greg[u];
    }
  };
  const int32_t last = k0 < k1 ? k0 + (k1 - 1 - k0) / kDepth * kDepth : k0 - 1;
  if (k0 < k1) {
    load_rows(k0);
    load(k0);
    if (last > k0) load_rows(k0 + kDepth);
    stage(Gs[0]);
  }
  __syncthreads();
  int p = 0;
  for (int32_t i0 = k0; i0 <= last; i0 += kDepth, p ^= 1) {
    double av[D][4];
#pragma unroll
    for (int g = 0; g < D; ++g)
#pragma unroll
      for (int h = 0; h < 4; ++h) av[g][h] = wreg[g][h];
    const bool more = i0 < last;
    if (more) {
      load(i0 + kDepth);
      if (i0 + kDepth < last) load_rows(i0 + 2 * kDepth);
    }
    if (i0 + kDepth > wave_k0)
#pragma unroll
      for (int g = 0; g < D; ++g)
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          double bv[NB];
#pragma unroll
          for (int n = 0; n < NB; ++n) bv[n] = Gs[p][16 * g + 4 * lk + h][16 * n + li];
#pragma unroll
          for (int n = 0; n < NB; ++n) acc[n] = mfma16x16x4(av[g][h], bv[n], acc[n]);
        }
    if (more) {
      stage(Gs[p ^ 1]);
      __syncthreads();
    }
  }
  if (!cols_live) return;
  // Epilogue: the iterate's entries are all loaded before any store (see the forward tile).
  double xv[NB][4] = {};
  if (kIterate && slot < 0) {
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      const int q = q0 + 16 * n + li;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int32_t j = j0 + 16 * wave + lk + 4 * v;
        if (q < kk && j < nc) xv[n][v] = a.x[static_cast<int64_t>(c0 + j) * kk + q];
      }
    }
  }
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    const int q = q0 + 16 * n + li;
    if (q >= kk) continue;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int32_t jj = 16 * wave + lk + 4 * v;
      const int32_t j = j0 + jj;
      if (j >= nc) continue;
      const double value = acc[n][v];
      if (slot >= 0) {
        a.partials[(static_cast<int64_t>(slot) * kTile + jj) * kk + q] = value;
      } else {
        const int64_t at = static_cast<int64_t>(c0 + j) * kk + q;
        a.d[at] = value;
        if (kIterate) a.x_next[at] = xv[n][v] + value;
      }
    }
  }
}

__global__ __launch_bounds__(256) void bwd_reduce_kernel(const int4* __restrict__ rdesc,
                                                         SweepArgs a) {
  const Task g = load_task(rdesc, xcd_block());
  const int32_t j0 = g.tile;
  const int32_t first = g.k0, count = g.k1;
  const int32_t nc = g.nc, c0 = g.c0;
  const int32_t kk = a.kk;
  constexpr int kRows = kTile / kReduceSplit;
  const int32_t lo = blockIdx.y * kRows;
  const int32_t cols = min(kRows, nc - j0 - lo);
  // Each thread's (at most four) entries: every load before any store.
  const bool iterate = a.x != nullptr;
  double sum[4] = {}, xv[4] = {};
  int64_t off[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int32_t e = threadIdx.x + 256 * u;
    off[u] = e < cols * kk ? static_cast<int64_t>(lo + e / kk) * kk + e % kk : 0;
    if (iterate && e < cols * kk)
      xv[u] = a.x[static_cast<int64_t>(c0 + j0 + lo + e / kk) * kk + e % kk];
  }
  add_partials(a.partials, static_cast<int64_t>(kTile) * kk, first, count, off, sum);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int32_t e = threadIdx.x + 256 * u;
    if (e >= cols * kk) continue;
    const int32_t jj = lo + e / kk, q = e % kk;
    const int64_t at = static_cast<int64_t>(c0 + j0 + jj) * kk + q;
    a.d[at] = sum[u];
    if (iterate) a.x_next[at] = xv[u] + sum[u];
  }
}

// Raises *flag once per block that fails, and not at all once the flag reads set: with every row
// failing in a solve's first rounds, an atomic a wave on one word serializes the whole launch.
// Block-collective.
__device__ __forceinline__ void raise_flag(bool fail, int32_t* flag) {
  const int any = __syncthreads_or(fail ? 1 : 0);
  if (any && threadIdx.x == 0 &&
      __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
    atomicOr(flag, 1);
}

// r = b - A x in the elimination order and whether any row is still above tolerance
// (componentwise against (|A||x| + |b|)_i, normwise against the larger of that and the column's
// largest |b|; kernels/cholesky.py:1393-1440). Pinned rows are dropped. One thread a (row,
// right-hand side), for one and two right-hand sides.
__global__ void residual_kernel(const int32_t* __restrict__ offsets,
                                const int32_t* __restrict__ columns,
                                const double* __restrict__ values, const double* __restrict__ b,
                                const double* __restrict__ x, const int32_t* __restrict__ pinned,
                                const double* __restrict__ bmax, int64_t n, int32_t kk,
                                double tolerance, int32_t componentwise, double* __restrict__ r,
                                int32_t* __restrict__ pending) {
  int64_t t = static_cast<int64_t>(xcd_block()) * blockDim.x + threadIdx.x;
  bool fail = false;
  if (t < n * kk) {
    const int64_t i = t / kk;
    const int64_t q = t % kk;
    const double bi = b[t];
    const bool dropped = pinned && pinned[i];
    const double bscale = componentwise ? 0.0 : bmax[q];
    double total = bi, scale = fabs(bi);
    // Eight entries at a time (a row of a triangle mesh has about seven): their column and value
    // loads, then their iterate loads, issue together; entries past the row's end repeat its last
    // one and are not added, and the sums stay in entry order.
    const int32_t e0 = offsets[i], e1 = offsets[i + 1];
    for (int32_t e = e0; e < e1; e += 8) {
      int32_t c[8];
      double v[8], xv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int32_t at = min(e + u, e1 - 1);
        c[u] = columns[at];
        v[u] = values[at];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) xv[u] = x[static_cast<int64_t>(c[u]) * kk + q];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const double term = e + u < e1 ? v[u] * xv[u] : 0.0;  // subtracting 0 changes nothing
        total -= term;
        scale += fabs(term);
      }
    }
    if (r) r[t] = dropped ? 0.0 : total;
    if (!componentwise) scale = fmax(scale, bscale);
    fail = !dropped && !(fabs(total) <= tolerance * scale);
  }
  raise_flag(fail, pending);
}

// The residual of residual_kernel for three right-hand sides and more: a lane holds two columns of a
// row (the last lane of an odd number repeats one), a block the rows of pair_rows, whose entries it
// first brings into LDS (they lie in one run); a block of rows with more entries than it can hold reads
// them where they lie. A thread's first row of the right-hand side and of the iterate are loaded before
// the entries are (the iterate's for the caches alone: its row is some row's entry), which hides part of
// the chain offsets, entries, iterate (icosphere(9) at 16 columns: 267 us against 286). Sums keep entry
// order. 524,288-row torus: 32 columns 105 us (a lane a column 204), 64 columns 197 (214), where the
// rows fetched twice from beyond L2 hold it (850 MB at 4.4 TB/s; 570 are needed). The heat step's
// right-hand side is read where the bitmap of seeded rows has one (197 to 163).
// kLong: the plan has rows of more than kLongRow entries, which are dealt over the block's groups of
// lanes, a row at a time (a vertex of 8,000 neighbours, 20 columns: 1.6 ms with a wave a row, 2.5 with
// one group reading them all, 0.05 so; an instance of its own, since it takes 82 registers to 58).
constexpr int32_t kPairEntries = 1024;
constexpr int32_t kLongRow = 64;
template <bool kLong>
__global__ __launch_bounds__(256) void residual_pairs_kernel(
    const int32_t* __restrict__ offsets, const int32_t* __restrict__ columns,
    const double* __restrict__ values, const double* __restrict__ b,
    const double* __restrict__ x, const int32_t* __restrict__ pinned,
    const double* __restrict__ bmax, const uint32_t* __restrict__ seeded, int64_t n, int32_t kk,
    int32_t rows, double tolerance, int32_t componentwise, double* __restrict__ r,
    int32_t* __restrict__ pending) {
  __shared__ int32_t ptr[kPairRows + 1];
  __shared__ int32_t named[kPairEntries];
  __shared__ double staged[kPairEntries];
  constexpr int B = 8;
  const int32_t tid = static_cast<int32_t>(threadIdx.x);
  const int64_t first = static_cast<int64_t>(xcd_block()) * rows;
  const int32_t here = static_cast<int32_t>(min(static_cast<int64_t>(rows), n - first));
  if (tid <= here) ptr[tid] = offsets[first + tid];
  const int32_t lanes = (kk + 1) / 2, per = 256 / lanes, s0 = tid / lanes;
  const int32_t q = min(2 * (tid % lanes), kk - 2);
  const bool takes = s0 < min(per, here);
  // b's entries of row s; seeded (nullable): only rows flagged there have any.
  auto right_hand_side = [&](int32_t s) {
    const int64_t i = first + s;
    if (seeded && !(seeded[i / 32] >> (i % 32) & 1)) return Pair{0.0, 0.0};
    return __builtin_nontemporal_load(reinterpret_cast<const Pair*>(b + i * kk + q));
  };
  Pair b0 = {0.0, 0.0}, x0 = {0.0, 0.0};
  if (takes) {
    b0 = right_hand_side(s0);
    x0 = *reinterpret_cast<const Pair*>(x + (first + s0) * kk + q);
  }
  __syncthreads();
  const int32_t base = ptr[0], count = ptr[here] - base;
  const bool fits = count <= kPairEntries;
  if (fits)
    for (int32_t e = tid; e < count; e += 256) {
      named[e] = columns[base + e];
      staged[e] = values[base + e];
    }
  __syncthreads();
  asm volatile("" ::"v"(x0));  // loaded, though nothing takes its value
  const Pair bscale = componentwise ? Pair{0.0, 0.0} : *reinterpret_cast<const Pair*>(bmax + q);
  bool fail = false;
  auto within = [&](Pair total, Pair scale) {
    return fabs(total.x) <= tolerance * fmax(scale.x, bscale.x) &&
           fabs(total.y) <= tolerance * fmax(scale.y, bscale.y);
  };
  auto row = [&](int32_t s, const int32_t* names, const double* v) {
    if (kLong && ptr[s + 1] - ptr[s] > kLongRow) return;
    const int64_t i = first + s, at = i * kk + q;
    Pair total = s == s0 ? b0 : right_hand_side(s);
    Pair scale = {fabs(total.x), fabs(total.y)};
    const bool dropped = pinned && pinned[i];
    const int32_t e1 = ptr[s + 1] - base;
    for (int32_t e = ptr[s] - base; e < e1; e += B) {
      Pair xv[B];
#pragma unroll
      for (int u = 0; u < B; ++u)
        xv[u] = *reinterpret_cast<const Pair*>(
            x + static_cast<int64_t>(names[min(e + u, e1 - 1)]) * kk + q);
#pragma unroll
      for (int u = 0; u < B; ++u) {
        if (e + u >= e1) break;
        const double a = v[e + u];
        const double t0 = a * xv[u].x, t1 = a * xv[u].y;
        total.x -= t0;
        total.y -= t1;
        scale.x += fabs(t0);
        scale.y += fabs(t1);
      }
    }
    if (r) *reinterpret_cast<Pair*>(r + at) = dropped ? Pair{0.0, 0.0} : total;
    fail |= !dropped && !within(total, scale);
  };
  if (takes) {
    if (fits)
      for (int32_t s = s0; s < here; s += per) row(s, named, staged);
    else
      for (int32_t s = s0; s < here; s += per) row(s, columns + base, values + base);
  }
  if (kLong && count > kLongRow) {
    Pair* parts = reinterpret_cast<Pair*>(staged);  // [256] of the sums, [256] of the scales
    __syncthreads();
    for (int32_t s = 0; s < here; ++s) {
      const int32_t e1 = ptr[s + 1];
      if (e1 - ptr[s] <= kLongRow) continue;
      Pair sum = {0.0, 0.0}, size = {0.0, 0.0};
      if (s0 < per)
        for (int32_t e = ptr[s] + B * s0; e < e1; e += B * per) {
          int32_t c[B];
          double a[B];
#pragma unroll
          for (int u = 0; u < B; ++u) {
            c[u] = columns[min(e + u, e1 - 1)];
            a[u] = e + u < e1 ? values[e + u] : 0.0;
          }
#pragma unroll
          for (int u = 0; u < B; ++u) {
            const Pair xv = *reinterpret_cast<const Pair*>(x + static_cast<int64_t>(c[u]) * kk + q);
            const double t0 = e + u < e1 ? a[u] * xv.x : 0.0, t1 = e + u < e1 ? a[u] * xv.y : 0.0;
            sum.x += t0;
            sum.y += t1;
            size.x += fabs(t0);
            size.y += fabs(t1);
          }
        }
      parts[tid] = sum;
      parts[256 + tid] = size;
      __syncthreads();
      if (s0 == 0) {
        const int64_t i = first + s;
        Pair total = right_hand_side(s);
        Pair scale = {fabs(total.x), fabs(total.y)};
        for (int32_t g = 0; g < per; ++g) {
          total -= parts[tid + g * lanes];
          scale += parts[256 + tid + g * lanes];
        }
        const bool dropped = pinned && pinned[i];
        if (r) *reinterpret_cast<Pair*>(r + i * kk + q) = dropped ? Pair{0.0, 0.0} : total;
        fail |= !dropped && !within(total, scale);
      }
      __syncthreads();
    }
  }
  raise_flag(fail, pending);
}

// Per-column partial maxima of |b| (user layout), one block a (chunk, column).
__global__ void absmax_partial_kernel(const double* __restrict__ b, int64_t n,
                                      double* __restrict__ partials) {
  __shared__ double scratch[256];
  const int64_t q = blockIdx.y;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  scratch[threadIdx.x] = i < n ? fabs(b[q * n + i]) : 0.0;
  __syncthreads();
  for (int stride = 128; stride > 0; stride >>= 1) {
    if (threadIdx.x < stride) scratch[threadIdx.x] = fmax(scratch[threadIdx.x], scratch[threadIdx.x + stride]);
    __syncthreads();
  }
  if (threadIdx.x == 0) partials[q * gridDim.x + blockIdx.x] = scratch[0];
}

// The columns' largest values, and a solve's verdict cleared for its first round.
__global__ __launch_bounds__(256) void absmax_final_kernel(ColumnMaxima maxima,
                                                           int32_t* __restrict__ pending) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *pending = 0;
  fold_maxima(maxima, blockIdx.x);
}

// Component sums for the null-space projection: block partials per (component chunk, column).
__global__ void component_partial_kernel(const int32_t* __restrict__ chunk_comp,
                                         const int32_t* __restrict__ chunk_first,
                                         const int32_t* __restrict__ comp_ptr,
                                         const int32_t* __restrict__ members, int64_t n,
                                         const double* __restrict__ x,
                                         double* __restrict__ partials) {
  __shared__ double scratch[256];
  const int32_t chunk = blockIdx.x;
  const int64_t q = blockIdx.y;
  const int32_t c = chunk_comp[chunk];
  const int32_t e = chunk_first[chunk] + threadIdx.x;
  scratch[threadIdx.x] = e < comp_ptr[c + 1] ? x[q * n + members[e]] : 0.0;
  __syncthreads();
  for (int stride = 128; stride > 0; stride >>= 1) {
    if (threadIdx.x < stride) scratch[threadIdx.x] += scratch[threadIdx.x + stride];
    __syncthreads();
  }
  if (threadIdx.x == 0) partials[q * gridDim.x + chunk] = scratch[0];
}

// Each (component, column)'s mean, from its chunks' partials in chunk order.
__global__ void component_mean_kernel(const int32_t* __restrict__ comp_chunk_ptr,
                                      const int32_t* __restrict__ comp_ptr, int32_t n_chunks,
                                      const double* __restrict__ partials,
                                      double* __restrict__ means) {
  __shared__ double scratch[256];
  const int32_t c = blockIdx.x;
  const int64_t q = blockIdx.y;
  double sum = 0.0;
  for (int32_t k = comp_chunk_ptr[c] + threadIdx.x; k < comp_chunk_ptr[c + 1]; k += 256)
    sum += partials[q * n_chunks + k];
  scratch[threadIdx.x] = sum;
  __syncthreads();
  for (int stride = 128; stride > 0; stride >>= 1) {
    if (threadIdx.x < stride) scratch[threadIdx.x] += scratch[threadIdx.x + stride];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    means[q * gridDim.x + c] = scratch[0] / static_cast<double>(comp_ptr[c + 1] - comp_ptr[c]);
}

__global__ void component_shift_kernel(const int32_t* __restrict__ chunk_comp,
                                       const int32_t* __restrict__ chunk_first,
                                       const int32_t* __restrict__ comp_ptr,
                                       const int32_t* __restrict__ members, int32_t n_comp,
                                       int64_t n, const double* __restrict__ means,
                                       double* __restrict__ x) {
  const int32_t chunk = blockIdx.x;
  const int64_t q = blockIdx.y;
  const int32_t c = chunk_comp[chunk];
  const int32_t e = chunk_first[chunk] + threadIdx.x;
  if (e < comp_ptr[c + 1]) x[q * n + members[e]] -= means[q * n_comp + c];
}

// ---- the distance from a Poisson solution stored by rows ------------------------------------
// Every component's rows are contiguous in the elimination order (each component is dissected on
// its own and numbered in component order), so the null-space chunks (256 members of one
// component) are row ranges too: chunk k covers rows [chunk_first[k], min(+256, comp end)).

// Column sums over each chunk: a lane holds two columns of a row (one column: one row a thread), whose
// rows are added in turn, then over the block. partials[q * n_chunks + k], the layout
// component_mean_kernel reads. 16 columns on icosphere(9): 55 us (a lane a column of 64: 116).
__global__ __launch_bounds__(256) void rows_partial_kernel(const int32_t* __restrict__ chunk_comp,
                                                           const int32_t* __restrict__ chunk_first,
                                                           const int32_t* __restrict__ comp_ptr,
                                                           const double* __restrict__ x,
                                                           int32_t kk,
                                                           double* __restrict__ partials) {
  __shared__ Pair part[256];
  const int32_t chunk = blockIdx.x, tid = static_cast<int32_t>(threadIdx.x);
  const int32_t first = chunk_first[chunk];
  const int32_t end = min(first + 256, comp_ptr[chunk_comp[chunk] + 1]);
  const int32_t lanes = (kk + 1) / 2, per = 256 / lanes, s = tid / lanes;
  const int32_t q = max(min(2 * (tid % lanes), kk - 2), 0);
  Pair sum = {0.0, 0.0};
  if (kk == 1) {
    if (first + s < end) sum.x = x[first + s];
  } else if (s < per) {
    for (int32_t r = first + s; r < end; r += 8 * per) {
      Pair v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        v[u] = *reinterpret_cast<const Pair*>(
            x + static_cast<int64_t>(min(r + u * per, end - 1)) * kk + q);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (r + u * per < end) sum += v[u];
    }
  }
  part[tid] = sum;
  for (int32_t c = per; c > 1;) {
    const int32_t half = (c + 1) / 2;
    __syncthreads();
    if (s < c - half) part[tid] += part[tid + half * lanes];
    c = half;
  }
  if (s > 0) return;
  partials[static_cast<int64_t>(q) * gridDim.x + chunk] = part[tid].x;
  if (kk > 1) partials[static_cast<int64_t>(q + 1) * gridDim.x + chunk] = part[tid].y;
}

// One block per column q, after each component's mean (component_mean_kernel,
// kernels/cholesky.py:1467-1660): the shift of the mean-removed field (kernels/heat.py:3383-3424),
// offset = its mean over the column's sources (vertex v at row iperm[v]), negated when its mean
// over every vertex (the chunks' sums less their share of the means) is below the offset.
// shift[2q] = offset, shift[2q + 1] = 1 to negate. own_mean: the one component's mean is formed here
// too (a launch less: 4.7 us of a small call), and left in means.
__global__ __launch_bounds__(256) void rows_decide_kernel(
    const int32_t* __restrict__ comp_ptr, const int32_t* __restrict__ chunk_comp,
    const int32_t* __restrict__ chunk_first, int32_t n_comp, int32_t n_chunks,
    const double* __restrict__ partials, double* means, bool own_mean,
    const double* __restrict__ x, int32_t kk, int64_t n, const int32_t* __restrict__ iperm,
    const int32_t* __restrict__ labels, const int32_t* __restrict__ sources,
    const int64_t* __restrict__ source_offsets, double* __restrict__ shift) {
  __shared__ double s_total[256];
  __shared__ double s_src[256];
  const int q = blockIdx.x, t = threadIdx.x;
  double* mean = means + static_cast<int64_t>(q) * n_comp;
  if (own_mean) {
    double sum = 0.0;
#pragma unroll 8
    for (int32_t k = t; k < n_chunks; k += 256)
      sum += partials[static_cast<int64_t>(q) * n_chunks + k];
    s_total[t] = sum;
    __syncthreads();
    for (int stride = 128; stride > 0; stride >>= 1) {
      if (t < stride) s_total[t] += s_total[t + stride];
      __syncthreads();
    }
    if (t == 0) mean[0] = s_total[0] / static_cast<double>(comp_ptr[1] - comp_ptr[0]);
    __syncthreads();
  }
  double total = 0.0;
#pragma unroll 4
  for (int32_t k = t; k < n_chunks; k += 256) {
    const int32_t c = chunk_comp[k];
    const int32_t len = min(256, comp_ptr[c + 1] - chunk_first[k]);
    total += partials[static_cast<int64_t>(q) * n_chunks + k] - static_cast<double>(len) * mean[c];
  }
  const int64_t first = source_offsets[q], last = source_offsets[q + 1];
  double src = 0.0;
  for (int64_t e = first + t; e < last; e += 256) {
    const int32_t v = sources[e];
    if (v < 0 || v >= n) continue;  // out of range: the call fails once the stream is synced
    src += x[static_cast<int64_t>(iperm[v]) * kk + q] - mean[labels[v]];
  }
  s_total[t] = total;
  s_src[t] = src;
  __syncthreads();
  for (int stride = 128; stride > 0; stride >>= 1) {
    if (t < stride) {
      s_total[t] += s_total[t + stride];
      s_src[t] += s_src[t + stride];
    }
    __syncthreads();
  }
  if (t == 0) {
    const int64_t count = last - first;
    const double offset = count > 0 ? s_src[0] / static_cast<double>(count) : 0.0;
    shift[2 * q] = offset;
    shift[2 * q + 1] =
        (count > 0 && s_total[0] / static_cast<double>(n) - offset < 0.0) ? 1.0 : 0.0;
  }
}

// The distance in the caller's layout (column q at q * n): vertex v's entry is the mean-removed
// value at row iperm[v], shifted and oriented. 64 vertices a block, transposed through LDS so the
// row reads and the column writes are both contiguous: a lane reads two columns of each of its rows,
// all of them before any is used, and the tile is W columns wide (16, 32 or 64: a wider one than the
// chunk keeps blocks off the unit). 16 columns on icosphere(9): 131 us (64 wide, an element a lane: 275).
template <int W>
__global__ __launch_bounds__(256) void rows_out_kernel(const double* __restrict__ x, int32_t kk,
                                                       int64_t n, const int32_t* __restrict__ iperm,
                                                       const int32_t* __restrict__ labels,
                                                       int32_t n_comp,
                                                       const double* __restrict__ means,
                                                       const double* __restrict__ shift,
                                                       double* const* __restrict__ out_slot) {
  constexpr int kTurns = W / 8;  // rows a thread takes: 64 over the 256 / (W / 2) read at once
  __shared__ double tile[kTile][W + 1];
  double* __restrict__ out = *out_slot;
  const int64_t v0 = static_cast<int64_t>(blockIdx.x) * kTile;
  const int32_t rows = static_cast<int32_t>(min<int64_t>(kTile, n - v0));
  const int32_t tid = static_cast<int32_t>(threadIdx.x);
  if (kk == 1) {
    if (tid < rows) {
      const double value = x[iperm[v0 + tid]] - means[n_comp > 1 ? labels[v0 + tid] : 0];
      out[v0 + tid] = shift[1] != 0.0 ? shift[0] - value : value - shift[0];
    }
    return;
  }
  const int32_t lanes = (kk + 1) / 2, per = 256 / lanes, s = tid / lanes;
  const int32_t q = min(2 * (tid % lanes), kk - 2);
  if (s < per) {
    const double offset0 = shift[2 * q], offset1 = shift[2 * q + 2];
    const bool flip0 = shift[2 * q + 1] != 0.0, flip1 = shift[2 * q + 3] != 0.0;
    Pair xv[kTurns], mv[kTurns];
#pragma unroll
    for (int j = 0; j < kTurns; ++j) {
      const int64_t v = v0 + min(s + j * per, rows - 1);
      xv[j] = *reinterpret_cast<const Pair*>(x + static_cast<int64_t>(iperm[v]) * kk + q);
      const int32_t c = n_comp > 1 ? labels[v] : 0;
      mv[j] = Pair{means[static_cast<int64_t>(q) * n_comp + c],
                   means[static_cast<int64_t>(q + 1) * n_comp + c]};
    }
#pragma unroll
    for (int j = 0; j < kTurns; ++j) {
      const int32_t lv = s + j * per;
      if (lv >= rows) break;
      const Pair value = xv[j] - mv[j];
      tile[lv][q] = flip0 ? offset0 - value.x : value.x - offset0;
      tile[lv][q + 1] = flip1 ? offset1 - value.y : value.y - offset1;
    }
  }
  __syncthreads();
  const int lv = threadIdx.x % kTile, qq = threadIdx.x / kTile;
  if (lv >= rows) return;
  for (int q = qq; q < kk; q += 4) out[static_cast<int64_t>(q) * n + v0 + lv] = tile[lv][q];
}

// Marks every front from each source's row's to its root. The heat step's right-hand side is 64
// seeds on the 524,288-row torus, whose forward sweep reaches 2 % of the leaves: skipping the rest,
// and in the backward sweep the leading blocks they would multiply by zero, takes that sweep from
// 1,200 to 795 us (16 seeds on icosphere(9) 2,480 to 1,420, one on the torus 415 to 276).
__global__ __launch_bounds__(256) void mark_fronts_kernel(
    const int32_t* __restrict__ sources, const int64_t* __restrict__ offsets, int32_t kk,
    int64_t count, int64_t n, const int32_t* __restrict__ iperm,
    const int32_t* __restrict__ row_front, const int32_t* __restrict__ parent,
    int32_t* __restrict__ live) {
  const int64_t first = offsets ? offsets[0] : 0, last = offsets ? offsets[kk] : count;
  for (int64_t e = first + static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; e < last;
       e += static_cast<int64_t>(gridDim.x) * 256) {
    const int32_t v = sources[e];
    if (v < 0 || v >= n) continue;  // out of range: the call fails once the stream is synced
    // A front already marked has its ancestors marked, or being marked by whoever marked it.
    for (int32_t s = row_front[iperm[v]]; s >= 0 && atomicExch(live + s, 1) == 0; s = parent[s]) {
    }
  }
}

// The gather pairs of the live fronts' rows, without the contributions of fronts that are not. A wave
// a front, eight of each lane's rows at a time: the largest fronts, a thousand rows and more, are
// the launch's length (one source on icosphere(7): 21.5 us a row a lane at a time, 10.4 so; 16 on icosphere(9) 84 and 40).
__global__ __launch_bounds__(256) void live_pairs_kernel(
    const int32_t* __restrict__ live, const int32_t* __restrict__ ncol,
    const int32_t* __restrict__ nrow, const int64_t* __restrict__ vec_off,
    const int32_t* __restrict__ vec_front, const int2* __restrict__ pairs, int32_t n_super,
    int2* __restrict__ out) {
  const int32_t s = static_cast<int32_t>(blockIdx.x) * 4 + static_cast<int32_t>(threadIdx.x) / 64;
  if (s >= n_super || !live[s]) return;
  const int64_t base = vec_off[s];
  const int32_t m = ncol[s] + nrow[s];
  constexpr int U = 8;
  for (int32_t i = static_cast<int32_t>(threadIdx.x) % 64; i < m; i += 64 * U) {
    int2 p[U];
    int32_t fx[U], fy[U];
#pragma unroll
    for (int u = 0; u < U; ++u) p[u] = pairs[base + min(i + 64 * u, m - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      fx[u] = p[u].x >= 0 ? vec_front[p[u].x] : s;  // the front itself is live
      fy[u] = p[u].y >= 0 ? vec_front[p[u].y] : s;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      fx[u] = live[fx[u]];
      fy[u] = live[fy[u]];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i + 64 * u < m)
        out[base + i + 64 * u] = make_int2(fx[u] ? p[u].x : -1, fy[u] ? p[u].y : -1);
  }
}

inline unsigned blocks_for(int64_t n) { return static_cast<unsigned>((n + 255) / 256); }

// A tile kernel for 16 NB right-hand sides a block, and the blocks a tile's columns take. The matrix
// cores take right-hand sides sixteen at a time, so a chunk is padded to 16, 32 or 64: 5 columns on
// the 524,288-row torus took 898 us a sweep padded to 64 and take 636 padded to 16, 32 took 1,043 and
// take 884, 16 on icosphere(9) 3.75 ms and 2.58. Five waves a SIMD for the 64-column instances (six
// spill: 1.32 -> 1.78 ms).
template <typename Kernel>
struct TileChoice {
  Kernel kernel;
  int32_t parts;
};

template <typename TW>
using TileKernel = void (*)(const int4*, int32_t, const TW*, SweepArgs);

template <typename TW>
TileChoice<TileKernel<TW>> forward_tile(int32_t kk, int32_t blocks, bool gathers) {
  const int32_t parts = (kk + 16 * blocks - 1) / (16 * blocks);
  if (blocks == 1) return {gathers ? fwd_tile_kernel<TW, 1, true> : fwd_tile_kernel<TW, 1, false>, parts};
  if (blocks == 2) return {gathers ? fwd_tile_kernel<TW, 2, true> : fwd_tile_kernel<TW, 2, false>, parts};
  return {gathers ? fwd_tile_kernel<TW, 4, true> : fwd_tile_kernel<TW, 4, false>, parts};
}

template <typename TW>
TileChoice<TileKernel<TW>> backward_tile(int32_t kk, int32_t blocks, bool iterate) {
  const int32_t parts = (kk + 16 * blocks - 1) / (16 * blocks);
  if (blocks == 1) return {iterate ? bwd_tile_kernel<TW, 1, true> : bwd_tile_kernel<TW, 1, false>, parts};
  if (blocks == 2) return {iterate ? bwd_tile_kernel<TW, 2, true> : bwd_tile_kernel<TW, 2, false>, parts};
  return {iterate ? bwd_tile_kernel<TW, 4, true> : bwd_tile_kernel<TW, 4, false>, parts};
}

// The leaves are bound by their bytes and take a tile's columns in one block (split in two, the
// forward leaves took 25 us more of 235 on the 524,288-row torus). Past them a level is bound by its
// tiles' chains of dependent loads, and splitting its columns over blocks shortens and multiplies
// them: 32 columns a block, 16 in a level of few tiles (64 columns, a sweep, with whole tiles, with
// halves, with quarters: torus 1,304, 1,274 and 1,314 us, icosphere(7) 562, 523 and 518).
constexpr int32_t kNarrowTasks = 512;

int32_t column_blocks(int32_t kk, int32_t tasks, bool leaves) {
  const int32_t most = kk <= 16 ? 1 : kk <= 32 ? 2 : 4;
  if (leaves) return most;
  return tasks >= kNarrowTasks ? std::min(most, 2) : 1;
}

template <typename TW>
void sweep(const DevicePlan& plan, const TW* w, SweepArgs a, hipStream_t stream) {
  const int list = a.kk <= 16 ? 0 : 1;
  const DevicePlan::SweepTasks& F = plan.fwd[list];
  const DevicePlan::SweepTasks& B = plan.bwd[list];
  for (int32_t level = 0; level < plan.n_levels; ++level) {
    const int32_t t0 = F.level_ptr[level];
    const int32_t tasks = F.level_ptr[level + 1] - t0;
    if (tasks == 0) continue;
    a.gathers = plan.level_gathers[level];
    const auto tile = forward_tile<TW>(a.kk, column_blocks(a.kk, tasks, !a.gathers), a.gathers);
    tile.kernel<<<tasks * tile.parts, 256, 0, stream>>>(F.desc.ptr + 3 * static_cast<int64_t>(t0),
                                                        tile.parts, w, a);
    const int32_t r0 = F.reduce_ptr[level];
    const int32_t groups = F.reduce_ptr[level + 1] - r0;
    if (groups > 0) {
      fwd_reduce_kernel<<<dim3(groups, kReduceSplit), 256, 0, stream>>>(
          F.rdesc.ptr + 3 * static_cast<int64_t>(r0), a);
    }
  }
  a.gathers = 0;
  for (int32_t level = plan.n_levels - 1; level >= 0; --level) {
    const int32_t t0 = B.level_ptr[level];
    const int32_t tasks = B.level_ptr[level + 1] - t0;
    if (tasks == 0) continue;
    const auto tile = backward_tile<TW>(a.kk, column_blocks(a.kk, tasks, level == 0), a.x != nullptr);
    tile.kernel<<<tasks * tile.parts, 256, 0, stream>>>(B.desc.ptr + 3 * static_cast<int64_t>(t0),
                                                        tile.parts, w, a);
    const int32_t r0 = B.reduce_ptr[level];
    const int32_t groups = B.reduce_ptr[level + 1] - r0;
    if (groups > 0) {
      bwd_reduce_kernel<<<dim3(groups, kReduceSplit), 256, 0, stream>>>(
          B.rdesc.ptr + 3 * static_cast<int64_t>(r0), a);
    }
  }
  HG_HIP(hipGetLastError());
}

}  // namespace

void SolveWorkspace::reserve(const DevicePlan& plan, int64_t kk_needed) {
  // Sized for the next power of two of columns: a caller whose batches vary in width reallocates
  // (a hipFree waits on every stream's work) a handful of times, not once per new width.
  int64_t kk = 1;
  while (kk < kk_needed) kk *= 2;
  kk = std::min<int64_t>(kk, kCols);
  const int64_t entries = plan.n * kk;
  if (capacity < entries) {
    capacity = 0;  // while any of them may be missing
    bp.allocate(entries);
    xa.allocate(entries);
    xb.allocate(entries);
    r.allocate(entries);
    y.allocate(entries);
    d.allocate(entries);
    capacity = entries;
  }
  if (fcap < plan.vec_size * kk) {
    fcap = 0;
    fvec.allocate(plan.vec_size * kk + kCols);  // the gathers' padding
    fcap = plan.vec_size * kk;
  }
  const int64_t pentries = std::max(plan.max_slots[0] * std::min<int64_t>(kk, 16),
                                    kk > 16 ? plan.max_slots[1] * kk : 0) * kTile;
  if (pcap < pentries) {
    pcap = 0;
    partials.allocate(std::max<int64_t>(pentries, 1));
    pcap = pentries;
  }
  const int64_t absmax = static_cast<int64_t>(blocks_for(plan.n)) * kCols + kCols;
  if (bmax.size < absmax) bmax.allocate(absmax);
  if (pending.size < 1) pending.allocate(1);
  if (live.size < plan.n_super) live.allocate(plan.n_super);
  if (live_pairs.size < 2 * plan.vec_size) live_pairs.allocate(2 * plan.vec_size);
}

int32_t refined_solve(const DevicePlan& plan, const Factor& factor, bool use_fp32,
                      double* b, double* x, int64_t k, double tolerance, bool componentwise,
                      int32_t max_rounds, const int32_t* pinned_new, SolveWorkspace& ws,
                      hipStream_t stream, PhaseTimer* timer, int sweep_phase,
                      FieldLayout b_layout, FieldLayout x_layout, int32_t* speculate,
                      const SourceRows* nonzero, const double* maxima) {
  const int64_t n = plan.n;
  HG_REQUIRE(b_layout == FieldLayout::kColumns || componentwise || maxima, HG_ERR_RUNTIME,
             "a normwise solve of a right-hand side stored by rows takes its blocks' maxima");
  if (n == 0 || k == 0) return 0;
  int32_t max_used = 0;
  if (use_fp32) speculate = nullptr;
  for (int64_t q0 = 0; q0 < k; q0 += kCols) {
    const int32_t kk = static_cast<int32_t>(std::min<int64_t>(kCols, k - q0));
    // The backward tiles address a chunk's fields with 32-bit element offsets.
    HG_REQUIRE(n * kk < (int64_t{1} << 31), HG_ERR_VALUE,
               "a solve chunk of " + std::to_string(n) + " rows x " + std::to_string(kk) +
                   " columns exceeds 2^31 entries; solve fewer columns per call");
    ws.reserve(plan, kk);
    int32_t* const verdict = speculate ? speculate + q0 / kCols : ws.pending.ptr;
    double* bq = b + q0 * n;
    double* xq = x + q0 * n;
    const unsigned grid = blocks_for(n * kk);
    const unsigned row_tiles = static_cast<unsigned>((n + kTile - 1) / kTile);
    // The right-hand side in the elimination order with its pinned rows zero: b itself by rows
    // (zeroed in place below, or by what wrote a normwise solve's), else permuted into ws.bp.
    double* bp = b_layout == FieldLayout::kRows ? bq : ws.bp.ptr;
    if (b_layout == FieldLayout::kColumns)
      perm_in_kernel<<<row_tiles, 256, 0, stream>>>(bq, plan.perm.ptr, pinned_new, n, kk, bp);
    double* bmax = ws.bmax.ptr + static_cast<int64_t>(blocks_for(n)) * kCols;
    // The normwise scale: folded from blocks' maxima, which b stored by rows comes with, in the launch
    // that readies the first sweep.
    ColumnMaxima fold{};
    if (!componentwise) {
      const int64_t blocks =
          b_layout == FieldLayout::kRows ? divergence_blocks(n, kk) : blocks_for(n);
      if (b_layout == FieldLayout::kColumns)
        absmax_partial_kernel<<<dim3(static_cast<unsigned>(blocks), kk), 256, 0, stream>>>(
            bq, n, ws.bmax.ptr);
      fold = ColumnMaxima{b_layout == FieldLayout::kRows
                              ? maxima + q0 * divergence_blocks(n, kCols)
                              : ws.bmax.ptr,
                          static_cast<int32_t>(blocks), bmax};
    }
    if (b_layout == FieldLayout::kRows && componentwise && pinned_new)
      zero_pinned_rows_kernel<<<blocks_for(n), 256, 0, stream>>>(pinned_new, n, kk, bp);
    SweepArgs a{};
    a.col_begin = plan.col_begin.ptr;
    a.ncol = plan.ncol.ptr;
    a.nrow = plan.nrow.ptr;
    a.row_ptr = plan.row_ptr.ptr;
    a.rows = plan.rows.ptr;
    a.w_off = plan.w_off.ptr;
    a.vec_off = plan.vec_off.ptr;
    a.gather_pair = plan.gather_pair.ptr;
    a.gather_ptr = plan.gather_ptr.ptr;
    a.gather_src = plan.gather_src.ptr;
    a.fvec = ws.fvec.ptr;
    a.y = ws.y.ptr;
    a.partials = ws.partials.ptr;
    a.kk = kk;
    a.vec_front = plan.vec_front.ptr;
    const bool sparse =
        nonzero && b_layout == FieldLayout::kRows && plan.n_super >= kSparseFronts;
    const uint32_t* seeded =
        nonzero && b_layout == FieldLayout::kRows ? nonzero->seeded : nullptr;
    const LiveFronts reached{ws.live.ptr, ws.live_pairs.ptr};
    // The first round solves for the iterate itself from x = 0: its right-hand side is b and its
    // correction is written straight into the iterate. Later rounds correct it: d into ws.d and
    // x + d into the other iterate buffer. By rows the iterate lives in x itself (and ws.xa).
    double* const x_home = x_layout == FieldLayout::kRows ? xq : ws.xb.ptr;
    double* x_cur = x_home;
    int32_t rounds = 0;
    // A few columns sweep in one launch (flow.hip) while no such launch has given up here and the
    // device is claimed for it: by the call where the solve only enqueues, else by the solve, which
    // waits for every round.
    const bool narrow = kk <= kFlowColumns && !ws.level_sweeps &&
                        (!use_fp32 || plan.w_size <= kFlowFp32Entries);
    const WaitClaim claim(narrow && !speculate, false);
    const bool claimed = narrow && (speculate ? ws.flows : claim.held());
    while (rounds < max_rounds) {
      const bool flows = claimed && !ws.level_sweeps;
      double* x_next = x_cur == x_home ? ws.xa.ptr : x_home;
      if (rounds == 0) {
        a.r = bp;
        a.x = nullptr;
        a.x_next = nullptr;
        a.d = x_cur;
      } else {
        a.r = ws.r.ptr;
        a.x = x_cur;
        a.x_next = x_next;
        a.d = ws.d.ptr;
      }
      {
        PhaseScope scope(timer, sweep_phase, stream);
        // Only the first round's right-hand side is the caller's; a residual is dense.
        const bool marked = sparse && rounds == 0;
        if (marked) {
          launch_zero(ws.live.ptr, static_cast<int64_t>(sizeof(int32_t)) * plan.n_super, stream);
          mark_fronts_kernel<<<64, 256, 0, stream>>>(
              nonzero->sources, nonzero->offsets ? nonzero->offsets + q0 : nullptr, kk,
              nonzero->count, n, plan.iperm.ptr, plan.row_front.ptr, plan.parent.ptr, ws.live.ptr);
          live_pairs_kernel<<<static_cast<unsigned>((plan.n_super + 3) / 4), 256, 0, stream>>>(
              ws.live.ptr, plan.ncol.ptr, plan.nrow.ptr, plan.vec_off.ptr, plan.vec_front.ptr,
              reinterpret_cast<const int2*>(plan.gather_pair.ptr), plan.n_super,
              reinterpret_cast<int2*>(ws.live_pairs.ptr));
        }
        a.live = marked ? reached.live : nullptr;
        a.gather_pair = marked ? reached.pairs : plan.gather_pair.ptr;
        ++(flows ? ws.flow_count : ws.level_count);
        if (!flows) {
          if (fold.partials)
            absmax_final_kernel<<<kk, 256, 0, stream>>>(fold, verdict);
          else
            launch_zero(verdict, sizeof(int32_t), stream);
        }
        if (flows)
          flow_sweep(plan, factor, use_fp32, a.r, a.fvec, a.y, a.d, a.x, a.x_next, kk, fold,
                     verdict, ws.patience, marked ? &reached : nullptr, stream);
        else if (use_fp32) sweep<float>(plan, factor.w32.ptr, a, stream);
        else sweep<double>(plan, factor.w64.ptr, a, stream);
      }
      fold.partials = nullptr;  // once
      if (rounds > 0) x_cur = x_next;
      ++rounds;
      // Through FP64 factors the first round almost always passes, so its residual is formed for
      // the test alone and written (a second pass) only when another round follows.
      const bool test_only = !use_fp32 && rounds == 1;
      auto residual = [&](double* r_out) {
        // Pairs from three columns on (on the 524,288-row torus 46 us for two against 63, 47 against 67
        // at four; the rows' entries read once a column below).
        if (kk >= 3) {
          const int32_t rows = pair_rows(kk, n);
          auto kernel = plan.longest_row > kLongRow ? residual_pairs_kernel<true>
                                                    : residual_pairs_kernel<false>;
          kernel<<<static_cast<unsigned>((n + rows - 1) / rows), 256, 0, stream>>>(
              plan.p_offsets.ptr, plan.p_columns.ptr, factor.pvalues.ptr, bp, x_cur, pinned_new,
              bmax, seeded, n, kk, rows, tolerance,
              componentwise ? 1 : 0, r_out, verdict);
        } else {
          residual_kernel<<<grid, 256, 0, stream>>>(
              plan.p_offsets.ptr, plan.p_columns.ptr, factor.pvalues.ptr, bp, x_cur, pinned_new,
              bmax, n, kk, tolerance, componentwise ? 1 : 0, r_out, verdict);
        }
      };
      {
        PhaseScope scope(timer, kPhaseResidual, stream);
        residual(test_only ? nullptr : ws.r.ptr);
      }
      HG_HIP(hipGetLastError());
      if (speculate) break;
      int32_t pending = 0;
      HG_HIP(hipMemcpyAsync(&pending, verdict, sizeof(int32_t), hipMemcpyDeviceToHost,
                            stream));
      HG_HIP(hipStreamSynchronize(stream));
      if (timer) timer->resolve();
      if (!pending) break;
      if (pending & kFlowAborted) {  // nothing the round wrote counts: start over level by level
        ws.gave_up();
        x_cur = x_home;
        rounds = 0;
        continue;
      }
      if (test_only && rounds < max_rounds) {
        PhaseScope scope(timer, kPhaseResidual, stream);
        residual(ws.r.ptr);
        HG_HIP(hipGetLastError());
      }
    }
    if (x_layout == FieldLayout::kColumns)
      perm_out_kernel<<<row_tiles, 256, 0, stream>>>(x_cur, plan.perm.ptr, n, kk, xq);
    else if (x_cur != xq)
      HG_HIP(hipMemcpyAsync(xq, x_cur, sizeof(double) * n * kk, hipMemcpyDeviceToDevice, stream));
    HG_HIP(hipGetLastError());
    max_used = std::max(max_used, rounds);
  }
  return max_used;
}

void NullSpace::build(const std::vector<int32_t>& comp_ptr_host, hipStream_t stream) {
  n_comp = static_cast<int32_t>(comp_ptr_host.size()) - 1;
  std::vector<int32_t> cc, cf, ccp(n_comp + 1, 0);
  for (int32_t c = 0; c < n_comp; ++c) {
    for (int32_t e = comp_ptr_host[c]; e < comp_ptr_host[c + 1]; e += 256) {
      cc.push_back(c);
      cf.push_back(e);
    }
    ccp[c + 1] = static_cast<int32_t>(cc.size());
  }
  n_chunks = static_cast<int32_t>(cc.size());
  chunk_comp.upload(cc, stream);
  chunk_first.upload(cf, stream);
  comp_chunk_ptr.upload(ccp, stream);
}

void remove_null_space(const NullSpace& ns, const int32_t* comp_ptr, const int32_t* members,
                       int64_t n, int64_t k, double* x, DeviceArray<double>& scratch,
                       hipStream_t stream) {
  if (ns.n_chunks == 0 || k == 0) return;
  const int64_t need = static_cast<int64_t>(ns.n_chunks) * k + static_cast<int64_t>(ns.n_comp) * k;
  if (scratch.size < need) scratch.allocate(need);
  double* partials = scratch.ptr;
  double* means = scratch.ptr + static_cast<int64_t>(ns.n_chunks) * k;
  dim3 grid(static_cast<unsigned>(ns.n_chunks), static_cast<unsigned>(k));
  component_partial_kernel<<<grid, 256, 0, stream>>>(ns.chunk_comp.ptr, ns.chunk_first.ptr,
                                                     comp_ptr, members, n, x, partials);
  component_mean_kernel<<<dim3(static_cast<unsigned>(ns.n_comp), static_cast<unsigned>(k)), 256, 0,
                          stream>>>(ns.comp_chunk_ptr.ptr, comp_ptr, ns.n_chunks, partials, means);
  component_shift_kernel<<<grid, 256, 0, stream>>>(ns.chunk_comp.ptr, ns.chunk_first.ptr,
                                                   comp_ptr, members, ns.n_comp, n, means, x);
  HG_HIP(hipGetLastError());
}

void finish_rows(const DevicePlan& plan, const NullSpace& ns, const int32_t* comp_ptr,
                 const int32_t* labels, const double* x, int64_t k, const int32_t* sources,
                 const int64_t* source_offsets, double* const* out_slots,
                 DeviceArray<double>& scratch, hipStream_t stream, bool remove_means) {
  const int64_t n = plan.n;
  if (n == 0 || k == 0 || ns.n_chunks == 0) return;
  const int64_t need = static_cast<int64_t>(ns.n_chunks) * kCols +
                       static_cast<int64_t>(ns.n_comp) * kCols + 2 * kCols;
  if (scratch.size < need) scratch.allocate(need);
  double* partials = scratch.ptr;
  double* means = partials + static_cast<int64_t>(ns.n_chunks) * kCols;
  double* shift = means + static_cast<int64_t>(ns.n_comp) * kCols;
  for (int64_t q0 = 0; q0 < k; q0 += kCols) {
    const int32_t kk = static_cast<int32_t>(std::min<int64_t>(kCols, k - q0));
    const double* xq = x + q0 * n;
    rows_partial_kernel<<<static_cast<unsigned>(ns.n_chunks), 256, 0, stream>>>(
        ns.chunk_comp.ptr, ns.chunk_first.ptr, comp_ptr, xq, kk, partials);
    const bool own_mean = remove_means && ns.n_comp == 1;
    if (remove_means && !own_mean)
      component_mean_kernel<<<dim3(static_cast<unsigned>(ns.n_comp), static_cast<unsigned>(kk)),
                              256, 0, stream>>>(ns.comp_chunk_ptr.ptr, comp_ptr, ns.n_chunks,
                                                partials, means);
    else if (!remove_means)
      launch_zero(means, static_cast<int64_t>(sizeof(double)) * ns.n_comp * kk, stream);
    rows_decide_kernel<<<static_cast<unsigned>(kk), 256, 0, stream>>>(
        comp_ptr, ns.chunk_comp.ptr, ns.chunk_first.ptr, ns.n_comp, ns.n_chunks, partials, means,
        own_mean, xq, kk, n, plan.iperm.ptr, labels, sources, source_offsets + q0, shift);
    auto out = kk <= 16 ? rows_out_kernel<16> : kk <= 32 ? rows_out_kernel<32> : rows_out_kernel<64>;
    out<<<static_cast<unsigned>((n + kTile - 1) / kTile), 256, 0, stream>>>(
        xq, kk, n, plan.iperm.ptr, labels, ns.n_comp, means, shift, out_slots + q0 / kCols);
  }
  HG_HIP(hipGetLastError());
}

}  // namespace hg
