// The triangular sweeps of a few right-hand sides as one launch.
//
// Level by level (solve.hip) a sweep of one column is up to 60 launches, and past the leaves each
// is a chain of dependent loads over a few megabytes: 10 us a level and 5 more for its split
// products' sums, where the level's inverse factors pass in 1-2 us. Here the whole sweep, forward
// and backward, is one launch of independent tasks in dependency order. A task is a tile of one
// front over its whole inner range; it loads its part of the inverse factor into registers first,
// then waits for the values it multiplies, so the factor's bytes arrive while the levels below are
// still at work, and a level costs one hand-over: the update vectors, y and d are words that are
// their own arrival flags (words.h).
//
// A task waits only for tasks before it in the list. The hardware dispatches blocks in order, so
// the first unfinished task is always running and its inputs are there; every wait is bounded
// all the same, and a launch that gave up reports it (kFlowAborted in the pending word), upon
// which the solve starts over level by level.
//
// Both sweeps of a one-source query, level by level before this and now: icosphere(4) 180 -> 39 us (its
// three levels are six hand-overs of about 2.5 us a sweep), icosphere(7) 730 -> 248 us (the heat step's,
// over the fronts its source reaches, 105), the 524,288-row torus 1.77 ms -> 632 us (216 and 416: the
// second reads 1.49 GB, at 3.6 TB/s where 1.5).
//
// A forward task is 256 / LN rows of a front, LN threads a row splitting the inner range; a
// backward task is 16 * PASS columns, sixteen lanes a column along its rows. Every output is one
// task's: no partial products cross blocks, and each sum has one fixed order.
#include <exception>
#include <mutex>

#include "cholesky.h"
#include "words.h"

namespace hg {
namespace {

constexpr int kThreads = 256;
constexpr int kStage = 1024;  // staged vector entries

struct FlowArgs {
  const int4* desc;
  int32_t n_forward;
  int32_t kk;
  const double* r;
  double* fvec;
  double* y;
  double* d;
  const double* x;  // null on the first round
  double* x_next;
  const int2* gather_pair;
  const int32_t* gather_ptr;
  const int32_t* gather_src;
  const int32_t* rows;
  const int32_t* live;       // null: every front is
  const int32_t* vec_front;
  int32_t* pending;
  int64_t spin_limit;
};

struct FlowTask {
  int32_t shape, tile, inner, gathers, nc, c0, m, s;
  int64_t w_off, other;
};

__device__ __forceinline__ FlowTask load_flow(const int4* __restrict__ desc) {
  const int4 d0 = desc[0], d1 = desc[1], d2 = desc[2];
  FlowTask t;
  t.shape = d0.x;
  t.tile = d0.y;
  t.inner = d0.z;
  t.gathers = d0.w;
  t.nc = d1.x;
  t.c0 = d1.y;
  t.m = d1.z;
  t.s = d1.w;
  t.w_off = static_cast<int64_t>(static_cast<uint32_t>(d2.x)) | (static_cast<int64_t>(d2.y) << 32);
  t.other = static_cast<int64_t>(static_cast<uint32_t>(d2.z)) | (static_cast<int64_t>(d2.w) << 32);
  return t;
}

// The entry `bytes` past a block-uniform base: one address register a lane for a whole run of loads.
template <typename T>
__device__ __forceinline__ T load_at(const T* base, uint32_t bytes) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + bytes);
}

struct Patience {
  const FlowArgs& a;
  bool aborted = false;
  // The word's value, waiting for it from what a first look found.
  __device__ __forceinline__ double await(const double* word, uint64_t bits) {
    int32_t polls = 0;
    while (bits == kEmpty && wait_on(a.pending, kFlowAborted, a.spin_limit, polls, aborted)) {
      bits = peek(word);
    }
    return __builtin_bit_cast(double, bits);
  }
};

// N front-vector entries (row[u], column q[u]; live[u]): v[u] plus the children's update words in
// ascending child order. Every first look is issued before any is waited for.
template <int N>
__device__ __forceinline__ void gather_words(const FlowArgs& a, Patience& wait,
                                             const int2 (&pair)[N], const int64_t (&row)[N],
                                             const int32_t (&q)[N], double (&v)[N]) {
  uint64_t first[N], second[N];
#pragma unroll
  for (int u = 0; u < N; ++u) {
    first[u] = pair[u].x >= 0 ? peek(a.fvec + static_cast<int64_t>(pair[u].x) * a.kk + q[u]) : 0;
    second[u] = pair[u].y >= 0 ? peek(a.fvec + static_cast<int64_t>(pair[u].y) * a.kk + q[u]) : 0;
  }
#pragma unroll
  for (int u = 0; u < N; ++u) {
    if (pair[u].x >= 0)
      v[u] += wait.await(a.fvec + static_cast<int64_t>(pair[u].x) * a.kk + q[u], first[u]);
    if (pair[u].y >= 0) {
      v[u] += wait.await(a.fvec + static_cast<int64_t>(pair[u].y) * a.kk + q[u], second[u]);
    } else if (pair[u].y == -2) {
      for (int32_t g = a.gather_ptr[row[u]] + 1; g < a.gather_ptr[row[u] + 1]; ++g) {
        if (a.live && !a.live[a.vec_front[a.gather_src[g]]]) continue;
        const double* word = a.fvec + static_cast<int64_t>(a.gather_src[g]) * a.kk + q[u];
        v[u] += wait.await(word, peek(word));
      }
    }
  }
}

// Rows [tile, tile + 256 / LN) of a front's inverse factor times f over columns [0, inner): y and
// the update words.
template <typename TW, int KC, int LN>
__device__ __forceinline__ void forward_task(const FlowArgs& a, const FlowTask& tk,
                                             const TW* __restrict__ w, double* staged,
                                             double* parts) {
  constexpr int T = kThreads / LN;
  constexpr int P = 16;                // inverse-factor entries a thread loads ahead
  constexpr int kChunk = kStage / KC;  // inner indices staged at a time
  const int t = threadIdx.x, ii = t % T, kl = t / T;
  const int32_t kk = a.kk, K = tk.inner, m = tk.m, nc = tk.nc;
  const int32_t i = tk.tile + ii;
  const int64_t vbase = tk.other;
  // Entry (i, kl + LN u) is a lane's offset past column LN u's base. Lanes past the front's rows
  // or the inner range read an entry inside it, which nothing uses.
  const TW* W = w + tk.w_off;
  const uint32_t lane = (static_cast<uint32_t>(min(kl, K - 1)) * static_cast<uint32_t>(m) +
                         static_cast<uint32_t>(min(i, m - 1))) * sizeof(TW);
  auto entry = [&](int32_t j) {  // of column j + kl, j block-uniform
    return load_at(W + static_cast<int64_t>(j) * m, lane);
  };
  TW ahead[P];
#pragma unroll
  for (int u = 0; u < P; ++u)
    ahead[u] = LN * u + LN <= K || LN * u + kl < K ? entry(LN * u) : TW(0);
  Patience wait{a};
  double acc[KC];
#pragma unroll
  for (int q = 0; q < KC; ++q) acc[q] = 0.0;
  for (int32_t k0 = 0; k0 < K; k0 += kChunk) {
    const int32_t ke = min(kChunk, K - k0);
    {
      // f = r(cols) plus the children's update words, four entries a thread.
      constexpr int N = kStage / kThreads;
      int2 pair[N];
      int64_t row[N];
      int32_t q[N];
      double v[N];
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const int32_t e = t + kThreads * u;
        const bool live = e < ke * kk;
        row[u] = vbase + k0 + (live ? e / kk : 0);
        q[u] = live ? e % kk : 0;
        v[u] = live ? a.r[static_cast<int64_t>(tk.c0 + k0) * kk + e] : 0.0;
        pair[u] = live && tk.gathers ? a.gather_pair[row[u]] : make_int2(-1, -1);
      }
      gather_words<N>(a, wait, pair, row, q, v);
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const int32_t e = t + kThreads * u;
        if (e < ke * kk) staged[(e / kk) * KC + e % kk] = v[u];
      }
    }
    __syncthreads();
    int32_t j0 = 0;  // this thread's next index of the chunk, less kl
    if (k0 == 0) {
#pragma unroll
      for (int u = 0; u < P; ++u) {
        if (LN * u < ke) {  // block-uniform
          const double wv = static_cast<double>(ahead[u]);
          const double* f = staged + min(kl + LN * u, ke - 1) * KC;
#pragma unroll
          for (int q = 0; q < KC; ++q) acc[q] += wv * f[q];
        }
      }
      j0 = LN * P;
    }
    for (; j0 < ke; j0 += 8 * LN) {
      TW next[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        next[u] = j0 + LN * u + kl < ke ? entry(k0 + j0 + LN * u) : TW(0);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (j0 + LN * u + kl < ke) {
          const double wv = static_cast<double>(next[u]);
#pragma unroll
          for (int q = 0; q < KC; ++q) acc[q] += wv * staged[(j0 + LN * u + kl) * KC + q];
        }
    }
    if (k0 + kChunk < K) __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < KC; ++q) parts[(kl * T + ii) * KC + q] = acc[q];
  __syncthreads();
  for (int32_t o = t; o < T * kk; o += kThreads) {
    const int32_t lr = o / kk, q = o % kk, row = tk.tile + lr;
    if (row >= m) break;
    double sum = parts[lr * KC + q];
    for (int l = 1; l < LN; ++l) sum += parts[(l * T + lr) * KC + q];
    if (row < nc) {
      publish(a.y + static_cast<int64_t>(tk.c0 + row) * kk + q, sum);
    } else {
      double base[1] = {0.0};
      if (tk.gathers) {
        const int64_t at[1] = {vbase + row};
        const int32_t column[1] = {q};
        const int2 pair[1] = {a.gather_pair[at[0]]};
        gather_words<1>(a, wait, pair, at, column, base);
      }
      publish(a.fvec + (vbase + row) * kk + q, base[0] + sum);
    }
  }
}

// Columns [tile, tile + 16 PASS) of a front's inverse factor, transposed, times [y(cols); d(rows)]
// over rows [top, m): d and, after the first round, x + d. top is the tile, whose rows above are
// zero, or the first row past the leading block of a front whose y is.
template <typename TW, int KC, int PASS>
__device__ __forceinline__ void backward_task(const FlowArgs& a, const FlowTask& tk, int32_t top,
                                              const TW* __restrict__ w, double* staged) {
  constexpr int U = 16 / PASS;  // entries of a column a lane loads ahead
  constexpr int kChunk = kStage / KC;
  const int t = threadIdx.x, sub = t % 16, group = t / 16;
  const int32_t kk = a.kk, m = tk.m, nc = tk.nc, j0 = tk.tile;
  const int32_t* srows = a.rows + tk.other;
  const TW* W = w + tk.w_off;
  // Entry (top + sub + 16 u, j0 + group + 16 p) is a lane's offset past (top + 16 u, j0 + 16 p), the
  // group's column clamped to the front's last.
  uint32_t lane[PASS];
  auto entry = [&](int p, int32_t i) {  // of row top + i + sub, i block-uniform
    return load_at(W + static_cast<int64_t>(min(j0 + 16 * p, nc - 1)) * m + top + i, lane[p]);
  };
  TW ahead[PASS][U];
#pragma unroll
  for (int p = 0; p < PASS; ++p) {
    const int32_t last = max(0, nc - 1 - j0 - 16 * p);
    lane[p] = (static_cast<uint32_t>(min(group, last)) * static_cast<uint32_t>(m) + sub) * sizeof(TW);
#pragma unroll
    for (int u = 0; u < U; ++u) ahead[p][u] = top + sub + 16 * u < m ? entry(p, 16 * u) : TW(0);
  }
  Patience wait{a};
  double acc[PASS][KC];
#pragma unroll
  for (int p = 0; p < PASS; ++p)
#pragma unroll
    for (int q = 0; q < KC; ++q) acc[p][q] = 0.0;
  for (int32_t s0 = top; s0 < m; s0 += kChunk) {
    const int32_t se = min(kChunk, m - s0);
    {
      constexpr int N = kStage / kThreads;
      const double* word[N];
      uint64_t bits[N];
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const int32_t e = t + kThreads * u;
        const bool live = e < se * kk;
        const int32_t i = s0 + (live ? e / kk : 0), q = live ? e % kk : 0;
        word[u] = i < nc ? a.y + static_cast<int64_t>(tk.c0 + i) * kk + q
                         : a.d + static_cast<int64_t>(srows[i - nc]) * kk + q;
        bits[u] = live ? 1 : 0;
      }
#pragma unroll
      for (int u = 0; u < N; ++u)
        if (bits[u]) bits[u] = peek(word[u]);
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const int32_t e = t + kThreads * u;
        if (e < se * kk) staged[(e / kk) * KC + e % kk] = wait.await(word[u], bits[u]);
      }
    }
    __syncthreads();
    int32_t i0 = 0;  // this lane's next row of the chunk, less sub
    if (s0 == top) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (16 * u < se) {  // block-uniform
          const double* g = staged + min(sub + 16 * u, se - 1) * KC;
#pragma unroll
          for (int p = 0; p < PASS; ++p) {
            const double wv = static_cast<double>(ahead[p][u]);
#pragma unroll
            for (int q = 0; q < KC; ++q) acc[p][q] += wv * g[q];
          }
        }
      }
      i0 = 16 * U;
    }
    constexpr int B = PASS == 1 ? 8 : 2;
    for (; i0 < se; i0 += 16 * B) {
      TW next[PASS][B];
#pragma unroll
      for (int p = 0; p < PASS; ++p)
#pragma unroll
        for (int u = 0; u < B; ++u)
          next[p][u] = i0 + 16 * u + sub < se ? entry(p, s0 - top + i0 + 16 * u) : TW(0);
#pragma unroll
      for (int u = 0; u < B; ++u)
        if (i0 + 16 * u + sub < se) {
          const double* g = staged + (i0 + 16 * u + sub) * KC;
#pragma unroll
          for (int p = 0; p < PASS; ++p) {
            const double wv = static_cast<double>(next[p][u]);
#pragma unroll
            for (int q = 0; q < KC; ++q) acc[p][q] += wv * g[q];
          }
        }
    }
    if (s0 + kChunk < m) __syncthreads();
  }
#pragma unroll
  for (int p = 0; p < PASS; ++p) {
#pragma unroll
    for (int q = 0; q < KC; ++q)
#pragma unroll
      for (int offset = 8; offset >= 1; offset >>= 1)
        acc[p][q] += __shfl_xor(acc[p][q], offset, 16);
    const int32_t j = j0 + group + 16 * p;
    if (j >= nc || sub >= kk) continue;
    double mine = acc[p][0];
#pragma unroll
    for (int q = 1; q < KC; ++q)
      if (q == sub) mine = acc[p][q];
    const int64_t at = static_cast<int64_t>(tk.c0 + j) * kk + sub;
    publish(a.d + at, mine);
    if (a.x) a.x_next[at] = a.x[at] + mine;
  }
}

// Four blocks a compute unit, with sixteen entries a thread loaded ahead: icosphere(7) takes 160 us a
// sweep so; two blocks with 32 entries 184, six with eight (spilling) 226.
template <typename TW, int KC>
__global__ __launch_bounds__(kThreads, 4) void flow_kernel(const TW* __restrict__ w, FlowArgs a) {
  __shared__ double staged[kStage];
  __shared__ double parts[kThreads * KC];
  const FlowTask tk = load_flow(a.desc + 3 * static_cast<int64_t>(blockIdx.x));
  if (static_cast<int32_t>(blockIdx.x) < a.n_forward) {
    if (a.live && !a.live[tk.s]) return;  // y = 0 and no updates, which nobody waits for
    if (tk.shape == 1) forward_task<TW, KC, 1>(a, tk, w, staged, parts);
    else if (tk.shape == 4) forward_task<TW, KC, 4>(a, tk, w, staged, parts);
    else forward_task<TW, KC, 16>(a, tk, w, staged, parts);
  } else {
    const int32_t top = a.live && !a.live[tk.s] ? tk.nc : tk.tile;
    if (tk.shape == 4) backward_task<TW, KC, 4>(a, tk, top, w, staged);
    else backward_task<TW, KC, 1>(a, tk, top, w, staged);
  }
}

// Every word the sweep hands over emptied, the solve's verdict cleared, and (partials not null) the
// columns' largest values folded by its first blocks.
__global__ __launch_bounds__(256) void flow_empty_kernel(uint64_t* __restrict__ y,
                                                         uint64_t* __restrict__ d,
                                                         int64_t entries,
                                                         uint64_t* __restrict__ fvec,
                                                         int64_t updates,
                                                         int32_t* __restrict__ pending,
                                                         ColumnMaxima maxima, int32_t kk) {
  if (maxima.partials)
    for (int32_t q = static_cast<int32_t>(blockIdx.x); q < kk; q += static_cast<int32_t>(gridDim.x)) {
      fold_maxima(maxima, q);
      __syncthreads();
    }
  const int64_t first = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  if (first == 0) *pending = 0;
  for (int64_t e = first; e < entries; e += stride) {
    y[e] = kEmpty;
    d[e] = kEmpty;
  }
  for (int64_t e = first; e < updates; e += stride) fvec[e] = kEmpty;
}

template <typename TW>
void launch_flow(const TW* w, const FlowArgs& a, unsigned tasks, hipStream_t stream) {
  auto kernel = a.kk == 1   ? flow_kernel<TW, 1>
                : a.kk == 2 ? flow_kernel<TW, 2>
                            : flow_kernel<TW, 4>;
  kernel<<<tasks, kThreads, 0, stream>>>(w, a);
}

}  // namespace

HostFlow flow_tasks(const Plan& plan) {
  HostFlow out;
  auto push = [&](int32_t shape, int32_t tile, int32_t inner, int32_t s, int64_t other) {
    const int32_t nc = plan.ncol[s], m = nc + plan.nrow[s];
    const int32_t gathers = plan.child_ptr[s + 1] > plan.child_ptr[s] ? 1 : 0;
    const int64_t w = plan.w_off[s];
    for (int32_t v : {shape, tile, inner, gathers, nc, plan.col_begin[s], m, s,
                      static_cast<int32_t>(static_cast<uint32_t>(w)), static_cast<int32_t>(w >> 32),
                      static_cast<int32_t>(static_cast<uint32_t>(other)),
                      static_cast<int32_t>(other >> 32)})
      out.desc.push_back(v);
  };
  // Tiles of a level: 64 wide where that makes enough of them to fill the compute units, else 16.
  auto tiles = [&](int32_t level, bool forward) {
    int64_t total = 0;
    for (int32_t k = plan.level_ptr[level]; k < plan.level_ptr[level + 1]; ++k) {
      const int32_t s = plan.level_nodes[k];
      total += (plan.ncol[s] + (forward ? plan.nrow[s] : 0) + 63) / 64;
    }
    return total;
  };
  for (int32_t level = 0; level < plan.n_levels; ++level) {
    const bool wide = tiles(level, true) >= kFlowWideTiles;
    for (int32_t k = plan.level_ptr[level]; k < plan.level_ptr[level + 1]; ++k) {
      const int32_t s = plan.level_nodes[k];
      const int32_t nc = plan.ncol[s], m = nc + plan.nrow[s];
      const int32_t shape = nc <= 32 ? 1 : wide ? 4 : 16;
      const int32_t rows = 256 / shape;
      for (int32_t tile = 0; tile < m; tile += rows)  // the leading block is lower triangular
        push(shape, tile, std::min(nc, tile + rows), s, plan.vec_off[s]);
    }
  }
  out.n_forward = static_cast<int32_t>(out.desc.size() / 12);
  for (int32_t level = plan.n_levels - 1; level >= 0; --level) {
    const bool wide = tiles(level, false) >= kFlowWideTiles;
    for (int32_t k = plan.level_ptr[level]; k < plan.level_ptr[level + 1]; ++k) {
      const int32_t s = plan.level_nodes[k];
      const int32_t nc = plan.ncol[s];
      const int32_t shape = wide && nc > 16 ? 4 : 1;
      for (int32_t tile = 0; tile < nc; tile += 16 * shape)
        push(shape, tile, 0, s, plan.row_ptr[s]);
    }
  }
  return out;
}

namespace {
constexpr int kClaimDevices = 64;
std::mutex g_wait_claims[kClaimDevices];
thread_local bool t_holds_claim[kClaimDevices] = {};
}  // namespace

WaitClaim::WaitClaim(bool wanted, bool wait) {
  if (!wanted) return;
  HG_HIP(hipGetDevice(&device_));
  if (device_ >= kClaimDevices) return;
  held_ = t_holds_claim[device_];
  if (held_) return;
  if (wait) g_wait_claims[device_].lock();
  else if (!g_wait_claims[device_].try_lock()) return;
  unwinding_ = std::uncaught_exceptions();
  held_ = owner_ = t_holds_claim[device_] = true;
}

WaitClaim::~WaitClaim() {
  if (!owner_) return;
  // A call that throws leaves work running.
  if (std::uncaught_exceptions() > unwinding_) (void)hipDeviceSynchronize();
  t_holds_claim[device_] = false;
  g_wait_claims[device_].unlock();
}

void flow_sweep(const DevicePlan& plan, const Factor& factor, bool use_fp32, const double* r,
                double* fvec, double* y, double* d, const double* x, double* x_next, int32_t kk,
                const ColumnMaxima& maxima, int32_t* pending, int64_t patience, const LiveFronts* live_fronts,
                hipStream_t stream) {
  FlowArgs a{};
  a.desc = plan.flow_desc.ptr;
  a.n_forward = plan.flow_forward;
  a.kk = kk;
  a.r = r;
  a.fvec = fvec;
  a.y = y;
  a.d = d;
  a.x = x;
  a.x_next = x_next;
  a.gather_pair =
      reinterpret_cast<const int2*>(live_fronts ? live_fronts->pairs : plan.gather_pair.ptr);
  a.live = live_fronts ? live_fronts->live : nullptr;
  a.vec_front = plan.vec_front.ptr;
  a.gather_ptr = plan.gather_ptr.ptr;
  a.gather_src = plan.gather_src.ptr;
  a.rows = plan.rows.ptr;
  a.pending = pending;
  a.spin_limit = patience;
  const int64_t entries = plan.n * kk, updates = plan.vec_size * kk;
  flow_empty_kernel<<<static_cast<unsigned>(std::min<int64_t>((updates + entries + 255) / 256, 2048)),
                      256, 0, stream>>>(reinterpret_cast<uint64_t*>(y),
                                        reinterpret_cast<uint64_t*>(d), entries,
                                        reinterpret_cast<uint64_t*>(fvec), updates, pending, maxima, kk);
  const unsigned tasks = static_cast<unsigned>(plan.flow_desc.size / 3);
  if (use_fp32) launch_flow<float>(factor.w32.ptr, a, tasks, stream);
  else launch_flow<double>(factor.w64.ptr, a, tasks, stream);
  HG_HIP(hipGetLastError());
}

}  // namespace hg
