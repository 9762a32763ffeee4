// Persistent conjugate-gradient solves: the settled Jacobi-CG of the heat step and the
// Jacobi-Chebyshev preconditioned CG of the Poisson step, each one cooperative launch.
//
// The iteration is ordito's Chronopoulos-Gear form (kernels/algorithms/conjugate_gradient.py:
// 381-866): a round is w = A u with the three dots r.u, w.u, r.r in one pass, then
// beta = gamma/gamma_old, alpha = gamma / (delta - beta gamma / alpha_old) and the update
// p = u + beta p, s = w + beta s, x += alpha p, r -= alpha s, u = M^-1 r. Where ordito records
// two launches a round into a conditional CUDA graph, this runs the whole loop -- rounds, the
// settle monitor (conjugate_gradient.py:1491-1580) and the stop decisions -- inside one kernel
// with grid-wide barriers, so nothing returns to the host until the solve ends. Every block folds
// the per-block partials in the same fixed order, so all blocks agree on alpha, beta and the stop
// decision bit for bit (the redundant fold ordito uses instead of a barrier, here beside one).
#include <utility>

#include <hipcub/hipcub.hpp>

#include "kernels.h"
#include "words.h"

namespace hg {
namespace {

constexpr int kMaxColumns = 64;

struct CgArgs {
  int64_t n;
  int32_t k;
  const int32_t* offsets;
  const int32_t* columns;
  const float* values32;
  const double* values64;
  const double* inv_diag;
  const double* rhs;
  const double* guess;  // the initial iterate, or null for zero (may alias x)
  double* x;
  double* r;
  double* u;
  double* p;
  double* s;
  double* w;
  double* prev;
  double* res;
  double* da;
  double* db;
  // cg_resident_kernel: the rows' spatial order and its inverse, and the exchanged words.
  const int32_t* order;
  const int32_t* inverse;
  double* exchange;  // [kPhases][n]
  double* slots;     // [kSlotPhases][G][kSlotWidth]
  double* partials;  // [k][G][3], then [G][2] for the settle check, then [k][G] for |b|^2
  // [0] stepped rounds, [1] set when a grid barrier gave up waiting, [2] barrier groups arrived
  // at the current barrier, [3] barrier generation, [4, 12) each group's blocks arrived; [1..12)
  // zero at launch.
  int32_t* counters;
  int64_t spin_limit;  // polls of a grid barrier before it gives up (every block then exits)
  int32_t settle;
  int32_t check_rounds;
  double change_tolerance;
  int32_t settle_rounds;
  double tol_sq;
  int64_t maxiter;
  int32_t cheb_steps;
  double theta;
  double delta;
};

// A block's view of the grid barrier: the generation it waits past and whether a barrier gave up.
struct SyncState {
  int32_t generation;
  int32_t aborted;
};

// Grid-wide barrier over co-resident blocks (the launch is cooperative), counted in two stages so
// no counter takes more than about a sixteenth of the grid's arrivals: a block's thread 0 releases
// the block's writes and counts itself into its group's counter (blocks b with the same b mod 8,
// the XCD the hardware deals b to); the last of a group counts the group into the grid's counter,
// and the last group resets the counts and advances the generation the others poll. The polls are
// relaxed loads, one acquire after the wait. The wait is bounded: past a.spin_limit polls, or once
// another block has given up, the block records the abort and stops waiting, and every later
// barrier returns at once, so each block leaves its loop within a round and the kernel ends; the
// host reads the abort and fails the call.
constexpr int kBarrierGroups = 8;

template <int kThreads, bool kSingle>
__device__ __forceinline__ void barrier(const CgArgs& a, SyncState* sync) {
  if constexpr (kSingle) {
    __syncthreads();
  } else {
    __syncthreads();
    if (threadIdx.x == 0 && !sync->aborted) {
      int32_t* abort = a.counters + 1;
      int32_t* grid_count = a.counters + 2;
      int32_t* generation = a.counters + 3;
      int32_t* group_count = a.counters + 4;
      const int32_t blocks = static_cast<int32_t>(gridDim.x);
      const int32_t group = static_cast<int32_t>(blockIdx.x) % kBarrierGroups;
      const int32_t groups = min(blocks, kBarrierGroups);
      const int32_t members = blocks / kBarrierGroups + (group < blocks % kBarrierGroups ? 1 : 0);
      const int32_t gen = sync->generation;
      const int32_t in_group = __hip_atomic_fetch_add(group_count + group, 1, __ATOMIC_ACQ_REL,
                                                      __HIP_MEMORY_SCOPE_AGENT);
      bool last = false;
      if (in_group == members - 1) {
        __hip_atomic_store(group_count + group, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int32_t in_grid = __hip_atomic_fetch_add(grid_count, 1, __ATOMIC_ACQ_REL,
                                                       __HIP_MEMORY_SCOPE_AGENT);
        last = in_grid == groups - 1;
      }
      if (last) {
        __hip_atomic_store(grid_count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(generation, gen + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        int64_t polls = 0;
        while (__hip_atomic_load(generation, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gen) {
          if (__hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 ||
              ++polls > a.spin_limit) {
            __hip_atomic_store(abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            sync->aborted = 1;
            break;
          }
          __builtin_amdgcn_s_sleep(2);
        }
        __atomic_thread_fence(__ATOMIC_ACQUIRE);
      }
      sync->generation = gen + 1;
    }
    __syncthreads();
  }
}

// Fixed-order block sum of up to three values, every thread getting the same bits: a butterfly
// within each wave (each step adds two lanes' values, which commute, so every lane holds the
// same sum), then the waves' sums in wave order. Two block barriers.
template <int kThreads, int kWidth>
__device__ __forceinline__ void block_sum(double (&v)[kWidth], double* scratch) {
  constexpr int kWaves = kThreads / 64;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
#pragma unroll
  for (int c = 0; c < kWidth; ++c)
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) v[c] += __shfl_xor(v[c], offset, 64);
  if (lane == 0)
#pragma unroll
    for (int c = 0; c < kWidth; ++c) scratch[c * kWaves + wave] = v[c];
  __syncthreads();
#pragma unroll
  for (int c = 0; c < kWidth; ++c) {
    double total = 0.0;
    for (int w = 0; w < kWaves; ++w) total += scratch[c * kWaves + w];
    v[c] = total;
  }
  __syncthreads();
}

template <int kThreads>
__device__ __forceinline__ double block_max(double v, double* scratch) {
  constexpr int kWaves = kThreads / 64;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1) v = fmax(v, __shfl_xor(v, offset, 64));
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  double out = scratch[0];
  for (int w = 1; w < kWaves; ++w) out = fmax(out, scratch[w]);
  __syncthreads();
  return out;
}

__device__ __forceinline__ double row_dot(const CgArgs& a, int64_t i, const double* vec) {
  double sum = 0.0;
  const int32_t begin = a.offsets[i], end = a.offsets[i + 1];
  if (a.values32) {
    for (int32_t e = begin; e < end; ++e)
      sum += static_cast<double>(a.values32[e]) * vec[a.columns[e]];
  } else {
    for (int32_t e = begin; e < end; ++e) sum += a.values64[e] * vec[a.columns[e]];
  }
  return sum;
}

// u = p(D^-1 A) D^-1 r for every column: the Chebyshev semi-iteration on D^-1 A z = D^-1 r from
// z = 0 (Saad, Iterative Methods for Sparse Linear Systems, 2nd ed., Algorithm 12.1), cheb_steps
// steps, cheb_steps - 1 products; the search direction is double-buffered so each step is one
// barrier. Leaves every thread past a barrier.
template <int kThreads, bool kSingle>
__device__ void chebyshev_apply(const CgArgs& a, SyncState* sync) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  const double sigma = a.theta / a.delta;
  double rho = 1.0 / sigma;
  for (int32_t q = 0; q < a.k; ++q) {
    const int64_t o = static_cast<int64_t>(q) * a.n;
    for (int64_t i = first; i < a.n; i += stride) {
      double c = a.inv_diag[i] * a.r[o + i];
      double d = c / a.theta;
      a.res[o + i] = c;
      a.da[o + i] = d;
      a.u[o + i] = d;
    }
  }
  barrier<kThreads, kSingle>(a, sync);
  double* d_old = a.da;
  double* d_new = a.db;
  for (int32_t step = 1; step < a.cheb_steps; ++step) {
    const double rho_new = 1.0 / (2.0 * sigma - rho);
    const double keep = rho_new * rho;
    const double push = 2.0 * rho_new / a.delta;
    for (int32_t q = 0; q < a.k; ++q) {
      const int64_t o = static_cast<int64_t>(q) * a.n;
      for (int64_t i = first; i < a.n; i += stride) {
        double ad = row_dot(a, i, d_old + o);
        double res = a.res[o + i] - a.inv_diag[i] * ad;
        a.res[o + i] = res;
        double d = keep * d_old[o + i] + push * res;
        d_new[o + i] = d;
        a.u[o + i] += d;
      }
    }
    rho = rho_new;
    barrier<kThreads, kSingle>(a, sync);
    double* t = d_old;
    d_old = d_new;
    d_new = t;
  }
}

template <int kThreads, bool kSingle>
__global__ __launch_bounds__(kThreads) void cg_kernel(CgArgs a) {
  __shared__ double scratch[3 * kThreads];
  __shared__ double gamma_old[kMaxColumns];
  __shared__ double alpha_old[kMaxColumns];
  __shared__ double atol_sq[kMaxColumns];
  __shared__ double coeff[2 * kMaxColumns];
  __shared__ int stepping[kMaxColumns];
  __shared__ SyncState sync_state;
  SyncState* sync = &sync_state;
  if (threadIdx.x == 0) {
    sync_state.generation = 0;
    sync_state.aborted = 0;
  }
  __syncthreads();

  const int32_t G = gridDim.x;
  const int64_t stride = static_cast<int64_t>(G) * kThreads;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  double* round_partials = a.partials;
  double* settle_partials = a.partials + static_cast<int64_t>(a.k) * G * 3;
  double* norm_partials = settle_partials + 2 * G;

  // Initial state from x = 0 (or the guess x0): r = b - A x0, p = s = 0, |b|^2 for the
  // tolerance. Each thread writes only its own rows of x, with the guess's own value.
  for (int32_t q = 0; q < a.k; ++q) {
    const int64_t o = static_cast<int64_t>(q) * a.n;
    double acc[1] = {0.0};
    for (int64_t i = first; i < a.n; i += stride) {
      const double b = a.rhs[o + i];
      double ri = b, xi = 0.0;
      if (a.guess) {
        xi = a.guess[o + i];
        ri = b - row_dot(a, i, a.guess + o);
      }
      a.x[o + i] = xi;
      a.r[o + i] = ri;
      a.p[o + i] = 0.0;
      a.s[o + i] = 0.0;
      a.prev[o + i] = 0.0;
      if (a.cheb_steps == 0) a.u[o + i] = a.inv_diag[i] * ri;
      acc[0] += b * b;
    }
    block_sum<kThreads, 1>(acc, scratch);
    if (threadIdx.x == 0) norm_partials[static_cast<int64_t>(q) * G + blockIdx.x] = acc[0];
  }
  barrier<kThreads, kSingle>(a, sync);
  if (a.cheb_steps > 0) chebyshev_apply<kThreads, kSingle>(a, sync);
  for (int32_t q = 0; q < a.k; ++q) {
    double acc[1] = {0.0};
    for (int32_t b = threadIdx.x; b < G; b += kThreads)
      acc[0] += norm_partials[static_cast<int64_t>(q) * G + b];
    block_sum<kThreads, 1>(acc, scratch);
    if (threadIdx.x == 0) {
      atol_sq[q] = a.tol_sq * acc[0];
      gamma_old[q] = INFINITY;
      alpha_old[q] = 1.0;
    }
  }
  __syncthreads();

  int32_t stepped_rounds = 0;
  int64_t round = 0;
  double settle_previous = 0.0, reach_check = 0.0, checks = 0.0;
  bool running = true;
  while (running) {
    if (sync->aborted) break;
    ++round;
    // w = A u and the round's three dots.
    for (int32_t q = 0; q < a.k; ++q) {
      const int64_t o = static_cast<int64_t>(q) * a.n;
      double acc[3] = {0.0, 0.0, 0.0};
      for (int64_t i = first; i < a.n; i += stride) {
        double wi = row_dot(a, i, a.u + o);
        a.w[o + i] = wi;
        double ri = a.r[o + i], ui = a.u[o + i];
        acc[0] += ri * ui;
        acc[1] += wi * ui;
        acc[2] += ri * ri;
      }
      block_sum<kThreads, 3>(acc, scratch);
      if (threadIdx.x == 0) {
        double* dst = round_partials + (static_cast<int64_t>(q) * G + blockIdx.x) * 3;
        dst[0] = acc[0];
        dst[1] = acc[1];
        dst[2] = acc[2];
      }
    }
    barrier<kThreads, kSingle>(a, sync);
    // Every block folds every column's partials in block order: alpha, beta, whether it steps.
    for (int32_t q = 0; q < a.k; ++q) {
      double acc[3] = {0.0, 0.0, 0.0};
      for (int32_t b = threadIdx.x; b < G; b += kThreads) {
        const double* src = round_partials + (static_cast<int64_t>(q) * G + b) * 3;
        acc[0] += src[0];
        acc[1] += src[1];
        acc[2] += src[2];
      }
      block_sum<kThreads, 3>(acc, scratch);
      if (threadIdx.x == 0) {
        int step = 0;
        double alpha = 0.0, beta = 0.0;
        if (acc[2] > atol_sq[q] && round <= a.maxiter && acc[0] != 0.0) {
          beta = acc[0] / gamma_old[q];
          double denominator = acc[1] - beta * acc[0] / alpha_old[q];
          if (denominator != 0.0) {
            alpha = acc[0] / denominator;
            step = 1;
          }
        }
        stepping[q] = step;
        coeff[2 * q] = alpha;
        coeff[2 * q + 1] = beta;
        if (step) {
          gamma_old[q] = acc[0];
          alpha_old[q] = alpha;
        }
      }
    }
    __syncthreads();
    bool any = false;
    for (int32_t q = 0; q < a.k; ++q) any = any || stepping[q];
    if (!any) break;
    ++stepped_rounds;
    for (int32_t q = 0; q < a.k; ++q) {
      if (!stepping[q]) continue;
      const double alpha = coeff[2 * q], beta = coeff[2 * q + 1];
      const int64_t o = static_cast<int64_t>(q) * a.n;
      for (int64_t i = first; i < a.n; i += stride) {
        double pk = a.u[o + i] + beta * a.p[o + i];
        double sk = a.w[o + i] + beta * a.s[o + i];
        a.p[o + i] = pk;
        a.s[o + i] = sk;
        a.x[o + i] += alpha * pk;
        double rk = a.r[o + i] - alpha * sk;
        a.r[o + i] = rk;
        if (a.cheb_steps == 0) a.u[o + i] = a.inv_diag[i] * rk;
      }
    }
    if (round >= a.maxiter) running = false;
    if (a.cheb_steps > 0) {
      barrier<kThreads, kSingle>(a, sync);
      chebyshev_apply<kThreads, kSingle>(a, sync);
    }
    if (a.settle && round % a.check_rounds == 0) {
      // Per-entry relative change since the last check and the count of reached entries.
      double change = 0.0;
      double reached[1] = {0.0};
      for (int32_t q = 0; q < a.k; ++q) {
        const int64_t o = static_cast<int64_t>(q) * a.n;
        for (int64_t i = first; i < a.n; i += stride) {
          double xv = a.x[o + i];
          if (xv != 0.0) {
            change = fmax(change, fabs(xv - a.prev[o + i]) / fabs(xv));
            reached[0] += 1.0;
          }
          a.prev[o + i] = xv;
        }
      }
      change = block_max<kThreads>(change, scratch);
      block_sum<kThreads, 1>(reached, scratch);
      if (threadIdx.x == 0) {
        settle_partials[2 * blockIdx.x] = change;
        settle_partials[2 * blockIdx.x + 1] = reached[0];
      }
      barrier<kThreads, kSingle>(a, sync);
      double c = 0.0;
      double count[1] = {0.0};
      for (int32_t b = threadIdx.x; b < G; b += kThreads) {
        c = fmax(c, settle_partials[2 * b]);
        count[0] += settle_partials[2 * b + 1];
      }
      c = block_max<kThreads>(c, scratch);
      block_sum<kThreads, 1>(count, scratch);
      checks += 1.0;
      double total = count[0] + 1.0;
      if (total != settle_previous) {
        settle_previous = total;
        reach_check = checks;
      } else {
        double idle = (checks - reach_check) * static_cast<double>(a.check_rounds);
        if (c < a.change_tolerance || idle >= static_cast<double>(a.settle_rounds)) running = false;
      }
    } else if (a.cheb_steps == 0) {
      barrier<kThreads, kSingle>(a, sync);
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) a.counters[0] = stepped_rounds;
}

// ---- one column, its whole state on the chip ---------------------------------------------------
//
// cg_kernel keeps the iteration's vectors in memory, and its grid barrier makes them visible to
// the other XCDs by writing back and invalidating the L2s, so every round re-reads its vectors and
// the operator from beyond the L2: 20-35 us a product on systems of 41-164 thousand rows whose
// data would fit the compute units several times over. Here a thread owns R rows and keeps their
// operator entries (E a row; longer rows read the rest through the L2) and their vectors in
// registers and LDS for the whole solve. Only two things leave a block:
//   - the values the products gather (u, or a Chebyshev direction) of rows that have a neighbour
//     in another block, written through to `exchange` where that neighbour's thread waits for them;
//   - a block's three partial sums, written through to `slots`, where every block waits for all.
// Both are words that are their own arrival flags (words.h), so one store-to-load latency replaces
// a barrier's several, nothing is written back or invalidated, and the read-only operator stays
// cached.
//
// Blocks own consecutive rows of a spatial order of the vertices (spatial_order), so nearly all
// of a row's neighbours are its block's and read from LDS. A published word is emptied again two
// phases later by its owner: product k reads phase k's words; having read its neighbours' phase
// k - 1, a row's thread knows that they have read phase k - 2 (they publish k - 1 after it, and
// the pattern is symmetric), so in phase k it empties its word of phase k - 2, waits for that store
// before it publishes phase k + 1, and nobody polls phase k + 2 in that word before reading that.
// So four buffers of n words serve. The sums' slots rotate over three in the same way: a block
// publishes sum q - 1 once all its threads have read sum q - 2.
//
// Sums keep a fixed order (a thread's rows, then butterflies over lanes, waves and blocks), so a
// solve repeats bit for bit. Every wait is bounded as the grid barrier's are.
constexpr int kPhases = 4, kSlotPhases = 3, kSlotWidth = 4;

// A row's thread reads up to so many entries past those in registers, each a chain of three loads. A
// longer row's are dealt over its wave (kLong), 64 chains at a time: a one-shot call on a cone whose
// apex has 400 neighbours (8,001 rows) takes 9.0 ms so, 40 with the thread reading them all and 27
// with the state in memory; 8,000 neighbours (64,001 rows) 73, 670 and 266 ms. Instances of their own,
// for systems that have such a row: the four rows a thread of the largest have no registers to spare.
constexpr int32_t kOwnExtra = 16;

// A thread's value of a vector for each of its rows, in registers or in LDS (l = the thread's
// first entry, entries kStride apart).
template <int R, int kStride, bool kLds>
struct RowVector {
  double reg[kLds ? 1 : R];
  double* lds;
  __device__ __forceinline__ double get(int j) const {
    if constexpr (kLds) return lds[kStride * j];
    else return reg[j];
  }
  __device__ __forceinline__ void set(int j, double v) {
    if constexpr (kLds) lds[kStride * j] = v;
    else reg[j] = v;
  }
};

// T threads a block, R rows a thread, E operator entries of a row in registers, TV the operator's
// values (float: the narrowed heat operator), kCheb the polynomial preconditioner, kGrid more than
// one block, kLong some rows of more than E + kOwnExtra entries. Instances with double values keep x, p, s and r in LDS: they are touched once a round,
// and the registers are the operator's.
template <int T, int R, int E, typename TV, bool kCheb, bool kGrid, bool kLong>
__global__ __launch_bounds__(T) void cg_resident_kernel(CgArgs a) {
  constexpr int L = R * T, kWaves = T / 64;
  static_assert((kWaves & (kWaves - 1)) == 0, "the waves' sums fold in a butterfly");
  constexpr bool kLds = sizeof(TV) == 8;
  // The values the products gather, two phases; entry L stays zero (the padding of a short row).
  __shared__ double vec[2][L + 1];
  __shared__ double state[kLds ? 4 * L : 1];
  __shared__ double scratch[2][3 * kWaves];
  const int t = threadIdx.x, wave = t / 64, lane = t % 64;
  const int32_t n = static_cast<int32_t>(a.n);
  const int32_t G = static_cast<int32_t>(gridDim.x);
  const int32_t block = kGrid ? xcd_block() : 0;
  const int32_t per_block = kGrid ? (n + G - 1) / G : n;
  const int32_t base = block * per_block;
  const int32_t count = max(0, min(per_block, n - base));  // this block's rows
  const TV* values = sizeof(TV) == 4 ? reinterpret_cast<const TV*>(a.values32)
                                     : reinterpret_cast<const TV*>(a.values64);
  bool aborted = false;
  if (t < 2) vec[t][L] = 0.0;

  // The thread's rows: local index t + T j, row base + t + T j of the order. An operator column is
  // held as the byte offset of its value: >= 0 in a phase's LDS vector, < 0 (complemented) in a
  // phase's exchange, for a row of another block.
  int32_t old_row[R], begin[R], extra[R];  // extra: entries past E
  int32_t col[R][E];
  TV val[R][E];
#pragma unroll
  for (int j = 0; j < R; ++j)
#pragma unroll
    for (int e = 0; e < E; ++e) {
      col[j][e] = 8 * L;
      val[j][e] = TV(0);
    }
  double dinv[R];
  uint32_t live = 0, outer = 0;  // row j exists; row j has a neighbour in another block
  auto locate = [&](int32_t c) {
    if constexpr (!kGrid) return 8 * c;
    const int32_t at = a.inverse[c] - base;
    return at >= 0 && at < count ? 8 * at : ~(8 * (at + base));
  };
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int32_t l = t + T * j;
    const bool has = l < count;
    if (has) live |= 1u << j;
    old_row[j] = has ? (kGrid ? a.order[base + l] : l) : 0;
    begin[j] = has ? a.offsets[old_row[j]] : 0;
    const int32_t degree = has ? a.offsets[old_row[j] + 1] - begin[j] : 0;
    extra[j] = max(0, degree - E);
    dinv[j] = has ? a.inv_diag[old_row[j]] : 0.0;
    // Entries past the row's end load one that exists, so the loads need no branches.
    const int32_t last = a.offsets[n] - 1;
    if (last < 0) continue;
    int32_t c[E];
#pragma unroll
    for (int e = 0; e < E; ++e) c[e] = a.columns[min(begin[j] + e, last)];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const bool stored = e < degree;
      const TV v = values[min(begin[j] + e, last)];
      const int32_t at = locate(c[e]);
      col[j][e] = stored ? at : 8 * L;
      val[j][e] = stored ? v : TV(0);
      if (kGrid && stored && at < 0) outer |= 1u << j;
    }
    if (kGrid)
#pragma unroll 1
      for (int32_t e = E; e < (kLong && extra[j] > kOwnExtra ? 0 : degree); ++e)
        if (locate(a.columns[begin[j] + e]) < 0) outer |= 1u << j;
    if constexpr (kGrid && kLong)
      for (uint64_t rows = __ballot(extra[j] > kOwnExtra); rows; rows &= rows - 1) {
        const int owner = __ffsll(static_cast<unsigned long long>(rows)) - 1;
        const int32_t from = __shfl(begin[j], owner, 64) + E, more = __shfl(extra[j], owner, 64);
        bool any = false;
        for (int32_t e = lane; e < more; e += 64) any |= locate(a.columns[from + e]) < 0;
        if (__any(any) && lane == owner) outer |= 1u << j;
      }
  }

  // Phase k of the exchange: this thread's rows' values, into LDS and, for rows with a neighbour
  // elsewhere, into the exchange.
  int32_t phase = -1;
  auto phase_words = [&](int32_t k) { return a.exchange + static_cast<int64_t>(k % kPhases) * n; };
  auto offer = [&](int j, double v) {
    vec[phase & 1][t + T * j] = v;
    if (kGrid && (outer >> j & 1)) publish(phase_words(phase) + base + t + T * j, v);
  };
  // Before a phase's offers: the words emptied in the last product have landed.
  auto next_phase = [&]() {
    ++phase;
    if (kGrid) drain_stores();
  };
  // out = A v over this thread's rows, v the current phase's values, each row in its entry order.
  auto product = [&](double (&out)[R]) {
    const char* local = reinterpret_cast<const char*>(vec[phase & 1]);
    const char* remote = nullptr;
    auto at_local = [&](int32_t c) {
      return *reinterpret_cast<const uint64_t*>(local + static_cast<uint32_t>(c));
    };
    auto at_remote = [&](int32_t c) {
      return peek(reinterpret_cast<const double*>(remote + static_cast<uint32_t>(~c)));
    };
    if (kGrid) {
      remote = reinterpret_cast<const char*>(phase_words(phase));
      double* spent = phase_words(phase + 2) + base + t;
#pragma unroll
      for (int j = 0; j < R; ++j)
        if (outer >> j & 1) empty(spent + T * j);
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
      uint64_t raw[E];
#pragma unroll
      for (int e = 0; e < E; ++e) raw[e] = at_local(kGrid ? max(col[j][e], 0) : col[j][e]);
      if (kGrid && (outer >> j & 1)) {
#pragma unroll
        for (int e = 0; e < E; ++e)
          if (col[j][e] < 0) raw[e] = at_remote(col[j][e]);
        int32_t polls = 0;
        for (;;) {
          bool waiting = false;
#pragma unroll
          for (int e = 0; e < E; ++e)
            if (raw[e] == kEmpty) {  // only a remote word can read so
              raw[e] = at_remote(col[j][e]);
              waiting = true;
            }
          if (!waiting || !wait_on(a.counters + 1, 1, a.spin_limit, polls, aborted)) break;
        }
      }
      double sum = 0.0;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        // Widened here each time: the widened values of a whole row would not fit the registers.
        if constexpr (sizeof(TV) == 4) asm volatile("" : "+v"(val[j][e]));
        sum += static_cast<double>(val[j][e]) * __builtin_bit_cast(double, raw[e]);
      }
#pragma unroll 1
      for (int32_t e = 0; e < (kLong && extra[j] > kOwnExtra ? 0 : extra[j]); ++e) {
        // The rest of a row longer than E.
        const int32_t c = locate(a.columns[begin[j] + E + e]);
        uint64_t bits;
        if (kGrid && c < 0) {
          int32_t polls = 0;
          while ((bits = at_remote(c)) == kEmpty && wait_on(a.counters + 1, 1, a.spin_limit, polls, aborted)) {
          }
        } else {
          bits = at_local(c);
        }
        sum += static_cast<double>(values[begin[j] + E + e]) * __builtin_bit_cast(double, bits);
      }
      if constexpr (kLong)
        for (uint64_t rows = __ballot(extra[j] > kOwnExtra); rows; rows &= rows - 1) {
          const int owner = __ffsll(static_cast<unsigned long long>(rows)) - 1;
          const int32_t from = __shfl(begin[j], owner, 64) + E, more = __shfl(extra[j], owner, 64);
          double part = 0.0;
#pragma unroll 1
          for (int32_t e = lane; e < more; e += 64) {
            const int32_t c = locate(a.columns[from + e]);
            uint64_t bits;
            if (kGrid && c < 0) {
              int32_t polls = 0;
              while ((bits = at_remote(c)) == kEmpty && wait_on(a.counters + 1, 1, a.spin_limit, polls, aborted)) {
              }
            } else {
              bits = at_local(c);
            }
            part += static_cast<double>(values[from + e]) * __builtin_bit_cast(double, bits);
          }
#pragma unroll
          for (int offset = 32; offset > 0; offset >>= 1) part += __shfl_xor(part, offset, 64);
          if (lane == owner) sum += part;
        }
      out[j] = sum;
    }
  };

  // The sums of v[0..2] over every thread of every block, v[0]'s maximum instead when kMax, left in
  // v on every thread. Scratch alternates between calls, so one block barrier a fold suffices.
  int32_t folds = 0, sums = 0;
  auto fold_block = [&](double (&v)[3], bool max_first) {
    double* mine = scratch[folds++ & 1];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int offset = 32; offset > 0; offset >>= 1) {
        const double other = __shfl_xor(v[c], offset, 64);
        v[c] = c == 0 && max_first ? fmax(v[c], other) : v[c] + other;
      }
    if (lane == 0)
#pragma unroll
      for (int c = 0; c < 3; ++c) mine[c * kWaves + wave] = v[c];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      v[c] = mine[c * kWaves + lane % kWaves];
#pragma unroll
      for (int offset = kWaves / 2; offset > 0; offset >>= 1) {
        const double other = __shfl_xor(v[c], offset, kWaves);
        v[c] = c == 0 && max_first ? fmax(v[c], other) : v[c] + other;
      }
    }
  };
  auto fold = [&](double (&v)[3], bool max_first = false) {
    if (!kGrid) {
      fold_block(v, max_first);
      return;
    }
    const int32_t q = sums++;
    double* slots = a.slots + static_cast<int64_t>(q % kSlotPhases) * G * kSlotWidth;
    double* spent = a.slots + static_cast<int64_t>((q + 1) % kSlotPhases) * G * kSlotWidth;
    if (t < 3) empty(spent + block * kSlotWidth + t);
    fold_block(v, max_first);
    if (t < 3) {
      drain_stores();
      publish(slots + block * kSlotWidth + t, t == 0 ? v[0] : t == 1 ? v[1] : v[2]);
    }
    uint64_t got[3] = {0, 0, 0};  // +0.0: the identity of these sums and of a maximum of magnitudes
    if (t < G) {
      const double* theirs = slots + t * kSlotWidth;
#pragma unroll
      for (int c = 0; c < 3; ++c) got[c] = peek(theirs + c);
      int32_t polls = 0;
      while (got[0] == kEmpty || got[1] == kEmpty || got[2] == kEmpty) {
        if (!wait_on(a.counters + 1, 1, a.spin_limit, polls, aborted)) break;
#pragma unroll
        for (int c = 0; c < 3; ++c)
          if (got[c] == kEmpty) got[c] = peek(theirs + c);
      }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = __builtin_bit_cast(double, got[c]);
    fold_block(v, max_first);
  };

  RowVector<R, T, kLds> x, r, p, s;
  x.lds = state + t;
  r.lds = state + (kLds ? L : 0) + t;
  p.lds = state + (kLds ? 2 * L : 0) + t;
  s.lds = state + (kLds ? 3 * L : 0) + t;
  double u[R];
  // r = b - A x0 (x0 the guess, else zero); the guess is read where the caller holds it.
  double norm[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const bool has = live >> j & 1;
    const double b = has ? a.rhs[old_row[j]] : 0.0;
    double ri = b, xi = 0.0;
    if (a.guess && has) {
      double ax = 0.0;
      xi = a.guess[old_row[j]];
#pragma unroll 1
      for (int32_t e = begin[j]; e < a.offsets[old_row[j] + 1]; ++e)
        ax += static_cast<double>(values[e]) * a.guess[a.columns[e]];
      ri = b - ax;
    }
    x.set(j, xi);
    r.set(j, ri);
    p.set(j, 0.0);
    s.set(j, 0.0);
    u[j] = dinv[j] * ri;
    norm[0] += b * b;
  }
  fold(norm);
  const double atol_sq = a.tol_sq * norm[0];

  // u = p(D^-1 A) D^-1 r (chebyshev_apply's recurrence).
  const double sigma = kCheb ? a.theta / a.delta : 0.0;
  auto chebyshev = [&]() {
    if constexpr (kCheb) {
      double rho = 1.0 / sigma;
      double res[R], d[R];
      next_phase();
#pragma unroll
      for (int j = 0; j < R; ++j) {
        res[j] = dinv[j] * r.get(j);
        d[j] = res[j] / a.theta;
        u[j] = d[j];
        offer(j, d[j]);
      }
      __syncthreads();
      for (int32_t step = 1; step < a.cheb_steps; ++step) {
        const double rho_new = 1.0 / (2.0 * sigma - rho);
        const double keep = rho_new * rho;
        const double push = 2.0 * rho_new / a.delta;
        double ad[R];
        product(ad);
        const bool more = step + 1 < a.cheb_steps;
        if (more) next_phase();
#pragma unroll
        for (int j = 0; j < R; ++j) {
          res[j] = res[j] - dinv[j] * ad[j];
          d[j] = keep * d[j] + push * res[j];
          u[j] += d[j];
          if (more) offer(j, d[j]);
        }
        rho = rho_new;
        if (more) __syncthreads();
      }
    }
  };

  double prev[kCheb ? 1 : R];
  if constexpr (!kCheb)
#pragma unroll
    for (int j = 0; j < R; ++j) prev[j] = 0.0;
  double gamma_old = INFINITY, alpha_old = 1.0;
  int32_t stepped_rounds = 0;
  int64_t round = 0;
  double settle_previous = 0.0, reach_check = 0.0, checks = 0.0;
  bool running = true;
  if (kCheb) chebyshev();
  while (running) {
    ++round;
    // w = A u and the round's three dots.
    next_phase();
#pragma unroll
    for (int j = 0; j < R; ++j) offer(j, u[j]);
    if (__syncthreads_or(aborted ? 1 : 0)) break;
    double w[R];
    double acc[3] = {0.0, 0.0, 0.0};
    product(w);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const double rj = r.get(j);
      acc[0] += rj * u[j];
      acc[1] += w[j] * u[j];
      acc[2] += rj * rj;
    }
    fold(acc);
    double alpha = 0.0, beta = 0.0;
    bool step = false;
    if (acc[2] > atol_sq && round <= a.maxiter && acc[0] != 0.0) {
      beta = acc[0] / gamma_old;
      const double denominator = acc[1] - beta * acc[0] / alpha_old;
      if (denominator != 0.0) {
        alpha = acc[0] / denominator;
        step = true;
      }
    }
    if (!step) break;
    gamma_old = acc[0];
    alpha_old = alpha;
    ++stepped_rounds;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const double pj = u[j] + beta * p.get(j);
      const double sj = w[j] + beta * s.get(j);
      p.set(j, pj);
      s.set(j, sj);
      x.set(j, x.get(j) + alpha * pj);
      const double rj = r.get(j) - alpha * sj;
      r.set(j, rj);
      if (!kCheb) u[j] = dinv[j] * rj;
    }
    if (round >= a.maxiter) running = false;
    if (kCheb) chebyshev();
    if constexpr (!kCheb) {
      if (a.settle && round % a.check_rounds == 0) {
        double verdict[3] = {0.0, 0.0, 0.0};  // the largest relative change, entries reached
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const double xj = x.get(j);
          if ((live >> j & 1) && xj != 0.0) {
            verdict[0] = fmax(verdict[0], fabs(xj - prev[j]) / fabs(xj));
            verdict[1] += 1.0;
          }
          prev[j] = xj;
        }
        fold(verdict, true);
        checks += 1.0;
        const double total = verdict[1] + 1.0;
        if (total != settle_previous) {
          settle_previous = total;
          reach_check = checks;
        } else {
          const double idle = (checks - reach_check) * static_cast<double>(a.check_rounds);
          if (verdict[0] < a.change_tolerance || idle >= static_cast<double>(a.settle_rounds))
            running = false;
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < R; ++j)
    if (live >> j & 1) a.x[old_row[j]] = x.get(j);
  if (block == 0 && t == 0) a.counters[0] = stepped_rounds;
}

// ---- a spatial order of the vertices -----------------------------------------------------------

// Order-preserving integers of floats, for atomic minima and maxima.
__device__ __forceinline__ uint32_t ordered_bits(float v) {
  const uint32_t b = __builtin_bit_cast(uint32_t, v);
  return b & 0x80000000u ? ~b : b | 0x80000000u;
}

__device__ __forceinline__ float from_ordered_bits(uint32_t b) {
  return __builtin_bit_cast(float, b & 0x80000000u ? b & 0x7FFFFFFFu : ~b);
}

// The finite coordinates' bounds into bounds[0..3) (minima, held complemented) and [3..6)
// (maxima), all zero at launch.
__global__ __launch_bounds__(kBlock) void bounds_kernel(const float* __restrict__ xyz, int64_t n,
                                                        uint32_t* __restrict__ bounds) {
  uint32_t best[6] = {0, 0, 0, 0, 0, 0};
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * kBlock)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const float v = xyz[3 * i + d];
      if (!(fabsf(v) < INFINITY)) continue;
      const uint32_t b = ordered_bits(v);
      best[d] = max(best[d], ~b);
      best[3 + d] = max(best[3 + d], b);
    }
#pragma unroll
  for (int c = 0; c < 6; ++c) {
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1)
      best[c] = max(best[c], static_cast<uint32_t>(__shfl_xor(static_cast<int>(best[c]), offset, 64)));
    if (threadIdx.x % 64 == 0) atomicMax(bounds + c, best[c]);
  }
}

__device__ __forceinline__ uint32_t spread3(uint32_t v) {  // ten bits, two zeros after each
  v = (v | v << 16) & 0x030000FFu;
  v = (v | v << 8) & 0x0300F00Fu;
  v = (v | v << 4) & 0x030C30C3u;
  return (v | v << 2) & 0x09249249u;
}

// Each vertex's Morton code over the bounds' cube, ten bits an axis (a non-finite coordinate in the
// first cell), and its index.
__global__ __launch_bounds__(kBlock) void morton_kernel(const float* __restrict__ xyz, int64_t n,
                                                        const uint32_t* __restrict__ bounds,
                                                        uint32_t* __restrict__ keys,
                                                        int32_t* __restrict__ ids) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  float extent = 0.0f, low[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    low[d] = from_ordered_bits(~bounds[d]);
    extent = fmaxf(extent, from_ordered_bits(bounds[3 + d]) - low[d]);
  }
  const float scale = extent > 0.0f ? 1024.0f / extent : 0.0f;
  uint32_t key = 0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float cell = (xyz[3 * i + d] - low[d]) * scale;
    const uint32_t c = cell > 0.0f ? static_cast<uint32_t>(fminf(cell, 1023.0f)) : 0u;
    key |= spread3(c) << d;
  }
  keys[i] = key;
  ids[i] = static_cast<int32_t>(i);
}

__global__ __launch_bounds__(kBlock) void invert_kernel(const int32_t* __restrict__ order, int64_t n,
                                                        int32_t* __restrict__ inverse) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i < n) inverse[order[i]] = static_cast<int32_t>(i);
}

__global__ __launch_bounds__(kBlock) void fill_empty_kernel(uint64_t* __restrict__ words,
                                                            int64_t count) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < count;
       i += static_cast<int64_t>(gridDim.x) * kBlock)
    words[i] = kEmpty;
}

// Componentwise backward error flag (kernels/linalg.py:1128-1230): "not within" so NaN flags.
__global__ void backward_error_kernel(const int32_t* __restrict__ offsets,
                                      const int32_t* __restrict__ columns,
                                      const double* __restrict__ values,
                                      const double* __restrict__ x, const double* __restrict__ b,
                                      int64_t n, double tolerance, int32_t* __restrict__ flag) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  int64_t q = blockIdx.y;
  bool fail = false;
  if (i < n) {
    const double* xq = x + q * n;
    double bi = b[q * n + i];
    double total = bi, scale = fabs(bi);
    for (int32_t e = offsets[i]; e < offsets[i + 1]; ++e) {
      double term = values[e] * xq[columns[e]];
      total -= term;
      scale += fabs(term);
    }
    fail = !(fabs(total) <= tolerance * scale);
  }
  // One atomic a failing block, none once the flag reads set.
  const int any = __syncthreads_or(fail ? 1 : 0);
  if (any && threadIdx.x == 0 &&
      __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
    atomicOr(flag, 1);
}

__global__ void dominance_partial_kernel(const int32_t* __restrict__ offsets,
                                         const int32_t* __restrict__ columns,
                                         const double* __restrict__ values, int64_t n,
                                         double* __restrict__ partials) {
  __shared__ double scratch[kBlock];
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  double ratio = 0.0;
  if (i < n) {
    double diag = 0.0, off = 0.0;
    for (int32_t e = offsets[i]; e < offsets[i + 1]; ++e) {
      if (columns[e] == i) diag = fabs(values[e]);
      else off += fabs(values[e]);
    }
    if (diag > 0.0) ratio = off / diag;
  }
  ratio = block_max<kBlock>(ratio, scratch);
  if (threadIdx.x == 0) partials[blockIdx.x] = ratio;
}

__global__ void dominance_final_kernel(const double* __restrict__ partials, int32_t blocks,
                                       double* __restrict__ out) {
  __shared__ double scratch[kBlock];
  double v = 0.0;
  for (int32_t b = threadIdx.x; b < blocks; b += kBlock) v = fmax(v, partials[b]);
  v = block_max<kBlock>(v, scratch);
  if (threadIdx.x == 0) out[0] = v;
}

// The multi-block solve's grid: one 1024-lane block per compute unit at most (every block folds
// every block's partials each round, and each grid barrier counts every block in, so fewer, wider
// blocks keep a round short), and never more blocks than can be resident at once.
int32_t cooperative_grid(int64_t n) {
  int device = 0;
  HG_HIP(hipGetDevice(&device));
  int cus = 0;
  HG_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  int per_cu = 0;
  HG_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, cg_kernel<1024, false>, 1024, 0));
  HG_REQUIRE(per_cu >= 1, HG_ERR_RUNTIME, "the conjugate-gradient kernel fits no compute unit");
  const int64_t needed = (n + 1023) / 1024;
  return static_cast<int32_t>(std::max<int64_t>(1, std::min<int64_t>(cus, needed)));
}

using CgKernel = void (*)(CgArgs);

// Blocks of a resident solve at most: one a compute unit, and no more than a block has threads to
// read the sums of.
int64_t resident_units() {
  int device = 0, cus = 0;
  HG_HIP(hipGetDevice(&device));
  HG_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  return std::min<int64_t>(cus, 256);
}

struct ResidentChoice {
  CgKernel kernel = nullptr;
  int32_t threads = 0, rows = 0;  // rows a block
};

template <int T, int R, int E, bool kGrid, bool kLong>
ResidentChoice resident_instance(bool cheb, bool narrow) {
  ResidentChoice c;
  c.threads = T;
  c.rows = T * R;
  if (cheb) c.kernel = cg_resident_kernel<T, R, E, double, true, kGrid, kLong>;
  else if (narrow) c.kernel = cg_resident_kernel<T, R, E, float, false, kGrid, kLong>;
  else if constexpr (!kGrid) c.kernel = cg_resident_kernel<T, R, E, double, false, kGrid, kLong>;
  return c;
}

template <int T, int R, int E, bool kGrid>
ResidentChoice resident_choice(const CgProblem& p, bool cheb, bool narrow) {
  // One block's vectors are all in its LDS, where a thread reads a long row quickly enough.
  if constexpr (kGrid)
    if (p.longest_row > E + kOwnExtra) return resident_instance<T, R, E, kGrid, true>(cheb, narrow);
  return resident_instance<T, R, E, kGrid, false>(cheb, narrow);
}

// The resident kernel for a one-column problem: its threads, rows a thread and function, by size.
// Up to 1,024 rows one block, which exchanges nothing, of 256, 512 or 1024 threads: a round waits for all
// its waves, idle ones too (the heat solve of 162 rows 136 us in 256 threads, 246 in 1024; of 258 rows 233
// in 512, 363 in 1024). Up to 3,072 too where there is no spatial order; with one, 2,562 rows took
// 1.04 ms for both solves of a one-shot call in one block, which reads three rows' entries out of one
// compute unit's LDS, and 0.88 ms in eleven of 256 threads.
// Up to 65,536 rows a row a thread in blocks of 256, as few blocks as hold them (icosphere(6),
// 40,962 rows: 3.51 ms; blocks of 512, 3.56; of 1024, 4.73). Past that every compute unit gets a
// block of 512 threads with two rows each (icosphere(7), 163,842 rows: 11.7 ms; as few blocks as
// hold them 12.0, 1024 threads with one row 12.1, 256 with four 15.2), or four with seven entries
// in registers (torus of 524,288 rows, the heat solve: 10.8 ms; nine entries spill, 13.4 ms; 1024
// threads with two rows 13.6 and 18.8 ms).
ResidentChoice choose_resident(const CgProblem& p) {
  const bool cheb = p.chebyshev_steps > 0, narrow = p.values32 != nullptr;
  if (p.n_columns != 1 || (cheb && narrow)) return {};
  if (p.n <= 256) return resident_choice<256, 1, 9, false>(p, cheb, narrow);
  if (p.n <= 512) return resident_choice<512, 1, 9, false>(p, cheb, narrow);
  if (p.n <= 1024) return resident_choice<1024, 1, 9, false>(p, cheb, narrow);
  if (!p.order || !p.inverse) {
    if (p.n <= 2048) return resident_choice<1024, 2, 9, false>(p, cheb, narrow);
    if (p.n <= 3072) return resident_choice<1024, 3, 5, false>(p, cheb, narrow);
    return {};
  }
  const int64_t units = resident_units();
  if (p.n <= 256 * units) return resident_choice<256, 1, 9, true>(p, cheb, narrow);
  if (p.n <= 1024 * units) return resident_choice<512, 2, 9, true>(p, cheb, narrow);
  if (p.n <= 2048 * units) return resident_choice<512, 4, 7, true>(p, cheb, narrow);
  return {};
}

// The exchange of a resident solve of n rows in at most 256 blocks, in doubles.
int64_t exchange_words(int64_t n) { return kPhases * n + kSlotPhases * kSlotWidth * 256; }

void reserve_exchange(CgWorkspace& ws, int64_t words) {
  if (ws.exchange.size < words) ws.exchange.allocate(words);
}

int32_t launched_rounds(CgWorkspace& ws, hipStream_t stream) {
  int32_t words[2] = {0, 0};
  HG_HIP(hipMemcpyAsync(words, ws.counters.ptr, sizeof(words), hipMemcpyDeviceToHost, stream));
  HG_HIP(hipStreamSynchronize(stream));
  HG_REQUIRE(words[1] == 0, HG_ERR_RUNTIME,
             "conjugate gradient: a grid barrier waited past its limit; the solve was abandoned");
  return words[0];
}

}  // namespace

bool wants_spatial_order(int64_t n, int64_t n_columns) {
  return n_columns == 1 && n > 1024 && n <= 2048 * resident_units();
}

void spatial_order(const float* xyz, int64_t n, SpatialOrder& out, CgWorkspace& ws,
                   hipStream_t stream) {
  // `out` takes the order once it is complete: one that could not be built is built by a later call.
  SpatialOrder built;
  built.order.allocate(std::max<int64_t>(n, 1));
  built.inverse.allocate(std::max<int64_t>(n, 1));
  if (n == 0) {
    out = std::move(built);
    return;
  }
  // Keys, sorted keys, indices, bounds and the sort's storage, in the exchange of the solve that
  // follows.
  size_t bytes = 0;
  uint32_t* keys = nullptr;
  int32_t* ids = nullptr;
  HG_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, keys, keys, ids, built.order.ptr,
                                            static_cast<int>(n), 0, 30, stream));
  const int64_t head = (4 * (3 * n + 6) + 255) / 256 * 256;
  reserve_exchange(ws, std::max(exchange_words(n), (head + static_cast<int64_t>(bytes) + 7) / 8));
  keys = reinterpret_cast<uint32_t*>(ws.exchange.ptr);
  ids = reinterpret_cast<int32_t*>(keys + 2 * n);
  uint32_t* bounds = keys + 3 * n;
  void* temp = reinterpret_cast<uint8_t*>(keys) + head;
  const unsigned blocks = static_cast<unsigned>((n + kBlock - 1) / kBlock);
  launch_zero(bounds, 6 * sizeof(uint32_t), stream);
  bounds_kernel<<<std::min(blocks, 256u), kBlock, 0, stream>>>(xyz, n, bounds);
  morton_kernel<<<blocks, kBlock, 0, stream>>>(xyz, n, bounds, keys, ids);
  HG_HIP(hipGetLastError());
  HG_HIP(hipcub::DeviceRadixSort::SortPairs(temp, bytes, keys, keys + n, ids, built.order.ptr,
                                            static_cast<int>(n), 0, 30, stream));
  invert_kernel<<<blocks, kBlock, 0, stream>>>(built.order.ptr, n, built.inverse.ptr);
  HG_HIP(hipGetLastError());
  out = std::move(built);
}

int32_t run_cg(const CgProblem& problem, CgWorkspace& ws, hipStream_t stream) {
  const int64_t n = problem.n;
  const int64_t k = problem.n_columns;
  HG_REQUIRE(k >= 1 && k <= kMaxColumns, HG_ERR_VALUE, "conjugate gradient takes 1-64 columns");
  if (n == 0) return 0;
  if (ws.counters.size < 4 + kBarrierGroups) ws.counters.allocate(4 + kBarrierGroups);
  CgArgs a{};
  a.n = n;
  a.k = static_cast<int32_t>(k);
  a.offsets = problem.offsets;
  a.columns = problem.columns;
  a.values32 = problem.values32;
  a.values64 = problem.values64;
  a.inv_diag = problem.inv_diag;
  a.rhs = problem.rhs;
  a.guess = problem.guess;
  a.x = problem.x;
  a.counters = ws.counters.ptr;
  a.spin_limit = kSpinLimit;
  a.settle = problem.settle;
  a.check_rounds = std::max(problem.check_rounds, 1);
  a.change_tolerance = problem.change_tolerance;
  a.settle_rounds = problem.settle_rounds;
  a.tol_sq = problem.settle ? 0.0 : problem.tolerance * problem.tolerance;
  a.maxiter = problem.maxiter > 0 ? problem.maxiter : 10 * n;
  a.cheb_steps = problem.chebyshev_steps;
  a.theta = 0.5 * (problem.lambda_max + problem.lambda_min);
  a.delta = 0.5 * (problem.lambda_max - problem.lambda_min);
  void* args[] = {&a};
  launch_zero(ws.counters.ptr, sizeof(int32_t) * (4 + kBarrierGroups), stream);
  const ResidentChoice choice = choose_resident(problem);
  if (choice.kernel) {
    if (n <= choice.rows) {
      hipLaunchKernelGGL(choice.kernel, dim3(1), dim3(choice.threads), 0, stream, a);
      HG_HIP(hipGetLastError());
      return launched_rounds(ws, stream);
    }
    const int64_t G = choice.rows > choice.threads ? resident_units()
                                                   : (n + choice.rows - 1) / choice.rows;
    const int64_t words = exchange_words(n);
    reserve_exchange(ws, words);
    a.order = problem.order;
    a.inverse = problem.inverse;
    a.exchange = ws.exchange.ptr;
    a.slots = ws.exchange.ptr + kPhases * n;
    fill_empty_kernel<<<static_cast<unsigned>(std::min<int64_t>((words + kBlock - 1) / kBlock, 2048)),
                        kBlock, 0, stream>>>(reinterpret_cast<uint64_t*>(ws.exchange.ptr), words);
    HG_HIP(hipGetLastError());
    // Cooperative: every block waits for words of the others, so all must be resident.
    const WaitClaim claim(true, true);
    HG_HIP(hipLaunchCooperativeKernel(reinterpret_cast<const void*>(choice.kernel),
                                      dim3(static_cast<unsigned>(G)), dim3(choice.threads), args,
                                      0, stream));
    return launched_rounds(ws, stream);
  }
  // Several columns, systems past the compute units' registers, and systems with no spatial order:
  // the state in memory. Small ones run in one block of 1024 lanes with block barriers only.
  const bool single = n <= 8192;
  const int32_t G = single ? 1 : cooperative_grid(n);
  const int64_t entries = n * k;
  if (ws.capacity_entries < entries) {
    ws.capacity_entries = 0;
    ws.vectors.allocate(9 * entries);
    ws.capacity_entries = entries;
  }
  const int64_t partial_size = k * G * 3 + 2 * G + k * G;
  if (ws.partials.size < partial_size) ws.partials.allocate(partial_size);
  double* base = ws.vectors.ptr;
  a.r = base;
  a.u = base + entries;
  a.p = base + 2 * entries;
  a.s = base + 3 * entries;
  a.w = base + 4 * entries;
  a.prev = base + 5 * entries;
  a.res = base + 6 * entries;
  a.da = base + 7 * entries;
  a.db = base + 8 * entries;
  a.partials = ws.partials.ptr;
  const WaitClaim claim(!single, true);
  if (single) {
    hipLaunchKernelGGL((cg_kernel<1024, true>), dim3(1), dim3(1024), 0, stream, a);
    HG_HIP(hipGetLastError());
  } else {
    HG_HIP(hipLaunchCooperativeKernel(reinterpret_cast<const void*>(&cg_kernel<1024, false>),
                                      dim3(G), dim3(1024), args, 0, stream));
  }
  return launched_rounds(ws, stream);
}

void launch_backward_error(const int32_t* offsets, const int32_t* columns, const double* values,
                           const double* x, const double* b, int64_t n, int64_t n_columns,
                           double tolerance, int32_t* flag, hipStream_t stream) {
  if (n == 0) return;
  dim3 grid(static_cast<unsigned>((n + kBlock - 1) / kBlock), static_cast<unsigned>(n_columns));
  backward_error_kernel<<<grid, kBlock, 0, stream>>>(offsets, columns, values, x, b, n, tolerance,
                                                     flag);
  HG_HIP(hipGetLastError());
}

void launch_dominance_bound(const int32_t* offsets, const int32_t* columns, const double* values,
                            int64_t n, double* partials, double* out, hipStream_t stream) {
  int32_t blocks = static_cast<int32_t>((std::max<int64_t>(n, 1) + kBlock - 1) / kBlock);
  if (n > 0)
    dominance_partial_kernel<<<blocks, kBlock, 0, stream>>>(offsets, columns, values, n, partials);
  else
    HG_HIP(hipMemsetAsync(partials, 0, sizeof(double) * blocks, stream));
  dominance_final_kernel<<<1, kBlock, 0, stream>>>(partials, blocks, out);
  HG_HIP(hipGetLastError());
}

}  // namespace hg
