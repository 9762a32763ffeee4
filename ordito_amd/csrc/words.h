// Words that are their own arrival flags, for blocks of one launch that hand values to each other.
//
// A word holds kEmpty until its value is published. A reader polls the very word it needs, so a
// hand-over costs one store-to-load latency; there is no separate flag to order after the data.
// Publishing and reading are agent-scope relaxed atomics: such stores write through to where every
// XCD sees them and such loads look there, so no L2 is written back or invalidated, as the
// release and acquire of a grid barrier would.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace hg {

constexpr uint64_t kEmpty = 0x7FF4A5A5C3C3F00Dull;  // a signaling NaN, which no arithmetic returns
constexpr uint64_t kQuietNan = 0x7FF8000000000000ull;

// Polls of a wait before it gives up: each poll is an agent-scope load (about a microsecond), so
// about two seconds, thousands of times the longest legitimate wait.
constexpr int64_t kSpinLimit = int64_t{1} << 21;

__device__ __forceinline__ void publish(double* word, double v) {
  uint64_t bits = __builtin_bit_cast(uint64_t, v);
  if (bits == kEmpty) bits = kQuietNan;
  __hip_atomic_store(reinterpret_cast<uint64_t*>(word), bits, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void empty(double* word) {
  __hip_atomic_store(reinterpret_cast<uint64_t*>(word), kEmpty, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint64_t peek(const double* word) {
  return __hip_atomic_load(reinterpret_cast<const uint64_t*>(word), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}

// This wave's stores have reached the point of coherence.
__device__ __forceinline__ void drain_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The most polls a wait may be told to make: its count of them goes one further.
constexpr int64_t kMostPolls = (int64_t{1} << 31) - 2;

// A wait's patience: false once it has polled past `limit` (at most kMostPolls) or another wait has
// given up, which it then tells everyone by setting `bit` of *flag.
__device__ __forceinline__ bool wait_on(int32_t* flag, int32_t bit, int64_t limit, int32_t& polls,
                                        bool& aborted) {
  if (aborted) return false;
  if ((++polls & 255) == 0 || polls > limit) {
    if (polls > limit ||
        (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit) != 0) {
      __hip_atomic_fetch_or(flag, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      aborted = true;
      return false;
    }
  }
  return true;
}

}  // namespace hg
