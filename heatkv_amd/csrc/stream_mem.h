// Non-temporal accesses for the streaming kernels (copies, the producer).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hkv {

// Written once and read by a later launch.  Only for stores of which one wave
// instruction fills whole 128-byte lines: a line filled by several
// non-temporal stores reaches memory in pieces (the producer's fp32 q rows in
// two 16-byte halves per lane: 65 us with them against 47 us without at 4096
// tokens, B=2, 16 heads).
template <typename T, typename U>
__device__ __forceinline__ void stream_store(T* p, U v) {
  __builtin_nontemporal_store(v, p);
}

// Read once.
template <typename T>
__device__ __forceinline__ T stream_load(const T* p) {
  return __builtin_nontemporal_load(p);
}

}  // namespace hkv
