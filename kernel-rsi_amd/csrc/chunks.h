// 16-byte chunks of rows, for the memory-bound kernels. RAGGED rows have any length (at least a chunk) and
// alignment (of the element) and go through the unaligned 128-bit accesses that the hardware takes. The last
// chunk of a ragged row ends at the row's end: it shares columns with the chunk before it, and both
// chunks' threads compute and store the same values there. Ragged rows share cache lines between
// waves and rows, so they are loaded and stored normally where aligned ones stream.
#pragma once

#include "krsi_device.h"

namespace krsi {

typedef u32x4 u32x4_any __attribute__((aligned(2)));
typedef f32x4 f32x4_any __attribute__((aligned(4)));

// Read once: non-temporal where aligned.
template <bool RAGGED, typename T>
__device__ __forceinline__ u32x4 stream_chunk(const T* p) {
  if constexpr (RAGGED) return *reinterpret_cast<const u32x4_any*>(p);
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}
template <bool RAGGED, typename T>
__device__ __forceinline__ u32x4 load_chunk(const T* p) {
  if constexpr (RAGGED) return *reinterpret_cast<const u32x4_any*>(p);
  return *reinterpret_cast<const u32x4*>(p);
}
template <bool RAGGED, typename T>
__device__ __forceinline__ void store_chunk(T* p, const u32x4& v) {
  if constexpr (RAGGED)
    *reinterpret_cast<u32x4_any*>(p) = v;
  else
    __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
}

// First column of chunk c (of E elements) of a row of n, and how many of its leading columns the chunk before it has.
template <bool RAGGED, int E>
__device__ __forceinline__ int chunk_col(int c, int n) {
  return RAGGED ? min(c * E, n - E) : c * E;
}
template <bool RAGGED, int E>
__device__ __forceinline__ int chunk_shared(int c, int n) {
  return RAGGED ? max(c * E - (n - E), 0) : 0;
}
// The chunk's address. Aligned rows index whole chunks: added to the row's offset as a count of elements, each
// chunk held one more address register (RMSNorm backward, fp32 rows of 8192: one wave per SIMD instead of two).
template <bool RAGGED, int E, typename T>
__device__ __forceinline__ const T* chunk_at(const T* row, int c, int n) {
  if constexpr (RAGGED) return row + chunk_col<true, E>(c, n);
  return reinterpret_cast<const T*>(reinterpret_cast<const u32x4*>(row) + c);
}
template <bool RAGGED, int E, typename T>
__device__ __forceinline__ T* chunk_at(T* row, int c, int n) {
  if constexpr (RAGGED) return row + chunk_col<true, E>(c, n);
  return reinterpret_cast<T*>(reinterpret_cast<u32x4*>(row) + c);
}

}  // namespace krsi
