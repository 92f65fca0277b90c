// Loads through raw buffer resources, straight into LDS where asked, and the transposed LDS reads that the
// 16-bit MFMA operands take: shared by the attention and projection kernels.
#pragma once

#include "krsi_device.h"

namespace krsi {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) void lds_void;

// Raw buffer resources (gfx9 descriptor word 3): a load whose byte offset is at or
// past num_records returns zero.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
constexpr int kRsrcWord3 = 0x00020000;
__device__ __forceinline__ rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, kRsrcWord3);
}

// The whole byte offset must reach the instruction in the VGPR: the range check is
// made on the VGPR offset, so a constant the compiler split off into the immediate
// field would turn a valid offset whose variable part is negative into a zero read.
// An empty asm makes the offset opaque, so no constant can be split off.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

// One buffer_load_dwordx4 ... lds: 16 bytes per lane from the buffer to LDS at m0 + 16 * lane. It is issued
// from asm on purpose: the compiler treats the builtin form as an LDS write of unknown extent and
// waits for it before every later LDS read, which would complete each step's prefetch before
// that step's own compute. Invisible to the compiler, the request stays in flight until the
// kernel's explicit wait before the step that reads it; the compiler's own vmcnt waits only ever
// over-wait because of it.
__device__ __forceinline__ void dma16(rsrc_t r, uint32_t voff, uint32_t m0) {
  asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(r), "{m0}"(m0) : "memory");
}

// Chunk j (16 bytes) of a staged row r of W 16-bit elements sits at j ^ swz16<W>(r): conflict-free for 128-bit reads
// of 16 rows (lane bit 5 and the parity of bits 2-4 fixed) and for transposed 64-bit reads of 8 rows x 2 chunks.
template <int W>
__device__ __forceinline__ int swz16(int r) {
  constexpr int C = W / 8;
  int s = ((r >> 2) & 1) << 1;
  if constexpr (C == 8) s |= ((r >> 1) & 1) << 2;
  if constexpr (C == 16) s |= (r & 3) << 2;
  return s;
}

// Per-lane element offsets into a tile of rows of W elements so staged, for 16x16x32 products with NS 32-wide steps
// and NC 16-wide blocks of columns. row[s]: the 128-bit read of row l % 16, columns 32 s + 8 (l / 16) .. + 7.
// tr[c]: the transposed read of rows 4 (l / 16) .. + 3 of column 16 c + l % 16 (lane s of a 16-lane group
// addresses row s / 4, columns 4 (s % 4) .. + 3 of the 4 x 16 block).
template <int W, int NS, int NC>
struct LaneOffsets16 {
  static constexpr int LD = W, KS = NS, CB = NC;
  int row[KS], tr[CB];
  static __device__ __forceinline__ int off(int r, int j) { return r * LD + 8 * (j ^ swz16<LD>(r)); }
  __device__ __forceinline__ void init(int g, int l16) {  // l / 16 and l % 16
#pragma unroll
    for (int s = 0; s < KS; ++s) row[s] = off(l16, 4 * s + g);
#pragma unroll
    for (int c = 0; c < CB; ++c) tr[c] = off(4 * g + (l16 >> 2), 2 * c + ((l16 & 3) >> 1)) + 4 * (l16 & 1);
  }
};

}  // namespace krsi
