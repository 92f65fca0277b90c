// Merged gate|up projection with the GEGLU epilogue in one kernel, for gfx950:
//   u   = T(x w^T)                   x [rows, K], w = [Wg; Wu] [2F, K] (nn.Linear layout), T = dtype
//   out = T( T(gelu(u[:, :F])) * u[:, F:] )                                          [rows, F]
// This is library/geglu.py's operation on the output of the merged GEMM its docstring names
// (geglu.py:3-5), without writing u to HBM and reading it back. The rounding points are the
// unfused pair's: the fp32 GEMM accumulators are rounded to T (u's dtype), then the GEGLU
// forward of geglu.hip (the same gelu from gelu_math.h) runs on them.
//
// The backward's first step is the same kernel with another epilogue: u is recomputed (the forward
// never wrote it), and with g the GEGLU backward of geglu.hip gives du [rows, 2F] = [da | db] of it.
//
// Tiling (bf16 / fp16 MFMA v_mfma_f32_16x16x32, fp32 accumulate):
//   * Workgroup = 8 waves, 256 rows x 128 output columns (4 waves, 128 x 64, where that leaves CUs
//     idle). The weight tile stacks the gate and the up rows of those columns, so each lane holds
//     gate and up of the same outputs and the epilogue runs in registers, with no exchange.
//   * Wave: 128 rows x 32 output columns (64 x 32 in the small tile).
//   * K is streamed in stages of 64 through double-buffered LDS. Both operands are 16-byte
//     chunks of K-contiguous rows, so both are 128-bit row reads, XOR-swizzled per row to be
//     conflict-free. Stages go HBM -> LDS directly (buffer_load ... lds).
//   * One barrier per stage, before its last products, and a persistent grid whose tiles form one
//     stream of stages (both explained at the loop).
//   * Rows past the end read as zero (buffer range check) and are not stored.
// What bounds it: the card's power limit. At x [8192, 4096], F = 4096 on random data the matrix cores
// are busy 67-72 % of the cycles at 1.9 GHz; on zeros the same instructions run at 2.4 GHz, a fifth
// faster. So what counts is work per joule as much as idle cycles: 16x16x32 products in place of 32x32x16
// (a loop of nothing else: 2140 against 1920 TFLOP/s on random data, both 2450 on zeros), large
// tiles (half the staged bytes per product of 128 x 64), 128-byte row segments (stages of 32 through a
// five-deep ring, whose segments are 64 bytes: 416 against 392 us at an earlier stage of this kernel).
// Measured there: 552 us with 128 x 64 tiles of 32x32x16 and a barrier before each stage's first
// products; 446 us with 256 x 128 tiles and the barrier moved; 392 us with 16x16x32; 383 us persistent, the
// epilogue in registers; 370 us with the requests spread over the products (1485 TFLOP/s; the vendor
// GEMM alone, without the GEGLU step, 352 us on that card).
// The backward's u and du at x [1000, 1024], F = 2816: the vendor GEMM and the GEGLU kernel took
// 22.8 + 8.1 us, this kernel 25.0.
// Requires K % 64 == 0 and F % 64 == 0; the host checks.
#include "gelu_math.h"
#include "krsi_device.h"
#include "krsi_internal.h"
#include "lds_dma.h"
#include "relpos_common.h"

namespace krsi {
namespace {

constexpr int kGlK = 64;       // K per stage
constexpr int kGlGroup = 4;    // row blocks per tile group (tile order, below)

// Every vector memory request and LDS access of the wave done, then the workgroup's barrier.
__device__ __forceinline__ void drain_and_sync() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Chunk j (16 bytes) of staged row r sits at position j ^ swz(r) of the row's 8 chunks: the 16
// lanes of a 128-bit read phase (lane bit 5 and the parity of bits 2-4 fixed) hit distinct bank quads.
__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }

// Four consecutive elements; aligned: the tensor starts on an 8-byte boundary (F % 64 == 0 keeps
// every group of four on one).
template <int DT>
__device__ __forceinline__ void load4(const uint16_t* p, bool aligned, float* f) {
  if (aligned) {
    const u32x2 v = *reinterpret_cast<const u32x2*>(p);
#pragma unroll
    for (int r = 0; r < 4; ++r) f[r] = Elem<DT>::load((uint16_t)(v[r / 2] >> (16 * (r % 2))));
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) f[r] = Elem<DT>::load(p[r]);
  }
}
template <int DT>
__device__ __forceinline__ void store4(uint16_t* p, bool aligned, const float* f) {
  if (aligned) {
    *reinterpret_cast<u32x2*>(p) = u32x2{Elem<DT>::pack2(f[0], f[1]), Elem<DT>::pack2(f[2], f[3])};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] = Elem<DT>::store(f[r]);
  }
}

// Tile of a workgroup of WM x WN waves: each wave computes 16 RB rows x 16 CB output columns (gate
// and up: 16 RB x 32 CB of the GEMM).
template <int WM, int WN, int RB, int CB>
struct GlTile {
  static constexpr int kThreads = 64 * WM * WN;
  static constexpr int kRows = 16 * RB * WM;       // rows of x and out per workgroup
  static constexpr int kCols = 16 * CB * WN;       // output columns: 2 kCols rows of w
  static constexpr int kX = kRows * kGlK;          // 16-bit elements of a staged x tile
  static constexpr int kW = 2 * kCols * kGlK;      // and of a staged w tile
  static constexpr int kXDma = kX / 8 / kThreads;  // 16-byte requests per thread and stage
  static constexpr int kWDma = kW / 8 / kThreads;
  static constexpr int kDma = kXDma + kWDma;
  static constexpr int kPerCu = 160 * 1024 / (4 * (kX + kW));  // workgroups whose two buffers a CU holds
  static_assert(kX / 8 % kThreads == 0 && kW / 8 % kThreads == 0 && kWDma % 2 == 0, "whole chunks per thread");
};

template <int DT, bool TANH, bool BWD, int WM, int WN, int RB, int CB>
__global__ __launch_bounds__(64 * WM * WN, (GlTile<WM, WN, RB, CB>::kPerCu * WM * WN / 4)) void
geglu_linear_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const uint16_t* __restrict__ gout,
                    uint16_t* __restrict__ out, int64_t rows, int K, int F, int ncb, int nrb, int tiles) {
  using Tl = GlTile<WM, WN, RB, CB>;
  using El = Elem<DT>;
  __shared__ __attribute__((aligned(16))) uint16_t lds[2 * (Tl::kX + Tl::kW)];
  uint16_t *const Xs = lds, *const Ws = lds + 2 * Tl::kX;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, l16 = lane & 15;
  const int wr = wave / WN, wc = wave % WN;
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  const int nk = K / kGlK;

  // DMA: chunk p = k * threads + tid of a tile is staged row p / 8, position p % 8, which holds
  // logical chunk (p % 8) ^ swz(row). The first half of the w tile's rows are gate rows c0 ..,
  // the second half up rows F + c0 ...
  uint32_t xoff[Tl::kXDma], woff[Tl::kWDma];
#pragma unroll
  for (int k = 0; k < Tl::kXDma; ++k) {
    const int p = k * Tl::kThreads + tid, row = p >> 3;
    xoff[k] = opaque((uint32_t)(row * K + 8 * ((p & 7) ^ swz(row))) * 2u);
  }
#pragma unroll
  for (int k = 0; k < Tl::kWDma; ++k) {
    const int p = k * Tl::kThreads + tid, row = p >> 3;
    woff[k] = opaque((uint32_t)((row & (Tl::kCols - 1)) * K + 8 * ((p & 7) ^ swz(row))) * 2u);
  }

  // Tile order. xcd_tile gives each XCD a contiguous range of tiles. Inside it the tiles go in
  // groups of kGlGroup row blocks: consecutive tiles walk the group's row blocks first, then
  // its column blocks. The workgroups in flight on one XCD then share a few row blocks of x
  // and a few column blocks of w in that XCD's L2. Walking one row block across every column
  // block instead made each XCD stream all of w once per row block it owns: 4.4 GB fetched per
  // call at x [8192, 4096], F = 4096, against 0.13 GB of inputs.
  struct Where {
    int64_t m0;
    int c0;
  };
  auto locate = [&](int v) {
    const int tile = xcd_tile(v, tiles);
    const int per_group = kGlGroup * ncb;
    const int grp = tile / per_group, in_grp = tile - grp * per_group;
    const int rb0 = grp * kGlGroup;
    const int gsz = min(kGlGroup, nrb - rb0);
    return Where{(int64_t)(rb0 + in_grp % gsz) * Tl::kRows, (in_grp / gsz) * Tl::kCols};
  };
  // A tile's sources. Rows of x past the end, and (F % kCols != 0) rows of w past its gate or up
  // half, fall past the resource and read as zero.
  struct Source {
    const uint16_t *x, *g, *u;
    uint32_t xbytes, wbytes;
  };
  auto source = [&](const Where& t) {
    return Source{x + t.m0 * K, w + (int64_t)t.c0 * K, w + ((int64_t)F + t.c0) * K,
                  (uint32_t)min((int64_t)Tl::kRows, rows - t.m0) * (uint32_t)K * 2u,
                  (uint32_t)(min(Tl::kCols, F - t.c0) * K) * 2u};
  };
  // Request i (of kDma) of this thread for stage kt of a tile into buffer buf.
  auto request = [&](const Source& t, int kt, int buf, int i) {
    const uint32_t kb = (uint32_t)kt * (kGlK * 2);
    if (i < Tl::kXDma) {
      dma16(make_rsrc(t.x + kt * kGlK, t.xbytes - kb), xoff[i],
            (uint32_t)(uintptr_t)(lds_void*)(Xs + buf * Tl::kX + (i * Tl::kThreads + 64 * wv) * 8));
    } else {
      const int k = i - Tl::kXDma;
      dma16(make_rsrc((k < Tl::kWDma / 2 ? t.g : t.u) + kt * kGlK, t.wbytes - kb), woff[k],
            (uint32_t)(uintptr_t)(lds_void*)(Ws + buf * Tl::kW + (k * Tl::kThreads + 64 * wv) * 8));
    }
  };

  // k-step s (32 of the stage's 64) reads chunk 4 s + g of x rows 16 (RB wr + i) + l16 and of w rows
  // 16 (CB wc + j) + l16 (gate) and kCols beyond (up). swz depends on l16 alone.
  u32x4 xa[2][RB], wb[2][2 * CB];
  constexpr int kReads = RB + 2 * CB, kProducts = RB * 2 * CB;
  auto read = [&](int s, int buf, int o) {
    const int ch = 8 * ((4 * s + g) ^ swz(l16));
    if (o < 2 * CB) {
      const int row = (o < CB ? 0 : Tl::kCols) + 16 * (CB * wc + o % CB) + l16;
      wb[s][o] = *reinterpret_cast<const u32x4*>(Ws + buf * Tl::kW + row * kGlK + ch);
    } else {
      const int row = 16 * (RB * wr + o - 2 * CB) + l16;
      xa[s][o - 2 * CB] = *reinterpret_cast<const u32x4*>(Xs + buf * Tl::kX + row * kGlK + ch);
    }
  };
  f32x4 acc[RB][2 * CB];  // [row block][gate blocks, up blocks]
  // The products of k-step s. Operand reads of the next k-step (from buffer rbuf) go out after the
  // even ones, in k-step 1 the requests of stage dt of tile d spread over all of them (every fourth
  // product instead of every second: 379 -> 370 us at x [8192, 4096], F = 4096). The w operand first:
  // the output tile is transposed, a lane holds one row's columns.
  constexpr int kEvery = kProducts / Tl::kDma;
  auto products = [&](int s, int rbuf, const Source& d, int dt) {
#pragma unroll
    for (int m = 0; m < kProducts; ++m) {
      const int i = m / (2 * CB), j = m % (2 * CB);
      acc[i][j] = mfma16x16x32<DT>(wb[s][j], xa[s][i], acc[i][j]);
      if (m % 2 == 0 && m / 2 < kReads) read(s ^ 1, rbuf, m / 2);
      if (s == 1 && m % kEvery == 1) request(d, dt, rbuf ^ 1, m / kEvery);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  static_assert(kReads * 2 <= kProducts && kEvery >= 2 && kEvery * Tl::kDma == kProducts,
                "one k-step's products hold them");

  // Persistent: workgroup b takes tiles b, b + grid, ... (the grid is a multiple of the XCD count or
  // covers every tile), whose stages form one stream through the two buffers. The barrier of a
  // stage stands before its last products, whose operands are in registers by then: every wave has
  // read all of the stage, whose buffer takes the stage after the next, and the next stage has
  // landed. So those products cover the barrier, the requests and the first operand reads of the next
  // stage, and the epilogue of a tile the first loads of the next tile.
  int v = blockIdx.x, buf = 0;
  Where here = locate(v);
  Source cur = source(here);
#pragma unroll
  for (int i = 0; i < Tl::kDma; ++i) request(cur, 0, 0, i);
  drain_and_sync();
#pragma unroll
  for (int o = 0; o < kReads; ++o) read(0, 0, o);
  Where next = locate(min(v + (int)gridDim.x, tiles - 1));
  Source nxt = source(next);
#pragma unroll
  for (int i = 0; i < Tl::kDma; ++i) request(cur, 1, 1, i);  // K = 64: the unused rest of the rows
  for (;;) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < 2 * CB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int kt = 0; kt < nk; ++kt) {
      products(0, buf, cur, 0);
      drain_and_sync();
      // Stage kt + 2 of this tile, or stage kt + 2 - nk of the next one (after the last tile some
      // tile's, not used; also with K = 64, where a workgroup has one tile).
      const bool in = kt + 2 < nk;
      const Source d{in ? cur.x : nxt.x, in ? cur.g : nxt.g, in ? cur.u : nxt.u, in ? cur.xbytes : nxt.xbytes,
                     in ? cur.wbytes : nxt.wbytes};
      products(1, buf ^ 1, d, in ? kt + 2 : kt + 2 - nk);
      buf ^= 1;
    }
    // Epilogue, in registers: u rounded to T as the unfused GEMM stores it, then the GEGLU step.
    // acc[i][j] holds row 16 (RB wr + i) + l16, columns 16 (CB wc + j) + 4 g + r of the gate, acc[i][CB + j]
    // the same of the up half.
    const bool aligned = (((uintptr_t)out | (uintptr_t)gout) & 7) == 0;
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      const int64_t row = here.m0 + 16 * (RB * wr + i) + l16;
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        const int col = here.c0 + 16 * (CB * wc + j) + 4 * g;
        if (row >= rows || col >= F) continue;
        float a[4], b[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          a[r] = El::round(acc[i][j][r]);
          b[r] = El::round(acc[i][CB + j][r]);
        }
        if constexpr (BWD) {
          float gg[4], da[4], db[4];
          load4<DT>(gout + row * F + col, aligned, gg);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float d;
            const float gel = gelu_fwd_bwd<DT, TANH>(a[r], d);
            db[r] = gg[r] * El::round(gel);
            da[r] = El::round(gg[r] * b[r]) * d;
          }
          uint16_t* p = out + row * 2 * F + col;
          store4<DT>(p, aligned, da);
          store4<DT>(p + F, aligned, db);
        } else {
          float o[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = El::round(gelu_fwd<DT, TANH>(a[r])) * b[r];
          store4<DT>(out + row * F + col, aligned, o);
        }
      }
    }
    v += gridDim.x;
    if (v >= tiles) break;
    here = next;
    cur = nxt;
    next = locate(min(v + (int)gridDim.x, tiles - 1));
    nxt = source(next);
  }
  drain_and_sync();  // the unused requests land before the workgroup's LDS is released
}

constexpr int kCus = 256;

template <int DT, bool TANH, bool BWD, int WM, int WN, int RB, int CB>
int launch_tile(const uint16_t* x, const uint16_t* w, const uint16_t* g, uint16_t* out, int64_t rows, int K, int F,
                hipStream_t st) {
  using Tl = GlTile<WM, WN, RB, CB>;
  const int ncb = (int)ceil_div(F, Tl::kCols);
  const int64_t nrb = ceil_div(rows, Tl::kRows);
  const int64_t tiles = nrb * ncb;
  if (tiles > 0x7fffffff) return KRSI_ERR_BAD_SHAPE;
  // The kernel's stream of stages reaches one tile ahead, two stages: with one stage per tile every
  // workgroup takes one tile.
  const int64_t resident = K > kGlK ? kCus * Tl::kPerCu : tiles;
  hipLaunchKernelGGL((geglu_linear_kernel<DT, TANH, BWD, WM, WN, RB, CB>),
                     dim3((unsigned)(tiles < resident ? tiles : resident)), dim3(Tl::kThreads), 0, st, x, w, g, out,
                     rows, K, F, ncb, (int)nrb, (int)tiles);
  return launch_status();
}

// 256 x 128 tiles, one workgroup per CU, or 128 x 64, two per CU, a round of which covers half as
// much. At full rounds the large tile runs 1.2 times faster (x [8192, 4096], F = 4096: 370 against
// 452 us; it reads and stages less per product); it loses when its last round leaves CUs idle (x
// [1000, 1024], F = 2816: 88 tiles, 26.2 against 18.1 us; x [4096, 1024], F = 2816: 352 tiles, 50.8
// against 48.3). So: the large tile when its rounds cost no more at 1.2 small rounds of half the work
// (and its byte offsets stay below 2^31).
template <int DT, bool TANH, bool BWD>
int launch_geglu_linear(const void* x, const void* w, const void* g, void* out, int64_t rows, int K, int F,
                        hipStream_t st) {
  using Large = GlTile<2, 4, 8, 2>;
  using Small = GlTile<2, 2, 4, 2>;
  const uint16_t *xp = (const uint16_t*)x, *wp = (const uint16_t*)w, *gp = (const uint16_t*)g;
  uint16_t* op = (uint16_t*)out;
  const int64_t large = ceil_div(ceil_div(rows, Large::kRows) * ceil_div(F, Large::kCols), kCus * Large::kPerCu);
  const int64_t small = ceil_div(ceil_div(rows, Small::kRows) * ceil_div(F, Small::kCols), kCus * Small::kPerCu);
  if (5 * large <= 3 * small && (int64_t)Large::kRows * K * 2 < ((int64_t)1 << 31))
    return launch_tile<DT, TANH, BWD, 2, 4, 8, 2>(xp, wp, gp, op, rows, K, F, st);
  return launch_tile<DT, TANH, BWD, 2, 2, 4, 2>(xp, wp, gp, op, rows, K, F, st);
}

int check(int64_t rows, int32_t k, int32_t f, int32_t approximate, int32_t dtype) {
  if (dtype != kBf16 && dtype != kF16) return KRSI_ERR_UNSUPPORTED;
  if (approximate != 0 && approximate != 1) return KRSI_ERR_UNSUPPORTED;
  if (rows < 0 || k <= 0 || f <= 0) return KRSI_ERR_BAD_SHAPE;
  if (k % 64 != 0 || f % 64 != 0) return KRSI_ERR_UNSUPPORTED;
  // Buffer resources: the byte offsets of a small tile (128 rows of x, 64 of w) stay below 2^31.
  if ((int64_t)128 * k * 2 >= ((int64_t)1 << 31)) return KRSI_ERR_UNSUPPORTED;
  return KRSI_OK;
}

template <bool BWD>
int geglu_linear(const void* x, const void* w, const void* g, void* out, int64_t rows, int k, int f, bool tanh_form,
                 int dtype, hipStream_t st) {
  if (tanh_form)
    return dtype == kF16 ? launch_geglu_linear<kF16, true, BWD>(x, w, g, out, rows, k, f, st)
                         : launch_geglu_linear<kBf16, true, BWD>(x, w, g, out, rows, k, f, st);
  return dtype == kF16 ? launch_geglu_linear<kF16, false, BWD>(x, w, g, out, rows, k, f, st)
                       : launch_geglu_linear<kBf16, false, BWD>(x, w, g, out, rows, k, f, st);
}

}  // namespace
}  // namespace krsi

extern "C" {

int krsi_geglu_linear_fwd(const void* x, const void* w, void* out, int64_t rows, int32_t k, int32_t f,
                          int32_t approximate, int32_t dtype, void* stream) {
  using namespace krsi;
  const int rc = check(rows, k, f, approximate, dtype);
  if (rc != KRSI_OK) return rc;
  if (rows == 0) return KRSI_OK;
  if (!x || !w || !out) return KRSI_ERR_NULL_POINTER;
  if (!aligned16(x) || !aligned16(w)) return KRSI_ERR_MISALIGNED;
  return geglu_linear<false>(x, w, nullptr, out, rows, k, f, approximate == 1, dtype, as_stream(stream));
}

int krsi_geglu_linear_bwd(const void* g, const void* x, const void* w, void* du, int64_t rows, int32_t k, int32_t f,
                          int32_t approximate, int32_t dtype, void* stream) {
  using namespace krsi;
  const int rc = check(rows, k, f, approximate, dtype);
  if (rc != KRSI_OK) return rc;
  if (rows == 0) return KRSI_OK;
  if (!g || !x || !w || !du) return KRSI_ERR_NULL_POINTER;
  if (!aligned16(x) || !aligned16(w)) return KRSI_ERR_MISALIGNED;
  return geglu_linear<true>(x, w, g, du, rows, k, f, approximate == 1, dtype, as_stream(stream));
}

}  // extern "C"
