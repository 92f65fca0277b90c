// The two products of geglu_linear's backward in one launch, for gfx950:
//   dx = T(du w)     [rows, K]     du [rows, 2F], w [2F, K]
//   dw = T(du^T x)   [2F, K]       x [rows, K]
// (fp32 accumulate, T = bf16 or fp16), for sizes at which either product alone leaves CUs idle. dx has few
// output tiles and a long sum: it is split over workgroups, whose fp32 parts a second kernel adds in
// order, so results are reproducible and depend on the sizes alone. dw's tiles fill the rest of the chip.
//
// What bounds it: at these sizes the staging of operands through each XCD's L2 and the length of a
// workgroup's chain of stages. At rows 1000, K 1024, F 2816 (23 Gflop) the vendor's products take 33.2 +
// 26.8 us in two launches, this 39.8 (580 TFLOP/s) with the addition of dx's parts; a training step there
// 97.2 -> 79.9 us.
//
// Tiling (bf16 / fp16 MFMA v_mfma_f32_16x16x32):
//   * Workgroup = 4 waves of 64 x 64, 128 x 128 outputs, 64 KB of LDS: two per CU.
//   * The sum is streamed in stages of 64 through double-buffered LDS, memory -> LDS directly, one
//     barrier per stage before its last products (as in geglu_linear_kernel).
//   * du in dx holds the summed index contiguously: 128-bit row reads. The other three operands hold the
//     output index contiguously: transposed 64-bit reads (ds_read_b64_tr_b16), of rows 8 g .. 8 g + 3 and
//     8 g + 4 .. 8 g + 7 of a k-step for lane group g, which is the operand order of row reads too.
//   * Rows and columns past an end read as zero (buffer range check) and are not stored.
#include "krsi_device.h"
#include "krsi_internal.h"
#include "lds_dma.h"
#include "relpos_common.h"

namespace krsi {
namespace {

constexpr int kGk = 64;         // summed index per stage
constexpr int kGt = 128;        // rows and columns of an output tile
constexpr int kGThreads = 256;
constexpr int kGTile = kGt * kGk;                      // 16-bit elements of a staged tile
constexpr int kGDma = kGTile / 8 / kGThreads;          // 16-byte requests per thread and tile
constexpr int kGGroup = 4;                             // row blocks per tile group (order of the tiles)
constexpr int kGSlots = 512;                           // workgroups that the chip holds: two per CU
constexpr int kGMinStages = 16;                        // stages of a part of a split sum, about
constexpr uint32_t kGOob = 0x7ffffff0u;                // past every resource

// Every vector memory request and LDS access of the wave done, then the workgroup's barrier.
__device__ __forceinline__ void drain_and_sync() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Chunk j (16 bytes) of a staged row r sits at j ^ swz: of 8 chunks where rows are output rows, conflict-free
// for 128-bit reads of 16 rows; of 16 chunks where rows are the summed index, conflict-free for transposed
// 64-bit reads of rows 0-3 and 8-11 (or 4-7 and 12-15) of 16 x 2 chunks.
__device__ __forceinline__ int swz_row(int r) { return (r >> 1) & 7; }
__device__ __forceinline__ int swz_tr(int r) { return ((r & 3) | ((r >> 3) & 1) << 2) << 1; }

// out [M, N] = a b over `sum` indices; a is [M, sum] (rows) or [sum, M] (transposed), b [sum, N].
struct Product {
  const uint16_t *a, *b;
  uint16_t* out;
  float* part;       // [splits, M, N] where splits > 1
  int64_t lda, ldb;  // elements; out is contiguous
  int64_t M, sum;
  int N, nmb, nnb, splits, per;  // tiles down and across, workgroups per tile, stages of each
  int blocks;                    // nmb nnb splits
};

template <int DT, bool TA>
__device__ __forceinline__ void product_tile(const Product& p, int v, uint16_t* lds) {
  uint16_t *const As = lds, *const Bs = lds + 2 * kGTile;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, l16 = lane & 15;
  const int wr = wave >> 1, wc = wave & 1;
  const int wv = __builtin_amdgcn_readfirstlane(wave);

  // Each XCD takes a contiguous range; consecutive tiles walk a group's row blocks, then the columns.
  const int tiles = p.nmb * p.nnb;
  const int vv = xcd_tile(v, p.blocks), split = vv / tiles, tile = vv - split * tiles;
  const int per_group = kGGroup * p.nnb, grp = tile / per_group, in_grp = tile - grp * per_group;
  const int gsz = min(kGGroup, p.nmb - grp * kGGroup);
  const int64_t m0 = (int64_t)(grp * kGGroup + in_grp % gsz) * kGt;
  const int n0 = in_grp / gsz * kGt;
  const int stages = (int)((p.sum + kGk - 1) / kGk);
  const int s0 = split * p.per, s1 = min(stages, s0 + p.per);

  // DMA: chunk q = i * threads + tid of a tile.
  uint32_t aoff[kGDma], boff[kGDma];
#pragma unroll
  for (int i = 0; i < kGDma; ++i) {
    const int q = i * kGThreads + tid;
    const int r = q >> 4, col = 8 * ((q & 15) ^ swz_tr(r));
    if (TA) {
      aoff[i] = opaque(m0 + col < p.M ? (uint32_t)(r * p.lda + col) * 2u : kGOob);
    } else {
      const int ar = q >> 3;
      aoff[i] = opaque((uint32_t)(ar * p.lda + 8 * ((q & 7) ^ swz_row(ar))) * 2u);
    }
    boff[i] = opaque(n0 + col < p.N ? (uint32_t)(r * p.ldb + col) * 2u : kGOob);
  }
  // Stage st into buffer buf; request i of 2 kGDma.
  auto request = [&](int st, int buf, int i) {
    const int64_t k0 = (int64_t)st * kGk;
    const int left = (int)min((int64_t)kGk, p.sum - k0);
    if (i < kGDma) {
      const uint16_t* base = TA ? p.a + k0 * p.lda + m0 : p.a + m0 * p.lda + k0;
      const int64_t n = TA ? left * p.lda - m0 : min((int64_t)kGt, p.M - m0) * p.lda - k0;
      dma16(make_rsrc(base, (uint32_t)(n * 2)), aoff[i],
            (uint32_t)(uintptr_t)(lds_void*)(As + buf * kGTile + (i * kGThreads + 64 * wv) * 8));
    } else {
      const int k = i - kGDma;
      dma16(make_rsrc(p.b + k0 * p.ldb + n0, (uint32_t)((left * p.ldb - n0) * 2)), boff[k],
            (uint32_t)(uintptr_t)(lds_void*)(Bs + buf * kGTile + (k * kGThreads + 64 * wv) * 8));
    }
  };

  u32x4 a[2][4], b[2][4];
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int trow = 8 * g + (l16 >> 2), tsw = swz_tr(trow), tb = (l16 & 3) >> 1, te = 4 * (l16 & 1);
  // Columns 16 c + l16 of a [64, 128] tile, rows 32 s + 8 g .. + 7.
  auto read_tr = [&](const uint16_t* t, int s, int c) {
    const uint16_t* q = t + (32 * s + trow) * kGt + 8 * ((2 * c + tb) ^ tsw) + te;
    const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)q));
    const u32x2 y = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(q + 4 * kGt)));
    return u32x4{x[0], x[1], y[0], y[1]};
  };
  auto read = [&](int s, int buf, int o) {
    if (o < 4) {
      b[s][o] = read_tr(Bs + buf * kGTile, s, 4 * wc + o);
    } else if (TA) {
      a[s][o - 4] = read_tr(As + buf * kGTile, s, 4 * wr + o - 4);
    } else {
      const int row = 16 * (4 * wr + o - 4) + l16;
      a[s][o - 4] = *reinterpret_cast<const u32x4*>(As + buf * kGTile + row * kGk + 8 * ((4 * s + g) ^ swz_row(l16)));
    }
  };
  // The products of k-step s, with the operand reads of the next k-step and (s = 1) the requests of stage
  // st among them. b first: the output is transposed, a lane holds four columns of one row.
  auto products = [&](int s, int rbuf, bool reads, bool requests, int st) {
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      acc[m / 4][m % 4] = mfma16x16x32<DT>(b[s][m % 4], a[s][m / 4], acc[m / 4][m % 4]);
      if (m % 2 == 0 && reads) read(s ^ 1, rbuf, m / 2);
      if (m % 2 == 1 && requests) request(st, rbuf ^ 1, m / 2);
    }
  };

#pragma unroll
  for (int i = 0; i < 2 * kGDma; ++i) request(s0, 0, i);
  drain_and_sync();
#pragma unroll
  for (int o = 0; o < 8; ++o) read(0, 0, o);
  if (s0 + 1 < s1) {
#pragma unroll
    for (int i = 0; i < 2 * kGDma; ++i) request(s0 + 1, 1, i);
  }
  int buf = 0;
  for (int st = s0; st + 1 < s1; ++st) {
    products(0, buf, true, false, 0);
    drain_and_sync();  // all of stage st is in registers, stage st + 1 has landed
    if (st + 2 < s1)
      products(1, buf ^ 1, true, true, st + 2);
    else
      products(1, buf ^ 1, true, false, 0);
    buf ^= 1;
  }
  products(0, buf, true, false, 0);
  products(1, buf, false, false, 0);

  const bool aligned = ((uintptr_t)p.out & 7) == 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t row = m0 + 16 * (4 * wr + i) + l16;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = n0 + 16 * (4 * wc + j) + 4 * g;
      if (row >= p.M || col >= p.N) continue;
      const f32x4 v4 = acc[i][j];
      if (p.splits > 1) {
        *reinterpret_cast<f32x4*>(p.part + ((int64_t)split * p.M + row) * p.N + col) = v4;
      } else if (aligned) {
        *reinterpret_cast<u32x2*>(p.out + row * p.N + col) =
            u32x2{Elem<DT>::pack2(v4[0], v4[1]), Elem<DT>::pack2(v4[2], v4[3])};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) p.out[row * p.N + col + r] = Elem<DT>::store(v4[r]);
      }
    }
  }
}

template <int DT>
__global__ __launch_bounds__(kGThreads, 2) void geglu_linear_grads_kernel(Product dx, Product dw) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[4 * kGTile];
  if ((int)blockIdx.x < dx.blocks)
    product_tile<DT, false>(dx, blockIdx.x, lds);
  else
    product_tile<DT, true>(dw, blockIdx.x - dx.blocks, lds);
}

// out = the parts' sum, in order; zero where there is none.
template <int DT>
__global__ __launch_bounds__(256) void geglu_linear_grads_sum(Product dx, Product dw, int dx_blocks) {
  const bool first = (int)blockIdx.x < dx_blocks;
  const Product& p = first ? dx : dw;
  const int64_t n = p.M * p.N, i = ((int64_t)(first ? blockIdx.x : blockIdx.x - dx_blocks) * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  f32x4 s = p.splits ? *reinterpret_cast<const f32x4*>(p.part + i) : f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k = 1; k < p.splits; ++k) s += *reinterpret_cast<const f32x4*>(p.part + k * n + i);
  if (((uintptr_t)p.out & 7) == 0) {
    *reinterpret_cast<u32x2*>(p.out + i) = u32x2{Elem<DT>::pack2(s[0], s[1]), Elem<DT>::pack2(s[2], s[3])};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) p.out[i + r] = Elem<DT>::store(s[r]);
  }
}

// Stages of all tiles of both products.
int64_t total_stages(int64_t rows, int k, int f) {
  return ceil_div(k, kGt) * (ceil_div(rows, kGt) * ceil_div(2 * (int64_t)f, kGk) +
                             ceil_div(2 * (int64_t)f, kGt) * ceil_div(rows, kGk));
}

// Both products by sizes alone. Stages per workgroup: what spreads all stages of both products over
// the chip once, but no fewer than 16, below which adding the parts costs more than the chain it cuts
// (with 8, dx alone at rows 951, K 3136, F 320, 10 stages in two parts, took 22.8 us).
void plan(int64_t rows, int k, int f, Product& dx, Product& dw) {
  const int64_t f2 = 2 * (int64_t)f;
  dx = Product{};
  dw = Product{};
  dx.lda = f2, dx.ldb = k, dx.M = rows, dx.sum = f2;
  dw.lda = f2, dw.ldb = k, dw.M = f2, dw.sum = rows;
  for (Product* p : {&dx, &dw}) {
    p->N = k;
    p->nmb = (int)ceil_div(p->M, kGt);
    p->nnb = (int)ceil_div(k, kGt);
  }
  const int64_t even = total_stages(rows, k, f) / kGSlots + 1, target = even < kGMinStages ? kGMinStages : even;
  for (Product* p : {&dx, &dw}) {
    const int64_t stages = ceil_div(p->sum, kGk);
    p->per = (int)ceil_div(stages, ceil_div(stages, target));
    p->splits = (int)ceil_div(stages, p->per);
    p->blocks = p->nmb * p->nnb * p->splits;
  }
}
size_t part_bytes(const Product& p) { return p.splits > 1 ? align256((size_t)p.splits * p.M * p.N * 4) : 0; }

template <int DT>
int launch(Product dx, Product dw, hipStream_t st) {
  hipLaunchKernelGGL((geglu_linear_grads_kernel<DT>), dim3((unsigned)(dx.blocks + dw.blocks)), dim3(kGThreads), 0, st,
                     dx, dw);
  const int64_t a = dx.blocks && dx.splits > 1 ? ceil_div(dx.M * dx.N, 1024) : 0;
  const int64_t b = dw.blocks && dw.splits > 1 ? ceil_div(dw.M * dw.N, 1024) : 0;
  if (a + b)
    hipLaunchKernelGGL((geglu_linear_grads_sum<DT>), dim3((unsigned)(a + b)), dim3(256), 0, st, dx, dw, (int)a);
  return launch_status();
}

// dw of an empty batch is zero.
template <int DT>
int launch_empty(void* dw, int k, int f, hipStream_t st) {
  Product none{}, z{};
  z.out = (uint16_t*)dw, z.M = 2 * (int64_t)f, z.N = k;
  hipLaunchKernelGGL((geglu_linear_grads_sum<DT>), dim3((unsigned)ceil_div(z.M * z.N, 1024)), dim3(256), 0, st, none, z,
                     0);
  return launch_status();
}

// Sizes that the kernel takes: whole 64-column blocks, byte offsets of a tile below 2^31, grids of int.
bool takes(int64_t rows, int32_t k, int32_t f) {
  return rows > 0 && rows <= 0x7fffffff / 4 && k > 0 && f > 0 && k % 64 == 0 && f % 64 == 0 && k <= (1 << 22) &&
         f <= (1 << 21) && ceil_div(rows, kGt) * ceil_div(k, kGt) < (1 << 20) &&
         ceil_div(2 * (int64_t)f, kGt) * ceil_div(k, kGt) < (1 << 20);
}

// Sizes at which this kernel is the faster one (bf16; us of the vendor's products / of this kernel, in graphs).
// Each product has tiles of 128 x 128 and stages of 64; n stages in all tiles of both. Measured over rows
// 64-65536 (131072 for dw alone), K 64-8192 and F 64-8192; not above.
// Both: the kernel wins by one launch and dx's split while the work is small, and by dw's split where rows are
// many, which the library does not cut (rows 65536, K 512, F 512: 331 / 203). It loses to the library's
// larger tiles once dx has work for every CU (tiles 1024: 8192, 2048, 1024 152.4 / 160.2, 4096, 4096, 1536
// 182.8 / 206.1; tiles 768: 4096, 3072, 1024, n 49152 1.07 times faster, 4096, 3072, 2048, n 98304 193 / 201;
// tiles 512: 2000, 4096, 2816, n 90112 1.06 times faster; n 131072: 248 / 238 to 235 / 242). At n up to 32768 it
// was 0.99 to 6 times as fast throughout.
// dw alone: tiles up to 512 (1024 of 8 stages: 512, 2048, 4096 26.8 / 29.5) and more than one stage (64, 8192,
// 8192 69.6 / 89.9), where it was 0.96-7 times as fast. Its parts are planned for both products, so that dw
// is bitwise the same with and without dx: 193-256 tiles of 33-64 stages are then not cut and leave
// half of the chip idle (4096, 2048, 1024 50.1 / 54.3). And not one narrow column of many tiles (4096, 128, 8192
// 37.7 / 44.4).
// dx alone (K from 256): long sums of few tiles, which are cut (64, 1024, 2816 27.0 / 15.0; 1000, 1024, 2816 34.8 / 26.7;
// 8192, 256, 4096 84.0 / 53.4); not where the library cuts them too (8 tiles and less at K below 512: 130,
// 448, 2304 11.1 / 14.9), and the shorter the sum, the fewer the tiles (72 stages: 3000, 320 and 300, 3072, 72
// tiles 0.96 times as fast; 128 tiles 128 stages 1.17-1.21). And sums of at most 8 stages on 129-256
// tiles, one round of one workgroup per CU (1000, 4096, 256 12.5 / 10.3); not on fewer (512, 1024, 128 5.8 / 6.9)
// or more (49152, 4096, 128 0.82 times as fast).
bool pays(int64_t rows, int k, int f, bool dx, bool dw) {
  if (rows > 131072 || k > 8192 || f > 8192) return false;
  const int64_t n = total_stages(rows, k, f), across = ceil_div(k, kGt);
  const int64_t dx_tiles = ceil_div(rows, kGt) * across, dx_stages = ceil_div(2 * (int64_t)f, kGk);
  const int64_t dw_tiles = ceil_div(2 * (int64_t)f, kGt) * across, dw_stages = ceil_div(rows, kGk);
  if (dx && dw)
    return n <= 32768 || (n <= 65536 && (dx_tiles <= 768 || rows >= 16384)) || (n <= 98304 && dx_tiles <= 512);
  if (dw)
    return n <= 32768 && dw_stages > 1 && dw_tiles <= 512 && (k >= 256 || f <= 4096) &&
           (dw_tiles <= 192 || dw_tiles > 256 || dw_stages <= 32);
  if (!dx || k < 256 || dx_stages > 128) return false;
  if (dx_stages <= 8) return dx_tiles > 128 && dx_tiles <= 256;
  if (dx_tiles <= 8 && k < 512) return false;
  return dx_tiles <= (dx_stages >= 126 ? 128 : dx_stages >= 96 ? 96 : dx_stages >= 72 ? 64 : 0);
}

}  // namespace
}  // namespace krsi

extern "C" {

int krsi_geglu_linear_grads_pays(int64_t rows, int32_t k, int32_t f, int32_t dx, int32_t dw) {
  using namespace krsi;
  return takes(rows, k, f) && pays(rows, k, f, dx != 0, dw != 0) ? 1 : 0;
}

size_t krsi_geglu_linear_grads_workspace_bytes(int64_t rows, int32_t k, int32_t f) {
  using namespace krsi;
  if (!takes(rows, k, f)) return 0;
  Product dx, dw;
  plan(rows, k, f, dx, dw);
  return part_bytes(dx) + part_bytes(dw);
}

int krsi_geglu_linear_grads(const void* du, const void* x, const void* w, void* dx, void* dw, void* workspace,
                            size_t workspace_bytes, int64_t rows, int32_t k, int32_t f, int32_t dtype, void* stream) {
  using namespace krsi;
  if (dtype != kBf16 && dtype != kF16) return KRSI_ERR_UNSUPPORTED;
  if (rows < 0 || k <= 0 || f <= 0) return KRSI_ERR_BAD_SHAPE;
  if (!takes(rows ? rows : 1, k, f)) return KRSI_ERR_UNSUPPORTED;
  if (rows == 0) {
    if (!dw) return KRSI_OK;
    return dtype == kF16 ? launch_empty<kF16>(dw, k, f, as_stream(stream))
                         : launch_empty<kBf16>(dw, k, f, as_stream(stream));
  }
  if (!du || !x || !w || (!dx && !dw)) return KRSI_ERR_NULL_POINTER;
  if (!aligned16(du) || !aligned16(x) || !aligned16(w)) return KRSI_ERR_MISALIGNED;
  Product px, pw;
  plan(rows, k, f, px, pw);
  const size_t need = part_bytes(px) + part_bytes(pw);
  if (need && (!workspace || workspace_bytes < need)) return KRSI_ERR_WORKSPACE;
  if (need && !aligned16(workspace)) return KRSI_ERR_MISALIGNED;
  px.a = pw.a = (const uint16_t*)du;
  px.b = (const uint16_t*)w;
  pw.b = (const uint16_t*)x;
  px.out = (uint16_t*)dx;
  pw.out = (uint16_t*)dw;
  px.part = (float*)workspace;
  pw.part = (float*)((char*)workspace + part_bytes(px));
  if (!dx) px.blocks = 0;
  if (!dw) pw.blocks = 0;
  return dtype == kF16 ? launch<kF16>(px, pw, as_stream(stream)) : launch<kBf16>(px, pw, as_stream(stream));
}

}  // extern "C"
