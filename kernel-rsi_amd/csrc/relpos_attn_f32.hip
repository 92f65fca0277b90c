// Relative-position-bias flash attention with fp32 activations.
//
// The semantics are those of the 16-bit kernels in relpos_attn.hip, and so of
// library/relpos_attention.py of the reference (kernel-rsi):
//   * :46 for the scores;
//   * :26-59 for the forward;
//   * :62-126 and :144-156 for the backward.
// With fp32 activations the reference rounds P and dS to fp32, which is no rounding at
// all (`p.to(v.dtype)`, :53; `ds.to(q.dtype)`, :92, :125), so no product here rounds its operands.
//
// Products of split operands. gfx950 has no reduced-precision fp32 matrix path, and its fp32 matrix
// instructions run at a sixteenth of the bf16 rate. So each fp32 operand is split into three bf16 (8 + 8 + 7
// bits, exact for |x| >= 2^-102 up to bf16's largest, and for zero) and a product is six bf16 MFMAs
// (v_mfma_f32_16x16x32_bf16, fp32 accumulate), the five small ones into an accumulator of their own where
// they are summed apart. What is left out is at most 2^-24 of a product, no more than one fp32 rounding;
// accumulating 32 products per instruction instead of 2 rounds less often, and the measured error
// against 64 bits is below that of fp32 products in every output (2-norm of out / dqkv / dpd at B2 S1024 H16
// D72: 6.9e-7 / 7.8e-7 / 5.3e-7 with fp32 products, 5.3e-7 / 6.1e-7 / 4.0e-7 here; likewise over S 200-2048,
// D 16-128, scores of one dominant product and operands of mixed exponents. At D = 8, whose fp32 sums round
// four times only, it is below for normal operands and 1.2 times for scores of one dominant product).
// Time there, forward / backward: 133 / 432 us with fp32 products, 83 / 253 us here; B4 S2048 H16 D64 612 /
// 2393 -> 414 / 1320, B2 S1024 H16 D128 181 / 615 -> 99 / 450. What bounds it: splitting the staged tiles, P
// and dS takes about as many VALU cycles as the products take matrix cycles, and between the two barriers
// of a step the waves of a SIMD do the former at the same time.
// A workgroup that meets an operand that does not split (infinite, NaN, past bf16's largest, or tiny in a tensor
// that an output is proportional to) computes its tile again with fp32 products
// (v_mfma_f32_32x32x2_f32), below "fp32 products". A tiny element of q or k in the scores is off by 2^-134 at
// most, which moves no score while the other side times |scale| is below 2^100, and is not tested for there
// (testing v alone in the forward instead of k and v: B4 S2048 H16 D64 430 -> 414 us).
//
// Layout (wave64, 16x16 output blocks; see mfma16x16x32 in krsi_device.h):
//   * Workgroup = 8 waves x 16 queries (forward, dQ) or keys (dK/dV), XCD-aware grid. 16 rows per wave keep
//     the resident operand planes (36 registers each at D = 72) and the accumulators within 256
//     registers, so two waves share a SIMD; dK/dV, which holds two operands and two outputs, spills 69-74
//     of them at padded D 80-96 and 179-200 at 112-128. (32 rows per wave: 106 / 315 us at one wave per
//     SIMD, 81 / 365 us with the keys halved between two groups of waves, whose backward spills more.)
//   * Streamed tiles (64 positions x D) are loaded into registers a step ahead, split once by the
//     workgroup and staged in LDS as three bf16 planes, XOR-swizzled so that the 128-bit row reads of
//     the head-dim contractions and the transposed 64-bit reads (ds_read_b64_tr_b16) of the position
//     contractions are both conflict-free.
//   * Scores are computed transposed (S^T = K Q^T) in the forward and dQ: a lane owns one query. Two score
//     blocks' registers hold positions 4 g + {0..3} and 16 + 4 g + {0..3} (g = lane / 16), which is what two
//     transposed reads return, so P and dS are split in place and no register moves between lanes.
//   * The dpd partial rows use the 16-bit kernels' layout (one row of S + 128 diagonals per
//     128-key block), so relpos_dpd_reduce sums them the same way. In the dK/dV kernel the
//     workgroup writes its fp32 dS block [64 queries x 128 keys] to LDS each step, by diagonals. One
//     thread per diagonal then sums that diagonal in query order into a 256-slot ring. Diagonals that
//     can get no further contribution are stored to the partial row. The order is fixed, so
//     dpd is bitwise reproducible.
#include <math.h>

#include "krsi_device.h"
#include "krsi_internal.h"
#include "lds_dma.h"
#include "relpos_common.h"

namespace krsi {
namespace {

constexpr int kRowsF = 128;                 // queries (forward, dQ) or keys (dK/dV) per workgroup
constexpr int kStepF = 64;                  // streamed positions per step
constexpr int kThreadsS = 512;              // threads of a workgroup: 8 waves x 16 rows
constexpr int kThreadsF = 256;              // threads of the fp32 products: 4 waves x 32 rows
constexpr int kWinF = kRowsF + kStepF - 1;  // bias-window entries of one step
static_assert(kRowsF == kKvRows, "the dpd partial rows are shared with the 16-bit kernels");

// (q.k scale + bias) in log2 units, rounded on its own: never fused with the subtraction of the
// running max (forward) or of lse (backward), so both passes form bitwise the same exponent
// argument (at S = 1, p is then exactly 1 in the backward, as in the forward).
__device__ __forceinline__ float log2_units(float t) {
#pragma clang fp contract(off)
  return t * kLog2e;
}

// The dS block of one step by diagonals: entry [x][iq] is query iq and key kk = x + iq - 63 of the block.
// Entries whose key falls outside the block stay zero, so every term of a diagonal sum is a plain
// load (+0 leaves the sum bitwise unchanged). The odd row stride spreads the writes (one query, a run
// of keys) and the reads (one query, 64 diagonals) over the banks.
constexpr int kDiagLd = kStepF + 1;
constexpr int kRing = 256;  // > the 191 diagonals live across two steps
struct KvShared {
  float dsb[kWinF * kDiagLd];
  float ring[kRing];
  float bw[kWinF];
  __attribute__((aligned(16))) float Lq[kStepF];
  __attribute__((aligned(16))) float Dq[kStepF];
};

constexpr int cmax(int a, int b) { return a > b ? a : b; }

// ------------------------------------------------------------- fp32 products
// The path of a workgroup that met a non-finite element (or of row strides past kMaxLdS), on its first
// four waves (32 rows each). Not inlined: the rare path would cost the split loops registers.
//   A operand: lane l holds A[m = l % 32][k = l / 32];
//   B operand: lane l holds B[k = l / 32][n = l % 32].
//   * Head-dim contractions (scores, dP) split D into two halves. Lane half g = l / 32 takes
//     d = g * D/2 + s at step s, for s < D/2, so each lane reads 4 consecutive d with one
//     128-bit load.
//   * Position contractions (P V, dS K, P^T dO, dS^T Q) take one register of the score
//     block per step. The score block's lane l holds positions 8 (r / 4) + 4 g + r % 4 in
//     register r. Step j pairs register j of the B operand with position 8 (j / 4) + 4 g + j % 4
//     of the A operand, so no register is moved between lanes.
//   * Streamed tiles are staged with a row stride of 32 DB + 4 floats, columns [D, 32 DB) zero.
template <int DB>
struct GeoF {
  static constexpr int LD = 32 * DB + 4;  // LDS row stride of a staged tile, floats
  static constexpr int HM = 16 * DB;      // contraction steps per half, at most (D / 2 <= 16 DB)
  static constexpr int TILE = kStepF * LD;
};

__device__ __forceinline__ f32x16 mma(float a, float b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = 0.f;
  return z;
}

// One step's tile rows held in registers between their global loads and their LDS stores, so
// the loads of step t + 1 are in flight while step t computes. Thread t holds 16-byte chunks
// t, t + 256, ... of the tile (at most 2 DB of them: D <= 32 DB). The stored tile holds rows
// p0 .. p0 + 63 of the [S, D] slice at `base` (row stride ld floats), zero past S; columns
// [D, 32 DB) keep what zero_tile_pad wrote. Every load reads a valid address (the last row,
// masked, stands in for rows past S) so none waits behind a branch.
template <int DB>
struct TileRegs {
  static constexpr int CPT = 2 * DB;
  f32x4 v[CPT];
  __device__ __forceinline__ void load(const float* base, int64_t ld, int p0, int S, int D) {
    const int cpr = D >> 2, n = kStepF * cpr;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int c = min((int)threadIdx.x + k * kThreadsF, n - 1);
      const int r = c / cpr, j = c - r * cpr;
      const bool ok = (int)threadIdx.x + k * kThreadsF < n && p0 + r < S;
      const int row = p0 + r < S ? p0 + r : S - 1;
      f32x4 x = *reinterpret_cast<const f32x4*>(base + (int64_t)row * ld + 4 * j);
      if (!ok) x = f32x4{0.f, 0.f, 0.f, 0.f};
      v[k] = x;
    }
  }
  __device__ __forceinline__ void store(float* tile, int D) const {
    const int cpr = D >> 2, n = kStepF * cpr;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int c = threadIdx.x + k * kThreadsF;
      if (c < n) {
        const int r = c / cpr, j = c - r * cpr;
        *reinterpret_cast<f32x4*>(tile + r * GeoF<DB>::LD + 4 * j) = v[k];
      }
    }
  }
};

// Bias window entry x = threadIdx.x (x < kWinF): pd[h, wb + x], zero outside [0, 2S - 1), loaded
// into a register one step ahead.
__device__ __forceinline__ float window_entry(const float* pdh, int npd, int wb) {
  const int k = wb + (int)threadIdx.x;
  return (threadIdx.x < (unsigned)kWinF && k >= 0 && k < npd) ? pdh[k] : 0.f;
}
__device__ __forceinline__ void store_window(float* bw, float v) {
  if (threadIdx.x < (unsigned)kWinF) bw[threadIdx.x] = v;
}

template <int DB>
__device__ __forceinline__ void zero_tile_pad(float* tile, int D) {
  constexpr int LD = GeoF<DB>::LD;
  const int w = LD - D;
  for (int c = threadIdx.x; c < kStepF * w; c += kThreadsF) {
    const int r = c / w;
    tile[r * LD + D + (c - r * w)] = 0.f;
  }
}

// The lane's half of a row of D floats into registers: dst[s] = row[s] for s < ns = D / 2
// (row points at column g D/2), zero past ns or when !ok.
template <int DB>
__device__ __forceinline__ void load_half_row(float* dst, const float* row, int ns, bool ok) {
#pragma unroll
  for (int s = 0; s < GeoF<DB>::HM; s += 4) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (ok && s < ns) v = *reinterpret_cast<const f32x4*>(row + s);
#pragma unroll
    for (int e = 0; e < 4; ++e) dst[s + e] = v[e];
  }
}

// Head-dim contraction: acc += A B with A's row m = row `row0 + l32` of a staged tile and
// B's column n = the lane's register half `breg`.
template <int DB>
__device__ __forceinline__ f32x16 dot_rows(const float* tile, int row, int g, int ns, const float* breg,
                                           f32x16 acc) {
  const float* a = tile + row * GeoF<DB>::LD + g * ns;
#pragma unroll
  for (int s = 0; s < GeoF<DB>::HM; s += 4) {
    if (s < ns) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(a + s);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = mma(v[e], breg[s + e], acc);
    }
  }
  return acc;
}

// Position contraction: acc[db] += sum over the 32 positions base + 8 (j / 4) + 4 g + j % 4 of
// tile[position][32 db + l32] * b[j]: output rows are head dims, columns the lane's own.
template <int DB>
__device__ __forceinline__ void dot_positions(const float* tile, int base, int g, int l32,
                                              const f32x16& b, f32x16* acc) {
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const float* rowp = tile + (base + 8 * (j >> 2) + 4 * g + (j & 3)) * GeoF<DB>::LD + l32;
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[db] = mma(rowp[32 * db], b[j], acc[db]);
  }
}

// Store a 32x32-block accumulator column (head dims 32 db + 8 a + 4 g .. + 3 of this lane's
// position) times `mul` to row `dst` (16-byte aligned, D % 8 == 0).
template <int DB>
__device__ __forceinline__ void store_dims(float* dst, const f32x16* acc, float mul, int g, int D) {
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int d0 = 32 * db + 8 * a + 4 * g;
      if (d0 < D) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[db][4 * a + e] * mul;
        *reinterpret_cast<f32x4*>(dst + d0) = v;
      }
    }
}

template <int DP>
__device__ __noinline__ void fwd_fp32(float* Ks, float* Vs, float* bw, const float* qkv, int64_t ld, const float* pd,
                                         float* out, float* out32, float* lse, int S, int H, int D, float scale) {
  constexpr int DB = (DP + 31) / 32;
  using G = GeoF<DB>;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 5, l32 = lane & 31;
  const int nqb = (S + kRowsF - 1) / kRowsF;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int bh = tile / nqb, b = bh / H, h = bh - b * H;
  const int i_wg = (tile - bh * nqb) * kRowsF;
  const int ii = wave * 32 + l32, qi = i_wg + ii;
  const bool qvalid = qi < S;
  const int ns = D >> 1;
  const int64_t HD = (int64_t)H * D;
  const float* q0 = qkv + (int64_t)b * S * ld + (int64_t)h * D;
  const int npd = 2 * S - 1;
  const float* pdh = pd + (int64_t)h * npd;

  float qr[G::HM];
  load_half_row<DB>(qr, q0 + (int64_t)(qvalid ? qi : 0) * ld + g * ns, ns, qvalid);
  zero_tile_pad<DB>(Ks, D);
  zero_tile_pad<DB>(Vs, D);
  f32x16 oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) oacc[db] = zero16();
  // The most negative finite float, not -inf: a step whose scores are all -inf (keys masked by
  // -inf bias entries) gives p = 0, not exp2(-inf - -inf) = NaN.
  float m_run = -3.40282347e+38f, l_run = 0.f;

  const int T = (S + kStepF - 1) / kStepF;
  const int wb0 = -i_wg - (kRowsF - 1) + S - 1;
  TileRegs<DB> kn, vn;
  kn.load(q0 + HD, ld, 0, S, D);
  vn.load(q0 + 2 * HD, ld, 0, S, D);
  float wn = window_entry(pdh, npd, wb0);
  for (int t = 0; t < T; ++t) {
    const int j0 = t * kStepF;
    __syncthreads();  // every wave is done with the previous step's tiles
    kn.store(Ks, D);
    vn.store(Vs, D);
    store_window(bw, wn);
    __syncthreads();
    if (t + 1 < T) {  // step t + 1's loads, in flight while step t computes
      kn.load(q0 + HD, ld, j0 + kStepF, S, D);
      vn.load(q0 + 2 * HD, ld, j0 + kStepF, S, D);
      wn = window_entry(pdh, npd, wb0 + j0 + kStepF);
    }
    // Scores in log2 units, (q.k scale + bias) log2(e), keys past S at -inf; exact running max.
    f32x16 sc[2];
    float mx = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      sc[kb] = dot_rows<DB>(Ks, kb * 32 + l32, g, ns, qr, zero16());
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int jj = kb * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
        // The window entry (index in [0, kWinF)) is read for every key, so the read does not
        // wait behind the key test; keys past S then take -inf.
        const float xv = log2_units(fmaf(sc[kb][r], scale, bw[jj - ii + kRowsF - 1]));
        const float x = j0 + jj < S ? xv : -INFINITY;
        sc[kb][r] = x;
        mx = fmaxf(mx, x);
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m_run, mx);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    l_run *= alpha;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
    m_run = m_new;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = __builtin_amdgcn_exp2f(sc[kb][r] - m_new);
        sc[kb][r] = p;
        l_run += p;
      }
      dot_positions<DB>(Vs, kb * 32, g, l32, sc[kb], oacc);
    }
  }
  const float l = l_run + __shfl_xor(l_run, 32);
  if (qvalid) {
    const int64_t ob = ((int64_t)b * S + qi) * HD + (int64_t)h * D;
    store_dims<DB>(out + ob, oacc, 1.f / l, g, D);
    if (out32 && out32 != out) store_dims<DB>(out32 + ob, oacc, 1.f / l, g, D);
    if (g == 0 && lse) lse[(int64_t)bh * S + qi] = m_run + log2f(l);
  }
}

template <int DP>
__device__ __noinline__ void dq_fp32(float* Ks, float* Vs, float* bw, const float* qkv, int64_t ld, const float* pd,
                                        const float* dout, const float* out32, const float* lse, float* delta_ws,
                                        float* dqkv, int64_t ldd, int S, int H, int D, float scale) {
  constexpr int DB = (DP + 31) / 32;
  using G = GeoF<DB>;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 5, l32 = lane & 31;
  const int nqb = (S + kRowsF - 1) / kRowsF;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int bh = tile / nqb, b = bh / H, h = bh - b * H;
  const int i_wg = (tile - bh * nqb) * kRowsF;
  const int ii = wave * 32 + l32, qi = i_wg + ii;
  const bool qvalid = qi < S;
  const int ns = D >> 1;
  const int64_t HD = (int64_t)H * D;
  const float* q0 = qkv + (int64_t)b * S * ld + (int64_t)h * D;
  const int npd = 2 * S - 1;
  const float* pdh = pd + (int64_t)h * npd;

  float qr[G::HM], dr[G::HM];
  const int qs = qvalid ? qi : 0;
  load_half_row<DB>(qr, q0 + (int64_t)qs * ld + g * ns, ns, qvalid);
  const int64_t ob = ((int64_t)b * S + qs) * HD + (int64_t)h * D + g * ns;
  load_half_row<DB>(dr, dout + ob, ns, qvalid);
  float delta;
  {
    float o[G::HM];
    load_half_row<DB>(o, out32 + ob, ns, qvalid);
    float part = 0.f;
#pragma unroll
    for (int s = 0; s < G::HM; ++s) part = fmaf(dr[s], o[s], part);
    delta = part + __shfl_xor(part, 32);
  }
  if (qvalid && g == 0) delta_ws[(int64_t)bh * S + qi] = delta;
  // +inf makes p = exp2(x - lse) exactly 0 on query lanes past S.
  const float nlse = qvalid ? lse[(int64_t)bh * S + qi] : INFINITY;
  zero_tile_pad<DB>(Ks, D);
  zero_tile_pad<DB>(Vs, D);
  f32x16 dq[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dq[db] = zero16();

  const int T = (S + kStepF - 1) / kStepF;
  const int wb0 = -i_wg - (kRowsF - 1) + S - 1;
  TileRegs<DB> kn, vn;
  kn.load(q0 + HD, ld, 0, S, D);
  vn.load(q0 + 2 * HD, ld, 0, S, D);
  float wn = window_entry(pdh, npd, wb0);
  for (int t = 0; t < T; ++t) {
    const int j0 = t * kStepF;
    __syncthreads();
    kn.store(Ks, D);
    vn.store(Vs, D);
    store_window(bw, wn);
    __syncthreads();
    if (t + 1 < T) {
      kn.load(q0 + HD, ld, j0 + kStepF, S, D);
      vn.load(q0 + 2 * HD, ld, j0 + kStepF, S, D);
      wn = window_entry(pdh, npd, wb0 + j0 + kStepF);
    }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      f32x16 s = dot_rows<DB>(Ks, kb * 32 + l32, g, ns, qr, zero16());
      const f32x16 dp = dot_rows<DB>(Vs, kb * 32 + l32, g, ns, dr, zero16());
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int jj = kb * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
        // Computed for every key (the window read and exp2 do not wait behind the key test;
        // keys past S have zero K rows and window entries, so the value is finite) and then
        // dropped past S.
        const float pv = __builtin_amdgcn_exp2f(log2_units(fmaf(s[r], scale, bw[jj - ii + kRowsF - 1])) - nlse);
        const float p = j0 + jj < S ? pv : 0.f;
        s[r] = p * (dp[r] - delta);  // ds
      }
      dot_positions<DB>(Ks, kb * 32, g, l32, s, dq);
    }
  }
  if (qvalid) store_dims<DB>(dqkv + ((int64_t)b * S + qi) * ldd + (int64_t)h * D, dq, scale, g, D);
}

template <int DP>
__device__ __noinline__ void dkdv_fp32(float* Qs, float* Os, KvShared& sh, const float* qkv, int64_t ld,
                                          const float* pd, const float* dout, const float* lse, const float* delta_ws,
                                          float* dqkv, int64_t ldd, float* part, int S, int H, int D, float scale,
                                          int kb0, int nkc) {
  constexpr int DB = (DP + 31) / 32;
  using G = GeoF<DB>;
  float *const dsb = sh.dsb, *const ring = sh.ring, *const bw = sh.bw, *const Lq = sh.Lq, *const Dq = sh.Dq;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 5, l32 = lane & 31;
  // Key blocks [kb0, kb0 + nkc) of every (batch, head).
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int bh = tile / nkc, b = bh / H, h = bh - b * H;
  const int kbl = tile - bh * nkc;
  const int j_wg = (kb0 + kbl) * kRowsF;
  const int kk = wave * 32 + l32, kj = j_wg + kk;
  const bool kvalid = kj < S;
  const int ns = D >> 1;
  const int64_t HD = (int64_t)H * D;
  const float* q0 = qkv + (int64_t)b * S * ld + (int64_t)h * D;
  const float* o0 = dout + (int64_t)b * S * HD + (int64_t)h * D;
  const int npd = 2 * S - 1;
  const float* pdh = pd + (int64_t)h * npd;
  const float* lse_bh = lse + (int64_t)bh * S;
  const float* dl_bh = delta_ws + (int64_t)bh * S;
  float* prow = part + ((int64_t)bh * nkc + kbl) * (S + kRowsF);
  const int rlen = S + kRowsF - 1;  // diagonals of the partial row

  float kr[G::HM], vr[G::HM];
  const int64_t krow = (int64_t)(kvalid ? kj : 0) * ld + g * ns;
  load_half_row<DB>(kr, q0 + HD + krow, ns, kvalid);
  load_half_row<DB>(vr, q0 + 2 * HD + krow, ns, kvalid);
  zero_tile_pad<DB>(Qs, D);
  zero_tile_pad<DB>(Os, D);
  for (int e = tid; e < kRing; e += kThreadsF) ring[e] = 0.f;
  for (int e = tid; e < kWinF * kDiagLd; e += kThreadsF) dsb[e] = 0.f;
  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dk[db] = dv[db] = zero16();

  const int T = (S + kStepF - 1) / kStepF;
  // Window entry x = kk - iq + 63 holds pd[h, (j_wg + kk) - (i0 + iq) + S - 1].
  const int wb0 = j_wg - (kStepF - 1) + S - 1;
  TileRegs<DB> qn, on;
  qn.load(q0, ld, 0, S, D);
  on.load(o0, HD, 0, S, D);
  float wn = window_entry(pdh, npd, wb0);
  float ln = 0.f, dn = 0.f;  // lse and delta of query tid (threads tid < 64)
  auto stats = [&](int i0) {
    const int q = min(i0 + tid, S - 1);
    ln = lse_bh[q];
    dn = dl_bh[q];
  };
  stats(0);
  for (int t = 0; t < T; ++t) {
    const int i0 = t * kStepF;
    __syncthreads();
    qn.store(Qs, D);
    on.store(Os, D);
    store_window(bw, wn);
    if (tid < kStepF) {
      const bool ok = i0 + tid < S;
      Lq[tid] = ok ? ln : INFINITY;  // queries past S: p = 0
      Dq[tid] = ok ? dn : 0.f;
    }
    __syncthreads();
    if (t + 1 < T) {
      qn.load(q0, ld, i0 + kStepF, S, D);
      on.load(o0, HD, i0 + kStepF, S, D);
      wn = window_entry(pdh, npd, wb0 - i0 - kStepF);
      stats(i0 + kStepF);
    }
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      // S and dP [query][key]: rows are this step's queries, columns the lane's key.
      f32x16 p = dot_rows<DB>(Qs, qb * 32 + l32, g, ns, kr, zero16());
      f32x16 ds = dot_rows<DB>(Os, qb * 32 + l32, g, ns, vr, zero16());
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int iq = qb * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
        const float pv = __builtin_amdgcn_exp2f(log2_units(fmaf(p[r], scale, bw[kk - iq + kStepF - 1])) - Lq[iq]);
        // Keys past S have p != 0 (their bias is real) but no gradient: their dK and dV are
        // never stored and their dS is kept out of dpd.
        const float dd = Dq[iq];  // read for every lane, so it does not wait behind kvalid
        const float dsv = kvalid ? pv * (ds[r] - dd) : 0.f;
        p[r] = pv;
        ds[r] = dsv;
        dsb[(kk - iq + kStepF - 1) * kDiagLd + iq] = dsv;
      }
      dot_positions<DB>(Os, qb * 32, g, l32, p, dv);   // dV^T += dO^T P
      dot_positions<DB>(Qs, qb * 32, g, l32, ds, dk);  // dK^T += Q^T dS
    }
    __syncthreads();
    // Local diagonal x = kk - iq + 63 of this step is partial-row entry R = x - 64 - i0 + S.
    if (tid < kWinF) {
      float acc = 0.f;
#pragma unroll 16
      for (int iq = 0; iq < kStepF; ++iq) acc += dsb[tid * kDiagLd + iq];
      const int R = tid - kStepF - i0 + S;
      if (R >= 0) ring[R & (kRing - 1)] += acc;
    }
    __syncthreads();
    // Later steps reach R <= S + 62 - i0 only: entries [S + 63 - i0, S + 126 - i0] are final.
    if (tid < kStepF) {
      const int R = S + (kStepF - 1) - i0 + tid;
      if (R >= 0 && R < rlen) {
        prow[R] = ring[R & (kRing - 1)];
        ring[R & (kRing - 1)] = 0.f;
      }
    }
  }
  __syncthreads();
  const int rmax = S + kStepF - 2 - kStepF * (T - 1);  // the rest: [0, rmax]
  for (int R = tid; R <= rmax; R += kThreadsF)
    if (R < rlen) prow[R] = ring[R & (kRing - 1)];

  if (kvalid) {
    float* row = dqkv + ((int64_t)b * S + kj) * ldd + (int64_t)h * D;
    store_dims<DB>(row + HD, dk, scale, g, D);
    store_dims<DB>(row + 2 * HD, dv, 1.f, g, D);
  }
}

// ------------------------------------------------------------ split products
// An fp32 value as three bf16: the nearest one, the nearest one to the rest, what is left (at most 7 bits).
// The sum is exact unless that last part is subnormal, so for every |x| >= 2^-102 up to bf16's largest;
// of a larger or non-finite x the parts are infinite or NaN. tiny, if given, is set by a subnormal last part.
__device__ __forceinline__ void split3(float x, float y, uint32_t* p, bool* tiny = nullptr) {
  p[0] = pack_bf16x2(x, y);
  float rx = x - bf_lo(p[0]), ry = y - bf_hi(p[0]);
  p[1] = pack_bf16x2(rx, ry);
  rx -= bf_lo(p[1]);
  ry -= bf_hi(p[1]);
  p[2] = pack_bf16x2(rx, ry);
  constexpr int kSubnormal = 0x090;  // v_cmp_class: negative and positive subnormals
  if (tiny) *tiny |= __builtin_amdgcn_classf(rx, kSubnormal) | __builtin_amdgcn_classf(ry, kSubnormal);
}
// Eight values as the three planes of one MFMA operand.
__device__ __forceinline__ void split8(const f32x4& lo, const f32x4& hi, u32x4* planes, bool* tiny = nullptr) {
  uint32_t p[4][3];
  split3(lo[0], lo[1], p[0], tiny);
  split3(lo[2], lo[3], p[1], tiny);
  split3(hi[0], hi[1], p[2], tiny);
  split3(hi[2], hi[3], p[3], tiny);
#pragma unroll
  for (int k = 0; k < 3; ++k) planes[k] = u32x4{p[0][k], p[1][k], p[2][k], p[3][k]};
}
// P and dS are split times 2^32, which comes off their sums: every normal P (2^-126 and up; exp2 gives no
// subnormals) then splits exactly, with no test that an unlikely key would fail.
constexpr float kUp = 0x1p32f, kDown = 0x1p-32f;

// The six partial products that matter: five small ones, then the large one (plane 0 x 0, at the
// callers). Those left out (planes 1 x 2, 2 x 1 and 2 x 2) come to 2^-24 of the product at most (measured over
// random mantissas 2^-24.1, rms 5.3e-9; one fp32 rounding: 2^-24, 2.5e-8), of either sign. FLIP
// exchanges the roles of a and b, so that q k^T and k q^T add the same terms in the same order. N chains at
// once: each product waits for the one before it in its chain, so two chains in turn hide that.
template <bool FLIP, int N>
__device__ __forceinline__ void mma_small(const u32x4 (*a)[3], const u32x4* b, f32x4* c) {
  constexpr int ia[5] = {FLIP ? 0 : 2, FLIP ? 2 : 0, 1, FLIP ? 0 : 1, FLIP ? 1 : 0};
  constexpr int ib[5] = {FLIP ? 2 : 0, FLIP ? 0 : 2, 1, FLIP ? 1 : 0, FLIP ? 0 : 1};
#pragma unroll
  for (int i = 0; i < 5; ++i)
#pragma unroll
    for (int n = 0; n < N; ++n) c[n] = mfma16x16x32(a[n][ia[i]], b[ib[i]], c[n]);
}

// One step's tile rows of a thread, between their global loads and their LDS stores (the loads of step
// t + 1 are in flight while step t computes): 16-byte chunks t, t + 512, ... of the tile. off: their
// byte offsets from the tile's first row; the buffer resource ends at the last row of the slice, so rows
// past S read as zero with no per-step test. Offsets are opaque: the range check is made on the
// register, so no constant may be split off into the instruction's immediate field.
template <int DP>
struct Chunks {
  static constexpr int CPT = (kStepF * DP / 4 + kThreadsS - 1) / kThreadsS;
  // Chunk k is inside the tile for every thread, whatever D in (DP - 16, DP].
  static constexpr bool whole(int k) { return (k + 1) * kThreadsS <= kStepF * (DP - 8) / 4; }
  uint32_t off[CPT];
  __device__ __forceinline__ void init(int64_t ld, int D) {
    const int cpr = D >> 2;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int c = threadIdx.x + k * kThreadsS, r = c / cpr, j = c - r * cpr;
      off[k] = opaque(whole(k) || r < kStepF ? (uint32_t)(r * (int)ld + 4 * j) * 4u : 0x80000000u);
    }
  }
  __device__ __forceinline__ void load(f32x4* v, const float* base, int64_t ld, int p0, int S, int D) const {
    const int rows = min(S - p0, kStepF);
    const rsrc_t r = make_rsrc(base + (int64_t)p0 * ld, (uint32_t)(((rows - 1) * (int)ld + D) * 4));
#pragma unroll
    for (int k = 0; k < CPT; ++k)
      v[k] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off[k], 0, 0));
  }
};
// Row strides whose 64-row tiles such offsets span; beyond, fp32 products.
constexpr int64_t kMaxLdS = (int64_t(1) << 31) / (4 * kStepF) - 256;

// Staged tiles: three planes of 64 rows x 32 KS bf16 (zero past D), swizzled as LaneOffsets16 reads them.
template <int DP>
struct Planes {
  static constexpr int KS = (DP + 31) / 32;  // 32-wide steps of the head-dim contractions
  static constexpr int CB = DP / 16;         // 16-wide blocks of the head-dim outputs
  static constexpr int LD = 32 * KS;         // row stride, elements
  static constexpr int PL = kStepF * LD;     // elements of a plane
  static constexpr int BYTES = 3 * PL * 2;
  using Lanes = LaneOffsets16<LD, KS, CB>;
  static __device__ __forceinline__ int off(int r, int j) { return Lanes::off(r, j); }
  // Columns [D, LD) of every plane, zero for the kernel's life.
  static __device__ __forceinline__ void zero_pad(uint16_t* t, int D) {
    const int first = D >> 3, w = LD / 8 - first;
    for (int c = threadIdx.x; c < kStepF * w; c += kThreadsS) {
      const int r = c / w, j = first + (c - r * w);
#pragma unroll
      for (int k = 0; k < 3; ++k) *reinterpret_cast<u32x4*>(t + k * PL + off(r, j)) = u32x4{0u, 0u, 0u, 0u};
    }
  }
  // The rows a thread holds, split, into the tile.
  static __device__ __forceinline__ void store(uint16_t* t, const f32x4* v, int D, bool* tiny = nullptr) {
    const int cpr = D >> 2, n = kStepF * cpr;
#pragma unroll
    for (int k = 0; k < Chunks<DP>::CPT; ++k) {
      const int c = threadIdx.x + k * kThreadsS;
      if (Chunks<DP>::whole(k) || c < n) {
        const int r = c / cpr, j = c - r * cpr;
        uint32_t lo[3], hi[3];
        split3(v[k][0], v[k][1], lo, tiny);
        split3(v[k][2], v[k][3], hi, tiny);
#pragma unroll
        for (int q = 0; q < 3; ++q)
          *reinterpret_cast<uint2*>(t + q * PL + off(r, j >> 1) + 4 * (j & 1)) = make_uint2(lo[q], hi[q]);
      }
    }
  }
};

template <int DP>
using LaneOff = typename Planes<DP>::Lanes;

// The lane's row of D floats as operand planes: columns 32 s + 8 g .. + 7 at step s, zero past D or
// when !ok (every lane loads, from column 0 where it has none). dot, if given, takes the lane's
// share of the row's dot product with row o.
template <int DP>
__device__ __forceinline__ void load_row(u32x4 (*dst)[3], const float* row, int g, int D, bool ok,
                                         bool* tiny = nullptr, const float* o = nullptr, float* dot = nullptr) {
#pragma unroll
  for (int s = 0; s < Planes<DP>::KS; ++s) {
    const int d = 32 * s + 8 * g;
    const bool in = ok && d < D;
    const float* p = row + (in ? d : 0);
    f32x4 f[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(p + 4 * e);
#pragma unroll
      for (int i = 0; i < 4; ++i) f[e][i] = in ? v[i] : 0.f;
    }
    if (dot) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(o + (in ? d : 0) + 4 * e);
#pragma unroll
        for (int i = 0; i < 4; ++i) *dot = fmaf(f[e][i], in ? v[i] : 0.f, *dot);
      }
    }
    split8(f[0], f[1], dst[s], tiny);
  }
}

// Head-dim contractions of two row blocks: out[n] = the tile's rows 16 (blk + n) + l % 16 against the lane's
// resident row. The small products are summed apart, so the large ones round KS times only, and
// the one sum of D <= 32 starts from theirs.
template <int DP, bool FLIP>
__device__ __forceinline__ void dot_row_blocks(const uint16_t* t, const LaneOff<DP>& L, int blk, const u32x4 (*b)[3],
                                               f32x4* out) {
  using P = Planes<DP>;
  f32x4 lo[2];
#pragma unroll
  for (int n = 0; n < 2; ++n) lo[n] = out[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < P::KS; ++s) {
    u32x4 a[2][3];
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int k = 0; k < 3; ++k)
        a[n][k] = *reinterpret_cast<const u32x4*>(t + k * P::PL + 16 * (blk + n) * P::LD + L.row[s]);
    mma_small<FLIP, 2>(a, b[s], lo);
#pragma unroll
    for (int n = 0; n < 2; ++n) out[n] = mfma16x16x32(a[n][0], b[s][0], P::KS == 1 ? lo[n] : out[n]);
  }
  if constexpr (P::KS > 1) {
#pragma unroll
    for (int n = 0; n < 2; ++n) out[n] += lo[n];
  }
}

// Position contraction over 32 positions (score blocks 2 half and 2 half + 1, v0 and v1, split here):
// acc[c] += tile[position][16 c + l16] * v[position].
template <int DP, int N>
__device__ __forceinline__ void dot_positions_cols(const uint16_t* t, const LaneOff<DP>& L, int c, const u32x4* b,
                                                   f32x4* acc) {
  using P = Planes<DP>;
  u32x4 a[N][3];
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const uint16_t* p = t + k * P::PL + L.tr[c + n];
      const uint2 x = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
      const uint2 y = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 16 * P::LD)));
      a[n][k] = u32x4{x.x, x.y, y.x, y.y};
    }
  mma_small<false, N>(a, b, acc + c);
#pragma unroll
  for (int n = 0; n < N; ++n) acc[c + n] = mfma16x16x32(a[n][0], b[0], acc[c + n]);
}
template <int DP>
__device__ __forceinline__ void dot_positions_half(const uint16_t* t, const LaneOff<DP>& L, int half, const f32x4& v0,
                                                   const f32x4& v1, f32x4* acc) {
  constexpr int CB = Planes<DP>::CB;
  u32x4 b[3];
  split8(v0, v1, b);
#pragma unroll
  for (int c = 0; c + 1 < CB; c += 2) dot_positions_cols<DP, 2>(t + 32 * half * Planes<DP>::LD, L, c, b, acc);
  if constexpr (CB % 2) dot_positions_cols<DP, 1>(t + 32 * half * Planes<DP>::LD, L, CB - 1, b, acc);
}

// acc (head dims 16 c + 4 g .. + 3 of this lane's row) times kDown mul to row dst (16-byte aligned).
template <int DP>
__device__ __forceinline__ void store_row(float* dst, const f32x4* acc, float mul, int g, int D) {
#pragma unroll
  for (int c = 0; c < Planes<DP>::CB; ++c) {
    const int d = 16 * c + 4 * g;
    if (d < D) *reinterpret_cast<f32x4*>(dst + d) = acc[c] * kDown * mul;
  }
}
template <int DP>
__device__ __forceinline__ void zero_acc(f32x4* acc) {
#pragma unroll
  for (int c = 0; c < Planes<DP>::CB; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
}
// Whether one of the lane's sums is not finite: some operand was not (every output sum of a row or column
// has a product with each of its P or dS, which have one with each input), or kUp took it past fp32's range.
template <int DP>
__device__ __forceinline__ bool overflowed(const f32x4* acc) {
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < Planes<DP>::CB; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) s = fmaf(acc[c][r], 0.f, s);
  return s != s;
}
// Sum and max over the four lanes (g = 0..3) that share a row.
__device__ __forceinline__ float row_sum(float v) {
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}
__device__ __forceinline__ float row_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16));
  return fmaxf(v, __shfl_xor(v, 32));
}
// The barriers of a loop that the workgroup's first four waves run alone.
__device__ __forceinline__ void barriers(int n) {
  for (int i = 0; i < n; ++i) __syncthreads();
}

// LDS of one staged tile, for either kind of products.
template <int DP>
constexpr int kTileBytes = cmax(Planes<DP>::BYTES, GeoF<(DP + 31) / 32>::TILE * 4);

// -------------------------------------------------------------------- forward
template <int DP>
__global__ __launch_bounds__(kThreadsS, 2) void relpos_fwd_f32_kernel(
    const float* __restrict__ qkv, int64_t ld, const float* __restrict__ pd, float* __restrict__ out,
    float* __restrict__ out32, float* __restrict__ lse, int S, int H, int D, float scale) {
  __shared__ __attribute__((aligned(256))) unsigned char tiles[2 * kTileBytes<DP>];
  __shared__ float bw[kWinF];
  uint16_t* const Ks = reinterpret_cast<uint16_t*>(tiles);
  uint16_t* const Vs = reinterpret_cast<uint16_t*>(tiles + kTileBytes<DP>);

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4,
            l16 = lane & 15;
  const int nqb = (S + kRowsF - 1) / kRowsF;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int bh = tile / nqb, b = bh / H, h = bh - b * H;
  const int i_wg = (tile - bh * nqb) * kRowsF;
  const int ii = wave * 16 + l16, qi = i_wg + ii;
  const bool qvalid = qi < S;
  const int64_t HD = (int64_t)H * D;
  const float* q0 = qkv + (int64_t)b * S * ld + (int64_t)h * D;
  const int npd = 2 * S - 1;
  const float* pdh = pd + (int64_t)h * npd;
  LaneOff<DP> L;
  L.init(g, l16);

  bool tiny = false;
  u32x4 qr[Planes<DP>::KS][3];
  load_row<DP>(qr, q0 + (int64_t)(qvalid ? qi : 0) * ld, g, D, qvalid);
  Planes<DP>::zero_pad(Ks, D);
  Planes<DP>::zero_pad(Vs, D);
  f32x4 oacc[Planes<DP>::CB];
  zero_acc<DP>(oacc);
  // The most negative finite float, not -inf: a step whose scores are all -inf (keys masked by
  // -inf bias entries) gives p = 0, not exp2(-inf - -inf) = NaN.
  float m_run = -3.40282347e+38f, l_run = 0.f;

  const bool narrow = ld <= kMaxLdS;
  const int T = narrow ? (S + kStepF - 1) / kStepF : 0;
  const int wb0 = -i_wg - (kRowsF - 1) + S - 1;
  Chunks<DP> ch;
  ch.init(ld, D);
  f32x4 kn[Chunks<DP>::CPT], vn[Chunks<DP>::CPT];
  if (T) {
    ch.load(kn, q0 + HD, ld, 0, S, D);
    ch.load(vn, q0 + 2 * HD, ld, 0, S, D);
  }
  float wn = window_entry(pdh, npd, wb0);
  for (int t = 0; t < T; ++t) {
    const int j0 = t * kStepF;
    __syncthreads();  // every wave is done with the previous step's tiles
    Planes<DP>::store(Ks, kn, D);
    Planes<DP>::store(Vs, vn, D, &tiny);
    store_window(bw, wn);
    __syncthreads();
    if (t + 1 < T) {  // step t + 1's loads, in flight while step t computes
      ch.load(kn, q0 + HD, ld, j0 + kStepF, S, D);
      ch.load(vn, q0 + 2 * HD, ld, j0 + kStepF, S, D);
      wn = window_entry(pdh, npd, wb0 + j0 + kStepF);
    }
    // Scores in log2 units, (q.k scale + bias) log2(e), keys past S at -inf; exact running max.
    f32x4 sc[4];
    const float* bk = bw + (4 * g - ii + kRowsF - 1);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      if (kb % 2 == 0) dot_row_blocks<DP, false>(Ks, L, kb, qr, sc + kb);
#pragma unroll
      for (int r = 0; r < 4; ++r) sc[kb][r] = log2_units(fmaf(sc[kb][r], scale, bk[16 * kb + r]));
    }
    if (j0 + kStepF > S) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (j0 + 16 * kb + 4 * g + r >= S) sc[kb][r] = -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, sc[kb][r]);
    const float m_new = fmaxf(m_run, row_max(mx));
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    l_run *= alpha;
#pragma unroll
    for (int c = 0; c < Planes<DP>::CB; ++c) oacc[c] *= alpha;
    m_run = m_new;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int kb = 2 * half; kb < 2 * half + 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sc[kb][r] = __builtin_amdgcn_exp2f(sc[kb][r] - m_new);
          l_run += sc[kb][r];
          sc[kb][r] *= kUp;
        }
      dot_positions_half<DP>(Vs, L, half, sc[2 * half], sc[2 * half + 1], oacc);
    }
  }
  if (__syncthreads_or(!narrow || tiny || overflowed<DP>(oacc))) {
    if (wave < 4)
      fwd_fp32<DP>(reinterpret_cast<float*>(Ks), reinterpret_cast<float*>(Vs), bw, qkv, ld, pd, out, out32, lse, S, H,
                   D, scale);
    else
      barriers(2 * ((S + kStepF - 1) / kStepF));
    return;
  }
  const float l = row_sum(l_run);
  if (qvalid) {
    const int64_t ob = ((int64_t)b * S + qi) * HD + (int64_t)h * D;
    store_row<DP>(out + ob, oacc, 1.f / l, g, D);
    if (out32 && out32 != out) store_row<DP>(out32 + ob, oacc, 1.f / l, g, D);
    if (g == 0 && lse) lse[(int64_t)bh * S + qi] = m_run + log2f(l);
  }
}

// --------------------------------------------------------- backward: delta and dQ
template <int DP>
__global__ __launch_bounds__(kThreadsS, 2) void relpos_bwd_dq_f32_kernel(
    const float* __restrict__ qkv, int64_t ld, const float* __restrict__ pd,
    const float* __restrict__ dout, const float* __restrict__ out32, const float* __restrict__ lse,
    float* __restrict__ delta_ws, float* __restrict__ dqkv, int64_t ldd, int S, int H, int D,
    float scale) {
  __shared__ __attribute__((aligned(256))) unsigned char tiles[2 * kTileBytes<DP>];
  __shared__ float bw[kWinF];
  uint16_t* const Ks = reinterpret_cast<uint16_t*>(tiles);
  uint16_t* const Vs = reinterpret_cast<uint16_t*>(tiles + kTileBytes<DP>);

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4,
            l16 = lane & 15;
  const int nqb = (S + kRowsF - 1) / kRowsF;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int bh = tile / nqb, b = bh / H, h = bh - b * H;
  const int i_wg = (tile - bh * nqb) * kRowsF;
  const int ii = wave * 16 + l16, qi = i_wg + ii;
  const bool qvalid = qi < S;
  const int64_t HD = (int64_t)H * D;
  const float* q0 = qkv + (int64_t)b * S * ld + (int64_t)h * D;
  const int npd = 2 * S - 1;
  const float* pdh = pd + (int64_t)h * npd;
  LaneOff<DP> L;
  L.init(g, l16);

  bool tiny = false;
  float part = 0.f;
  u32x4 qr[Planes<DP>::KS][3], dr[Planes<DP>::KS][3];
  const int qs = qvalid ? qi : 0;
  const int64_t ob = ((int64_t)b * S + qs) * HD + (int64_t)h * D;
  load_row<DP>(qr, q0 + (int64_t)qs * ld, g, D, qvalid);
  load_row<DP>(dr, dout + ob, g, D, qvalid, &tiny, out32 + ob, &part);
  const float delta = row_sum(part);
  // +inf makes p = exp2(x - lse) exactly 0 on query lanes past S.
  const float nlse = qvalid ? lse[(int64_t)bh * S + qi] : INFINITY;
  Planes<DP>::zero_pad(Ks, D);
  Planes<DP>::zero_pad(Vs, D);
  f32x4 dq[Planes<DP>::CB];
  zero_acc<DP>(dq);

  const bool narrow = ld <= kMaxLdS;
  const int T = narrow ? (S + kStepF - 1) / kStepF : 0;
  const int wb0 = -i_wg - (kRowsF - 1) + S - 1;
  Chunks<DP> ch;
  ch.init(ld, D);
  f32x4 kn[Chunks<DP>::CPT], vn[Chunks<DP>::CPT];
  if (T) {
    ch.load(kn, q0 + HD, ld, 0, S, D);
    ch.load(vn, q0 + 2 * HD, ld, 0, S, D);
  }
  float wn = window_entry(pdh, npd, wb0);
  for (int t = 0; t < T; ++t) {
    const int j0 = t * kStepF;
    __syncthreads();
    Planes<DP>::store(Ks, kn, D, &tiny);
    Planes<DP>::store(Vs, vn, D, &tiny);
    store_window(bw, wn);
    __syncthreads();
    if (t + 1 < T) {
      ch.load(kn, q0 + HD, ld, j0 + kStepF, S, D);
      ch.load(vn, q0 + 2 * HD, ld, j0 + kStepF, S, D);
      wn = window_entry(pdh, npd, wb0 + j0 + kStepF);
    }
    const float* bk = bw + (4 * g - ii + kRowsF - 1);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      f32x4 sc[2], dp[2];
      dot_row_blocks<DP, false>(Ks, L, 2 * half, qr, sc);
      dot_row_blocks<DP, false>(Vs, L, 2 * half, dr, dp);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int kb = 2 * half + i;
        f32x4& s = sc[i];
        // Keys past S have zero K rows and window entries, so p is finite there; it is then dropped.
#pragma unroll
        for (int r = 0; r < 4; ++r)
          s[r] = __builtin_amdgcn_exp2f(log2_units(fmaf(s[r], scale, bk[16 * kb + r])) - nlse);
        if (j0 + kStepF > S) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (j0 + 16 * kb + 4 * g + r >= S) s[r] = 0.f;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] *= fmaf(dp[i][r], kUp, -delta * kUp);  // ds times kUp
      }
      dot_positions_half<DP>(Ks, L, half, sc[0], sc[1], dq);
    }
  }
  if (__syncthreads_or(!narrow || tiny || overflowed<DP>(dq))) {
    if (wave < 4)
      dq_fp32<DP>(reinterpret_cast<float*>(Ks), reinterpret_cast<float*>(Vs), bw, qkv, ld, pd, dout, out32, lse,
                  delta_ws, dqkv, ldd, S, H, D, scale);
    else
      barriers(2 * ((S + kStepF - 1) / kStepF));
    return;
  }
  if (qvalid) {
    if (g == 0) delta_ws[(int64_t)bh * S + qi] = delta;
    store_row<DP>(dqkv + ((int64_t)b * S + qi) * ldd + (int64_t)h * D, dq, scale, g, D);
  }
}

// ------------------------------------------------------ backward: dK, dV and dpd
template <int DP>
__global__ __launch_bounds__(kThreadsS, 2) void relpos_bwd_dkdv_f32_kernel(
    const float* __restrict__ qkv, int64_t ld, const float* __restrict__ pd,
    const float* __restrict__ dout, const float* __restrict__ lse, const float* __restrict__ delta_ws,
    float* __restrict__ dqkv, int64_t ldd, float* __restrict__ part, int S, int H, int D, float scale,
    int kb0, int nkc) {
  __shared__ __attribute__((aligned(256))) unsigned char tiles[2 * kTileBytes<DP>];
  __shared__ KvShared sh;
  static_assert(2 * kTileBytes<DP> + sizeof(KvShared) <= 160 * 1024, "LDS of a CU");
  uint16_t* const Qs = reinterpret_cast<uint16_t*>(tiles);
  uint16_t* const Os = reinterpret_cast<uint16_t*>(tiles + kTileBytes<DP>);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4,
            l16 = lane & 15;
  // Key blocks [kb0, kb0 + nkc) of every (batch, head).
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int bh = tile / nkc, b = bh / H, h = bh - b * H;
  const int kbl = tile - bh * nkc;
  const int j_wg = (kb0 + kbl) * kRowsF;
  const int kk = wave * 16 + l16, kj = j_wg + kk;
  const bool kvalid = kj < S;
  const uint32_t kmask = lane_mask(kvalid);
  const int64_t HD = (int64_t)H * D;
  const float* q0 = qkv + (int64_t)b * S * ld + (int64_t)h * D;
  const float* o0 = dout + (int64_t)b * S * HD + (int64_t)h * D;
  const int npd = 2 * S - 1;
  const float* pdh = pd + (int64_t)h * npd;
  const float* lse_bh = lse + (int64_t)bh * S;
  const float* dl_bh = delta_ws + (int64_t)bh * S;
  float* prow = part + ((int64_t)bh * nkc + kbl) * (S + kRowsF);
  const int rlen = S + kRowsF - 1;  // diagonals of the partial row
  LaneOff<DP> L;
  L.init(g, l16);

  bool tiny = false, over = false;
  u32x4 kr[Planes<DP>::KS][3], vr[Planes<DP>::KS][3];
  const int64_t krow = (int64_t)(kvalid ? kj : 0) * ld;
  load_row<DP>(kr, q0 + HD + krow, g, D, kvalid);
  load_row<DP>(vr, q0 + 2 * HD + krow, g, D, kvalid, &tiny);
  Planes<DP>::zero_pad(Qs, D);
  Planes<DP>::zero_pad(Os, D);
  for (int e = tid; e < kRing; e += kThreadsS) sh.ring[e] = 0.f;
  for (int e = tid; e < kWinF * kDiagLd; e += kThreadsS) sh.dsb[e] = 0.f;
  f32x4 dk[Planes<DP>::CB], dv[Planes<DP>::CB];
  zero_acc<DP>(dk);
  zero_acc<DP>(dv);

  const bool narrow = ld <= kMaxLdS;
  const int T = narrow ? (S + kStepF - 1) / kStepF : 0;
  // Window entry x = kk - iq + 63 holds pd[h, (j_wg + kk) - (i0 + iq) + S - 1].
  const int wb0 = j_wg - (kStepF - 1) + S - 1;
  Chunks<DP> cq, co;
  cq.init(ld, D);
  co.init(HD, D);
  f32x4 qn[Chunks<DP>::CPT], on[Chunks<DP>::CPT];
  if (T) {
    cq.load(qn, q0, ld, 0, S, D);
    co.load(on, o0, HD, 0, S, D);
  }
  float wn = window_entry(pdh, npd, wb0);
  float ln = 0.f, dn = 0.f;  // lse and delta of query tid (threads tid < 64)
  auto stats = [&](int i0) {
    const int q = min(i0 + tid, S - 1);
    ln = lse_bh[q];
    dn = dl_bh[q];
  };
  // Query iq = 4 g + z of the step (z = 32 half + 16 i + r <= kYMax) against key kk: window entry kk - iq + 63
  // and dS entry [kk - iq + 63][iq], from the lowest address, so every z is a positive offset.
  constexpr int kYMax = 51;
  const float* const bwl = sh.bw + (kk - 4 * g + kStepF - 1 - kYMax);
  float* const dsl = sh.dsb + (kk - 4 * g + kStepF - 1 - kYMax) * kDiagLd + 4 * g + kYMax;
  if (tid < kStepF) stats(0);
  for (int t = 0; t < T; ++t) {
    const int i0 = t * kStepF;
    __syncthreads();
    Planes<DP>::store(Qs, qn, D, &tiny);
    Planes<DP>::store(Os, on, D, &tiny);
    store_window(sh.bw, wn);
    if (tid < kStepF) {
      const bool ok = i0 + tid < S;
      sh.Lq[tid] = ok ? ln : INFINITY;  // queries past S: p = 0
      sh.Dq[tid] = ok ? dn * kUp : 0.f;
    }
    __syncthreads();
    if (t + 1 < T) {
      cq.load(qn, q0, ld, i0 + kStepF, S, D);
      co.load(on, o0, HD, i0 + kStepF, S, D);
      wn = window_entry(pdh, npd, wb0 - i0 - kStepF);
      if (tid < kStepF) stats(i0 + kStepF);
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      // S and dP [query][key]: rows are this step's queries, columns the lane's key.
      f32x4 p[2], ds[2];
      dot_row_blocks<DP, true>(Qs, L, 2 * half, kr, p);
      dot_row_blocks<DP, true>(Os, L, 2 * half, vr, ds);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int iq0 = 32 * half + 16 * i + 4 * g;  // query of register 0
        const f32x4 lq = *reinterpret_cast<const f32x4*>(sh.Lq + iq0);
        const f32x4 dd = *reinterpret_cast<const f32x4*>(sh.Dq + iq0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int y = kYMax - (32 * half + 16 * i + r);
          p[i][r] = __builtin_amdgcn_exp2f(log2_units(fmaf(p[i][r], scale, bwl[y])) - lq[r]);
          // Keys past S have p != 0 (their bias is real) but no gradient: their dK and dV are
          // never stored and their dS is kept out of dpd.
          ds[i][r] = __uint_as_float(__float_as_uint(p[i][r] * fmaf(ds[i][r], kUp, -dd[r])) & kmask);
          dsl[y * (kDiagLd - 1)] = ds[i][r];
        }
      }
      dot_positions_half<DP>(Os, L, half, p[0] * kUp, p[1] * kUp, dv);  // dV^T += dO^T P
      dot_positions_half<DP>(Qs, L, half, ds[0], ds[1], dk);            // dK^T += Q^T dS
    }
    __syncthreads();
    // Local diagonal x = kk - iq + 63 of this step is partial-row entry R = x - 64 - i0 + S.
    if (tid < kWinF) {
      float acc = 0.f;
#pragma unroll 16
      for (int iq = 0; iq < kStepF; ++iq) acc += sh.dsb[tid * kDiagLd + iq];
      const int R = tid - kStepF - i0 + S;
      if (R >= 0) sh.ring[R & (kRing - 1)] += acc;
    }
    __syncthreads();
    // Later steps reach R <= S + 62 - i0 only: entries [S + 63 - i0, S + 126 - i0] are final.
    if (tid < kStepF) {
      const int R = S + (kStepF - 1) - i0 + tid;
      if (R >= 0 && R < rlen) {
        const float v = sh.ring[R & (kRing - 1)];
        over |= !isfinite(v);
        prow[R] = v * kDown;
        sh.ring[R & (kRing - 1)] = 0.f;
      }
    }
  }
  const int rmax = S + kStepF - 2 - kStepF * (T - 1);  // diagonals not stored yet: [0, rmax]
  if (T)
    for (int R = tid; R <= rmax; R += kThreadsS) over |= !isfinite(sh.ring[R & (kRing - 1)]);
  if (__syncthreads_or(!narrow || tiny || over || overflowed<DP>(dk) || overflowed<DP>(dv))) {
    if (wave < 4)
      dkdv_fp32<DP>(reinterpret_cast<float*>(Qs), reinterpret_cast<float*>(Os), sh, qkv, ld, pd, dout, lse, delta_ws,
                    dqkv, ldd, part, S, H, D, scale, kb0, nkc);
    else
      barriers(4 * ((S + kStepF - 1) / kStepF) + 1);
    return;
  }
  for (int R = tid; R <= rmax; R += kThreadsS)
    if (R < rlen) prow[R] = sh.ring[R & (kRing - 1)] * kDown;

  if (kvalid) {
    float* row = dqkv + ((int64_t)b * S + kj) * ldd + (int64_t)h * D;
    store_row<DP>(row + HD, dk, scale, g, D);
    store_row<DP>(row + 2 * HD, dv, 1.f, g, D);
  }
}

template <int DP>
void launch_fwd_f32(const float* qkv, int64_t ld, const float* pd, float* out, float* out32, float* lse,
                    int B, int S, int H, int D, float scale, hipStream_t st) {
  const dim3 grid((unsigned)(ceil_div(S, kRowsF) * B * H));
  hipLaunchKernelGGL((relpos_fwd_f32_kernel<DP>), grid, dim3(kThreadsS), 0, st, qkv, ld, pd, out, out32,
                     lse, S, H, D, scale);
}

template <int DP>
void launch_bwd_f32(const float* dout, const float* qkv, int64_t ld, const float* pd, const float* out32,
                    const float* lse, float* dqkv, int64_t ldd, float* dpd, float* delta, float* part,
                    int nkc, int B, int S, int H, int D, float scale, hipStream_t st) {
  const int nkb = (int)ceil_div(S, kRowsF);
  hipLaunchKernelGGL((relpos_bwd_dq_f32_kernel<DP>), dim3((unsigned)(nkb * B * H)), dim3(kThreadsS), 0, st, qkv,
                     ld, pd, dout, out32, lse, delta, dqkv, ldd, S, H, D, scale);
  // Key blocks in chunks of nkc (all of them with the full workspace); each chunk's partial
  // rows are summed into dpd before the next chunk overwrites them.
  for (int kb0 = 0; kb0 < nkb; kb0 += nkc) {
    const int n = min(nkc, nkb - kb0);
    hipLaunchKernelGGL((relpos_bwd_dkdv_f32_kernel<DP>), dim3((unsigned)(n * B * H)), dim3(kThreadsS), 0, st,
                       qkv, ld, pd, dout, lse, (const float*)delta, dqkv, ldd, part, S, H, D, scale, kb0, n);
    launch_dpd_reduce(part, dpd, B, S, H, kb0, n, kb0 > 0, st);
  }
}

}  // namespace

int relpos_fwd_f32(const float* qkv, int64_t ld, const float* pd, float* out, float* out32, float* lse,
                   int B, int S, int H, int D, float scale, hipStream_t st) {
#define KRSI_FWD_F32(DP_) \
  case DP_ / 16: launch_fwd_f32<DP_>(qkv, ld, pd, out, out32, lse, B, S, H, D, scale, st); break;
  switch ((D + 15) / 16) {
    KRSI_FWD_F32(16) KRSI_FWD_F32(32) KRSI_FWD_F32(48) KRSI_FWD_F32(64)
    KRSI_FWD_F32(80) KRSI_FWD_F32(96) KRSI_FWD_F32(112) KRSI_FWD_F32(128)
    default: return KRSI_ERR_UNSUPPORTED;
  }
#undef KRSI_FWD_F32
  return launch_status();
}

int relpos_bwd_f32(const float* dout, const float* qkv, int64_t ld, const float* pd, const float* out32,
                   const float* lse, float* dqkv, int64_t ldd, float* dpd, float* delta, float* part,
                   int nkc, int B, int S, int H, int D, float scale, hipStream_t st) {
#define KRSI_BWD_F32(DP_)                                                                                     \
  case DP_ / 16:                                                                                              \
    launch_bwd_f32<DP_>(dout, qkv, ld, pd, out32, lse, dqkv, ldd, dpd, delta, part, nkc, B, S, H, D, scale, st); \
    break;
  switch ((D + 15) / 16) {
    KRSI_BWD_F32(16) KRSI_BWD_F32(32) KRSI_BWD_F32(48) KRSI_BWD_F32(64)
    KRSI_BWD_F32(80) KRSI_BWD_F32(96) KRSI_BWD_F32(112) KRSI_BWD_F32(128)
    default: return KRSI_ERR_UNSUPPORTED;
  }
#undef KRSI_BWD_F32
  return launch_status();
}

}  // namespace krsi
