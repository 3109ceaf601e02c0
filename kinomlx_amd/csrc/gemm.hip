// Linear layers on gfx950 MFMA: the entry points, the affine int4 / int8 and mxfp8 weight-quantized
// products, the few-column (gate logit) products, and the register-staged fallback. Dense products with
// K % 64 == 0 run in gemm_dense.hip.
//
// c[m, n] = epilogue(sum_k a[m, k] * w[n, k]) — both operands K-contiguous (the reference's
// (out, in) weight layout), fp32 accumulation, one rounding to the 16-bit type (bf16, or fp16 for
// dense operands, template H).
//
// The register-staged kernel (v_mfma_f32_32x32x16): a BM x BN output tile per workgroup of WM x WN
// waves; each wave owns a (BM/WM) x (BN/WN) sub-tile as a grid of 32x32 MFMA blocks. K advances in stages of 64: the
// next stage's global loads are issued into registers before the current stage's MFMAs and
// written to the other half of a double-buffered LDS tile afterwards, so one barrier per stage
// suffices. LDS rows are 128 bytes (64 bf16) with the 16-byte chunk index XOR-swizzled by the
// row, so the 32-row fragment reads of an MFMA operand are bank-conflict free.
//
// The MFMA A operand is the weight tile and the B operand the activation tile, so that the
// accumulator's lane holds one output row m and runs of 4 consecutive columns n: the epilogue
// stores 8-byte vectors along the output row.
//
// Quantized weights: the stage's packed words and per-group bf16 scale/bias are loaded instead,
// and dequantized (bf16(fp32(scale) * q + fp32(bias))) inside the mainloop. mxfp8 weights (OCP
// MX: FP8 E4M3 elements, one E8M0 scale byte per 32 along K) take the same route: each element is
// converted to fp32 exactly (v_cvt_pk_f32_fp8) and multiplied by its power-of-two scale (exact),
// so the bf16 operand equals the format's value.
#include <stdlib.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "gemm.h"

namespace kx {
namespace {

constexpr int BK = 64;        // K per stage
constexpr int ROWB = BK * 2;  // bytes per LDS tile row

struct QuantW {
  const uint32_t* words;  // (n, k * bits / 32)
  const uint16_t* scales;  // (n, k / 64)
  const uint16_t* biases;  // (n, k / 64)
  const uint8_t* e8m0;     // mxfp8: (n, k / 32) scale bytes
};

// Weight-mode template code: 0 dense bf16, 4 / 8 affine int4 / int8, QMX8 mxfp8 (8-bit codes).
constexpr int QMX8 = 9;
template <int QB>
constexpr int qbits() { return QB == QMX8 ? 8 : QB; }

// 2^(s - 127) for an E8M0 scale byte (s = 0: 2^-127, an fp32 subnormal; s = 255: NaN).
__device__ __forceinline__ float e8m0_f32(uint32_t s) {
  const uint32_t bits = s == 0 ? 0x00400000u : (s == 255 ? 0x7FC00000u : s << 23);
  return __uint_as_float(bits);
}

// Four E4M3 bytes of w (lowest first) times a power-of-two scale, as four bf16 (two words). The
// fp8 -> fp32 conversion is exact, and so is the product while it stays in the fp32 normal range.
__device__ __forceinline__ uint2 mx8_quad(uint32_t w, float scale) {
  const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(w, false);
  const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(w, true);
  return make_uint2(pack2(lo.x * scale, lo.y * scale), pack2(hi.x * scale, hi.y * scale));
}

__device__ __forceinline__ int lds_off(int r, int c) { return r * ROWB + ((c ^ (r & 7)) << 4); }

template <int BITS>
__device__ __forceinline__ uint4 dequant8(const uint32_t* wd, float s, float b) {
  if constexpr (BITS == QMX8) {
    const uint2 q0 = mx8_quad(wd[0], s), q1 = mx8_quad(wd[1], s);
    return make_uint4(q0.x, q0.y, q1.x, q1.y);
  }
  float v[8];
  if (BITS == 4) {
    const uint32_t w = wd[0];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = fmaf(s, (float)((w >> (4 * j)) & 15u), b);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = fmaf(s, (float)((wd[0] >> (8 * j)) & 255u), b);
      v[4 + j] = fmaf(s, (float)((wd[1] >> (8 * j)) & 255u), b);
    }
  }
  return pack8(v);
}

// QB = 0: dense bf16 weights; QB = 4 / 8: affine quantized weights of that many bits; QMX8: mxfp8.
template <int BM, int BN, int WM, int WN, int QB, bool H = false>
__global__ __launch_bounds__(WM* WN * 64) void gemm_kernel(
    const uint16_t* __restrict__ A, int64_t lda, const uint16_t* __restrict__ W, int64_t ldw,
    QuantW qw, void* __restrict__ C, int64_t ldc, int M, int N, int K, Epilogue epi) {
  constexpr int NT = WM * WN * 64;
  constexpr int WT_M = BM / WM, WT_N = BN / WN;
  constexpr int MB = WT_M / 32, NB = WT_N / 32;
  constexpr int A_PER = BM * (BK / 8) / NT;
  constexpr int W_PER = BN * (BK / 8) / NT;
  constexpr int QBITS = qbits<QB>();
  constexpr int QWORDS = QBITS == 8 ? 2 : 1;
  static_assert(A_PER * NT == BM * (BK / 8) && W_PER * NT == BN * (BK / 8), "tile/threads");
  static_assert(MB >= 1 && NB >= 1, "wave tile");
  constexpr int STAGE = (BM + BN) * ROWB;

  __shared__ __attribute__((aligned(16))) uint8_t smem[2 * STAGE];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave % WM, wn = wave / WM;

  // ---- tile coordinates: XCD-contiguous, then grouped by 8 tile rows for L2 reuse
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const int t = xcd_remap(blockIdx.x, tiles_m * tiles_n);
  constexpr int GM = 8;
  const int group_width = GM * tiles_n;
  const int first_m = (t / group_width) * GM;
  const int gsz = min(tiles_m - first_m, GM);
  const int tm = first_m + (t % group_width) % gsz;
  const int tn = (t % group_width) / gsz;
  const int m0 = tm * BM, n0 = tn * BN;

  // ---- global -> register prefetch
  uint4 ra[A_PER];
  uint4 rw[QB == 0 ? W_PER : 1];
  uint32_t rq[QB == 0 ? 1 : W_PER][QWORDS];
  float rs[QB == 0 ? 1 : W_PER], rb[QB == 0 ? 1 : W_PER];

  auto load_stage = [&](int k0) {
#pragma unroll
    for (int i = 0; i < A_PER; ++i) {
      const int q = tid + i * NT;
      const int r = q >> 3, c = q & 7;
      const int gm = min(m0 + r, M - 1);
      const int gk = k0 + c * 8;
      // Branch-free K tail: read a valid chunk, then zero it (K % 8 == 0, so K - 8 >= 0).
      uint4 v = *reinterpret_cast<const uint4*>(A + (int64_t)gm * lda + min(gk, K - 8));
      if (gk >= K) v = make_uint4(0, 0, 0, 0);
      ra[i] = v;
    }
#pragma unroll
    for (int i = 0; i < W_PER; ++i) {
      const int q = tid + i * NT;
      const int r = q >> 3, c = q & 7;
      const int gn = min(n0 + r, N - 1);
      const int gk = k0 + c * 8;
      if (QB == 0) {
        uint4 v = *reinterpret_cast<const uint4*>(W + (int64_t)gn * ldw + min(gk, K - 8));
        if (gk >= K) v = make_uint4(0, 0, 0, 0);
        rw[i] = v;
      } else if constexpr (QB == QMX8) {
        // K % 32 == 0: a stage's second 32-wide half may lie past K; it reads the last group and
        // is zeroed (zero codes dequantize to zero)
        const int gkc = min(gk, K - 8);
        const int64_t wrow = (int64_t)gn * (K / 4);
#pragma unroll
        for (int j = 0; j < 2; ++j) rq[i][j] = gk < K ? qw.words[wrow + gkc / 4 + j] : 0u;
        rs[i] = e8m0_f32(qw.e8m0[(int64_t)gn * (K / 32) + gkc / 32]);
        rb[i] = 0.0f;
      } else {
        const int64_t wrow = (int64_t)gn * (K * QB / 32);
#pragma unroll
        for (int j = 0; j < QWORDS; ++j) rq[i][j] = qw.words[wrow + gk * QB / 32 + j];
        const int64_t g = (int64_t)gn * (K / 64) + k0 / 64;
        rs[i] = bf2f(qw.scales[g]);
        rb[i] = bf2f(qw.biases[g]);
      }
    }
  };

  auto store_stage = [&](uint8_t* buf) {
#pragma unroll
    for (int i = 0; i < A_PER; ++i) {
      const int q = tid + i * NT;
      *reinterpret_cast<uint4*>(buf + lds_off(q >> 3, q & 7)) = ra[i];
    }
    uint8_t* wbuf = buf + BM * ROWB;
#pragma unroll
    for (int i = 0; i < W_PER; ++i) {
      const int q = tid + i * NT;
      uint4 v;
      if (QB == 0)
        v = rw[i];
      else
        v = dequant8<QB>(rq[i], rs[i], rb[i]);
      *reinterpret_cast<uint4*>(wbuf + lds_off(q >> 3, q & 7)) = v;
    }
  };

  f32x16 acc[NB][MB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  const int stages = (K + BK - 1) / BK;
  load_stage(0);
  store_stage(smem);
  __syncthreads();

  const int lrow = lane & 31, lhalf = lane >> 5;
  for (int kt = 0; kt < stages; ++kt) {
    uint8_t* cur = smem + (kt & 1) * STAGE;
    const bool more = kt + 1 < stages;
    if (more) load_stage((kt + 1) * BK);
    const uint8_t* tA = cur;
    const uint8_t* tW = cur + BM * ROWB;
#pragma unroll
    for (int s = 0; s < BK / 16; ++s) {
      const int c = 2 * s + lhalf;
      bf16x8 af[MB], wf[NB];
#pragma unroll
      for (int j = 0; j < MB; ++j)
        af[j] = *reinterpret_cast<const bf16x8*>(tA + lds_off(wm * WT_M + j * 32 + lrow, c));
#pragma unroll
      for (int i = 0; i < NB; ++i)
        wf[i] = *reinterpret_cast<const bf16x8*>(tW + lds_off(wn * WT_N + i * 32 + lrow, c));
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j)
          acc[i][j] = mfma32x32x16<H>(wf[i], af[j], acc[i][j]);
    }
    if (more) store_stage(smem + ((kt + 1) & 1) * STAGE);
    __syncthreads();
  }

  // ---- epilogue, staged through LDS one 32-column block at a time. The unrolled part only
  // moves accumulators (static indices, so they stay in registers); bias, activation and the
  // gated residual run in a plain loop over rows with each lane on 4 consecutive columns.
  constexpr int EP_LD = 36;  // padded fp32 row: 16-byte writes from 16 rows hit distinct banks
  static_assert(WM * WN * WT_M * EP_LD * 4 <= 2 * STAGE, "epilogue staging must fit in LDS");
  float* ep = reinterpret_cast<float*>(smem) + wave * (WT_M * EP_LD);
  const int act = (epi.flags >> 4) & 15;
  const bool has_bias = epi.flags & KX_EPI_BIAS;
  const bool gated = epi.flags & KX_EPI_GATED_RESIDUAL;
  const bool resid_f32 = epi.flags & KX_EPI_RESID_F32;
  const bool out_f32 = epi.flags & KX_EPI_OUT_F32;
  const bool vec_store = (ldc % 4 == 0) && (!gated || epi.ldr % 4 == 0);
  const int col4 = (lane & 7) * 4;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
#pragma unroll
    for (int j = 0; j < MB; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float4 v;
        v.x = acc[i][j][g * 4 + 0];
        v.y = acc[i][j][g * 4 + 1];
        v.z = acc[i][j][g * 4 + 2];
        v.w = acc[i][j][g * 4 + 3];
        *reinterpret_cast<float4*>(ep + (j * 32 + lrow) * EP_LD + g * 8 + lhalf * 4) = v;
      }
    __syncthreads();
    const int n = n0 + wn * WT_N + i * 32 + col4;
    float bias4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (has_bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) bias4[e] = n + e < N ? e2f<H>(epi.bias[n + e]) : 0.0f;
    }
#pragma unroll 2
    for (int r = lane >> 3; r < WT_M; r += 8) {
      const int m = m0 + wm * WT_M + r;
      if (m >= M || n >= N) continue;
      const float4 a4 = *reinterpret_cast<const float4*>(ep + r * EP_LD + col4);
      float v[4] = {a4.x + bias4[0], a4.y + bias4[1], a4.z + bias4[2], a4.w + bias4[3]};
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = apply_act(v[e], act);
      const int64_t ro = (int64_t)m * epi.ldr + n;
      const int64_t co = (int64_t)m * ldc + n;
      if (vec_store && n + 3 < N) {
        if (gated) {
          const float* grow = epi.gate + (m / epi.gate_div) * epi.gate_stride;
          const float4 gv = *reinterpret_cast<const float4*>(grow + n);
          float rv[4];
          if (resid_f32) {
            const float4 rr = *reinterpret_cast<const float4*>(static_cast<const float*>(epi.resid) + ro);
            rv[0] = rr.x; rv[1] = rr.y; rv[2] = rr.z; rv[3] = rr.w;
          } else {
            const uint2 rr = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(epi.resid) + ro);
            rv[0] = e_lo<H>(rr.x); rv[1] = e_hi<H>(rr.x); rv[2] = e_lo<H>(rr.y); rv[3] = e_hi<H>(rr.y);
          }
          v[0] = rv[0] + gv.x * v[0];
          v[1] = rv[1] + gv.y * v[1];
          v[2] = rv[2] + gv.z * v[2];
          v[3] = rv[3] + gv.w * v[3];
        }
        if (out_f32) {
          *reinterpret_cast<float4*>(static_cast<float*>(C) + co) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
          uint2 o;
          o.x = e_pack2<H>(v[0], v[1]);
          o.y = e_pack2<H>(v[2], v[3]);
          *reinterpret_cast<uint2*>(static_cast<uint16_t*>(C) + co) = o;
        }
      } else {
        for (int e = 0; e < 4 && n + e < N; ++e) {
          float x = v[e];
          if (gated) {
            const float rv = resid_f32 ? static_cast<const float*>(epi.resid)[ro + e]
                                       : e2f<H>(static_cast<const uint16_t*>(epi.resid)[ro + e]);
            x = rv + epi.gate[(m / epi.gate_div) * epi.gate_stride + n + e] * x;
          }
          if (out_f32)
            static_cast<float*>(C)[co + e] = x;
          else
            static_cast<uint16_t*>(C)[co + e] = f2e<H>(x);
        }
      }
    }
    __syncthreads();
  }
}

template <int BITS>
__global__ __launch_bounds__(256) void dequant_kernel(const uint32_t* __restrict__ words,
                                                      const uint16_t* __restrict__ scales,
                                                      const uint16_t* __restrict__ biases,
                                                      uint16_t* __restrict__ out, int64_t n,
                                                      int64_t k, int group) {
  const int64_t chunks_per_row = k / 8;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n * chunks_per_row) return;
  const int64_t r = idx / chunks_per_row, c = idx - r * chunks_per_row;
  const int64_t kk = c * 8;
  const int64_t g = r * (k / group) + kk / group;
  const uint32_t* wd = words + r * (k * BITS / 32) + kk * BITS / 32;
  uint32_t tmp[2] = {wd[0], BITS == 8 ? wd[1] : 0u};
  *reinterpret_cast<uint4*>(out + r * k + kk) = dequant8<BITS>(tmp, bf2f(scales[g]), bf2f(biases[g]));
}

// mxfp8 in the reference layout: (n, k / 4) words and (n, k / 32) scale bytes -> (n, k) bf16, eight
// values per thread.
__global__ __launch_bounds__(256) void dequant_mx8_kernel(const uint32_t* __restrict__ words,
                                                          const uint8_t* __restrict__ scales,
                                                          uint16_t* __restrict__ out, int64_t n, int64_t k) {
  const int64_t chunks_per_row = k / 8;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n * chunks_per_row) return;
  const int64_t r = idx / chunks_per_row, c = idx - r * chunks_per_row;
  const uint2 w = *reinterpret_cast<const uint2*>(words + r * (k / 4) + 2 * c);
  uint32_t tmp[2] = {w.x, w.y};
  *reinterpret_cast<uint4*>(out + r * k + 8 * c) =
      dequant8<QMX8>(tmp, e8m0_f32(scales[r * (k / 32) + c / 4]), 0.0f);
}

// mxfp4 / nvfp4: (n, k / 8) words of eight E2M1 codes and (n, k / G) scale bytes (G = 32: E8M0,
// G = 16: E4M3) -> (n, k) bf16, eight values (one word) per thread. Every value is exact: an E2M1
// magnitude has at most 2 significant bits and the scale at most 4.
__device__ __forceinline__ float e2m1_f32(uint32_t c) {
  const uint32_t m3 = c & 7u;
  // 0, 0.5, then 1, 1.5, 2, 3, 4, 6: from code 2 on, the fp32 bits step by 2^22 from 1.0
  const float mag = m3 < 2u ? 0.5f * (float)m3 : __uint_as_float(0x3F800000u + ((m3 - 2u) << 22));
  return __uint_as_float(__float_as_uint(mag) | ((c & 8u) << 28));
}
__device__ __forceinline__ float e4m3_f32(uint32_t b) {
  const uint32_t e = (b >> 3) & 15u, m = b & 7u;
  const float mag = e == 0 ? (float)m * 0.001953125f : ldexpf(1.0f + (float)m * 0.125f, (int)e - 7);
  return (b & 0x80u) ? -mag : mag;
}
template <bool NV>
__global__ __launch_bounds__(256) void dequant_fp4_kernel(const uint32_t* __restrict__ words,
                                                          const uint8_t* __restrict__ scales,
                                                          uint16_t* __restrict__ out, int64_t n, int64_t k) {
  constexpr int G = NV ? 16 : 32;
  const int64_t words_per_row = k / 8;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n * words_per_row) return;
  const int64_t r = idx / words_per_row, c = idx - r * words_per_row;
  const uint32_t w = words[idx];
  const uint32_t sb = scales[r * (k / G) + (8 * c) / G];
  const float sc = NV ? e4m3_f32(sb) : e8m0_f32(sb);
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = e2m1_f32((w >> (4 * j)) & 15u) * sc;
  *reinterpret_cast<uint4*>(out + r * k + 8 * c) = pack8(v);
}

// mxfp8 in the pretransposed layout (quantized from weight.T: (k, n / 4) words and (k, n / 32)
// scale bytes, groups along n) -> the (n, k) bf16 weight, through 64 x 64 LDS tiles: a thread
// dequantizes 16 consecutive n of one k row and writes them transposed into the tile, then
// writes 16 consecutive k of one n row. n % 32 == 0 and k % 8 == 0 keep every 16-run of n and
// every 8-run of k either wholly inside the matrix or wholly outside.
__global__ __launch_bounds__(256) void dequant_mx8_t_kernel(const uint32_t* __restrict__ words,
                                                            const uint8_t* __restrict__ scales,
                                                            uint16_t* __restrict__ out, int64_t n, int64_t k) {
  __shared__ uint16_t tile[64][64 + 2];
  const int t = threadIdx.x;
  const int64_t n0 = (int64_t)blockIdx.x * 64, k0 = (int64_t)blockIdx.y * 64;
  {
    const int kl = t >> 2, nl = (t & 3) * 16;
    const int64_t kk = k0 + kl, nn = n0 + nl;
    if (kk < k && nn < n) {
      const uint4 w = *reinterpret_cast<const uint4*>(words + kk * (n / 4) + nn / 4);
      const float sc = e8m0_f32(scales[kk * (n / 32) + nn / 32]);
      const uint32_t wv[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint2 q = mx8_quad(wv[j], sc);
        tile[nl + 4 * j][kl] = (uint16_t)(q.x & 0xffffu);
        tile[nl + 4 * j + 1][kl] = (uint16_t)(q.x >> 16);
        tile[nl + 4 * j + 2][kl] = (uint16_t)(q.y & 0xffffu);
        tile[nl + 4 * j + 3][kl] = (uint16_t)(q.y >> 16);
      }
    }
  }
  __syncthreads();
  const int nl = t >> 2, kl = (t & 3) * 16;
  const int64_t nn = n0 + nl;
  if (nn >= n) return;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int64_t kk = k0 + kl + 8 * h;
    if (kk >= k) break;
    const uint16_t* src = &tile[nl][kl + 8 * h];
    uint4 v;
    v.x = src[0] | ((uint32_t)src[1] << 16);
    v.y = src[2] | ((uint32_t)src[3] << 16);
    v.z = src[4] | ((uint32_t)src[5] << 16);
    v.w = src[6] | ((uint32_t)src[7] << 16);
    *reinterpret_cast<uint4*>(out + nn * k + kk) = v;
  }
}

// ---- quantized direct-to-LDS kernel (K % 128 == 0) -----------------------------------------------
//
// Operand tiles go from global memory straight into LDS (no VGPR staging): one wave instruction fills
// 64 lanes x 16 B = DRPI rows of DBK bf16, from a scalar tile base plus a loop-invariant 32-bit lane
// offset. A ring of four stages of 32 along K; the DMA for stage kt+3 goes out between the MFMAs of
// stage kt. Every k16 step is one scheduling region: wait for this step's fragments (read one step
// earlier), issue the fragment reads of the next step, then the step's MFMAs, so LDS latency hides
// under a full step of MFMAs and never more than MB + NB reads are outstanding (lgkmcnt counts to
// 15). The last step of a stage holds the stage's only workgroup barrier. The 16-byte slots of a
// row are XOR-swizzled so that both the DMA writes and the 32-row fragment reads are bank-conflict
// free.
//
// Epilogue: each wave stages half of its fp32 tile in LDS at a time and writes it back in rows,
// 4 columns per lane, so bias / gate / residual loads and the stores are contiguous runs. Full,
// aligned tiles take a compile-time specialisation per residual mode (GMODE 0: none, 1: bf16
// residual, 2: fp32 residual) and output type; edge tiles take the generic masked path.

// 8-bit packed weight rows (32 bytes per stage): chunk swizzle of row r
__device__ __forceinline__ int qswz(int r) { return (r >> 3) & 1; }
// One full-tile epilogue row piece: bias + activation (+ gated residual), then the store of 4
// consecutive columns. Values by value so that nothing of the caller's frame is addressed.
template <int GMODE, bool OUTF32, int ACT, typename ResidT>
__device__ __forceinline__ void epi_row4(float4 a4, ResidT res, float b0, float b1, float b2, float b3,
                                         int act, float4 gv, char* dst) {
  float v[4] = {a4.x + b0, a4.y + b1, a4.z + b2, a4.w + b3};
  if (ACT != 0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = act_c<ACT>(v[e], act);
  }
  if constexpr (GMODE != 0) {
    float rv[4];
    if constexpr (GMODE == 2) {
      rv[0] = res.x; rv[1] = res.y; rv[2] = res.z; rv[3] = res.w;
    } else {
      rv[0] = lo_f(res.x); rv[1] = hi_f(res.x); rv[2] = lo_f(res.y); rv[3] = hi_f(res.y);
    }
    v[0] = rv[0] + gv.x * v[0];
    v[1] = rv[1] + gv.y * v[1];
    v[2] = rv[2] + gv.z * v[2];
    v[3] = rv[3] + gv.w * v[3];
  }
  if constexpr (OUTF32) {
    *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    uint2 o;
    o.x = pack2(v[0], v[1]);
    o.y = pack2(v[2], v[3]);
    *reinterpret_cast<uint2*>(dst) = o;
  }
}

// QB = 4 / 8 (affine) and QMX8 (mxfp8): each stage DMAs the activations, the packed weight bytes and the scale (/ bias) words of its group, and every wave
// dequantizes its own weight fragments in registers (bit-exact, the arithmetic of dequant8)
// between the MFMAs of the previous k16 step: the stage's weights cross LDS once, packed, and no
// bf16 copy of them is written. TL: the affine weights are in the tiled layout (one contiguous
// block per 256-row tile and stage, see kx_qweight_tile_affine), else in the reference layout
// (one 16- or 32-byte piece per row).
template <int BM, int BN, int QB, bool TL, int GMODE, bool OUTF32>
__global__ __launch_bounds__(256) void gemm_lds_kernel(
    const uint16_t* __restrict__ A, int64_t lda, QuantW qw, void* __restrict__ C, int64_t ldc, int M, int N, int K, Epilogue epi) {
  // stage geometry: 32-wide stages in a 4-stage ring; a row's 16-byte slots are XOR-swizzled (by
  // (r >> 2) & 3) so that the DMA writes and the 32-row fragment reads are bank-conflict free
  constexpr int DBK = 32;                   // K per LDS stage
  constexpr int DROW = DBK * 2;             // bytes per LDS row
  constexpr int DCPR = DBK / 8;             // 16-byte chunks per row
  constexpr int DRPI = 64 / DCPR;           // rows one DMA instruction fills
  constexpr int DNS = 4;                    // stages in the ring
  const auto dswz = [](int r) { return (r >> 2) & 3; };
  constexpr int A_INST = BM / DRPI / 4;
  constexpr int QROW = DBK * qbits<QB>() / 8;                         // packed bytes per row
  constexpr int WQ_INST = BN * QROW / 1024 / 4;                       // packed words, per wave
  constexpr int SB_BYTES = QB == QMX8 ? 4 : 8;                        // scale (bias) bytes per row
  constexpr int SB_INST = SB_BYTES * BN / 256 / 4;                    // scale and bias pairs
  constexpr int W_INST = WQ_INST + SB_INST;
  constexpr int PER = A_INST + W_INST;  // DMA instructions per wave per stage
  constexpr int W_BYTES = BN * QROW + BN * SB_BYTES;
  constexpr int STAGE = BM * DROW + W_BYTES;
  constexpr int RING = DNS * STAGE;
  // wave layout: 1 x 4 waves of BM x (BN / 4), so that each weight column is dequantized by one wave
  // only (a 2 x 2 layout dequantizes every column twice) for the same LDS fragment traffic per MFMA
  constexpr int WGM = 1, WGN = 4;
  constexpr int WT_M = BM / WGM, WT_N = BN / WGN;
  constexpr int MB = WT_M / 32, NB = WT_N / 32;
  constexpr int KS = DBK / 16;
  constexpr int DPS = (PER + KS - 1) / KS;  // DMA instructions per k16 step
  // At the wait in the last k16 step, stages kt+2 .. kt+NS-2 and the DMA of this iteration's
  // earlier steps may stay in flight: stage kt+1 is then complete.
  constexpr int NBEFORE = (KS - 1) * DPS < PER ? (KS - 1) * DPS : PER;
  constexpr int WAITN = (DNS - 3) * PER + NBEFORE;
  constexpr int PITCH = WT_N / 2 + 4;  // staged epilogue row, floats
  constexpr int EP_BYTES = 4 * WT_M * PITCH * 4;
  constexpr int SMEM = RING > EP_BYTES ? RING : EP_BYTES;
  static_assert(A_INST * DRPI * 4 == BM && MB >= 1 && NB >= 2, "tile");
  static_assert(BN == 256 && WQ_INST >= 1, "weight tile");
  static_assert(MB + NB <= 15 && WAITN >= 0, "pipeline");
  static_assert(!(TL && QB == QMX8), "mxfp8 weights are read in the reference layout only");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[SMEM];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WGM, wn = wave / WGM;
  const int lrow = lane & 31, lhalf = lane >> 5;

  // tile coordinates (see lds_tile_of)
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  int2 tile = lds_tile_of(blockIdx.x, tiles_m, tiles_n);
  if (epi.rows_desc) tile.x = tiles_m - 1 - tile.x;
  const int m0 = tile.x * BM, n0 = tile.y * BN;

  // per-lane DMA sources: lane -> row lane / DCPR of the instruction's rows, slot lane % DCPR;
  // rows past the end re-read the last row (in bounds; their results are never stored)
  const int r_in = lane / DCPR, slot = lane % DCPR;
  uint32_t vo[PER];
#pragma unroll
  for (int i = 0; i < A_INST; ++i) {
    const int r = (wave * A_INST + i) * DRPI + r_in;
    vo[i] = (uint32_t)(((int64_t)(min(m0 + r, M - 1) - m0) * lda + (slot ^ dswz(r)) * 8) * 2);
  }
  const char* a_base = reinterpret_cast<const char*>(A + (int64_t)m0 * lda);
  const char* w_base;            // the packed words
  const char* s_base = nullptr;  // scale pairs (bias pairs follow at b_base)
  const char* b_base = nullptr;
  const int64_t qrow_bytes = (int64_t)K * qbits<QB>() / 8, groups = K / 64;
  if constexpr (TL) {
    // tiled: the stage's packed words (BN * QROW bytes) and scale / bias pairs (BN * 8 bytes of
    // its 128-wide window) are contiguous blocks (8-bit rows: chunk swizzle as below)
#pragma unroll
    for (int i = 0; i < WQ_INST; ++i) {
      const int r = (wave * WQ_INST + i) * (1024 / QROW) + lane / (QROW / 16);
      const int chunk = QROW == 32 ? (lane & 1) ^ qswz(r) : 0;
      vo[A_INST + i] = (uint32_t)(r * QROW + chunk * 16);
    }
#pragma unroll
    for (int i = 0; i < SB_INST; ++i) vo[A_INST + WQ_INST + i] = (uint32_t)((wave * SB_INST + i) * 256 + lane * 4);
    const int64_t nb = n0 / BN;
    w_base = reinterpret_cast<const char*>(qw.words) + nb * (K / DBK) * (int64_t)(BN * QROW);
    s_base = reinterpret_cast<const char*>(qw.scales) + nb * (K / 128) * (int64_t)(BN * 8);
  } else {
    // packed words: RPW rows per instruction, QROW / 16 chunks per row; an 8-bit row's two
    // chunks trade places when (r >> 3) & 1, so that the 16-byte fragment reads of 16 rows
    // cover every bank once
    constexpr int RPW = 1024 / QROW;
#pragma unroll
    for (int i = 0; i < WQ_INST; ++i) {
      const int r = (wave * WQ_INST + i) * RPW + lane / (QROW / 16);
      const int chunk = QROW == 32 ? (lane & 1) ^ qswz(r) : 0;
      vo[A_INST + i] = (uint32_t)((int64_t)(min(n0 + r, N - 1) - n0) * qrow_bytes + chunk * 16);
    }
    // scale / bias pairs (mxfp8: scale-byte quads): 64 rows x 4 bytes per instruction
    const int64_t sb_row = QB == QMX8 ? K / 32 : groups * 2;  // bytes per row of the scale array
#pragma unroll
    for (int i = 0; i < SB_INST; ++i) {
      const int g = wave * SB_INST + i;
      const int r = (g % (BN / 64)) * 64 + lane;
      vo[A_INST + WQ_INST + i] = (uint32_t)((int64_t)(min(n0 + r, N - 1) - n0) * sb_row);
    }
    w_base = reinterpret_cast<const char*>(qw.words) + (int64_t)n0 * qrow_bytes;
    if constexpr (QB == QMX8) {
      s_base = reinterpret_cast<const char*>(qw.e8m0) + (int64_t)n0 * sb_row;
    } else {
      s_base = reinterpret_cast<const char*>(qw.scales) + (int64_t)n0 * sb_row;
      b_base = reinterpret_cast<const char*>(qw.biases) + (int64_t)n0 * sb_row;
    }
  }
  // activations: buffer loads (the tile base as the resource; lane offsets < 2^31, K offsets < 2^23
  // by the dispatch's stride limits)
  const rsrc_t a_rsrc = raw_rsrc(a_base);
  auto dma = [&](int i, uint8_t* buf, int k0) {
    if (i < A_INST) {
      buffer_lds16(a_rsrc, buf + (wave * A_INST + i) * DRPI * DROW, vo[i], (uint32_t)k0 * 2);
    } else if (TL && i < A_INST + WQ_INST) {
      __builtin_amdgcn_global_load_lds((const void*)(w_base + (int64_t)(k0 / DBK) * (BN * QROW) + vo[i]),
                                       KX_LDS(buf + BM * DROW + (wave * WQ_INST + i - A_INST) * 1024), 16, 0, 0);
    } else if (TL) {
      const int g = wave * SB_INST + (i - A_INST - WQ_INST);
      __builtin_amdgcn_global_load_lds((const void*)(s_base + (int64_t)(k0 / 128) * (BN * 8) + vo[i]),
                                       KX_LDS(buf + BM * DROW + BN * QROW + g * 256), 4, 0, 0);
    } else if (i < A_INST + WQ_INST) {
      __builtin_amdgcn_global_load_lds((const void*)(w_base + (int64_t)k0 * qbits<QB>() / 8 + vo[i]),
                                       KX_LDS(buf + BM * DROW + (wave * WQ_INST + i - A_INST) * 1024), 16, 0, 0);
    } else if constexpr (QB == QMX8) {
      // the scale-byte quad holding group k0 / 32 (k0 / 32 rounded down to a multiple of 4)
      const int g = wave * SB_INST + (i - A_INST - WQ_INST);
      __builtin_amdgcn_global_load_lds((const void*)(s_base + (int64_t)((k0 >> 5) & ~3) + vo[i]),
                                       KX_LDS(buf + BM * DROW + BN * QROW + g * 256), 4, 0, 0);
    } else {
      // the pair of groups holding group k0 / 64 (k0 / 64 rounded down to even)
      const int g = wave * SB_INST + (i - A_INST - WQ_INST);
      const char* src = (g < BN / 64 ? s_base : b_base) + (int64_t)((k0 >> 6) & ~1) * 2 + vo[i];
      __builtin_amdgcn_global_load_lds((const void*)src, KX_LDS(buf + BM * DROW + BN * QROW + g * 256), 4, 0, 0);
    }
  };

  // fragment byte offsets, per k16 step (the MFMA A operand is the weight tile): step s of lane
  // half h covers k = 16 h + 8 s .. + 7 of the stage (the same permutation of the sum on both
  // operands), so that a lane's packed weight bytes of both steps are contiguous and come in one
  // read per stage
  int a_off[KS][MB];
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int j = 0; j < MB; ++j) {
      const int r = j * 32 + lrow;
      a_off[s][j] = r * DROW + (((2 * lhalf + s) ^ dswz(r)) << 4);
    }

  f32x16 acc[NB][MB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  const int stages = K / DBK;
#pragma unroll
  for (int p = 0; p < DNS - 1; ++p)
#pragma unroll
    for (int i = 0; i < PER; ++i) dma(i, smem + p * STAGE, min(p, stages - 1) * DBK);
  wait_vmcnt<(DNS - 2) * PER>();
  KX_BARRIER();
  bf16x8 fa[2][MB], fw[2][NB];
  int cur_i = 0;
  {
    // ---- mainloop: every wave dequantizes its own weight fragments in registers ----
    // A lane's packed bytes of weight block i for the whole stage (both k16 steps of its row)
    // and the row's scale (and bias) word; read once per stage, right after the stage's barrier.
    using Raw = typename std::conditional<qbits<QB>() == 4, uint2, uint4>::type;
    Raw raw[NB];
    uint32_t rsw[NB], rbw[NB];
    int wr_off[NB], ws_off[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int r = wn * WT_N + i * 32 + lrow;
      wr_off[i] = BM * DROW + (QROW == 16 ? r * 16 + 8 * lhalf : r * 32 + ((lhalf ^ qswz(r)) << 4));
      ws_off[i] = BM * DROW + BN * QROW + (TL && QB != QMX8 ? 8 * r : 4 * r);
    }
    // scale (and bias) of each block's rows for stage kt: affine, group kt / 2 of the pair (64-wide
    // groups); mxfp8, scale byte kt % 4 of the word (32-wide groups)
    float scl[NB], bia[NB];
    auto stage_scales = [&](int kt) {
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        if constexpr (QB == QMX8) {
          scl[i] = e8m0_f32((rsw[i] >> (8 * (kt & 3))) & 255u);
          bia[i] = 0.0f;
        } else {
          const bool half = (kt >> 1) & 1;
          scl[i] = half ? hi_f(rsw[i]) : lo_f(rsw[i]);
          bia[i] = half ? hi_f(rbw[i]) : lo_f(rbw[i]);
        }
      }
    };
    // values 2p, 2p+1 of block i's fragment for k16 step s, as two bf16 (dequant8's arithmetic)
    auto dq_pair = [&](int i, int s, int p) -> uint32_t {
      if constexpr (QB == QMX8) {
        const uint32_t w = (2 * s + (p >> 1)) == 0 ? raw[i].x : (2 * s + (p >> 1)) == 1 ? raw[i].y
                           : (2 * s + (p >> 1)) == 2 ? raw[i].z : raw[i].w;
        const f32x2 v = (p & 1) ? __builtin_amdgcn_cvt_pk_f32_fp8(w, true) : __builtin_amdgcn_cvt_pk_f32_fp8(w, false);
        return pack2(v.x * scl[i], v.y * scl[i]);
      } else if constexpr (QB == 8) {
        const uint32_t w = (2 * s + (p >> 1)) == 0 ? raw[i].x : (2 * s + (p >> 1)) == 1 ? raw[i].y
                           : (2 * s + (p >> 1)) == 2 ? raw[i].z : raw[i].w;
        const int b = 2 * (p & 1);
        return pack2(fmaf(scl[i], (float)((w >> (8 * b)) & 255u), bia[i]),
                     fmaf(scl[i], (float)((w >> (8 * b + 8)) & 255u), bia[i]));
      } else {
        // even nibbles in the low halves of the bytes of lo, odd ones in hi: each value is one
        // byte conversion (v_cvt_f32_ubyte), the masks are shared by the word's four pairs
        const uint32_t w = s ? raw[i].y : raw[i].x;
        uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
        // the masked words opaque to the optimizer, which would otherwise fold the masks back
        // into one bit-field extract per value
        asm("" : "+v"(lo));
        asm("" : "+v"(hi));
        return pack2(fmaf(scl[i], (float)((lo >> (8 * p)) & 255u), bia[i]),
                     fmaf(scl[i], (float)((hi >> (8 * p)) & 255u), bia[i]));
      }
    };
    // the fragment under construction, four pairs
    uint32_t part[NB][4];
    auto dq_step = [&](int idx, int s) {  // pair idx of the step's NB * 4 pairs
      const int i = idx >> 2, p = idx & 3;
      part[i][p] = dq_pair(i, s, p);
    };
    auto dq_commit = [&](bf16x8* wf) {
#pragma unroll
      for (int i = 0; i < NB; ++i) wf[i] = __builtin_bit_cast(bf16x8, make_uint4(part[i][0], part[i][1], part[i][2], part[i][3]));
    };
    constexpr int NMF = NB * MB;
    constexpr int NPAIR = NB * 4;
    constexpr int SB_RD = QB == QMX8 || TL ? 1 : 2;  // scale (bias) reads per block
    constexpr int NRD1 = MB + NB * (1 + SB_RD);      // LDS reads at a stage's start
    constexpr int NRQ = NB * (1 + SB_RD);             // of which the packed weights and scales
    constexpr int QSPLIT = 4;                         // MFMAs before the wait for those
    static_assert(NMF > QSPLIT, "MFMAs per step");
    // LDS read r of a stage's start: the raw blocks and scale words (needed first, by the
    // dequantization of the stage's step 0), then the A fragments of its step 0
    auto stage_read = [&](int r, const uint8_t* buf) {
      if (r >= NRQ) {
        fa[0][r - NRQ] = *reinterpret_cast<const bf16x8*>(buf + a_off[0][r - NRQ]);
      } else if (r < NB) {
        raw[r] = *reinterpret_cast<const Raw*>(buf + wr_off[r]);
      } else {
        const int q = r - NB, i = q % NB;
        if constexpr (QB == QMX8) {
          rsw[i] = *reinterpret_cast<const uint32_t*>(buf + ws_off[i]);
        } else if constexpr (TL) {
          const uint2 pr = *reinterpret_cast<const uint2*>(buf + ws_off[i]);
          rsw[i] = pr.x;
          rbw[i] = pr.y;
        } else if (q < NB) {
          rsw[i] = *reinterpret_cast<const uint32_t*>(buf + ws_off[i]);
        } else {
          rbw[i] = *reinterpret_cast<const uint32_t*>(buf + ws_off[i] + 4 * BN);
        }
      }
    };

#pragma unroll
    for (int r = 0; r < NRD1; ++r) stage_read(r, smem);
    wait_lgkmcnt0();
    stage_scales(0);
#pragma unroll
    for (int q = 0; q < NPAIR; ++q) dq_step(q, 0);
    dq_commit(fw[0]);
    for (int kt = 0; kt < stages; ++kt) {
      const uint8_t* cur = smem + cur_i * STAGE;
      const int nxt_i = cur_i + 1 == DNS ? 0 : cur_i + 1;
      const uint8_t* nxt = smem + nxt_i * STAGE;
      uint8_t* iss = smem + (cur_i == 0 ? DNS - 1 : cur_i - 1) * STAGE;
      const int k_iss = min(kt + DNS - 1, stages - 1) * DBK;
      // step 0, in a fixed order: each MFMA, then its share of the pairs of step 1's weight
      // fragments (the arithmetic runs while the MFMA executes); the A fragments of step 1 and
      // the first DMA issues ride along the first MFMAs
      __builtin_amdgcn_sched_barrier(0);
      wait_lgkmcnt0();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < NMF; ++q) {
        const int i = q / MB, j = q % MB;
        acc[i][j] = mfma32x32x16<false>(fw[0][i], fa[0][j], acc[i][j]);
        if (q < MB) fa[1][q] = *reinterpret_cast<const bf16x8*>(cur + a_off[1][q]);
        if (q < DPS && q < PER) dma(q, iss, k_iss);
#pragma unroll
        for (int idx = q * NPAIR / NMF; idx < (q + 1) * NPAIR / NMF; ++idx) dq_step(idx, 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      dq_commit(fw[1]);
      // step 1: stage kt+1 has landed for this wave and its reads of stage kt-1's buffer ended
      // one step ago; after the barrier this holds for every wave. The stage-start reads of stage
      // kt+1 and the remaining DMA issues ride along the first QSPLIT MFMAs; after the wait for
      // those reads, each further MFMA is followed by pairs of stage kt+1's step-0 fragments.
      __builtin_amdgcn_sched_barrier(0);
      wait_lgkmcnt0();
      wait_vmcnt<WAITN>();
      KX_BARRIER();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < QSPLIT; ++q) {
        const int i = q / MB, j = q % MB;
        acc[i][j] = mfma32x32x16<false>(fw[1][i], fa[1][j], acc[i][j]);
#pragma unroll
        for (int r = q * NRD1 / QSPLIT; r < (q + 1) * NRD1 / QSPLIT; ++r) stage_read(r, nxt);
#pragma unroll
        for (int d = DPS + q * (PER - DPS) / QSPLIT; d < DPS + (q + 1) * (PER - DPS) / QSPLIT; ++d)
          dma(d, iss, k_iss);
        __builtin_amdgcn_sched_barrier(0);
      }
      wait_lgkmcnt<MB>();
      stage_scales(kt + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = QSPLIT; q < NMF; ++q) {
        const int i = q / MB, j = q % MB;
        acc[i][j] = mfma32x32x16<false>(fw[1][i], fa[1][j], acc[i][j]);
#pragma unroll
        for (int idx = (q - QSPLIT) * NPAIR / (NMF - QSPLIT); idx < (q - QSPLIT + 1) * NPAIR / (NMF - QSPLIT); ++idx)
          dq_step(idx, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      dq_commit(fw[0]);
      cur_i = nxt_i;
    }
  }
  wait_vmcnt<0>();

  // ---- epilogue: the accumulator lane holds row m = j*32 + lrow and columns 8g + 4 lhalf + e of
  // block i; staged per half of the wave's columns into a private LDS region.
  const bool vec_ok = (ldc % 4 == 0) && (!(epi.flags & KX_EPI_GATED_RESIDUAL) || epi.ldr % 4 == 0);
  const bool full = vec_ok && m0 + BM <= M && n0 + BN <= N;
  float* ep = reinterpret_cast<float*>(smem) + wave * (WT_M * PITCH);
  constexpr int HALF_N = WT_N / 2;
  constexpr int LPR = HALF_N / 4;  // lanes per staged row
  constexpr int RPI_EP = 64 / LPR;   // rows per read-back iteration
  const int q = lane % LPR, rr = lane / LPR;
  const int act = (epi.flags >> 4) & 15;
  const bool has_bias = epi.flags & KX_EPI_BIAS;
  const int mrow0 = m0 + wm * WT_M;
  using ResidT = typename std::conditional<GMODE == 2, float4, uint2>::type;
  const int64_t resid_es = GMODE == 2 ? 4 : 2;
  const char* rbase = GMODE == 0 ? nullptr
      : reinterpret_cast<const char*>(epi.resid) + ((int64_t)mrow0 * epi.ldr + n0 + wn * WT_N + 4 * q) * resid_es;
  KX_BARRIER();  // every wave is done with the main loop's LDS
  // The half loop is not unrolled (its body is large); each half stages its accumulator blocks
  // under its own branch so that every accumulator index stays a compile-time constant.
#define KX_STAGE_BLOCK(ii, i)                                                                     \
  _Pragma("unroll") for (int j = 0; j < MB; ++j)                                                  \
  _Pragma("unroll") for (int g = 0; g < 4; ++g)                                                   \
      *reinterpret_cast<float4*>(ep + (j * 32 + lrow) * PITCH + (ii) * 32 + 8 * g + 4 * lhalf) =  \
          make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
#pragma unroll 1
  for (int h = 0; h < 2; ++h) {
    if (h == 0) {
#pragma unroll
      for (int ii = 0; ii < NB / 2; ++ii) { KX_STAGE_BLOCK(ii, ii) }
    } else {
#pragma unroll
      for (int ii = 0; ii < NB / 2; ++ii) { KX_STAGE_BLOCK(ii, NB / 2 + ii) }
    }
#undef KX_STAGE_BLOCK
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int n = n0 + wn * WT_N + h * HALF_N + 4 * q;
    if (full) {
      // column data is fixed per lane: bias, and the gate when one gate row covers the rows
      float b4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (has_bias) {
        const uint2 bb = *reinterpret_cast<const uint2*>(epi.bias + n);
        b4[0] = lo_f(bb.x); b4[1] = hi_f(bb.x); b4[2] = lo_f(bb.y); b4[3] = hi_f(bb.y);
      }
      const int64_t gstride = epi.gate_stride, gdiv = epi.gate_div;
      const bool gate_const = GMODE == 0 || gstride == 0 || (mrow0 / gdiv) == ((mrow0 + WT_M - 1) / gdiv);
      float4 g4c = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (GMODE != 0 && gate_const) g4c = *reinterpret_cast<const float4*>(epi.gate + (mrow0 / gdiv) * gstride + n);
      char* cbase = reinterpret_cast<char*>(C) + ((int64_t)mrow0 * ldc + n) * (OUTF32 ? 4 : 2);
      // the rows with the activation fixed at compile time (a run-time choice per value put a
      // chain of scalar branches around every value and serialised them)
      auto full_rows = [&](auto act_tag, auto gate_tag) {
        constexpr int ACT = decltype(act_tag)::value;
        constexpr bool GC = decltype(gate_tag)::value;  // one gate row covers the wave's rows
#pragma unroll 4
        for (int r = rr; r < WT_M; r += RPI_EP) {
          ResidT res{};
          float4 gv = g4c;
          if constexpr (GMODE != 0) {
            res = *reinterpret_cast<const ResidT*>(rbase + ((int64_t)r * epi.ldr + h * HALF_N) * resid_es);
            if constexpr (!GC) {
              const int64_t grow = gdiv == 1 ? (int64_t)(mrow0 + r) : (int64_t)(mrow0 + r) / gdiv;
              gv = *reinterpret_cast<const float4*>(epi.gate + grow * gstride + n);
            }
          }
          epi_row4<GMODE, OUTF32, ACT>(*reinterpret_cast<const float4*>(ep + r * PITCH + 4 * q), res, b4[0],
                                       b4[1], b4[2], b4[3], act, gv, cbase + (int64_t)r * ldc * (OUTF32 ? 4 : 2));
        }
      };
      using Const = std::true_type;
      using PerRow = std::integral_constant<bool, GMODE == 0>;  // GMODE 0 reads no gate
      if (act == 0 && gate_const) full_rows(std::integral_constant<int, 0>{}, Const{});
      else if (act == 0) full_rows(std::integral_constant<int, 0>{}, PerRow{});
      else if (GMODE == 0 && act == 1) full_rows(std::integral_constant<int, GMODE == 0 ? 1 : -1>{}, Const{});
      else if (GMODE == 0 && act == 2) full_rows(std::integral_constant<int, GMODE == 0 ? 2 : -1>{}, Const{});
      else full_rows(std::integral_constant<int, -1>{}, PerRow{});
    } else {
#pragma unroll 2
      for (int r = rr; r < WT_M; r += RPI_EP) {
        const int m = mrow0 + r;
        const float4 a4 = *reinterpret_cast<const float4*>(ep + r * PITCH + 4 * q);
        if (m < M && n < N) {
          float v[4] = {a4.x, a4.y, a4.z, a4.w};
          epilogue_store4<false>(v, m, n, N, epi, C, ldc, vec_ok);
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

// ---- skinny kernel (N <= 64: the gate-logit projections) ------------------------------------
//
// One workgroup per R rows x 32 columns, R = ceil(M / 256) (at least 16, at most 128), so that the
// rows spread evenly over the 256 CUs: the kernel is bound by each CU's operand stream, and 32-row
// workgroups (288 of them at 9216 rows) left 32 CUs with twice the rows of the others. The R rows
// are RB = ceil(R / 16) MFMA row blocks; rows past R or M re-read the last valid row (the same
// cache lines as its own lanes) and are not stored. The NWK waves split K into NWK slices and
// read both MFMA operands straight from global memory (the weight is a few hundred KB and stays
// in L2, each activation row is read once), then add their partial tiles through LDS. The products are
// 16x16x32 MFMAs: a 16-byte operand load then spans 16 rows (four lanes of 64 contiguous bytes per
// row) instead of the 32 rows of a 32x32x16 operand, which halves the cache lines each load
// instruction touches, the limit of this kernel.
// Quantized weights are dequantized in registers with the arithmetic of the other kernels.
template <int QB, int NWK, int RB, bool H = false>
__global__ __launch_bounds__(NWK * 64) void gemm_skinny_kernel(
    const uint16_t* __restrict__ A, int64_t lda, const uint16_t* __restrict__ W, int64_t ldw,
    QuantW qw, void* __restrict__ C, int64_t ldc, int M, int N, int K, int R, Epilogue epi) {
  __shared__ __attribute__((aligned(16))) float part[NWK][2 * RB * 4][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  const int m0 = blockIdx.x * R, n0 = blockIdx.y * 32;
  const int mend = min(m0 + R, M);
  // operand rows of this lane: activation rows m0 + 16 rb + l16 (clamped to the last valid row),
  // weight rows n0 + 16 cb + l16
  int wrow_i[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) wrow_i[b] = min(n0 + 16 * b + l16, N - 1);
  const uint16_t* arow[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) arow[b] = A + (int64_t)min(m0 + 16 * b + l16, mend - 1) * lda + 8 * lq;
  const int kq = K / NWK, kbeg = wave * kq;
  // accumulator (cb, rb): lane holds weight rows n0 + 16 cb + 4 lq + e, activation row m0 + 16 rb + l16
  f32x4 acc[2][RB];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[cb][rb][e] = 0.0f;
  auto wfrag = [&](int n, int k) -> bf16x8 {  // row n, this lane's 8 values start at k (k % 8 == 0)
    if constexpr (QB == 0) {
      return *reinterpret_cast<const bf16x8*>(W + (int64_t)n * ldw + k);
    } else if constexpr (QB == QMX8) {
      const float sc = e8m0_f32(qw.e8m0[(int64_t)n * (K / 32) + k / 32]);
      const uint32_t* wd = qw.words + (int64_t)n * (K / 4) + k / 4;
      uint32_t tmp[2] = {wd[0], wd[1]};
      return __builtin_bit_cast(bf16x8, dequant8<QMX8>(tmp, sc, 0.0f));
    } else {
      const int64_t g = (int64_t)n * (K / 64) + k / 64;
      const float sc = bf2f(qw.scales[g]), bi = bf2f(qw.biases[g]);
      const uint32_t* wd = qw.words + (int64_t)n * (K * QB / 32) + k * QB / 32;
      uint32_t tmp[2] = {wd[0], QB == 8 ? wd[1] : 0u};
      return __builtin_bit_cast(bf16x8, dequant8<QB>(tmp, sc, bi));
    }
  };
#pragma unroll 2
  for (int k = kbeg; k < kbeg + kq; k += 32) {
    const bf16x8 w0 = wfrag(wrow_i[0], k + 8 * lq), w1 = wfrag(wrow_i[1], k + 8 * lq);
    bf16x8 x[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) x[b] = *reinterpret_cast<const bf16x8*>(arow[b] + k);
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      acc[0][b] = mfma16x16x32<H>(w0, x[b], acc[0][b]);
      acc[1][b] = mfma16x16x32<H>(w1, x[b], acc[1][b]);
    }
  }
#pragma unroll
  for (int a = 0; a < 2 * RB; ++a)
#pragma unroll
    for (int e = 0; e < 4; ++e) part[wave][4 * a + e][lane] = acc[a / RB][a % RB][e];
  __syncthreads();
  // wave w finishes accumulators a = w, w + NWK, ...: (cb, rb) = (a / RB, a % RB), 4 consecutive
  // columns of one row per lane
  const bool vec_ok = (ldc % 4 == 0) && (!(epi.flags & KX_EPI_GATED_RESIDUAL) || epi.ldr % 4 == 0);
  for (int a = wave; a < 2 * RB; a += NWK) {
    const int cb = a / RB, rb = a % RB;
    const int row = m0 + 16 * rb + l16;
    const int col = n0 + 16 * cb + 4 * lq;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int p = 0; p < NWK; ++p)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += part[p][4 * a + e][lane];
    if (row < mend && col < N) epilogue_store4<H>(v, row, col, N, epi, C, ldc, vec_ok);
  }
}

// LDS-staged form for bf16 / fp16 weights and K % 256 == 0. The register form's 16-byte operand
// loads cover four lanes (64 bytes) of a row: every L1 -> L2 request is half a cache line, and the
// per-CU stream (requests in flight x latency) holds the activation read to ~2.4 TB/s. Here each
// wave streams its K quarter through a private ring of SKS stages in LDS: per stage its R
// activation rows and 32 weight rows x 64 K, DMA'd by buffer loads of 8 rows x 128 bytes (one
// full-line request per row), slots XOR-swizzled by (row >> 1) & 7 so that the 16-row fragment
// reads are conflict free. A wave only reads stages it copied itself, so the ring needs its own
// vmcnt waits and no barrier.
template <int A_I, bool H>
__global__ __launch_bounds__(256) void gemm_skinny_lds_kernel(
    const uint16_t* __restrict__ A, int64_t lda, const uint16_t* __restrict__ W, int64_t ldw,
    void* __restrict__ C, int64_t ldc, int M, int N, int K, int R, Epilogue epi) {
  constexpr int SKS = 3;                          // stages per wave ring
  constexpr int AROWS = A_I * 8;                  // activation rows per stage (R <= AROWS)
  constexpr int RB = (AROWS + 15) / 16;           // MFMA row blocks; rows past AROWS read the
                                                  // weight rows that follow (never stored)
  constexpr int W_I = 4;                          // weight DMA instructions per stage
  constexpr int STG = (AROWS + 32) * 128;         // bytes per stage
  constexpr int RING_W = SKS * STG;               // bytes per wave
  constexpr int PART = 4 * 2 * RB * 4 * 64 * 4;   // partial tiles of the 4 waves
  constexpr int SMEM = 4 * RING_W > PART ? 4 * RING_W : PART;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[SMEM];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  const int m0 = blockIdx.x * R, n0 = blockIdx.y * 32;
  const int mend = min(m0 + R, M);
  uint8_t* ring = smem + wave * RING_W;
  // DMA lanes: row lane / 8 of the instruction's 8, 16-byte slot lane % 8 (global chunk slot ^ swz)
  const int r8 = lane >> 3, slot = lane & 7;
  const int kq = K / 4, kbeg = wave * kq, nst = kq / 64;
  uint32_t av[A_I], wv[W_I];
#pragma unroll
  for (int i = 0; i < A_I; ++i) {
    const int r = 8 * i + r8;
    av[i] = (uint32_t)(((int64_t)(min(m0 + r, mend - 1) - m0) * lda + kbeg + 8 * (slot ^ ((r >> 1) & 7))) * 2);
  }
#pragma unroll
  for (int i = 0; i < W_I; ++i) {
    const int r = 8 * i + r8;
    wv[i] = (uint32_t)(((int64_t)(min(n0 + r, N - 1) - n0) * ldw + kbeg + 8 * (slot ^ ((r >> 1) & 7))) * 2);
  }
  const rsrc_t a_rsrc = raw_rsrc(A + (int64_t)m0 * lda), w_rsrc = raw_rsrc(W + (int64_t)n0 * ldw);
  auto issue = [&](int st) {  // stage st of this wave's K quarter (clamped: re-reads the last)
    uint8_t* buf = ring + (st % SKS) * STG;
    const uint32_t ko = (uint32_t)(min(st, nst - 1) * 64 * 2);
#pragma unroll
    for (int i = 0; i < A_I; ++i) buffer_lds16(a_rsrc, buf + i * 1024, av[i], ko);
#pragma unroll
    for (int i = 0; i < W_I; ++i) buffer_lds16(w_rsrc, buf + AROWS * 128 + i * 1024, wv[i], ko);
  };
  // fragment offsets: row r, 16-byte chunk c = 4 h + lq of k32 half h
  int fo[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) fo[h] = l16 * 128 + (((4 * h + lq) ^ ((l16 >> 1) & 7)) << 4);
  f32x4 acc[2][RB];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[cb][rb][e] = 0.0f;
#pragma unroll
  for (int st = 0; st < SKS - 1; ++st) issue(st);
  for (int st = 0; st < nst; ++st) {
    // stage st landed (stage st + 1 may still be in flight)
    wait_vmcnt<(SKS - 2) * (A_I + W_I)>();
    const uint8_t* buf = ring + (st % SKS) * STG;
    bf16x8 wf[2][2], xf[2][RB];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // 16-row blocks are 2 KB apart; the swizzle depends on the row within its block only
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
        wf[h][cb] = *reinterpret_cast<const bf16x8*>(buf + AROWS * 128 + cb * 2048 + fo[h]);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) xf[h][rb] = *reinterpret_cast<const bf16x8*>(buf + rb * 2048 + fo[h]);
    }
    wait_lgkmcnt0();
    // the slot of stage st + SKS - 1 is stage st - 1's: read out one iteration ago
    issue(st + SKS - 1);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        acc[0][rb] = mfma16x16x32<H>(wf[h][0], xf[h][rb], acc[0][rb]);
        acc[1][rb] = mfma16x16x32<H>(wf[h][1], xf[h][rb], acc[1][rb]);
      }
  }
  wait_vmcnt<0>();
  __syncthreads();
  float* part = reinterpret_cast<float*>(smem);  // [wave][2 RB * 4][64]
#pragma unroll
  for (int a = 0; a < 2 * RB; ++a)
#pragma unroll
    for (int e = 0; e < 4; ++e) part[(wave * 2 * RB * 4 + 4 * a + e) * 64 + lane] = acc[a / RB][a % RB][e];
  __syncthreads();
  const bool vec_ok = (ldc % 4 == 0) && (!(epi.flags & KX_EPI_GATED_RESIDUAL) || epi.ldr % 4 == 0);
  for (int a = wave; a < 2 * RB; a += 4) {
    const int cb = a / RB, rb = a % RB;
    const int row = m0 + 16 * rb + l16;
    const int col = n0 + 16 * cb + 4 * lq;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += part[(p * 2 * RB * 4 + 4 * a + e) * 64 + lane];
    if (row < mend && col < N) epilogue_store4<H>(v, row, col, N, epi, C, ldc, vec_ok);
  }
}

template <bool H, int AI>
void launch_skinny_lds_ai(const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, void* c, int64_t ldc,
                          int m, int n, int k, int r, const Epilogue& epi, hipStream_t s) {
  const dim3 grid((unsigned)((m + r - 1) / r), (unsigned)((n + 31) / 32));
  gemm_skinny_lds_kernel<AI, H><<<grid, 256, 0, s>>>(a, lda, w, ldw, c, ldc, m, n, k, r, epi);
}

// Rows per skinny workgroup (see above) and its launch.
template <int QB, bool H, int RB>
void launch_skinny_rb(const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, QuantW qw, void* c,
                      int64_t ldc, int m, int n, int k, int r, const Epilogue& epi, hipStream_t s) {
  const dim3 grid((unsigned)((m + r - 1) / r), (unsigned)((n + 31) / 32));
  gemm_skinny_kernel<QB, 4, RB, H><<<grid, 256, 0, s>>>(a, lda, w, ldw, qw, c, ldc, m, n, k, r, epi);
}

template <int QB, bool H>
void launch_skinny(const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, QuantW qw, void* c,
                   int64_t ldc, int m, int n, int k, const Epilogue& epi, hipStream_t s) {
  if (QB == 0 && k % 256 == 0 && lda <= (1 << 22) && ldw <= (1 << 22)) {
    // rows per workgroup: the rows spread over the 256 CUs in the fewest rounds of at most 64
    // rows (at least 16)
    const int per_cu = (m + 255) / 256, rounds = (per_cu + 63) / 64;
    const int r = std::max((m + 256 * rounds - 1) / (256 * rounds), 16);
    switch ((r + 7) / 8) {
      case 2: return launch_skinny_lds_ai<H, 2>(a, lda, w, ldw, c, ldc, m, n, k, r, epi, s);
      case 3: return launch_skinny_lds_ai<H, 3>(a, lda, w, ldw, c, ldc, m, n, k, r, epi, s);
      case 4: return launch_skinny_lds_ai<H, 4>(a, lda, w, ldw, c, ldc, m, n, k, r, epi, s);
      case 5: return launch_skinny_lds_ai<H, 5>(a, lda, w, ldw, c, ldc, m, n, k, r, epi, s);
      case 6: return launch_skinny_lds_ai<H, 6>(a, lda, w, ldw, c, ldc, m, n, k, r, epi, s);
      case 7: return launch_skinny_lds_ai<H, 7>(a, lda, w, ldw, c, ldc, m, n, k, r, epi, s);
      default: return launch_skinny_lds_ai<H, 8>(a, lda, w, ldw, c, ldc, m, n, k, r, epi, s);
    }
  }
  const int r = std::min(std::max((m + 255) / 256, 16), 128);
  switch ((r + 15) / 16) {
    case 1: return launch_skinny_rb<QB, H, 1>(a, lda, w, ldw, qw, c, ldc, m, n, k, r, epi, s);
    case 2: return launch_skinny_rb<QB, H, 2>(a, lda, w, ldw, qw, c, ldc, m, n, k, r, epi, s);
    case 3: return launch_skinny_rb<QB, H, 3>(a, lda, w, ldw, qw, c, ldc, m, n, k, r, epi, s);
    case 4: return launch_skinny_rb<QB, H, 4>(a, lda, w, ldw, qw, c, ldc, m, n, k, r, epi, s);
    case 5:
    case 6: return launch_skinny_rb<QB, H, 6>(a, lda, w, ldw, qw, c, ldc, m, n, k, r, epi, s);
    default: return launch_skinny_rb<QB, H, 8>(a, lda, w, ldw, qw, c, ldc, m, n, k, r, epi, s);
  }
}

// ---- dispatch ---------------------------------------------------------------------------------

enum TileCfg { T256x256 = 0, T256x128 = 1, T128x128 = 2, T64x64 = 3, T128x64 = 4 };

template <int BM, int BN, int WM, int WN, int QB, bool H = false>
int launch_cfg(const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, QuantW qw,
               void* c, int64_t ldc, int m, int n, int k, const Epilogue& epi,
               hipStream_t s) {
  const int tiles = ((m + BM - 1) / BM) * ((n + BN - 1) / BN);
  gemm_kernel<BM, BN, WM, WN, QB, H><<<tiles, WM * WN * 64, 0, s>>>(a, lda, w, ldw, qw, c, ldc, m, n,
                                                                k, epi);
  return KX_OK;
}

int pick_cfg(int64_t m, int64_t n) {
  const char* env = getenv("KX355_GEMM_TILE");
  if (env && *env) {
    const int v = atoi(env);
    if (v >= 0 && v <= 4) return v;
  }
  if (m < 512 || n < 512) return (m * n >= 256 * 1024) ? T128x64 : T64x64;
  // Prefer the largest tile whose last wave of workgroups keeps the 256 CUs mostly busy.
  auto eff = [](int64_t tiles) {
    const int64_t waves = (tiles + 255) / 256;
    return (double)tiles / (double)(waves * 256);
  };
  const int64_t t256 = ((m + 255) / 256) * ((n + 255) / 256);
  const int64_t t128 = ((m + 255) / 256) * ((n + 127) / 128);
  if (eff(t256) >= 0.85) return T256x256;
  if (eff(t128) >= 0.85 || t128 >= 1024) return T256x128;
  return T128x128;
}

template <int BM, int QB, bool TL, int GMODE, bool OUTF32>
void launch_lds_t(const uint16_t* a, int64_t lda, QuantW qw, void* c, int64_t ldc, int m, int n, int k,
                  const Epilogue& epi, hipStream_t s) {
  const int tiles = ((m + BM - 1) / BM) * ((n + 255) / 256);
  Epilogue e = epi;
  e.rows_desc = rows_last_first(m, k);
  gemm_lds_kernel<BM, 256, QB, TL, GMODE, OUTF32><<<tiles, 256, 0, s>>>(a, lda, qw, c, ldc, m, n, k, e);
}

// Residual mode (none / bf16 / fp32) and output type select the epilogue specialisation.
template <int BM, int QB, bool TL = false>
void launch_lds(const uint16_t* a, int64_t lda, QuantW qw, void* c, int64_t ldc, int m, int n, int k,
                const Epilogue& epi, hipStream_t s) {
  const int gmode = (epi.flags & KX_EPI_GATED_RESIDUAL) ? ((epi.flags & KX_EPI_RESID_F32) ? 2 : 1) : 0;
  const bool out32 = epi.flags & KX_EPI_OUT_F32;
  switch (gmode * 2 + (out32 ? 1 : 0)) {
    case 0: return launch_lds_t<BM, QB, TL, 0, false>(a, lda, qw, c, ldc, m, n, k, epi, s);
    case 1: return launch_lds_t<BM, QB, TL, 0, true>(a, lda, qw, c, ldc, m, n, k, epi, s);
    case 2: return launch_lds_t<BM, QB, TL, 1, false>(a, lda, qw, c, ldc, m, n, k, epi, s);
    case 3: return launch_lds_t<BM, QB, TL, 1, true>(a, lda, qw, c, ldc, m, n, k, epi, s);
    case 4: return launch_lds_t<BM, QB, TL, 2, false>(a, lda, qw, c, ldc, m, n, k, epi, s);
    default: return launch_lds_t<BM, QB, TL, 2, true>(a, lda, qw, c, ldc, m, n, k, epi, s);
  }
}

// Tile height of the quantized direct-to-LDS kernel (256-wide tiles): the fewest rounds of 256
// workgroups times their rows (KX355_GEMM_LDS_TILE = 0 / 1 forces 256 / 192).
bool quantized_tall(int64_t m, int64_t n) {
  const char* env = getenv("KX355_GEMM_LDS_TILE");
  if (env && (env[0] == '0' || env[0] == '1')) return env[0] == '0';
  const int64_t t256 = ((m + 255) / 256) * ((n + 255) / 256), t192 = ((m + 191) / 192) * ((n + 255) / 256);
  return (t256 + 255) / 256 * 256 <= (t192 + 255) / 256 * 192;
}

template <int QB, bool H = false>
int dispatch(const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, QuantW qw,
             void* c, int64_t ldc, int64_t m, int64_t n, int64_t k, const Epilogue& epi,
             hipStream_t s) {
  const char* legacy = getenv("KX355_GEMM_TILE");
  const bool use_legacy = legacy && *legacy;
  if (QB == 0 && m <= FEW_ROWS && !use_legacy) {
    launch_few_rows(H, a, lda, w, ldw, c, ldc, (int)m, (int)n, (int)k, epi, s);
    return KX_OK;
  }
  if (n <= 64 && k % 128 == 0 && !use_legacy) {
    launch_skinny<QB, H>(a, lda, w, ldw, qw, c, ldc, (int)m, (int)n, (int)k, epi, s);
    return KX_OK;
  }
  // the direct-to-LDS kernels keep per-lane 32-bit byte offsets within a 256-row tile
  if (QB == 0 && k % DENSE_BK == 0 && lda <= (1 << 22) && ldw <= (1 << 22) && !use_legacy) {
    launch_dense(H, a, lda, w, ldw, c, ldc, (int)m, (int)n, (int)k, epi, s);
    return KX_OK;
  }
  // quantized weights: the direct-to-LDS kernel with in-LDS dequantization needs whole 128-wide
  // K blocks (scale / bias pairs of two groups), 16-byte aligned packed rows and 4-byte aligned
  // scale / bias rows; tile 2 (or a narrow N) selects the register-staged kernel
  // (a few hundred rows leave most CUs idle with its 192 / 256-row tiles: they take the
  // register-staged kernel's small tiles instead)
  const bool sb_aligned = QB == QMX8 ? (reinterpret_cast<uintptr_t>(qw.e8m0) & 3) == 0
                                     : (reinterpret_cast<uintptr_t>(qw.scales) & 3) == 0 &&
                                           (reinterpret_cast<uintptr_t>(qw.biases) & 3) == 0;
  if (QB != 0 && k % 128 == 0 && lda <= (1 << 22) && n >= 128 && m >= 512 && !use_legacy &&
      aligned16(qw.words) && sb_aligned) {
    const char* env = getenv("KX355_GEMM_LDS_TILE");
    if (!env || env[0] != '2') {
      if constexpr (QB != 0) {
        if (quantized_tall(m, n)) launch_lds<256, QB>(a, lda, qw, c, ldc, (int)m, (int)n, (int)k, epi, s);
        else launch_lds<192, QB>(a, lda, qw, c, ldc, (int)m, (int)n, (int)k, epi, s);
      }
      return KX_OK;
    }
  }
  switch (pick_cfg(m, n)) {
    case T256x256:
      return launch_cfg<256, 256, 2, 2, QB, H>(a, lda, w, ldw, qw, c, ldc, (int)m, (int)n, (int)k,
                                            epi, s);
    case T256x128:
      return launch_cfg<256, 128, 2, 2, QB, H>(a, lda, w, ldw, qw, c, ldc, (int)m, (int)n, (int)k,
                                            epi, s);
    case T128x128:
      return launch_cfg<128, 128, 2, 2, QB, H>(a, lda, w, ldw, qw, c, ldc, (int)m, (int)n, (int)k,
                                            epi, s);
    case T128x64:
      return launch_cfg<128, 64, 2, 2, QB, H>(a, lda, w, ldw, qw, c, ldc, (int)m, (int)n, (int)k,
                                           epi, s);
    default:
      return launch_cfg<64, 64, 2, 2, QB, H>(a, lda, w, ldw, qw, c, ldc, (int)m, (int)n, (int)k, epi,
                                          s);
  }
}

// Split-K reduction: c = epilogue(sum over the planes of the fp32 partial products), 4 columns
// of one row per thread (the planes are (M, N) fp32, N a multiple of 4).
template <bool H>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ parts, int splits,
                                                            int M, int N, void* __restrict__ C, int64_t ldc,
                                                            Epilogue epi, bool vec_ok) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per_row = N / 4;
  if (idx >= (int64_t)M * per_row) return;
  const int m = (int)(idx / per_row), n = (int)(idx - m * per_row) * 4;
  const int64_t plane = (int64_t)M * N;
  float4 acc = *reinterpret_cast<const float4*>(parts + (int64_t)m * N + n);
  for (int y = 1; y < splits; ++y) {
    const float4 p = *reinterpret_cast<const float4*>(parts + y * plane + (int64_t)m * N + n);
    acc.x += p.x;
    acc.y += p.y;
    acc.z += p.z;
    acc.w += p.w;
  }
  float v[4] = {acc.x, acc.y, acc.z, acc.w};
  epilogue_store4<H>(v, m, n, N, epi, C, ldc, vec_ok);
}

// Tiled affine weights: for 256-row tile nb and 32-wide K stage kb, the rows' packed bytes of the
// stage are one block of 256 * (32 * bits / 8) bytes; for the 128-wide window p, the rows'
// (scale 2p, scale 2p+1, bias 2p, bias 2p+1) are one block of 256 * 8 bytes. Rows past n repeat
// row n - 1 (their products are never stored).
template <int BITS>
__global__ __launch_bounds__(256) void tile_weights_kernel(const uint32_t* __restrict__ words,
                                                           const uint16_t* __restrict__ scales,
                                                           const uint16_t* __restrict__ biases,
                                                           uint8_t* __restrict__ wt, uint8_t* __restrict__ sbt,
                                                           int64_t n, int64_t k) {
  constexpr int QROW = 32 * BITS / 8;
  const int64_t npad = (n + 255) / 256 * 256;
  const int64_t kb_count = k / 32, p_count = k / 128;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t rows_x_kb = npad * kb_count;
  if (idx < rows_x_kb) {
    const int64_t r = idx % npad, kb = idx / npad;  // consecutive threads: consecutive rows
    const int64_t src_row = r < n ? r : n - 1;
    const uint32_t* src = words + src_row * (k * BITS / 32) + kb * (QROW / 4);
    uint32_t* dst = reinterpret_cast<uint32_t*>(wt + (((r / 256) * kb_count + kb) * 256 + (r % 256)) * QROW);
#pragma unroll
    for (int j = 0; j < QROW / 4; ++j) dst[j] = src[j];
  }
  if (idx < npad * p_count) {
    const int64_t r = idx % npad, p = idx / npad;
    const int64_t src_row = r < n ? r : n - 1;
    const int64_t g = src_row * (k / 64) + 2 * p;
    uint16_t* dst = reinterpret_cast<uint16_t*>(sbt + (((r / 256) * p_count + p) * 256 + (r % 256)) * 8);
    dst[0] = scales[g];
    dst[1] = scales[g + 1];
    dst[2] = biases[g];
    dst[3] = biases[g + 1];
  }
}

int check_epilogue(const char* name, int epilogue, const void* bias, const void* c,
                   int64_t ldc, const void* resid, int64_t ldr, int64_t n, const float* gate,
                   int64_t gate_div, int64_t gate_stride) {
  const int act = (epilogue >> 4) & 15;
  const int known = KX_EPI_BIAS | (15 << 4) | KX_EPI_GATED_RESIDUAL | KX_EPI_RESID_F32 |
                    KX_EPI_OUT_F32;
  KX_REQUIRE((epilogue & ~known) == 0 && act <= 4, "%s: bad epilogue flags %d", name, epilogue);
  KX_REQUIRE(!(epilogue & KX_EPI_BIAS) || (bias && aligned8(bias)), "%s: bias missing or unaligned",
             name);
  KX_REQUIRE(!(epilogue & KX_EPI_OUT_F32) || (aligned16(c) && ldc % 4 == 0),
             "%s: an fp32 output needs 16-byte aligned rows", name);
  KX_REQUIRE(!(epilogue & KX_EPI_RESID_F32) || (epilogue & KX_EPI_GATED_RESIDUAL),
             "%s: KX_EPI_RESID_F32 without a gated residual", name);
  if (epilogue & KX_EPI_GATED_RESIDUAL) {
    KX_REQUIRE(resid && gate && ldr >= n && gate_div > 0 && gate_stride >= 0,
               "%s: gated residual needs resid, ldr >= n and gate rows", name);
    KX_REQUIRE(aligned16(gate) && gate_stride % 4 == 0, "%s: gate must be 16-byte aligned", name);
    if (epilogue & KX_EPI_RESID_F32)
      KX_REQUIRE(aligned16(resid) && ldr % 4 == 0, "%s: an fp32 residual needs 16-byte aligned rows",
                 name);
    else
      KX_REQUIRE(aligned8(resid), "%s: resid must be 8-byte aligned", name);
  }
  return KX_OK;
}

}  // namespace
}  // namespace kx

using namespace kx;

namespace {
template <bool H>
int gemm_entry(const void* a, int64_t lda, const void* w, int64_t ldw, const void* bias, void* c, int64_t ldc,
               int64_t m, int64_t n, int64_t k, int epilogue, const void* resid, int64_t ldr, const float* gate,
               int64_t gate_div, int64_t gate_stride, hipStream_t s) {
  const char* what = ename<H>("kx_gemm_bf16", "kx_gemm_f16");
  KX_REQUIRE(a && w && c, "%s: null tensor", what);
  KX_REQUIRE(m >= 0 && n >= 0 && k > 0 && m < (1ll << 31) && n < (1ll << 31) && k < (1ll << 30),
             "%s: bad shape (%lld, %lld, %lld)", what, (long long)m, (long long)n, (long long)k);
  KX_REQUIRE(k % 8 == 0 && lda % 8 == 0 && ldw % 8 == 0 && lda >= k && ldw >= k && ldc >= n,
             "%s: k, lda and ldw must be multiples of 8 (k=%lld lda=%lld ldw=%lld)", what, (long long)k,
             (long long)lda, (long long)ldw);
  KX_REQUIRE(aligned16(a) && aligned16(w) && aligned8(c), "%s: a/w must be 16-byte and c 8-byte aligned", what);
  const int rc = check_epilogue(what, epilogue, bias, c, ldc, resid, ldr, n, gate, gate_div, gate_stride);
  if (rc) return rc;
  if (m == 0 || n == 0) return KX_OK;
  const Epilogue epi{(const uint16_t*)bias, resid, ldr, gate, gate_div, gate_stride, epilogue};
  dispatch<0, H>((const uint16_t*)a, lda, (const uint16_t*)w, ldw, QuantW{}, c, ldc, m, n, k, epi, s);
  return check_launch(what);
}
}  // namespace

extern "C" int kx_gemm_bf16(const void* a, int64_t lda, const void* w, int64_t ldw, const void* bias, void* c,
                            int64_t ldc, int64_t m, int64_t n, int64_t k, int epilogue, const void* resid,
                            int64_t ldr, const float* gate, int64_t gate_div, int64_t gate_stride,
                            kx_stream_t stream) {
  return gemm_entry<false>(a, lda, w, ldw, bias, c, ldc, m, n, k, epilogue, resid, ldr, gate, gate_div, gate_stride,
                           (hipStream_t)stream);
}

extern "C" int kx_gemm_f16(const void* a, int64_t lda, const void* w, int64_t ldw, const void* bias, void* c,
                           int64_t ldc, int64_t m, int64_t n, int64_t k, int epilogue, const void* resid,
                           int64_t ldr, const float* gate, int64_t gate_div, int64_t gate_stride,
                           kx_stream_t stream) {
  return gemm_entry<true>(a, lda, w, ldw, bias, c, ldc, m, n, k, epilogue, resid, ldr, gate, gate_div, gate_stride,
                          (hipStream_t)stream);
}

namespace {
// The column forms' shared entry: query / key heads of head_dim columns normalized and rotated, the
// columns from swiglu_begin on a SwiGLU pair written to c2.
int gemm_columns(const char* what, const void* a, int64_t lda, const void* w, int64_t ldw, const void* bias, void* c,
                 int64_t ldc, int64_t m, int64_t n, int64_t k, int64_t q_end, int64_t k_end, int64_t head_dim,
                 const void* norm_q, const void* norm_k, int norm_dtype, float eps, float weight_offset,
                 const float* cos, const float* sin, int64_t table_ld, int64_t table_hs, int64_t table_rows,
                 int64_t table_bs, int64_t swiglu_begin, void* c2, int64_t ldc2, hipStream_t s) {
  KX_REQUIRE(a && w && (c || swiglu_begin == 0) && (c2 || swiglu_begin == n), "%s: null tensor", what);
  KX_REQUIRE(k_end == 0 || (norm_q && norm_k && cos && sin), "%s: null tensor", what);
  KX_REQUIRE(m >= 0 && n > 0 && k > 0 && m < (1ll << 31) && n < (1ll << 31) && k < (1ll << 30) &&
                 k % DENSE_BK == 0,
             "%s: bad shape (m=%lld n=%lld k=%lld; k %% 64 == 0)", what, (long long)m, (long long)n, (long long)k);
  KX_REQUIRE(head_dim == 64 || head_dim == 128, "%s: head_dim must be 64 or 128, got %lld", what, (long long)head_dim);
  KX_REQUIRE(q_end >= 0 && q_end % 128 == 0 && k_end >= q_end && k_end % 128 == 0 && k_end <= swiglu_begin,
             "%s: the query and key columns must be whole 128-wide heads inside n (q_end=%lld k_end=%lld)", what,
             (long long)q_end, (long long)k_end);
  KX_REQUIRE(swiglu_begin >= 0 && swiglu_begin <= n &&
                 (swiglu_begin == n || (swiglu_begin % 256 == 0 && (n - swiglu_begin) % 256 == 0)),
             "%s: the SwiGLU columns must start at a multiple of 256 and be a multiple of 256 (begin=%lld n=%lld)",
             what, (long long)swiglu_begin, (long long)n);
  KX_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && lda >= k && ldw >= k && lda <= (1 << 22) && ldw <= (1 << 22) &&
                 (swiglu_begin == 0 || (ldc >= swiglu_begin && ldc % 4 == 0)) &&
                 (swiglu_begin == n || (ldc2 >= (n - swiglu_begin) / 2 && ldc2 % 4 == 0)),
             "%s: bad strides", what);
  // a SwiGLU tile addresses its up rows from its gate rows with a 32-bit byte offset
  KX_REQUIRE(swiglu_begin == n || ((n - swiglu_begin) / 2 + 256) * ldw * 2 < (1ll << 32),
             "%s: SwiGLU weight rows are too far apart", what);
  KX_REQUIRE(aligned16(a) && aligned16(w) && aligned8(c) && aligned8(c2) && (!bias || aligned8(bias)),
             "%s: misaligned tensor", what);
  Epilogue epi{(const uint16_t*)bias, nullptr, 0, nullptr, 1, 0, bias ? KX_EPI_BIAS : 0};
  epi.sw_begin = swiglu_begin;
  epi.sw_width = (n - swiglu_begin) / 2;
  epi.c2 = c2;
  epi.ldc2 = ldc2;
  if (k_end > 0) {
    KX_REQUIRE(norm_dtype == KX_F32 || norm_dtype == KX_BF16, "%s: norm weights must be KX_F32 or KX_BF16", what);
    KX_REQUIRE(norm_dtype == KX_BF16 ? (aligned8(norm_q) && aligned8(norm_k))
                                     : (aligned16(norm_q) && aligned16(norm_k)),
               "%s: misaligned norm weights", what);
    KX_REQUIRE(aligned16(cos) && aligned16(sin) && table_ld % 4 == 0 && table_hs % 4 == 0 && table_bs % 4 == 0 &&
                   table_rows > 0 && table_rows < (1ll << 31),
               "%s: tables need 16-byte aligned rows (table_ld, table_hs, table_bs multiples of 4)", what);
    // the kernel indexes the tables with 32-bit offsets
    const int64_t heads = std::max(q_end, k_end - q_end) / head_dim;
    const int64_t last = (m > 0 ? (m - 1) / table_rows : 0) * table_bs + std::min(m, table_rows) * table_ld +
                         std::max<int64_t>(heads - 1, 0) * table_hs + head_dim;
    KX_REQUIRE(table_ld >= 0 && table_hs >= 0 && table_bs >= 0 && last < (1ll << 31),
               "%s: table offsets must be non-negative and below 2^31 elements", what);
    epi.nq = norm_q;
    epi.nk = norm_k;
    epi.n_bf16 = norm_dtype == KX_BF16;
    epi.head_dim = (int)head_dim;
    epi.n_eps = eps;
    epi.n_off = weight_offset;
    epi.q_end = q_end;
    epi.k_end = k_end;
    epi.cosp = cos;
    epi.sinp = sin;
    epi.t_ld = table_ld;
    epi.t_hs = table_hs;
    epi.t_rows = table_rows;
    epi.t_bs = table_bs;
    // division by the invariant table_rows (round-up method): shift = ceil(log2 d),
    // magic = floor(2^32 (2^shift - d) / d) + 1
    int shift = 0;
    while ((1ll << shift) < table_rows) ++shift;
    epi.t_shift = shift;
    epi.t_magic = (uint32_t)(((((unsigned __int128)1 << 32) * (uint64_t)((1ll << shift) - table_rows)) /
                              (uint64_t)table_rows) + 1);
  }
  if (m == 0) return KX_OK;
  launch_dense_columns((const uint16_t*)a, lda, (const uint16_t*)w, ldw, c, ldc, (int)m, (int)n, (int)k, epi, s);
  return check_launch(what);
}
}  // namespace

extern "C" int kx_gemm_qknorm_rope_bf16(const void* a, int64_t lda, const void* w, int64_t ldw, const void* bias,
                                        void* c, int64_t ldc, int64_t m, int64_t n, int64_t k, int64_t q_end,
                                        int64_t k_end, const void* norm_q, const void* norm_k, int norm_dtype,
                                        float eps, float weight_offset, const float* cos, const float* sin,
                                        int64_t table_ld, int64_t table_hs, int64_t table_rows, int64_t table_bs,
                                        kx_stream_t stream) {
  const char* what = "kx_gemm_qknorm_rope_bf16";
  KX_REQUIRE(c && norm_q && norm_k && cos && sin, "%s: null tensor", what);
  return gemm_columns(what, a, lda, w, ldw, bias, c, ldc, m, n, k, q_end, k_end, 128, norm_q, norm_k, norm_dtype, eps,
                      weight_offset, cos, sin, table_ld, table_hs, table_rows, table_bs, n, nullptr, 0,
                      (hipStream_t)stream);
}

extern "C" int kx_gemm_columns_bf16(const void* a, int64_t lda, const void* w, int64_t ldw, const void* bias, void* c,
                                    int64_t ldc, int64_t m, int64_t n, int64_t k, int64_t q_end, int64_t k_end,
                                    int64_t head_dim, const void* norm_q, const void* norm_k, int norm_dtype,
                                    float eps, float weight_offset, const float* cos, const float* sin,
                                    int64_t table_ld, int64_t table_hs, int64_t table_rows, int64_t table_bs,
                                    int64_t swiglu_begin, void* c2, int64_t ldc2, kx_stream_t stream) {
  return gemm_columns("kx_gemm_columns_bf16", a, lda, w, ldw, bias, c, ldc, m, n, k, q_end, k_end, head_dim, norm_q,
                      norm_k, norm_dtype, eps, weight_offset, cos, sin, table_ld, table_hs, table_rows, table_bs,
                      swiglu_begin, c2, ldc2, (hipStream_t)stream);
}

extern "C" int kx_qgemm_affine_bf16(const void* a, int64_t lda, const uint32_t* wq,
                                    const void* scales, const void* biases, const void* bias,
                                    void* c, int64_t ldc, int64_t m, int64_t n, int64_t k,
                                    int group_size, int bits, int epilogue, const void* resid,
                                    int64_t ldr, const float* gate, int64_t gate_div,
                                    int64_t gate_stride, kx_stream_t stream) {
  KX_REQUIRE(a && wq && scales && biases && c, "kx_qgemm_affine_bf16: null tensor");
  KX_REQUIRE(bits == 4 || bits == 8, "kx_qgemm_affine_bf16: bits must be 4 or 8, got %d", bits);
  KX_REQUIRE(group_size == 64, "kx_qgemm_affine_bf16: group_size must be 64, got %d", group_size);
  KX_REQUIRE(m >= 0 && n >= 0 && k > 0 && k % 64 == 0 && m < (1ll << 31) && n < (1ll << 31) &&
                 k < (1ll << 30),
             "kx_qgemm_affine_bf16: bad shape (k must be a multiple of 64)");
  KX_REQUIRE(lda % 8 == 0 && lda >= k && ldc >= n && aligned16(a) && aligned8(c),
             "kx_qgemm_affine_bf16: bad stride or alignment");
  const int rc = check_epilogue("kx_qgemm_affine_bf16", epilogue, bias, c, ldc, resid, ldr, n,
                                gate, gate_div, gate_stride);
  if (rc) return rc;
  if (m == 0 || n == 0) return KX_OK;
  const Epilogue epi{(const uint16_t*)bias, resid, ldr, gate, gate_div, gate_stride, epilogue};
  const QuantW qw{wq, (const uint16_t*)scales, (const uint16_t*)biases};
  if (bits == 4)
    dispatch<4>((const uint16_t*)a, lda, nullptr, 0, qw, c, ldc, m, n, k, epi, (hipStream_t)stream);
  else
    dispatch<8>((const uint16_t*)a, lda, nullptr, 0, qw, c, ldc, m, n, k, epi, (hipStream_t)stream);
  return check_launch("kx_qgemm_affine_bf16");
}

extern "C" int kx_dequant_affine_bf16(const uint32_t* wq, const void* scales, const void* biases,
                                      void* out, int64_t n, int64_t k, int group_size, int bits,
                                      kx_stream_t stream) {
  KX_REQUIRE(wq && scales && biases && out, "kx_dequant_affine_bf16: null tensor");
  KX_REQUIRE(bits == 4 || bits == 8, "kx_dequant_affine_bf16: bits must be 4 or 8");
  KX_REQUIRE(group_size > 0 && group_size % 8 == 0 && n >= 0 && k > 0 && k % group_size == 0,
             "kx_dequant_affine_bf16: k must be a multiple of group_size (a multiple of 8)");
  KX_REQUIRE(aligned16(out), "kx_dequant_affine_bf16: out must be 16-byte aligned");
  const int64_t total = n * (k / 8);
  if (total == 0) return KX_OK;
  const unsigned blocks = (unsigned)((total + 255) / 256);
  if (bits == 4)
    dequant_kernel<4><<<blocks, 256, 0, (hipStream_t)stream>>>(
        wq, (const uint16_t*)scales, (const uint16_t*)biases, (uint16_t*)out, n, k, group_size);
  else
    dequant_kernel<8><<<blocks, 256, 0, (hipStream_t)stream>>>(
        wq, (const uint16_t*)scales, (const uint16_t*)biases, (uint16_t*)out, n, k, group_size);
  return check_launch("kx_dequant_affine_bf16");
}

extern "C" int kx_qgemm_mxfp8_bf16(const void* a, int64_t lda, const uint32_t* wq, const void* scales,
                                   const void* bias, void* c, int64_t ldc, int64_t m, int64_t n, int64_t k,
                                   int group_size, int epilogue, const void* resid, int64_t ldr, const float* gate,
                                   int64_t gate_div, int64_t gate_stride, kx_stream_t stream) {
  const char* what = "kx_qgemm_mxfp8_bf16";
  KX_REQUIRE(a && wq && scales && c, "%s: null tensor", what);
  KX_REQUIRE(group_size == 32, "%s: group_size must be 32, got %d", what, group_size);
  KX_REQUIRE(m >= 0 && n >= 0 && k > 0 && k % 32 == 0 && m < (1ll << 31) && n < (1ll << 31) && k < (1ll << 30),
             "%s: bad shape (m=%lld n=%lld k=%lld; k must be a multiple of 32)", what, (long long)m, (long long)n,
             (long long)k);
  KX_REQUIRE(lda % 8 == 0 && lda >= k && ldc >= n && aligned16(a) && aligned8(c) && aligned8(wq),
             "%s: bad stride or alignment", what);
  const int rc = check_epilogue(what, epilogue, bias, c, ldc, resid, ldr, n, gate, gate_div, gate_stride);
  if (rc) return rc;
  if (m == 0 || n == 0) return KX_OK;
  const Epilogue epi{(const uint16_t*)bias, resid, ldr, gate, gate_div, gate_stride, epilogue};
  const QuantW qw{wq, nullptr, nullptr, (const uint8_t*)scales};
  dispatch<QMX8>((const uint16_t*)a, lda, nullptr, 0, qw, c, ldc, m, n, k, epi, (hipStream_t)stream);
  return check_launch(what);
}

extern "C" int kx_dequant_mxfp8_bf16(const uint32_t* wq, const void* scales, void* out, int64_t n, int64_t k,
                                     int group_size, int transposed, kx_stream_t stream) {
  const char* what = "kx_dequant_mxfp8_bf16";
  KX_REQUIRE(wq && scales && out, "%s: null tensor", what);
  KX_REQUIRE(group_size == 32, "%s: group_size must be 32, got %d", what, group_size);
  KX_REQUIRE(n >= 0 && k >= 0 && n < (1ll << 31) && k < (1ll << 31), "%s: bad shape", what);
  KX_REQUIRE(transposed ? (n % 32 == 0 && k % 8 == 0) : k % 32 == 0,
             "%s: the grouped axis must be a multiple of 32 (and k of 8 when transposed): n=%lld k=%lld", what,
             (long long)n, (long long)k);
  KX_REQUIRE(aligned16(out) && (transposed ? aligned16(wq) : aligned8(wq)), "%s: out (and wq) misaligned", what);
  if (n == 0 || k == 0) return KX_OK;
  hipStream_t s = (hipStream_t)stream;
  if (transposed) {
    const dim3 grid((unsigned)((n + 63) / 64), (unsigned)((k + 63) / 64));
    dequant_mx8_t_kernel<<<grid, 256, 0, s>>>(wq, (const uint8_t*)scales, (uint16_t*)out, n, k);
  } else {
    const int64_t total = n * (k / 8);
    dequant_mx8_kernel<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(wq, (const uint8_t*)scales, (uint16_t*)out,
                                                                       n, k);
  }
  return check_launch(what);
}

extern "C" int kx_dequant_fp4_bf16(const uint32_t* wq, const void* scales, void* out, int64_t n, int64_t k,
                                   int group_size, int scale_kind, kx_stream_t stream) {
  const char* what = "kx_dequant_fp4_bf16";
  KX_REQUIRE(wq && scales && out, "%s: null tensor", what);
  KX_REQUIRE(scale_kind == KX_FP4_MX || scale_kind == KX_FP4_NV, "%s: bad scale kind %d", what, scale_kind);
  const int gs = scale_kind == KX_FP4_NV ? 16 : 32;
  KX_REQUIRE(group_size == gs, "%s: group_size must be %d for this scale kind, got %d", what, gs, group_size);
  KX_REQUIRE(n >= 0 && k > 0 && k % gs == 0, "%s: k must be a multiple of the group size (n=%lld k=%lld)", what,
             (long long)n, (long long)k);
  KX_REQUIRE(aligned16(out), "%s: out must be 16-byte aligned", what);
  const int64_t total = n * (k / 8);
  KX_REQUIRE(total / 256 < (1ll << 31), "%s: too many elements", what);
  if (total == 0) return KX_OK;
  const unsigned grid = (unsigned)((total + 255) / 256);
  if (scale_kind == KX_FP4_NV)
    dequant_fp4_kernel<true><<<grid, 256, 0, (hipStream_t)stream>>>(wq, (const uint8_t*)scales, (uint16_t*)out, n, k);
  else
    dequant_fp4_kernel<false><<<grid, 256, 0, (hipStream_t)stream>>>(wq, (const uint8_t*)scales, (uint16_t*)out, n, k);
  return check_launch(what);
}

extern "C" int kx_qweight_tile_affine(const uint32_t* wq, const void* scales, const void* biases,
                                      void* wt, void* sbt, int64_t n, int64_t k, int group_size,
                                      int bits, kx_stream_t stream) {
  KX_REQUIRE(wq && scales && biases && wt && sbt, "kx_qweight_tile_affine: null tensor");
  KX_REQUIRE(bits == 4 || bits == 8, "kx_qweight_tile_affine: bits must be 4 or 8, got %d", bits);
  KX_REQUIRE(group_size == 64, "kx_qweight_tile_affine: group_size must be 64, got %d", group_size);
  KX_REQUIRE(n > 0 && k > 0 && k % 128 == 0 && n < (1ll << 31) && k < (1ll << 30),
             "kx_qweight_tile_affine: k must be a positive multiple of 128");
  KX_REQUIRE(aligned16(wt) && aligned8(sbt), "kx_qweight_tile_affine: wt must be 16-byte and sbt 8-byte aligned");
  const int64_t npad = (n + 255) / 256 * 256;
  const int64_t work = npad * (k / 32);
  const unsigned blocks = (unsigned)((work + 255) / 256);
  if (bits == 4)
    tile_weights_kernel<4><<<blocks, 256, 0, (hipStream_t)stream>>>(
        wq, (const uint16_t*)scales, (const uint16_t*)biases, (uint8_t*)wt, (uint8_t*)sbt, n, k);
  else
    tile_weights_kernel<8><<<blocks, 256, 0, (hipStream_t)stream>>>(
        wq, (const uint16_t*)scales, (const uint16_t*)biases, (uint8_t*)wt, (uint8_t*)sbt, n, k);
  return check_launch("kx_qweight_tile_affine");
}

extern "C" int kx_qgemm_affine_tiled_bf16(const void* a, int64_t lda, const void* wt, const void* sbt,
                                          const void* bias, void* c, int64_t ldc, int64_t m, int64_t n,
                                          int64_t k, int bits, int epilogue, const void* resid,
                                          int64_t ldr, const float* gate, int64_t gate_div,
                                          int64_t gate_stride, kx_stream_t stream) {
  KX_REQUIRE(a && wt && sbt && c, "kx_qgemm_affine_tiled_bf16: null tensor");
  KX_REQUIRE(bits == 4 || bits == 8, "kx_qgemm_affine_tiled_bf16: bits must be 4 or 8, got %d", bits);
  KX_REQUIRE(m >= 0 && n > 0 && k > 0 && k % 128 == 0 && m < (1ll << 31) && n < (1ll << 31) &&
                 k < (1ll << 30),
             "kx_qgemm_affine_tiled_bf16: bad shape (k must be a multiple of 128)");
  KX_REQUIRE(lda % 8 == 0 && lda >= k && lda <= (1 << 22) && ldc >= n && aligned16(a) && aligned8(c) &&
                 aligned16(wt) && aligned8(sbt),
             "kx_qgemm_affine_tiled_bf16: bad stride or alignment");
  const int rc = check_epilogue("kx_qgemm_affine_tiled_bf16", epilogue, bias, c, ldc, resid, ldr, n,
                                gate, gate_div, gate_stride);
  if (rc) return rc;
  if (m == 0) return KX_OK;
  const Epilogue epi{(const uint16_t*)bias, resid, ldr, gate, gate_div, gate_stride, epilogue};
  const QuantW qw{(const uint32_t*)wt, (const uint16_t*)sbt, nullptr};
  const bool tall = quantized_tall(m, n);
  hipStream_t s = (hipStream_t)stream;
  if (bits == 4) {
    if (tall) launch_lds<256, 4, true>((const uint16_t*)a, lda, qw, c, ldc, (int)m, (int)n, (int)k, epi, s);
    else launch_lds<192, 4, true>((const uint16_t*)a, lda, qw, c, ldc, (int)m, (int)n, (int)k, epi, s);
  } else {
    if (tall) launch_lds<256, 8, true>((const uint16_t*)a, lda, qw, c, ldc, (int)m, (int)n, (int)k, epi, s);
    else launch_lds<192, 8, true>((const uint16_t*)a, lda, qw, c, ldc, (int)m, (int)n, (int)k, epi, s);
  }
  return check_launch("kx_qgemm_affine_tiled_bf16");
}

namespace {

// Argument checks shared by the two split-K entry points (no GPU call).
int check_splitk(const char* what, const void* a, int64_t lda, const void* w, int64_t ldw, const void* bias,
                 void* c, int64_t ldc, int64_t m, int64_t n, int64_t k, int epilogue, const void* resid,
                 int64_t ldr, const float* gate, int64_t gate_div, int64_t gate_stride, int splits) {
  KX_REQUIRE(a && w && c, "%s: null tensor", what);
  KX_REQUIRE(splits >= 2 && splits <= 64, "%s: splits must be 2..64, got %d", what, splits);
  KX_REQUIRE(m > 0 && n > 0 && k > 0 && m < (1ll << 31) && n < (1ll << 31) && k < (1ll << 30) && n % 4 == 0 &&
                 k % (splits * DENSE_BK) == 0,
             "%s: bad shape (m=%lld n=%lld k=%lld; n %% 4 == 0, k %% (64 splits) == 0)", what, (long long)m,
             (long long)n, (long long)k);
  KX_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && lda >= k && ldw >= k && ldc >= n && lda <= (1 << 22) &&
                 ldw <= (1 << 22),
             "%s: bad strides", what);
  KX_REQUIRE(aligned16(a) && aligned16(w) && aligned8(c), "%s: a/w must be 16-byte and c 8-byte aligned", what);
  return check_epilogue(what, epilogue, bias, c, ldc, resid, ldr, n, gate, gate_div, gate_stride);
}

// Both passes of a split-K product on `parts` (splits * m * n floats): every slice writes all of its
// (m, n) plane before the reduction reads it, so `parts` needs no clearing between calls.
template <bool H>
int run_splitk(const char* what, const void* a, int64_t lda, const void* w, int64_t ldw, const void* bias,
               void* c, int64_t ldc, int64_t m, int64_t n, int64_t k, int epilogue, const void* resid,
               int64_t ldr, const float* gate, int64_t gate_div, int64_t gate_stride, float* parts, int splits,
               hipStream_t s) {
  launch_dense_slices(H, (const uint16_t*)a, lda, (const uint16_t*)w, ldw, parts, (int)m, (int)n, (int)k, splits, s);
  const Epilogue epi{(const uint16_t*)bias, resid, ldr, gate, gate_div, gate_stride, epilogue};
  const bool vec_ok = (ldc % 4 == 0) && (!(epilogue & KX_EPI_GATED_RESIDUAL) || ldr % 4 == 0);
  const int64_t threads = m * (n / 4);
  splitk_reduce_kernel<H><<<(unsigned)((threads + 255) / 256), 256, 0, s>>>(parts, splits, (int)m, (int)n, c, ldc, epi,
                                                                         vec_ok);
  return check_launch(what);
}

// The no-allocation variant's partial products: one static array per device (the HIP runtime
// places a copy on each device that loads this code object, for the life of the process). Host
// code never passes `scratch` itself to a kernel (on the host it names a stand-in, not a device
// address); it passes the device address hipGetSymbolAddress returns for the current device.
static __device__ __align__(256) float scratch[KX_SPLITK_SCRATCH_BYTES / 4];

constexpr int KX_MAX_DEVICES = 64;
std::mutex g_scratch_mutex;
float* g_scratch_ptr[KX_MAX_DEVICES] = {};

// The current device's address of `scratch`, looked up on the first call on that device (with the
// device current) and kept per device.
int scratch_address(const char* what, float** out) {
  int dev = -1;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return set_error(KX_ERR_LAUNCH, "%s: hipGetDevice failed: %s", what, hipGetErrorString(err));
  if (dev < 0 || dev >= KX_MAX_DEVICES) return set_error(KX_ERR_UNSUPPORTED, "%s: device %d out of range", what, dev);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess || !p)
      return set_error(KX_ERR_LAUNCH, "%s: hipGetSymbolAddress(scratch) failed on device %d: %s", what, dev,
                       hipGetErrorString(err));
    g_scratch_ptr[dev] = static_cast<float*>(p);
  }
  *out = g_scratch_ptr[dev];
  return KX_OK;
}

}  // namespace

namespace {
template <bool H>
int splitk_entry(const void* a, int64_t lda, const void* w, int64_t ldw, const void* bias, void* c, int64_t ldc,
                 int64_t m, int64_t n, int64_t k, int epilogue, const void* resid, int64_t ldr, const float* gate,
                 int64_t gate_div, int64_t gate_stride, void* workspace, int64_t workspace_bytes, int splits,
                 hipStream_t s) {
  const char* what = ename<H>("kx_gemm_splitk_bf16", "kx_gemm_splitk_f16");
  KX_REQUIRE(workspace, "%s: null tensor", what);
  const int rc = check_splitk(what, a, lda, w, ldw, bias, c, ldc, m, n, k, epilogue, resid, ldr, gate, gate_div,
                              gate_stride, splits);
  if (rc) return rc;
  KX_REQUIRE(aligned16(workspace), "%s: workspace must be 16-byte aligned", what);
  KX_REQUIRE(workspace_bytes >= (int64_t)splits * m * n * 4,
             "%s: workspace of %lld bytes is below splits * m * n * 4 = %lld", what, (long long)workspace_bytes,
             (long long)splits * m * n * 4);
  return run_splitk<H>(what, a, lda, w, ldw, bias, c, ldc, m, n, k, epilogue, resid, ldr, gate, gate_div,
                       gate_stride, static_cast<float*>(workspace), splits, s);
}
}  // namespace

#define KX_SPLITK_ENTRY(SUFFIX, H)                                                                                \
  extern "C" int kx_gemm_splitk_##SUFFIX(const void* a, int64_t lda, const void* w, int64_t ldw, const void* bias, \
                                         void* c, int64_t ldc, int64_t m, int64_t n, int64_t k, int epilogue,     \
                                         const void* resid, int64_t ldr, const float* gate, int64_t gate_div,     \
                                         int64_t gate_stride, void* workspace, int64_t workspace_bytes,           \
                                         int splits, kx_stream_t stream) {                                        \
    return splitk_entry<H>(a, lda, w, ldw, bias, c, ldc, m, n, k, epilogue, resid, ldr, gate, gate_div,          \
                           gate_stride, workspace, workspace_bytes, splits, (hipStream_t)stream);                \
  }

KX_SPLITK_ENTRY(bf16, false)
KX_SPLITK_ENTRY(f16, true)

extern "C" int kx_gemm_splits(int64_t m, int64_t n, int64_t k, int* splits) {
  KX_REQUIRE(splits, "kx_gemm_splits: null result");
  KX_REQUIRE(m >= 0 && n >= 0 && k > 0 && m < (1ll << 31) && n < (1ll << 31) && k < (1ll << 30),
             "kx_gemm_splits: bad shape (%lld, %lld, %lld)", (long long)m, (long long)n, (long long)k);
  *splits = m <= FEW_ROWS || n == 0 || n % 4 || k % DENSE_BK ? 1 : dense_splits(m, n, k);
  return KX_OK;
}

extern "C" int kx_gemm_kernels(int64_t m, int64_t n, int64_t k, int* count) {
  KX_REQUIRE(count, "kx_gemm_kernels: null result");
  KX_REQUIRE(m >= 0 && n >= 0 && k > 0 && m < (1ll << 31) && n < (1ll << 31) && k < (1ll << 30),
             "kx_gemm_kernels: bad shape (%lld, %lld, %lld)", (long long)m, (long long)n, (long long)k);
  if (m == 0 || n == 0) *count = 0;
  else *count = m <= FEW_ROWS || (n <= 64 && k % 128 == 0) || k % DENSE_BK ? 1 : dense_kernels(m, n, k);
  return KX_OK;
}

extern "C" int kx_gemm_splitk_noalloc_bf16(const void* a, int64_t lda, const void* w, int64_t ldw,
                                           const void* bias, void* c, int64_t ldc, int64_t m, int64_t n, int64_t k,
                                           int epilogue, const void* resid, int64_t ldr, const float* gate,
                                           int64_t gate_div, int64_t gate_stride, int splits, kx_stream_t stream) {
  const char* what = "kx_gemm_splitk_noalloc_bf16";
  const int rc = check_splitk(what, a, lda, w, ldw, bias, c, ldc, m, n, k, epilogue, resid, ldr, gate, gate_div,
                              gate_stride, splits);
  if (rc) return rc;
  KX_REQUIRE((int64_t)splits * m * n * 4 <= KX_SPLITK_SCRATCH_BYTES,
             "%s: splits * m * n * 4 = %lld bytes exceeds the %lld-byte static scratch", what,
             (long long)splits * m * n * 4, (long long)KX_SPLITK_SCRATCH_BYTES);
  float* parts = nullptr;
  const int arc = scratch_address(what, &parts);
  if (arc) return arc;
  return run_splitk<false>(what, a, lda, w, ldw, bias, c, ldc, m, n, k, epilogue, resid, ldr, gate, gate_div,
                           gate_stride, parts, splits, (hipStream_t)stream);
}
