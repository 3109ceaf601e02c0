// Dense bf16 / fp16 products on gfx950 MFMA: c[m, n] = epilogue(sum_k a[m, k] * w[n, k]), both
// operands K-contiguous, K % 64 == 0, fp32 accumulation in v_mfma_f32_16x16x32 (the weight tile is
// the MFMA A operand, so an accumulator lane holds one output row and 4 consecutive columns).
//
// Two kernels over one operand stream: tiles go from global memory straight into LDS by
// buffer_load_dwordx4 ... lds, 8 rows x 128 bytes (one full cache line per row and 64-wide K stage)
// per instruction, the 16-byte slots of a row XOR-swizzled by (row >> 1) & 7 so that the copies and
// the 16-row fragment reads are free of bank conflicts. Every tile sums K in the same order, so a
// product's bits do not depend on the tile that the dispatch picks.
//
// gemm_pp_kernel (256 x 256 and 128 x 256 tiles, 8 waves, two per SIMD): the matrix cores are the
// bound, and what kept them idle with one wave per SIMD was everything the wave itself issues
// between MFMAs (fragment reads, copies, waits). Here waves 0-3 and 4-7 form two groups, one wave of
// each per SIMD, that alternate: while one group runs a section of MFMAs from registers, the other
// reads the fragments of its next section from LDS and issues copies; a workgroup barrier swaps
// them. Measured at 9216 x 16384 x 4096: 809 us (1529 TFLOP/s) against 903 us for the one-wave-per-
// SIMD kernel it replaced (32x32x16 MFMAs, fragment reads between them) on the same card; with
// 32x32x16 MFMAs in this schedule 860 us (the 16x16x32 form's smaller accumulator traffic lets the
// power-limited clock rise), with four sections per stage instead of two 826 us.
#include <stdlib.h>

#include "gemm.h"

namespace kx {
namespace {

typedef __attribute__((ext_vector_type(4))) int i32x4;

// A raw buffer resource over 4 GiB from a 64-bit base.
__device__ __forceinline__ i32x4 buffer_of(const void* base) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  return (i32x4){(int)(uint32_t)a, (int)(uint32_t)(a >> 32), -1, 0x00020000};
}

// One 16-byte-per-lane buffer -> LDS copy (M0 holds the wave's LDS address). Inline assembly, so
// that the compiler's wait-count pass does not order the LDS reads after it: the kernels order the
// copies themselves (a vmcnt wait, then the workgroup barrier, before any wave reads them).
__device__ __forceinline__ void copy16(i32x4 rsrc, uint32_t voff, uint32_t soff, uint32_t lds) {
  asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(rsrc), "s"(soff), "{m0}"(lds)
               : "memory");
}
__device__ __forceinline__ uint32_t lds_address(const void* p) { return (uint32_t)(uintptr_t)KX_LDS(p); }

constexpr int PITCH = 132;  // staged epilogue row of 128 columns, floats (4 of padding)

// ---- the epilogue of a 128-column strip staged in LDS --------------------------------------------
// 32 lanes hold a row (4 columns each), THREADS / 32 rows at a time, NROW rows per thread.

// Rows mrow + rr + q * STEP of the strip at columns n .. n + 3 of this thread, all inside C: bias,
// activation, gated residual (its rows in `res`) and the store, with the activation fixed at
// compile time (a choice per value puts a chain of scalar branches around every value).
template <int GMODE>
using ResidOf = typename std::conditional<GMODE == 2, float4, uint2>::type;

template <bool H, int GMODE, bool OUTF32, int NROW, int STEP, int ACT, bool GC>
__device__ __forceinline__ void strip_rows(const float* st, int rr, int c4, int mrow, int n, const Epilogue& epi,
                                           const ResidOf<GMODE>* res, void* C, int64_t ldc) {
  float b[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (epi.flags & KX_EPI_BIAS) {
    const uint2 bb = *reinterpret_cast<const uint2*>(epi.bias + n);
    b[0] = e_lo<H>(bb.x); b[1] = e_hi<H>(bb.x); b[2] = e_lo<H>(bb.y); b[3] = e_hi<H>(bb.y);
  }
  const int act = (epi.flags >> 4) & 15;
  float4 g4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (GMODE != 0 && GC) g4 = *reinterpret_cast<const float4*>(epi.gate + ((mrow + epi.row0) / epi.gate_div) * epi.gate_stride + n);
  char* dst = reinterpret_cast<char*>(C) + ((int64_t)(mrow + rr) * ldc + n) * (OUTF32 ? 4 : 2);
#pragma unroll
  for (int q = 0; q < NROW; ++q) {
    const int r = rr + q * STEP;
    const float4 a4 = *reinterpret_cast<const float4*>(st + r * PITCH + c4);
    float v[4] = {a4.x + b[0], a4.y + b[1], a4.z + b[2], a4.w + b[3]};
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = act_c<ACT>(v[e], act);
    if constexpr (GMODE != 0) {
      float4 gv = g4;
      if constexpr (!GC)
        gv = *reinterpret_cast<const float4*>(epi.gate + ((mrow + r + epi.row0) / epi.gate_div) * epi.gate_stride + n);
      float rv[4];
      if constexpr (GMODE == 2) {
        rv[0] = res[q].x; rv[1] = res[q].y; rv[2] = res[q].z; rv[3] = res[q].w;
      } else {
        rv[0] = e_lo<H>(res[q].x); rv[1] = e_hi<H>(res[q].x); rv[2] = e_lo<H>(res[q].y); rv[3] = e_hi<H>(res[q].y);
      }
      v[0] = fmaf(gv.x, v[0], rv[0]);
      v[1] = fmaf(gv.y, v[1], rv[1]);
      v[2] = fmaf(gv.z, v[2], rv[2]);
      v[3] = fmaf(gv.w, v[3], rv[3]);
    }
    if constexpr (OUTF32) {
      *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
      uint2 o;
      o.x = e_pack2<H>(v[0], v[1]);
      o.y = e_pack2<H>(v[2], v[3]);
      *reinterpret_cast<uint2*>(dst) = o;
    }
    dst += (int64_t)STEP * ldc * (OUTF32 ? 4 : 2);
  }
}

// The residual of a strip's rows, loaded before the strip is staged: the loads are in flight
// together under the staging and its barrier.
template <int GMODE, int NROW, int STEP>
__device__ __forceinline__ void strip_resid(ResidOf<GMODE>* res, int row, int n, const Epilogue& epi) {
  const char* p = reinterpret_cast<const char*>(epi.resid) + ((int64_t)row * epi.ldr + n) * (GMODE == 2 ? 4 : 2);
#pragma unroll
  for (int q = 0; q < NROW; ++q)
    res[q] = *reinterpret_cast<const ResidOf<GMODE>*>(p + (int64_t)(q * STEP) * epi.ldr * (GMODE == 2 ? 4 : 2));
}

// A staged strip to memory: whole and aligned (`full`), or masked at the edges of C.
template <bool H, int GMODE, bool OUTF32, int NROW, int STEP>
__device__ __forceinline__ void strip_store(const float* st, int rr, int c4, int mrow, int n, int M, int N,
                                            const Epilogue& epi, bool full, bool vec_ok, const ResidOf<GMODE>* res,
                                            void* C, int64_t ldc) {
  if (full) {
    const int act = (epi.flags >> 4) & 15;
    constexpr int LAST = NROW * STEP - 1;
    const bool gc = GMODE == 0 || epi.gate_stride == 0 ||
                    (mrow + epi.row0) / epi.gate_div == (mrow + epi.row0 + LAST) / epi.gate_div;
#define KX_STRIP(ACT, GC) strip_rows<H, GMODE, OUTF32, NROW, STEP, ACT, GC>(st, rr, c4, mrow, n, epi, res, C, ldc)
    if constexpr (GMODE == 0) {
      if (act == 0) KX_STRIP(0, true);
      else if (act == 1) KX_STRIP(1, true);
      else if (act == 2) KX_STRIP(2, true);
      else KX_STRIP(-1, true);
    } else {
      if (act == 0 && gc) KX_STRIP(0, true);
      else if (act == 0) KX_STRIP(0, false);
      else KX_STRIP(-1, false);
    }
#undef KX_STRIP
    return;
  }
#pragma unroll 2
  for (int q = 0; q < NROW; ++q) {
    const int r = rr + q * STEP, m = mrow + r;
    const float4 a4 = *reinterpret_cast<const float4*>(st + r * PITCH + c4);
    if (m < M && n < N) {
      float v[4] = {a4.x, a4.y, a4.z, a4.w};
      epilogue_store4<H>(v, m, n, N, epi, C, ldc, vec_ok);
    }
  }
}

// The sum over the 16 (64-wide heads) or 32 (128-wide) lanes that hold a row's head.
__device__ __forceinline__ float head_sum(float v, bool wide) {
  v = row16_sum(v);
  if (wide) {
    // adds the neighbouring 16-lane row (lanes 0-15 with 16-31, 32-47 with 48-63)
    const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  return v;
}

// A strip of query or key heads: bias, one rounding to bf16 (the projection's), the weighted
// RMSNorm per head and the adjacent-pair rotation in fp32, each product of the rotation rounded
// before the sum (as the standalone norm + RoPE kernel does). Rows go GR at a time: their table rows
// are in flight together.
template <int NROW, int STEP>
__device__ __forceinline__ void strip_norm_rope(const float* st, int rr, int c4, int mrow, int n, int M,
                                                const Epilogue& epi, uint16_t* C, int64_t ldc) {
  constexpr int GR = 4;
  static_assert(NROW % GR == 0, "row groups");
  const bool isq = n < epi.q_end, wide = epi.head_dim == 128;
  const int col = isq ? n : n - (int)epi.q_end;
  const int d = wide ? col & 127 : col & 63, head = wide ? col >> 7 : col >> 6;
  const void* nw = isq ? epi.nq : epi.nk;
  float b[4] = {0.0f, 0.0f, 0.0f, 0.0f}, w[4];
  if (epi.flags & KX_EPI_BIAS) {
    const uint2 bb = *reinterpret_cast<const uint2*>(epi.bias + n);
    b[0] = lo_f(bb.x); b[1] = hi_f(bb.x); b[2] = lo_f(bb.y); b[3] = hi_f(bb.y);
  }
  if (epi.n_bf16) {
    const uint2 ww = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(nw) + d);
    w[0] = lo_f(ww.x); w[1] = hi_f(ww.x); w[2] = lo_f(ww.y); w[3] = hi_f(ww.y);
  } else {
    const float4 ww = *reinterpret_cast<const float4*>(static_cast<const float*>(nw) + d);
    w[0] = ww.x; w[1] = ww.y; w[2] = ww.z; w[3] = ww.w;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] += epi.n_off;
  const float* ct = epi.cosp + head * epi.t_hs + d;
  const float* sn = epi.sinp + head * epi.t_hs + d;
  const uint32_t t_rows = (uint32_t)epi.t_rows, t_bs = (uint32_t)epi.t_bs, t_ld = (uint32_t)epi.t_ld;
  const float inv_width = wide ? 1.0f / 128.0f : 1.0f / 64.0f;
#pragma unroll
  for (int g = 0; g < NROW; g += GR) {
    float4 c[GR], s[GR];
#pragma unroll
    for (int j = 0; j < GR; ++j) {
      // table row of output row m (a row past the end reads the last one's): m / t_rows by the
      // host's magic number (m < 2^31: umulhi(m, magic) + m fits 32 bits)
      const uint32_t m = (uint32_t)(min(mrow + rr + (g + j) * STEP, M - 1) + (int)epi.row0);
      const uint32_t seq = (__umulhi(m, epi.t_magic) + m) >> epi.t_shift;
      const uint32_t row = seq * t_bs + (m - seq * t_rows) * t_ld;  // < 2^31 (host check)
      c[j] = *reinterpret_cast<const float4*>(ct + row);
      s[j] = *reinterpret_cast<const float4*>(sn + row);
    }
#pragma unroll
    for (int j = 0; j < GR; ++j) {
      const int r = rr + (g + j) * STEP, m = mrow + r;
      const float4 a4 = *reinterpret_cast<const float4*>(st + r * PITCH + c4);
      const float v0 = bf2f(f2bf(a4.x + b[0])), v1 = bf2f(f2bf(a4.y + b[1]));
      const float v2 = bf2f(f2bf(a4.z + b[2])), v3 = bf2f(f2bf(a4.w + b[3]));
      const float ss = head_sum(fmaf(v3, v3, fmaf(v2, v2, fmaf(v1, v1, v0 * v0))), wide);
      const float inv = rsqrtf(ss * inv_width + epi.n_eps);
      const float x0 = v0 * inv * w[0], x1 = v1 * inv * w[1], x2 = v2 * inv * w[2], x3 = v3 * inv * w[3];
      float o[4];
      {
#pragma clang fp contract(off)
        const float p0 = x0 * c[j].x, q0 = (-x1) * s[j].x, p1 = x1 * c[j].y, q1 = x0 * s[j].y;
        const float p2 = x2 * c[j].z, q2 = (-x3) * s[j].z, p3 = x3 * c[j].w, q3 = x2 * s[j].w;
        o[0] = p0 + q0;
        o[1] = p1 + q1;
        o[2] = p2 + q2;
        o[3] = p3 + q3;
      }
      uint2 sv;
      sv.x = pack2(o[0], o[1]);
      sv.y = pack2(o[2], o[3]);
      if (m < M) *reinterpret_cast<uint2*>(C + (int64_t)m * ldc + n) = sv;
    }
  }
}

// silu(gate) * up of 4 columns of a row staged at g and u.
__device__ __forceinline__ uint2 swiglu4(const float* g, const float* u, const float* bg, const float* bu) {
  const float4 a = *reinterpret_cast<const float4*>(g), b = *reinterpret_cast<const float4*>(u);
  uint2 o;
  o.x = pack2(fast_silu(a.x + bg[0]) * (b.x + bu[0]), fast_silu(a.y + bg[1]) * (b.y + bu[1]));
  o.y = pack2(fast_silu(a.z + bg[2]) * (b.z + bu[2]), fast_silu(a.w + bg[3]) * (b.w + bu[3]));
  return o;
}
__device__ __forceinline__ void swiglu_bias(const Epilogue& epi, int ng, int nu, float* bg, float* bu) {
#pragma unroll
  for (int e = 0; e < 4; ++e) bg[e] = bu[e] = 0.0f;
  if (epi.flags & KX_EPI_BIAS) {
    const uint2 x = *reinterpret_cast<const uint2*>(epi.bias + ng);
    const uint2 y = *reinterpret_cast<const uint2*>(epi.bias + nu);
    bg[0] = lo_f(x.x); bg[1] = hi_f(x.x); bg[2] = lo_f(x.y); bg[3] = hi_f(x.y);
    bu[0] = lo_f(y.x); bu[1] = hi_f(y.x); bu[2] = lo_f(y.y); bu[3] = hi_f(y.y);
  }
}

// ---- 256 x 256 and 128 x 256 tiles ---------------------------------------------------------------
//
// Waves 2 (rows) x 4 (columns); the tile's rows and columns are two halves each, and a wave owns
// BM / 4 rows of each row half and 32 columns of each column half. A stage of K = 64 is two sections:
// P1 reads both weight halves and the first activation half and multiplies them, P2 reads the
// second activation half (the weight fragments stay in registers) and multiplies that. Per section:
//   [fragment reads, copies, waits] barrier [2 x 2 x 2 x JB MFMAs] barrier
// with the second group one barrier behind, so its reads run beside the first group's MFMAs.
// Copies: P1 of stage kt fills the activation halves of stage kt + NST - 1 (their slot's last reader
// was P2 of kt - 1), P2 the weight halves of kt + NST (read in P1 of kt). A group's reads have
// returned (lgkmcnt 0) before the barrier that lets the other group's copies over them start, and
// a copy is complete (vmcnt, the counts below) in every wave before the barrier ahead of its first
// read. Past the last stage the last one is copied again into slots that nobody reads, which
// keeps the loop free of branches and the counts uniform.
// LDS: 128 KB for two stages of 256 x 256; 144 KB for three of 128 x 256, whose sections are half as
// long and need the deeper prefetch.
//
// NS: the fused-projection column forms. SwiGLU column tiles pair 128 gate columns (first column
// half) with their 128 up columns (second half): the product of both leaves the tile as
// silu(gate) * up, half the stores, and the (m, 2 F) intermediate never exists.
template <int BM, int GMODE, bool OUTF32, bool NS, bool H>
__global__ __launch_bounds__(512, 2) void gemm_pp_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                         const uint16_t* __restrict__ W, int64_t ldw,
                                                         void* __restrict__ C, int64_t ldc, int M, int N, int K,
                                                         Epilogue epi) {
  constexpr int HA = BM / 2;                  // rows of an activation half
  constexpr int HAB = HA * 128, HWB = 16384;  // bytes of a half's stage
  constexpr int STAGE = 2 * HAB + 2 * HWB;
  constexpr int NST = BM == 256 ? 2 : 3;
  constexpr int AI = HA / 64, WI = 2;  // copies per wave and half
  constexpr int PER = 2 * AI + 2 * WI;
  constexpr int JB = HA / 32;  // 16-row blocks per wave and half
  constexpr int WAIT1 = (NST - 1) * PER, WAIT2 = AI + 2 * WI + (NST - 2) * PER;
  constexpr int STRIP = HA * PITCH;  // floats of a staged quadrant
  constexpr int SMEM = NST * STAGE > 2 * STRIP * 4 ? NST * STAGE : 2 * STRIP * 4;
  static_assert(!NS || (GMODE == 0 && !OUTF32 && !H), "the column forms: plain bf16 output");
  static_assert(WAIT1 < 64, "vmcnt");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[SMEM];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int l16 = lane & 15, lq = lane >> 4;
  if constexpr (GMODE == 0 && OUTF32) {
    // K slices (grid.y > 1): workgroup row y multiplies slice y (K is its length) into plane y
    const int64_t y = blockIdx.y;
    A += y * K;
    W += y * K;
    C = static_cast<float*>(C) + y * (int64_t)M * ldc;
  }
  const int tiles_m = (M + BM - 1) / BM;
  int plain_n = (N + 255) / 256, tiles_n = plain_n;
  if constexpr (NS) {
    plain_n = ((int)epi.sw_begin + 255) / 256;
    tiles_n = plain_n + (int)(epi.sw_width / 128);
  }
  int2 tile = lds_tile_of(blockIdx.x, tiles_m, tiles_n);
  if (epi.rows_desc) tile.x = tiles_m - 1 - tile.x;
  const int m0 = tile.x * BM;
  const bool swiglu = NS && tile.y >= plain_n;
  // first weight row of the tile, and the distance to its second column half's rows
  const int n0 = swiglu ? (int)epi.sw_begin + (tile.y - plain_n) * 128 : tile.y * 256;
  const int whalf = swiglu ? (int)epi.sw_width : 128;

  // copies: lane -> row lane / 8 of the instruction's 8 rows, slot lane % 8; rows past the end re-read
  // the last row (their results are never stored)
  const i32x4 abuf = buffer_of(A + (int64_t)m0 * lda), wbuf = buffer_of(W + (int64_t)n0 * ldw);
  const int r8 = lane >> 3, slot = lane & 7;
  uint32_t va[2 * AI], vw[2 * WI];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int i = 0; i < AI; ++i) {
      const int r = 8 * (AI * wave + i) + r8;
      va[h * AI + i] =
          (uint32_t)(((int64_t)(min(m0 + h * HA + r, M - 1) - m0) * lda + (slot ^ ((r >> 1) & 7)) * 8) * 2);
    }
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      const int r = 8 * (WI * wave + i) + r8;
      vw[h * WI + i] =
          (uint32_t)(((int64_t)(min(n0 + h * whalf + r, N - 1) - n0) * ldw + (slot ^ ((r >> 1) & 7)) * 8) * 2);
    }
  }
  const uint32_t lds0 = lds_address(smem);
  const int stages = K / DENSE_BK;
  auto copy_a = [&](int buf, int kt) {
    const uint32_t ko = (uint32_t)min(kt, stages - 1) * 128;
#pragma unroll
    for (int i = 0; i < 2 * AI; ++i)
      copy16(abuf, va[i], ko, lds0 + buf * STAGE + (i / AI) * HAB + (AI * wave + i % AI) * 1024);
  };
  auto copy_w = [&](int buf, int kt) {
    const uint32_t ko = (uint32_t)min(kt, stages - 1) * 128;
#pragma unroll
    for (int i = 0; i < 2 * WI; ++i)
      copy16(wbuf, vw[i], ko, lds0 + buf * STAGE + 2 * HAB + (i / WI) * HWB + (WI * wave + i % WI) * 1024);
  };

  // fragments: row block offsets are immediates (the swizzle depends on the row within 16 only)
  int ao[2], wo[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int ch = ((4 * s + lq) ^ ((l16 >> 1) & 7)) << 4;
    ao[s] = (wm * (HA / 2) + l16) * 128 + ch;
    wo[s] = 2 * HAB + (wn * 32 + l16) * 128 + ch;
  }
  f32x4 acc[2][2][2][JB];  // [column half][16-column block][row half][16-row block]
#pragma unroll
  for (int hw = 0; hw < 2; ++hw)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int ha = 0; ha < 2; ++ha)
#pragma unroll
        for (int j = 0; j < JB; ++j) acc[hw][i][ha][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  bf16x8 fa[2][JB], fw[2][2][2];
  auto read_a = [&](const uint8_t* st, int h) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < JB; ++j) fa[s][j] = *reinterpret_cast<const bf16x8*>(st + ao[s] + h * HAB + j * 2048);
  };
  auto read_w = [&](const uint8_t* st, int h) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i) fw[h][s][i] = *reinterpret_cast<const bf16x8*>(st + wo[s] + h * HWB + i * 2048);
  };
  auto section = [&](int ha) {
    __builtin_amdgcn_sched_barrier(0);
    KX_BARRIER();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int hw = 0; hw < 2; ++hw)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < JB; ++j) acc[hw][i][ha][j] = mfma16x16x32<H>(fw[hw][s][i], fa[s][j], acc[hw][i][ha][j]);
    __builtin_amdgcn_sched_barrier(0);
    KX_BARRIER();
    __builtin_amdgcn_sched_barrier(0);
  };

#pragma unroll
  for (int p = 0; p < NST - 1; ++p) {
    copy_w(p, p);
    copy_a(p, p);
  }
  copy_w(NST - 1, NST - 1);
  wait_vm<WAIT2>();
  KX_BARRIER();
  if (wave >= 4) KX_BARRIER();  // the second group runs one barrier behind
  int cur = 0;
  for (int kt = 0; kt < stages; ++kt) {
    const uint8_t* st = smem + cur * STAGE;
    read_w(st, 0);
    read_a(st, 0);
    read_w(st, 1);
    __builtin_amdgcn_sched_barrier(0);
    copy_a(cur == 0 ? NST - 1 : cur - 1, kt + NST - 1);
    wait_vm<WAIT1>();
    wait_lgkmcnt0();
    section(0);
    read_a(st, 1);
    __builtin_amdgcn_sched_barrier(0);
    copy_w(cur, kt + NST);
    wait_vm<WAIT2>();
    wait_lgkmcnt0();
    section(1);
    cur = cur + 1 == NST ? 0 : cur + 1;
  }
  if (wave < 4) KX_BARRIER();
  wait_vm<0>();
  KX_BARRIER();  // every copy has landed and every read is done: the ring's memory takes the staging

  // ---- epilogue: a quadrant (row half x column half) at a time through one of two LDS strips
  constexpr int STEP = 16, NROW = HA / STEP;
  float* const strip = reinterpret_cast<float*>(smem);
  const int c4 = (tid & 31) * 4, rr = tid >> 5;
  const bool vec_ok = (ldc % 4 == 0) && (!(epi.flags & KX_EPI_GATED_RESIDUAL) || epi.ldr % 4 == 0);
  const bool full = vec_ok && m0 + BM <= M && n0 + 256 <= N;
#define KX_STAGE(st, hw, ha)                                                                              \
  _Pragma("unroll") for (int i = 0; i < 2; ++i) _Pragma("unroll") for (int j = 0; j < JB; ++j)            \
      *reinterpret_cast<float4*>((st) + (wm * (HA / 2) + j * 16 + l16) * PITCH + wn * 32 + i * 16 + 4 * lq) = \
          make_float4(acc[hw][i][ha][j][0], acc[hw][i][ha][j][1], acc[hw][i][ha][j][2], acc[hw][i][ha][j][3]);
  if constexpr (NS) {
    if (swiglu) {
      uint16_t* out = static_cast<uint16_t*>(epi.c2) + (n0 - (int)epi.sw_begin) + c4;
      float bg[4], bu[4];
      swiglu_bias(epi, n0 + c4, n0 + whalf + c4, bg, bu);
#pragma unroll
      for (int ha = 0; ha < 2; ++ha) {
        if (ha) KX_BARRIER();  // the first half's strips have been read
        KX_STAGE(strip, 0, ha)
        KX_STAGE(strip + STRIP, 1, ha)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        KX_BARRIER();
#pragma unroll
        for (int q = 0; q < NROW; ++q) {
          const int r = rr + q * STEP, m = m0 + ha * HA + r;
          const uint2 o = swiglu4(strip + r * PITCH + c4, strip + STRIP + r * PITCH + c4, bg, bu);
          if (m < M) *reinterpret_cast<uint2*>(out + (int64_t)m * epi.ldc2) = o;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
      return;
    }
  }
#pragma unroll 1
  for (int q = 0; q < 4; ++q) {
    const int ha = q >> 1, hw = q & 1;
    float* st = strip + hw * STRIP;
    const int mrow = m0 + ha * HA, n = n0 + hw * 128 + c4;
    ResidOf<GMODE> res[GMODE ? NROW : 1];
    if constexpr (GMODE != 0) {
      if (full) strip_resid<GMODE, NROW, STEP>(res, mrow + rr, n, epi);
    }
    // (a strip's readers of two quadrants ago have passed the last quadrant's barrier)
    if (q == 0) { KX_STAGE(st, 0, 0) }
    else if (q == 1) { KX_STAGE(st, 1, 0) }
    else if (q == 2) { KX_STAGE(st, 0, 1) }
    else { KX_STAGE(st, 1, 1) }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    KX_BARRIER();
    if (NS && n0 + hw * 128 < epi.k_end)
      strip_norm_rope<NROW, STEP>(st, rr, c4, mrow, n, M, epi, static_cast<uint16_t*>(C), ldc);
    else
      strip_store<H, GMODE, OUTF32, NROW, STEP>(st, rr, c4, mrow, n, M, NS ? min(N, (int)epi.sw_begin) : N, epi,
                                                full, vec_ok, res, C, ldc);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
#undef KX_STAGE
}

// ---- 128 x 128 and 64 x 128 tiles ----------------------------------------------------------------
//
// Few rows: the product is bound by the weight stream's latency, so more, smaller workgroups. Four
// waves (2 x 2), a ring of four 64-wide stages with the copies three stages ahead between the MFMAs;
// every k32 step waits for its fragments (read one step earlier), then each MFMA is followed by its
// share of the next step's reads and of the copies. The last step of a stage holds its only barrier.
// NS: the column forms, as in gemm_pp_kernel; a SwiGLU tile pairs 64 gate with 64 up columns.
template <int BM, int GMODE, bool OUTF32, bool NS, bool H>
__global__ __launch_bounds__(256) void gemm_ring_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                        const uint16_t* __restrict__ W, int64_t ldw,
                                                        void* __restrict__ C, int64_t ldc, int M, int N, int K,
                                                        Epilogue epi) {
  constexpr int BN = 128, DNS = 4;
  constexpr int A_INST = BM / 32, W_INST = BN / 32;  // copies per wave and stage
  constexpr int PER = A_INST + W_INST;
  constexpr int STAGE = (BM + BN) * 128;
  constexpr int MB = BM / 32, NB = BN / 32;  // 16-wide blocks of a wave's (BM / 2) x (BN / 2)
  constexpr int KS = 2, DPS = PER / KS;      // k32 steps per stage, copies per step
  static_assert(DPS * KS == PER, "copies per step");
  constexpr int WAITN = (DNS - 3) * PER + DPS;  // stage kt + 1 complete at the wait of stage kt
  constexpr int SMEM = DNS * STAGE;
  static_assert(BM * PITCH * 4 <= SMEM, "staging");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[SMEM];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int l16 = lane & 15, lq = lane >> 4;
  if constexpr (GMODE == 0 && OUTF32) {
    const int64_t y = blockIdx.y;  // K slices, as in gemm_pp_kernel
    A += y * K;
    W += y * K;
    C = static_cast<float*>(C) + y * (int64_t)M * ldc;
  }
  const int tiles_m = (M + BM - 1) / BM;
  int plain_n = (N + BN - 1) / BN, tiles_n = plain_n;
  if constexpr (NS) {
    plain_n = ((int)epi.sw_begin + BN - 1) / BN;
    tiles_n = plain_n + (int)(epi.sw_width / 64);
  }
  int2 tile = lds_tile_of(blockIdx.x, tiles_m, tiles_n);
  if (epi.rows_desc) tile.x = tiles_m - 1 - tile.x;
  const int m0 = tile.x * BM;
  const bool swiglu = NS && tile.y >= plain_n;
  const int n0 = swiglu ? (int)epi.sw_begin + (tile.y - plain_n) * 64 : tile.y * BN;
  const int wskip = swiglu ? (int)epi.sw_width - 64 : 0;  // weight rows between the tile's two halves
  const i32x4 abuf = buffer_of(A + (int64_t)m0 * lda), wbuf = buffer_of(W + (int64_t)n0 * ldw);
  const int r8 = lane >> 3, slot = lane & 7;
  uint32_t vo[PER];
#pragma unroll
  for (int i = 0; i < A_INST; ++i) {
    const int r = (wave * A_INST + i) * 8 + r8;
    vo[i] = (uint32_t)(((int64_t)(min(m0 + r, M - 1) - m0) * lda + (slot ^ ((r >> 1) & 7)) * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < W_INST; ++i) {
    const int r = (wave * W_INST + i) * 8 + r8;
    const int wr = r + (r < 64 ? 0 : wskip);
    vo[A_INST + i] = (uint32_t)(((int64_t)(min(n0 + wr, N - 1) - n0) * ldw + (slot ^ ((r >> 1) & 7)) * 8) * 2);
  }
  const uint32_t lds0 = lds_address(smem);
  auto copy = [&](int i, int buf, uint32_t ko) {
    if (i < A_INST)
      copy16(abuf, vo[i], ko, lds0 + buf * STAGE + (wave * A_INST + i) * 1024);
    else
      copy16(wbuf, vo[i], ko, lds0 + buf * STAGE + BM * 128 + (wave * W_INST + i - A_INST) * 1024);
  };
  int ao[KS], wo[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int ch = ((4 * s + lq) ^ ((l16 >> 1) & 7)) << 4;
    ao[s] = (wm * (BM / 2) + l16) * 128 + ch;
    wo[s] = BM * 128 + (wn * (BN / 2) + l16) * 128 + ch;
  }
  f32x4 acc[NB][MB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) acc[i][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  const int stages = K / DENSE_BK;
#pragma unroll
  for (int p = 0; p < DNS - 1; ++p)
#pragma unroll
    for (int i = 0; i < PER; ++i) copy(i, p, (uint32_t)min(p, stages - 1) * 128);
  wait_vm<(DNS - 2) * PER>();
  KX_BARRIER();
  bf16x8 fa[2][MB], fw[2][NB];
  auto read = [&](const uint8_t* st, int s, int r, bf16x8* a, bf16x8* w) {
    if (r < MB) a[r] = *reinterpret_cast<const bf16x8*>(st + ao[s] + r * 2048);
    else w[r - MB] = *reinterpret_cast<const bf16x8*>(st + wo[s] + (r - MB) * 2048);
  };
#pragma unroll
  for (int r = 0; r < MB + NB; ++r) read(smem, 0, r, fa[0], fw[0]);
  int cur = 0;
  for (int kt = 0; kt < stages; ++kt) {
    const int nxt = cur + 1 == DNS ? 0 : cur + 1;
    // stage kt + 3 goes into the slot stage kt - 1 used; past the end the last stage is copied again
    const int iss = cur == 0 ? DNS - 1 : cur - 1;
    const uint32_t ko = (uint32_t)min(kt + DNS - 1, stages - 1) * 128;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      wait_lgkmcnt0();
      if (s + 1 == KS) {
        // stage kt + 1 has landed for this wave and its reads of stage kt are done; after the
        // barrier this holds for every wave
        wait_vm<WAITN>();
        KX_BARRIER();
      }
      __builtin_amdgcn_sched_barrier(0);
      const uint8_t* rbuf = smem + (s + 1 < KS ? cur : nxt) * STAGE;
      constexpr int NRD = MB + NB, NMF = NB * MB;
#pragma unroll
      for (int q = 0; q < NMF; ++q) {
        const int i = q / MB, j = q % MB;
        acc[i][j] = mfma16x16x32<H>(fw[s][i], fa[s][j], acc[i][j]);
#pragma unroll
        for (int r = q * NRD / NMF; r < (q + 1) * NRD / NMF; ++r) read(rbuf, s ^ 1, r, fa[s ^ 1], fw[s ^ 1]);
#pragma unroll
        for (int d = q * DPS / NMF; d < (q + 1) * DPS / NMF; ++d) copy(s * DPS + d, iss, ko);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    cur = nxt;
  }
  wait_vm<0>();
  wait_lgkmcnt0();

  // epilogue: the whole tile staged at once
  constexpr int STEP = 8, NROW = BM / STEP;
  float* const strip = reinterpret_cast<float*>(smem);
  const int c4 = (tid & 31) * 4, rr = tid >> 5;
  const bool vec_ok = (ldc % 4 == 0) && (!(epi.flags & KX_EPI_GATED_RESIDUAL) || epi.ldr % 4 == 0);
  const bool full = vec_ok && m0 + BM <= M && n0 + BN <= N;
  ResidOf<GMODE> res[GMODE ? NROW : 1];
  if constexpr (GMODE != 0) {
    if (full) strip_resid<GMODE, NROW, STEP>(res, m0 + rr, n0 + c4, epi);
  }
  KX_BARRIER();  // every wave is done with the ring
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j)
      *reinterpret_cast<float4*>(strip + (wm * (BM / 2) + j * 16 + l16) * PITCH + wn * (BN / 2) + i * 16 + 4 * lq) =
          make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  KX_BARRIER();
  if constexpr (NS) {
    if (swiglu) {
      const int p4 = (tid & 15) * 4;
      float bg[4], bu[4];
      swiglu_bias(epi, n0 + p4, n0 + (int)epi.sw_width + p4, bg, bu);
      uint16_t* out = static_cast<uint16_t*>(epi.c2) + (n0 - (int)epi.sw_begin) + p4;
#pragma unroll
      for (int q = 0; q < BM / 16; ++q) {
        const int r = (tid >> 4) + q * 16, m = m0 + r;
        const uint2 o = swiglu4(strip + r * PITCH + p4, strip + r * PITCH + 64 + p4, bg, bu);
        if (m < M) *reinterpret_cast<uint2*>(out + (int64_t)m * epi.ldc2) = o;
      }
      return;
    }
    if (n0 < epi.k_end) {
      strip_norm_rope<NROW, STEP>(strip, rr, c4, m0, n0 + c4, M, epi, static_cast<uint16_t*>(C), ldc);
      return;
    }
  }
  strip_store<H, GMODE, OUTF32, NROW, STEP>(strip, rr, c4, m0, n0 + c4, M, NS ? min(N, (int)epi.sw_begin) : N, epi,
                                            full, vec_ok, res, C, ldc);
}

// ---- launches ------------------------------------------------------------------------------------

struct Call {
  const uint16_t* a;
  int64_t lda;
  const uint16_t* w;
  int64_t ldw;
  void* c;
  int64_t ldc;
  int m, n, k, splits;
  hipStream_t s;
};

template <int BM, int GMODE, bool OUTF32, bool NS, bool H>
void run_pp(const Call& x, const Epilogue& epi, int tiles_n) {
  const dim3 grid((unsigned)(((x.m + BM - 1) / BM) * tiles_n), (unsigned)x.splits);
  gemm_pp_kernel<BM, GMODE, OUTF32, NS, H><<<grid, 512, 0, x.s>>>(x.a, x.lda, x.w, x.ldw, x.c, x.ldc, x.m, x.n, x.k, epi);
}
template <int BM, int GMODE, bool OUTF32, bool NS, bool H>
void run_ring(const Call& x, const Epilogue& epi, int tiles_n) {
  const dim3 grid((unsigned)(((x.m + BM - 1) / BM) * tiles_n), (unsigned)x.splits);
  gemm_ring_kernel<BM, GMODE, OUTF32, NS, H><<<grid, 256, 0, x.s>>>(x.a, x.lda, x.w, x.ldw, x.c, x.ldc, x.m, x.n, x.k, epi);
}

// tiles_256, tiles_128: the product's column tiles of either width
template <int GMODE, bool OUTF32, bool NS, bool H>
void run_tile(int tile, const Call& x, const Epilogue& epi, int tiles_256, int tiles_128) {
  switch (tile) {
    case DT256x256: return run_pp<256, GMODE, OUTF32, NS, H>(x, epi, tiles_256);
    case DT128x256: return run_pp<128, GMODE, OUTF32, NS, H>(x, epi, tiles_256);
    case DT128x128: return run_ring<128, GMODE, OUTF32, NS, H>(x, epi, tiles_128);
    default: return run_ring<64, GMODE, OUTF32, NS, H>(x, epi, tiles_128);
  }
}
template <int GMODE, bool OUTF32, bool H>
void run_plain(int tile, const Call& x, const Epilogue& epi) {
  run_tile<GMODE, OUTF32, false, H>(tile, x, epi, (x.n + 255) / 256, (x.n + 127) / 128);
}

// Residual mode (none / 16-bit / fp32) and output type select the epilogue.
template <bool H>
void run_epilogue(int tile, const Call& x, const Epilogue& epi) {
  const int gmode = (epi.flags & KX_EPI_GATED_RESIDUAL) ? ((epi.flags & KX_EPI_RESID_F32) ? 2 : 1) : 0;
  const bool out32 = epi.flags & KX_EPI_OUT_F32;
  switch (gmode * 2 + (out32 ? 1 : 0)) {
    case 0: return run_plain<0, false, H>(tile, x, epi);
    case 1: return run_plain<0, true, H>(tile, x, epi);
    case 2: return run_plain<1, false, H>(tile, x, epi);
    case 3: return run_plain<1, true, H>(tile, x, epi);
    case 4: return run_plain<2, false, H>(tile, x, epi);
    default: return run_plain<2, true, H>(tile, x, epi);
  }
}

}  // namespace

// Whether a product visits its tile rows last to first. Every producer of an activation in
// this library writes its rows in ascending order, so the last rows written are the ones most
// likely still in the 256 MB memory-side cache. When the input is too large for that cache to
// hold whole (above 128 MiB: the 9216 x 16384 feed-forward hidden state, 302 MB, read by the
// down projection right after the up projection wrote it), reading its rows newest first turns
// part of the operand stream into cache hits (down projection 964 -> 927 us in the config-3
// block). The order of tiles does not change any result.
bool rows_last_first(int64_t m, int64_t k) { return m * k * 2 > (128ll << 20); }

namespace {

// ---- the tile and row-split rule -----------------------------------------------------------------
//
// Time of a (m, n, k) product on one tile size, in us: fixed + per round of 256 workgroups a prologue
// and epilogue + per 64-wide stage of a full round `full`, of a partial round `part` + `load` times
// its share of the 256 CUs (a partly filled chip clocks higher and shares the L2s among fewer
// streams). Fitted to 14 row counts (127 .. 9216) x 10 weight shapes per tile; the mean error of the
// fit is 4 %. Per FLOP the tiles cost 1 : 1.2 : 1.9 : 2.2 (full rounds): the smaller ones are bound by
// their operand stream (about 50 GB/s per CU out of the L2 for all of them), but waste less of the
// chip on few rows: 2048 x 4096 x 4096 79 us on 256 x 256 tiles (128 of them) and 62 on 128 x 256;
// 480 x 4096 x 4096 82, 52, 50 and 32.
struct TileCost {
  int bm, bn;
  double fixed, round, full, part, load;
};
constexpr TileCost kTiles[4] = {{256, 256, 3.9, 7.9, 1.41, 0.89, 0.40},
                                {128, 256, 4.2, 4.8, 0.84, 0.57, 0.20},
                                {128, 128, 4.1, 3.0, 0.655, 0.55, 0.10},
                                {64, 128, 3.1, 2.3, 0.384, 0.334, 0.037}};
constexpr int64_t kCUs = 256;

double tile_cost(const TileCost& t, int64_t m, int64_t n, int64_t k, int64_t slices = 1) {
  const int64_t tiles = ((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn) * slices;
  const int64_t full = tiles / kCUs, rest = tiles % kCUs;
  const double stages = (double)(k / DENSE_BK) / (double)slices;
  return t.fixed + t.round * (double)(full + (rest > 0)) + stages * t.full * (double)full +
         (rest > 0 ? stages * (t.part + t.load * (double)rest / (double)kCUs) : 0.0);
}

// The fastest tile size.
int best_tile(int64_t m, int64_t n, int64_t k, double* cost) {
  int best = 0;
  for (int i = 0; i < 4; ++i) {
    const double c = tile_cost(kTiles[i], m, n, k);
    if (i == 0 || c < *cost) {
      best = i;
      *cost = c;
    }
  }
  return best;
}

// Rows that run as 256 x 256 tiles filling whole rounds, the rest as the tile that suits them best:
// a product whose 256 x 256 tiles end in a nearly empty round (1111 x 16384 x 4096: 320 tiles, 1.25
// rounds) pays a whole round for them otherwise. rows = 0: one tile size for all rows. Measured:
// 4608 x 4096 x 4096 162 -> 132 us, 1111 x 16384 x 4096 171 -> 131 us.
struct RowPlan {
  int64_t rows;
  int tile, rest_tile;
};
RowPlan row_plan(int64_t m, int64_t n, int64_t k) {
  double cost = 0.0;
  RowPlan plan{0, best_tile(m, n, k, &cost), 0};
  const int64_t tiles_n = (n + 255) / 256, tiles_m = (m + 255) / 256;
  // a split has to win 4 %, the error of the rule
  double limit = 0.96 * cost;
  const int64_t rounds = tiles_m * tiles_n / kCUs;
  for (int64_t r = std::max<int64_t>(rounds - 1, 1); r <= rounds; ++r) {
    const int64_t rows = r * kCUs / tiles_n * 256;
    if (rows == 0 || rows >= m) continue;
    double rest = 0.0;
    const int rest_tile = best_tile(m - rows, n, k, &rest);
    const double c = tile_cost(kTiles[0], rows, n, k) + rest;
    if (c < limit) {
      limit = c;
      plan = RowPlan{rows, DT256x256, rest_tile};
    }
  }
  return plan;
}

int forced_tile() {
  const char* env = getenv("KX355_GEMM_LDS_TILE");
  if (!env || !*env) return -1;
  const int v = atoi(env);
  return v >= 0 && v <= 3 ? v : -1;
}

// Call `run(first row, rows, tile)` for each part of the plan; the last rows first (their producer
// wrote them most recently, and their pass leaves the weight in the memory-side cache).
template <typename F>
void run_rows(int64_t m, int64_t n, int64_t k, F run) {
  const int forced = forced_tile();
  const RowPlan p = forced >= 0 ? RowPlan{0, forced, 0} : row_plan(m, n, k);
  if (p.rows) run(p.rows, m - p.rows, p.rest_tile);
  run(0, p.rows ? p.rows : m, p.tile);
}

// The tile for `s` K slices, and the time with the reduction of their fp32 partial products (a
// launch, and 0.22 us per MB written and read back; mean error of the fit 6 %).
int slice_tile(int64_t m, int64_t n, int64_t k, int s, double* cost) {
  int best = 0;
  for (int i = 0; i < 4; ++i) {
    const double c = tile_cost(kTiles[i], m, n, k, s);
    if (i == 0 || c < *cost) {
      best = i;
      *cost = c;
    }
  }
  *cost += 4.0 + 0.22e-6 * (double)(m * n) * 4.0 * s;
  return best;
}

}  // namespace

int dense_splits(int64_t m, int64_t n, int64_t k) {
  // a row plan's parts cost the sum of theirs
  double cost = 0.0;
  const RowPlan p = row_plan(m, n, k);
  if (p.rows) {
    best_tile(m - p.rows, n, k, &cost);
    cost += tile_cost(kTiles[0], p.rows, n, k);
  } else {
    cost = tile_cost(kTiles[p.tile], m, n, k);
  }
  int best = 1;
  double limit = 0.94 * cost;  // the error of the rule with slices
  for (const int s : {2, 4, 8, 16}) {
    if (k % (DENSE_BK * s) || k / s < 256) break;
    double c = 0.0;
    slice_tile(m, n, k, s, &c);
    if (c < limit) {
      limit = c;
      best = s;
    }
  }
  return best;
}

int dense_kernels(int64_t m, int64_t n, int64_t k) {
  int count = 0;
  run_rows(m, n, k, [&](int64_t, int64_t, int) { ++count; });
  return count;
}

void launch_dense(bool half, const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, void* c, int64_t ldc,
                  int m, int n, int k, const Epilogue& epi, hipStream_t s) {
  run_rows(m, n, k, [&](int64_t row0, int64_t rows, int tile) {
    Epilogue e = epi;
    e.rows_desc = rows_last_first(rows, k);
    e.row0 = row0;
    if (epi.resid)
      e.resid = static_cast<const char*>(epi.resid) + row0 * epi.ldr * (epi.flags & KX_EPI_RESID_F32 ? 4 : 2);
    const Call x{a + row0 * lda, lda, w, ldw, static_cast<char*>(c) + row0 * ldc * (epi.flags & KX_EPI_OUT_F32 ? 4 : 2),
                 ldc, (int)rows, n, k, 1, s};
    if (half) run_epilogue<true>(tile, x, e);
    else run_epilogue<false>(tile, x, e);
  });
}

void launch_dense_slices(bool half, const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, float* parts,
                         int m, int n, int k, int splits, hipStream_t s) {
  Epilogue plain{};
  plain.gate_div = 1;
  plain.flags = KX_EPI_OUT_F32;
  const int forced = forced_tile();
  double cost = 0.0;
  const int tile = forced >= 0 ? forced : slice_tile(m, n, k, splits, &cost);
  const Call x{a, lda, w, ldw, parts, n, m, n, k / splits, splits, s};
  if (half) run_plain<0, true, true>(tile, x, plain);
  else run_plain<0, true, false>(tile, x, plain);
}

void launch_dense_columns(const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, void* c, int64_t ldc, int m,
                          int n, int k, const Epilogue& epi, hipStream_t s) {
  const int t256 = (int)((epi.sw_begin + 255) / 256 + epi.sw_width / 128);
  const int t128 = (int)((epi.sw_begin + 127) / 128 + epi.sw_width / 64);
  run_rows(m, n, k, [&](int64_t row0, int64_t rows, int tile) {
    Epilogue e = epi;
    e.rows_desc = rows_last_first(rows, k);
    e.row0 = row0;
    if (epi.c2) e.c2 = static_cast<uint16_t*>(epi.c2) + row0 * epi.ldc2;
    const Call x{a + row0 * lda, lda, w, ldw, static_cast<uint16_t*>(c) + row0 * ldc, ldc, (int)rows, n, k, 1, s};
    run_tile<0, false, true, false>(tile, x, e, t256, t128);
  });
}

}  // namespace kx
