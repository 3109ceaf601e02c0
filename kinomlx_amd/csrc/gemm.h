// Shared by the GEMM translation units: the epilogue arguments and their application to a run of
// four columns, the workgroup -> tile map, and the buffer -> LDS copy and wait helpers.
#pragma once

#include <algorithm>
#include <type_traits>

#include "common.h"

namespace kx {

struct Epilogue {
  const uint16_t* bias;
  const void* resid;  // bf16, or fp32 with KX_EPI_RESID_F32
  int64_t ldr;
  const float* gate;
  int64_t gate_div;
  int64_t gate_stride;
  int flags;
  // set by the launcher, not part of the C ABI: visit the tile rows last to first (see
  // rows_last_first); the call's first row in the whole product (gate and table rows count from there)
  int rows_desc;
  int64_t row0;
  // The column forms (the fused-projection kernels): columns [0, q_end) are query heads and
  // [q_end, k_end) key heads of head_dim (64 or 128) columns; each row's head is RMS-normalized
  // (weights nq / nk, fp32 or bf16, plus n_off; n_eps), then rotated in adjacent pairs by the row's
  // cos / sin table row: tables + (m / t_rows) * t_bs + (m % t_rows) * t_ld + head * t_hs + d.
  const void* nq;
  const void* nk;
  int n_bf16;
  int head_dim;
  float n_eps, n_off;
  int64_t q_end, k_end;
  const float* cosp;
  const float* sinp;
  int64_t t_ld, t_hs, t_rows, t_bs;
  uint32_t t_magic;  // m / t_rows = (umulhi(m, t_magic) + m) >> t_shift for m < 2^31
  int t_shift;
  // columns from sw_begin on are a SwiGLU pair: sw_width gate columns, then as many up columns;
  // silu(gate) * up goes to columns [0, sw_width) of c2
  int64_t sw_begin, sw_width;
  void* c2;
  int64_t ldc2;
};

// ---- dense products (gemm_dense.hip) ------------------------------------------------------------

// Output tiles of the dense kernels: 256 x 256 and 128 x 256 (the alternating-group kernel), 128 x 128
// and 64 x 128 (the four-wave ring kernel).
enum DenseTile { DT256x256 = 0, DT128x256 = 1, DT128x128 = 2, DT64x128 = 3 };
constexpr int DENSE_BK = 64;  // K per stage: a row's 128 bytes of a stage are one full cache line

// Whether an (m, k) input is visited last rows first.
bool rows_last_first(int64_t m, int64_t k);
// c = epilogue(a w^T) for k % 64 == 0 and 16-byte aligned rows of at most 2^22 elements
// (KX355_GEMM_LDS_TILE = 0 .. 3 forces one tile size).
void launch_dense(bool half, const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, void* c, int64_t ldc,
                  int m, int n, int k, const Epilogue& epi, hipStream_t s);
// The kernels that launch_dense runs for these sizes (2 with a row split).
int dense_kernels(int64_t m, int64_t n, int64_t k);
// The K slices (1, 2, 4, 8 or 16) in which a product is fastest, its reduction included.
int dense_splits(int64_t m, int64_t n, int64_t k);
// parts[y] = a[:, slice y] w[:, slice y]^T in fp32, (splits, m, n): k / splits wide slices.
void launch_dense_slices(bool half, const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, float* parts,
                         int m, int n, int k, int splits, hipStream_t s);
// The bf16 product with the epilogue's column forms (256-column tiles).
void launch_dense_columns(const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, void* c, int64_t ldc, int m,
                          int n, int k, const Epilogue& epi, hipStream_t s);
// ---- few rows (gemm_rows.hip) -------------------------------------------------------------------

// c = epilogue(a w^T) for 1 <= m <= FEW_ROWS, k % 8 == 0 and 16-byte aligned rows.
constexpr int FEW_ROWS = 4;
void launch_few_rows(bool half, const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, void* c, int64_t ldc,
                     int m, int n, int k, const Epilogue& epi, hipStream_t s);

namespace {

__device__ __forceinline__ float apply_act(float v, int act) {
  switch (act) {
    case 1: return fast_gelu_tanh(v);
    case 2: return fast_silu(v);
    case 3: return fast_sigmoid2(v);
    case 4: return fast_sigmoid(v);
    default: return v;
  }
}

// Tile of workgroup `bid` for the direct-to-LDS kernel, as (tile row, tile column). The 256
// workgroups of a round run at once, 32 per XCD, and the XCDs' L2s are separate. When the tile
// columns divide a round (8, 16, 32 or 64 of them) and the rows fill whole rounds, each round
// covers R = 256 / tiles_n whole tile rows, and each XCD an a x b block of them with the fewest
// operand panels (a + b = 12 for 32 tiles): every activation panel is then read in one round
// only, so a product whose operands exceed the last-level cache re-reads them from HBM once per
// round rather than once per round and XCD pair (the 9216 x 4096 x 16384 down projection: mean
// L1 -> L2 request latency 688 -> 505 cycles, 2.5 % faster). Otherwise: XCD-contiguous tiles,
// grouped by 8 tile rows.
__device__ __forceinline__ int2 lds_tile_of(int bid, int tiles_m, int tiles_n) {
  const int rows = 256 / tiles_n;
  if ((tiles_n == 8 || tiles_n == 16 || tiles_n == 32 || tiles_n == 64) && tiles_m % rows == 0) {
    // XCD x: block (x % ra, x / ra) of an ra x cb grid over the round, ra * cb = 8
    const int ra = tiles_n >= 32 ? 1 : tiles_n == 16 ? 2 : 8, cb = 8 / ra;
    const int a = rows / ra, b = tiles_n / cb;  // block rows x columns, a * b = 32
    const int x = bid % 8, i = bid / 8, r = i / 32, j = i % 32;
    return make_int2(r * rows + (x % ra) * a + j % a, (x / ra) * b + j / a);
  }
  const int t = xcd_remap(bid, tiles_m * tiles_n);
  constexpr int GM = 8;
  const int group_width = GM * tiles_n;
  const int first_m = (t / group_width) * GM;
  const int gsz = min(tiles_m - first_m, GM);
  return make_int2(first_m + (t % group_width) % gsz, (t % group_width) / gsz);
}

#define KX_LDS(p) ((__attribute__((address_space(3))) void*)(p))
// Raw buffer resource over `base` (stride 0, 4 GiB range; dword 3 as for every gfx9 raw buffer)
// and a 16-byte-per-lane buffer load into LDS (M0 + lane * 16) from base + voff + soff: the
// offsets are one loop-invariant 32-bit lane offset and a scalar K offset, so a DMA issue needs
// no 64-bit address arithmetic (3 % on the block GEMMs against global_load_lds with per-issue
// 64-bit VALU adds). The host compilation pass has no buffer builtins; kernels only run on the
// device.
#if defined(__HIP_DEVICE_COMPILE__)
using rsrc_t = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ rsrc_t raw_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, -1, 0x00020000);
}
__device__ __forceinline__ void buffer_lds16(rsrc_t r, void* lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, KX_LDS(lds), 16, voff, soff, 0, 0);
}
#else
struct rsrc_t {};
__device__ inline rsrc_t raw_rsrc(const void*) { return {}; }
__device__ inline void buffer_lds16(rsrc_t, void*, uint32_t, uint32_t) {}
#endif
// A workgroup barrier that the compiler may not move memory accesses across.
#define KX_BARRIER() asm volatile("s_barrier" ::: "memory")

// gfx9 s_waitcnt immediate that waits for vmcnt <= N only.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// s_waitcnt vmcnt(N) that also keeps the compiler from moving memory accesses across it.
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void wait_lgkmcnt0() { __builtin_amdgcn_s_waitcnt(0xC07F); }
// gfx9 s_waitcnt immediate that waits for lgkmcnt <= N only (LDS reads complete in order).
template <int N>
__device__ __forceinline__ void wait_lgkmcnt() {
  static_assert(N >= 0 && N < 16, "lgkmcnt");
  __builtin_amdgcn_s_waitcnt(0xC07F | (N << 8));
}

// bias + activation + gated residual on 4 consecutive columns n..n+3 of row m, then the store.
template <bool H>
__device__ __forceinline__ void epilogue_store4(float v[4], int m, int n, int N, const Epilogue& epi,
                                                void* __restrict__ C, int64_t ldc, bool vec_ok) {
  const int act = (epi.flags >> 4) & 15;
  const bool gated = epi.flags & KX_EPI_GATED_RESIDUAL;
  const bool resid_f32 = epi.flags & KX_EPI_RESID_F32;
  const bool out_f32 = epi.flags & KX_EPI_OUT_F32;
  const int64_t ro = (int64_t)m * epi.ldr + n;
  const int64_t co = (int64_t)m * ldc + n;
  if (vec_ok && n + 3 < N) {
    if (epi.flags & KX_EPI_BIAS) {
      const uint2 bb = *reinterpret_cast<const uint2*>(epi.bias + n);
      v[0] += e_lo<H>(bb.x); v[1] += e_hi<H>(bb.x); v[2] += e_lo<H>(bb.y); v[3] += e_hi<H>(bb.y);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = apply_act(v[e], act);
    if (gated) {
      const int64_t grow = (m + epi.row0) / epi.gate_div;
      const float4 gv = *reinterpret_cast<const float4*>(epi.gate + grow * epi.gate_stride + n);
      float rv[4];
      if (resid_f32) {
        const float4 rr = *reinterpret_cast<const float4*>(static_cast<const float*>(epi.resid) + ro);
        rv[0] = rr.x; rv[1] = rr.y; rv[2] = rr.z; rv[3] = rr.w;
      } else {
        const uint2 rr = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(epi.resid) + ro);
        rv[0] = e_lo<H>(rr.x); rv[1] = e_hi<H>(rr.x); rv[2] = e_lo<H>(rr.y); rv[3] = e_hi<H>(rr.y);
      }
      v[0] = fmaf(gv.x, v[0], rv[0]);
      v[1] = fmaf(gv.y, v[1], rv[1]);
      v[2] = fmaf(gv.z, v[2], rv[2]);
      v[3] = fmaf(gv.w, v[3], rv[3]);
    }
    if (out_f32) {
      *reinterpret_cast<float4*>(static_cast<float*>(C) + co) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
      uint2 o;
      o.x = e_pack2<H>(v[0], v[1]);
      o.y = e_pack2<H>(v[2], v[3]);
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(C) + co) = o;
    }
    return;
  }
  for (int e = 0; e < 4 && n + e < N; ++e) {
    float x = v[e];
    if (epi.flags & KX_EPI_BIAS) x += e2f<H>(epi.bias[n + e]);
    x = apply_act(x, act);
    if (gated) {
      const float rv = resid_f32 ? static_cast<const float*>(epi.resid)[ro + e]
                                 : e2f<H>(static_cast<const uint16_t*>(epi.resid)[ro + e]);
      x = fmaf(epi.gate[((m + epi.row0) / epi.gate_div) * epi.gate_stride + n + e], x, rv);
    }
    if (out_f32)
      static_cast<float*>(C)[co + e] = x;
    else
      static_cast<uint16_t*>(C)[co + e] = f2e<H>(x);
  }
}

// The activation as a compile-time choice (ACT = the epilogue's activation code; -1: chosen at
// run time per value).
template <int ACT>
__device__ __forceinline__ float act_c(float v, int act) {
  if constexpr (ACT == 1) return fast_gelu_tanh(v);
  else if constexpr (ACT == 2) return fast_silu(v);
  else if constexpr (ACT == 0) return v;
  else return apply_act(v, act);
}

// One 16x16x32 MFMA on 16-bit operands (bf16, or fp16 with H).
template <bool H>
__device__ __forceinline__ f32x4 mfma16x16x32(bf16x8 a, bf16x8 b, f32x4 c) {
  if constexpr (H)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

}  // namespace
}  // namespace kx
