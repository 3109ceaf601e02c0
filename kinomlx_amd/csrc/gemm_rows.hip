// C = epilogue(A W^T) for 1 to 4 rows: the AdaLN producers of one denoising step, whose weights are
// read once for a row or two. The weight stream is the whole cost, so nothing is staged: a wave
// reads 4 weight rows 1 KB at a time (64 lanes x 16 bytes, one fully used request per load), without
// keeping them in the caches, multiplies them in registers with its piece of the few activation
// rows, and asks for the next 1 KB of each before it uses the last. The 4 waves of a workgroup share
// the K axis, so that 4096 columns still put 16 waves on each CU; their sums meet in LDS.
//
// Measured (bf16, us, against the 64 x 128 MFMA tiles with K slices and their reduction): 1 x 36864 x 4096
// 74.9 -> 43.3 (7.0 TB/s), 1 x 4096 x 4096 13.3 -> 7.5, 1 x 18432 x 2048 20.6 -> 13.0, 4 x 36864 x 4096
// 74.8 -> 50.3, 1 x 4096 x 256 5.1 -> 3.4. One wave per weight row group (K not shared) takes 51.0 and 8.7 on
// the first two, cached loads 48.6 and 8.0, 8 weight rows per wave 47.0 and 7.8. From 5 rows on the
// vector unit is the limit (8 rows: 93 us against the tiles' 72): those rows stay with the tiles.
#include "gemm.h"

namespace kx {
namespace {

typedef uint32_t words4 __attribute__((ext_vector_type(4)));
constexpr int COLS = 4;  // weight rows (output columns) per workgroup

template <int ROWS, bool H>
__global__ __launch_bounds__(256) void gemm_rows_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                        const uint16_t* __restrict__ W, int64_t ldw,
                                                        void* __restrict__ C, int64_t ldc, int M, int N, int K,
                                                        Epilogue epi, bool vec_ok) {
  constexpr int V = ROWS * COLS;  // sums per lane: value m * COLS + c
  __shared__ float part[4][V];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * COLS;
  const int chunks = (K + 511) / 512;  // of 512 K; wave w takes w, w + 4, ..
  float acc[V];
#pragma unroll
  for (int v = 0; v < V; ++v) acc[v] = 0.0f;
  const uint16_t* wrow[COLS];  // columns past N repeat the last (never stored)
#pragma unroll
  for (int c = 0; c < COLS; ++c) wrow[c] = W + (int64_t)min(n0 + c, N - 1) * ldw;
  words4 x[2][ROWS], w[2][COLS];
  auto load = [&](int b, int chunk) {
    const int k = chunk * 512 + 8 * lane;
    const bool in = k < K;  // K % 8 == 0
#pragma unroll
    for (int m = 0; m < ROWS; ++m) {
      x[b][m] = words4{0, 0, 0, 0};
      if (in) x[b][m] = *reinterpret_cast<const words4*>(A + min(m, M - 1) * lda + k);
    }
#pragma unroll
    for (int c = 0; c < COLS; ++c) {
      w[b][c] = words4{0, 0, 0, 0};
      if (in) w[b][c] = __builtin_nontemporal_load(reinterpret_cast<const words4*>(wrow[c] + k));
    }
  };
  auto multiply = [&](int b) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int c = 0; c < COLS; ++c) {
        const float lo = e_lo<H>(w[b][c][j]), hi = e_hi<H>(w[b][c][j]);
#pragma unroll
        for (int m = 0; m < ROWS; ++m) {
          acc[m * COLS + c] = fmaf(lo, e_lo<H>(x[b][m][j]), acc[m * COLS + c]);
          acc[m * COLS + c] = fmaf(hi, e_hi<H>(x[b][m][j]), acc[m * COLS + c]);
        }
      }
  };
  int chunk = wave;
  if (chunk < chunks) load(0, chunk);
  for (; chunk < chunks; chunk += 8) {
    if (chunk + 4 < chunks) load(1, chunk + 4);
    multiply(0);
    if (chunk + 4 >= chunks) break;
    if (chunk + 8 < chunks) load(0, chunk + 8);
    multiply(1);
  }
  // Sum over the lanes, half the values at a time: lanes with the mask bit set go on with the upper half.
  // Value v ends in the lanes whose high bits are v.
  int mask = 32;
#pragma unroll
  for (int half = V / 2; half; half /= 2, mask /= 2) {
    const bool up = lane & mask;
#pragma unroll
    for (int v = 0; v < half; ++v) {
      const float keep = up ? acc[v + half] : acc[v], send = up ? acc[v] : acc[v + half];
      acc[v] = keep + __shfl_xor(send, mask);
    }
  }
  for (; mask; mask /= 2) acc[0] += __shfl_xor(acc[0], mask);
  if (lane % (64 / V) == 0) part[wave][lane / (64 / V)] = acc[0];
  __syncthreads();
  const int m = threadIdx.x;
  if (m >= M) return;
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = (part[0][m * COLS + e] + part[1][m * COLS + e]) +
                                     (part[2][m * COLS + e] + part[3][m * COLS + e]);
  epilogue_store4<H>(v, m, n0, N, epi, C, ldc, vec_ok);
}

template <bool H>
void launch_rows(const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, void* c, int64_t ldc, int m, int n,
                 int k, const Epilogue& epi, hipStream_t s) {
  const bool vec_ok = ldc % 4 == 0 && (!(epi.flags & KX_EPI_GATED_RESIDUAL) || epi.ldr % 4 == 0);
  const unsigned grid = (unsigned)((n + COLS - 1) / COLS);
  if (m == 1) gemm_rows_kernel<1, H><<<grid, 256, 0, s>>>(a, lda, w, ldw, c, ldc, m, n, k, epi, vec_ok);
  else if (m == 2) gemm_rows_kernel<2, H><<<grid, 256, 0, s>>>(a, lda, w, ldw, c, ldc, m, n, k, epi, vec_ok);
  else gemm_rows_kernel<4, H><<<grid, 256, 0, s>>>(a, lda, w, ldw, c, ldc, m, n, k, epi, vec_ok);
}

}  // namespace

void launch_few_rows(bool half, const uint16_t* a, int64_t lda, const uint16_t* w, int64_t ldw, void* c, int64_t ldc,
                     int m, int n, int k, const Epilogue& epi, hipStream_t s) {
  if (half) launch_rows<true>(a, lda, w, ldw, c, ldc, m, n, k, epi, s);
  else launch_rows<false>(a, lda, w, ldw, c, ldc, m, n, k, epi, s);
}

}  // namespace kx
