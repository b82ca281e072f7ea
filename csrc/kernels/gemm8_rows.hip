// gemm8 (gemm8_core.h) for any number of rows and with K in parts: prompt passes of every model family, ragged
// training batches.
#include "gemm8_core.h"

using namespace mx;

// Any number of rows: C[M, N] = A op(B) with A [M][K] and B [N][K] (b_kc) or [K][N], or, swiglu (B = [gate; up], b_kc),
// C[M, N / 2] = silu(gate) up of that product, which is not stored.  bf16, beta 0, 4-phase schedule; N a multiple of
// 256, K of 64.  Prompt passes and ragged training batches: the library's solutions are tuned for round row counts
// (gate-up with SwiGLU, us, library + SwiGLU pass -> here: 2048 x 16384 at 2600 rows 205 -> 142, 4096 x 28672 at 4096
// 706 -> 640, the rest beside the rule in mxllm/ops/gemm.py).  Returns -1 (nothing launched) for other shapes.
extern "C" int mx_gemm8_rows(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, int b_kc, uint16_t* C,
                             int64_t ldc, int M, int N, int K, int swiglu, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || (N & 255) || K % G8_BK || (swiglu && !b_kc)) return -1;
  if (lda % 8 || ldb % 8 || ldc % 8 || lda < K || ldb < (b_kc ? K : N) || ldc < (swiglu ? N / 2 : N)) return -1;
  if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 15) return -1;
  const int64_t aspan = 256 * lda, bspan = (swiglu ? N : b_kc ? 256 : (int64_t)K) * ldb;
  if (aspan * 2 >= ((int64_t)1 << 31) || bspan * 2 >= ((int64_t)1 << 31)) return -1;
  const int64_t grid = ((M + 255LL) >> 8) * (N >> 8);
  if (grid > INT32_MAX) return -1;
#define G8_R(BK_, E) \
  gemm8_kernel<true, BK_, false, false, 0, 4, E><<<(int)grid, 512, 0, stream>>>(A, lda, B, ldb, C, ldc, M, N, K, nullptr, 1.f)
  if (swiglu) G8_R(true, G8_EPI_ROWS_SWIGLU);
  else if (b_kc) G8_R(true, G8_EPI_ROWS);
  else G8_R(false, G8_EPI_ROWS);
#undef G8_R
  return (int)hipGetLastError();
}

// mx_gemm8_rows with K in S parts (S * its tiles workgroups into the S fp32 images of `ws`, S * M * N floats, then one
// pass that adds them in order): for a long K whose tiles leave most CUs idle (14336 x 4096 at 400 rows, 32 tiles: 210 us
// whole, 57 in 8 parts, the library 80; 16384 x 2048, 4096 rows, 128 tiles: 272, 211 in 2, 237).
extern "C" int mx_gemm8_parts(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, int b_kc, uint16_t* C,
                              int64_t ldc, int M, int N, int K, int swiglu, int S, float* ws, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || (N & 255) || K % G8_BK || (swiglu && !b_kc) || S < 2 || S > K / G8_BK) return -1;
  if (lda % 8 || ldb % 8 || ldc % 8 || lda < K || ldb < (b_kc ? K : N) || ldc < (swiglu ? N / 2 : N)) return -1;
  if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C | (uintptr_t)ws) & 15) return -1;
  const int64_t aspan = 256 * lda, bspan = (b_kc ? 256 : (int64_t)K) * ldb;
  if (aspan * 2 >= ((int64_t)1 << 31) || bspan * 2 >= ((int64_t)1 << 31)) return -1;
  const int64_t grid = ((M + 255LL) >> 8) * (N >> 8) * S, part = (int64_t)M * N;
  if (grid > INT32_MAX) return -1;
  if (b_kc)
    gemm8_kernel<true, true, true, false, 0, 4, G8_EPI_PART><<<(int)grid, 512, 0, stream>>>(A, lda, B, ldb, ws, N, M, N, K,
                                                                                         nullptr, 1.f, S, part);
  else
    gemm8_kernel<true, false, true, false, 0, 4, G8_EPI_PART><<<(int)grid, 512, 0, stream>>>(A, lda, B, ldb, ws, N, M, N, K,
                                                                                          nullptr, 1.f, S, part);
  const int64_t units = (int64_t)M * (swiglu ? N / 2 : N) / 8;
  const int blocks = (int)(units < 256 * 4096 ? (units + 255) / 256 : 4096);
  if (swiglu)
    g8_parts_kernel<true><<<blocks, 256, 0, stream>>>(ws, part, S, N, C, ldc, units);
  else
    g8_parts_kernel<false><<<blocks, 256, 0, stream>>>(ws, part, S, N, C, ldc, units);
  return (int)hipGetLastError();
}
