// A training step's gradients by one turn of tiles (gemm_tile_core.h), operands as they are stored:
//   NN  C[M, N] = A[M, K] . B[K, N]     an input gradient, dX = dY W
//   TT  C[M, N] = A[K, M]^T . B[K, N]   a weight gradient, dW = dY^T X of K tokens, or C += it (summed in f32, rounded once)
//
// What bounds the narrow ones is how many CUs have a tile: 2048 x 2048 is 64 tiles of 256 x 256, and the library's kernels for
// TT ask for two transposes first and read a K that is no multiple of 64 slowly.  The 64 x 64 to 256 x 128 tiles of one turn fill the
// chip; an operand stored [K][rows] comes to LDS as it is and is turned by the reads (ds_read_b64_tr_b16).
// us, transposes and library (or gemm8, marked *) -> here:
//   TT 2048 x 2048 of 4096 / 2048 / 3001 / 1000 tokens 51.7 / 34.5 / 56.3* / 25.8* -> 34.5 / 19.9 / 26.5 / 12.5
//      3072 x 2048 63.8 / 41.3 / 56.8* / 26.4* -> 47.4 / 27.0 / 37.2 / 16.8
//   NN 4096 rows of 2048 x 2048 / 3072 x 2048 37.9 / 50.9 -> 31.6 / 43.4;  2709 rows 39.7 / 39.5 -> 24.9 / 33.8
//      300 rows of 2048 x 2048 13.6 -> 9.3
// Over 480 random sizes that the plan takes: TT .38 of the time, NN .66 (profiles/gemm_routes/forms.txt).
// Left: 0.5 us a step of 64 k where the matrix cores need 0.3 (128 x 128), the L2's rate beside 256 CUs.
#include "gemm_tile_core.h"

namespace mx {

// The tiles and what a turn of them takes, us: start + steps of 64 k (step + load tiles / 256) + out MB of C.  Fitted to 19,600
// runs of TT and 7,800 of NN (2 to 4 % off in the mean; the tile so chosen is 0.3 and 0.2 % behind the best one).
struct GtForm {
  int tm, tn;
  float start, step, load, out;
};
constexpr GtForm kGtNN[] = {{64, 64, 4.83f, .169f, .037f, .084f},   {64, 128, 5.11f, .250f, .059f, .117f},
                            {128, 128, 5.03f, .315f, .099f, .171f}, {128, 192, 6.18f, .415f, .180f, .139f},
                            {192, 128, 6.09f, .402f, .165f, .143f}, {256, 128, 7.00f, .424f, .296f, .128f},
                            {192, 192, 7.59f, .501f, .325f, .109f}};
constexpr GtForm kGtTT[] = {{64, 64, 4.67f, .189f, .035f, .168f},   {64, 128, 5.07f, .276f, .059f, .119f},
                            {128, 128, 5.42f, .336f, .112f, .140f}, {128, 192, 6.07f, .451f, .162f, .153f},
                            {192, 128, 6.16f, .466f, .163f, .152f}, {256, 128, 7.35f, .445f, .347f, .089f},
                            {192, 192, 7.33f, .550f, .311f, .120f}};
constexpr int kGtForms = sizeof(kGtNN) / sizeof(GtForm);

static int64_t gt_form_units(const GtForm& t, int64_t M, int64_t N) { return (M + t.tm - 1) / t.tm * ((N + t.tn - 1) / t.tn); }

template <int EPI, bool AK>
static void gt_form_launch(int tile, int grid, const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, void* C,
                           int64_t ldc, int M, int N, int K, hipStream_t s) {
#define GT(I, TM, TN, WM, WN, S, O)                                                                                     \
  case I:                                                                                                               \
    gemm_tile_kernel<TM, TN, WM, WN, S, O, EPI, AK, false><<<grid, 64 * WM * WN, 0, s>>>(A, lda, B, ldb, C, ldc, M, N, K, 1); \
    break
  switch (tile) {
    GT(0, 64, 64, 2, 2, 4, 2);
    GT(1, 64, 128, 2, 2, 4, 1);
    GT(2, 128, 128, 2, 4, 3, 1);
    GT(3, 128, 192, 4, 2, 3, 1);
    GT(4, 192, 128, 2, 4, 3, 1);
    GT(5, 256, 128, 4, 2, 3, 1);
    GT(6, 192, 192, 4, 2, 3, 1);
  }
#undef GT
}

}  // namespace mx

using namespace mx;

// The tile for a product, -1: more than one turn of the largest, or the other kernels have it faster.  Where the lines lie:
//  * TT: always, but past 6,144 tokens with fewer than 48 tiles of 64 x 64, where the library's split of K is the quicker one for
//    a third (.84 in the mean; 256 x 256 of 8192 22.3 -> 28.8, 512 x 512 31.7 -> 37.0; 48 tiles and more .60);
//  * NN: a K below 4096.  From there on this is the faster one too (1000 rows of 4096 x 4096 41 -> 33), but the library cuts K where it has
//    few tiles, and one sum in order rounds otherwise: as near to 64 bits (1.3 % of the moments in either), but in the second optimizer
//    step of six layers of 4096 channels, 1,328 tokens, single elements of the first moment are then .59 of its rms apart.  That is
//    more than results may move by for 1 % of that step.  A K of 1,025 and more from 24 tiles on (16 to 23 tiles 1.1),
//    16 channels below a K of 1024 (.66; from there on .97 and up to 1.44, 2634 rows of 16 x 3584 9.1 -> 13.1).
extern "C" int mx_gemm_tile_form_plan(int tt, int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || N % 16 || (tt ? M % 16 != 0 : K % 64 != 0 || K >= 4096)) return -1;
  const int64_t small = gt_form_units(kGtNN[0], M, N);
  if (tt ? K > 6144 && small < 48 : small < (K > 1024 ? 24 : 1) || (N < 32 && K >= 1024)) return -1;
  const float nk = (float)((K + 63) / 64), mb = (float)M * N * 2e-6f;
  float best = INFINITY;
  int tile = -1;
  for (int i = 0; i < kGtForms; ++i) {
    const GtForm& t = tt ? kGtTT[i] : kGtNN[i];
    const int64_t u = gt_form_units(t, M, N);
    const float us = t.start + nk * (t.step + t.load * u / 256) + t.out * mb;
    if (u <= 256 && us < best) best = us, tile = i;
  }
  return tile;
}

// C[M, N] (bf16) = A . B (NN) or A^T . B (TT; add: C + that) by tile `tile`.  -1 (nothing launched) for shapes, strides and
// addresses that are not taken.
extern "C" int mx_gemm_tile_form(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, uint16_t* C, int64_t ldc, int M,
                                 int N, int K, int tt, int add, int tile, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || N % 16 || (tt ? M % 16 != 0 : K % 64 != 0 || add) || tile < 0 || tile >= kGtForms) return -1;
  if (lda % 8 || ldb % 8 || ldc % 8 || lda < (tt ? M : K) || ldb < N || ldc < N) return -1;
  if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 15) return -1;
  const GtForm& t = kGtNN[tile];
  // byte offsets of 31 bits: the 32nd marks those past K
  const int64_t rows = ((int64_t)K + 63) / 64 * 64;
  if ((tt ? rows : t.tm) * lda >= 1 << 30 || rows * ldb >= 1 << 30) return -1;
  const int64_t grid = gt_form_units(t, M, N);
  if (grid > INT32_MAX) return -1;
  if (!tt) gt_form_launch<kGtPlain, true>(tile, (int)grid, A, lda, B, ldb, C, ldc, M, N, K, stream);
  else if (add) gt_form_launch<kGtAdd, false>(tile, (int)grid, A, lda, B, ldb, C, ldc, M, N, K, stream);
  else gt_form_launch<kGtPlain, false>(tile, (int)grid, A, lda, B, ldb, C, ldc, M, N, K, stream);
  return (int)hipGetLastError();
}
