// bf16 GEMMs whose output is one turn of tiles: C[M, N] = A[M, K] . B[N, K]^T, any number of rows, f32 sums; with SwiGLU (B =
// [gate; up], F rows each) C[M, F] = silu(gate) up.  Projections of prompt passes past the decode GEMMs' 32 rows.
//
// What bounds these products is not the matrix cores' rate but how many CUs have a tile and how long a tile waits: gemm8's 256 x
// 256 tiles leave most CUs of a short prompt without one, and a long walk over K behind one tile is as long as its
// loads' latency.  Here the tile fits the output (64 x 64 to 192 x 192, at most one a CU), and where even that
// leaves CUs idle K is cut in parts, whose f32 images a second launch adds in order.  mx_gemm_tile_plan picks both.
//  * A and B by LDS-DMA (gemm8_core.h: images of 128-B rows, their 16-B chunks XOR-permuted at the source, so that the
//    MFMA-operand reads are free of bank conflicts), S K-tiles of 64 in LDS;
//  * a wave's fragments are read one step of 32 k ahead of their MFMAs, in two register sets, between the MFMAs of the step before
//    (counted lgkmcnt waits: a row of MFMAs waits for its own fragments only); so are the DMA pieces, spread over both steps;
//  * one barrier a K-tile, a quarter into its second step, when the reads of that stage are long done: behind it the next
//    tile is read and tile kt + S asked for.  Wherever LDS allows it is asked for S - 1 tiles ahead of its use; past K the
//    loads are out of the descriptor's range and write zeros into a stage that nobody reads, so every wait has one count;
//  * 8 waves (two a SIMD) where the tile can be dealt to them, 4 where it cannot: 128 x 256, K 4096, few tiles: 36.8 against 39.6 us.
// us, weights from memory, hipBLASLt (or gemm8, K in parts, marked *) -> here:
//   2048 x 2048 at 48 / 330 / 1024 / 2709 / 4096 rows 8.7 / 11.1 / 17.4 / 27.8 / 33.4 -> 7.8 / 8.9 / 15.9 / 23.8 / 30.3
//   3072 x 2048 at 48 / 256 / 2709 11.7 / 13.2 / 42 -> 9.2 / 11.8 / 32
//   2048 x 8192 at 64 / 330 / 1024 / 2709 23.1 / 31.9 / 55.1 / 95 -> 13.2 / 26.5 / 42.7 / 82
//   4096 x 4096 at 48 / 128 / 1024 / 2048 13.8 / 24.8 / 42.1 / 60 -> 12.0 / 16.7 / 38.9 / 54
//   4096 x 14336 at 48 / 64 / 256 36.9 / 35.0* / 60.3* -> 27.8 / 28.3 / 47.6;  8192 x 512 at 128 / 1024 1.8 and 1.2 times as fast.
// Left: 2709 rows of 2048 x 8192 run at 1.1 PF/s.  A CU alone has its 128 x 192 x 64 step in 0.44 us, 242 of them at once in 0.6: the
// L2's 15 TB/s (40 KB a step and CU) and the clock under load.
#include <algorithm>

#include "gemm_tile_core.h"

namespace mx {

// The tiles, and what a turn of them takes, us: start + steps of 64 k (step + load units / 256) + memory MB of weights + with K
// in parts, sum + part parts (part + glu with SwiGLU) + image MB of f32 images.  Fitted to 89,000 runs of 350 sizes of weights
// at 9 to 4,200 rows, weights from memory: 4 to 6 % off in the mean, the tile so chosen 1 % behind the best one.  One tile a CU
// at most: two of 64 x 64 on a CU take 1.8 times as long.
struct GtTile {
  int tm, tn;
  float start, step, load, sum, part, image, memory, glu;
};
constexpr GtTile kGtTiles[] = {{64, 64, 2.55f, .169f, .065f, 1.90f, .152f, .497f, .080f, .250f},
                               {64, 128, 2.86f, .253f, .101f, 1.81f, .153f, .487f, .087f, .263f},
                               {128, 128, 3.49f, .411f, .078f, 1.38f, .143f, .482f, .066f, .293f},
                               {128, 192, 4.86f, .474f, .136f, 1.31f, .151f, .373f, .063f, .232f},
                               {128, 256, 5.96f, .593f, .138f, 2.01f, .102f, .294f, .065f, .189f},
                               {160, 192, 6.79f, .571f, .084f, .21f, .097f, .349f, .058f, .171f},
                               {192, 192, 6.97f, .547f, .202f, 1.14f, .093f, .316f, .056f, .138f}};
constexpr int kGtCount = sizeof(kGtTiles) / sizeof(GtTile), kGtPlaces = 256;

// What the library takes where it has a good kernel, us: the quickest tenth of the same sizes.  Its tiles are not known; it is
// as quick as the best of these would be, in as many turns as they need.  It is slower by 16 % in the mean, and by half and
// more between the sizes that it is tuned for.
static float gt_library(int64_t M, int64_t N, int64_t K) {
  constexpr int edge[] = {32, 64, 96, 128, 160, 192, 224, 256};
  float step = INFINITY;
  for (int tm : edge)
    for (int tn : edge) {
      const int64_t u = (M + tm - 1) / tm * ((N + tn - 1) / tn);
      const float load = .0041f + .0538f * std::min(1.f, (float)u / kGtPlaces);
      step = std::min(step, (float)((u + kGtPlaces - 1) / kGtPlaces) * (.0149f + .0442f * tm * tn / 4096 + load * (tm + tn) / 64));
    }
  return 5.33f + .0908f * N * K * 2e-6f + .299f * M * N * 2e-6f + K / 64 * step;
}

static int64_t gt_units(const GtTile& t, int64_t M, int64_t N) { return (M + t.tm - 1) / t.tm * ((N + t.tn - 1) / t.tn); }

template <int EPI>
static void gt_launch(int tile, int grid, const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, void* C, int64_t ldc,
                      int M, int N, int K, int parts, hipStream_t s, float limit = 0.f) {
#define GT(I, TM, TN, WM, WN, S, O) \
  case I: gemm_tile_kernel<TM, TN, WM, WN, S, O, EPI><<<grid, 64 * WM * WN, 0, s>>>(A, lda, B, ldb, C, ldc, M, N, K, parts, limit); break
  switch (tile) {
    GT(0, 64, 64, 2, 2, 4, 2);
    GT(1, 64, 128, 2, 2, 4, 1);
    GT(2, 128, 128, 4, 2, 3, 1);
    GT(3, 128, 192, 4, 2, 3, 1);
    GT(4, 128, 256, 2, 4, 3, 1);
    GT(5, 160, 192, 2, 2, 3, 1);
    GT(6, 192, 192, 4, 2, 3, 1);
  }
#undef GT
}

}  // namespace mx

using namespace mx;

// Tile and parts of K for a product, as 64 tile + parts, by the modelled time; -1: it is not one turn of tiles, or the library,
// or another kernel, may have it faster.  Where the lines lie (us, hipBLASLt, or gemm8 marked * -> here):
//  * K in one part of more than 1,024: a tile past 64 x 64 only where enough of the CUs have one. The share, and the mean time
//    against the library's at 256 to 4,400 rows below it and at it: 64 x 128 13/16, past a K of 2,048 7/8 (K 2048 at 12/16 .99, a
//    quarter of the sizes slower by more than 3 %, at 13/16 .91; K 3072 at 13/16 1.10); 128 x 128 13/16 (K 4096 1.08, .92), up to a K of
//    2,048 1/2 (.85; 2048 x 2048 at 1,045 to 1,628 rows 19 -> 15); 128 x 192 5/8 (.98); larger ones 13/16 (1.05 - 1.1, .95); past a
//    K of 4,096 7/8 (.98 at 13/16, but a quarter slower). Below them the library's kernels are as quick (6144 x 4096 at 386 rows,
//    192 tiles, 30.9 -> 36.8; 4096 x 4096 at 687, 192, 32.3 -> 36.5). A K up to 1,024 is over before it matters (8192 x 512 at 181
//    rows, 192 tiles, 9.3 -> 5.9);
//  * not where the library at its best (gt_library, with SwiGLU and its activation's launch) would be faster. The model may be
//    longer than that by 3 % (64 x 128; in parts that leave CUs idle); up to 32 rows by 5 % (12 with SwiGLU of more than 44 M
//    weights); up to 192 rows, where the library is seldom at its best, by 12 % (6144 x 4096 at 150 39.6 -> 24.9); in one part of
//    the smallest or the larger tiles by 10 % (2048 x 8192 at 2709 91 -> 84), in parts for 7 of 8 CUs by 9 (1,800 sizes past 3
//    .87; past 9 6144 x 4096 at 386 31.3 -> 34.1); of 128 x 128 and a K up to 2,048 by 18 % (3072 x 2048 at 643 to 768 rows .86). Past each of these lines more than one size of 50 is
//    slower here; of 20,000 sizes of 760 weights at 33 rows and more that go here and that neither lines nor model were fitted to,
//    2.6 % are by more than 3 %, most of them by the next line, and all together take .82 of the library's time
//    (profiles/gemm_routes/tile.txt);
//  * past 32 rows what is over in 17 us (24 with SwiGLU) is taken all the same: the library's call costs the host 21 us, this
//    one 11, in parts 15. A prompt of 290 / 370 / 430 tokens of llama3.2-1b takes 2.85 / 2.83 / 2.82 ms with the library's
//    products and 1.94 / 1.98 / 2.00 with these, though 370 rows of 3072 x 2048 alone are 15.1 us there and 16.1 here. A
//    step of 33 and more sequences is replayed without the host, but there these are the quicker ones too: 38 sizes of 33 to 256
//    rows that this line decides take .87 of the library's time in the mean (10240 x 2048 at 65 rows 21.6 -> 15.6), one is slower
//    by more than 3 % (20480 x 1536 at 64 19.3 -> 21.1);
//  * more than 44 M weights (12288 x 4096 and up) are read at the rate of memory by the library as well, from 256 rows (K of
//    8192: 128) on it falls behind: 12288 x 4096 at 64 / 256 / 700 rows 26.7 / 1.21 / 1.23 times as fast here (26.8 at 64),
//    16384 x 4096 at 128 37.3 -> 41.8, 8192 x 8192 at 64 / 128 / 256 33.6 / 50.9 / 1.66 times (39.0, 43.0). So they are by a
//    step of up to 32 sequences from 20 M weights on (6144 x 4096 at 17 / 24 / 32 rows .89, .99, 1.0 times as fast, 16384 x
//    2048 1.03, .97, .96; but 4096 x 4096 1.18, 1.16, 1.16, 2048 x 8192 1.16, 1.14, 1.33), but for a K of 12288 and more of up
//    to 4096 channels past 16 rows (4096 x 14336 at 10 / 17 / 32 26.3 / 28.6 / 32.6 -> 27.1 / 26.0 / 26.4; 6144 x 16384 at 22
//    42.2 -> 50.7). With SwiGLU, whose launch is saved, up to 128 M (28672 x 4096 at 22 / 37 / 110 rows 54.2 / 51.0 / 54.7 ->
//    46.3 / 46.7 / 50.7; 57344 x 8192 is gemm8's), from 129 to 192 rows 100 M (28672 x 4096 at 130 / 157 / 205 61.4 / 60.5 /
//    73.7 -> 63.3 / 61.8 / 68.0, 21504 x 4096 at 135 61.1 -> 52.5), and a K of 12288 and more from 33 rows on (7168 x 16384 at
//    16 51.5 -> 66.9);
//  * a K of 12288 and more: up to 2^20 outputs, then gemm8 in parts of K (4096 x 14336 at 256 / 512 / 1024 rows 60.3* / 68.5* /
//    103.6* -> 47.6 / 68.4 / 119; 2048 x 12288 at 512 / 1400 1.18 and .87 times as fast);
//  * up to 256 channels, which are gates and routers, are not cut along K, whatever the rows: the side gate of sigusun-8b, 64 x
//    4096, takes 8 us for the library's 11 at 48 to 400 rows and 13 for 20 at 2048, 1 % of the pass, but f32 sums in parts
//    round otherwise than one sum in order, and where an expert's choice is close that shows in a pass' outputs (one of 17
//    differed by 3 %; the other way round as often). In one part, of which no line above is stretched for them, the library
//    mostly has it faster.
extern "C" int mx_gemm_tile_plan(int M, int N, int K, int swiglu) {
  if (M <= 0 || N <= 0 || K <= 0 || N % 16 || K % 64) return -1;
  const int64_t weights = (int64_t)N * K;
  const bool lengthy = K >= 12288;
  if (lengthy && (int64_t)M * N > (1 << 20)) return -1;
  if (swiglu ? weights > (M <= 128 || M > 192 ? 128000000 : 100000000) || (lengthy && M <= 32)
             : (!lengthy && weights > 44000000 && M < (K >= 8192 ? 128 : 256)) ||
                   (M <= 32 && weights > 20000000 && (!lengthy || M <= 16 || N > 4096)))
    return -1;
  const int nk = K / 64;
  const float quick = M <= 32 || N <= 256 ? 0.f : swiglu ? 24.f : 17.f;
  float best = INFINITY;
  int plan = -1;
  for (int i = 0; i < kGtCount; ++i) {
    const GtTile& t = kGtTiles[i];
    const int64_t tiles = gt_units(t, M, N);
    for (int S : {1, 2, 3, 4, 6, 8, 12, 16}) {
      const int64_t u = tiles * S;
      if (u > kGtPlaces || (S > 1 && (nk < 4 * S || N <= 256))) break;
      float us = t.start + (float)nk / S * (t.step + t.load * u / kGtPlaces) + t.memory * weights * 2e-6f;
      if (S > 1) us += t.sum + (t.part + (swiglu ? t.glu : 0.f)) * S + t.image * ((float)S * M * N * 4e-6f);
      const int least = i == 3 && K <= 4096 ? 10 : i == 2 && K <= 2048 ? 8 : K <= (i == 1 ? 2048 : 4096) ? 13 : 14;  // sixteenths
      if (S == 1 && i && !swiglu && K > 1024 && 16 * u < least * kGtPlaces && us > quick) continue;
      if (us < best) {
        best = us;
        plan = 64 * i + S;
      }
    }
  }
  if (plan < 0) return -1;
  const int tile = plan / 64, S = plan % 64;
  const bool filled = 8 * gt_units(kGtTiles[tile], M, N) * S >= 7 * kGtPlaces;
  const bool flat = !swiglu && S == 1 && tile == 2 && K <= 2048;
  const bool steady = !swiglu && (S == 1 ? tile < 1 || tile > 2 || K <= 1024 : filled && !lengthy);
  float most = gt_library(M, N, K);
  if (swiglu) most += 1.5f + .3f * ((float)M * N * 3e-6f);  // (its bytes: N in, N / 2 out)
  if (N > 256)
    most *= M <= 32 ? (swiglu && weights > 44000000 ? 1.12f : 1.05f)
                    : flat ? 1.18f : M <= 192 ? 1.12f : steady ? (S == 1 ? 1.1f : 1.09f) : 1.03f;
  return best < std::max(most, quick) ? plan : -1;
}

// C[M, N] = A . B^T, or (glu 1) C[M, N / 2] = silu(gate) up, by tile `tile` with K in `parts`; parts > 1: ws holds
// parts * M * N floats.  glu 2, one part only: the unit of inputs clipped to `limit` instead (sigusun's shared expert: 32 launches
// and a trip of the product of a prompt; sigusun-8b, 2048 tokens, 21.85 -> 21.69 ms).
// -1 (nothing launched) for shapes, strides and addresses that are not taken.
extern "C" int mx_gemm_tile(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, uint16_t* C, int64_t ldc, int M, int N,
                            int K, int glu, float limit, int tile, int parts, float* ws, hipStream_t stream) {
  const bool swiglu = glu != 0;
  if (glu < 0 || glu > 2 || (glu == 2 && parts != 1)) return -1;
  if (M <= 0 || N <= 0 || K <= 0 || N % 16 || K % 64 || tile < 0 || tile >= kGtCount || parts < 1 || parts > K / 64) return -1;
  if (lda % 8 || ldb % 8 || ldc % 8 || lda < K || ldb < K || ldc < (swiglu ? N / 2 : N)) return -1;
  if ((((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 15) || (parts > 1 && (!ws || ((uintptr_t)ws & 15)))) return -1;
  const GtTile& t = kGtTiles[tile];
  // offsets of 31 bits: the 32nd marks those past K
  if (t.tm * lda >= 1 << 30 || (swiglu ? N : t.tn) * ldb >= 1 << 30) return -1;
  const int64_t grid = gt_units(t, M, N) * parts;
  if (grid > INT32_MAX) return -1;
  if (parts > 1) {
    gt_launch<kGtPart>(tile, (int)grid, A, lda, B, ldb, ws, N, M, N, K, parts, stream);
    const int64_t units = (int64_t)M * (swiglu ? N / 2 : N) / 8;
    const int blocks = (int)std::min<int64_t>((units + 255) / 256, 4096);
    if (swiglu) g8_parts_kernel<true><<<blocks, 256, 0, stream>>>(ws, (int64_t)M * N, parts, N, C, ldc, units);
    else g8_parts_kernel<false><<<blocks, 256, 0, stream>>>(ws, (int64_t)M * N, parts, N, C, ldc, units);
  } else if (glu == 2) {
    gt_launch<kGtClipped>(tile, (int)grid, A, lda, B, ldb, C, ldc, M, N, K, 1, stream, limit);
  } else if (swiglu) {
    gt_launch<kGtSwiglu>(tile, (int)grid, A, lda, B, ldb, C, ldc, M, N, K, 1, stream);
  } else {
    gt_launch<kGtPlain>(tile, (int)grid, A, lda, B, ldb, C, ldc, M, N, K, 1, stream);
  }
  return (int)hipGetLastError();
}
