// The tile loop of the bf16 GEMMs whose output is one turn of tiles (gemm_tile.hip: projections of prompt passes, where its
// structure is told; gemm_tile_forms.hip: a training step's gradients).
#pragma once

#include "gemm8_core.h"
#include "hybrid.h"

namespace mx {

constexpr int kGtPlain = 0, kGtSwiglu = 1, kGtPart = 2, kGtAdd = 3, kGtClipped = 4;
constexpr bool gt_glu(int epi) { return epi == kGtSwiglu || epi == kGtClipped; }

template <int N>
__device__ __forceinline__ void gt_vm_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// row of B behind virtual column v of tile pn: with SwiGLU a wave's first half of columns are gate's, the second the same
// channels of up
template <int TN, int WN, int EPI>
__device__ __forceinline__ int gt_row(int v, int pn, int F) {
  if constexpr (!gt_glu(EPI)) return pn * TN + v;
  constexpr int HW = TN / WN / 2;
  const int q = v % (2 * HW);
  return (q < HW ? 0 : F) + pn * (TN / 2) + v / (2 * HW) * HW + q % HW;
}

// An operand stored [K][rows] (a weight gradient's two, an input gradient's weights): a stage holds its tile as blocks of 64 rows,
// [64 k][64], 128 B a k.  Chunk c of a k lies at c ^ 2 f(k): the 32 lanes of half a transposed read take 32 B of 8 k (4 g + q of
// two g) and meet every bank once.
__device__ __forceinline__ int gt_f(int k) { return ((k >> 1) & 1) | ((k >> 3) & 1) << 1; }
// lane part of the address of a transposed read of rows 16 idx .. + 15 of a block, k 8 g .. + 3 of a step (4 k on: + 512 B)
__device__ __forceinline__ uint32_t gt_mn_lane(int lane, int idx) {
  const int g = lane >> 4, q = (lane & 15) >> 2, p = lane & 3, k = 8 * g + q;
  return (uint32_t)(k * 128 + 32 * (idx ^ gt_f(k)) + 8 * p);
}

// TM x TN tile by WM x WN waves, S stages of LDS, OCC workgroups a CU (a launch bound: 256 registers a wave at 2).  kGtPart: C is
// f32 [parts][M][N]; kGtAdd: the product is added to C; kGtClipped: as kGtSwiglu, the unit of inputs clipped to `limit` (hybrid.h).
// AK, BK: A is [M][K], B is [N][K]; else [K][M], [K][N].
template <int TM, int TN, int WM, int WN, int S, int OCC, int EPI, bool AK = true, bool BK = true>
__global__ void __launch_bounds__(64 * WM * WN, OCC)
gemm_tile_kernel(const uint16_t* __restrict__ A, int64_t lda, const uint16_t* __restrict__ B, int64_t ldb, void* __restrict__ C,
                 int64_t ldc, int M, int N, int K, int parts, float limit = 0.f) {
  constexpr int NW = WM * WN, BI = TM / WM / 16, BJ = TN / WN / 16, STG = (TM + TN) * 128;
  constexpr int QA = TM / 8 / NW, QB = TN / 8 / NW, P = QA + QB;  // DMA pieces of 8 rows of a wave: of A, of B
  constexpr int NM = BI * BJ, NR = BI + BJ;                      // MFMAs and fragments of a step
  constexpr int NB = NM / 4 < NM - NR ? NM / 4 : NM - NR;        // MFMAs of the second step ahead of the barrier
  constexpr int RA = AK ? 1 : 2, RB = BK ? 1 : 2;                // LDS reads of a fragment
  constexpr int R0 = NM >= 2 * NR ? 2 : 1, R1 = NM - NB >= 2 * NR ? 2 : 1;         // MFMAs from one fragment read to the next
  constexpr int D0 = NM / (P - P / 2), D1 = (NM - NB) / (P / 2);  // and from one DMA piece to the next
  static_assert(TM % (8 * NW) == 0 && TN % (8 * NW) == 0 && BJ % 2 == 0 && S >= 3 && NB >= 0 && D0 > 0 && D1 > 0, "tile");
  __shared__ __attribute__((aligned(1024))) char smem[S * STG];
  const int nM = (M + TM - 1) / TM, nN = (N + TN - 1) / TN, F = N / 2;
  int pm, pn, nk = AK || BK ? K / 64 : (K + 63) / 64;
  {
    int L = xcd_remap(blockIdx.x, gridDim.x);
    if constexpr (EPI == kGtPart) {  // parts after each other: an XCD's tiles share the panels of one part of K
      const int kp = L / (nM * nN), t0 = nk * kp / parts, t1 = nk * (kp + 1) / parts;
      L -= kp * nM * nN;
      A += AK ? t0 * 64 : (int64_t)t0 * 64 * lda;
      B += BK ? t0 * 64 : (int64_t)t0 * 64 * ldb;
      K -= t0 * 64;
      nk = t1 - t0;
      C = reinterpret_cast<float*>(C) + (int64_t)kp * M * N;
    }
    constexpr int GM = 8;  // a band of 8 tiles down, then across: an XCD's tiles share their panels in its L2
    const int per = GM * nN, grp = L / per, first = grp * GM;
    const int rows = min(GM, nM - first), in = L - grp * per;
    pm = first + in % rows;
    pn = in / rows;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / WN, wn = w % WN;
  // rows past M and N read the last one again: their products are not stored
  const int mrem = M - pm * TM;
  const uint16_t* ab = A + (int64_t)pm * TM * (AK ? lda : 1);
  const uint16_t* bb = B + (gt_glu(EPI) ? 0 : (int64_t)pn * TN * (BK ? ldb : 1));
  const int brows = gt_glu(EPI) ? N : min(N - pn * TN, TN);
  const int64_t arec = AK ? (min(mrem, TM) - 1) * lda + K : (K - 1) * lda + mrem;
  const int64_t brec = BK ? (brows - 1) * ldb + K : (K - 1) * ldb + N - pn * TN;
  const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc((void*)ab, 0, (uint32_t)(arec * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc((void*)bb, 0, (uint32_t)(brec * 2), 0x00020000);
  const uint32_t astep = AK ? 128 : (uint32_t)(128 * lda), bstep = BK ? 128 : (uint32_t)(128 * ldb);  // bytes of 64 k
  uint32_t off[P];
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int pc = j < QA ? w * QA + j : w * QB + j - QA, r = 8 * pc + (lane >> 3);
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    if (j < QA ? !AK : !BK) {  // (rows past the tile's end: others of the same k, or past the end; not stored either)
      const int k = 8 * (pc & 7) + (lane >> 3);
      off[j] = (uint32_t)((k * (j < QA ? lda : ldb) + 64 * (pc >> 3) + 8 * ((lane & 7) ^ (2 * gt_f(k)))) * 2);
    } else if (j < QA) {
      off[j] = (uint32_t)((min(r, mrem - 1) * lda + 8 * c) * 2);
    } else {
      const int b = min(gt_row<TN, WN, EPI>(r, pn, F), N - 1) - (gt_glu(EPI) ? 0 : pn * TN);
      off[j] = (uint32_t)((b * ldb + 8 * c) * 2);
    }
  }
  // kt: the tile of 64 k, or one past K: out of the descriptors' range
  auto piece = [&](int j, int kt, char* dst) __attribute__((always_inline)) {
    const uint32_t so = off[j] + (kt < nk ? (uint32_t)kt * (j < QA ? astep : bstep) : G8_OOB);
    char* d = dst + (j < QA ? (w * QA + j) * 1024 : TM * 128 + (w * QB + j - QA) * 1024);
    if (j < QA) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ars, (g8lptr_t)d, 16, so, 0, 0, 0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(brs, (g8lptr_t)d, 16, so, 0, 0, 0);
    }
  };
  const uint32_t lds0 = lds_addr(smem);
  uint32_t al[2], bl[2], am[BI], bm[BJ];  // [K][rows]: a fragment's rows each, steps and halves are immediates
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    al[s] = lds0 + g8_kc_lane(lane, s) + wm * (TM / WM) * 128;
    bl[s] = lds0 + g8_kc_lane(lane, s) + TM * 128 + wn * (TN / WN) * 128;
  }
#pragma unroll
  for (int i = 0; i < BI; ++i) {
    const int r = wm * BI + i;
    am[i] = lds0 + (r >> 2) * 8192 + gt_mn_lane(lane, r & 3);
  }
#pragma unroll
  for (int j = 0; j < BJ; ++j) {
    const int r = wn * BJ + j;
    bm[j] = lds0 + TM * 128 + (r >> 2) * 8192 + gt_mn_lane(lane, r & 3);
  }
  u16x8 fa[2][BI], fb[2][BJ];
  u16x4 ta[2][BI][2], tb[2][BJ][2];  // transposed reads' halves (put together behind their wait)
  f32x4 acc[BI][BJ];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // fragment r of set s, step s of stage `st`: B's first, then A's
  auto read = [&](int s, int r, uint32_t st) __attribute__((always_inline)) {
    if (r < BJ) {
      if constexpr (BK) {
        fb[s][r] = rd128_off(bl[s] + st, r * 2048);
      } else {
        tb[s][r][0] = trd_off(bm[r] + st, 4096 * s);
        tb[s][r][1] = trd_off(bm[r] + st, 4096 * s + 512);
      }
    } else {
      if constexpr (AK) {
        fa[s][r - BJ] = rd128_off(al[s] + st, (r - BJ) * 2048);
      } else {
        ta[s][r - BJ][0] = trd_off(am[r - BJ] + st, 4096 * s);
        ta[s][r - BJ][1] = trd_off(am[r - BJ] + st, 4096 * s + 512);
      }
    }
  };
  auto whole = [](const u16x4& x, const u16x4& y) { return u16x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]}; };
  // LDS reads of the first n fragments
  auto reads = [](int n) { return min(n, BJ) * RB + max(n - BJ, 0) * RA; };
  // A's fragment i of set s, and with the first all of B's, are there once at most `left` younger LDS reads are not
  auto have = [&](int s, int i, int left) __attribute__((always_inline)) {
    lds_wait_le(left > 15 ? 15 : left);
    if constexpr (AK) {
      pin(fa[s][i]);
    } else {
      pin(ta[s][i][0]);
      pin(ta[s][i][1]);
      fa[s][i] = whole(ta[s][i][0], ta[s][i][1]);
    }
    if (i == 0) {
#pragma unroll
      for (int j = 0; j < BJ; ++j) {
        if constexpr (BK) {
          pin(fb[s][j]);
        } else {
          pin(tb[s][j][0]);
          pin(tb[s][j][1]);
          fb[s][j] = whole(tb[s][j][0], tb[s][j][1]);
        }
      }
    }
  };

#pragma unroll
  for (int t = 0; t < S; ++t)
#pragma unroll
    for (int j = 0; j < P; ++j) piece(j, t, smem + t * STG);
  gt_vm_wait<(S - 1) * P>();
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int r = 0; r < NR; ++r) read(0, r, 0);
  int st = 0;  // stage of kt
  for (int kt = 0; kt < nk; ++kt) {
    const int nx = st + 1 == S ? 0 : st + 1;
    {  // step 0: multiply set 0, read set 1; the second half of tile kt + S - 1's pieces
      char* dst = smem + (st == 0 ? S - 1 : st - 1) * STG;
#pragma unroll
      for (int n = 0; n < NM; ++n) {
        const int i = n / BJ, j = n % BJ, r = n / R0, d = n / D0;
        if (j == 0) have(0, i, (BI - 1 - i) * RA + reads(min((n + R0 - 1) / R0, NR)));
        acc[i][j] = g8_mfma(fb[0][j], fa[0][i], acc[i][j]);
        if (n % R0 == 0 && r < NR) read(1, r, st * STG);
        if (n % D0 == D0 - 1 && d < P - P / 2 && kt > 0) piece(P / 2 + d, kt + S - 1, dst);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    {  // step 1: multiply set 1; behind the barrier read set 0 of the next tile, and the first half of tile kt + S's pieces
      char* dst = smem + st * STG;
#pragma unroll
      for (int n = 0; n < NM; ++n) {
        const int i = n / BJ, j = n % BJ, q = n - NB, r = q / R1, d = q / D1;
        if (q == 0) {  // this wave's reads of stage st are done, its pieces of tile kt + 1 landed
          lds_wait();
          gt_vm_wait<(S - 2) * P>();
          __builtin_amdgcn_s_barrier();
        }
        if (j == 0) have(1, i, q < 0 ? (BI - 1 - i) * RA : 15);
        acc[i][j] = g8_mfma(fb[1][j], fa[1][i], acc[i][j]);
        if (q >= 0 && q % R1 == 0 && r < NR) read(0, r, nx * STG);  // (behind the last tile: bytes that are not multiplied)
        if (q >= 0 && q % D1 == D1 - 1 && d < P / 2) piece(d, kt + S, dst);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    st = nx;
  }
  // the reads behind the last tile own their registers, and the DMA behind K its LDS, until here
#pragma unroll
  for (int i = 0; i < BI; ++i) have(0, i, 0);
  gt_vm_wait<0>();
  const int ml = pm * TM + wm * (TM / WM) + (lane & 15);
  if constexpr (EPI == kGtPart) {
    float* c = reinterpret_cast<float*>(C);
    const int n0 = pn * TN + wn * (TN / WN) + 4 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j)
        if (ml + 16 * i < M && n0 + 16 * j < N)
          *reinterpret_cast<f32x4*>(c + (int64_t)(ml + 16 * i) * N + n0 + 16 * j) = acc[i][j];
  } else if constexpr (EPI == kGtAdd) {  // the sum is rounded once
    uint16_t* c = reinterpret_cast<uint16_t*>(C);
    const int n0 = pn * TN + wn * (TN / WN) + 4 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < BI; ++i) {
      u16x4 o[BJ];
#pragma unroll
      for (int j = 0; j < BJ; ++j)
        if (ml + 16 * i < M && n0 + 16 * j < N) o[j] = *reinterpret_cast<const u16x4*>(c + (int64_t)(ml + 16 * i) * ldc + n0 + 16 * j);
#pragma unroll
      for (int j = 0; j < BJ; ++j)
        if (ml + 16 * i < M && n0 + 16 * j < N) {
#pragma unroll
          for (int e = 0; e < 4; ++e) o[j][e] = f2bf(acc[i][j][e] + bf2f(o[j][e]));
          *reinterpret_cast<u16x4*>(c + (int64_t)(ml + 16 * i) * ldc + n0 + 16 * j) = o[j];
        }
    }
  } else if constexpr (gt_glu(EPI)) {
    uint16_t* c = reinterpret_cast<uint16_t*>(C);
    const int n0 = pn * (TN / 2) + wn * (TN / WN / 2) + 4 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ / 2; ++j) {
        u16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g = g8_rbf(acc[i][j][e]), u = g8_rbf(acc[i][BJ / 2 + j][e]);
          o[e] = f2bf(EPI == kGtClipped ? clipped_glu<uint16_t>(g, u, limit) : g * g8_sigmoid(g) * u);
        }
        if (ml + 16 * i < M && n0 + 16 * j < F) *reinterpret_cast<u16x4*>(c + (int64_t)(ml + 16 * i) * ldc + n0 + 16 * j) = o;
      }
  } else {
    uint16_t* c = reinterpret_cast<uint16_t*>(C);
    const int n0 = pn * TN + wn * (TN / WN) + 16 * ((lane >> 4) & 1) + 8 * (lane >> 5);
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; j += 2) {
        const uint4 o = g8_pack8(acc[i][j], acc[i][j + 1]);  // lanes exchange: outside the row test
        if (ml + 16 * i < M && n0 + 16 * j < N) *reinterpret_cast<uint4*>(c + (int64_t)(ml + 16 * i) * ldc + n0 + 16 * j) = o;
      }
  }
}

}  // namespace mx
