// Causal GQA flash-attention backward for heads of 64 (training), in two passes that each form the scores again:
//
//   query pass   S^T = K Q^T, dP^T = V dO^T, dS^T = P^T (dP^T - delta), dQ^T += K^T dS^T; it also makes delta
//   key pass     S = Q K^T,   dP = dO V^T,   dS = P (dP - delta),       dV^T += dO^T P,  dK^T += Q^T dS
//   P = exp2(S * sl - lse)
//
// With dS^T handed from the key pass to the query pass through memory (as attn_bwd.hip does it for heads of 128) two
// sequences of 2,048 x 32 heads took 284 us: 290 MB written by a key pass of one wave a SIMD, 201 us, read again in 74, and
// delta.  At 64 channels a product is cheap next to that: forming S and dP once more is 8 MFMAs of 32 cycles a 32 x 32 block.
// The two passes take 74 + 88 us there, in a training step as those figures are (0.53 PF/s of the five products that a backward
// cannot do without).  Replayed alone 158 to 172 from card to card; one sequence of 4,096 480 -> 275, four of 777 113 -> 78, four of 150
// 24 -> 19.  What bounds them: products and exponentials of a wave follow each other, and two waves a SIMD hide about half of one
// behind the other (matrix cores busy 45 % of the time, vector ALU 44 %).
// At 128 channels the products double and the bytes of dS^T stay: there the image is the cheaper one.
//
// Both kernels: workgroup = 4 waves, 32 rows (queries or keys) a wave, which sit in registers as B operands of
// v_mfma_f32_32x32x16_bf16 while 64-row tiles of the other side come through LDS.  Accumulators rounded to bf16 are the next
// product's B operand as they are; its A operand is a transposed read (ds_read_b64_tr_b16) of the same tile.  The scores of a
// tile's two blocks are formed ahead of both their exponentials, so that the second block's products can run under the
// first's exponentials (174 -> 149 us; an order of instructions given by sched_group_barrier 162).  Tiles that need masks are
// the first or the last ones and have a loop of their own: the other one has no branches.
#include <algorithm>

#include "common.h"

namespace mx {
namespace {

typedef __bf16 bf16x8_q __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4_q;

constexpr int kD = 64, kRowB = 128, kTile = 64 * kRowB;  // a tile of 64 rows, [64][64] bf16

__device__ __forceinline__ f32x16 mma(const u16x8& a, const u16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_q, a), __builtin_bit_cast(bf16x8_q, b), c, 0,
                                                 0, 0);
}
// 16-byte chunks of a row are stored at chunk ^ swz(row): both reads below are free of bank conflicts, and rows 16 apart
// share it
__device__ __forceinline__ int swz(int row) { return (((row >> 1) & 1) << 2) | ((row >> 2) & 3); }
__device__ __forceinline__ u16x8 row_frag(const char* tile, int at) {
  return *reinterpret_cast<const u16x8*>(tile + at);
}
// rows a .. a + 3 and a + 8 .. a + 11 of 16 (those an accumulator's eight registers hold), 32 columns
__device__ __forceinline__ u16x8 col_frag(const char* tile, int a, int b) {
  const u16x4 x = __builtin_bit_cast(u16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_q*)(tile + a)));
  const u16x4 y = __builtin_bit_cast(u16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_q*)(tile + b)));
  return u16x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
}
__device__ __forceinline__ u16x8 pack8(const f32x16& v, int at) {
  u16x8 r;
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = f2bf(v[at + j]);
  return r;
}
// lane J of each sixteen to all of them: the value of accumulator register J where lane l holds that of row
// (l & 3) + 8 ((l & 15) >> 2) + 4 (l >> 5)
template <int J>
__device__ __forceinline__ float of_reg(float v) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(v), 0x150 + J, 0xF, 0xF, true));
}
template <int J = 0, typename F>
__device__ __forceinline__ void each_reg(F&& f) {
  f(std::integral_constant<int, J>{});
  if constexpr (J + 1 < 16) each_reg<J + 1>(f);
}
__device__ __forceinline__ f32x16 all16(float v) {
  f32x16 z;
#pragma unroll
  for (int j = 0; j < 16; ++j) z[j] = v;
  return z;
}
__device__ __forceinline__ u16x8 load16(__amdgpu_buffer_rsrc_t rs, int at) {  // (past the end: zeros)
  return __builtin_bit_cast(u16x8, __builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, 0));
}

// dQ of 128 query rows of one head, 32 a wave, and what the key pass takes of them: -delta = -sum_d dO O.  The tiles of K and
// V come through registers (two LDS buffers): a tile's loads are asked for before the products of the one ahead of it and
// stored after them.  dq f32 [B, Hq, S, 64]; or with dqkv its q columns (rows of ldq): scaled, turned back by the rotation
// and rounded once, as rope_merge_bwd_kernel does it; columns d and d + 32 of a row are registers of one lane.
template <bool CAUSAL>
__global__ void __launch_bounds__(256, 2)
attn_bwd64_q_kernel(const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K, const uint16_t* __restrict__ V,
                    const uint16_t* __restrict__ O, const uint16_t* __restrict__ dO, const float* __restrict__ LSE,
                    float* __restrict__ NDELTA, float* __restrict__ dQ, uint16_t* __restrict__ dqkv,
                    const float* __restrict__ cosb, const float* __restrict__ sinb, int B, int Hq, int Hkv, int S, int Sk,
                    int off, float sl, float scale, int64_t ldo, int64_t ldq) {
  constexpr int BM = 128, BN = 64;
  __shared__ __attribute__((aligned(1024))) char smem[2 * 2 * kTile];
  const int nqb = (S + BM - 1) / BM, BH = B * Hq;
  const int bid = xcd_balance(blockIdx.x, gridDim.x, BH, Hq / Hkv);
  const int qb = nqb - 1 - bid / BH, bh = bid % BH;  // the blocks with most keys first
  const int b = bh / Hq, h = bh % Hq, hk = h / (Hq / Hkv);
  const __amdgpu_buffer_rsrc_t krs =
      __builtin_amdgcn_make_buffer_rsrc((void*)(K + (size_t)(b * Hkv + hk) * Sk * kD), 0, Sk * kRowB, 0x00020000);
  const __amdgpu_buffer_rsrc_t vrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)(V + (size_t)(b * Hkv + hk) * Sk * kD), 0, Sk * kRowB, 0x00020000);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, hh = lane >> 5;
  const int g = lane >> 4, tq = (lane & 15) >> 2, tp = lane & 3;
  const int q0 = qb * BM + 32 * w, q = q0 + r, qld = min(q, S - 1);

  // staging: chunks tid and tid + 256 of a tile
  const int srow = tid >> 3, sch = tid & 7;
  char* const sat = smem + srow * kRowB + 16 * (sch ^ swz(srow));
  const int nkt = CAUSAL ? max(0, (min(Sk, qb * BM + BM + off) + BN - 1) / BN) : (Sk + BN - 1) / BN;
  // tiles that every row of the workgroup sees whole
  const int nfull = CAUSAL ? min(max(0, (qb * BM + off + 1) / BN), Sk / BN) : Sk / BN;
  u16x8 k0s, k1s, v0s, v1s;
  auto fetch = [&](int kt) {
    const int at = kt * kTile + tid * 16;
    k0s = load16(krs, at), v0s = load16(vrs, at);
    k1s = load16(krs, at + kTile / 2), v1s = load16(vrs, at + kTile / 2);
  };
  auto stage = [&](int buf) {
    char* t = sat + buf * 2 * kTile;
    *reinterpret_cast<u16x8*>(t) = k0s;
    *reinterpret_cast<u16x8*>(t + kTile / 2) = k1s;
    *reinterpret_cast<u16x8*>(t + kTile) = v0s;
    *reinterpret_cast<u16x8*>(t + kTile + kTile / 2) = v1s;
  };
  if (nkt > 0) fetch(0);

  u16x8 qf[4], gf[4];
  const uint16_t* Qr = Q + ((size_t)bh * S + qld) * kD + 8 * hh;
  const uint16_t* Gr = dO + ((size_t)b * S + qld) * Hq * kD + h * kD + 8 * hh;
  const uint16_t* Or = O + ((size_t)b * S + qld) * ldo + h * kD + 8 * hh;
  float nd = 0.f;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    qf[s] = *reinterpret_cast<const u16x8*>(Qr + 16 * s);
    gf[s] = *reinterpret_cast<const u16x8*>(Gr + 16 * s);
    const u16x8 x = *reinterpret_cast<const u16x8*>(Or + 16 * s);
#pragma unroll
    for (int j = 0; j < 8; ++j) nd -= bf2f(gf[s][j]) * bf2f(x[j]);
  }
  nd = lane_sum<32>(nd);
  if (hh == 0 && q < S) NDELTA[(size_t)bh * S + q] = nd;
  const float nl = -LSE[(size_t)bh * S + qld];

  // byte offsets within a tile: row r at k step s is ra ^ 32 s
  const int ra = r * kRowB + 16 * (hh ^ swz(r));
  const int rA = 4 * hh + tq, rB = rA + 8, cch = (16 * (g & 1) + 4 * tp) >> 3;
  const int ca = rA * kRowB + 16 * (cch ^ swz(rA)) + 8 * (tp & 1), cb = rB * kRowB + 16 * (cch ^ swz(rB)) + 8 * (tp & 1);
  f32x16 acc0 = all16(0.f), acc1 = all16(0.f);

  auto tile = [&](int kt, auto masked) {
    const char* kimg = smem + (kt & 1) * 2 * kTile;
    const char* vimg = kimg + kTile;
    f32x16 sa[2], dp[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      sa[n] = all16(0.f), dp[n] = all16(nd);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        sa[n] = mma(row_frag(kimg, (ra ^ (32 * s)) + 32 * n * kRowB), qf[s], sa[n]);
        dp[n] = mma(row_frag(vimg, (ra ^ (32 * s)) + 32 * n * kRowB), gf[s], dp[n]);
      }
    }
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      // register j: key kt BN + 32 n + (j & 3) + 8 (j >> 2) + 4 hh; lane: query
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sa[n][j], sl, nl));
        if constexpr (masked.value) {
          const int key = kt * BN + 32 * n + (j & 3) + 8 * (j >> 2) + 4 * hh;
          p = (key >= Sk) | (CAUSAL & (key > q + off)) ? 0.f : p;
        }
        dp[n][j] *= p;
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const u16x8 ds = pack8(dp[n], 8 * s);
        const char* t = kimg + (32 * n + 16 * s) * kRowB;
        acc0 = mma(col_frag(t, ca, cb), ds, acc0);
        acc1 = mma(col_frag(t, ca ^ 64, cb ^ 64), ds, acc1);  // (channels 32 .. 63: chunk + 4)
      }
    }
  };
  if (nkt > 0) stage(0);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // (all loads so far: the loop is left to wait for its own alone)
  __syncthreads();
  for (int kt = 0; kt < nfull; ++kt) {
    if (kt + 1 < nkt) fetch(kt + 1);
    tile(kt, std::false_type{});
    if (kt + 1 < nkt) stage((kt + 1) & 1);  // last read a tile ago, before the barrier
    __syncthreads();
  }
  for (int kt = nfull; kt < nkt; ++kt) {
    if (kt + 1 < nkt) fetch(kt + 1);
    if (!CAUSAL || kt * BN <= q0 + 31 + off) tile(kt, std::true_type{});  // some row of this wave sees the tile
    if (kt + 1 < nkt) stage((kt + 1) & 1);
    __syncthreads();
  }
  if (q >= S) return;
  // register j of acc0, acc1: channel (j & 3) + 8 (j >> 2) + 4 hh, and 32 on
  if (dqkv) {
    const float* cp = cosb + (int64_t)q * (kD / 2) + 4 * hh;
    const float* sp = sinb + (int64_t)q * (kD / 2) + 4 * hh;
    uint16_t* dst = dqkv + ((int64_t)b * S + q) * ldq + (int64_t)h * kD + 4 * hh;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const f32x4 c = *reinterpret_cast<const f32x4*>(cp + 8 * t), s = *reinterpret_cast<const f32x4*>(sp + 8 * t);
      u16x4 y1, y2;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float a1 = acc0[4 * t + j] * scale, a2 = acc1[4 * t + j] * scale;
        y1[j] = f2bf(__builtin_fmaf(a1, c[j], a2 * s[j]));  // the contraction of rope_merge_bwd_kernel
        y2[j] = f2bf(__builtin_fmaf(a2, c[j], -(a1 * s[j])));
      }
      *reinterpret_cast<u16x4*>(dst + 8 * t) = y1;
      *reinterpret_cast<u16x4*>(dst + 8 * t + kD / 2) = y2;
    }
  } else {
    float* dst = dQ + ((size_t)bh * S + q) * kD + 4 * hh;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      *reinterpret_cast<f32x4*>(dst + 8 * t) =
          f32x4{acc0[4 * t] * scale, acc0[4 * t + 1] * scale, acc0[4 * t + 2] * scale, acc0[4 * t + 3] * scale};
      *reinterpret_cast<f32x4*>(dst + 32 + 8 * t) =
          f32x4{acc1[4 * t] * scale, acc1[4 * t + 1] * scale, acc1[4 * t + 2] * scale, acc1[4 * t + 3] * scale};
    }
  }
}

// dK and dV of 128 keys for one query head, 32 a wave (the partials [B, Hq, Sk, 64] f32 that rope_merge_bwd sums over a KV
// head's query heads).  A query's lse and delta are needed by the register that holds its row: a lane holds one row's, and
// a row of sixteen lanes hands each out by DPP (four 16-byte LDS reads of each a block would make LDS the slowest part);
// -delta is what dP's sum starts from.  Keys past Sk are lanes that are not stored; queries past S have zero rows and an lse
// of infinity, so P is 0.
template <bool CAUSAL>
__global__ void __launch_bounds__(256, 2)
attn_bwd64_kv_kernel(const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K, const uint16_t* __restrict__ V,
                     const uint16_t* __restrict__ dO, const float* __restrict__ LSE, const float* __restrict__ NDELTA,
                     float* __restrict__ dKp, float* __restrict__ dVp, int B, int Hq, int Hkv, int S, int Sk, int off,
                     float sl, float scale) {
  constexpr int BN = 128, BQ = 64;
  __shared__ __attribute__((aligned(1024))) char smem[2 * 2 * kTile];
  const int BH = B * Hq;
  const int bid = xcd_balance(blockIdx.x, gridDim.x, BH, Hq / Hkv);
  const int kb = bid / BH, bh = bid % BH;  // causal: the first keys are seen by most queries
  const int b = bh / Hq, h = bh % Hq, hk = h / (Hq / Hkv);
  const int grow = Hq * kRowB;  // bytes of a row of dO
  const __amdgpu_buffer_rsrc_t qrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)(Q + (size_t)bh * S * kD), 0, S * kRowB, 0x00020000);
  const uint16_t* gbase = dO + ((size_t)b * S * Hq + h) * kD;
  const float* lsep = LSE + (size_t)bh * S;
  const float* ndp = NDELTA + (size_t)bh * S;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, hh = lane >> 5;
  const int g = lane >> 4, tq = (lane & 15) >> 2, tp = lane & 3;
  const int k0 = kb * BN + 32 * w, key = k0 + r;

  const int srow = tid >> 3, sch = tid & 7;
  char* const sat = smem + srow * kRowB + 16 * (sch ^ swz(srow));
  const int qstart = CAUSAL ? max(0, (kb * BN - off) / BQ * BQ) : 0;
  const int nqt = qstart < S ? (S - qstart + BQ - 1) / BQ : 0;
  // the first tiles, which not all keys of the workgroup are seen in whole
  const int nmask = CAUSAL ? min(nqt, max(0, (kb * BN + BN - 1 - off - qstart + BQ - 1) / BQ)) : 0;
  const int lrow = qstart + (lane & 3) + 8 * ((lane & 15) >> 2) + 4 * hh;
  u16x8 q0s, q1s, g0s, g1s;
  float l0n, l1n, d0n, d1n;  // the lane's row of each 32: lse, -delta
  auto fetch = [&](int it) {
    const int at = (qstart * kRowB) + it * kTile + tid * 16;
    // (a descriptor a tile: a sequence's dO can be longer than 4 GiB)
    const int row = qstart + it * BQ, ga = srow * grow + 16 * sch;
    const __amdgpu_buffer_rsrc_t grs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(gbase + (size_t)row * Hq * kD), 0, (min(S - row, BQ) - 1) * grow + kRowB, 0x00020000);
    q0s = load16(qrs, at), g0s = load16(grs, ga);
    q1s = load16(qrs, at + kTile / 2), g1s = load16(grs, ga + 32 * grow);
    const int a = min(lrow + it * BQ, S - 1), c = min(lrow + it * BQ + 32, S - 1);
    l0n = lsep[a], l1n = lsep[c], d0n = ndp[a], d1n = ndp[c];
  };
  auto stage = [&](int buf) {
    char* t = sat + buf * 2 * kTile;
    *reinterpret_cast<u16x8*>(t) = q0s;
    *reinterpret_cast<u16x8*>(t + kTile / 2) = q1s;
    *reinterpret_cast<u16x8*>(t + kTile) = g0s;
    *reinterpret_cast<u16x8*>(t + kTile + kTile / 2) = g1s;
  };
  if (nqt > 0) fetch(0);

  u16x8 kf[4], vf[4];
  const size_t kat = ((size_t)(b * Hkv + hk) * Sk + min(key, Sk - 1)) * kD + 8 * hh;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    kf[s] = *reinterpret_cast<const u16x8*>(K + kat + 16 * s);
    vf[s] = *reinterpret_cast<const u16x8*>(V + kat + 16 * s);
  }
  const int ra = r * kRowB + 16 * (hh ^ swz(r));
  const int rA = 4 * hh + tq, rB = rA + 8, cch = (16 * (g & 1) + 4 * tp) >> 3;
  const int ca = rA * kRowB + 16 * (cch ^ swz(rA)) + 8 * (tp & 1), cb = rB * kRowB + 16 * (cch ^ swz(rB)) + 8 * (tp & 1);
  f32x16 dk0 = all16(0.f), dk1 = all16(0.f), dv0 = all16(0.f), dv1 = all16(0.f);

  auto tile = [&](int it, float l0, float l1, float d0, float d1, auto masked) {
    const int q0 = qstart + it * BQ;
    const char* qimg = smem + (it & 1) * 2 * kTile;
    const char* gimg = qimg + kTile;
    f32x16 sa[2], dp[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const float nd = m ? d1 : d0;
      sa[m] = all16(0.f);
      each_reg([&](auto jc) { dp[m][jc.value] = of_reg<jc.value>(nd); });
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        sa[m] = mma(row_frag(qimg, (ra ^ (32 * s)) + 32 * m * kRowB), kf[s], sa[m]);
        dp[m] = mma(row_frag(gimg, (ra ^ (32 * s)) + 32 * m * kRowB), vf[s], dp[m]);
      }
    }
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const float l = m ? l1 : l0;
      // register j: query q0 + 32 m + (j & 3) + 8 (j >> 2) + 4 hh; lane: key
      each_reg([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sa[m][j], sl, -of_reg<j>(l)));
        if constexpr (masked.value) p = key > q0 + 32 * m + (j & 3) + 8 * (j >> 2) + 4 * hh + off ? 0.f : p;
        sa[m][j] = p;
        dp[m][j] *= p;
      });
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const u16x8 p = pack8(sa[m], 8 * s), ds = pack8(dp[m], 8 * s);
        const int at = (32 * m + 16 * s) * kRowB;
        dv0 = mma(col_frag(gimg + at, ca, cb), p, dv0);
        dv1 = mma(col_frag(gimg + at, ca ^ 64, cb ^ 64), p, dv1);
        dk0 = mma(col_frag(qimg + at, ca, cb), ds, dk0);
        dk1 = mma(col_frag(qimg + at, ca ^ 64, cb ^ 64), ds, dk1);
      }
    }
  };
  auto step = [&](int it, auto masked) {
    const int q = lrow + it * BQ;
    const float l0 = q < S ? l0n : INFINITY, l1 = q + 32 < S ? l1n : INFINITY, d0 = d0n, d1 = d1n;
    if (it + 1 < nqt) fetch(it + 1);
    // (masked: nothing where no row of the tile sees a key of this wave)
    if (!masked.value || k0 <= qstart + it * BQ + BQ - 1 + off) tile(it, l0, l1, d0, d1, masked);
    if (it + 1 < nqt) stage((it + 1) & 1);
    __syncthreads();
  };
  if (nqt > 0) stage(0);
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  for (int it = 0; it < nmask; ++it) step(it, std::true_type{});
  for (int it = nmask; it < nqt; ++it) step(it, std::false_type{});
  if (key >= Sk) return;
  float* dkq = dKp + ((size_t)bh * Sk + key) * kD + 4 * hh;
  float* dvq = dVp + ((size_t)bh * Sk + key) * kD + 4 * hh;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    *reinterpret_cast<f32x4*>(dkq + 8 * t) =
        f32x4{dk0[4 * t] * scale, dk0[4 * t + 1] * scale, dk0[4 * t + 2] * scale, dk0[4 * t + 3] * scale};
    *reinterpret_cast<f32x4*>(dkq + 32 + 8 * t) =
        f32x4{dk1[4 * t] * scale, dk1[4 * t + 1] * scale, dk1[4 * t + 2] * scale, dk1[4 * t + 3] * scale};
    *reinterpret_cast<f32x4*>(dvq + 8 * t) = f32x4{dv0[4 * t], dv0[4 * t + 1], dv0[4 * t + 2], dv0[4 * t + 3]};
    *reinterpret_cast<f32x4*>(dvq + 32 + 8 * t) = f32x4{dv1[4 * t], dv1[4 * t + 1], dv1[4 * t + 2], dv1[4 * t + 3]};
  }
}

}  // namespace
}  // namespace mx

using namespace mx;

// The arguments of mx_attn_bwd (attn_bwd.hip), which checks them; dq is not written where dqkv is given.  -1 (nothing launched):
// more rows of a head, or heads, than the byte offsets of 31 bits within a head's q, k and v and a tile of dO reach.
int mx_attn_bwd64(const uint16_t* q, const uint16_t* k, const uint16_t* v, const uint16_t* o, const uint16_t* dout,
                  const float* lse, float* delta, float* dq, float* dkp, float* dvp, int B, int Hq, int Hkv, int S, int Sk,
                  bool causal, float scale, int64_t ldo, uint16_t* dqkv, int64_t ldq, const float* cosb,
                  const float* sinb, hipStream_t stream) {
  constexpr int kMost = (1 << 24) - 128;  // rows: x 128 B
  if (S > kMost || Sk > kMost || Hq > (1 << 18) || (int64_t)((std::max(S, Sk) + 127) / 128) * B * Hq > INT32_MAX) return -1;
  const float sl = scale * 1.4426950408889634f;
  const int off = Sk - S, qgrid = (S + 127) / 128 * B * Hq, kgrid = (Sk + 127) / 128 * B * Hq;
#define MX_BWD64(C)                                                                                                      \
  do {                                                                                                                   \
    attn_bwd64_q_kernel<C><<<qgrid, 256, 0, stream>>>(q, k, v, o, dout, lse, delta, dq, dqkv, cosb, sinb, B, Hq, Hkv, S,  \
                                                      Sk, off, sl, scale, ldo, ldq);                                     \
    attn_bwd64_kv_kernel<C><<<kgrid, 256, 0, stream>>>(q, k, v, dout, lse, delta, dkp, dvp, B, Hq, Hkv, S, Sk, off, sl,   \
                                                       scale);                                                           \
  } while (0)
  if (causal) MX_BWD64(true);
  else MX_BWD64(false);
#undef MX_BWD64
  return (int)hipGetLastError();
}
