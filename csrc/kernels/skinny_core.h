// Weight-streaming core of the bf16 decode GEMMs (skinny_gemm.hip, hybrid_skinny.hip; its fragments and sums also in
// stream_core.h): a workgroup of 8 waves computes 16 NC output channels for 8 TB token rows.
//
// What bounds it is how memory likes to be asked.  An instruction reads 8 rows x 128 B, whole cache lines, marked
// nontemporal (read once, never found again), and a wave has at least 1 KB of each row in turn: 8 K parts of 16 rows,
// or for a K of 2048 4 parts of 8 rows.  Reads alone, in a chain of launches: 50 MB of K 2048 9.4 us, of K 4096 9.1; with
// 16 rows x 64 B and 8 parts 13.0 and 10.9 (nontemporal 14.4 and 12.0: the other half of each line is asked for again).
//
// Lane (c, g) of v_mfma_f32_16x16x32_bf16, the weights as the A operand, holds 8 k from 32 (c >> 3) + 8 g of a 64-k chunk of
// weight row c & 7; the B operand has token c & 7's at the same k.  Of a product, (channel, token) of the first halves and
// (channel + 8, token + 8) of the second ones are of use: they are added with the waves' parts.
#pragma once

#include <type_traits>

#include "common.h"

namespace mx {

typedef __bf16 bf16x8_sk __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x4 mfma16_sk(const u16x8& a, const u16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_sk, a), __builtin_bit_cast(bf16x8_sk, b),
                                                 c, 0, 0, 0);
}
template <typename V = u16x8>
__device__ __forceinline__ V sk_weights(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const V*>(p));
}

constexpr int kSkWaves = 8;
// K parts of a workgroup: 8, each wave's 16 rows; or 4, waves 0 .. 3 rows 0 .. 7 and waves 4 .. 7 the others.  With 4 a wave
// reads twice as much of X for its weights: past 16 token rows that is what lasts (16384 x 2048, 16 / 32 rows 15.4 / 18.6 us, with
// 8 parts 16.3 / 17.7), and a shorter K has little to gain (128256 x 1536, 8 rows 71 -> 89).
constexpr int sk_parts(int M, int K) { return K == 2048 && M <= 16 ? 4 : 8; }
// Whether fragments of 16 rows x 64 B and 16 tokens, without the halves, are the better ones: past 16 token rows, and past 8 of a
// K under 2048, the products and sums of each 8 tokens show beside the few bytes (4096 x 1024, 12 / 32 rows 4.8 / 7.2 us in
// blocks of 8, 4.6 / 5.9 so; stream_gemm.hip, 16384 x 2048, 32 rows 20.0, 18.6 so).  So do they where a wave's part is 6 or 7
// chunks, whose loads go out in two or three turns either way (2048 x 3072, 9 / 16 rows 7.7 / 8.7, 7.4 / 8.1 so; 2048 x 3584, 16
// rows 9.7, 9.3 so; of 5 chunks, 2048 x 2560, 6.7 / 7.7, 6.9 / 7.7 so; of 9, 2048 x 4608, 9.7 / 11.1, 10.3 / 11.9 so).
constexpr bool sk_wide(int M, int K) { return M > 16 || (M > 8 && (K < 2048 || (K > 2560 && K < 4096))); }
// 8-row blocks of a wave for NC groups of 16 channels
template <int KP, int NC>
constexpr int kSkBlocks = NC * KP / 4;
// a wave's K part, and the half (0, 1) of a group's channels that its block rb is
template <int KP>
__device__ __forceinline__ int sk_part(int w) { return KP == 8 ? w : w & 3; }
template <int KP>
__device__ __forceinline__ int sk_half(int w, int rb) { return KP == 8 ? rb & 1 : w >> 2; }
// the lane's k in a chunk
__device__ __forceinline__ int sk_lane_k(int c, int g) { return 32 * (c >> 3) + 8 * g; }

// 64-k chunks whose loads are issued before the first is used
constexpr int sk_unr(int nc) { return nc == 1 ? 8 : 4; }

// a product's useful parts added: channels 4 g .. + 3 of token c in lanes c < 8, g < 2
__device__ __forceinline__ f32x4 sk_both_halves(const f32x4& v) {
  f32x4 s;
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // lane l + lane (l ^ 8) + 32: without the LDS, whose round trips showed at 9 rows and more
    const uint32_t t = __builtin_amdgcn_mov_dpp(__float_as_uint(v[i]), 0x128, 0xF, 0xF, true);  // row_ror:8
    s[i] = v[i] + __uint_as_float(__builtin_amdgcn_permlane32_swap(t, t, false, false)[1]);
  }
  return s;
}

// Sums of the waves' parts.  red: 16 places a (wave, block, token block); a whole wave adds the halves and stores its own,
// and after a barrier lane (c, g) of any wave gets channels 4 g .. + 3 of token 16 mb + c of group j.
template <int TB, int NC, int KP>
struct SkSum {
  static constexpr int RB = kSkBlocks<KP, NC>, PLACES = kSkWaves * RB * TB * 16;
  f32x4* red;
  static __device__ __forceinline__ int at(int w, int rb, int tb) { return ((w * RB + rb) * TB + tb) * 16; }
  __device__ __forceinline__ void put(int w, int c, int g, const f32x4 (&acc)[RB][TB]) const {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) {
        const f32x4 s = sk_both_halves(acc[rb][tb]);
        if (c < 8 && g < 2) red[at(w, rb, tb) + 8 * g + c] = s;
      }
  }
  __device__ __forceinline__ f32x4 get(int c, int g, int j, int mb) const {
    const int tb = min(2 * mb + (c >> 3), TB - 1), e = 8 * (g & 1) + (c & 7);
    const int w0 = KP == 8 ? 0 : 4 * (g >> 1), rb = KP == 8 ? 2 * j + (g >> 1) : j;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < KP; ++w) s += red[at(w0 + w, rb, tb) + e];
    return s;
  }
};

// the first block of weight loads, issued ahead of a prologue that builds X in LDS (half a block where K has no
// more)
template <int NC, int RB>
__device__ __forceinline__ void sk_prefetch(const uint16_t* const (&wrow)[RB], int nit, u16x8 (&apre)[sk_unr(NC)][RB]) {
  constexpr int UNR = sk_unr(NC);
  auto load = [&](auto from, auto to) {
#pragma unroll
    for (int u = from; u < to; ++u)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) apre[u][rb] = sk_weights(wrow[rb] + u * 64);
  };
  using std::integral_constant;
  if (nit >= UNR / 2) load(integral_constant<int, 0>{}, integral_constant<int, UNR / 2>{});
  if (nit >= UNR) load(integral_constant<int, UNR / 2>{}, integral_constant<int, UNR>{});
}

// acc[rb][tb] (zeroed here) = this wave's K part of block rb's rows; PRE: apre holds the first block's weights.
// DEEP: a block's loads all go out ahead of its products, at 126 registers; left to itself the compiler keeps half of them
// back for the sake of more waves, which few workgroups do not have.
// WIDE: fragments of 16 rows x 64 B and 16 tokens; the two blocks are the halves of a chunk and add up in acc[0].
// WHOLE: the chunks of a K part, all in flight together.
// A K part goes by blocks of UNR chunks, then of half as many down to one: whatever K leaves over is in flight
// together.
template <int TB, int NC, bool PRE, bool WIDE = false, bool DEEP = false, int WHOLE = 0, int RB>
__device__ __forceinline__ void sk_stream(const uint16_t* const (&wrow)[RB], const uint16_t* const (&xr)[TB], int nit,
                                          const u16x8 (&apre)[sk_unr(NC)][RB], f32x4 (&acc)[RB][TB]) {
  constexpr int UNR = sk_unr(NC), XH = WIDE ? 2 : 1;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) acc[rb][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto loadx = [&](int k, u16x8 (&b)[TB][XH]) {
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
      for (int h = 0; h < XH; ++h) b[tb][h] = *reinterpret_cast<const u16x8*>(xr[tb] + k + 32 * h);
  };
  auto loadw = [&](const uint16_t* p) {
    if constexpr (WIDE) return *reinterpret_cast<const u16x8*>(p);  // half lines: the other half is still to come
    else return sk_weights(p);
  };
  auto step = [&](const u16x8 (&a)[RB], const u16x8 (&b)[TB][XH]) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) {
        f32x4& s = acc[WIDE ? 0 : rb][tb];
        s = mfma16_sk(a[rb], b[tb][WIDE ? rb : 0], s);
      }
  };
  auto block = [&](auto n, int it) {
    constexpr int U = n;
    u16x8 a[U][RB], b[U][TB][XH];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) a[u][rb] = loadw(wrow[rb] + (it + u) * 64);
      loadx((it + u) * 64, b[u]);
    }
    if constexpr (DEEP || WHOLE > 0) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) step(a[u], b[u]);
  };
  auto first = [&](auto n) {  // weights prefetched above, X fragments from LDS
    constexpr int U = n;
    u16x8 b[U][TB][XH];
#pragma unroll
    for (int u = 0; u < U; ++u) loadx(u * 64, b[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) step(apre[u], b[u]);
  };
  using std::integral_constant;
  if constexpr (WHOLE > 0) {
    block(integral_constant<int, WHOLE>{}, 0);
    return;
  }
  int it = 0;
  if constexpr (PRE) {
    if (nit >= UNR) {
      first(integral_constant<int, UNR>{});
      it = UNR;
    } else if (nit >= UNR / 2) {
      first(integral_constant<int, UNR / 2>{});
      it = UNR / 2;
    }
  }
  for (; it + UNR <= nit; it += UNR) block(integral_constant<int, UNR>{}, it);
  if constexpr (UNR >= 8) {
    if (it + 4 <= nit) { block(integral_constant<int, 4>{}, it); it += 4; }
  }
  if (it + 2 <= nit) { block(integral_constant<int, 2>{}, it); it += 2; }
  if (it < nit) block(integral_constant<int, 1>{}, it);
}

}  // namespace mx
