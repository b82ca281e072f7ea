// Weight-streaming core of the bf16 decode GEMMs (skinny_gemm.hip, hybrid_skinny.hip): a workgroup of
// 8 waves computes 16 NC output channels for 16 MB token rows; wave w owns K part [w K / 8, (w + 1) K / 8)
// in 64-k chunks, two v_mfma_f32_16x16x32_bf16 each with the weights as the A operand.  Lane (c, g)
// reads 16 g .. 16 g + 15 of its chunk of weight row c and of token row c.
#pragma once

#include <type_traits>

#include "common.h"

namespace mx {

typedef __bf16 bf16x8_sk __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x4 mfma16_sk(const u16x8& a, const u16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_sk, a), __builtin_bit_cast(bf16x8_sk, b),
                                                 c, 0, 0, 0);
}

constexpr int kSkWaves = 8;
// 64-k chunks whose loads are issued before the first is used
constexpr int sk_unr(int nc) { return nc == 1 ? 8 : 4; }

// the first block of weight loads, issued ahead of a prologue that builds X in LDS (half a block where K has no
// more: at K 2048 a wave's part is 4 chunks)
template <int NC>
__device__ __forceinline__ void sk_prefetch(const uint16_t* const (&wrow)[NC], int nit,
                                            u16x8 (&apre)[sk_unr(NC)][NC][2]) {
  constexpr int UNR = sk_unr(NC);
  auto load = [&](auto from, auto to) {
#pragma unroll
    for (int u = from; u < to; ++u)
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        apre[u][j][0] = *reinterpret_cast<const u16x8*>(wrow[j] + u * 64);
        apre[u][j][1] = *reinterpret_cast<const u16x8*>(wrow[j] + u * 64 + 8);
      }
  };
  using std::integral_constant;
  if (nit >= UNR / 2) load(integral_constant<int, 0>{}, integral_constant<int, UNR / 2>{});
  if (nit >= UNR) load(integral_constant<int, UNR / 2>{}, integral_constant<int, UNR>{});
}

// acc[j][mb] (zeroed here) = this wave's K part; PRE: apre holds the first block's weights.
// A K part goes by blocks of UNR chunks, then of half as many down to one: whatever K leaves over is in flight
// together (chunk by chunk, a K of 2048 waited for memory four times: 6.0 us for a 12.6 MB projection of one row
// against 5.5; with the norm in the prologue, whose prefetch such a K now has, 7.1 against 5.6, and 17.3 against 14.9
// for the 67 MB gate-up projection).
template <int MB, int NC, bool PRE>
__device__ __forceinline__ void sk_stream(const uint16_t* const (&wrow)[NC], const uint16_t* const (&xr)[MB], int nit,
                                          const u16x8 (&apre)[sk_unr(NC)][NC][2], f32x4 (&acc)[NC][MB]) {
  constexpr int UNR = sk_unr(NC);
#pragma unroll
  for (int j = 0; j < NC; ++j)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[j][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto loadx = [&](int k, u16x8 (&b)[MB][2]) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      b[mb][0] = *reinterpret_cast<const u16x8*>(xr[mb] + k);
      b[mb][1] = *reinterpret_cast<const u16x8*>(xr[mb] + k + 8);
    }
  };
  auto step = [&](const u16x8 (&a)[NC][2], const u16x8 (&b)[MB][2]) {
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        acc[j][mb] = mfma16_sk(a[j][0], b[mb][0], acc[j][mb]);
        acc[j][mb] = mfma16_sk(a[j][1], b[mb][1], acc[j][mb]);
      }
  };
  auto block = [&](auto n, int it) {
    constexpr int U = n;
    u16x8 a[U][NC][2], b[U][MB][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        a[u][j][0] = *reinterpret_cast<const u16x8*>(wrow[j] + (it + u) * 64);
        a[u][j][1] = *reinterpret_cast<const u16x8*>(wrow[j] + (it + u) * 64 + 8);
      }
      loadx((it + u) * 64, b[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) step(a[u], b[u]);
  };
  auto first = [&](auto n) {  // weights prefetched above, X fragments from LDS
    constexpr int U = n;
    u16x8 b[U][MB][2];
#pragma unroll
    for (int u = 0; u < U; ++u) loadx(u * 64, b[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) step(apre[u], b[u]);
  };
  using std::integral_constant;
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
