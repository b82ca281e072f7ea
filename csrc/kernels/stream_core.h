// The walk of the decode GEMMs over few workgroups that stay (stream_gemm.hip, moe_stream.hip): a workgroup of 8
// waves holds its token rows X in LDS and goes over channel groups grp = first, + step, ... < groups, only weights in its
// load queue, two blocks of U 64-k chunks in flight.
//   row(grp): weight row of channel 0 of a group; off(ch): rows from there to channel ch's, the same in every group (a
//     scalar base and 32-bit offsets: as 64-bit addresses a lane's two rows spilled registers);
//   stage(xs, ldx, ahead): fills xs [M, K] (row stride ldx) and ends with a barrier; calls ahead(), the first weight
//     loads, behind its own reads and in front of the work on them;
//   finish(sum, mb, grp): called by one whole wave, lane (c, g): channels 4 g .. + 3 of token 16 mb + c.
#pragma once

#include "e4m3.h"
#include "skinny_core.h"

namespace mx {

// How a kernel reads its weights: bf16 in blocks of 8 rows x 128 B and of 8 tokens (up to 16 rows of X), or of 16 rows x 64 B
// and 16 tokens; e4m3 codes, which a lane widens to the two MFMA operands of a chunk, the same two ways: 8 rows x 128 codes and 8
// tokens (4 K parts), or 16 rows x 64 and 16.
enum { kStLines, kStWide, kStF8, kStF8Lines };

// NL loads of weights in flight, chunk by chunk and block by block
template <int KIND, int NL, int RB>
struct WFrag {
  u16x8 a[NL / RB][RB];
  __device__ __forceinline__ void load(const char* p, const uint32_t (&o)[RB]) {
#pragma unroll
    for (int u = 0; u < NL / RB; ++u)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) a[u][rb] = KIND == kStWide ? *reinterpret_cast<const u16x8*>(p + o[rb] + u * 128) : sk_weights(p + o[rb] + u * 128);
  }
};
template <bool LINES, int NL>
struct WCodes {
  u32x4 a[NL];
  __device__ __forceinline__ void load(const char* p, const uint32_t (&o)[1]) {
#pragma unroll
    for (int u = 0; u < NL; ++u)
      a[u] = LINES ? sk_weights<u32x4>(p + o[0] + u * 128) : *reinterpret_cast<const u32x4*>(p + o[0] + u * 64);
  }
  __device__ __forceinline__ void get(int u, u16x8& x, u16x8& y) const {
    x = dequant8(a[u][0], a[u][1]);
    y = dequant8(a[u][2], a[u][3]);
  }
};

template <int NL>
struct WFrag<kStF8, NL, 1> : WCodes<false, NL> {};
template <int NL>
struct WFrag<kStF8Lines, NL, 1> : WCodes<true, NL> {};

// rows of X [M, K] as they are: XP 16-B pieces a thread holds at once, all or the last ones
template <int XP, typename Ahead>
__device__ __forceinline__ void stream_rows_in(const uint16_t* __restrict__ X, int64_t ldX, int M, int K, uint16_t* xs,
                                               int ldx, const Ahead& ahead) {
  const int tid = threadIdx.x, per = K / 8, total = M * per;
  u16x8 v[XP];
  auto fetch = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XP; ++i) {
      const int p = min(p0 + tid + 512 * i, total - 1), m = p / per;
      v[i] = *reinterpret_cast<const u16x8*>(X + (int64_t)m * ldX + (p - m * per) * 8);
    }
  };
  auto put = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XP; ++i) {
      const int p = p0 + tid + 512 * i, m = p / per;
      if (p < total) *reinterpret_cast<u16x8*>(xs + m * ldx + (p - m * per) * 8) = v[i];
    }
  };
  int p0 = 0;
  for (; p0 + XP * 512 < total; p0 += XP * 512) {
    fetch(p0);
    put(p0);
  }
  fetch(p0);
  ahead();
  put(p0);
  lds_barrier();
}

// the partial sums' images: two of up to 8 KB (the waves take turns at a group's sum and what follows, the others go
// on), or one of 16
template <int KIND, int TB, int KP>
constexpr int kStreamPlaces = KIND == kStLines || KIND == kStF8Lines ? SkSum<TB, 1, KP>::PLACES : kSkWaves * TB * 64;
template <int KIND, int TB, int KP>
constexpr int kStreamImages = kStreamPlaces<KIND, TB, KP> * 16 <= 8192 ? 2 : 1;
template <int KIND, int TB, int KP>
constexpr int kStreamRed = kStreamPlaces<KIND, TB, KP> * kStreamImages<KIND, TB, KP> * 16;  // bytes, 16 KB at most

// TB blocks of 8 (lines) or 16 tokens, KP K parts (kStF8Lines: 4, without lines: 8)
template <int KIND, int TB, int KP, int NL, typename Row, typename Off, typename Stage, typename Finish>
__device__ __forceinline__ void stream_walk(const void* W, int64_t ldw, const float* scale, int M, int K, int first,
                                            int step, int groups, char* smem, const Row& row, const Off& off, const Stage& stage,
                                            const Finish& finish) {
  constexpr bool F8 = KIND == kStF8 || KIND == kStF8Lines, LINES = KIND == kStLines || KIND == kStF8Lines;
  static_assert(KIND != kStF8Lines || KP == 4, "one block of codes a wave");
  constexpr int NW = kSkWaves, WB = F8 ? 1 : 2, RB = F8 ? 1 : kSkBlocks<KP, 1>, MB = LINES ? (TB + 1) / 2 : TB;
  constexpr int AB = LINES ? RB : 1;  // blocks with sums of their own (kStWide: the halves of a chunk share them)
  constexpr int CK = KIND == kStF8Lines ? 128 : 64, CH = NL / RB;  // k of a chunk, chunks of a block
  typedef SkSum<TB, 1, KP> Sum;  // kStLines
  constexpr int PLACES = kStreamPlaces<KIND, TB, KP>, NRED = kStreamImages<KIND, TB, KP>;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int kq = K / KP, nblk = kq / (CK * CH), ldx = K + 8;
  f32x4* red = reinterpret_cast<f32x4*>(smem);
  uint16_t* xs = reinterpret_cast<uint16_t*>(smem + kStreamRed<KIND, TB, KP>);
  const int k0 = sk_part<KP>(w) * kq + (F8 && LINES ? 2 * sk_lane_k(c, g) : LINES ? sk_lane_k(c, g) : F8 ? 16 * g : 8 * g);
  // the block to load next: group lg, block lb
  int lg = first, lb = 0;
  uint32_t lo[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
    lo[rb] = (uint32_t)(off(LINES ? 8 * sk_half<KP>(w, rb) + (c & 7) : c) * (uint32_t)ldw + (uint32_t)k0 +
                        (LINES ? 0 : 32 * rb)) * WB;
  const char* lp = reinterpret_cast<const char*>(W) + row(lg) * ldw * WB;
  auto load = [&](WFrag<KIND, NL, RB>& f) __attribute__((always_inline)) {
    f.load(lp, lo);
    lp += CH * CK * WB;
    if (++lb == nblk) {
      lb = 0;
      lg += step;
      lp = reinterpret_cast<const char*>(W) + row(min(lg, groups - 1)) * ldw * WB;
    }
  };
  WFrag<KIND, NL, RB> f0, f1;
  stage(xs, ldx, [&]() __attribute__((always_inline)) { load(f0); });
  const uint16_t* xr[TB];
#pragma unroll
  for (int tb = 0; tb < TB; ++tb) xr[tb] = xs + min(LINES ? tb * 8 + (c & 7) : tb * 16 + c, M - 1) * ldx + k0;

  f32x4 acc[AB][TB];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int rb = 0; rb < AB; ++rb)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) acc[rb][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  int cg = first, cb = 0, turn = 0;
  auto multiply = [&](const WFrag<KIND, NL, RB>& f) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int k = (cb * CH + u) * CK;
      if constexpr (F8) {
        u16x8 a0, a1;
        f.get(u, a0, a1);
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
          acc[0][tb] = mfma16_sk(a0, *reinterpret_cast<const u16x8*>(xr[tb] + k), acc[0][tb]);
          acc[0][tb] = mfma16_sk(a1, *reinterpret_cast<const u16x8*>(xr[tb] + k + 8), acc[0][tb]);
        }
      } else if constexpr (LINES) {
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
          const u16x8 b = *reinterpret_cast<const u16x8*>(xr[tb] + k);
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) acc[rb][tb] = mfma16_sk(f.a[u][rb], b, acc[rb][tb]);
        }
      } else {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
          for (int tb = 0; tb < TB; ++tb)
            acc[0][tb] = mfma16_sk(f.a[u][rb], *reinterpret_cast<const u16x8*>(xr[tb] + k + 32 * rb), acc[0][tb]);
      }
    }
    if (++cb < nblk) return;
    cb = 0;
    f32x4* const img = red + (NRED == 2 ? turn & 1 : 0) * PLACES;
    const Sum sum{img};
    if constexpr (LINES) {
      sum.put(w, c, g, acc);
    } else {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) img[(w * MB + mb) * 64 + lane] = acc[0][mb];
    }
    clear();
    lds_barrier();
    if (w == (turn & (NW - 1))) {
      f32x4 sc = {1.f, 1.f, 1.f, 1.f};
      if constexpr (F8) sc = *reinterpret_cast<const f32x4*>(scale + row(cg) + off(4 * g));
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        f32x4 s;
        if constexpr (LINES) {
          s = sum.get(c, g, 0, mb);
        } else {
          s = img[mb * 64 + lane];
#pragma unroll
          for (int ww = 1; ww < NW; ++ww) s += img[(ww * MB + mb) * 64 + lane];
        }
        if constexpr (F8) s *= sc;
        finish(s, mb, cg);
      }
    }
    if constexpr (NRED == 1) lds_barrier();  // one image: its sum is read before the next group's parts
    ++turn;
    cg += step;
  };
  const int steps = (groups - first + step - 1) / step * nblk;
  if (steps == 1) {
    multiply(f0);
    return;
  }
  load(f1);
  int s = 0;
  for (; s + 3 < steps; s += 2) {
    multiply(f0);
    load(f0);
    multiply(f1);
    load(f1);
  }
  multiply(f0);
  if (steps - s == 3) {
    load(f0);
    multiply(f1);
    multiply(f0);
  } else {
    multiply(f1);
  }
}

// One group and, more >= 0, half of another (more: twice the group + the half): a wave's loads of both in flight at once.
// Half h is channels 4 h .. + 3 and 8 + 4 h .. + 3, which an epilogue pairs: 8 rows.  finish has a fourth
// argument, whether the lane's four channels are of that half.  For the K whose part is one block (4096: kStLines of 8 parts,
// NL 16; kStF8Lines, NL 8).
template <int KIND, int TB, int KP, int NL, typename Row, typename Off, typename Stage, typename Finish>
__device__ __forceinline__ void stream_and_half(const void* W, int64_t ldw, const float* scale, int M, int K, int grp,
                                                int more, char* smem, const Row& row, const Off& off, const Stage& stage,
                                                const Finish& finish) {
  constexpr bool F8 = KIND == kStF8Lines;
  static_assert(KIND == kStLines || F8, "blocks of 8 rows");
  constexpr int WB = F8 ? 1 : 2, RB = F8 ? 1 : kSkBlocks<KP, 1>, MB = (TB + 1) / 2;
  constexpr int CK = F8 ? 128 : 64, CH = NL / RB;  // chunks of a wave's part
  static_assert(kStreamImages<KIND, TB, KP> == 2, "sums of both");
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4, ldx = K + 8;
  f32x4* const red = reinterpret_cast<f32x4*>(smem);
  f32x4* const hred = red + kStreamPlaces<KIND, TB, KP>;
  uint16_t* const xs = reinterpret_cast<uint16_t*>(smem + kStreamRed<KIND, TB, KP>);
  const int kl = F8 ? 2 * sk_lane_k(c, g) : sk_lane_k(c, g), k0 = sk_part<KP>(w) * (K / KP) + kl;
  const int hg = more >> 1, h = more & 1, hc = 4 * h + (c & 3) + 8 * (c >> 2 & 1);
  WFrag<KIND, NL, RB> f;
  WFrag<KIND, CH, 1> f2;
  const bool extra = more >= 0 && w < KP;  // (the same parts and sums as a whole group's: the same bits)
  stage(xs, ldx, [&]() __attribute__((always_inline)) {
    uint32_t o[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
      o[rb] = (uint32_t)(off(8 * sk_half<KP>(w, rb) + (c & 7)) * (uint32_t)ldw + (uint32_t)k0) * WB;
    f.load(reinterpret_cast<const char*>(W) + row(grp) * ldw * WB, o);
    if (extra) {
      const uint32_t o2[1] = {(uint32_t)(off(hc) * (uint32_t)ldw + (uint32_t)k0) * WB};
      f2.load(reinterpret_cast<const char*>(W) + row(hg) * ldw * WB, o2);
    }
  });
  auto products = [&](const auto& fr, auto& acc) __attribute__((always_inline)) {
    constexpr int R = std::extent<std::remove_reference_t<decltype(acc)>>::value;
    const uint16_t* xr[TB];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) xr[tb] = xs + min(tb * 8 + (c & 7), M - 1) * ldx + k0;
#pragma unroll
    for (int rb = 0; rb < R; ++rb)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) acc[rb][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      if constexpr (F8) {
        u16x8 a0, a1;
        fr.get(u, a0, a1);
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
          acc[0][tb] = mfma16_sk(a0, *reinterpret_cast<const u16x8*>(xr[tb] + u * CK), acc[0][tb]);
          acc[0][tb] = mfma16_sk(a1, *reinterpret_cast<const u16x8*>(xr[tb] + u * CK + 8), acc[0][tb]);
        }
      } else {
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
          const u16x8 b = *reinterpret_cast<const u16x8*>(xr[tb] + u * CK);
#pragma unroll
          for (int rb = 0; rb < R; ++rb) acc[rb][tb] = mfma16_sk(fr.a[u][rb], b, acc[rb][tb]);
        }
      }
    }
  };
  const SkSum<TB, 1, KP> sum{red};
  {
    f32x4 acc[RB][TB];
    products(f, acc);
    sum.put(w, c, g, acc);
  }
  if (extra) {
    f32x4 acc[1][TB];
    products(f2, acc);
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
      const f32x4 s = sk_both_halves(acc[0][tb]);
      if (c < 8 && g < 2) hred[(w * TB + tb) * 16 + 8 * g + c] = s;
    }
  }
  lds_barrier();
  if (w > (more >= 0 ? 1 : 0)) return;
  const int cg = w ? hg : grp;
  f32x4 sc = {1.f, 1.f, 1.f, 1.f};
  if constexpr (F8) sc = *reinterpret_cast<const f32x4*>(scale + row(cg) + off(4 * g));
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    f32x4 s;
    if (w == 0) {
      s = sum.get(c, g, 0, mb);
    } else {
      s = f32x4{0.f, 0.f, 0.f, 0.f};
      const int e = min(2 * mb + (c >> 3), TB - 1) * 16 + 8 * (g >> 1) + (c & 7);
#pragma unroll
      for (int i = 0; i < KP; ++i) s += hred[i * TB * 16 + e];
    }
    if constexpr (F8) s *= sc;
    finish(s, mb, cg, w == 0 || (g & 1) == h);
  }
}

}  // namespace mx
