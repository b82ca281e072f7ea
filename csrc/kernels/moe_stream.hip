// The experts' gated products of a decode step (bf16, gfx950), over workgroups that stay: each has one expert (or the shared
// one) and a run of its channel groups, holds the rows of the tokens that chose it in LDS and streams the weights past
// them (stream_core.h).
//
// moe_few_kernel gives 16 channels a workgroup of their own: 512 of 128 KB of weights (1B sizes) or 1,800 of 256 KB (8B), each with
// its own choices, list and rows in front of the first load, two a CU and in uneven turns (3.2 to 4.7 TB/s).  Here a CU does
// that once, and has the next block of weights in flight throughout.  One launch, 8 / 16 / 32 tokens, us: 1B sizes (67 MB)
// 16.6 / 17.9 -> 15.0 / 16.2; 8B sizes (268 MB) 46.2 / 50.0 / 57.1 -> 38.9 / 43.6 / 55.4; steps of 8 / 16 sequences 1310 / 1396 ->
// 1242 / 1333 and 4709 / 5141 -> 4549 / 4970.  Rows go 16 at a time: past 16 tokens the shared expert's weights are read twice.
// At 1B sizes that, or 32 rows in LDS in 16-row fragments, is what lasts (32 tokens alone 21.1 -> 18.8, but with a model's uneven
// choices steps of 24 sequences 1521 -> 1536 us): those stay.  The first weights asked for ahead of the choices gained
// nothing (14.8 / 16.9).
#include <algorithm>
#include <climits>

#include "decode_fuse.h"
#include "hybrid.h"
#include "moe_route.h"
#include "stream_core.h"
#include "sublayer.h"

namespace mx {

constexpr int kMoeStreamTokens = 32, kMoeStreamLds = 158 * 1024;

struct MoeWalk {
  MoeFew a;
  int per, sper;  // channel groups of a workgroup: 8 gate and the 8 matching up rows each
  int we, ws;     // workgroups of an expert, of the shared one (the first ones)
  int cap;        // rows at a time
};

// K of 2,048: four K parts and blocks of 8 loads; of a multiple of 4,096: eight and 16
template <int KP, int NL>
__global__ void __launch_bounds__(512, 2) moe_stream_kernel(MoeWalk p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int16_t list[64];  // the pairs of the tokens that chose this expert
  const MoeFew& a = p.a;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
  const bool shared = (int)blockIdx.x < p.ws;
  const int unit = shared ? blockIdx.x : blockIdx.x - p.ws, expert = shared ? 0 : unit / p.we;
  const int per = shared ? p.sper : p.per, F = shared ? a.sN : a.N;
  const int first = (shared ? unit : unit % p.we) * per, groups = min(F / 8, first + per);
  int n = a.T;
  if (!shared) {
    if (unit == p.we - 1) {  // the last of the first expert, whose run may be the shorter one, stores the choices
      constexpr int TW = kMoeStreamTokens / 8;  // tokens of a wave, their logits asked for together
      float z[TW];
#pragma unroll
      for (int i = 0; i < TW; ++i) z[i] = a.logits[(int64_t)min(w + 8 * i, a.T - 1) * a.E + min(lane, a.E - 1)];
#pragma unroll
      for (int i = 0; i < TW; ++i) {
        const int t = w + 8 * i;
        if (t >= a.T) break;
        moe_choose64(z[i], a.E, a.top, lane, [&](int k, float wt) {
          a.ids_out[t * a.top + k] = lane;
          a.wts_out[t * a.top + k] = wt;
        });
      }
    }
    n = moe_list(moe_place(a.logits, a.E, a.top, a.T, expert, lane), a.top, lane, list);
    if (n == 0) return;
  }
  const uint16_t* W = shared ? a.sw : a.w + (int64_t)expert * 2 * a.N * a.K;
  uint16_t* const y = shared ? a.sy : a.y;
  const float limit = shared ? a.slimit : a.limit;
  auto row = [&](int grp) __attribute__((always_inline)) -> int64_t { return dfuse_row<true>(grp, 0, F); };
  auto off = [&](int ch) __attribute__((always_inline)) -> int { return (int)dfuse_row<true>(0, ch, F); };
  for (int r0 = 0; r0 < n; r0 += p.cap) {
    const int rows = min(p.cap, n - r0);
    auto stage = [&](uint16_t* xs, int ldx, auto ahead) __attribute__((always_inline)) {
      const int pieces = a.K / 8, total = rows * pieces;
      constexpr int XP = 8;
      u32x4 v[XP];
      auto fetch = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < XP; ++i) {
          const int q = min(p0 + tid + 512 * i, total - 1), m = q / pieces;
          const int t = shared ? r0 + m : list[r0 + m] / a.top;
          v[i] = *reinterpret_cast<const u32x4*>(a.x + (int64_t)t * a.ldx + (q - m * pieces) * 8);
        }
      };
      auto put = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < XP; ++i) {
          const int q = p0 + tid + 512 * i, m = q / pieces;
          if (q < total) *reinterpret_cast<u32x4*>(xs + m * ldx + (q - m * pieces) * 8) = v[i];
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
    };
    auto finish = [&](const f32x4& s, int mb, int grp) __attribute__((always_inline)) {
      const int m = mb * 16 + c;
      u16x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float up = __uint_as_float(lane_pair<32>(__float_as_uint(s[i])).b);
        o[i] = f2bf(clipped_glu<uint16_t>(s[i], up, limit));
      }
      if (m < rows && g < 2) {
        const int64_t at = shared ? r0 + m : list[r0 + m];
        *reinterpret_cast<u16x4*>(y + at * F + 8 * grp + 4 * g) = o;
      }
    };
    if (r0) __syncthreads();  // the rows and sums of the last walk are read
    if (rows <= 8)
      stream_walk<kStLines, 1, KP, NL>(W, a.K, nullptr, rows, a.K, first, 1, groups, smem, row, off, stage, finish);
    else
      stream_walk<kStLines, 2, KP, NL>(W, a.K, nullptr, rows, a.K, first, 1, groups, smem, row, off, stage, finish);
  }
}

template <int KP, int NL>
static int moe_stream_launch(const MoeWalk& p, int grid, size_t lds, hipStream_t stream) {
  static const bool big = hipFuncSetAttribute((const void*)moe_stream_kernel<KP, NL>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                              kMoeStreamLds) == hipSuccess;
  if (!big) return -1;
  moe_stream_kernel<KP, NL><<<grid, 512, lds, stream>>>(p);
  return (int)hipGetLastError();
}

}  // namespace mx

using namespace mx;

// What mx_moe_few takes, more pairs than experts, up to 32 tokens; -1: sizes for that kernel, nothing launched
extern "C" int mx_moe_stream(const MoeFew* pa, hipStream_t stream) {
  const MoeFew& a = *pa;
  if (a.T <= 0 || a.T > kMoeStreamTokens || !a.logits || a.E > 64 || a.T * a.top <= a.E || a.K <= 0 ||
      (a.K != 2048 && a.K % 4096) || (a.K == 2048 && a.T > 16) || a.N <= 0 || a.N % 8 || (a.sw && (a.sN <= 0 || a.sN % 8 || a.sK != a.K)) ||
      (int64_t)(std::max(a.N, a.sN) + 16) * a.K * 2 >> 32)
    return -1;
  MoeWalk p{a};
  p.cap = std::min(a.T, 16);
  const size_t lds = 16 * 1024 + (size_t)p.cap * (a.K + 8) * 2;
  if (lds > kMoeStreamLds - 512) return -1;
  // One workgroup a CU.  What one takes, in quarters of a row of K: the 16 weight rows of a group, again for each turn of the
  // shared expert's rows, and its tokens' rows, which come from L2 (counted whole, 32 tokens at 1B sizes took 20.5 us for 18.8).
  const int turns = (a.T + p.cap - 1) / p.cap, gx = a.N / 8, sx = a.sw ? a.sN / 8 : 0, mean = a.T * a.top / a.E;
  int64_t best = INT64_MAX;
  for (int per = 1; per <= gx; ++per) {
    const int we = (gx + per - 1) / per, left = 256 - a.E * we;
    if (left < (sx ? 1 : 0) && per < gx) continue;
    const int sper = sx ? (sx + std::max(left, 1) - 1) / std::max(left, 1) : 0;
    const int64_t cost = std::max(64 * per + mean, sx ? 64 * sper * turns + a.T : 0);
    if (cost < best) {
      best = cost;
      p.per = per, p.we = we, p.sper = sper, p.ws = sx ? (sx + sper - 1) / sper : 0;
    }
  }
  const int grid = a.E * p.we + p.ws;
  return a.K == 2048 ? moe_stream_launch<4, 8>(p, grid, lds, stream) : moe_stream_launch<8, 16>(p, grid, lds, stream);
}
