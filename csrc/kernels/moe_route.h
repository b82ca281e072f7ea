// Choice of experts from a token's router logits, by one wave.
#pragma once

#include "hybrid.h"

namespace mx {

// z [E] in LDS (destroyed): the `top` largest, in falling order (equal logits: the lower index), and the
// softmax over them alone
template <typename T>
__device__ __forceinline__ void moe_select(float* z, int E, int top, int lane, int32_t* ids, float* wts) {
  float zmax = 0.f, sum = 0.f;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int at = E;
    for (int e = lane; e < E; e += 64)
      if (z[e] > best) best = z[e], at = e;
    wave_pick(best, at);
    if (at >= E) at = 0;  // logits that are not numbers: some expert of the table
    if (k == 0) zmax = best;
    const float w = exp_t<float>(best - zmax);
    sum += w;
    if (lane == 0) {
      ids[k] = at;
      wts[k] = w;
      z[at] = -INFINITY;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the other lanes see the choice taken out
    __builtin_amdgcn_wave_barrier();
  }
  if (lane == 0)
    for (int k = 0; k < top; ++k) wts[k] /= sum;
}

// the same for at most 64 experts: lane e holds expert e's logit (other lanes anything); put(k, weight) on the
// lane of the k-th choice
template <typename F>
__device__ __forceinline__ void moe_choose64(float z, int E, int top, int lane, F put) {
  z = lane < E && z == z ? z : -INFINITY;  // (not a number: chosen last)
  int rank = 0;
  float zmax = -INFINITY;
  for (int e = 0; e < E; ++e) {
    const float v = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(z), e));
    rank += v > z || (v == z && e < lane);
    zmax = fmaxf(zmax, v);
  }
  const bool on = lane < E && rank < top;
  const float w = on ? exp_t<float>(z - zmax) : 0.f;
  const float sum = wave_sum(w);
  if (on) put(rank, w / sum);
}
// The same seen from one expert: lane t's answer is its place among the choices of token t (-1: not chosen, or t >= T).
// A workgroup of one expert needs no more than that, a token a lane; with all tokens' choices made in each, 8 waves had
// 600 instructions apiece for 32 tokens of 16 experts.
__device__ __forceinline__ int moe_place(const float* z, int E, int top, int T, int expert, int lane) {
  const float* zr = z + (int64_t)min(lane, T - 1) * E;
  auto number = [](float x) { return x == x ? x : -INFINITY; };  // (not a number: chosen last)
  const float own = number(zr[expert]);
  int rank = 0;
  auto count = [&](float x, int e) __attribute__((always_inline)) {
    const float u = number(x);
    rank += (int)(u > own) | ((int)(u == own) & (int)(e < expert));  // (no branches)
  };
  int e0 = 0;
  if (E % 4 == 0 && ((uintptr_t)z & 15) == 0)
    for (; e0 + 16 <= E; e0 += 16) {
      f32x4 v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const f32x4*>(zr + e0 + 4 * i);
#pragma unroll
      for (int i = 0; i < 16; ++i) count(v[i >> 2][i & 3], e0 + i);
    }
  for (; e0 < E; ++e0) count(zr[e0], e0);
  return lane < T && rank < top ? rank : -1;
}
// list[0 ..]: the pairs t top + place of the tokens that chose the expert; their number.  Every wave writes the whole
// list (the same values) and reads what it wrote: no barrier.
__device__ __forceinline__ int moe_list(int place, int top, int lane, int16_t* list) {
  const uint64_t on = __ballot(place >= 0);
  if (place >= 0) list[__popcll(on & ((1ull << lane) - 1))] = (int16_t)(lane * top + place);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  return __builtin_amdgcn_readfirstlane(__popcll(on));
}
__device__ __forceinline__ void moe_select64(float z, int E, int top, int lane, int32_t* ids, float* wts) {
  moe_choose64(z, E, top, lane, [&](int k, float w) {
    ids[k] = lane;
    wts[k] = w;
  });
}

}  // namespace mx
