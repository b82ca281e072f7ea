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
__device__ __forceinline__ void moe_select64(float z, int E, int top, int lane, int32_t* ids, float* wts) {
  moe_choose64(z, E, top, lane, [&](int k, float w) {
    ids[k] = lane;
    wts[k] = w;
  });
}

}  // namespace mx
