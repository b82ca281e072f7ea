// The grouped RMS norm of an f32 residual in front of the workgroups that stay (stream_gemm.hip, stream_hybrid.hip).
#pragma once

#include "stream_core.h"

namespace mx {

struct StreamGroups {
  const float* h;         // [M, K] dense
  const uint16_t* delta;  // or nullptr
  int64_t ldd;
  const float* gamma;
  float* h_out;
  float eps;
};

// up to 4 rows of (rms(h + delta) gamma), K = 512 EPT, in 8 parts, one a wave, so that its sum needs no barrier, into xs [M, K] (row
// stride ldx); ends with a barrier, calls ahead() behind its own reads.  Workgroup 0 stores h + delta.
template <int EPT, typename Ahead>
__device__ __forceinline__ void stream_groups_in(const StreamGroups& n, int M, uint16_t* xs, int ldx, const Ahead& ahead) {
  constexpr int K = 512 * EPT, Q = EPT / 4;
  const int tid = threadIdx.x, cc = tid * EPT;
  f32x4 h[4][Q], gm[Q];
  u16x4 d[4][Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    gm[i] = *reinterpret_cast<const f32x4*>(n.gamma + cc + 4 * i);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int mm = min(m, M - 1);
      h[m][i] = *reinterpret_cast<const f32x4*>(n.h + (int64_t)mm * K + cc + 4 * i);
      d[m][i] = n.delta ? *reinterpret_cast<const u16x4*>(n.delta + (int64_t)mm * n.ldd + cc + 4 * i) : u16x4{0, 0, 0, 0};
    }
  }
  ahead();
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    if (m >= M) break;
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      if (n.delta) {
#pragma unroll
        for (int j = 0; j < 4; ++j) h[m][i][j] += bf2f(d[m][i][j]);
        if (blockIdx.x == 0) *reinterpret_cast<f32x4*>(n.h_out + (int64_t)m * K + cc + 4 * i) = h[m][i];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) ss += h[m][i][j] * h[m][i][j];
    }
    const float rs = 1.f / sqrtf(wave_sum(ss) / (float)(K / 8) + n.eps);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      u16x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = f2bf(h[m][i][j] * rs * gm[i][j]);
      *reinterpret_cast<u16x4*>(xs + m * ldx + cc + 4 * i) = o;
    }
  }
  lds_barrier();
}

}  // namespace mx
