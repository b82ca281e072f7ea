// Prompt rows of sigusun (mxllm/models/sigusun.py) behind a layer's mixer, one launch: h += rms(src) w with its copy, as post_norm_kernel
// has it, and the experts of each row, as moe_route_mfma_kernel chooses them.
#include "hybrid.h"
#include "moe_route.h"
#include "skinny_core.h"
#include "sublayer.h"

namespace mx {

constexpr int kPrRows = 8;  // rows of a workgroup, one a wave

// W = 1024 NIT, up to 16 experts.  What bounds it: the rows' bytes.  The router read 16 MB of copies again that had just been written, in
// a launch of its own.  Here a wave norms a row (lane l holds the columns of post_norm_kernel's threads l, 64 + l, 128 + l and 192 + l and
// sums as that one does) and leaves its copy in LDS; then the waves share K as the router's do, with weights asked for ahead of the
// barrier: 128 KB a workgroup for W 4096, which is little beside the rows (the second embedding's
// matrices, eight times as much, are not: a kernel that had them as well behind the experts' mix was level).  Two launches -> one, replayed,
// us, 33 / 300 / 1000 / 2048 / 4096 / 8192 rows: W 4096 14.3 / 15.5 / 19.9 / 27.0 / 41.7 / 81.9 -> 11.5 / 12.2 / 14.7 / 19.4 / 36.8 / 75.0,
// 2048 13.5 / 14.3 / 16.4 / 19.5 / 27.6 / 51.3 -> 7.3 / 7.8 / 8.8 / 11.4 / 19.8 / 35.1.  In a prompt pass of 2048 rows of W 4096, whose
// rows come from further away, 18 + 12 -> 26.5.  All of W 4096's stream asked for at once spills
// (2048 rows 24.4).
template <int NIT>
__global__ void __launch_bounds__(512, 4) post_route_kernel(PostRoute a) {
  constexpr int W = 1024 * NIT, NC = 4 * NIT, XS = 2 * W + 64, US = W / 512;
  __shared__ __attribute__((aligned(16))) char xs[kPrRows * XS];
  __shared__ f32x4 red[8][64];
  __shared__ float z[kPrRows][16];
  const PostNorm& p = a.p;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, g = lane >> 4;
  const int64_t r = (int64_t)blockIdx.x * kPrRows + wv, row = min(r, p.T - 1);
  const bool on = r < p.T;
  const uint16_t* src = reinterpret_cast<const uint16_t*>(p.src) + row * p.lds + 4 * lane;
  float* hp = p.h + row * W + 4 * lane;
  {
    u16x4 v[NC];  // chunk i: columns 256 i + 4 lane
    f32x4 h[NC];  // AH of them ahead
    constexpr int AH = NC < 8 ? NC : 8;
#pragma unroll
    for (int i = 0; i < NC; ++i) v[i] = *reinterpret_cast<const u16x4*>(src + 256 * i);
#pragma unroll
    for (int i = 0; i < AH; ++i) h[i] = *reinterpret_cast<const f32x4*>(hp + 256 * i);
    __builtin_amdgcn_sched_barrier(0);
    float tot = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float ss = 0.f;
#pragma unroll
      for (int it = 0; it < NIT; ++it)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float x = bf2f(v[4 * it + q][j]);
          ss += x * x;
        }
      tot += wave_sum(ss);
    }
    const float rs = 1.f / sqrtf(tot / (float)W + p.eps);
    uint16_t* yp = reinterpret_cast<uint16_t*>(p.y) + row * W + 4 * lane;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const f32x4 w = *reinterpret_cast<const f32x4*>(p.w + 256 * i + 4 * lane);
      if (i + AH < NC) h[i + AH] = *reinterpret_cast<const f32x4*>(hp + 256 * (i + AH));
      u16x4 x;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        h[i][j] += bf2f(v[i][j]) * rs * w[j];
        x[j] = f2bf(h[i][j]);
      }
      *reinterpret_cast<u16x4*>(xs + wv * XS + 2 * (256 * i + 4 * lane)) = x;
      if (on) {
        *reinterpret_cast<f32x4*>(hp + 256 * i) = h[i];
        *reinterpret_cast<u16x4*>(yp + 256 * i) = x;
      }
      if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (four chunks' loads at a time: registers)
    }
  }
  u16x8 m[US][2];
  const uint16_t* wr = a.m + (int64_t)min(c, a.E - 1) * W + 64 * wv + 16 * g;
#pragma unroll
  for (int u = 0; u < US; ++u) {
    m[u][0] = *reinterpret_cast<const u16x8*>(wr + 512 * u);
    m[u][1] = *reinterpret_cast<const u16x8*>(wr + 512 * u + 8);
  }
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  const char* xr = xs + (c & 7) * XS + 2 * (64 * wv + 16 * g);  // (columns 8 .. 15 of the products are not used)
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < US; ++u) {
    acc = mfma16_sk(m[u][0], *reinterpret_cast<const u16x8*>(xr + 1024 * u), acc);
    acc = mfma16_sk(m[u][1], *reinterpret_cast<const u16x8*>(xr + 1024 * u + 16), acc);
  }
  red[wv][lane] = acc;
  __syncthreads();
  if (wv == 0) {
    f32x4 s = red[0][lane];
#pragma unroll
    for (int i = 1; i < 8; ++i) s += red[i][lane];
    if (c < kPrRows)
#pragma unroll
      for (int i = 0; i < 4; ++i) z[c][4 * g + i] = s[i];
  }
  __syncthreads();
  if (on) moe_select64(lane < 16 ? z[wv][lane] : 0.f, a.E, a.top, lane, a.ids + row * a.top, a.wts + row * a.top);
}

}  // namespace mx

using namespace mx;

// bf16 rows; -1 (nothing launched): sizes it does not take
extern "C" int mx_post_route(const PostRoute* pa, hipStream_t stream) {
  const PostRoute& a = *pa;
  const PostNorm& p = a.p;
  if (p.T <= 0) return 0;
  if (p.mode != PostNorm::kRows || !p.src || !p.h || !p.w || !p.y || !a.m || !a.ids || !a.wts || a.E <= 0 || a.E > 16 || a.top <= 0 ||
      a.top > a.E || p.W <= 0 || p.W > 4096 || p.W % 1024 || p.lds % 4 || p.T > (int64_t)INT32_MAX * kPrRows ||
      (((uintptr_t)p.h | (uintptr_t)p.w | (uintptr_t)a.m) & 15) || (((uintptr_t)p.src | (uintptr_t)p.y) & 7))
    return -1;
  const unsigned grid = (unsigned)((p.T + kPrRows - 1) / kPrRows);
#define PR(N) post_route_kernel<N><<<grid, 512, 0, stream>>>(a)
  if (p.W == 1024) PR(1);
  else if (p.W == 2048) PR(2);
  else if (p.W == 3072) PR(3);
  else PR(4);
#undef PR
  return (int)hipGetLastError();
}
