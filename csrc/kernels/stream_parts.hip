// Decode GEMMs of 9 to 32 token rows whose K is too long for LDS: K in segments, a workgroup holds its segment of X in LDS and
// streams the weights of a run of channel groups past it (stream_core.h); the segments' sums, f32, are added by whatever
// reads the product next (parts_norm_kernel here), which was a launch of its own before.
//
// What bounds it: weights read once.  skinny_gemm.hip reads X beside each 16 channels (16 rows: as many bytes as the
// weights), the library's kernels reach 4.4 TB/s.  With the norm behind it, 16 rows, us: 4096 x 14336 30.7 -> 26.5 (5.0 TB/s by
// itself), 2048 x 8192 16.1 -> 13.6, 2048 x 12288 21.7 -> 15.6, 4096 x 21504 (skinny_gemm; past 16 rows the library's 125)
// 51.5 -> 40.6.  More segments are more workgroups' worth of groups dealt evenly and less of X in front of the first product, but
// more parts to write and add.
#include <algorithm>
#include <climits>

#include "stream_core.h"

namespace mx {

constexpr int kPartsRows = 32, kPartsLds = 158 * 1024;

struct PartsArgs {
  const uint16_t* X;
  int64_t ldx;
  const uint16_t* W;
  int64_t ldw;
  float* Y;  // [segments, M, N]
  int M, N, seg;
};

template <int KIND, int NL>
__global__ void __launch_bounds__(512, 2) stream_parts_kernel(PartsArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int c = threadIdx.x & 15, g = threadIdx.x >> 4 & 3, M = a.M;
  const int64_t k0 = (int64_t)blockIdx.y * a.seg;
  float* const y = a.Y + (int64_t)blockIdx.y * M * a.N;
  auto row = [&](int grp) __attribute__((always_inline)) -> int64_t { return (int64_t)grp * 16; };
  auto off = [&](int ch) __attribute__((always_inline)) -> int { return ch; };
  auto stage = [&](uint16_t* xs, int ldx, auto ahead) __attribute__((always_inline)) {
    stream_rows_in<8>(a.X + k0, a.ldx, M, a.seg, xs, ldx, ahead);
  };
  auto finish = [&](const f32x4& s, int mb, int grp) __attribute__((always_inline)) {
    const int m = mb * 16 + c;
    if (m < M) *reinterpret_cast<f32x4*>(y + (int64_t)m * a.N + (int64_t)grp * 16 + 4 * g) = s;
  };
  stream_walk<KIND, 2, 8, NL>(a.W + k0, a.ldw, nullptr, M, a.seg, (int)blockIdx.x, (int)gridDim.x, a.N / 16, smem, row, off,
                              stage, finish);
}

template <int KIND, int NL>
static int parts_launch(const PartsArgs& a, dim3 grid, size_t lds, hipStream_t stream) {
  static const bool big = hipFuncSetAttribute((const void*)stream_parts_kernel<KIND, NL>,
                                              hipFuncAttributeMaxDynamicSharedMemorySize, kPartsLds) == hipSuccess;
  if (!big) return -1;
  stream_parts_kernel<KIND, NL><<<grid, 512, lds, stream>>>(a);
  return (int)hipGetLastError();
}

// rmsnorm.hip's norm of (parts summed and rounded to bf16) + residual: a row a workgroup of 1,024 threads, so that the parts'
// loads are in flight together (256 threads took 4.3 us with 4 parts of 4,096, 6.0 with 7)
template <int ITERS>
__global__ void __launch_bounds__(1024) parts_norm_kernel(const float* __restrict__ parts, int S, int64_t seg,
                                                          const uint16_t* __restrict__ res, const uint16_t* __restrict__ w,
                                                          uint16_t* __restrict__ y, uint16_t* __restrict__ h_out, int H, float eps) {
  __shared__ float scratch[16];
  const size_t base = (size_t)blockIdx.x * H;
  f32x4 v[ITERS];
  u16x4 gw[ITERS], rv[ITERS];
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = min((it * 1024 + (int)threadIdx.x) * 4, H - 4);  // (past the end: read, not used)
    v[it] = f32x4{0.f, 0.f, 0.f, 0.f};
    gw[it] = *reinterpret_cast<const u16x4*>(w + c);
    rv[it] = *reinterpret_cast<const u16x4*>(res + base + c);
  }
  for (int s0 = 0; s0 < S; s0 += 8) {
    f32x4 p[8][ITERS];
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int it = 0; it < ITERS; ++it)
        p[s][it] = *reinterpret_cast<const f32x4*>(parts + min(s0 + s, S - 1) * seg + base +
                                                   min((it * 1024 + (int)threadIdx.x) * 4, H - 4));
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int it = 0; it < ITERS; ++it)
        if (s0 + s < S) v[it] += p[s][it];
  }
  float ss = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * 1024 + (int)threadIdx.x) * 4;
    if (c < H) {
      u16x4 hb;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        hb[j] = f2bf(bf2f(f2bf(v[it][j])) + bf2f(rv[it][j]));
        v[it][j] = bf2f(hb[j]);
        ss += v[it][j] * v[it][j];
      }
      *reinterpret_cast<u16x4*>(h_out + base + c) = hb;
    }
  }
  ss = block_sum(ss, scratch);
  const float rs = rsqrtf(ss / (float)H + eps);
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * 1024 + (int)threadIdx.x) * 4;
    if (c < H) {
      u16x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = f2bf(v[it][j] * rs * bf2f(gw[it][j]));
      *reinterpret_cast<u16x4*>(y + base + c) = o;
    }
  }
}

// chunks of 512 k (64 a wave) of a block of loads, two in flight: the longest of these that divides a segment's
static int parts_block(int chunks) {
  for (int u : {8, 7, 6, 4, 3})
    if (chunks % u == 0) return u;
  return 0;
}

}  // namespace mx

using namespace mx;

// Segments of K for M rows times [N, K]; 0: not taken.  A workgroup a CU; what the busiest reads, weights and its segment of X,
// and its share of the parts, written and read.
extern "C" int mx_stream_parts_segments(int M, int N, int K) {
  if (M < 1 || M > kPartsRows || N <= 0 || N % 16 || K <= 0 || K % 512) return 0;
  int best = 0;
  int64_t least = INT64_MAX;
  for (int s = 1; s <= 16; ++s) {
    const int seg = K / s;
    if (K % s || seg % 512 || !parts_block(seg / 512) || 16 * 1024 + (int64_t)M * (seg + 8) * 2 > kPartsLds) continue;
    const int wgs = 256 / s, turns = (N / 16 + wgs - 1) / wgs;
    const int64_t cost = (int64_t)seg * (16 * turns + M) + (int64_t)s * M * N / 64;
    if (cost < least) best = s, least = cost;
  }
  return best;
}

// parts [segments, M, N] f32 = X's segments times W's; -1: sizes, strides or addresses it does not take
extern "C" int mx_stream_parts(const uint16_t* x, int64_t ldx, const uint16_t* w, int64_t ldw, float* parts, int M, int N, int K,
                               hipStream_t stream) {
  const int s = mx_stream_parts_segments(M, N, K);
  if (!s || ldx % 8 || ldw % 8 || ldx < K || ldw < K || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)parts) & 15) ||
      ldw * 512 >> 32)
    return -1;
  const int seg = K / s;
  PartsArgs a{x, ldx, w, ldw, parts, M, N, seg};
  const dim3 grid(std::min(256 / s, N / 16), s);
  const size_t lds = 16 * 1024 + (size_t)M * (seg + 8) * 2;
#define MX_SP(U) \
  return M <= 16 ? parts_launch<kStLines, 2 * U>(a, grid, lds, stream) : parts_launch<kStWide, 2 * U>(a, grid, lds, stream)
  switch (parts_block(seg / 512)) {
    case 8: MX_SP(8);
    case 7: MX_SP(7);
    case 6: MX_SP(6);
    case 4: MX_SP(4);
    default: MX_SP(3);
  }
#undef MX_SP
}

// y [M, H] = rmsnorm(h_out) * w, h_out = res + the parts' sum rounded to bf16
extern "C" int mx_parts_norm(const float* parts, int S, const uint16_t* res, const uint16_t* w, uint16_t* y, uint16_t* h_out,
                             int M, int H, float eps, hipStream_t stream) {
  if (M <= 0) return 0;
  if (S < 1 || H <= 0 || H % 8 || H > 8192 ||
      (((uintptr_t)parts | (uintptr_t)res | (uintptr_t)w | (uintptr_t)y | (uintptr_t)h_out) & 15))
    return -1;
  const int64_t seg = (int64_t)M * H;
#define MX_PN(I) parts_norm_kernel<I><<<M, 1024, 0, stream>>>(parts, S, seg, res, w, y, h_out, H, eps)
  if (H <= 4096) MX_PN(1);
  else MX_PN(2);
#undef MX_PN
  return (int)hipGetLastError();
}
