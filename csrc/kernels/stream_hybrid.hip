// Fused decode projections of the recurrent / chunked-attention decoders on the workgroups that stay (stream_core.h), up to 16 rows:
// the epilogues of hybrid_skinny.hip (minGRU step; convolution, rotation and cache append), X in LDS once a workgroup, and for up to 4
// rows of a norm in 8 parts the norm in its prologue.
//
// What bounds it: as hybrid_skinny.hip, a workgroup to every 16 channels that reads its rows of X beside the weights, the
// projections of 25 MB ran at 2.6 TB/s, and the norm of 3 and 4 rows was a launch of its own.
// Norm and projection, us (apart or in hybrid_skinny.hip's prologue -> here), 1 / 2 / 4 rows, weights from memory, 8 parts:
//   minGRU, 3 x 2048 x 2048 8.7 / 10.2 / 12.1 -> 8.7 / 9.1 / 10.1; 3 x 4096 x 4096 23.8 / 24.7 / 25.5 -> 23.7 / 23.7 / 24.8;
//   convolved, 5120 x 2048 9.0 / 10.0 / 11.6 -> 8.3 / 8.4 / 9.4; 10240 x 4096 20.7 / 20.6 / 21.2 -> 20.7 / 20.4 / 22.0 (in a step, where
//   the norm's launch costs more, 3 and 4 rows gain 0.6 %);
// rows that were normed before, 5 / 8 / 16: minGRU 9.5 / 10.9 / 14.5 -> 8.8 / 9.5 / 10.8 and, up to 8 rows, 22.3 / 25.2 -> 21.2 / 22.4;
// convolved 9.1 / 10.4 / 13.6 -> 8.5 / 8.9 / 9.6.  Those of 4096 stay where they were: the convolution's up to 8 rows (10240 x 4096, 640
// groups on 512 places are dealt unevenly: 5 / 8 18.6 / 20.0 -> 20.3 / 20.8; a workgroup a group 24.3 / 25.4), both past them, where
// steps of the 8B size are faster with the library's products (16 sequences 4181, here 4214).
// Steps of the 1B size, 700 keys, 2 / 3 / 4 / 8 / 9 / 16 sequences: 819 / 871 / 901 / 994 / 998 / 1057 -> 800 / 827 / 853 / 970 / 959 / 1021 us.
// Left: 25 MB in 8.8 us; a minGRU workgroup has one group of rows, a quarter of whose fragment is idle, and ends with two
// loads behind each other (slot, state).  Those asked for behind the first weights: 0.3 us less, the convolution's 0.8 more.
#include <algorithm>

#include "hybrid_fuse.h"
#include "stream_groups.h"

namespace mx {

struct StreamHybrid {
  const uint16_t* X;  // or the norm's h
  int64_t ldx;
  const uint16_t* W;
  int64_t ldw;
  uint16_t* Y;
  int M, K, groups;
  StreamGroups n;
};

// EPT: elements of a row a thread of the norm (K = 512 EPT); 0: X as it is
template <bool GRU, int TB, int KP, int EPT>
__global__ void __launch_bounds__(512, 4) stream_hybrid_kernel(StreamHybrid a, HsGru gr, HsConv cv) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4, M = a.M;
  auto row = [&](int grp) __attribute__((always_inline)) -> int64_t { return GRU ? (int64_t)grp * 4 : (int64_t)grp * 16; };
  auto off = [&](int ch) __attribute__((always_inline)) -> int { return GRU ? (int)hs_gru_row(0, ch, gr.W) : ch; };
  auto stage = [&](uint16_t* xs, int ldx, auto ahead) __attribute__((always_inline)) {
    if constexpr (EPT) stream_groups_in<EPT>(a.n, M, xs, ldx, ahead);
    else stream_rows_in<8>(a.X, a.ldx, M, a.K, xs, ldx, ahead);
  };
  auto finish = [&](const f32x4& s, int mb, int cg) __attribute__((always_inline)) {
    if constexpr (GRU) hs_gru_store(s, lane, M, cg, gr, a.Y);
    else hs_conv_store(s, cg * 16 + 4 * g, c, M, cv);
  };
  stream_walk<kStLines, TB, KP, 8>(a.W, a.ldw, nullptr, M, EPT ? 512 * EPT : a.K, (int)blockIdx.x, (int)gridDim.x, a.groups, smem,
                                    row, off, stage, finish);
}

template <bool GRU, int TB, int KP, int EPT>
static int sh_launch(const StreamHybrid& a, const HsGru& gr, const HsConv& cv, hipStream_t stream) {
  const size_t lds = kStreamRed<kStLines, TB, KP> + (size_t)a.M * (a.K + 8) * 2;
  static const bool big = hipFuncSetAttribute((const void*)stream_hybrid_kernel<GRU, TB, KP, EPT>,
                                              hipFuncAttributeMaxDynamicSharedMemorySize, 159 * 1024) == hipSuccess;
  if (!big) return -1;
  const int per_cu = lds <= 80 * 1024 ? 2 : 1;  // (as stream_gemm.hip)
  stream_hybrid_kernel<GRU, TB, KP, EPT><<<std::min(a.groups, 256 * per_cu), 512, lds, stream>>>(a, gr, cv);
  return (int)hipGetLastError();
}

// whether the rows, and the norm where there is one, fit; -1 and nothing launched where they do not
template <bool GRU>
static int sh_run(const StreamHybrid& a, int parts, const HsGru& gr, const HsConv& cv, hipStream_t stream) {
  const bool norm = a.n.h != nullptr;
  if (a.M < 1 || a.M > (norm ? 4 : 16) || (a.K != 2048 && a.K != 4096) || a.groups <= 0 || a.ldw % 8 || a.ldw < a.K) return -1;
  if (!norm && a.K == 4096 && (!GRU || a.M > 8)) return -1;  // (above)
  const int64_t span = (GRU ? 2 * (int64_t)gr.W + 4 : 16) * a.ldw * 2;  // offsets of 32 bits inside a group
  if (span >> 32) return -1;
  if (norm ? parts != 8 || (a.n.delta && (!a.n.h_out || a.n.ldd % 4 || a.n.ldd < a.K)) : !a.X || a.ldx % 8 || a.ldx < a.K) return -1;
  if (((uintptr_t)a.X | (uintptr_t)a.W | (uintptr_t)a.n.h | (uintptr_t)a.n.delta | (uintptr_t)a.n.gamma | (uintptr_t)a.n.h_out) & 15)
    return -1;
  if (norm) return a.K == 2048 ? sh_launch<GRU, 1, 4, 4>(a, gr, cv, stream) : sh_launch<GRU, 1, 8, 8>(a, gr, cv, stream);
  if (a.K == 2048)
    return a.M <= 8 ? sh_launch<GRU, 1, 4, 0>(a, gr, cv, stream) : sh_launch<GRU, 2, 4, 0>(a, gr, cv, stream);
  if constexpr (GRU) return sh_launch<true, 1, 8, 0>(a, gr, cv, stream);
  return -1;
}

}  // namespace mx

using namespace mx;

// As mx_hs_gru_gemm and mx_hs_conv_gemm (hybrid_skinny.hip), which ask them first; -1: not taken, nothing launched.
extern "C" int mx_stream_gru(const uint16_t* x, int64_t ldx, const uint16_t* delta, int64_t ldd, const float* h, const float* gamma,
                             float* h_out, int groups, float eps, const uint16_t* w, int64_t ldw, const float* bias,
                             const int32_t* slots, float* state, uint16_t* y, int M, int W, int K, hipStream_t stream) {
  if (W <= 0 || W % 4) return -1;
  const StreamHybrid a{h ? nullptr : x, ldx, w, ldw, y, M, K, W / 4, StreamGroups{h, delta, ldd, gamma, h_out, eps}};
  return sh_run<true>(a, groups, HsGru{bias, slots, state, W}, HsConv{}, stream);
}

extern "C" int mx_stream_conv(const uint16_t* x, int64_t ldx, const uint16_t* delta, int64_t ldd, const float* h,
                              const float* gamma, float* h_out, int groups, float eps, const uint16_t* w, int64_t ldw,
                              const ConvRope* pa, const int32_t* pos, const int32_t* slots, uint16_t* gate, int M, int K,
                              hipStream_t stream) {
  const int N = hs_conv_rows(*pa);
  const StreamHybrid a{h ? nullptr : x, ldx, w, ldw, nullptr, M, K, N / 16, StreamGroups{h, delta, ldd, gamma, h_out, eps}};
  return sh_run<false>(a, groups, HsGru{}, HsConv{*pa, pos, slots, gate}, stream);
}
