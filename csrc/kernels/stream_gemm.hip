// Decode GEMMs over few workgroups that stay: Y[M, N] = X[M, K] . W[N, K]^T for M <= 32 token rows, bf16 or e4m3
// weights, X held in LDS.
//
// What bounds it: every weight is read once, at the rate memory gives it.  skinny_gemm.hip and fp8_gemm.hip give
// each 16 output channels a workgroup of their own, and each reads its K part of X beside its weights: as many
// bytes as the weights' at 16 rows (at 8 for e4m3), through the same load queue.  Here a workgroup stages X in LDS
// once (2 M K bytes) and walks over channel groups; only weights are left in the queue, and the next block of them
// is in flight while the last one is multiplied and summed.
//  * fragments, K parts and sums of skinny_core.h, or of fp8_gemm.hip for e4m3: the products and sums of the kernels
//    above, bit for bit;
//  * X is asked for in front of the first weights and worked on behind them: loads return in order, and __syncthreads
//    waits for all of them (with the weights in front and that barrier, 6144 x 4096 at 16 rows 17.6 us in a step, now
//    14.8; the e4m3 gate-up projection of 4 rows with its norm 26.5, now 23.6);
//  * blocks of 16 loads (K a multiple of 4096) or 8 (of 2048), two in flight: 128 or 64 registers, so that with up to
//    80 KB of LDS two workgroups share a CU;
//  * LDS rows are K + 8 long: the 16 rows that a fragment read touches start 4 banks apart;
//  * the waves take turns at a group's sum and epilogue (two LDS images, one barrier a group), the others go on;
//  * epilogues: plain, SwiGLU (8 gate and the matching 8 up channels), RoPE + cache append (heads of 64 or 128);
//    prologue: the RMSNorm with the residual add, up to 4 rows (decode_fuse.h).
// 28672 x 4096 (235 MB), rows 1 / 4 / 8 / 16: 39.4 / 39.6 / 39.4 / 41.4 us (6.0 TB/s; in fragments of 16 rows x 64 B 43.0 / 43.5 /
// 43.7 / 44.4) against skinny_gemm's 39.8 / 41.0 / 42.8 / 54.6 and hipBLASLt's 61 to 64; 16384 x 2048 (67 MB), 4 / 8 / 16 rows 12.9 /
// 13.4 / 15.4 (15.8 / 16.4 / 16.5); in e4m3, 28672 x 4096, rows 1 / 4 / 8: 22.2 / 22.4 / 22.8 (24.6 / 25.4 / 25.7 in
// 16 rows x 64 B) against fp8_gemm's 27.1 / 31.5 / 34.1; 4096 x 14336, 1 / 4 rows 12.9 / 14.3 (14.3 / 16.1).
// 6144 x 4096 is 384 groups on 256 CUs: half of the CUs had two and ended at 9.2 us where the others did at 6.7 (e4m3, 4 rows,
// in a step). 257 to 384 groups go as one and a half a workgroup, all loads in flight (stream_and_half): steps of
// llama3.1-8b with 1 / 4 / 8 / 16 rows 2990 / 3183 / 3520 / 3760 -> 2913 / 3106 / 3434 / 3752 us, in e4m3 1 / 4 / 8 rows 2048 /
// 2289 / 2619 -> 2041 / 2275 / 2585 (eight parts of K for a half: other bits, and no faster).
// Left: the launch's own 2 us before the first bytes arrive.
#include <algorithm>

#include "decode_fuse.h"
#include "stream_groups.h"

namespace mx {

enum { kStPlain, kStSwiglu, kStRope128, kStRope64 };

struct StreamArgs {
  const uint16_t* X;
  int64_t ldx;
  const void* W;  // bf16 [N, K], or e4m3 codes
  int64_t ldw;
  const float* scale;  // e4m3: one a row
  uint16_t* Y;
  int64_t ldy;
  int M, K, F, groups;
  SkNorm na;
  SkRope rp;
};

// workgroups of up to 128 registers: two a CU where LDS allows it (X of 9 rows and more of a K over 2048 does not)
template <int KIND, int TB, int KP, int NL>
constexpr int kStWaves = KIND >= kStF8 ? (TB == 1 ? 4 : 2) : NL == 8 && (TB == 1 || KP == 4) ? 4 : 2;

// HALF: 256 workgroups, of which each has a group and, in front of the last groups' count, half of one of those
template <int KIND, int TB, int KP, int EPI, bool NORM, int NL, bool HALF = false>
__global__ void __launch_bounds__(512, (HALF ? 2 : kStWaves<KIND, TB, KP, NL>)) stream_gemm_kernel(StreamArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, c = tid & 15, g = tid >> 4 & 3;
  const int M = a.M, K = a.K;
  auto row = [&](int grp) __attribute__((always_inline)) -> int64_t {
    if constexpr (EPI == kStSwiglu) return dfuse_row<true>(grp, 0, a.F);
    else if constexpr (EPI == kStRope128) return dfuse_row<false, 64>(grp, 0, 0);
    else if constexpr (EPI == kStRope64) return dfuse_row<false, 32>(grp, 0, 0);
    else return (int64_t)grp * 16;
  };
  auto off = [&](int ch) __attribute__((always_inline)) -> int {
    if constexpr (EPI == kStSwiglu) return (int)dfuse_row<true>(0, ch, a.F);
    else if constexpr (EPI == kStRope128) return (int)dfuse_row<false, 64>(0, ch, 0);
    else if constexpr (EPI == kStRope64) return (int)dfuse_row<false, 32>(0, ch, 0);
    else return ch;
  };
  auto stage = [&](uint16_t* xs, int ldx, auto ahead) __attribute__((always_inline)) {
    if constexpr (NORM) {
      __shared__ float nscr[4][4];
      dfuse_norm_ahead(a.X, a.ldx, M, K, a.na, xs, ldx, nscr, ahead);
    } else {
      stream_rows_in<KIND < kStF8 && NL == 16 ? 16 : 8>(a.X, a.ldx, M, K, xs, ldx, ahead);
    }
  };
  auto finish = [&](const f32x4& s, int mb, int cg, bool on = true) __attribute__((always_inline)) {
    const int m = on ? mb * 16 + c : M;
    if constexpr (EPI == kStRope128) {
      dfuse_rope_store<64, HALF>(s, g, m, M, cg, a.rp);
    } else if constexpr (EPI == kStRope64) {
      dfuse_rope_store<32, HALF>(s, g, m, M, cg, a.rp);
    } else if constexpr (EPI == kStSwiglu) {
      dfuse_swiglu_store(s, g, m, M, a.Y, a.ldy, cg);
    } else if (m < M) {
      u16x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = f2bf(s[i]);
      *reinterpret_cast<u16x4*>(a.Y + (int64_t)m * a.ldy + (int64_t)cg * 16 + 4 * g) = o;
    }
  };
  const int x = blockIdx.x;
  if constexpr (HALF)
    stream_and_half<KIND, TB, KP, NL>(a.W, a.ldw, a.scale, M, K, x, x < 2 * (a.groups - 256) ? 512 + x : -1, smem, row, off,
                                      stage, finish);
  else
    stream_walk<KIND, TB, KP, NL>(a.W, a.ldw, a.scale, M, K, x, (int)gridDim.x, a.groups, smem, row, off, stage, finish);
}

constexpr int kTwoLds = 80 * 1024;  // LDS up to which two workgroups share a CU

template <int KIND, int TB, int KP, int EPI, bool NORM, int NL, bool HALF = false>
static int stream_launch(const StreamArgs& a, int per_cu, size_t lds, hipStream_t stream) {
  static const bool big = hipFuncSetAttribute((const void*)stream_gemm_kernel<KIND, TB, KP, EPI, NORM, NL, HALF>,
                                              hipFuncAttributeMaxDynamicSharedMemorySize, 159 * 1024) == hipSuccess;
  if (!big) return -1;
  stream_gemm_kernel<KIND, TB, KP, EPI, NORM, NL, HALF><<<std::min(a.groups, 256 * per_cu), 512, lds, stream>>>(a);
  return (int)hipGetLastError();
}

// bf16 blocks of 16 loads (150 registers and more) leave a CU to one workgroup: where its LDS does that anyway
template <int KIND, int TB, int EPI, bool NORM>
static int stream_blocks(const StreamArgs& a, hipStream_t stream) {
  const bool four = KIND == kStLines && sk_parts(a.M, a.K) == 4;
  constexpr int KP8 = KIND == kStF8Lines ? 4 : 8;
  const size_t lds = (four ? kStreamRed<KIND, TB, 4> : kStreamRed<KIND, TB, KP8>) + (size_t)a.M * (a.K + 8) * 2;
  const int per_cu = lds <= kTwoLds ? 2 : 1;
  // (A K of 2048 has two workgroups a CU, so 512 groups are one turn; of a longer one a part is more than one block, and the registers
  // do not hold two of those.)
  if constexpr (KIND == kStLines || KIND == kStF8Lines)
    if (a.K == 4096 && a.groups > 256 && a.groups <= 384)
      return stream_launch<KIND, TB, KP8, EPI, NORM, KIND == kStLines ? 16 : 8, true>(a, 1, lds, stream);
  if constexpr (KIND >= kStF8) {
    return a.K % 4096 == 0 ? stream_launch<KIND, TB, KP8, EPI, NORM, 8>(a, per_cu, lds, stream)
                           : stream_launch<KIND, TB, KP8, EPI, NORM, 4>(a, per_cu, lds, stream);
  } else {
    if constexpr (KIND == kStLines)
      if (four) return stream_launch<KIND, TB, 4, EPI, NORM, 8>(a, per_cu, lds, stream);
    return a.K % 4096 == 0 && per_cu == 1 ? stream_launch<KIND, TB, 8, EPI, NORM, 16>(a, per_cu, lds, stream)
                                          : stream_launch<KIND, TB, 8, EPI, NORM, 8>(a, per_cu, lds, stream);
  }
}

template <bool F8, int EPI>
static int stream_rows(const StreamArgs& a, bool norm, hipStream_t stream) {
  constexpr int LINES = F8 ? kStF8Lines : kStLines, WIDE = F8 ? kStF8 : kStWide;
  if (norm) return stream_blocks<LINES, 1, EPI, true>(a, stream);
  if (a.M <= 8) return stream_blocks<LINES, 1, EPI, false>(a, stream);
  // 9 to 16 rows: whole lines, but for a K of 4096 of few groups, where the first bytes and the rows in LDS are what lasts (us,
  // lines -> 16 rows, 9 / 16 rows: 1024 x 4096 8.3 / 9.1 -> 8.2 / 8.8, 2048 8.7 / 9.5 -> 8.4 / 9.1; but 12288 20.8 / 21.8 -> 21.4 /
  // 22.0; 2048 x 2048 5.4 / 6.1 -> 5.6 / 6.0).  Between 192 and 256 groups they are level, and skinny_gemm.hip has these
  // sizes with the bits of whole lines.
  const bool few = a.groups <= 192;
  if (a.M <= 16 && (F8 || (a.K == 4096 && few))) return stream_blocks<WIDE, 1, EPI, false>(a, stream);
  if (a.M <= 16) return stream_blocks<LINES, F8 ? 1 : 2, EPI, false>(a, stream);
  return stream_blocks<WIDE, 2, EPI, false>(a, stream);
}

// The same with a grouped RMS norm of an f32 residual (+ delta) in front, up to 4 rows: Y = (rms(h + delta) gamma) . W^T, parts of
// K / 8 elements, one a wave, so that its sum needs no barrier.  EPT: elements of a row a thread.  Every workgroup does the
// norm, for all its channels; workgroup 0 stores the sum.  1 / 2 / 4 rows, us: 12288 x 2048 in hybrid_skinny.hip's prologue (every
// 16 channels) 13.4 / 14.3 / 18.7, norm and product apart 12.5 / 12.9 / 13.3, here 10.5 / 10.9 / 12.2; 21504 x 4096 33.6 / 38.6 /
// 47.4, 35.3 / 35.0 / 35.4, here 33.0 / 33.3 / 35.0.
template <int KP, int EPT>
__global__ void __launch_bounds__(512, 4) stream_group_norm_kernel(StreamArgs a, StreamGroups n) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, c = tid & 15, g = tid >> 4 & 3, M = a.M;
  constexpr int K = 512 * EPT;
  auto row = [&](int grp) __attribute__((always_inline)) -> int64_t { return (int64_t)grp * 16; };
  auto off = [&](int ch) __attribute__((always_inline)) -> int { return ch; };
  auto stage = [&](uint16_t* xs, int ldx, auto ahead) __attribute__((always_inline)) {
    stream_groups_in<EPT>(n, M, xs, ldx, ahead);
  };
  auto finish = [&](const f32x4& s, int mb, int cg) __attribute__((always_inline)) {
    const int m = mb * 16 + c;
    if (m >= M) return;
    u16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = f2bf(s[i]);
    *reinterpret_cast<u16x4*>(a.Y + (int64_t)m * a.ldy + (int64_t)cg * 16 + 4 * g) = o;
  };
  stream_walk<kStLines, 1, KP, 8>(a.W, a.ldw, nullptr, M, K, (int)blockIdx.x, (int)gridDim.x, a.groups, smem, row, off, stage,
                                  finish);
}

}  // namespace mx

using namespace mx;

// y [M, N] = (grouped rmsnorm of h + delta in 8 parts, times gamma) . w^T, h [M, K] f32 dense, K 2048 or 4096, up to 4 rows;
// h_out gets h + delta where delta is given.  -1: not taken, nothing launched
extern "C" int mx_stream_group_norm(const float* h, const uint16_t* delta, int64_t ldd, const float* gamma, float eps,
                                    float* h_out, const uint16_t* w, int64_t ldw, uint16_t* y, int M, int N, int K,
                                    hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 4 || (K != 2048 && K != 4096) || N <= 0 || N % 16 || ldw % 8 || ldw < K || ldw * 512 >> 32 ||
      (delta && (!h_out || ldd % 4 || ldd < K)) ||
      (((uintptr_t)h | (uintptr_t)gamma | (uintptr_t)h_out | (uintptr_t)w | (uintptr_t)delta | (uintptr_t)y) & 15))
    return -1;
  const StreamArgs a{nullptr, 0, w, ldw, nullptr, y, N, M, K, 0, N / 16};
  const StreamGroups n{h, delta, ldd, gamma, h_out, eps};
  const unsigned grid = std::min(N / 16, 512);
  const size_t x = (size_t)M * (K + 8) * 2;  // both below the 64 KB that need no leave
  if (K == 2048) stream_group_norm_kernel<4, 4><<<grid, 512, kStreamRed<kStLines, 1, 4> + x, stream>>>(a, n);
  else stream_group_norm_kernel<8, 8><<<grid, 512, kStreamRed<kStLines, 1, 8> + x, stream>>>(a, n);
  return (int)hipGetLastError();
}

// Whether mx_stream_gemm takes M rows of K: X and the partial sums in 160 KB of LDS, whole blocks a wave.
extern "C" int mx_stream_ok(int M, int K, int norm) {
  const int64_t lds = 16 * 1024 + (int64_t)M * (K + 8) * 2;
  return M >= 1 && M <= (norm ? 4 : 32) && K % 2048 == 0 && lds <= 158 * 1024;
}

// epi 0: y [M, N]; 1: w = [gate; up], y [M, N / 2] = silu(g) u; 2 / 3: the QKV projection of heads of 128 / 64 (N =
// (Hq + 2 Hkv) heads), q rotated, K / V appended to the caches at (slot, pos).  scale: w is e4m3 codes, else bf16.
// gamma: X = rmsnorm(h + delta) of up to 4 rows (x = h; delta may be null, else h_out gets h + delta).  What is read,
// and h_out, 16-B aligned, the other outputs 8-B; other sizes, strides and addresses: -1, nothing launched.
extern "C" int mx_stream_gemm(const uint16_t* x, int64_t ldx, const void* w, int64_t ldw, const float* scale, uint16_t* y,
                              int64_t ldy, int M, int N, int K, int epi, const uint16_t* delta, int64_t ldd,
                              const uint16_t* gamma, float eps, uint16_t* h_out, const float* cosb, const float* sinb,
                              const int32_t* pos, const int32_t* slots, uint16_t* q, uint16_t* kc, uint16_t* vc, int Hq,
                              int Hkv, int max_seq, const int32_t* bt, int maxb, hipStream_t stream) {
  if (M <= 0) return 0;
  if (!mx_stream_ok(M, K, gamma != nullptr) || N % 16 || ldx % 8 || ldw % (scale ? 16 : 8) || ldx < K || ldw < K ||
      epi < 0 || epi > 3 || (delta && (!gamma || ldd % 8 || ldd < K || !h_out)))
    return -1;
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)scale | (uintptr_t)delta | (uintptr_t)gamma | (uintptr_t)h_out) & 15 ||
      ((uintptr_t)y | (uintptr_t)q | (uintptr_t)kc | (uintptr_t)vc) & 7)
    return -1;
  if (epi >= 2 ? N != (Hq + 2 * Hkv) * (epi == 2 ? 128 : 64) : (ldy % 4 || ldy < (epi == 1 ? N / 2 : N))) return -1;
  if ((int64_t)(epi == 1 ? N / 2 + 16 : 256) * ldw * (scale ? 1 : 2) >> 32) return -1;  // offsets inside a group
  StreamArgs a{x, ldx, w, ldw, scale, y, ldy, M, K, N / 2, N / 16, SkNorm{delta, ldd, gamma, h_out, eps},
               SkRope{cosb, sinb, pos, slots, q, kc, vc, Hq, Hkv, max_seq, bt, maxb}};
  const bool norm = gamma != nullptr;
#define MX_ST(E) return scale ? stream_rows<true, E>(a, norm, stream) : stream_rows<false, E>(a, norm, stream)
  if (epi == 0) MX_ST(kStPlain);
  if (epi == 1) MX_ST(kStSwiglu);
  if (epi == 2) MX_ST(kStRope128);
  MX_ST(kStRope64);
#undef MX_ST
}
