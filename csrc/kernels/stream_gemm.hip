// Decode GEMMs over few workgroups that stay: Y[M, N] = X[M, K] . W[N, K]^T for M <= 32 token rows, bf16 or e4m3
// weights, X held in LDS.
//
// What bounds it: every weight is read once, at the rate memory gives it.  skinny_gemm.hip and fp8_gemm.hip give
// each 16 output channels a workgroup of their own, and each reads its K part of X beside its weights: as many
// bytes as the weights' at 16 rows (at 8 for e4m3), through the same load queue.  Here a workgroup stages X in LDS
// once (2 M K bytes) and walks over channel groups; only weights are left in the queue, and the next block of them
// is in flight while the last one is multiplied and summed.
//  * 8 waves split K in eight contiguous parts, 64-k chunks of two v_mfma_f32_16x16x32_bf16 with the weights as
//    the A operand, partial sums in wave order: the products and sums of the kernels above, bit for bit;
//  * X is asked for in front of the first weights and worked on behind them: loads return in order, and __syncthreads
//    waits for all of them (with the weights in front and that barrier, 6144 x 4096 at 16 rows 17.6 us in a step, now
//    14.8; the e4m3 gate-up projection of 4 rows with its norm 26.5, now 23.6);
//  * blocks of U chunks, two in flight: 8 (K a multiple of 4096) or 4 (of 2048): 128 or 64 registers, so that
//    with up to 80 KB of LDS two workgroups share a CU;
//  * LDS rows are K + 8 long: the 16 rows that a fragment read touches start 4 banks apart;
//  * the waves take turns at a group's sum and epilogue (two LDS images, one barrier a group), the others go on;
//  * epilogues: plain, SwiGLU (8 gate and the matching 8 up channels), RoPE + cache append (heads of 64 or 128);
//    prologue: the RMSNorm with the residual add, up to 4 rows (decode_fuse.h).
// 28672 x 4096 (235 MB) with SwiGLU, rows 1 / 4 / 8 / 16: 42.6 / 42.9 / 43.3 / 43.8 us (5.5 TB/s) against skinny_gemm's
// 43.6 / 47.3 / 54.9 / 67.1 and hipBLASLt's 67; in e4m3, rows 1 / 4 / 8: 24.9 / 25.8 / 28.6 against fp8_gemm's 28.4 / 32.2
// / 36.4.  128256 x 2048, 8 rows: 98 against 109 and 114.
// Left: the last groups' uneven end (6144 x 4096 is 384 groups on 256 workgroups: 14.8 us for 50 MB; the last 128 as
// 256 halves: no change, a half's loads take a whole one's turns).
#include <algorithm>

#include "decode_fuse.h"
#include "e4m3.h"
#include "skinny_core.h"

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

template <bool F8, int U>
struct WFrag {
  u16x8 a[U][2];
  __device__ __forceinline__ void load(const char* p) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      a[u][0] = *reinterpret_cast<const u16x8*>(p + u * 128);
      a[u][1] = *reinterpret_cast<const u16x8*>(p + u * 128 + 16);
    }
  }
  __device__ __forceinline__ void get(int u, u16x8& x, u16x8& y) const { x = a[u][0], y = a[u][1]; }
};
template <int U>
struct WFrag<true, U> {
  u32x4 a[U];
  __device__ __forceinline__ void load(const char* p) {
#pragma unroll
    for (int u = 0; u < U; ++u) a[u] = *reinterpret_cast<const u32x4*>(p + u * 64);
  }
  __device__ __forceinline__ void get(int u, u16x8& x, u16x8& y) const {
    x = dequant8(a[u][0], a[u][1]);
    y = dequant8(a[u][2], a[u][3]);
  }
};

template <bool F8, int MB, int EPI, bool NORM, int U>
__global__ void __launch_bounds__(512, MB == 1 && (F8 || U == 4) ? 4 : 2) stream_gemm_kernel(StreamArgs a) {
  constexpr int NW = kSkWaves, NRED = MB == 1 ? 2 : 1, WB = F8 ? 1 : 2;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int M = a.M, K = a.K, kq = K / NW, nblk = kq / (64 * U), ldx = K + 8;
  f32x4(*red)[NW][MB][64] = reinterpret_cast<f32x4(*)[NW][MB][64]>(smem);
  uint16_t* xs = reinterpret_cast<uint16_t*>(smem + sizeof(f32x4) * NRED * NW * MB * 64);
  auto row = [&](int grp, int ch) -> int64_t {
    if constexpr (EPI == kStSwiglu) return dfuse_row<true>(grp, ch, a.F);
    else if constexpr (EPI == kStRope128) return dfuse_row<false, 64>(grp, ch, 0);
    else if constexpr (EPI == kStRope64) return dfuse_row<false, 32>(grp, ch, 0);
    else return (int64_t)grp * 16 + ch;
  };
  // the block to load next: group lg, block lb
  int lg = blockIdx.x, lb = 0;
  const char* base = reinterpret_cast<const char*>(a.W) + ((int64_t)w * kq + 16 * g) * WB;
  const char* lp = base + row(lg, c) * a.ldw * WB;
  auto load = [&](WFrag<F8, U>& f) {
    f.load(lp + (int64_t)lb * (U * 64 * WB));
    if (++lb == nblk) {
      lb = 0;
      lg += gridDim.x;
      lp = base + row(min(lg, a.groups - 1), c) * a.ldw * WB;
    }
  };
  WFrag<F8, U> f0, f1;
  // the first block goes out behind the reads of X, which return before it, and in front of the work on them
  if constexpr (NORM) {
    __shared__ float nscr[4][4];
    dfuse_norm_ahead(a.X, a.ldx, M, K, a.na, xs, ldx, nscr, [&]() __attribute__((always_inline)) { load(f0); });
  } else {
    constexpr int XP = !F8 && U == 8 ? 16 : 8;  // 16-B pieces of X a thread holds: all, or the last ones
    const int per = K / 8, total = M * per;
    u16x8 v[XP];
    auto fetch = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < XP; ++i) {
        const int p = min(p0 + tid + 512 * i, total - 1), m = p / per;
        v[i] = *reinterpret_cast<const u16x8*>(a.X + (int64_t)m * a.ldx + (p - m * per) * 8);
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
    load(f0);
    put(p0);
    lds_barrier();
  }
  const uint16_t* xr[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) xr[mb] = xs + min(mb * 16 + c, M - 1) * ldx + w * kq + 16 * g;

  f32x4 acc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  int cg = blockIdx.x, cb = 0, turn = 0;
  auto multiply = [&](const WFrag<F8, U>& f) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      u16x8 a0, a1;
      f.get(u, a0, a1);
      const int k = (cb * U + u) * 64;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        acc[mb] = mfma16_sk(a0, *reinterpret_cast<const u16x8*>(xr[mb] + k), acc[mb]);
        acc[mb] = mfma16_sk(a1, *reinterpret_cast<const u16x8*>(xr[mb] + k + 8), acc[mb]);
      }
    }
    if (++cb < nblk) return;
    cb = 0;
    const int par = NRED == 2 ? turn & 1 : 0;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      red[par][w][mb][lane] = acc[mb];
      acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    lds_barrier();
    if (w == (turn & (NW - 1))) {
      f32x4 sc = {1.f, 1.f, 1.f, 1.f};
      if constexpr (F8) sc = *reinterpret_cast<const f32x4*>(a.scale + row(cg, 4 * g));
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        f32x4 s = red[par][0][mb][lane];
#pragma unroll
        for (int ww = 1; ww < NW; ++ww) s += red[par][ww][mb][lane];
        if constexpr (F8) s *= sc;
        const int m = mb * 16 + c;
        if constexpr (EPI == kStRope128) {
          dfuse_rope_store<64>(s, g, m, M, cg, a.rp);
        } else if constexpr (EPI == kStRope64) {
          dfuse_rope_store<32>(s, g, m, M, cg, a.rp);
        } else if constexpr (EPI == kStSwiglu) {
          dfuse_swiglu_store(s, g, m, M, a.Y, a.ldy, cg);
        } else if (m < M) {
          u16x4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = f2bf(s[i]);
          *reinterpret_cast<u16x4*>(a.Y + (int64_t)m * a.ldy + (int64_t)cg * 16 + 4 * g) = o;
        }
      }
    }
    if constexpr (NRED == 1) lds_barrier();  // one image: its sum is read before the next group's parts
    ++turn;
    cg += gridDim.x;
  };
  const int steps = (a.groups - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x * nblk;
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

constexpr int kRedBytes = 16 * 1024;  // the partial sums' images
constexpr int kTwoLds = 80 * 1024;    // LDS up to which two workgroups share a CU

template <bool F8, int MB, int EPI, bool NORM, int U>
static int stream_launch(const StreamArgs& a, int per_cu, size_t lds, hipStream_t stream) {
  static const bool big = hipFuncSetAttribute((const void*)stream_gemm_kernel<F8, MB, EPI, NORM, U>,
                                              hipFuncAttributeMaxDynamicSharedMemorySize, 159 * 1024) == hipSuccess;
  if (!big) return -1;
  stream_gemm_kernel<F8, MB, EPI, NORM, U><<<std::min(a.groups, 256 * per_cu), 512, lds, stream>>>(a);
  return (int)hipGetLastError();
}

// bf16 blocks of 8 chunks (152 registers) leave a CU to one workgroup: where its LDS does that anyway
template <bool F8, int MB, int EPI, bool NORM>
static int stream_u(const StreamArgs& a, hipStream_t stream) {
  const size_t lds = kRedBytes + (size_t)a.M * (a.K + 8) * 2;
  const int per_cu = lds <= kTwoLds ? 2 : 1;
  return a.K % 4096 == 0 && (F8 || per_cu == 1) ? stream_launch<F8, MB, EPI, NORM, 8>(a, per_cu, lds, stream)
                                                : stream_launch<F8, MB, EPI, NORM, 4>(a, per_cu, lds, stream);
}

template <bool F8, int EPI>
static int stream_rows(const StreamArgs& a, bool norm, hipStream_t stream) {
  if (norm) return stream_u<F8, 1, EPI, true>(a, stream);
  return a.M <= 16 ? stream_u<F8, 1, EPI, false>(a, stream) : stream_u<F8, 2, EPI, false>(a, stream);
}

}  // namespace mx

using namespace mx;

// Whether mx_stream_gemm takes M rows of K: X and the partial sums in 160 KB of LDS, whole blocks a wave.
extern "C" int mx_stream_ok(int M, int K, int norm) {
  const int64_t lds = kRedBytes + (int64_t)M * (K + 8) * 2;
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
