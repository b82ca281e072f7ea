// Fused decode GEMMs of the recurrent / chunked-attention decoders on the weight-streaming core
// (skinny_core.h), M <= 16 bf16 rows, Y = X . W^T:
//   prologues (the rows are rebuilt in LDS by every workgroup; M K <= 16384 for the norm, 32768 for PolyNorm):
//     kProNorm : X = group_norm(h + delta) * gamma, f32 residual; workgroup 0 stores h + delta;
//     kProPoly : X = poly_norm(z), the feed-forward activation ahead of the down projection;
//   epilogues:
//     kEpiPlain: Y bf16;
//     kEpiGru  : W = [z; u; g]: a workgroup's 16 weight rows are 4 channels of each (a quarter
//                idle), so the wave that sums the K parts holds z, u and g of its channels, advances
//                the f32 state and writes S * silu(g);
//     kEpiConv : W = [q; k; v; gate]: the causal convolution against the ring of earlier projected
//                values, the pair rotation and the KV-cache append on the 4 consecutive channels a
//                lane holds; the gate's channels go out as they are.
// Each replaces two to four launches of a decode step.
#include "hybrid_fuse.h"
#include "skinny_core.h"

extern "C" int mx_stream_gru(const uint16_t* x, int64_t ldx, const uint16_t* delta, int64_t ldd, const float* h, const float* gamma,
                             float* h_out, int groups, float eps, const uint16_t* w, int64_t ldw, const float* bias,
                             const int32_t* slots, float* state, uint16_t* y, int M, int W, int K, hipStream_t stream);
extern "C" int mx_stream_conv(const uint16_t* x, int64_t ldx, const uint16_t* delta, int64_t ldd, const float* h,
                              const float* gamma, float* h_out, int groups, float eps, const uint16_t* w, int64_t ldw,
                              const mx::ConvRope* pa, const int32_t* pos, const int32_t* slots, uint16_t* gate, int M, int K,
                              hipStream_t stream);

namespace mx {

enum { kProNone, kProNorm, kProPoly };
enum { kEpiPlain, kEpiGru, kEpiConv };

constexpr int kHsMaxChunks = 4;  // 8-element pieces per thread: M K <= 512 * 8 * 4

// rows of h (+ delta), normalised, into xs [M, K]: piece sums of squares, then one wave per (row, part)
__device__ __forceinline__ void hs_norm_rows(const HsNorm& na, int M, int K, uint16_t* xs, float* psum, float* rs) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int np = M * K / 8, gs = K / na.groups, per = gs / 8;
  float v[kHsMaxChunks][8];
#pragma unroll
  for (int i = 0; i < kHsMaxChunks; ++i) {
    const int p = i * 512 + tid;
    if (p < np) {
      const int m = p / (K / 8), c = (p % (K / 8)) * 8;
      ldv<8>(na.h + (int64_t)m * K + c, v[i]);
      if (na.delta) {
        float d[8];
        ldv<8>(na.delta + (int64_t)m * na.ldd + c, d);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] += d[j];
        if (blockIdx.x == 0) stv<8>(na.h_out + (int64_t)m * K + c, v[i]);
      }
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += v[i][j] * v[i][j];
      psum[p] = ss;
    }
  }
  __syncthreads();
  for (int u = w; u < M * na.groups; u += kSkWaves) {  // part u: pieces [u per, (u + 1) per)
    float ss = 0.f;
    for (int i = lane; i < per; i += 64) ss += psum[u * per + i];
    ss = wave_sum(ss);
    if (lane == 0) rs[u] = 1.f / sqrtf(ss / (float)gs + na.eps);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kHsMaxChunks; ++i) {
    const int p = i * 512 + tid;
    if (p < np) {
      const int c = (p % (K / 8)) * 8;
      const float r = rs[p / per];
      float g[8], o[8];
      ldv<8>(na.gamma + c, g);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = v[i][j] * r * g[j];
      stv<8>(xs + (int64_t)p * 8, o);
    }
  }
  __syncthreads();
}

// poly_norm of the rows z [M, K] into xs [M, K]
__device__ __forceinline__ void hs_poly_rows(const uint16_t* __restrict__ z, int64_t ldz, const HsPoly& pp, int M, int K,
                                             uint16_t* xs, float (*red)[kSkWaves]) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int m = 0; m < M; ++m) {
    float s[3] = {0.f, 0.f, 0.f};
    for (int c = tid * 8; c < K; c += 4096) {
      const u16x8 zv = *reinterpret_cast<const u16x8*>(z + (int64_t)m * ldz + c);
      *reinterpret_cast<u16x8*>(xs + (int64_t)m * K + c) = zv;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float v = bf2f(zv[j]), q = v * v;
        s[0] += q;
        s[1] += q * q;
        s[2] += q * q * q;
      }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      s[k] = wave_sum(s[k]);
      if (lane == 0) red[k][w] = s[k];
    }
    __syncthreads();
    float kf[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      float t = 0.f;
#pragma unroll
      for (int i = 0; i < kSkWaves; ++i) t += red[k][i];
      kf[k] = pp.coef[k] / sqrtf(t / (float)K + pp.eps);
    }
    const float e = pp.coef[3];
    for (int c = tid * 8; c < K; c += 4096) {  // the pieces this thread stored
      u16x8* px = reinterpret_cast<u16x8*>(xs + (int64_t)m * K + c);
      const u16x8 zv = *px;
      u16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float v = bf2f(zv[j]);
        o[j] = f2bf(((kf[2] * v + kf[1]) * v + kf[0]) * v + e);
      }
      *px = o;
    }
    __syncthreads();
  }
}

template <int PRO, int EPI, int TB, int KP>
__global__ void __launch_bounds__(512) hybrid_skinny_kernel(const uint16_t* __restrict__ X, int64_t ldx,
                                                            const uint16_t* __restrict__ W, int64_t ldw,
                                                            uint16_t* __restrict__ Y, int64_t ldy, int M, int K,
                                                            HsNorm na, HsPoly pp, HsGru gr, HsConv cv) {
  typedef SkSum<TB, 1, KP> Sum;
  constexpr int RB = Sum::RB;
  __shared__ f32x4 red[Sum::PLACES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int blk = blockIdx.x, kq = K / KP, nit = kq / 64;
  const int64_t k0 = (int64_t)sk_part<KP>(w) * kq + sk_lane_k(c, g);
  const uint16_t* wrow[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int ch = 8 * sk_half<KP>(w, rb) + (c & 7);
    wrow[rb] = W + (EPI == kEpiGru ? hs_gru_row(blk, ch, gr.W) : (int64_t)blk * 16 + ch) * ldw + k0;
  }
  const uint16_t* xr[TB];
  u16x8 apre[sk_unr(1)][RB];
  if constexpr (PRO != kProNone) {
    extern __shared__ __attribute__((aligned(16))) uint16_t xs[];  // [M, K], then the norm's scratch
    sk_prefetch<1>(wrow, nit, apre);
    if constexpr (PRO == kProNorm) {
      float* psum = reinterpret_cast<float*>(xs + (int64_t)M * K);
      hs_norm_rows(na, M, K, xs, psum, psum + M * K / 8);
    } else {
      __shared__ float pred[3][kSkWaves];
      hs_poly_rows(X, ldx, pp, M, K, xs, pred);
    }
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) xr[tb] = xs + (int64_t)min(8 * tb + (c & 7), M - 1) * K + k0;
  } else {
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) xr[tb] = X + (int64_t)min(8 * tb + (c & 7), M - 1) * ldx + k0;
  }
  f32x4 acc[RB][TB];
  sk_stream<TB, 1, PRO != kProNone>(wrow, xr, nit, apre, acc);
  const Sum sum{red};
  sum.put(w, c, g, acc);
  __syncthreads();
  if (w == 0) {
    const f32x4 s = sum.get(c, g, 0, 0);
    if constexpr (EPI == kEpiGru) {
      hs_gru_store(s, lane, M, blk, gr, Y);
    } else if constexpr (EPI == kEpiConv) {
      hs_conv_store(s, blk * 16 + 4 * g, c, M, cv);
    } else if (c < M) {
      u16x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = f2bf(s[i]);
      *reinterpret_cast<u16x4*>(Y + (int64_t)c * ldy + blk * 16 + 4 * g) = o;
    }
  }
}

struct HsRun {
  int groups;
  size_t lds;
  const uint16_t* x;
  int64_t ldx;
  const uint16_t* w;
  int64_t ldw;
  uint16_t* y;
  int64_t ldy;
  int M, K;
};
template <int PRO, int EPI, int ROWS = 16>
static void hs_launch(const HsRun& r, const HsNorm& na, const HsPoly& pp, const HsGru& gr, const HsConv& cv, hipStream_t stream) {
  constexpr int TB = ROWS > 8 ? 2 : 1;
#define HS_RUN(TBV, KP) \
  hybrid_skinny_kernel<PRO, EPI, TBV, KP><<<r.groups, 512, r.lds, stream>>>(r.x, r.ldx, r.w, r.ldw, r.y, r.ldy, r.M, r.K, na, pp, gr, cv)
  if (sk_parts(r.M, r.K) == 4) {
    if (r.M <= 8) HS_RUN(1, 4); else HS_RUN(TB, 4);
  } else {
    if (r.M <= 8) HS_RUN(1, 8); else HS_RUN(TB, 8);
  }
#undef HS_RUN
}

static int hs_check(const uint16_t* x, int64_t ldx, int64_t ldw, int M, int K, int N) {
  if (M > 16 || K % 512 || ldw % 8 || ldw < K || N <= 0) return -1;
  if (x && (ldx % 8 || ldx < K)) return -1;
  return 0;
}
static int hs_norm_check(const HsNorm& na, int M, int K) {
  if (na.groups <= 0 || K % na.groups || (K / na.groups) % 8 || (int64_t)M * K > 512 * 8 * kHsMaxChunks ||
      M * na.groups > 512 || (na.delta && (na.ldd % 8 || na.ldd < K || !na.h_out)))
    return -1;
  return 0;
}
static size_t hs_norm_lds(int M, int K, int groups) { return (size_t)M * K * 2 + (size_t)M * K / 2 + (size_t)M * groups * 4; }

}  // namespace mx

using namespace mx;

// Common to the three: norm != 0: X = group_norm(h + delta) * gamma (x unused), else X = x bf16 rows.

// y [M, N] bf16
extern "C" int mx_hs_norm_gemm(const uint16_t* delta, int64_t ldd, const float* h, const float* gamma, float* h_out,
                               int groups, float eps, const uint16_t* w, int64_t ldw, uint16_t* y, int64_t ldy, int M,
                               int N, int K, hipStream_t stream) {
  if (M <= 0) return 0;
  const HsNorm na{delta, ldd, h, gamma, h_out, groups, eps};
  if (hs_check(nullptr, 0, ldw, M, K, N) || hs_norm_check(na, M, K) || N % 16 || ldy % 4 || ldy < N) return -1;
  hs_launch<kProNorm, kEpiPlain>({N / 16, hs_norm_lds(M, K, groups), nullptr, 0, w, ldw, y, ldy, M, K}, na, {}, {}, {}, stream);
  return (int)hipGetLastError();
}

// y [M, N] = poly_norm(z) . w^T, up to 8 rows
extern "C" int mx_hs_poly_gemm(const uint16_t* z, int64_t ldz, const float* coef, float eps, const uint16_t* w,
                               int64_t ldw, uint16_t* y, int64_t ldy, int M, int N, int K, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 8 || hs_check(z, ldz, ldw, M, K, N) || (int64_t)M * K > 32768 || N % 16 || ldy % 4 || ldy < N) return -1;
  hs_launch<kProPoly, kEpiPlain, 8>({N / 16, (size_t)M * K * 2, z, ldz, w, ldw, y, ldy, M, K}, {}, HsPoly{coef, eps}, {}, {}, stream);
  return (int)hipGetLastError();
}

// w [3 W, K] -> y [M, W] = S * silu(g), state advanced
extern "C" int mx_hs_gru_gemm(const uint16_t* x, int64_t ldx, int norm, const uint16_t* delta, int64_t ldd,
                              const float* h, const float* gamma, float* h_out, int groups, float eps,
                              const uint16_t* w, int64_t ldw, const float* bias, const int32_t* slots, float* state,
                              uint16_t* y, int M, int W, int K, hipStream_t stream) {
  if (M <= 0) return 0;
  const int rc = mx_stream_gru(x, ldx, delta, ldd, norm ? h : nullptr, gamma, h_out, groups, eps, w, ldw, bias, slots, state, y, M, W, K, stream);
  if (rc != -1) return rc;
  const HsNorm na{delta, ldd, h, gamma, h_out, groups, eps};
  if (hs_check(norm ? nullptr : x, ldx, ldw, M, K, W) || W % 4 || (norm && hs_norm_check(na, M, K)) || (!norm && !x))
    return -1;
  const HsGru gr{bias, slots, state, W};
  if (norm)
    hs_launch<kProNorm, kEpiGru>({W / 4, hs_norm_lds(M, K, groups), nullptr, 0, w, ldw, y, W, M, K}, na, {}, gr, {}, stream);
  else
    hs_launch<kProNone, kEpiGru>({W / 4, 0, x, ldx, w, ldw, y, W, M, K}, {}, {}, gr, {}, stream);
  return (int)hipGetLastError();
}

// w [C + H E, K] -> q [M, H, Dp] (in a), k / v cache rows, ring, gate [M, H E]
extern "C" int mx_hs_conv_gemm(const uint16_t* x, int64_t ldx, int norm, const uint16_t* delta, int64_t ldd,
                               const float* h, const float* gamma, float* h_out, int groups, float eps,
                               const uint16_t* w, int64_t ldw, const ConvRope* pa, const int32_t* pos,
                               const int32_t* slots, uint16_t* gate, int M, int K, hipStream_t stream) {
  if (M <= 0) return 0;
  const int rc = mx_stream_conv(x, ldx, delta, ldd, norm ? h : nullptr, gamma, h_out, groups, eps, w, ldw, pa, pos, slots, gate, M, K, stream);
  if (rc != -1) return rc;
  const HsNorm na{delta, ldd, h, gamma, h_out, groups, eps};
  const ConvRope& a = *pa;
  const int N = hs_conv_rows(a);
  if (hs_check(norm ? nullptr : x, ldx, ldw, M, K, N) || (norm && hs_norm_check(na, M, K)) || (!norm && !x)) return -1;
  const HsConv cv{a, pos, slots, gate};
  if (norm)
    hs_launch<kProNorm, kEpiConv>({N / 16, hs_norm_lds(M, K, groups), nullptr, 0, w, ldw, nullptr, 0, M, K}, na, {}, {}, cv, stream);
  else
    hs_launch<kProNone, kEpiConv>({N / 16, 0, x, ldx, w, ldw, nullptr, 0, M, K}, {}, {}, {}, cv, stream);
  return (int)hipGetLastError();
}
