// Post-normed sublayers on an f32 residual stream, for gfx950:
//   * post_norm   : h += rms(src) * w and the activation copy of h, where src is a sublayer's output, the
//                   weighted sum of a token's expert outputs (+ the shared expert's), or - without the
//                   add - an embedding row;
//   * side_act    : gelu_tanh(z) times the token's row of a second embedding;
//   * post_dots   : decode rows, the residual step with the products that read the new h next: the router's
//                   logits, or the second embedding's gate (with its activation);
//   * post_side   : decode rows, the second embedding's projection with the residual step behind it;
//   * clipped_glu : min(g, L) sigmoid(1.702 min(g, L)) (clamp(u, -L, L) + 1).
// Storage type T: bf16 (uint16_t) or float; every reduction and product is f32.
#include "hybrid.h"
#include "sublayer.h"

namespace mx {

// one row per TPU threads, held in registers (at most 16 elements a thread)
template <typename T, int MODE, int TPU, int VEC>
__global__ void __launch_bounds__(TPU < 256 ? 256 : TPU) post_norm_kernel(PostNorm a) {
  constexpr int ITERS = 16 / VEC;
  __shared__ float scratch[16];
  const int64_t r = TPU < 256 ? (int64_t)blockIdx.x * (256 / TPU) + threadIdx.x / TPU : (int64_t)blockIdx.x;
  const bool on = r < a.T;
  const int64_t row = on ? r : 0;
  const int t = threadIdx.x % TPU;
  const T* src = reinterpret_cast<const T*>(a.src);
  const T* sp = src + row * a.lds;
  if constexpr (MODE == PostNorm::kEmbed) {
    int64_t id = a.ids[row];
    id = id < 0 ? 0 : (id >= a.V ? a.V - 1 : id);  // ids are checked on the host; stays in the table either way
    sp = src + id * a.lds;
  }
  float v[ITERS][VEC];
  float ss = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * TPU + t) * VEC;
    if (on && c < a.W) {
      if constexpr (MODE == PostNorm::kMix) {
        if (a.shared) {
          ldv<VEC>(reinterpret_cast<const T*>(a.shared) + row * a.ldsh + c, v[it]);
        } else {
#pragma unroll
          for (int j = 0; j < VEC; ++j) v[it][j] = 0.f;
        }
#pragma unroll 4
        for (int k = 0; k < a.top; ++k) {
          const int64_t pr = row * a.top + k;
          const float wt = a.wts[pr];
          float e[VEC];
          ldv<VEC>(src + (a.inv ? a.inv[pr] : pr) * a.lds + c, e);
#pragma unroll
          for (int j = 0; j < VEC; ++j) v[it][j] += wt * e[j];
        }
      } else {
        ldv<VEC>(sp + c, v[it]);
      }
#pragma unroll
      for (int j = 0; j < VEC; ++j) ss += v[it][j] * v[it][j];
    }
  }
  ss = TPU == 64 ? wave_sum(ss) : block_sum(ss, scratch);
  const float rs = 1.f / sqrtf(ss / (float)a.W + a.eps);
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * TPU + t) * VEC;
    if (on && c < a.W) {
      float g[VEC], o[VEC];
      ldv<VEC>(a.w + c, g);
      float* hp = a.h + row * a.W + c;
      if constexpr (MODE == PostNorm::kEmbed) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) o[j] = v[it][j] * rs * g[j];
      } else {
        ldv<VEC>(hp, o);
#pragma unroll
        for (int j = 0; j < VEC; ++j) o[j] += v[it][j] * rs * g[j];
      }
      stv<VEC>(hp, o);
      if (a.y) stv<VEC>(reinterpret_cast<T*>(a.y) + row * a.W + c, o);
    }
  }
}

// decode rows (W <= 4096): a workgroup rebuilds the row's new h and takes kDotRows rows of the matrix; the first
// one stores h.  The matrix rows are requested ahead of the norm.
constexpr int kDotRows = 4;
template <int MODE, bool SIDE>
__global__ void __launch_bounds__(256) post_dots_kernel(PostDots a) {
  __shared__ float scratch[16];
  __shared__ float part[4][kDotRows];
  const int64_t row = blockIdx.y;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6, r0 = blockIdx.x * kDotRows, W = a.p.W;
  const uint16_t* src = reinterpret_cast<const uint16_t*>(a.p.src);
  float v[2][8], o[2][8], g[2][8], ss = 0.f;
  u16x8 m[kDotRows][2];
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int c = (it * 256 + t) * 8;
    if (c < W) {
#pragma unroll
      for (int r = 0; r < kDotRows; ++r) m[r][it] = *reinterpret_cast<const u16x8*>(a.m + (int64_t)min(r0 + r, a.R - 1) * W + c);
      if constexpr (MODE == PostNorm::kMix) {
        if (a.p.shared) {
          ldv<8>(reinterpret_cast<const uint16_t*>(a.p.shared) + row * a.p.ldsh + c, v[it]);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[it][j] = 0.f;
        }
#pragma unroll 4
        for (int k = 0; k < a.p.top; ++k) {
          const int64_t pr = row * a.p.top + k;
          const float wt = a.p.wts[pr];
          float e[8];
          ldv<8>(src + pr * a.p.lds + c, e);
#pragma unroll
          for (int j = 0; j < 8; ++j) v[it][j] += wt * e[j];
        }
      } else {
        ldv<8>(src + row * a.p.lds + c, v[it]);
      }
      ldv<8>(a.p.w + c, g[it]);
      ldv<8>(a.p.h + row * W + c, o[it]);
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += v[it][j] * v[it][j];
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // the matrix rows' loads stay ahead of the reduction
  ss = block_sum(ss, scratch);
  const float rs = 1.f / sqrtf(ss / (float)W + a.p.eps);
  float s[kDotRows] = {};
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int c = (it * 256 + t) * 8;
    if (c < W) {
#pragma unroll
      for (int j = 0; j < 8; ++j) o[it][j] += v[it][j] * rs * g[it][j];
      if (blockIdx.x == 0) {
        stv<8>(a.ho + row * W + c, o[it]);
        if (a.p.y) stv<8>(reinterpret_cast<uint16_t*>(a.p.y) + row * W + c, o[it]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = bf2f(f2bf(o[it][j]));
#pragma unroll
        for (int r = 0; r < kDotRows; ++r) s[r] += x * bf2f(m[r][it][j]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kDotRows; ++r) {
    s[r] = wave_sum(s[r]);
    if (lane == 0) part[wv][r] = s[r];
  }
  __syncthreads();
  const int ch = r0 + t;
  if (t >= kDotRows || ch >= a.R) return;
  const float z = part[0][t] + part[1][t] + part[2][t] + part[3][t];
  if constexpr (SIDE) {
    int64_t id = a.ids[row];
    id = id < 0 ? 0 : (id >= a.V ? a.V - 1 : id);
    a.side[row * a.R + ch] = f2bf(gelu_tanh_t<uint16_t>(bf2f(f2bf(z))) * bf2f(a.emb[id * a.lde + ch]));
  } else {
    a.logits[row * a.R + ch] = z;
  }
}

// decode rows (W <= 4096): h += rms(P g) * w and its copy, P [W, R] the second embedding's projection, g [T, R] its gated
// rows.  The product and the norm behind it were two launches that wait for each other, 4.7 us each; a workgroup of 16 waves
// reads P itself (256 KB at W 2048, 8.5 us).  R / 8 lanes take a row of P, whose products go to LDS rounded as the product's
// were.  The row's sum of squares is that of these products: as g^T (P^T P) g out of a matrix laid out before, several workgroups
// could share a row (65 us less in a step of 32 sequences, 1B size), but terms cancel (two columns alike to 1 in 256: the norm
// off by 2 to 4 %), and weights written later would meet the norm of the old ones.
template <int R>
__global__ void __launch_bounds__(1024) post_side_kernel(PostNorm a, const uint16_t* __restrict__ gs,
                                                         const uint16_t* __restrict__ P) {
  constexpr int LPR = R / 8, RPI = 64 / LPR, U = 16;
  __shared__ float scratch[16];
  __shared__ __attribute__((aligned(16))) float ybuf[4096];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6, W = a.W, c = min(4 * t, W - 4);
  const int64_t row = blockIdx.x;
  const u16x8 gr = *reinterpret_cast<const u16x8*>(gs + row * R + 8 * (lane % LPR));
  float* hp = a.h + row * W + c;
  float o[4], w[4], v[4], g[8];
  ldv<4>(hp, o);
  ldv<4>(a.w + c, w);
#pragma unroll
  for (int j = 0; j < 8; ++j) g[j] = bf2f(gr[j]);
  const int per = W / 16, n = per / RPI;  // rows of P a wave, loads of RPI of them
  const int first = wv * per + lane / LPR;
  const uint16_t* p0 = P + (int64_t)first * R + 8 * (lane % LPR);
  for (int i0 = 0; i0 < n; i0 += U) {
    u16x8 m[U];
#pragma unroll
    for (int u = 0; u < U; ++u) m[u] = *reinterpret_cast<const u16x8*>(p0 + min(i0 + u, n - 1) * (RPI * R));
    __builtin_amdgcn_sched_barrier(0);  // every load is in flight before the first product waits
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) s += g[j] * bf2f(m[u][j]);
#define MX_ADD_LANES(CTRL) \
  s += __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(s), CTRL, 0xF, 0xF, true))
      MX_ADD_LANES(0xB1);                           // lane ^ 1
      MX_ADD_LANES(0x4E);                           // lane ^ 2
      if constexpr (LPR >= 8) MX_ADD_LANES(0x141);  // the other quad of eight
      if constexpr (LPR >= 16) MX_ADD_LANES(0x140); // the other half of sixteen
#undef MX_ADD_LANES
      if (i0 + u < n && lane % LPR == 0) ybuf[first + (i0 + u) * RPI] = bf2f(f2bf(s));
    }
  }
  __syncthreads();
  float ss = 0.f;
  const bool on = 4 * t < W;
  ldv<4>(ybuf + c, v);
#pragma unroll
  for (int j = 0; j < 4; ++j) ss += on ? v[j] * v[j] : 0.f;
  ss = block_sum(ss, scratch);
  if (!on) return;
  const float rs = 1.f / sqrtf(ss / (float)W + a.eps);
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] += v[j] * rs * w[j];
  stv<4>(hp, o);
  stv<4>(reinterpret_cast<uint16_t*>(a.y) + row * W + c, o);
}

template <typename T, int VEC>
__global__ void __launch_bounds__(256) side_act_kernel(const T* __restrict__ z, int64_t ldz, const T* __restrict__ emb,
                                                       int64_t lde, const int64_t* __restrict__ ids, int V,
                                                       T* __restrict__ y, int64_t n, int dim) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int nv = dim / VEC;
  const int64_t row = i / nv;
  const int c = (int)(i % nv) * VEC;
  int64_t id = ids[row];
  id = id < 0 ? 0 : (id >= V ? V - 1 : id);
  float a[VEC], e[VEC];
  ldv<VEC>(z + row * ldz + c, a);
  ldv<VEC>(emb + id * lde + c, e);
#pragma unroll
  for (int j = 0; j < VEC; ++j) a[j] = gelu_tanh_t<T>(a[j]) * e[j];
  stv<VEC>(y + row * dim + c, a);
}

template <typename T, int VEC>
__global__ void __launch_bounds__(256) clipped_glu_kernel(const T* __restrict__ z, int64_t ldz, T* __restrict__ y,
                                                          int64_t n, int F, float limit) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int nv = F / VEC;
  const int64_t row = i / nv;
  const int c = (int)(i % nv) * VEC;
  float g[VEC], u[VEC];
  ldv<VEC>(z + row * ldz + c, g);
  ldv<VEC>(z + row * ldz + F + c, u);
#pragma unroll
  for (int j = 0; j < VEC; ++j) g[j] = clipped_glu<T>(g[j], u[j], limit);
  stv<VEC>(y + row * F + c, g);
}

}  // namespace mx

using namespace mx;

static bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

extern "C" int mx_post_norm(const PostNorm* pa, int f32, hipStream_t stream) {
  const PostNorm& a = *pa;
  if (a.T <= 0) return 0;
  if (a.W <= 0 || a.W > 16384 || !a.src || !a.h || !a.w || (a.mode == PostNorm::kEmbed && (!a.ids || a.V <= 0)) ||
      (a.mode == PostNorm::kMix && (!a.wts || a.top <= 0)))
    return -1;
  const bool v4 = a.W % 4 == 0 && a.lds % 4 == 0 && (!a.shared || a.ldsh % 4 == 0) && al16(a.src) && al16(a.h) &&
                  al16(a.w) && al16(a.shared) && al16(a.y);
#define PN(TT, MM, TPU, VV)                                                                                 \
  post_norm_kernel<TT, MM, TPU, VV>                                                                         \
      <<<(unsigned)(TPU == 64 ? (a.T + 3) / 4 : a.T), TPU == 64 ? 256 : TPU, 0, stream>>>(a)
#define PNV(TT, MM)                                                                                         \
  if (v4) { if (a.W <= 512) PN(TT, MM, 64, 4); else if (a.W <= 4096) PN(TT, MM, 256, 4); else PN(TT, MM, 1024, 4); } \
  else { if (a.W <= 1024) PN(TT, MM, 64, 1); else if (a.W <= 4096) PN(TT, MM, 256, 1); else PN(TT, MM, 1024, 1); }
#define PNM(TT)                                                                                             \
  if (a.mode == PostNorm::kRows) { PNV(TT, PostNorm::kRows) }                                               \
  else if (a.mode == PostNorm::kEmbed) { PNV(TT, PostNorm::kEmbed) }                                        \
  else { PNV(TT, PostNorm::kMix) }
  if (f32) { PNM(float) } else { PNM(uint16_t) }
#undef PNM
#undef PNV
#undef PN
  return (int)hipGetLastError();
}

// bf16 rows; -1 (nothing launched): sizes it does not take
extern "C" int mx_post_dots(const PostDots* pa, hipStream_t stream) {
  const PostDots& a = *pa;
  const PostNorm& p = a.p;
  if (p.T <= 0) return 0;
  if (p.T > 65535 || p.W <= 0 || p.W > 4096 || p.W % 8 || p.lds % 8 || (p.shared && p.ldsh % 8) || a.R <= 0 || !a.ho ||
      (p.mode != PostNorm::kRows && (p.mode != PostNorm::kMix || p.inv || !p.wts || p.top <= 0)) || !al16(p.src) ||
      !al16(p.shared) || !al16(p.h) || !al16(p.w) || !al16(p.y) || !al16(a.ho) || !al16(a.m) || (!a.side && !a.logits) ||
      (a.side && (!a.emb || !a.ids || a.V <= 0)))
    return -1;
  const dim3 g((a.R + kDotRows - 1) / kDotRows, (unsigned)p.T);
  if (p.mode == PostNorm::kRows) {
    if (a.side) post_dots_kernel<PostNorm::kRows, true><<<g, 256, 0, stream>>>(a);
    else post_dots_kernel<PostNorm::kRows, false><<<g, 256, 0, stream>>>(a);
  } else {
    if (a.side) post_dots_kernel<PostNorm::kMix, true><<<g, 256, 0, stream>>>(a);
    else post_dots_kernel<PostNorm::kMix, false><<<g, 256, 0, stream>>>(a);
  }
  return (int)hipGetLastError();
}

// bf16 rows g [T, R] and P [W, R], both dense; -1 (nothing launched): sizes it does not take
extern "C" int mx_post_side(const PostNorm* pa, const uint16_t* g, const uint16_t* P, int R, hipStream_t stream) {
  const PostNorm& a = *pa;
  if (a.T <= 0) return 0;
  if (a.T > 65535 || (R != 32 && R != 64 && R != 128) || a.W <= 0 || a.W > 4096 || a.W % (16 * 512 / R) || !a.h || !a.w || !a.y ||
      !al16(a.h) || !al16(a.w) || !al16(a.y) || !al16(g) || !al16(P))
    return -1;
#define PS(RR) post_side_kernel<RR><<<(unsigned)a.T, 1024, 0, stream>>>(a, g, P)
  if (R == 32) PS(32);
  else if (R == 64) PS(64);
  else PS(128);
#undef PS
  return (int)hipGetLastError();
}

extern "C" int mx_side_act(const void* z, int64_t ldz, const void* emb, int64_t lde, const int64_t* ids, int V, void* y,
                           int f32, int64_t T, int dim, hipStream_t stream) {
  if (T <= 0) return 0;
  if (dim <= 0 || V <= 0) return -1;
  const bool v4 = dim % 4 == 0 && ldz % 4 == 0 && lde % 4 == 0 && al16(z) && ((uintptr_t)emb & 7) == 0 && (!f32 || al16(emb));
  const int64_t n = T * (dim / (v4 ? 4 : 1));
  const unsigned g = (unsigned)((n + 255) / 256);
#define SA(TT, VV) side_act_kernel<TT, VV><<<g, 256, 0, stream>>>((const TT*)z, ldz, (const TT*)emb, lde, ids, V, (TT*)y, n, dim)
  if (f32) { if (v4) SA(float, 4); else SA(float, 1); }
  else { if (v4) SA(uint16_t, 4); else SA(uint16_t, 1); }
#undef SA
  return (int)hipGetLastError();
}

extern "C" int mx_clipped_glu(const void* z, int64_t ldz, void* y, int f32, int64_t T, int F, float limit,
                              hipStream_t stream) {
  if (T <= 0) return 0;
  if (F <= 0) return -1;
  const int vec = F % 8 == 0 && ldz % 8 == 0 && al16(z) && !f32 ? 8 : F % 4 == 0 && ldz % 4 == 0 && al16(z) ? 4 : 1;
  const int64_t n = T * (F / vec);
  const unsigned g = (unsigned)((n + 255) / 256);
#define CG(TT, VV) clipped_glu_kernel<TT, VV><<<g, 256, 0, stream>>>((const TT*)z, ldz, (TT*)y, n, F, limit)
  if (f32) { if (vec == 4) CG(float, 4); else CG(float, 1); }
  else { if (vec == 8) CG(uint16_t, 8); else if (vec == 4) CG(uint16_t, 4); else CG(uint16_t, 1); }
#undef CG
  return (int)hipGetLastError();
}
