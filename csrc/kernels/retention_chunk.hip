// Retention over whole prompts in chunks, f32 matrix cores (gfx950), bf16 or f32 storage (bf16 heads of 64 and 128, rotated
// whole: ends and out are retention_mfma.hip's, at half of the time).  Everything that
// enters the recurrence - rotated q and k, scores, decay powers, state - is f32, as in retention_seq.
// Three launches over runs of kRetChunk rows of one sequence:
//   ends  : U = sum_j decay^(n-1-j) k_j v_j^T of every run;
//   carry : the state ahead of every run (in place of U) and the sequence's last state;
//   out   : 128 rows at a time: decay^(i+1) q_i S_run + sum_(j <= i) decay^(i-j) (q_i . k_j) v_j, then the
//           norm per head and the gate.
// Powers of the decays come from a table [H, kRetChunk + 1].
#include "hybrid.h"
#include "sublayer.h"

namespace mx {

constexpr int kRetChunk = 256, kRetKeys = 32;

__device__ __forceinline__ f32x4 mfma4(float a, float b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// k rows [r0, r0 + n) at column `col` (width D) into dst [R][DP + 4], rotated by halves and times scale(row);
// rows past n and columns past D are zero
template <typename T, int R, int DP, typename F>
__device__ __forceinline__ void ret_stage_k(const RetentionChunks& a, int64_t r0, int n, int p0, int64_t col, F scale,
                                            float* dst) {
  const int D = a.D, rd = a.rd, half = rd / 2;
  const T* x = reinterpret_cast<const T*>(a.x) + r0 * a.ldx + col;
  if (a.v4) {  // D, half and every offset whole groups of four: a thread turns four pairs
    const int gr = half / 4, gp = (DP - rd) / 4;  // groups of pairs, of dims that pass
    for (int i = threadIdx.x; i < R * (gr + gp); i += blockDim.x) {
      const int r = i / (gr + gp), q = i - r * (gr + gp);
      const bool rot = q < gr, on = r < n;
      const int d = rot ? q * 4 : rd + (q - gr) * 4;
      float u[4] = {0.f, 0.f, 0.f, 0.f}, v[4] = {0.f, 0.f, 0.f, 0.f};
      if (on && d < D) {
        const T* xr = x + (int64_t)r * a.ldx;
        const float sc = scale(r);
        ldv<4>(xr + d, u);
        if (rot) {
          float c[4], s[4];
          ldv<4>(xr + d + half, v);
          ldv<4>(a.cosb + (int64_t)(p0 + r) * half + d, c);
          ldv<4>(a.sinb + (int64_t)(p0 + r) * half + d, s);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float x0 = u[j], x1 = v[j];
            u[j] = (x0 * c[j] - x1 * s[j]) * sc;
            v[j] = (x1 * c[j] + x0 * s[j]) * sc;
          }
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) u[j] *= sc;
        }
      }
      stv<4>(dst + r * (DP + 4) + d, u);
      if (rot) stv<4>(dst + r * (DP + 4) + d + half, v);
    }
    return;
  }
  for (int i = threadIdx.x; i < R * DP; i += blockDim.x) {
    const int r = i / DP, d = i % DP;
    float v = 0.f;
    if (r < n && d < D) {
      const T* xr = x + (int64_t)r * a.ldx;
      v = ld1(xr + d);
      if (d < rd) {
        const bool lo = d < half;
        const int64_t f = (int64_t)(p0 + r) * half + (lo ? d : d - half);
        const float o = ld1(xr + (lo ? d + half : d - half)), c = a.cosb[f], s = a.sinb[f];
        v = lo ? v * c - o * s : v * c + o * s;
      }
      v *= scale(r);
    }
    dst[r * (DP + 4) + d] = v;
  }
}

// four dims d .. d + 3 of a rotated q row at position p
template <typename T>
__device__ __forceinline__ f32x4 ret_q4(const RetentionChunks& a, const T* xr, int p, int d) {
  const int half = a.rd / 2;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  if (a.v4) {
    if (d >= a.D) return o;
    float v[4];
    ldv<4>(xr + d, v);
    if (d < a.rd) {
      const bool lo = d < half;
      const int64_t f = (int64_t)p * half + (lo ? d : d - half);
      float w[4], c[4], s[4];
      ldv<4>(xr + (lo ? d + half : d - half), w);
      ldv<4>(a.cosb + f, c);
      ldv<4>(a.sinb + f, s);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = lo ? v[j] * c[j] - w[j] * s[j] : v[j] * c[j] + w[j] * s[j];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = v[j];
    return o;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (d + j >= a.D) continue;
    float v = ld1(xr + d + j);
    if (d + j < a.rd) {
      const bool lo = d + j < half;
      const int e = lo ? d + j : d + j - half;
      const int64_t f = (int64_t)p * half + e;
      const float w = ld1(xr + (lo ? e + half : e));
      v = lo ? v * a.cosb[f] - w * a.sinb[f] : v * a.cosb[f] + w * a.sinb[f];
    }
    o[j] = v;
  }
  return o;
}

// rows [0, n) of src (row stride ld, width E from column e0) to dst [R][EP + 4], the rest zero: requested into
// registers, stored later, so that the requests of k and v are in flight together
template <typename T, int R, int EP, int NT>
struct RetRows {
  static constexpr int G = EP / 4, IT = (R * G + NT - 1) / NT;
  float v[IT][4];
  __device__ __forceinline__ void load(const T* src, int64_t ld, int n, int e0, int E, bool v4) {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int i = it * NT + threadIdx.x, r = i / G, e = e0 + (i % G) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[it][j] = 0.f;
      if (r < n && e < E) {  // (n <= R)
        if (v4) {
          ldv<4>(src + (int64_t)r * ld + e, v[it]);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (e + j < E) v[it][j] = ld1(src + (int64_t)r * ld + e + j);
        }
      }
    }
  }
  __device__ __forceinline__ void store(float* dst) const {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int i = it * NT + threadIdx.x, r = i / G, e = (i % G) * 4;
      if (r < R) stv<4>(dst + r * (EP + 4) + e, v[it]);
    }
  }
};

// acc[j] += x(k) b(k, 16 j + c) over the 16 N keys (or dims) k of a tile, four of them a step; the next step's
// row of b is read ahead of this one's products
template <int N, int EB, typename X>
__device__ __forceinline__ void ret_products(f32x4 (&acc)[EB], const float* b, int ldb, int g, int c, X x) {
  float v[2][EB];
  auto row = [&](int t, float(&d)[EB]) __attribute__((always_inline)) {
    const float* p = b + (16 * (t >> 2) + 4 * g + (t & 3)) * ldb + c;
#pragma unroll
    for (int j = 0; j < EB; ++j) d[j] = p[16 * j];
  };
  row(0, v[0]);
#pragma unroll
  for (int t = 0; t < 4 * N; ++t) {
    if (t + 1 < 4 * N) row(t + 1, v[(t + 1) & 1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < EB; ++j) acc[j] = mfma4(x(t >> 2, t & 3), v[t & 1][j], acc[j]);
  }
}

// ------------------------------------------------------------------ run sums
// wave w: 16-row blocks w, w + 4, ... of D, all EP columns of column block blockIdx.z
template <typename T, int DP, int EP>
__global__ void __launch_bounds__(256) retention_ends_kernel(RetentionChunks a) {
  constexpr int NB = DP / 64, EB = EP / 16, R = kRetKeys;
  __shared__ float ks[R * (DP + 4)], vs[R * (EP + 4)], pw[kRetChunk + 1];
  const int4 ch = reinterpret_cast<const int4*>(a.chunks)[blockIdx.y];  // (first row, rows, position, -)
  const int h = blockIdx.x, e0 = blockIdx.z * EP, w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4;
  for (int i = threadIdx.x; i <= kRetChunk; i += 256) pw[i] = a.pw[(int64_t)h * (kRetChunk + 1) + i];
  const float ksc = 1.f / sqrtf((float)a.D);
  const int64_t HD = (int64_t)a.H * a.D;
  f32x4 acc[NB][EB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < EB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < ch.y; j0 += R) {
    const int n = min(R, ch.y - j0);
    __syncthreads();
    RetRows<T, R, EP, 256> vr;
    vr.load(reinterpret_cast<const T*>(a.x) + (ch.x + j0) * a.ldx + 2 * HD + (int64_t)h * a.E, a.ldx, n, e0, a.E, a.v4);
    ret_stage_k<T, R, DP>(a, ch.x + j0, n, ch.z + j0, HD + (int64_t)h * a.D,
                          [&](int r) { return ksc * pw[ch.y - 1 - j0 - r]; }, ks);
    vr.store(vs);
    __syncthreads();
    auto row = [&](int t, float(&xk)[NB], float(&bv)[EB]) __attribute__((always_inline)) {
      const int key = 16 * (t >> 2) + 4 * g + (t & 3);
#pragma unroll
      for (int m = 0; m < NB; ++m) xk[m] = ks[key * (DP + 4) + 16 * (w + 4 * m) + c];
#pragma unroll
      for (int j = 0; j < EB; ++j) bv[j] = vs[key * (EP + 4) + 16 * j + c];
    };
    float xk[2][NB], bv[2][EB];
    row(0, xk[0], bv[0]);
#pragma unroll
    for (int t = 0; t < R / 4; ++t) {  // the next keys' values are read ahead of these products
      if (t + 1 < R / 4) row(t + 1, xk[(t + 1) & 1], bv[(t + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < NB; ++m)
#pragma unroll
        for (int j = 0; j < EB; ++j) acc[m][j] = mfma4(xk[t & 1][m], bv[t & 1][j], acc[m][j]);
    }
  }
  float* u = a.ws + ((int64_t)blockIdx.y * a.H + h) * a.D * a.E;
#pragma unroll
  for (int m = 0; m < NB; ++m)
#pragma unroll
    for (int j = 0; j < EB; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 16 * (w + 4 * m) + 4 * g + i, e = e0 + 16 * j + c;
        if (d < a.D && e < a.E) u[(int64_t)d * a.E + e] = acc[m][j][i];
      }
}

// ------------------------------------------------------------------ states ahead of the runs
__global__ void __launch_bounds__(256) retention_carry_kernel(RetentionChunks a) {
  const int4 sq = reinterpret_cast<const int4*>(a.seqs)[blockIdx.z];  // (first run, runs, slot or -1, -)
  const int h = blockIdx.y, n = a.D * a.E, i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float* pw = a.pw + (int64_t)h * (kRetChunk + 1);
  float S = 0.f;
  for (int c = 0; c < sq.y; ++c) {
    float* u = a.ws + ((int64_t)(sq.x + c) * a.H + h) * n + i;
    const float x = *u;
    *u = S;
    S = pw[reinterpret_cast<const int4*>(a.chunks)[sq.x + c].y] * S + x;
  }
  if (a.state && sq.z >= 0) a.state[((int64_t)sq.z * a.H + h) * n + i] = S;
}

// ------------------------------------------------------------------ outputs
// wave w: rows 16 w .. 16 w + 15 of the block
constexpr int kRetRows = 128;
template <typename T, int DP, int EP>
__global__ void __launch_bounds__(512, DP <= 128 && EP <= 128 ? 4 : 2) retention_out_kernel(RetentionChunks a) {
  constexpr int DS = DP / 16, EB = EP / 16, R = kRetKeys;
  __shared__ float ks[R * (DP + 4)], vs[R * (EP + 4)];  // a tile of k and v (or of the state)
  __shared__ float ps[8][16 * (R + 4)];
  __shared__ float pw[kRetChunk + 1];
  const int4 bl = reinterpret_cast<const int4*>(a.blocks)[blockIdx.y];  // (run, first row in it, -, -)
  const int4 ch = reinterpret_cast<const int4*>(a.chunks)[bl.x];
  const int h = blockIdx.x, i0 = bl.y, w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4, rows = min(kRetRows, ch.y - i0);
  for (int i = threadIdx.x; i <= kRetChunk; i += 512) pw[i] = a.pw[(int64_t)h * (kRetChunk + 1) + i];
  const float ksc = 1.f / sqrtf((float)a.D);
  const int64_t HD = (int64_t)a.H * a.D, HE = (int64_t)a.H * a.E;
  const T* x = reinterpret_cast<const T*>(a.x);

  f32x4 qf[DS];  // row c, dims 16 s + 4 g ..
  {
    const int qr = min(i0 + 16 * w + c, ch.y - 1);  // rows past the run are not stored
#pragma unroll
    for (int s = 0; s < DS; ++s)
      qf[s] = ret_q4<T>(a, x + (ch.x + qr) * a.ldx + (int64_t)h * a.D, ch.z + qr, 16 * s + 4 * g);
  }
  f32x4 acc[EB];
#pragma unroll
  for (int j = 0; j < EB; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (ch.z > 0) {  // a state ahead of this run
    const float* S = a.ws + ((int64_t)bl.x * a.H + h) * a.D * a.E;
    RetRows<float, R, EP, 512> sr;
    sr.load(S, a.E, min(R, a.D), 0, a.E, a.v4);
#pragma unroll
    for (int d0 = 0; d0 < DP; d0 += R) {
      __syncthreads();
      sr.store(vs);
      __syncthreads();
      if (d0 + R < DP) sr.load(S + (int64_t)(d0 + R) * a.E, a.E, min(R, a.D - d0 - R), 0, a.E, a.v4);
      ret_products<R / 16>(acc, vs, EP + 4, g, c, [&](int s, int i) { return qf[d0 / 16 + s][i]; });
    }
    __syncthreads();  // (pw is there also where no tile was)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float f = pw[min(i0 + 16 * w + 4 * g + i + 1, kRetChunk)];
#pragma unroll
      for (int j = 0; j < EB; ++j) acc[j][i] *= f;
    }
  }
  const int last = min(i0 + kRetRows, ch.y);
  for (int j0 = 0; j0 < last; j0 += R) {
    const int n = min(R, ch.y - j0);
    __syncthreads();
    RetRows<T, R, EP, 512> vr;
    vr.load(x + (ch.x + j0) * a.ldx + 2 * HD + (int64_t)h * a.E, a.ldx, n, 0, a.E, a.v4);
    ret_stage_k<T, R, DP>(a, ch.x + j0, n, ch.z + j0, HD + (int64_t)h * a.D, [&](int) { return ksc; }, ks);
    vr.store(vs);
    __syncthreads();
    const int top = i0 + 16 * w;  // this wave's first row: keys past its last one count for none
    if (j0 <= top + 15) {
      f32x4 s4[R / 16] = {}, k4[2][R / 16];
      auto row = [&](int s, f32x4(&d)[R / 16]) __attribute__((always_inline)) {
#pragma unroll
        for (int kb = 0; kb < R / 16; ++kb)
          d[kb] = *reinterpret_cast<const f32x4*>(ks + (16 * kb + c) * (DP + 4) + 16 * s + 4 * g);
      };
      row(0, k4[0]);
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        if (s + 1 < DS) row(s + 1, k4[(s + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int kb = 0; kb < R / 16; ++kb) s4[kb] = mfma4(qf[s][i], k4[s & 1][kb][i], s4[kb]);
      }
#pragma unroll
      for (int kb = 0; kb < R / 16; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int back = top + 4 * g + i - (j0 + 16 * kb + c);
          ps[w][(4 * g + i) * (R + 4) + 16 * kb + c] = back >= 0 ? s4[kb][i] * pw[min(back, kRetChunk)] : 0.f;
        }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wave reads its own scores back
      __builtin_amdgcn_wave_barrier();
      f32x4 p4[R / 16];
#pragma unroll
      for (int s = 0; s < R / 16; ++s) p4[s] = *reinterpret_cast<const f32x4*>(&ps[w][c * (R + 4) + 16 * s + 4 * g]);
      ret_products<R / 16>(acc, vs, EP + 4, g, c, [&](int s, int i) { return p4[s][i]; });
    }
  }
  T gt[4][EB];  // every gate is requested before the first is used
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t row = ch.x + i0 + min(16 * w + 4 * g + i, rows - 1);
    const T* gp = x + row * a.ldx + 2 * HD + HE + (int64_t)h * a.E;
#pragma unroll
    for (int j = 0; j < EB; ++j) gt[i][j] = gp[min(16 * j + c, a.E - 1)];
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < EB; ++j) ss += acc[j][i] * acc[j][i];  // columns past E are zero
    ss = row_sum(ss);
    const float rs = 1.f / sqrtf(ss / (float)a.E + a.eps);
    const int r = 16 * w + 4 * g + i;
    if (r < rows) {
      T* yp = reinterpret_cast<T*>(a.y) + (ch.x + i0 + r) * HE + (int64_t)h * a.E;
#pragma unroll
      for (int j = 0; j < EB; ++j)
        if (16 * j + c < a.E) st1(yp + 16 * j + c, acc[j][i] * rs * silu_t<T>(ld1(&gt[i][j])));
    }
  }
}

}  // namespace mx

using namespace mx;

extern "C" int mx_retention_mfma_takes(const RetentionChunks* a, int f32);  // retention_mfma.hip
extern "C" void mx_retention_mfma_ends(const RetentionChunks* a, hipStream_t stream);
extern "C" void mx_retention_mfma_out(const RetentionChunks* a, hipStream_t stream);

// -1 (nothing launched): heads wider than 256
extern "C" int mx_retention_chunks(const RetentionChunks* pa, int f32, hipStream_t stream) {
  RetentionChunks a = *pa;
  if (a.nblocks <= 0) return 0;
  if (a.H <= 0 || a.H > 65535 || a.D <= 0 || a.D > 256 || a.E <= 0 || a.E > 256 || a.rd < 0 || a.rd % 2 || a.rd > a.D ||
      a.ldx < 2ll * a.H * (a.D + a.E) || a.nchunks <= 0 || a.nchunks > 65535 || a.nblocks > 65535 || a.nseq <= 0 ||
      a.nseq > 65535 || !a.pw || (a.carry && !a.ws))
    return -1;
  a.v4 = a.D % 4 == 0 && a.E % 4 == 0 && a.rd % 8 == 0 && a.ldx % 4 == 0 && ((uintptr_t)a.x & 15) == 0 &&
         (((uintptr_t)a.cosb | (uintptr_t)a.sinb) & 15) == 0;
#define RE(TT, DP, EP)                                                                                             \
  retention_ends_kernel<TT, DP, EP><<<dim3(a.H, a.nchunks, (a.E + EP - 1) / EP), 256, 0, stream>>>(a)
#define RO(TT, DP, EP) retention_out_kernel<TT, DP, EP><<<dim3(a.H, a.nblocks), 512, 0, stream>>>(a)
#define RED(TT, DP) do { if (a.E <= 64) RE(TT, DP, 64); else RE(TT, DP, 128); } while (0)
#define ROD(TT, DP) do { if (a.E <= 64) RO(TT, DP, 64); else if (a.E <= 128) RO(TT, DP, 128); else RO(TT, DP, 256); } while (0)
#define RT(M, TT) do { if (a.D <= 64) M(TT, 64); else if (a.D <= 128) M(TT, 128); else M(TT, 256); } while (0)
  const bool split = mx_retention_mfma_takes(&a, f32);
  if (a.carry) {
    if (split) mx_retention_mfma_ends(&a, stream);
    else if (f32) RT(RED, float); else RT(RED, uint16_t);
    retention_carry_kernel<<<dim3((a.D * a.E + 255) / 256, a.H, a.nseq), 256, 0, stream>>>(a);
  }
  if (split) mx_retention_mfma_out(&a, stream);
  else if (f32) RT(ROD, float); else RT(ROD, uint16_t);
#undef RT
#undef ROD
#undef RED
#undef RO
#undef RE
  return (int)hipGetLastError();
}
