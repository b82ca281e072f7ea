// Mixture of experts for gfx950: routing, grouping of (token, choice) pairs by expert, and the experts'
// products on grouped rows.
//   * moe_route : router logits in f32, the largest `top` of every row, softmax over them;
//   * moe_group : pairs sorted by expert (counting sort in one workgroup) and the row tiles of the
//                 products, all on the device: nothing of it needs the host;
//   * moe_gemm  : Y = act(X_e W_e^T) on the rows of each expert, f32 arithmetic without matrix cores, any
//                 sizes (f32 storage, or sizes outside moe_mfma.hip).
#include "hybrid.h"
#include "moe_route.h"
#include "sublayer.h"

namespace mx {

constexpr int kMoeMaxExperts = 1024;

// ------------------------------------------------------------------ routing
// one workgroup of 4 waves a token: a wave takes every 4th expert's dot product, wave 0 selects
template <typename T, int VEC>
__global__ void __launch_bounds__(256) moe_route_kernel(const T* __restrict__ x, int64_t ldx, const T* __restrict__ w,
                                                        int32_t* __restrict__ ids, float* __restrict__ wts, int K, int E,
                                                        int top) {
  __shared__ float z[kMoeMaxExperts];
  const int row = blockIdx.x, wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const T* xp = x + row * ldx;
  for (int e = wv; e < E; e += 4) {
    float s = 0.f;
    for (int c = lane * VEC; c < K; c += 64 * VEC) {
      float a[VEC], b[VEC];
      ldv<VEC>(xp + c, a);
      ldv<VEC>(w + (int64_t)e * K + c, b);
#pragma unroll
      for (int j = 0; j < VEC; ++j) s += a[j] * b[j];
    }
    s = wave_sum(s);
    if (lane == 0) z[e] = s;
  }
  __syncthreads();
  if (wv) return;
  if (E <= 64) {
    moe_select64(lane < E ? z[lane] : 0.f, E, top, lane, ids + (int64_t)row * top, wts + (int64_t)row * top);
    return;
  }
  moe_select<T>(z, E, top, lane, ids + (int64_t)row * top, wts + (int64_t)row * top);
}

// ------------------------------------------------------------------ grouping
// ids [P] -> src (token of each sorted row), inv (sorted row of each pair), tiles of at most bm rows (expert, first
// row, rows, number of tiles), the unused ones last
__global__ void __launch_bounds__(1024) moe_group_kernel(const int32_t* __restrict__ ids, int P, int top, int E, int bm,
                                                         int32_t* __restrict__ src, int32_t* __restrict__ inv,
                                                         int4* __restrict__ tiles, int ntiles) {
  __shared__ int cnt[kMoeMaxExperts], first[kMoeMaxExperts], tfirst[kMoeMaxExperts + 1];
  const int t = threadIdx.x;
  for (int e = t; e < E; e += 1024) cnt[e] = 0;
  __syncthreads();
  for (int i = t; i < P; i += 1024) atomicAdd(&cnt[min(max(ids[i], 0), E - 1)], 1);
  __syncthreads();
  if (t < 64) {  // wave 0: running sums over the experts
    int rows = 0, tl = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + t, n = e < E ? cnt[e] : 0, m = (n + bm - 1) / bm;
      int a = n, b = m;
      for (int o = 1; o < 64; o <<= 1) {
        const int pa = __shfl_up(a, o, 64), pb = __shfl_up(b, o, 64);
        if (t >= o) a += pa, b += pb;
      }
      if (e < E) first[e] = rows + a - n, tfirst[e] = tl + b - m;
      rows += __shfl(a, 63, 64);
      tl += __shfl(b, 63, 64);
    }
    if (t == 0) tfirst[E] = tl;
  }
  __syncthreads();
  for (int e = t; e < E; e += 1024) {
    const int n = cnt[e];
    for (int j = 0, r = 0; r < n; ++j, r += bm)
      if (tfirst[e] + j < ntiles) tiles[tfirst[e] + j] = int4{e, first[e] + r, min(bm, n - r), tfirst[E]};
  }
  for (int i = tfirst[E] + t; i < ntiles; i += 1024) tiles[i] = int4{0, 0, 0, tfirst[E]};
  __syncthreads();
  for (int i = t; i < P; i += 1024) {
    const int pos = atomicAdd(&first[min(max(ids[i], 0), E - 1)], 1);
    src[pos] = i / top;
    inv[i] = pos;
  }
}

// ------------------------------------------------------------------ products, any sizes
// tile 64 rows x 64 columns, K in steps of 16 through LDS, 4 x 4 outputs a thread; GLU: gate and up
// columns side by side
constexpr int kMgB = 64, kMgK = 16;
template <typename T, bool GLU>
__global__ void __launch_bounds__(256) moe_gemm_kernel(MoeGemm a) {
  const int4 tl = reinterpret_cast<const int4*>(a.tiles)[blockIdx.y];
  const int rows = tl.z;
  if (rows == 0) return;
  __shared__ float xs[kMgK][kMgB + 4], ws[GLU ? 2 : 1][kMgK][kMgB + 4];
  const int t = threadIdx.x, tx = t & 15, ty = t >> 4, n0 = blockIdx.x * kMgB;
  const T* x = reinterpret_cast<const T*>(a.x);
  const T* w = reinterpret_cast<const T*>(a.w) + (int64_t)tl.x * (GLU ? 2 : 1) * a.N * a.K;
  const int lr = t >> 2, lk = (t & 3) * 4;  // staging: row, 4 k
  const bool xon = lr < rows, won = n0 + lr < a.N;
  const int xr = xon ? (a.src ? a.src[tl.y + lr] : tl.y + lr) : 0;
  float acc[GLU ? 2 : 1][4][4] = {};
  for (int k0 = 0; k0 < a.K; k0 += kMgK) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = k0 + lk + j;
      xs[lk + j][lr] = xon && k < a.K ? ld1(x + (int64_t)xr * a.ldx + k) : 0.f;
      ws[0][lk + j][lr] = won && k < a.K ? ld1(w + (int64_t)(n0 + lr) * a.K + k) : 0.f;
      if constexpr (GLU) ws[1][lk + j][lr] = won && k < a.K ? ld1(w + (int64_t)(a.N + n0 + lr) * a.K + k) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kMgK; ++k) {
      float xv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) xv[i] = xs[k][ty * 4 + i];
#pragma unroll
      for (int g = 0; g < (GLU ? 2 : 1); ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float wv = ws[g][k][tx * 4 + j];
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[g][i][j] += xv[i] * wv;
        }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = ty * 4 + i;
    if (r >= rows) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = n0 + tx * 4 + j;
      if (c < a.N)
        st1(reinterpret_cast<T*>(a.y) + (int64_t)(tl.y + r) * a.N + c,
            GLU ? clipped_glu<T>(acc[0][i][j], acc[GLU ? 1 : 0][i][j], a.limit) : acc[0][i][j]);
    }
  }
}

}  // namespace mx

using namespace mx;

extern "C" int mx_moe_route(const void* x, int64_t ldx, const void* w, int f32, int32_t* ids, float* wts, int T, int K,
                            int E, int top, hipStream_t stream) {
  if (T <= 0) return 0;
  if (K <= 0 || E <= 0 || E > kMoeMaxExperts || top <= 0 || top > E) return -1;
  const bool al = ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0;
#define MR(TT, VV) moe_route_kernel<TT, VV><<<T, 256, 0, stream>>>((const TT*)x, ldx, (const TT*)w, ids, wts, K, E, top)
  if (f32) { if (al && K % 4 == 0 && ldx % 4 == 0) MR(float, 4); else MR(float, 1); }
  else { if (al && K % 8 == 0 && ldx % 8 == 0) MR(uint16_t, 8); else MR(uint16_t, 1); }
#undef MR
  return (int)hipGetLastError();
}

extern "C" int mx_moe_group(const int32_t* ids, int P, int top, int E, int bm, int32_t* src, int32_t* inv, int32_t* tiles,
                            int ntiles, hipStream_t stream) {
  if (P <= 0) return 0;
  if (E <= 0 || E > kMoeMaxExperts || top <= 0 || bm <= 0 || ntiles < P / bm + (E < P ? E : P)) return -1;
  moe_group_kernel<<<1, 1024, 0, stream>>>(ids, P, top, E, bm, src, inv, (int4*)tiles, ntiles);
  return (int)hipGetLastError();
}

// tiles of at most 64 rows
extern "C" int mx_moe_gemm(const MoeGemm* pa, int f32, hipStream_t stream) {
  const MoeGemm& a = *pa;
  if (a.ntiles <= 0) return 0;
  if (a.N <= 0 || a.K <= 0 || a.ntiles > 65535 || a.ldx < a.K) return -1;
  const dim3 g((a.N + kMgB - 1) / kMgB, a.ntiles);
#define MG(TT, GG) moe_gemm_kernel<TT, GG><<<g, 256, 0, stream>>>(a)
  if (f32) { if (a.glu) MG(float, true); else MG(float, false); }
  else { if (a.glu) MG(uint16_t, true); else MG(uint16_t, false); }
#undef MG
  return (int)hipGetLastError();
}
