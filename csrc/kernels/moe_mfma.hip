// Expert mixtures on the matrix cores (gfx950, bf16 storage):
//   * moe_route_mfma : router logits of 16 tokens a workgroup in f32 accumulators, then the choice;
//   * moe_grouped    : the experts' products on rows sorted by expert (prompts): gemm8_core.h's tile loop
//                      with gathered rows, the gated unit in the epilogue;
//   * moe_few_up / moe_few_down : up to 64 tokens (decode steps): every workgroup finds its expert's pairs
//                      among the choices and streams 16-channel slices of the weights past them; the
//                      shared expert's slices run in the same launch.  Weights are read once for up to 64
//                      rows; experts nobody chose are not read, but for the first chunks of their down weights where
//                      these are asked for before the choices (FewLines).
#include "e4m3.h"
#include "gemm8_core.h"
#include "hybrid.h"
#include "moe_route.h"
#include "skinny_core.h"
#include "sublayer.h"

namespace mx {

// ------------------------------------------------------------------ routing
// 8 waves split K in 64-element steps; NB blocks of 16 experts
template <int NB>
__global__ void __launch_bounds__(512) moe_route_mfma_kernel(const uint16_t* __restrict__ x, int64_t ldx,
                                                             const uint16_t* __restrict__ w, int32_t* __restrict__ ids,
                                                             float* __restrict__ wts, int T, int K, int E, int top) {
  __shared__ f32x4 red[8][NB][64];
  __shared__ float z[16][NB * 16];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
  const int t0 = blockIdx.x * 16;
  const uint16_t* xr = x + (int64_t)min(t0 + c, T - 1) * ldx + 16 * g;
  const uint16_t* wr[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) wr[j] = w + (int64_t)min(16 * j + c, E - 1) * K + 16 * g;
  f32x4 acc[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int U = NB == 1 ? 8 : 4;
  for (int kb = wv * 64; kb < K; kb += 512 * U) {
    u16x8 fb[U][2], fa[U][NB][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool on = kb + 512 * u < K;
      const int k = on ? kb + 512 * u : 0;
      fb[u][0] = *reinterpret_cast<const u16x8*>(xr + k);
      fb[u][1] = *reinterpret_cast<const u16x8*>(xr + k + 8);
      if (!on) fb[u][0] = fb[u][1] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        fa[u][j][0] = *reinterpret_cast<const u16x8*>(wr[j] + k);
        fa[u][j][1] = *reinterpret_cast<const u16x8*>(wr[j] + k + 8);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        acc[j] = mfma16_sk(fa[u][j][0], fb[u][0], acc[j]);
        acc[j] = mfma16_sk(fa[u][j][1], fb[u][1], acc[j]);
      }
  }
#pragma unroll
  for (int j = 0; j < NB; ++j) red[wv][j][lane] = acc[j];
  __syncthreads();
  for (int j = wv; j < NB; j += 8) {
    f32x4 s = red[0][j][lane];
#pragma unroll
    for (int i = 1; i < 8; ++i) s += red[i][j][lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) z[c][16 * j + 4 * g + i] = s[i];
  }
  __syncthreads();
  for (int r = wv; r < 16; r += 8) {
    const int64_t row = t0 + r;
    if (row < T) moe_select64(lane < NB * 16 ? z[r][lane] : 0.f, E, top, lane, ids + row * top, wts + row * top);
  }
}

// ------------------------------------------------------------------ few tokens
constexpr int kFewTokens = 64, kFewPairs = 1024;

// What bounds them: weights read once (67 MB up, 34 MB down for 32 tokens at 1B sizes: 3.2 and 2.9 TB/s), and behind one another
// the choices, the list of an expert's pairs, its rows and its weights.  An expert has 8 rows on average there: a block of
// 16 rows instead of two is a quarter of the loads (up 22.6 -> 21.1 us, 48 tokens 26.4 -> 24.2; 8B sizes 60.7 -> 57.1,
// 70.5 -> 65.3).  Weights of an expert known by its place, asked for before the choices, gain little by themselves: several
// workgroups a CU hide each other's waits.
// One slice set: 16 weight rows a slice, 8 gate and the 8 matching up rows where GLU; KW of the 8 waves share the K
// of NC slices (a fragment of the rows feeds NC products), 8 / KW such sets a workgroup.  16 rows x 64 B a load: for many
// rows, whose fragments and sums are then what lasts.
template <bool GLU, int KW, int NC>
struct FewSlices {
  static constexpr int SL = 8 / KW * NC, CH = GLU ? 8 : 16, U = 2;
  typedef int64_t Off;  // of X's rows
  static constexpr int places(int rows) { return 8 * NC * 64 * ((rows + 15) / 16); }
  const uint16_t* wr[NC];
  int n0, k0, k1, ks;

  __device__ __forceinline__ FewSlices(const uint16_t* W, int bx, int N, int K, int w, int lane) {
    const int c = lane & 15;
    ks = w % KW;
    n0 = (bx * SL + w / KW * NC) * CH;
    const int steps = (K + 63) / 64, per = (steps + KW - 1) / KW;
    k0 = ks * per * 64, k1 = min(K, k0 + per * 64);
#pragma unroll
    for (int j = 0; j < NC; ++j)
      wr[j] = W + ((int64_t)(GLU && c >= 8 ? N : 0) + min(n0 + j * CH + (GLU ? c & 7 : c), N - 1)) * K;
  }
  __device__ __forceinline__ void ahead() {}
  __device__ __forceinline__ void move(int64_t by) {
#pragma unroll
    for (int j = 0; j < NC; ++j) wr[j] += by;
  }
  // n rows: xrow(r) reads, yrow(r) is the output's; limit of the unit; ROWS at a time; fresh: after ahead()
  template <int ROWS, typename X, typename Y>
  __device__ __forceinline__ void run(bool fresh, int n, int N, const uint16_t* xb, X xoff, Y yrow, uint16_t* y, float limit,
                                      f32x4* red, int w, int lane, int c, int g) {
    constexpr int MB = (ROWS + 15) / 16;
    auto slot = [&](int wv, int j, int mb) -> f32x4& { return red[((wv * NC + j) * MB + mb) * 64 + lane]; };
    for (int r0 = 0; r0 < n; r0 += 16 * MB) {
      const uint16_t* xr[MB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) xr[mb] = xb + xoff(min(r0 + 16 * mb + c, n - 1));
      f32x4 acc[NC][MB];
#pragma unroll
      for (int j = 0; j < NC; ++j)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[j][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int kb = k0; kb < k1; kb += 64 * U) {
        u16x8 fa[U][NC][2], fb[U][MB][2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = kb + 64 * u + 16 * g;
          const bool on = k < k1;  // K is a multiple of 16
          const int kk = on ? k : 0;
#pragma unroll
          for (int j = 0; j < NC; ++j) {
            fa[u][j][0] = *reinterpret_cast<const u16x8*>(wr[j] + kk);
            fa[u][j][1] = *reinterpret_cast<const u16x8*>(wr[j] + kk + 8);
          }
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) {
            fb[u][mb][0] = *reinterpret_cast<const u16x8*>(xr[mb] + kk);
            fb[u][mb][1] = *reinterpret_cast<const u16x8*>(xr[mb] + kk + 8);
            if (!on) fb[u][mb][0] = fb[u][mb][1] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
          }
        }
        __builtin_amdgcn_sched_barrier(0);  // every load is in flight before the first product waits
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < NC; ++j)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
              acc[j][mb] = mfma16_sk(fa[u][j][0], fb[u][mb][0], acc[j][mb]);
              acc[j][mb] = mfma16_sk(fa[u][j][1], fb[u][mb][1], acc[j][mb]);
            }
      }
      if (r0) __syncthreads();  // the previous rows' sums are read
#pragma unroll
      for (int j = 0; j < NC; ++j)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) slot(w, j, mb) = acc[j][mb];
      __syncthreads();
      for (int jm = ks; jm < NC * MB; jm += KW) {  // the K parts' waves share the sums
        const int j = jm % NC, mb = jm / NC;
        f32x4 s = slot(w - ks, j, mb);
#pragma unroll
        for (int i = 1; i < KW; ++i) s += slot(w - ks + i, j, mb);
        const int r = r0 + 16 * mb + c, ch = n0 + j * CH + 4 * g;
        u16x4 o;
        if constexpr (GLU) {  // rows 4 g .. of the slice: gate in groups 0 and 1, up in 2 and 3
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float up = __uint_as_float(lane_pair<32>(__float_as_uint(s[i])).b);
            o[i] = f2bf(clipped_glu<uint16_t>(s[i], up, limit));
          }
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = f2bf(s[i]);
        }
        if (r < n && ch < N && (!GLU || g < 2)) *reinterpret_cast<u16x4*>(y + (int64_t)yrow(r) * N + ch) = o;
      }
    }
  }
};

// The same slices for a few rows each, in the fragments of skinny_core.h: loads of 8 rows x 128 B, nontemporal, products of 8
// token rows with two useful blocks.  A wave's part of K is whole blocks of U chunks (loads past its end would cost as others do:
// 6 chunks in two parts, blocks of 4 13.6 us, of 3 11.8); the first is asked for before the rows are known.  Down products alone;
// offsets of 32 bits.
template <int KW, int NC, int UC>
struct FewLines {
  static constexpr int SL = 8 / KW * NC, CH = 16, RB = 2 * NC, U = UC;
  static constexpr int places(int rows) { return 8 * RB * 16 * ((rows + 7) / 8); }
  typedef uint32_t Off;  // of X's rows
  typedef u32x4 Frag[U][RB];  // (as vectors of 16 bits they come apart where paths join)
  const char* W;
  uint32_t wo[RB];
  int n0, c0, c1, ks;  // this wave's chunks of 64 k
  Frag pre;

  __device__ __forceinline__ FewLines(const uint16_t* w_, int bx, int N, int K, int w, int lane) {
    const int c = lane & 15, g = lane >> 4;
    W = reinterpret_cast<const char*>(w_);
    ks = w % KW;
    n0 = (bx * SL + w / KW * NC) * CH;
    const int per = K / 64 / KW;
    c0 = ks * per, c1 = c0 + per;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const int ch = n0 + (rb >> 1) * CH + 8 * (rb & 1) + (c & 7);
      wo[rb] = ((uint32_t)min(ch, N - 1) * (uint32_t)K + (uint32_t)sk_lane_k(c, g)) * 2;
    }
  }
  // (readfirstlane: a scalar base and 32-bit offsets; left alone the loop keeps 64-bit addresses a lane, 12 registers and a wave less)
  __device__ __forceinline__ void load(Frag& f, int c) const {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const char* p = W + 128 * (int64_t)__builtin_amdgcn_readfirstlane(c + u);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) f[u][rb] = sk_weights<u32x4>(p + wo[rb]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ void ahead() { load(pre, c0); }
  __device__ __forceinline__ void move(int64_t by) { W += 2 * by; }
  // xoff(r): offset of row r from X, in elements
  template <int ROWS, typename X, typename Y>
  __device__ __forceinline__ void run(bool fresh, int n, int N, const uint16_t* xb, X xoff, Y yrow, uint16_t* y, float limit,
                                      f32x4* red, int w, int lane, int c, int g) {
    constexpr int TB = (ROWS + 7) / 8, MB = (TB + 1) / 2, UX = TB == 1 || U < 4 ? U : U / 2;  // chunks of rows in flight
    auto at = [&](int wv, int rb, int tb) { return ((wv * RB + rb) * TB + tb) * 16; };
    // (the first rows apart: ahead()'s weights are then no longer held)
    auto rows = [&](int r0, auto first) __attribute__((always_inline)) {
      uint32_t xo[TB];
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) xo[tb] = (xoff(min(r0 + 8 * tb + (c & 7), n - 1)) + (uint32_t)sk_lane_k(c, g)) * 2;
      f32x4 acc[RB][TB];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) acc[rb][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
      auto step = [&](const Frag& f, int cb) __attribute__((always_inline)) {
#pragma unroll
        for (int u0 = 0; u0 < U; u0 += UX) {
          u32x4 fb[UX][TB];
#pragma unroll
          for (int u = 0; u < UX; ++u) {
            const char* p = reinterpret_cast<const char*>(xb) + 128 * (int64_t)__builtin_amdgcn_readfirstlane(cb + u0 + u);
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) fb[u][tb] = *reinterpret_cast<const u32x4*>(p + xo[tb]);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int u = 0; u < UX; ++u)
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
              for (int tb = 0; tb < TB; ++tb)
                acc[rb][tb] = mfma16_sk(__builtin_bit_cast(u16x8, f[u0 + u][rb]), __builtin_bit_cast(u16x8, fb[u][tb]),
                                        acc[rb][tb]);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      int cb = c0;
      if constexpr (first) {
        step(pre, cb);
        cb += U;
      }
      for (; cb < c1; cb += U) {
        Frag f;
        load(f, cb);
        step(f, cb);
      }
      if (r0) __syncthreads();  // the previous rows' sums are read
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
          const f32x4 s = sk_both_halves(acc[rb][tb]);
          if (c < 8 && g < 2) red[at(w, rb, tb) + 8 * g + c] = s;
        }
      __syncthreads();
      for (int jm = ks; jm < NC * MB; jm += KW) {  // the K parts' waves share the sums
        const int j = jm % NC, mb = jm / NC, tb = 2 * mb + (c >> 3);
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < KW; ++i)
          s += red[at(w - ks + i, 2 * j + (g >> 1), min(tb, TB - 1)) + 8 * (g & 1) + (c & 7)];
        const int r = r0 + 16 * mb + c, ch = n0 + j * CH + 4 * g;
        u16x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = f2bf(s[i]);
        if (tb < TB && r < n && ch < N) *reinterpret_cast<u16x4*>(y + (int64_t)yrow(r) * N + ch) = o;
      }
    };
    int r0 = 0;
    if (fresh) {
      rows(0, std::true_type{});
      r0 = 8 * TB;
    }
    for (; r0 < n; r0 += 8 * TB) rows(r0, std::false_type{});
  }
};

// GLU: y[pair] = clipped unit of x[token] through [gate | up]; else y[pair] = W x[pair].
// Workgroups: the shared expert's slices (its rows are the tokens), then those of every expert, or - fewer pairs
// than experts - of every pair whose expert no earlier pair has chosen.  Own, ROWS: the experts' slices (up to ROWS rows at a
// time; LESS: up to so many of them, fewer products); Shared, SROWS the shared one's, whose K is longer and whose rows are all
// tokens.  a.logits (GLU): the choices are made here from the router's logits; one workgroup stores them.  TMAX: most tokens.
template <bool GLU, typename Own, int ROWS, int LESS, typename Shared, int SROWS, int TMAX>
__global__ void __launch_bounds__(512, TMAX <= 32 ? 4 : 2) moe_few_kernel(MoeFew a) {
  __shared__ int16_t sel[kFewPairs], list[kFewPairs];
  __shared__ int count;
  __shared__ f32x4 red[Own::places(ROWS) > Shared::places(SROWS) ? Own::places(ROWS) : Shared::places(SROWS)];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  typedef typename Own::Off Off;
  constexpr int SCOLS = Shared::SL * Shared::CH, COLS = Own::SL * Own::CH;
  const int snx = a.sw ? (a.sN + SCOLS - 1) / SCOLS : 0, nx = (a.N + COLS - 1) / COLS, P = a.T * a.top;
  if ((int)blockIdx.x < snx) {
    Shared s(a.sw, blockIdx.x, a.sN, a.sK, w, lane);
    s.ahead();
    s.template run<SROWS>(
        true, a.T, a.sN, GLU ? a.x : a.sx, [&](int r) { return GLU ? r * (Off)a.ldx : r * (Off)a.sK; },
        [](int r) { return r; }, a.sy, a.slimit, red, w, lane, c, g);
    return;
  }
  const int bx = (blockIdx.x - snx) % nx, unit = (blockIdx.x - snx) / nx;
  // What the choices are made of is asked for first, all of it at once, and the weights of an expert known by its place behind
  // it: the choices do not wait for them (no barrier here drains the loads), and they do not wait for the choices.
  constexpr int TW = (TMAX + 7) / 8;  // tokens of a wave
  float z[TW];
  if (GLU && a.logits) {
#pragma unroll
    for (int i = 0; i < TW; ++i) z[i] = a.logits[(int64_t)min(w + 8 * i, a.T - 1) * a.E + min(lane, a.E - 1)];
  } else {
    for (int i = tid; i < P; i += 512) sel[i] = (int16_t)min(max(a.ids[i], 0), a.E - 1);
  }
  const int64_t wsize = (int64_t)(GLU ? 2 : 1) * a.N * a.K;
  const bool known = P > a.E;
  __builtin_amdgcn_sched_barrier(0);
  Own s(a.w + (known ? unit : 0) * wsize, bx, a.N, a.K, w, lane);
  if (known) s.ahead();
  if (GLU && a.logits) {
#pragma unroll
    for (int i = 0; i < TW; ++i) {
      const int t = w + 8 * i;
      if (t >= a.T) break;
      const int store = (int)blockIdx.x == snx;
      moe_choose64(z[i], a.E, a.top, lane, [&](int k, float wt) {
        sel[t * a.top + k] = (int16_t)lane;
        if (store) {
          a.ids_out[t * a.top + k] = lane;
          a.wts_out[t * a.top + k] = wt;
        }
      });
    }
  }
  lds_barrier();
  const int expert = known ? unit : __builtin_amdgcn_readfirstlane(sel[unit]);
  if (w == 0) {  // pairs whose choice this expert is
    int at = 0, first = P;
    for (int i0 = 0; i0 < P; i0 += 64) {
      const bool hit = i0 + lane < P && sel[i0 + lane] == expert;
      const uint64_t m = __ballot(hit);
      if (hit) list[at + __popcll(m & ((1ull << lane) - 1))] = (int16_t)(i0 + lane);
      if (m && first == P) first = i0 + __ffsll((unsigned long long)m) - 1;
      at += __popcll(m);
    }
    if (lane == 0) count = !known && first < unit ? 0 : at;
  }
  lds_barrier();
  const int n = __builtin_amdgcn_readfirstlane(count);
  if (n == 0) return;
  if (!known) s.move(expert * wsize);
  auto xoff = [&](int r) { return (Off)(GLU ? list[r] / a.top : list[r]) * (Off)a.ldx; };
  auto yrow = [&](int r) { return list[r]; };
  if (LESS < ROWS && n <= LESS) s.template run<LESS>(known, n, a.N, a.x, xoff, yrow, a.y, a.limit, red, w, lane, c, g);
  else s.template run<ROWS>(known, n, a.N, a.x, xoff, yrow, a.y, a.limit, red, w, lane, c, g);
}

// The gated products of more pairs than experts, chosen from the router's logits: y[pair] = clipped unit of x[token] through
// [gate | up].  Workgroups: the shared expert's slices (its rows are the tokens), those of every expert, and one that
// stores the choices, behind all others.  A wave finds its expert's tokens by itself (moe_route.h, moe_place): with all
// choices made by every workgroup and two barriers, the weights of half of them began 10 us into the launch (stamped; 32
// tokens, 1B sizes), now 7; steps of 24 / 32 / 48 sequences 1480 / 1567 / 1890 -> 1455 / 1528 / 1813 us, 8B sizes of
// 48 7190 -> 6760.  The other half's logits wait in their CU's queue behind the
// first half's weights: 67 MB come at 4.5 TB/s whatever is asked for first (half or all of a wave's weights ahead of the
// choices: within 0.4 %).
template <typename Own, int ROWS, int LESS, typename Shared, int SROWS, int TMAX>
__global__ void __launch_bounds__(512, TMAX <= 32 ? 4 : 2) moe_up_kernel(MoeFew a) {
  __shared__ int16_t list[kFewTokens];
  __shared__ f32x4 red[Own::places(ROWS) > Shared::places(SROWS) ? Own::places(ROWS) : Shared::places(SROWS)];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  typedef typename Own::Off Off;
  constexpr int SCOLS = Shared::SL * Shared::CH, COLS = Own::SL * Own::CH;
  const int snx = a.sw ? (a.sN + SCOLS - 1) / SCOLS : 0, nx = (a.N + COLS - 1) / COLS;
  if ((int)blockIdx.x < snx) {
    Shared s(a.sw, blockIdx.x, a.sN, a.sK, w, lane);
    s.template run<SROWS>(
        false, a.T, a.sN, a.x, [&](int r) { return r * (Off)a.ldx; }, [](int r) { return r; }, a.sy, a.slimit, red, w, lane,
        c, g);
    return;
  }
  if (blockIdx.x == gridDim.x - 1) {
    for (int t = w; t < a.T; t += 8)
      moe_choose64(a.logits[(int64_t)t * a.E + min(lane, a.E - 1)], a.E, a.top, lane, [&](int k, float wt) {
        a.ids_out[t * a.top + k] = lane;
        a.wts_out[t * a.top + k] = wt;
      });
    return;
  }
  const int bx = (blockIdx.x - snx) % nx, expert = (blockIdx.x - snx) / nx;
  const int n = moe_list(moe_place(a.logits, a.E, a.top, a.T, expert, lane), a.top, lane, list);
  if (n == 0) return;
  Own s(a.w + expert * (2 * (int64_t)a.N * a.K), bx, a.N, a.K, w, lane);
  auto xoff = [&](int r) { return (Off)(list[r] / a.top) * (Off)a.ldx; };
  auto yrow = [&](int r) { return list[r]; };
  if (LESS < ROWS && n <= LESS) s.template run<LESS>(false, n, a.N, a.x, xoff, yrow, a.y, a.limit, red, w, lane, c, g);
  else s.template run<ROWS>(false, n, a.N, a.x, xoff, yrow, a.y, a.limit, red, w, lane, c, g);
}

}  // namespace mx

using namespace mx;

extern "C" int mx_moe_route_mfma(const uint16_t* x, int64_t ldx, const uint16_t* w, int32_t* ids, float* wts, int T, int K,
                                 int E, int top, hipStream_t stream) {
  if (T <= 0) return 0;
  if (K <= 0 || K % 64 || E <= 0 || E > 64 || top <= 0 || top > E || ldx % 8 || ldx < K || (((uintptr_t)x | (uintptr_t)w) & 15))
    return -1;
  const unsigned g = (unsigned)((T + 15) / 16);
#define RM(NB) moe_route_mfma_kernel<NB><<<g, 512, 0, stream>>>(x, ldx, w, ids, wts, T, K, E, top)
  if (E <= 16) RM(1);
  else if (E <= 32) RM(2);
  else RM(4);
#undef RM
  return (int)hipGetLastError();
}

// rows sorted by expert, tiles of at most 256 rows; xrows: rows of x; -1: sizes it does not take
extern "C" int mx_moe_grouped(const MoeGemm* pa, int64_t xrows, hipStream_t stream) {
  const MoeGemm& a = *pa;
  if (a.ntiles <= 0) return 0;
  const int64_t abytes = ((xrows - 1) * a.ldx + a.K) * 2, bbytes = (int64_t)(a.glu ? 2 : 1) * a.N * a.K * 2;
  if (a.N <= 0 || a.K <= 0 || a.N % 8 || a.K % 8 || a.ldx % 8 || a.ldx < a.K || xrows <= 0 ||
      abytes >= ((int64_t)1 << 31) - 4096 || bbytes >= ((int64_t)1 << 31) - 4096 ||
      (((uintptr_t)a.x | (uintptr_t)a.w | (uintptr_t)a.y) & 15))
    return -1;
  G8Moe mo = {};
  mo.tiles = reinterpret_cast<const int4*>(a.tiles), mo.src = a.src, mo.arec = (uint32_t)abytes;
  mo.F = a.N, mo.limit = a.limit;
  const int nn = a.glu ? (a.N + 127) / 128 : (a.N + 255) / 256;
  const int64_t grid = (int64_t)a.ntiles * nn;
  if (grid > INT32_MAX || (int64_t)a.ntiles * 256 > INT32_MAX) return -1;
  const uint16_t* x = reinterpret_cast<const uint16_t*>(a.x);
  const uint16_t* w = reinterpret_cast<const uint16_t*>(a.w);
  if (a.glu)
    gemm8_kernel<true, true, false, false, 0, 4, G8_EPI_MOE_GLU><<<(unsigned)grid, 512, 0, stream>>>(
        x, a.ldx, w, a.K, a.y, a.N, a.ntiles * 256, nn * 256, a.K, nullptr, 1.f, 0, 0, G8Epi{}, mo);
  else
    gemm8_kernel<true, true, false, false, 0, 4, G8_EPI_MOE><<<(unsigned)grid, 512, 0, stream>>>(
        x, a.ldx, w, a.K, a.y, a.N, a.ntiles * 256, nn * 256, a.K, nullptr, 1.f, 0, 0, G8Epi{}, mo);
  return (int)hipGetLastError();
}

extern "C" int mx_moe_stream(const MoeFew* pa, hipStream_t stream);

extern "C" int mx_moe_few(const MoeFew* pa, int glu, hipStream_t stream) {
  const MoeFew& a = *pa;
  if (a.T <= 0) return 0;
  const uintptr_t al = (uintptr_t)a.x | (uintptr_t)a.w | (uintptr_t)a.sw | (uintptr_t)a.sx;
  if (a.T > kFewTokens || a.top <= 0 || a.T * a.top > kFewPairs || a.E <= 0 || a.E > 65534 ||
      (a.logits && (!glu || a.E > 64 || a.top > a.E)) || (!a.logits && !a.ids) || a.N <= 0 || a.N % 4 || a.K <= 0 || a.K % 16 || a.ldx % 8 || a.ldx < a.K || (al & 15) ||
      (a.sw && (a.sN <= 0 || a.sN % 4 || a.sK <= 0 || a.sK % 16)))
    return -1;
  if (glu) {
    const int r = mx_moe_stream(pa, stream);
    if (r != -1) return r;
  }
  // channels of a workgroup: up 16, from 33 tokens on 32 (the rows' fragments are then most of the traffic; first
  // moe_stream.hip, more pairs than experts);
  // down 64, for a few pairs 32 with K in four parts; the shared expert's down, whose K is the longest, 16 with K in
  // eight (its few workgroups were the last to end: K 2048 in two parts are 16 waits for memory one after another;
  // 32 tokens, 1B sizes 30.5 -> 16.1 us, 4 tokens 15.6 -> 10.3; 8B sizes 38.4 -> 33.1, 22.2 -> 18.7)
  const int64_t units = a.T * a.top <= a.E ? a.T * a.top : a.E;
#define MF(GLU, OWN, ROWS, LESS, SHARED, SROWS, TMAX)                                                            \
  do {                                                                                                           \
    typedef OWN Own;                                                                                             \
    typedef SHARED Shared;                                                                                       \
    const int64_t cols = Own::SL * Own::CH, sc = Shared::SL * Shared::CH;                                        \
    const int64_t gr = units * ((a.N + cols - 1) / cols) + (a.sw ? (a.sN + sc - 1) / sc : 0);                    \
    if (gr > INT32_MAX) return -1;                                                                               \
    moe_few_kernel<GLU, Own, ROWS, LESS, Shared, SROWS, TMAX><<<(unsigned)gr, 512, 0, stream>>>(a);              \
  } while (0)
#define FS(...) FewSlices<__VA_ARGS__>
#define FL(...) FewLines<__VA_ARGS__>
  // Down: FewLines for more than 8 pairs where both K parts are whole blocks of 3 chunks, past one block each from 17 tokens on
  // (and up to 16 tokens with the shared expert's eight in whole blocks of 4): loads past a part's end cost as others do.  us,
  // FewSlices -> FewLines: 2048 x 384, 16 / 64 / 128 pairs 8.2 -> 6.9, 8.7 -> 7.0, 10.0 -> 8.3; 4096 x 768 with a shared expert of
  // 2048, 128 pairs 28.5 -> 27.5; 2048 x 1152, 128 pairs 19.3 -> 17.5.  Elsewhere it loses: 1024 x 512, 2 to 8 pairs half as much
  // again, 2048 x 256, 256 pairs a third, 2 to 8 pairs of any K, where four K parts hide more, up to two thirds; 4096 x 768 with
  // few tokens' uneven choices, 20 pairs 18.0 -> 23.4, 48 22.8 -> 24.7.  Up stays with FewSlices (2 x 384 x 2048, 32 tokens
  // 21.1 us, 23.3 by FewLines; 768 x 4096 57.1, 62.4).
  const int pairs = a.T * a.top;
  const bool lines = !glu && a.K % 384 == 0 && pairs > 8 &&
                     (a.T > 16 || (a.K <= 384 && (!a.sw || a.sK % 2048 == 0))) &&
                     std::max(std::max((int64_t)a.N * a.K, (int64_t)a.sN * a.sK),
                              pairs * std::max(a.ldx, (int64_t)a.sK)) < (1ll << 31) - 4096;
#define MU(OWN, ROWS, LESS, SHARED, SROWS, TMAX)                                                                 \
  do {                                                                                                           \
    typedef OWN Own;                                                                                             \
    typedef SHARED Shared;                                                                                       \
    const int64_t cols = Own::SL * Own::CH, sc = Shared::SL * Shared::CH;                                        \
    const int64_t gr = a.E * ((a.N + cols - 1) / cols) + (a.sw ? (a.sN + sc - 1) / sc : 0) + 1;                  \
    if (gr > INT32_MAX) return -1;                                                                               \
    moe_up_kernel<Own, ROWS, LESS, Shared, SROWS, TMAX><<<(unsigned)gr, 512, 0, stream>>>(a);                    \
  } while (0)
  if (glu && a.logits && pairs > a.E) {
    if (a.T <= 16) MU(FS(true, 8, 2), 16, 16, FS(true, 8, 2), 16, 16);
    else if (a.T <= 32) MU(FS(true, 8, 2), 32, 16, FS(true, 8, 2), 32, 32);
    else MU(FS(true, 8, 4), 64, 16, FS(true, 8, 4), 64, 64);
  } else if (glu) {
    if (a.T <= 16) MF(true, FS(true, 8, 2), 16, 16, FS(true, 8, 2), 16, 16);
    else if (a.T <= 32) MF(true, FS(true, 8, 2), 32, 16, FS(true, 8, 2), 32, 32);
    else MF(true, FS(true, 8, 4), 64, 16, FS(true, 8, 4), 64, 64);
  } else if (pairs <= 8) {
    MF(false, FS(false, 4, 1), 16, 16, FS(false, 8, 1), 16, 16);
  } else if (lines) {
    if (a.T <= 8) MF(false, FL(2, 1, 3), 8, 8, FL(8, 1, 4), 8, 8);
    else if (a.T <= 16) MF(false, FL(2, 1, 3), 16, 8, FL(8, 1, 4), 16, 16);
    else if (a.T <= 32) MF(false, FL(2, 1, 3), 16, 8, FS(false, 8, 1), 32, 32);
    else MF(false, FL(2, 1, 3), 32, 16, FS(false, 8, 1), 64, 64);
  } else {
    if (a.T <= 16) MF(false, FS(false, 2, 1), 16, 16, FS(false, 8, 1), 16, 16);
    else if (a.T <= 32) MF(false, FS(false, 2, 1), 32, 16, FS(false, 8, 1), 32, 32);
    else MF(false, FS(false, 2, 1), 64, 16, FS(false, 8, 1), 64, 64);
  }
#undef FL
#undef FS
#undef MF
#undef MU
  return (int)hipGetLastError();
}
