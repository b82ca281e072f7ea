// Batched token sampler with per-row temperature / top-k / top-p.
//
// OpenAI / LiteLLM semantics (the reference's completion() endpoint,
// src/distributed_inference.py:37): probabilities are softmax(logits / T); the
// candidate set is the top_k most likely tokens (k <= 0: all), then the
// smallest most-likely prefix of those whose mass reaches top_p of the set
// (the token that crosses top_p is kept); one token is drawn from the
// renormalised candidates.  T <= 0 is greedy argmax.
//
// The draw is Gumbel-max restricted to the kept tokens: argmax of x / T + G(seed, step, index) is an EXACT
// sample of the renormalised distribution over them, with the same (seed, step, index) noise as the
// greedy / temperature kernel in decode.hip, so a request's stream does not depend on batching.
//
// Split form (vocabularies of kSplitV and more): four launches over (chunk, row), so a step's few rows fill the
// chip.  One workgroup a row kept 32 of 256 CUs on six to nine passes whose LDS atomics and logarithms bound it:
// 253 us for 32 rows of 128,256 bf16 logits of mixed parameters, where the four launches take 63 us (stats 6,
// hist 15, pick 24, final 18; all top-p 85 us, all top-k 38, temperature alone 26).
//  * stats: a chunk's largest (with its index) and smallest logit;
//  * hist: masses exp2((x - max) log2e / T) and counts in 2048 bins, linear in the exponent (64 bins a power of
//    two, finer where the row's whole range is under 32 of them).  A bin holds all tokens of a value, so bins
//    order tokens as their logits do.  Masses are summed as integers (2^-42): any order gives the same sums;
//  * pick: the bins where top-k and top-p cross, from the sums; tokens ahead of them compete at once, those
//    inside are listed (a value or two: tens to hundreds of tokens), the rest is dropped;
//  * final: exact counts and masses above each listed token, the kept ones compete with the chunks' winners.
// A row whose list overflows (thousands of tokens of one value at the boundary), and short vocabularies, take the
// one-workgroup form: no sort, the k-th largest key and then the top-p boundary key by a radix select over
// order-preserving 32-bit keys, 11 + 11 + 10 bits, over LDS histograms.  Its mass histogram uses float atomics: a
// boundary whose cumulative mass is within rounding of top_p * Z can move by one key between runs.
//
// Ties at a boundary are kept.
#include <algorithm>

#include "common.h"

namespace mx {

__device__ __forceinline__ uint32_t okey(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key2f(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

__device__ __forceinline__ uint32_t hash3s(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t h = a * 0x9E3779B1u ^ (b + 0x7F4A7C15u) * 0x85EBCA77u ^ (c + 0x165667B1u) * 0xC2B2AE3Du;
  h ^= h >> 15; h *= 0x2C1B3C6Du; h ^= h >> 12; h *= 0x297A2D39u; h ^= h >> 15;
  return h;
}

constexpr int kSampThreads = 1024;
constexpr int kBins = 2048;  // 11-bit digits

template <typename T>
struct RowReader {
  const T* x;
  int V;
  // calls f(index, value) for every element; 8 elements per lane per step (16 B bf16 / 2x16 B f32)
  template <typename F>
  __device__ __forceinline__ void each(F&& f) const {
    const int vec_end = (V / 8) * 8;
    const bool aligned = (((uintptr_t)x) & 15) == 0;
    if (aligned) {
      for (int base = threadIdx.x * 8; base < vec_end; base += kSampThreads * 8) {
        if constexpr (sizeof(T) == 2) {
          const u16x8 v = *reinterpret_cast<const u16x8*>(reinterpret_cast<const uint16_t*>(x) + base);
#pragma unroll
          for (int j = 0; j < 8; ++j) f(base + j, bf2f(v[j]));
        } else {
          const f32x4 a = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(x) + base);
          const f32x4 b = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(x) + base + 4);
#pragma unroll
          for (int j = 0; j < 4; ++j) f(base + j, a[j]);
#pragma unroll
          for (int j = 0; j < 4; ++j) f(base + 4 + j, b[j]);
        }
      }
    }
    for (int c = (aligned ? vec_end : 0) + threadIdx.x; c < V; c += kSampThreads) {
      float v;
      if constexpr (sizeof(T) == 2) v = bf2f(reinterpret_cast<const uint16_t*>(x)[c]);
      else v = reinterpret_cast<const float*>(x)[c];
      f(c, v);
    }
  }
};

// Radix-select step: over elements whose key matches `prefix` on the bits above
// `shift + nbits` (and passes `keep`), histogram the next `nbits` digit with weight
// wfn(value); pick the digit where the descending cumulative weight, starting at
// `*above`, first reaches `target`; fold the weight of higher digits into `*above`.
template <typename T, typename K, typename W>
__device__ __forceinline__ uint32_t radix_digit(const RowReader<T>& rd, float* hist, float* scan, int* sel,
                                                uint32_t prefix, int shift, int nbits, K keep, W wfn, float* above,
                                                float target) {
  const int nb = 1 << nbits;
  for (int i = threadIdx.x; i < kBins; i += kSampThreads) hist[i] = 0.f;
  __syncthreads();
  const uint32_t hi_mask = (shift + nbits >= 32) ? 0u : (0xffffffffu << (shift + nbits));
  rd.each([&](int idx, float v) {
    const uint32_t k = okey(v);
    if (((k ^ prefix) & hi_mask) == 0 && keep(k)) atomicAdd(&hist[(k >> shift) & (nb - 1)], wfn(v));
  });
  __syncthreads();
  // descending inclusive suffix sums: thread t owns bins 2t, 2t+1 (kBins = 2 * threads)
  const int t = threadIdx.x;
  const float h0 = t * 2 < nb ? hist[t * 2] : 0.f, h1 = t * 2 + 1 < nb ? hist[t * 2 + 1] : 0.f;
  float mine = h0 + h1;
  // block suffix scan over threads (descending order = reverse thread order)
  const int lane = t & 63, wv = t >> 6;
  float inc = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {  // inclusive suffix within the wave (lanes >= this lane)
    const float y = __shfl_down(inc, o, 64);
    if (lane + o < 64) inc += y;
  }
  if (lane == 0) scan[wv] = inc;  // wave total
  __syncthreads();
  float after = 0.f;  // total of the waves above this one
  for (int w2 = wv + 1; w2 < kSampThreads / 64; ++w2) after += scan[w2];
  const float suf1 = after + inc - h0;  // suffix including bin 2t+1
  const float suf0 = after + inc;       // suffix including bin 2t
  const float ab = *above;
  if (t == 0) *sel = 0;
  __syncthreads();
  // the digit d with ab + suffix_excl(d) < target <= ab + suffix_incl(d); digit 0 if none
  if (t * 2 + 1 < nb && ab + (suf1 - h1) < target && ab + suf1 >= target) *sel = t * 2 + 1;
  if (t * 2 < nb && ab + (suf0 - h0) < target && ab + suf0 >= target) *sel = t * 2;
  __syncthreads();
  const int d = *sel;
  // weight of the digits above d (suffix excluding d), published by its owner
  if ((d >> 1) == t) scan[32] = (d & 1) ? (suf1 - h1) : (suf0 - h0);
  __syncthreads();
  const float ex = scan[32];
  __syncthreads();
  *above = ab + ex;
  return prefix | ((uint32_t)d << shift);
}

// A row's parameters: device arrays, or by value where the caller has them on the host.
struct SampRow {
  float temp, p;
  int k;
  uint32_t seed, step;
};
constexpr int kSampGroup = 64;  // rows of one launch's by-value parameters
struct SampArgs {
  const float* temps;  // nullptr: rows[]
  const float* ps;
  const int32_t* ks;
  const int64_t* seeds;
  const int32_t* steps;
  SampRow rows[kSampGroup];
};
__device__ __forceinline__ SampRow samp_row(const SampArgs& a, int r) {
  if (a.temps) return SampRow{a.temps[r], a.ps[r], a.ks[r], (uint32_t)a.seeds[r], (uint32_t)a.steps[r]};
  return a.rows[r];
}

__device__ __forceinline__ float gumbel_score(float v, float inv_t, uint32_t seed, uint32_t step, int idx) {
  const uint32_t h = hash3s(seed, step, (uint32_t)idx);  // = decode.hip sample_kernel noise of a 1-row call
  const float u = ((h >> 8) + 0.5f) * (1.0f / 16777216.0f);
  return v * inv_t - __logf(-__logf(u));
}

// One row by one workgroup of kSampThreads.
struct SampScratch {
  float hist[kBins];
  float scan[40];
  int sel;
  float red[16];
  int redi[16];
};

template <typename T>
__device__ __forceinline__ int topkp_row(const T* __restrict__ x, int V, const SampRow& rp, SampScratch& sc) {
  float(&hist)[kBins] = sc.hist;
  float(&scan)[40] = sc.scan;
  int& sel = sc.sel;
  float(&red)[16] = sc.red;
  int(&redi)[16] = sc.redi;
  const RowReader<T> rd{x, V};
  const float temp = rp.temp;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint32_t seed = rp.seed, step = rp.step;

  // pass 1: max (greedy: argmax directly)
  float best = -INFINITY;
  int bi = 0x7fffffff;
  rd.each([&](int idx, float v) {
    if (v > best || (v == best && idx < bi)) { best = v; bi = idx; }
  });
  auto argmax_reduce = [&](float& b, int& i) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(b, o, 64);
      const int oi = __shfl_xor(i, o, 64);
      if (ov > b || (ov == b && oi < i)) { b = ov; i = oi; }
    }
    __syncthreads();
    if (lane == 0) { red[wv] = b; redi[wv] = i; }
    __syncthreads();
    b = red[0];
    i = redi[0];
    for (int w2 = 1; w2 < kSampThreads / 64; ++w2)
      if (red[w2] > b || (red[w2] == b && redi[w2] < i)) { b = red[w2]; i = redi[w2]; }
  };
  argmax_reduce(best, bi);
  if (bi >= V) bi = 0;  // no logit is a number
  if (!(temp > 0.f)) return bi;
  const float mx = best;
  const float c = 1.4426950408889634f / temp;  // exp2 domain
  const float inv_t = 1.f / temp;
  uint32_t thr = 0;  // keep keys >= thr
  const int k = rp.k;
  if (k > 0 && k < V) {  // k-th largest key (counts)
    float above = 0.f;
    uint32_t pre = 0;
    pre = radix_digit(rd, hist, scan, &sel, pre, 21, 11, [](uint32_t) { return true; },
                      [](float) { return 1.f; }, &above, (float)k);
    pre = radix_digit(rd, hist, scan, &sel, pre, 10, 11, [](uint32_t) { return true; },
                      [](float) { return 1.f; }, &above, (float)k);
    pre = radix_digit(rd, hist, scan, &sel, pre, 0, 10, [](uint32_t) { return true; },
                      [](float) { return 1.f; }, &above, (float)k);
    thr = pre;
  }
  const float p = rp.p;
  if (p < 1.f) {
    // Z over the kept set, then the top-p boundary by mass
    float z = 0.f;
    const uint32_t t0 = thr;
    rd.each([&](int, float v) {
      if (okey(v) >= t0) z += __builtin_amdgcn_exp2f((v - mx) * c);
    });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) z += __shfl_xor(z, o, 64);
    __syncthreads();
    if (lane == 0) red[wv] = z;
    __syncthreads();
    z = 0.f;
    for (int w2 = 0; w2 < kSampThreads / 64; ++w2) z += red[w2];
    const float target = fmaxf(p, 0.f) * z;
    float above = 0.f;
    uint32_t pre = 0;
    auto keep = [t0](uint32_t kk) { return kk >= t0; };
    auto wf = [mx, c](float v) { return __builtin_amdgcn_exp2f((v - mx) * c); };
    pre = radix_digit(rd, hist, scan, &sel, pre, 21, 11, keep, wf, &above, target);
    pre = radix_digit(rd, hist, scan, &sel, pre, 10, 11, keep, wf, &above, target);
    pre = radix_digit(rd, hist, scan, &sel, pre, 0, 10, keep, wf, &above, target);
    thr = max(thr, pre);
  }
  // Gumbel-max over the kept keys
  const uint32_t tf = thr;
  float gb = -INFINITY;
  int gi = 0x7fffffff;
  rd.each([&](int idx, float v) {
    if (okey(v) < tf) return;
    const float s = gumbel_score(v, inv_t, seed, step, idx);
    if (s > gb || (s == gb && idx < gi)) { gb = s; gi = idx; }
  });
  argmax_reduce(gb, gi);
  return gi < V ? gi : bi;
}

template <typename T>
__global__ void __launch_bounds__(kSampThreads) sample_topkp_kernel(const T* __restrict__ logits,
                                                                    int64_t* __restrict__ out, int V, SampArgs a) {
  __shared__ SampScratch sc;
  const int row = blockIdx.x;
  const int id = topkp_row(logits + (size_t)row * V, V, samp_row(a, row), sc);
  if (threadIdx.x == 0) out[row] = id;
}

// ------------------------------------------------------------------ split form
// Shorter rows: one workgroup, one launch.  32 top-p rows of 8,191: 30 us against 41 split; of 32,768: about 80
// (its time grows with the row) against 47.
constexpr int kSplitV = 16384;
constexpr int kSplitMaxV = (1 << 22) - 1;  // as many masses of up to 2^42 stay below 2^64
constexpr int kMBins = 2048;
constexpr int kMaxCh = 64;         // chunks a row (= one wave over their partials)
constexpr int kListCap = 1024;     // listed tokens a row
constexpr int kChThreads = 256;

struct SampWs {
  float *mx, *mn, *gv;   // [rows, nch]: largest, smallest finite logit; best score among tokens kept at once
  int *mi, *gi;          // their indexes
  unsigned long long* mass;  // [rows, kMBins]
  uint32_t* cnt;             // [rows, kMBins]
  unsigned long long* list;  // [rows, kListCap] key << 32 | index
  uint32_t* nlist;           // [rows]
};

__device__ __forceinline__ void pick(float& b, int& i, float ov, int oi) {
  if (ov > b || (ov == b && oi < i)) { b = ov; i = oi; }
}
__device__ __forceinline__ void wave_pick(float& b, int& i) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) pick(b, i, __shfl_xor(b, o, 64), __shfl_xor(i, o, 64));
}

// f(index, value) over [c0, c1) of a row; 16-B loads where the row and the chunk allow it
template <typename T, typename F>
__device__ __forceinline__ void each_in(const T* __restrict__ x, int c0, int c1, F&& f) {
  int c = c0;
  if ((((uintptr_t)(x + c0)) & 15) == 0) {
    const int ve = c0 + (c1 - c0) / 8 * 8;
    for (int b = c0 + (int)threadIdx.x * 8; b < ve; b += kChThreads * 8) {
      if constexpr (sizeof(T) == 2) {
        const u16x8 v = *reinterpret_cast<const u16x8*>(x + b);
#pragma unroll
        for (int j = 0; j < 8; ++j) f(b + j, bf2f(v[j]));
      } else {
        const f32x4 u = *reinterpret_cast<const f32x4*>(x + b), v = *reinterpret_cast<const f32x4*>(x + b + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) f(b + j, u[j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) f(b + 4 + j, v[j]);
      }
    }
    c = ve;
  }
  for (c += threadIdx.x; c < c1; c += kChThreads) {
    if constexpr (sizeof(T) == 2) f(c, bf2f(x[c]));
    else f(c, x[c]);
  }
}

template <typename T>
__global__ void __launch_bounds__(kChThreads) samp_stats_kernel(const T* __restrict__ logits, int V, int chunk,
                                                                SampWs ws) {
  __shared__ float sv[4], sm[4];
  __shared__ int si[4];
  const int row = blockIdx.y, nch = gridDim.x, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int i = blockIdx.x * kChThreads + threadIdx.x; i < kMBins; i += nch * kChThreads) {
    ws.mass[row * kMBins + i] = 0;
    ws.cnt[row * kMBins + i] = 0;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) ws.nlist[row] = 0;
  const int c0 = blockIdx.x * chunk;
  float b = -INFINITY, m = INFINITY;
  int bi = 0x7fffffff;
  each_in(logits + (size_t)row * V, c0, min(V, c0 + chunk), [&](int i, float v) {
    pick(b, bi, v, i);
    if (v > -INFINITY) m = fminf(m, v);
  });
  wave_pick(b, bi);
  m = -wave_max(-m);
  if (lane == 0) { sv[wv] = b; si[wv] = bi; sm[wv] = m; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kChThreads / 64; ++w) {
      pick(b, bi, sv[w], si[w]);
      m = fminf(m, sm[w]);
    }
    ws.mx[row * kMaxCh + blockIdx.x] = b;
    ws.mi[row * kMaxCh + blockIdx.x] = bi;
    ws.mn[row * kMaxCh + blockIdx.x] = m;
  }
}

// what the bins of a row are made of; every lane of a wave calls it
struct RowScale {
  float mx, c, scale;
  int mi;
  __device__ __forceinline__ int bin(float v) const {  // not-a-numbers: the first
    return (int)fminf(fmaxf((mx - v) * c * scale, 0.f), (float)(kMBins - 1));
  }
  __device__ __forceinline__ unsigned long long weight(float v) const {  // in 2^-42
    const float w = fminf(fmaxf(__builtin_amdgcn_exp2f((v - mx) * c), 0.f), 1.f) * 2097152.f;
    const uint32_t hi = (uint32_t)w;
    return ((unsigned long long)hi << 21) + (uint32_t)((w - (float)hi) * 2097152.f);
  }
};
__device__ __forceinline__ RowScale row_scale(const SampWs& ws, int row, int nch, float temp) {
  const int lane = threadIdx.x & 63;
  float b = lane < nch ? ws.mx[row * kMaxCh + lane] : -INFINITY, m = lane < nch ? ws.mn[row * kMaxCh + lane] : INFINITY;
  int bi = lane < nch ? ws.mi[row * kMaxCh + lane] : 0x7fffffff;
  wave_pick(b, bi);
  m = -wave_max(-m);
  RowScale r;
  r.mx = b;
  r.mi = bi;
  r.c = 1.4426950408889634f / temp;  // exp2 domain
  const float range = (b - m) * r.c;
  r.scale = range > 0.f && range < 31.9f ? (kMBins - 1) / range : 64.f;
  return r;
}

template <typename T>
__global__ void __launch_bounds__(kChThreads) samp_hist_kernel(const T* __restrict__ logits, int V, int chunk,
                                                               SampArgs a, int row0, SampWs ws) {
  __shared__ unsigned long long mass[kMBins];
  __shared__ uint32_t cnt[kMBins];
  const int row = blockIdx.y;
  const SampRow rp = samp_row(a, row0 + row);
  const bool hk = rp.k > 0 && rp.k < V, hp = rp.p < 1.f;
  if (!(rp.temp > 0.f) || !(hk || hp)) return;
  const RowScale rs = row_scale(ws, row, gridDim.x, rp.temp);
  for (int i = threadIdx.x; i < kMBins; i += kChThreads) { mass[i] = 0; cnt[i] = 0; }
  __syncthreads();
  const int c0 = blockIdx.x * chunk;
  each_in(logits + (size_t)row * V, c0, min(V, c0 + chunk), [&](int, float v) {
    const int b = rs.bin(v);
    if (hp) atomicAdd(&mass[b], rs.weight(v));
    if (hk) atomicAdd(&cnt[b], 1u);
  });
  __syncthreads();
  for (int i = threadIdx.x; i < kMBins; i += kChThreads) {
    if (mass[i]) atomicAdd(&ws.mass[row * kMBins + i], mass[i]);
    if (cnt[i]) atomicAdd(&ws.cnt[row * kMBins + i], cnt[i]);
  }
}

// Where a row's cuts lie: tokens of bins below `all` are kept, those of bins all .. last and of bin `bk` (the one
// the k-th token is in; kMBins: no top-k) are listed.
struct RowCut {
  int all, last, bk;
};
// pm / pc [kMBins]: mass and count of the bins ahead of each; every thread of NT calls it
template <int NT>
__device__ __forceinline__ RowCut row_cut(const SampWs& ws, int row, const SampRow& rp, bool hk, bool hp,
                                          unsigned long long* pm, uint32_t* pc, unsigned long long* wm, uint32_t* wc,
                                          RowCut* out) {
  constexpr int PER = kMBins / NT, NW = NT / 64;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  unsigned long long m[PER], sm = 0;
  uint32_t n[PER], sn = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    m[i] = hp ? ws.mass[row * kMBins + t * PER + i] : 0;
    n[i] = hk ? ws.cnt[row * kMBins + t * PER + i] : 0;
    sm += m[i];
    sn += n[i];
  }
  unsigned long long im = sm;
  uint32_t in = sn;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long y = __shfl_up(im, o, 64);
    const uint32_t z = __shfl_up(in, o, 64);
    if (lane >= o) { im += y; in += z; }
  }
  if (lane == 63) { wm[wv] = im; wc[wv] = in; }
  if (t == 0) *out = RowCut{0, kMBins - 1, hk ? kMBins - 1 : kMBins};
  __syncthreads();
  unsigned long long bm = im - sm, tot = 0;
  uint32_t bn = in - sn;
  for (int w = 0; w < NW; ++w) {
    if (w < wv) { bm += wm[w]; bn += wc[w]; }
    tot += wm[w];
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int b = t * PER + i;
    pm[b] = bm;
    pc[b] = bn;
    if (hk && bn < (uint32_t)rp.k && bn + n[i] >= (uint32_t)rp.k) out->bk = b;
    bm += m[i];
    bn += n[i];
  }
  __syncthreads();
  RowCut r = *out;
  __syncthreads();
  const bool lim = hp && tot > 0 && rp.p > 0.f;  // an empty mass restricts nothing
  if (lim) {
    // the kept set's mass lies between that of the bins ahead of bk and that with bk
    const double lo = (double)rp.p * (double)(hk ? pm[r.bk] : tot);
    const double hi = (double)rp.p * (double)(hk && r.bk + 1 < kMBins ? pm[r.bk + 1] : tot);
    // bins whose tokens are wholly under a target: a prefix of them
    int nlo = 0, nhi = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int b = t * PER + i;
      const double incl = (double)(b + 1 < kMBins ? pm[b + 1] : tot);
      nlo += incl < lo;
      nhi += incl < hi;
    }
    if (t == 0) { out->all = 0; out->last = 0; }
    __syncthreads();
    atomicAdd(&out->all, nlo);
    atomicAdd(&out->last, nhi);
    __syncthreads();
    r.all = out->all;
    r.last = min(out->last, kMBins - 1);
    r.all = min(r.all, min(r.bk, r.last));
    r.last = min(r.last, r.bk);
  } else {
    r.all = hk ? r.bk : kMBins;
    r.last = r.all - (hk ? 0 : 1);
  }
  return r;
}

template <typename T>
__global__ void __launch_bounds__(kChThreads) samp_pick_kernel(const T* __restrict__ logits, int V, int chunk,
                                                               SampArgs a, int row0, SampWs ws) {
  __shared__ unsigned long long pm[kMBins], wm[4];
  __shared__ uint32_t pc[kMBins], wc[4];
  __shared__ RowCut cut;
  __shared__ float sv[4];
  __shared__ int si[4];
  const int row = blockIdx.y, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const SampRow rp = samp_row(a, row0 + row);
  if (!(rp.temp > 0.f)) return;
  const bool hk = rp.k > 0 && rp.k < V, hp = rp.p < 1.f;
  const RowScale rs = row_scale(ws, row, gridDim.x, rp.temp);
  RowCut r{kMBins, kMBins - 1, kMBins};
  if (hk || hp) r = row_cut<kChThreads>(ws, row, rp, hk, hp, pm, pc, wm, wc, &cut);
  const float inv_t = 1.f / rp.temp;
  float gb = -INFINITY;
  int gi = 0x7fffffff;
  const int c0 = blockIdx.x * chunk;
  each_in(logits + (size_t)row * V, c0, min(V, c0 + chunk), [&](int i, float v) {
    const int b = hk || hp ? rs.bin(v) : 0;
    if (b < r.all) {
      pick(gb, gi, gumbel_score(v, inv_t, rp.seed, rp.step, i), i);
    } else if (b <= r.last || b == r.bk) {
      const uint32_t at = atomicAdd(&ws.nlist[row], 1u);
      if (at < kListCap) ws.list[row * kListCap + at] = ((unsigned long long)okey(v) << 32) | (uint32_t)i;
    }
  });
  wave_pick(gb, gi);
  if (lane == 0) { sv[wv] = gb; si[wv] = gi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kChThreads / 64; ++w) pick(gb, gi, sv[w], si[w]);
    ws.gv[row * kMaxCh + blockIdx.x] = gb;
    ws.gi[row * kMaxCh + blockIdx.x] = gi;
  }
}

template <typename T>
__global__ void __launch_bounds__(kSampThreads) samp_final_kernel(const T* __restrict__ logits,
                                                                  int64_t* __restrict__ out, int V, int nch,
                                                                  SampArgs a, int row0, SampWs ws) {
  __shared__ union {
    SampScratch slow;
    struct {
      unsigned long long pm[kMBins], wm[16], w[kListCap], above[kListCap], zk;
      uint32_t pc[kMBins], wc[16], key[kListCap], idx[kListCap], more[kListCap];
      uint16_t bin[kListCap];
      RowCut cut;
      float red[16];
      int redi[16];
    } f;
  } sh;
  const int row = blockIdx.x, t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const SampRow rp = samp_row(a, row0 + row);
  const bool hk = rp.k > 0 && rp.k < V, hp = rp.p < 1.f;
  if (rp.temp > 0.f && (hk || hp) && ws.nlist[row] > kListCap) {
    const int id = topkp_row(logits + (size_t)row * V, V, rp, sh.slow);
    if (t == 0) out[row] = id;
    return;
  }
  const RowScale rs = row_scale(ws, row, nch, rp.temp);
  if (!(rp.temp > 0.f)) {
    if (t == 0) out[row] = rs.mi < V ? rs.mi : 0;
    return;
  }
  float gb = lane < nch ? ws.gv[row * kMaxCh + lane] : -INFINITY;
  int gi = lane < nch ? ws.gi[row * kMaxCh + lane] : 0x7fffffff;
  if (hk || hp) {
    const int n = (int)ws.nlist[row];
    row_cut<kSampThreads>(ws, row, rp, hk, hp, sh.f.pm, sh.f.pc, sh.f.wm, sh.f.wc, &sh.f.cut);
    const int bk = [&] {  // row_cut leaves it in place
      __syncthreads();
      return sh.f.cut.bk;
    }();
    unsigned long long tot = 0;
    for (int w = 0; w < kSampThreads / 64; ++w) tot += sh.f.wm[w];
    for (int i = t; i < n; i += kSampThreads) {
      const unsigned long long e = ws.list[row * kListCap + i];
      const float v = key2f((uint32_t)(e >> 32));
      sh.f.key[i] = (uint32_t)(e >> 32);
      sh.f.idx[i] = (uint32_t)e;
      sh.f.bin[i] = (uint16_t)rs.bin(v);
      sh.f.w[i] = rs.weight(v);
      sh.f.above[i] = 0;
      sh.f.more[i] = 0;
    }
    if (t == 0) sh.f.zk = 0;
    __syncthreads();
    // mass and count of the tokens above each listed one in its bin: the workgroup's threads over (token, part)
    if (n > 0) {
      const int parts = max(1, kSampThreads / n), i = t % n, part = t / n;
      if (part < parts) {
        const uint32_t key = sh.f.key[i];
        const uint16_t bin = sh.f.bin[i];
        unsigned long long m = 0;
        uint32_t c = 0;
        for (int j = part; j < n; j += parts)
          if (sh.f.bin[j] == bin && sh.f.key[j] > key) { m += sh.f.w[j]; ++c; }
        if (m) atomicAdd(&sh.f.above[i], m);
        if (c) atomicAdd(&sh.f.more[i], c);
      }
    }
    __syncthreads();
    const bool in = t < n;
    const int b = in ? sh.f.bin[t] : 0;
    const bool keep_k = in && (!hk || sh.f.pc[b] + sh.f.more[t] < (uint32_t)rp.k);
    if (hk && keep_k && b == bk) atomicAdd(&sh.f.zk, sh.f.w[t]);
    __syncthreads();
    const unsigned long long z = hk ? sh.f.pm[bk] + sh.f.zk : tot;
    const bool lim = hp && tot > 0 && rp.p > 0.f;
    if (keep_k && (!lim || (double)(sh.f.pm[b] + sh.f.above[t]) < (double)rp.p * (double)z))
      pick(gb, gi, gumbel_score(key2f(sh.f.key[t]), 1.f / rp.temp, rp.seed, rp.step, (int)sh.f.idx[t]),
           (int)sh.f.idx[t]);
  }
  wave_pick(gb, gi);
  __syncthreads();
  if (lane == 0) { sh.f.red[wv] = gb; sh.f.redi[wv] = gi; }
  __syncthreads();
  if (t == 0) {
    for (int w = 1; w < kSampThreads / 64; ++w) pick(gb, gi, sh.f.red[w], sh.f.redi[w]);
    out[row] = gi < V ? gi : (rs.mi < V ? rs.mi : 0);
  }
}

}  // namespace mx

using namespace mx;

static int samp_chunks(int V) { return std::min(kMaxCh, (V + 4095) / 4096); }
static bool samp_split(int V) { return V >= kSplitV && V <= kSplitMaxV; }

// bytes of workspace of one call of mx_sample_rows / mx_sample_list
extern "C" int64_t mx_sample_rows_ws(int B, int V) {
  if (!samp_split(V)) return 0;
  const int64_t rows = std::min(B, kSampGroup);
  return rows * (kMBins * 12 + kListCap * 8 + kMaxCh * 20 + 8);
}

template <typename T>
static void samp_launch(const T* x, int64_t* out, int B, int V, const SampArgs& a, int row0, char* w,
                        hipStream_t stream) {
  if (!samp_split(V)) {
    SampArgs o = a;
    if (o.temps) {
      o.temps += row0; o.ps += row0; o.ks += row0; o.seeds += row0; o.steps += row0;
    }
    sample_topkp_kernel<T><<<B, kSampThreads, 0, stream>>>(x, out, V, o);
    return;
  }
  const size_t R = B;
  SampWs ws;
  ws.mass = (unsigned long long*)w;
  ws.list = ws.mass + R * kMBins;
  ws.cnt = (uint32_t*)(ws.list + R * kListCap);
  ws.mx = (float*)(ws.cnt + R * kMBins);
  ws.mn = ws.mx + R * kMaxCh;
  ws.gv = ws.mn + R * kMaxCh;
  ws.mi = (int*)(ws.gv + R * kMaxCh);
  ws.gi = ws.mi + R * kMaxCh;
  ws.nlist = (uint32_t*)(ws.gi + R * kMaxCh);
  const int nch0 = samp_chunks(V), chunk = ((V + nch0 - 1) / nch0 + 7) / 8 * 8, nch = (V + chunk - 1) / chunk;
  const dim3 grid(nch, B);
  samp_stats_kernel<T><<<grid, kChThreads, 0, stream>>>(x, V, chunk, ws);
  samp_hist_kernel<T><<<grid, kChThreads, 0, stream>>>(x, V, chunk, a, row0, ws);
  samp_pick_kernel<T><<<grid, kChThreads, 0, stream>>>(x, V, chunk, a, row0, ws);
  samp_final_kernel<T><<<B, kSampThreads, 0, stream>>>(x, out, V, nch, a, row0, ws);
}

// logits [B, V] bf16 (is_bf16) or f32; per-row parameters (device arrays of B):
// temperature f32 (<= 0: greedy), top_p f32 (>= 1: off), top_k i32 (<= 0: off),
// seed i64, step i32.  out ids [B] int64.  ws: mx_sample_rows_ws(B, V) bytes.
extern "C" int mx_sample_rows(const void* logits, int is_bf16, int64_t* out, int B, int V, const float* temps,
                              const float* top_ps, const int32_t* top_ks, const int64_t* seeds, const int32_t* steps,
                              void* ws, hipStream_t stream) {
  if (B <= 0) return 0;
  if (V <= 0 || !temps || (samp_split(V) && !ws)) return -1;
  SampArgs a{temps, top_ps, top_ks, seeds, steps, {}};
  const int step = samp_split(V) ? kSampGroup : B;  // one workgroup a row: all rows at once
  for (int r = 0; r < B; r += step) {
    const int n = std::min(step, B - r);
    if (is_bf16) samp_launch((const uint16_t*)logits + (size_t)r * V, out + r, n, V, a, r, (char*)ws, stream);
    else samp_launch((const float*)logits + (size_t)r * V, out + r, n, V, a, r, (char*)ws, stream);
  }
  return (int)hipGetLastError();
}

// the same with the parameters in host arrays of B: they travel with the launches, kSampGroup rows at a time
extern "C" int mx_sample_list(const void* logits, int is_bf16, int64_t* out, int B, int V, const double* temps,
                              const double* top_ps, const int64_t* top_ks, const int64_t* seeds, const int64_t* steps,
                              void* ws, hipStream_t stream) {
  if (B <= 0) return 0;
  if (V <= 0 || (samp_split(V) && !ws)) return -1;
  for (int r = 0; r < B; r += kSampGroup) {
    const int n = std::min(kSampGroup, B - r);
    SampArgs a{};
    for (int i = 0; i < n; ++i)
      a.rows[i] = SampRow{(float)temps[r + i], (float)top_ps[r + i],
                          (int)std::max<int64_t>(0, std::min<int64_t>(top_ks[r + i], 0x7fffffff)),
                          (uint32_t)seeds[r + i], (uint32_t)steps[r + i]};
    if (is_bf16) samp_launch((const uint16_t*)logits + (size_t)r * V, out + r, n, V, a, 0, (char*)ws, stream);
    else samp_launch((const float*)logits + (size_t)r * V, out + r, n, V, a, 0, (char*)ws, stream);
  }
  return (int)hipGetLastError();
}
