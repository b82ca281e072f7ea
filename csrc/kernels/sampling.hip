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
// Split form (vocabularies of kSplitV and more): three launches over (chunk, row), so a step's few rows fill the
// chip.  One workgroup a row kept 32 of 256 CUs on six to nine passes whose LDS atomics and logarithms bound it:
// 253 us for 32 rows of 128,256 bf16 logits of mixed parameters, where the three launches take 27 us a call behind one
// another (all top-p 28, all top-k 23, temperature alone 20.5; one row 19 - 21), of which the host's part is 21.  With
// lane shuffles for folds and scans, the last bin's atomics on one address, and the kept tokens scored on the lanes
// that hold them it was 32 (32 / 26 / 20.5; one row 23 - 25): see each.  What bounds them now (us within a call, stamped): stats
// 2.5, of which loads 0.8; a launch's gap 1.3 - 2; hist 8, of which parameters and partials 1.6, LDS atomics of 64 bits on
// random banks 3.7, the sums to memory 2; pick 12.5: loads 1.6, scan of bins and cuts 2.1, tokens 2.4, the row's list
// and counter 2.7, and its last workgroup's comparisons 3.
//  * stats: a chunk's largest (with its index) and smallest logit;
//  * hist: masses exp2((x - max) log2e / T) and counts in 2048 bins, linear in the exponent (64 bins a power of
//    two, finer where the row's whole range is under 32 of them).  A bin holds all tokens of a value, so bins
//    order tokens as their logits do.  Masses are summed as integers (2^-42): any order gives the same sums.
//    Rows without cuts compete here already;
//  * pick: the bins where top-k and top-p cross, from the sums; tokens ahead of them compete at once, those
//    inside are listed (a value or two: tens to hundreds of tokens), the rest is dropped.  A row's last workgroup has
//    exact counts and masses above each listed token; the kept ones compete with the chunks' winners.
// One workgroup of 1,024 threads a CU: each clears, adds up and scans 2,048 bins, so that four times as many of 256
// threads took 61 us for the 32 mixed rows (a global counter asked for each listed token, and a fourth launch with a
// scan of its own for the listed ones, were the other half of that).
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
    wave_pick(b, i);
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
    z = wave_sum(z);
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
// Shorter rows: one workgroup, one launch.  32 top-p rows of 8,191: 30 us against 41 split when that was four launches;
// of 32,768: about 80 (its time grows with the row) against 27 now.
constexpr int kSplitV = 16384;
constexpr int kSplitMaxV = (1 << 22) - 1;  // as many masses of up to 2^42 stay below 2^64
constexpr int kMBins = 2048;
constexpr int kMaxCh = 64;         // chunks a row (= one wave over their partials)
constexpr int kListCap = 1024;     // listed tokens a row
constexpr int kChThreads = 1024;
constexpr int kNearCap = 2048;     // tokens of a chunk above its row's cut that are dealt out evenly

// A token that only exact sums decide about, with the mass and count of the bins ahead of its own.
struct Listed {
  unsigned long long id, pm;  // id: key << 32 | index
  uint32_t pc, pad;
};
struct RowInfo {
  unsigned long long tot, pmk;  // mass of the row; of the bins ahead of the one the k-th token is in
  int bk;                       // that bin
};

struct SampWs {
  unsigned long long* mass;  // [rows, kMBins]
  Listed* list;              // [rows, kListCap]
  uint32_t* cnt;             // [rows, kMBins]
  float *mx, *mn, *gv;       // [rows, kMaxCh]: largest, smallest finite logit; best score among tokens kept at once
  int *mi, *gi;              // their indexes
  uint32_t *nlist, *done;    // [rows]: listed tokens, workgroups that are through
};

__device__ __forceinline__ void pick(float& b, int& i, float ov, int oi) {
  if (ov > b || (ov == b && oi < i)) { b = ov; i = oi; }
}

// [c0, c1) of a row by 16-B loads, two pieces of 8 a thread and turn; rows of any alignment (an odd vocabulary
// shifts every row) have their first and last few values apart
template <typename T>
struct Chunk {
  const T* x;
  int c0, c1, head, ve;
  struct Pieces {
    u16x8 u, v;
    __device__ __forceinline__ float at(int j) const { return bf2f(j < 8 ? u[j & 7] : v[j & 7]); }
  };
  struct Pieces32 {
    f32x4 u[2], v[2];
    __device__ __forceinline__ float at(int j) const { return j < 8 ? u[(j >> 2) & 1][j & 3] : v[(j >> 2) & 1][j & 3]; }
  };
  using P = std::conditional_t<sizeof(T) == 2, Pieces, Pieces32>;
  static constexpr int S = kChThreads * 8;

  __device__ __forceinline__ Chunk(const T* row, int a, int b) : x(row), c0(a), c1(b) {
    head = min(c1, c0 + (int)((16 - ((uintptr_t)(x + c0) & 15)) & 15) / (int)sizeof(T));
    ve = head + (c1 - head) / 8 * 8;
  }
  __device__ __forceinline__ int start() const { return head + (int)threadIdx.x * 8; }
  // pieces at b and, where the chunk has it, b + S (else the first again)
  __device__ __forceinline__ P load(int b) const {
    const T *p = x + b, *q = x + (b + S < ve ? b + S : b);
    P r;
    if constexpr (sizeof(T) == 2) {
      r.u = *reinterpret_cast<const u16x8*>(p), r.v = *reinterpret_cast<const u16x8*>(q);
    } else {
      r.u[0] = *reinterpret_cast<const f32x4*>(p), r.u[1] = *reinterpret_cast<const f32x4*>(p + 4);
      r.v[0] = *reinterpret_cast<const f32x4*>(q), r.v[1] = *reinterpret_cast<const f32x4*>(q + 4);
    }
    return r;
  }
  // the thread's values outside the pieces: f(index, value)
  template <typename F>
  __device__ __forceinline__ void ends(F&& f) const {
    const int t = threadIdx.x;
    auto one = [&](int c) {
      if constexpr (sizeof(T) == 2) f(c, bf2f(x[c]));
      else f(c, x[c]);
    };
    if (c0 + t < head) one(c0 + t);
    if (ve + t < c1) one(ve + t);
  }
  __device__ __forceinline__ P first() const {
    P p = {};
    if (start() < ve) p = load(start());
    return p;
  }
  template <typename F>
  __device__ __forceinline__ void each(F&& f) const {
    each(first(), f);
  }
  template <typename F>
  __device__ __forceinline__ void each(P p, F&& f) const {
    ends(f);
    for (int b = start(); b < ve; b += 2 * S) {
      if (b != start()) p = load(b);
#pragma unroll
      for (int j = 0; j < 8; ++j) f(b + j, p.at(j));
      if (b + S < ve) {
#pragma unroll
        for (int j = 8; j < 16; ++j) f(b + S + j - 8, p.at(j));
      }
    }
  }
};

// thread 0's (b, i): the best of the workgroup
__device__ __forceinline__ void group_pick(float& b, int& i, float* sv, int* si) {
  wave_pick(b, i);
  if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = b; si[threadIdx.x >> 6] = i; }
  __syncthreads();
  if (threadIdx.x < 64) {
    static_assert(kChThreads / 64 == 16, "a wave's best each: one row of lanes");
    b = sv[threadIdx.x & 15];
    i = si[threadIdx.x & 15];
    row_pick(b, i);
  }
}

template <typename T>
__global__ void __launch_bounds__(kChThreads) samp_stats_kernel(const T* __restrict__ logits, int V, int chunk,
                                                                SampWs ws) {
  __shared__ float sv[kChThreads / 64], sm[kChThreads / 64];
  __shared__ int si[kChThreads / 64];
  const int row = blockIdx.y, nch = gridDim.x, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int i = blockIdx.x * kChThreads + threadIdx.x; i < kMBins; i += nch * kChThreads) {
    ws.mass[row * kMBins + i] = 0;
    ws.cnt[row * kMBins + i] = 0;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) ws.nlist[row] = ws.done[row] = 0;
  const int c0 = blockIdx.x * chunk;
  const Chunk<T> ch(logits + (size_t)row * V, c0, min(V, c0 + chunk));
  const typename Chunk<T>::P first = ch.first();
  // two comparisons a token: where the largest lies is looked for by the waves that hold it, and the smallest finite one
  // again by those that have an infinity
  float b = -INFINITY, m = INFINITY;
  ch.each(first, [&](int, float v) {
    b = v > b ? v : b;
    m = v < m ? v : m;
  });
  if (__ballot(m == -INFINITY)) {
    m = INFINITY;
    ch.each(first, [&](int, float v) { m = v < m && v > -INFINITY ? v : m; });
  }
  b = wave_max(b);
  m = -wave_max(-m);
  if (lane == 0) sv[wv] = b, sm[wv] = m;
  __syncthreads();
  const float top = row_max(sv[lane & 15]);
  int bi = 0x7fffffff;
  if (b == top) {
    ch.each(first, [&](int i, float v) { bi = v == top && i < bi ? i : bi; });
    bi = wave_min(bi);
  }
  if (lane == 0) si[wv] = bi;
  __syncthreads();
  if (threadIdx.x < 64) {
    bi = row_min(si[lane & 15]);
    m = -row_max(-sm[lane & 15]);
  }
  if (threadIdx.x == 0) {
    b = top;
    ws.mx[row * kMaxCh + blockIdx.x] = b;
    ws.mi[row * kMaxCh + blockIdx.x] = bi;
    ws.mn[row * kMaxCh + blockIdx.x] = m;
  }
}

// what the bins of a row are made of; every lane of a wave calls it
struct RowScale {
  float mx, c, cs;
  int mi;
  __device__ __forceinline__ int bin(float v) const {  // not-a-numbers: the first (med3 is the least of the others then)
    return (int)__builtin_amdgcn_fmed3f((mx - v) * cs, 0.f, (float)(kMBins - 1));
  }
  // exp2((v - mx) c) in 2^-42, cut off: the power's mantissa where 1 has its own, moved down by its exponent (32 top-p
  // rows are bound by these instructions: a float's two conversions and their difference are half as many again).  What
  // is not a number has the largest exponent, and like zero moves past the end.
  __device__ __forceinline__ unsigned long long weight(float v) const {
    const uint32_t b = __float_as_uint(__builtin_amdgcn_exp2f((v - mx) * c));
    const uint32_t down = min(127u - (b >> 23), 63u);  // (no sign)
    return ((unsigned long long)((b & 0x7fffffu) | 0x800000u) << 19) >> down;
  }
};
struct RowParts {  // its chunks' statistics, one a lane
  float b, m;
  int bi;
  __device__ __forceinline__ RowParts(const SampWs& ws, int row, int nch) {
    const int lane = threadIdx.x & 63, at = row * kMaxCh + min(lane, nch - 1);  // (the last again: it changes nothing)
    b = ws.mx[at], m = ws.mn[at], bi = ws.mi[at];
  }
};
__device__ __forceinline__ RowScale row_scale(RowParts p, float temp) {
  float b = p.b, m = p.m;
  int bi = p.bi;
  wave_pick(b, bi);
  m = -wave_max(-m);
  b = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(b)));
  m = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(m)));
  bi = __builtin_amdgcn_readfirstlane(bi);
  RowScale r;
  r.mx = b;
  r.mi = bi;
  r.c = 1.4426950408889634f / temp;  // exp2 domain
  const float range = (b - m) * r.c;
  r.cs = r.c * (range > 0.f && range < 31.9f ? (kMBins - 1) / range : 64.f);
  return r;
}

template <typename T>
__global__ void __launch_bounds__(kChThreads) samp_hist_kernel(const T* __restrict__ logits, int V, int chunk,
                                                               SampArgs a, int row0, SampWs ws) {
  __shared__ unsigned long long mass[kMBins];
  __shared__ uint32_t cnt[kMBins];
  __shared__ float sv[kChThreads / 64];
  __shared__ int si[kChThreads / 64];
  const int row = blockIdx.y;
  const int c0 = blockIdx.x * chunk;
  const Chunk<T> ch(logits + (size_t)row * V, c0, min(V, c0 + chunk));
  const typename Chunk<T>::P first = ch.first();  // on its way, like the statistics, with the row's parameters
  const RowParts parts(ws, row, gridDim.x);
  __builtin_amdgcn_sched_barrier(0);
  const SampRow rp = samp_row(a, row0 + row);
  const bool hk = rp.k > 0 && rp.k < V, hp = rp.p < 1.f;
  if (!(rp.temp > 0.f)) return;
  if (!(hk || hp)) {  // every token competes: nothing to wait for
    const float inv_t = 1.f / rp.temp;
    float gb = -INFINITY;
    int gi = 0x7fffffff;
    ch.each(first, [&](int i, float v) { pick(gb, gi, gumbel_score(v, inv_t, rp.seed, rp.step, i), i); });
    group_pick(gb, gi, sv, si);
    if (threadIdx.x == 0) {
      ws.gv[row * kMaxCh + blockIdx.x] = gb;
      ws.gi[row * kMaxCh + blockIdx.x] = gi;
    }
    return;
  }
  for (int i = threadIdx.x; i < kMBins; i += kChThreads) { mass[i] = 0; cnt[i] = 0; }
  const RowScale rs = row_scale(parts, rp.temp);
  __syncthreads();
  // the last bin holds all that lies further away than it: a sixth of a row at a low temperature, whose atomics on one
  // address held a workgroup up for 5 us.  Its sums are the threads' own first.
  unsigned long long fm = 0;
  uint32_t fc = 0;
  ch.each(first, [&](int, float v) {
    const int b = rs.bin(v);
    const unsigned long long w = hp ? rs.weight(v) : 0;
    if (b == kMBins - 1) {
      fm += w;
      ++fc;
    } else {
      if (hp) atomicAdd(&mass[b], w);
      if (hk) atomicAdd(&cnt[b], 1u);
    }
  });
  if (__ballot(fc != 0)) {
    fm = wave_scan(fm);
    fc = wave_scan(fc);
    if ((threadIdx.x & 63) == 63) {
      if (hp) atomicAdd(&mass[kMBins - 1], fm);
      if (hk) atomicAdd(&cnt[kMBins - 1], fc);
    }
  }
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
  unsigned long long klo, khi;  // mass of the bins ahead of bk, and with it
};
// a thread's bins
struct Bins {
  static constexpr int PER = kMBins / kChThreads;
  unsigned long long m[PER];
  uint32_t n[PER];
  __device__ __forceinline__ Bins(const SampWs& ws, int row) {  // (zero where the row has no such cut)
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      m[i] = ws.mass[row * kMBins + threadIdx.x * PER + i];
      n[i] = ws.cnt[row * kMBins + threadIdx.x * PER + i];
    }
  }
};
// pm / pc [kMBins]: mass and count of the bins ahead of each; every thread calls it
__device__ __forceinline__ RowCut row_cut(const Bins& bins, const SampRow& rp, bool hk, bool hp,
                                          unsigned long long* pm, uint32_t* pc, unsigned long long* wm, uint32_t* wc,
                                          RowCut* out, unsigned long long& tot) {
  constexpr int PER = Bins::PER, NW = kChThreads / 64;
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const auto &m = bins.m;
  const auto &n = bins.n;
  unsigned long long sm = 0;
  uint32_t sn = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) sm += m[i], sn += n[i];
  const unsigned long long im = wave_scan(sm);
  const uint32_t in = wave_scan(sn);
  if (lane == 63) { wm[wv] = im; wc[wv] = in; }
  if (t == 0) *out = RowCut{0, 0, hk ? kMBins - 1 : kMBins, 0, 0};
  __syncthreads();
  const unsigned long long vm = wave_scan(lane < NW ? wm[lane] : 0ull);
  const uint32_t vn = wave_scan(lane < NW ? wc[lane] : 0u);
  tot = lane_value(vm, NW - 1);
  unsigned long long bm = im - sm + (wv ? lane_value(vm, wv - 1) : 0);
  uint32_t bn = in - sn + (wv ? (uint32_t)__builtin_amdgcn_readlane((int)vn, wv - 1) : 0);
  const unsigned long long bm0 = bm;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int b = t * PER + i;
    pm[b] = bm;
    pc[b] = bn;
    if (hk && bn < (uint32_t)rp.k && bn + n[i] >= (uint32_t)rp.k) {
      out->bk = b;
      out->klo = bm;
      out->khi = bm + m[i];
    }
    bm += m[i];
    bn += n[i];
  }
  __syncthreads();
  RowCut r = *out;
  const bool lim = hp && tot > 0 && rp.p > 0.f;  // an empty mass restricts nothing
  if (lim) {
    // the kept set's mass lies between that of the bins ahead of bk and that with bk; the bin that brings the mass
    // to p of either: no bin ahead of it does
    const double lo = (double)rp.p * (double)(hk ? r.klo : tot);
    const double hi = (double)rp.p * (double)(hk ? r.khi : tot);
    bm = bm0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const double excl = (double)bm, incl = (double)(bm + m[i]);
      if (excl < lo && incl >= lo) out->all = t * PER + i;
      if (excl < hi && incl >= hi) out->last = t * PER + i;
      bm += m[i];
    }
    __syncthreads();
    r.all = out->all;
    r.last = out->last;
    r.all = min(r.all, min(r.bk, r.last));
    r.last = min(r.last, r.bk);
  } else {
    r.all = hk ? r.bk : kMBins;
    r.last = r.all - (hk ? 0 : 1);
  }
  return r;
}

// Values that another workgroup of the same launch reads: written through to and read from where all XCDs see them, so
// that no fence has to write a whole L2 back (with a fence on each side 32 top-p rows took 69 us instead of 33).
template <typename T>
__device__ __forceinline__ void put_shared(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T get_shared(T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The listed tokens of a row (thread t: the t-th of n <= kListCap) against the exact counts and masses above them;
// those that stay compete with (gb, gi), every wave's best so far.
struct FinalScratch {
  struct {
    uint32_t key, bin;
    unsigned long long w;
  } e[kListCap];
  unsigned long long above[kListCap], zk;
  uint32_t more[kListCap];
};
__device__ __forceinline__ void final_listed(const Listed& e, int n, const RowScale& rs, const RowInfo& info,
                                             const SampRow& rp, bool hk, bool hp, FinalScratch& f, float& gb, int& gi) {
  const int t = threadIdx.x;
  const bool in = t < n;
  const float v = key2f((uint32_t)(e.id >> 32));
  const int b = rs.bin(v);
  const unsigned long long w = rs.weight(v);
  if (in) {
    f.e[t] = {(uint32_t)(e.id >> 32), (uint32_t)b, w};
    f.above[t] = 0;
    f.more[t] = 0;
  }
  if (t == 0) f.zk = 0;
  __syncthreads();
  // mass and count of the tokens above each listed one in its bin: the workgroup's threads over (token, part)
  const int parts = kChThreads / n, i = t % n, part = t / n;
  if (part < parts) {
    const uint32_t key = f.e[i].key, bin = f.e[i].bin;
    unsigned long long m = 0;
    uint32_t c = 0;
#pragma unroll 4
    for (int j = part; j < n; j += parts) {
      const auto o = f.e[j];
      const bool over = o.bin == bin && o.key > key;
      m += over ? o.w : 0;
      c += over;
    }
    if (m) atomicAdd(&f.above[i], m);
    if (c) atomicAdd(&f.more[i], c);
  }
  __syncthreads();
  const bool keep_k = in && (!hk || e.pc + f.more[t] < (uint32_t)rp.k);
  if (hk) {
    if (keep_k && b == info.bk) atomicAdd(&f.zk, w);
    __syncthreads();
  }
  const unsigned long long z = hk ? info.pmk + f.zk : info.tot;
  const bool lim = hp && info.tot > 0 && rp.p > 0.f;
  if (keep_k && (!lim || (double)(e.pm + f.above[t]) < (double)rp.p * (double)z))
    pick(gb, gi, gumbel_score(v, 1.f / rp.temp, rp.seed, rp.step, (int)(uint32_t)e.id), (int)(uint32_t)e.id);
}

// Picks over a row's chunks; the workgroup that comes last to a row's counter, with all of its lists in memory, ends
// it (rows without cuts: the first chunk's, from what the launches before left).
template <typename T>
__global__ void __launch_bounds__(kChThreads) samp_pick_kernel(const T* __restrict__ logits, int64_t* __restrict__ out,
                                                               int V, int chunk, SampArgs a, int row0, SampWs ws) {
  __shared__ union {
    struct {
      unsigned long long pm[kMBins], wm[kChThreads / 64], own[kListCap];
      uint32_t pc[kMBins], wc[kChThreads / 64];
      uint2 near[kNearCap];
      RowCut cut;
    } c;
    FinalScratch f;
    SampScratch slow;
  } sh;
  static_assert(kSampThreads == kChThreads && kListCap == kChThreads, "one workgroup shape; a thread a listed token");
  __shared__ uint32_t nown, nnear, at0, last;
  __shared__ float sv[kChThreads / 64];
  __shared__ int si[kChThreads / 64];
  const int row = blockIdx.y, nch = gridDim.x, t = threadIdx.x, lane = t & 63;
  const T* x = logits + (size_t)row * V;
  const int c0 = blockIdx.x * chunk;
  const Chunk<T> ch(x, c0, min(V, c0 + chunk));
  const Bins bins(ws, row);  // on their way, like the statistics and the first logits, with the row's parameters
  const RowParts parts(ws, row, nch);
  typename Chunk<T>::P p = ch.first();
  __builtin_amdgcn_sched_barrier(0);
  const SampRow rp = samp_row(a, row0 + row);
  const bool hk = rp.k > 0 && rp.k < V, hp = rp.p < 1.f, cutting = rp.temp > 0.f && (hk || hp);
  if (!cutting && blockIdx.x) return;
  const RowScale rs = row_scale(parts, rp.temp);
  auto end = [&](float gb, int gi) {  // thread 0
    out[row] = gi < V ? gi : (rs.mi < V ? rs.mi : 0);
  };
  if (!cutting) {
    float gb = lane < nch && rp.temp > 0.f ? ws.gv[row * kMaxCh + lane] : -INFINITY;
    int gi = lane < nch && rp.temp > 0.f ? ws.gi[row * kMaxCh + lane] : 0x7fffffff;
    wave_pick(gb, gi);
    if (t == 0) end(gb, gi);
    return;
  }
  if (t == 0) nown = nnear = 0;
  RowInfo info;
  const RowCut r = row_cut(bins, rp, hk, hp, sh.c.pm, sh.c.pc, sh.c.wm, sh.c.wc, &sh.c.cut, info.tot);
  info.pmk = r.klo;
  info.bk = r.bk;
  const float inv_t = 1.f / rp.temp;
  float gb = -INFINITY;
  int gi = 0x7fffffff;
  auto token = [&](int i, float v) {
    const int b = rs.bin(v);
    if (b < r.all) {
      pick(gb, gi, gumbel_score(v, inv_t, rp.seed, rp.step, i), i);
    } else if (b <= r.last || b == r.bk) {
      const uint32_t n = atomicAdd(&nown, 1u);
      if (n < kListCap) sh.c.own[n] = ((unsigned long long)okey(v) << 32) | (uint32_t)i;
    }
  };
  // Most tokens lie further from the largest than the last bin that counts reaches: a difference and a comparison
  // mark the others (and not-a-numbers).  Those are few and uneven, three or four on one lane of a wave and none on
  // most: they are gathered, and then scored by all threads alike.  What does not fit goes one a lane and turn.
  const int lim = max(max(r.last, hk ? r.bk : 0), r.all - 1);
  const float far = lim >= kMBins - 1 ? INFINITY : (float)(lim + 1) / rs.cs * 1.0001f + 1e-30f;
  ch.ends(token);
  for (int at = ch.start(); at - lane * 8 < ch.ve; at += 2 * ch.S) {  // whole waves, for the sums over lanes
    if (at != ch.start() && at < ch.ve) p = ch.load(at);
    uint32_t near = 0;
#pragma unroll
    for (int j = 0; j < 16; ++j) near |= !(rs.mx - p.at(j) > far) ? 1u << j : 0u;
    near &= at >= ch.ve ? 0u : at + ch.S >= ch.ve ? 0xffu : 0xffffu;
    const uint32_t c = __builtin_popcount(near), upto = wave_scan(c);
    const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)upto, 63);
    if (!all) continue;
    uint32_t from = 0;
    if (lane == 0) from = atomicAdd(&nnear, all);
    from = (uint32_t)__builtin_amdgcn_readfirstlane((int)from);
    if (from + all <= kNearCap) {
      uint2* q = sh.c.near + from + upto - c;
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (near >> j & 1) *q++ = {__float_as_uint(p.at(j)), (uint32_t)(at + (j & 7) + (j & 8 ? ch.S : 0))};
      continue;
    }
    for (uint32_t q = from + lane; q < kNearCap; q += 64) sh.c.near[q] = {0u, ~0u};  // (asked for, and not used)
    for (; near; near &= near - 1) {
      const int j = __builtin_ctz(near);
      float v = p.at(0);
#pragma unroll
      for (int k = 1; k < 16; ++k) v = j == k ? p.at(k) : v;
      token(at + (j & 7) + (j & 8 ? ch.S : 0), v);
    }
  }
  __syncthreads();
  for (uint32_t q = t, n = min(nnear, (uint32_t)kNearCap); q < n; q += kChThreads) {
    const uint2 e = sh.c.near[q];
    if (e.y != ~0u) token((int)e.y, __uint_as_float(e.x));
  }
  group_pick(gb, gi, sv, si);  // its barrier: the workgroup's list is whole
  const uint32_t mine = nown;
  if (t == 0) {
    put_shared(&ws.gv[row * kMaxCh + blockIdx.x], gb);
    put_shared(&ws.gi[row * kMaxCh + blockIdx.x], gi);
    at0 = mine ? atomicAdd(&ws.nlist[row], mine) : 0;
  }
  if (mine) {
    __syncthreads();
    if (t < mine && at0 + t < kListCap) {
      const unsigned long long id = sh.c.own[t];
      const int b = rs.bin(key2f((uint32_t)(id >> 32)));
      Listed* l = ws.list + row * kListCap + at0 + t;
      put_shared(&l->id, id);
      put_shared(&l->pm, sh.c.pm[b]);
      put_shared(&l->pc, sh.c.pc[b]);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every wave: what it wrote is where all XCDs see it
  __syncthreads();
  if (t == 0) last = atomicAdd(&ws.done[row], 1u) == (uint32_t)nch - 1;
  __syncthreads();
  if (!last) return;
  const int n = (int)get_shared(&ws.nlist[row]);
  Listed* l = ws.list + row * kListCap + t;  // asked for with its count: past it, used by no one
  const Listed e{get_shared(&l->id), get_shared(&l->pm), get_shared(&l->pc), 0};
  gb = lane < nch ? get_shared(&ws.gv[row * kMaxCh + lane]) : -INFINITY;
  gi = lane < nch ? get_shared(&ws.gi[row * kMaxCh + lane]) : 0x7fffffff;
  if (n > kListCap) {
    const int id = topkp_row(x, V, rp, sh.slow);
    if (t == 0) out[row] = id;
    return;
  }
  if (n > 0) final_listed(e, n, rs, info, rp, hk, hp, sh.f, gb, gi);
  group_pick(gb, gi, sv, si);
  if (t == 0) end(gb, gi);
}

}  // namespace mx

using namespace mx;

// Chunks of a row: as many workgroups of 1,024 threads as CUs over all rows, each with at least 8,192 logits (one
// 16-B piece a thread) and every chunk with a histogram of its own to clear, add up and scan.
static int samp_chunks(int B, int V) {
  return std::max(1, std::min({kMaxCh, (256 + B - 1) / B, (V + 8191) / 8192}));
}
static bool samp_split(int V) { return V >= kSplitV && V <= kSplitMaxV; }

// bytes of workspace of one call of mx_sample_rows / mx_sample_list
extern "C" int64_t mx_sample_rows_ws(int B, int V) {
  if (!samp_split(V)) return 0;
  const int64_t rows = std::min(B, kSampGroup);
  return rows * (kMBins * 12 + kListCap * (int64_t)sizeof(Listed) + kMaxCh * 20 + 8);
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
  ws.list = (Listed*)(ws.mass + R * kMBins);
  ws.cnt = (uint32_t*)(ws.list + R * kListCap);
  ws.mx = (float*)(ws.cnt + R * kMBins);
  ws.mn = ws.mx + R * kMaxCh;
  ws.gv = ws.mn + R * kMaxCh;
  ws.mi = (int*)(ws.gv + R * kMaxCh);
  ws.gi = ws.mi + R * kMaxCh;
  ws.nlist = (uint32_t*)(ws.gi + R * kMaxCh);
  ws.done = ws.nlist + R;
  const int nch0 = samp_chunks(B, V), chunk = ((V + nch0 - 1) / nch0 + 7) / 8 * 8, nch = (V + chunk - 1) / chunk;
  const dim3 grid(nch, B);
  samp_stats_kernel<T><<<grid, kChThreads, 0, stream>>>(x, V, chunk, ws);
  samp_hist_kernel<T><<<grid, kChThreads, 0, stream>>>(x, V, chunk, a, row0, ws);
  samp_pick_kernel<T><<<grid, kChThreads, 0, stream>>>(x, out, V, chunk, a, row0, ws);
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
