// Retention over whole prompts (retention_chunk.hip: the runs and the three launches) on the bf16 matrix cores, for bf16 storage,
// heads of 64 or 128 that are rotated whole.  What is f32 there - rotated q and k, scores, decay powers, state - stays f32 here: each
// factor is split into three bf16 pieces whose sum it is (8 bits each of the 24), and a product of two is the six of its nine
// products that are not below 2^-26 of it; v is bf16 as it comes.  The smaller products are added up among themselves or first, so
// a sum has fewer roundings at its full size than the f32 instruction's: against 64 bits states are off by 1.2e-7 of their size (2.9e-7
// there), and 0.016 % of the outputs are not the nearest bf16 (0.034 %).  A factor that is infinite has NaN for its smaller pieces, and
// one beside it zeros: a run's sum that is not finite is that of the largest pieces, an output row that comes out NaN is
// formed again in f32 (rm_row), so that infinite and zero products are what they are.
// Heads of 128, 32 of them, 2048 tokens, us: ends 62 -> 18, out 104 -> 50; heads of 64 with states and carry 72 -> 39.
#include "gemm8_core.h"
#include "hybrid.h"
#include "sublayer.h"

namespace mx {

typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int kRetRun = 256, kRetBlock = 128;  // rows of a run, of a block (the tables that the caller gives)

__device__ __forceinline__ f32x16 rm_mfma(const u16x8& a, const u16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_g, a), __builtin_bit_cast(bf16x8_g, b), c, 0, 0, 0);
}

// x = p[0] + p[1] + p[2]
__device__ __forceinline__ void rm_split(const float (&x)[8], u16x8 (&p)[3]) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  uint32_t o[3][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float a = x[2 * j], b = x[2 * j + 1];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
      o[i][j] = u;
      a -= __builtin_bit_cast(float, u << 16);
      b -= __builtin_bit_cast(float, u & 0xffff0000u);
    }
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) p[i] = __builtin_bit_cast(u16x8, make_uint4(o[i][0], o[i][1], o[i][2], o[i][3]));
}
typedef float rm_f2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ rm_f2 rm_rd2(uint32_t base, int off) {  // floats off, off + 1
  rm_f2 v;
  asm volatile("ds_read2_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(v) : "v"(base), "i"(off), "i"(off + 1));
  return v;
}

// LDS byte offsets of 16-byte chunk c of row r, rows of W values: for fragments read along the rows, and across them (transposed)
template <int W>
__device__ __forceinline__ uint32_t rm_along(int r, int c) {
  return r * 2 * W + 16 * (c ^ (W == 128 ? r & 15 : (r >> 1) & 7));
}
template <int W>
__device__ __forceinline__ uint32_t rm_across(int r, int c) {
  return r * 2 * W + 16 * (c ^ (W == 128 ? (r & 3) << 2 : (r << 1) & 4));
}
// lane part of a transposed read: of columns 32 b .. + 31 the lane's, four rows from K0 (lane >> 5) on
template <int W, int K0>
__device__ __forceinline__ uint32_t rm_tr(int lane, int b) {
  const int h = lane >> 5, q = (lane & 15) >> 2, p = lane & 3;
  return rm_across<W>(K0 * h + q, 4 * b + 2 * ((lane >> 4) & 1) + (p >> 1)) + 8 * (p & 1);
}
__device__ __forceinline__ u16x8 rm_whole(const u16x4& x, const u16x4& y) {
  return u16x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
}
__device__ __forceinline__ void rm_sync() {  // LDS stores and DMA of this wave are there, then the others' are
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// eight pairs of a k row: values d .. d + 7 and those D / 2 on
template <int D>
struct RmKey {
  u16x8 lo, hi;
  float c[8], s[8];
  __device__ __forceinline__ void load(const uint16_t* xr, int d) {
    lo = *reinterpret_cast<const u16x8*>(xr + d);
    hi = *reinterpret_cast<const u16x8*>(xr + d + D / 2);
  }
  __device__ __forceinline__ void turn(const float* cr, const float* sr) {
    ldv<4>(cr, reinterpret_cast<float(&)[4]>(c[0]));
    ldv<4>(cr + 4, reinterpret_cast<float(&)[4]>(c[4]));
    ldv<4>(sr, reinterpret_cast<float(&)[4]>(s[0]));
    ldv<4>(sr + 4, reinterpret_cast<float(&)[4]>(s[4]));
  }
  template <bool MASK>
  __device__ __forceinline__ void pieces(float sc, bool on, u16x8 (&pl)[3], u16x8 (&ph)[3]) const {
    float l[8], h[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float x0 = bf2f(lo[j]), x1 = bf2f(hi[j]);
      l[j] = (x0 * c[j] - x1 * s[j]) * sc;
      h[j] = (x1 * c[j] + x0 * s[j]) * sc;
      if (MASK && !on) l[j] = h[j] = 0.f;
    }
    rm_split(l, pl);
    rm_split(h, ph);
  }
};

// rows r0 .. r0 + R of W bf16 columns to LDS by the DMA of NW waves, `across` or `along`; rows from n on are zeros
template <int W, int R, int NW, bool ACROSS>
__device__ __forceinline__ void rm_rows(const __amdgpu_buffer_rsrc_t& rs, int64_t ld, int r0, int n, int w, int lane, char* dst) {
  constexpr int PR = 512 / W, PIECES = R / PR / NW;  // rows, pieces of a wave
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int r = (w * PIECES + i) * PR + lane / (W / 8), cc = lane % (W / 8);
    const int c = ACROSS ? cc ^ (W == 128 ? (r & 3) << 2 : (r << 1) & 4) : cc ^ (W == 128 ? r & 15 : (r >> 1) & 7);
    const uint32_t so = r0 + r < n ? (uint32_t)(((r0 + r) * ld + 8 * c) * 2) : G8_OOB;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (g8lptr_t)(dst + (w * PIECES + i) * 1024), 16, so, 0, 0, 0);
  }
}

// ------------------------------------------------------------------ run sums
// Bound by the chain of a workgroup, one a CU: 64 rows wait for their k and v, are rotated and split, and multiplied while the next
// ones come; the products are a seventh of the time.
// wave w: rows 32 (w % (D / 32)) .. of D, half w / (D / 32) of E
template <int D, int E>
__global__ void __launch_bounds__(4 * D, 1) retention_ends_mfma_kernel(RetentionChunks a) {
  constexpr int R = 64, NW = D / 16, EB = E / 64, KB = R * D * 2, BUF = 3 * KB + R * E * 2;
  __shared__ __attribute__((aligned(1024))) char sm[2 * BUF];
  __shared__ float pw[kRetRun + 1];
  const int4 ch = reinterpret_cast<const int4*>(a.chunks)[blockIdx.y];  // (first row, rows, position, -)
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int db = w % (D / 32), eh = w / (D / 32);
  const int64_t HD = (int64_t)a.H * D;
  const uint16_t* xk = reinterpret_cast<const uint16_t*>(a.x) + ch.x * a.ldx + HD + (int64_t)h * D;
  const uint16_t* xv = reinterpret_cast<const uint16_t*>(a.x) + ch.x * a.ldx + 2 * HD + (int64_t)h * E;
  const __amdgpu_buffer_rsrc_t vrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)xv, 0, (uint32_t)(((ch.y - 1) * a.ldx + E) * 2), 0x00020000);
  const float ksc = 1.f / sqrtf((float)D);
  const int r = tid / (D / 16), d = tid % (D / 16) * 8;
  RmKey<D> key;
  auto load = [&](int j0) __attribute__((always_inline)) {
    const int j = min(j0 + r, ch.y - 1);
    key.load(xk + j * a.ldx, d);
    key.turn(a.cosb + (int64_t)(ch.z + j) * (D / 2) + d, a.sinb + (int64_t)(ch.z + j) * (D / 2) + d);
  };
  auto stage = [&](int j0, char* b) __attribute__((always_inline)) {
    u16x8 pl[3], ph[3];
    const bool on = j0 + r < ch.y;
    key.template pieces<true>(ksc * pw[max(ch.y - 1 - j0 - r, 0)], on, pl, ph);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      *reinterpret_cast<u16x8*>(b + i * KB + rm_across<D>(r, d / 8)) = pl[i];
      *reinterpret_cast<u16x8*>(b + i * KB + rm_across<D>(r, d / 8 + D / 16)) = ph[i];
    }
  };
  rm_rows<E, R, NW, true>(vrs, a.ldx, 0, ch.y, w, lane, sm + 3 * KB);
  load(0);
  for (int i = tid; i <= kRetRun; i += 4 * D) pw[i] = a.pw[(int64_t)h * (kRetRun + 1) + i];
  rm_sync();
  stage(0, sm);
  rm_sync();
  const uint32_t lds0 = lds_addr(sm), ka = lds0 + rm_tr<D, 8>(lane, db);
  uint32_t va[EB];
#pragma unroll
  for (int j = 0; j < EB; ++j) va[j] = lds0 + 3 * KB + rm_tr<E, 8>(lane, eh * EB + j);
  f32x16 acc[EB] = {}, low[EB] = {};
  int st = 0;
  for (int j0 = 0; j0 < ch.y; j0 += R, st ^= 1) {
    const bool more = j0 + R < ch.y;
    if (more) {
      rm_rows<E, R, NW, true>(vrs, a.ldx, j0 + R, ch.y, w, lane, sm + (st ^ 1) * BUF + 3 * KB);
      load(j0 + R);
    }
    __builtin_amdgcn_sched_barrier(0);
    u16x4 tk[2][3][2], tv[2][EB][2];
    auto read = [&](int t, int b) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < EB; ++j) {
        tv[b][j][0] = trd_off(va[j] + st * BUF, t * 16 * 2 * E);
        tv[b][j][1] = trd_off(va[j] + st * BUF, (t * 16 + 4) * 2 * E);
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        tk[b][i][0] = trd_off(ka + st * BUF, i * KB + t * 16 * 2 * D);
        tk[b][i][1] = trd_off(ka + st * BUF, i * KB + (t * 16 + 4) * 2 * D);
      }
    };
    read(0, 0);
#pragma unroll
    for (int t = 0; t < R / 16; ++t) {
      const int b = t & 1;
      lds_wait();
#pragma unroll
      for (int j = 0; j < EB; ++j) pin(tv[b][j][0]), pin(tv[b][j][1]);
#pragma unroll
      for (int i = 0; i < 3; ++i) pin(tk[b][i][0]), pin(tk[b][i][1]);
      if (t + 1 < R / 16) read(t + 1, b ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      u16x8 k[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) k[i] = rm_whole(tk[b][i][0], tk[b][i][1]);
#pragma unroll
      for (int j = 0; j < EB; ++j) {
        const u16x8 v = rm_whole(tv[b][j][0], tv[b][j][1]);
        low[j] = rm_mfma(k[2], v, low[j]);
        low[j] = rm_mfma(k[1], v, low[j]);
        acc[j] = rm_mfma(k[0], v, acc[j]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (more) stage(j0 + R, sm + (st ^ 1) * BUF);
    rm_sync();
  }
  float* u = a.ws + ((int64_t)blockIdx.y * a.H + h) * D * E;
#pragma unroll
  for (int j = 0; j < EB; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i)
      u[(32 * db + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3)) * E + 32 * (eh * EB + j) + (lane & 31)] =
          acc[j][i] + (__builtin_isfinite(acc[j][i]) ? low[j][i] : 0.f);
}

// ------------------------------------------------------------------ outputs
// Row i of a run by one wave in f32, for rows that hold what is not finite; pw: powers of the decay.  Lane l has dims and channels l and
// l + 64.  Nothing is stored where all is NaN, as it is already.
template <int D, int E>
__device__ __forceinline__ void rm_row(const RetentionChunks& a, const int4& ch, int run, int h, int i, const float* pw, int lane) {
  constexpr int ND = D / 64, NE = E / 64;
  const int64_t HD = (int64_t)a.H * D, HE = (int64_t)a.H * E;
  const uint16_t* x = reinterpret_cast<const uint16_t*>(a.x) + ch.x * a.ldx;
  auto turned = [&](const uint16_t* xr, int j, float (&o)[ND]) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < ND; ++n) {
      const int d = lane + 64 * n, f = d % (D / 2);
      const float c = a.cosb[(int64_t)(ch.z + j) * (D / 2) + f], s = a.sinb[(int64_t)(ch.z + j) * (D / 2) + f];
      const float u = bf2f(xr[d]), v = bf2f(xr[d < D / 2 ? d + D / 2 : d - D / 2]);
      o[n] = d < D / 2 ? u * c - v * s : u * c + v * s;
    }
  };
  float q[ND], o[NE] = {};
  turned(x + i * a.ldx + (int64_t)h * D, i, q);
  auto lost = [&]() __attribute__((always_inline)) {  // sums that are NaN stay so
    bool all = true;
#pragma unroll
    for (int e = 0; e < NE; ++e) all = all && __builtin_isnan(o[e]);
    return __all(all);
  };
  if (ch.z > 0) {
    const float* S = a.ws + ((int64_t)run * a.H + h) * D * E + lane;
#pragma unroll
    for (int n = 0; n < ND; ++n)
      for (int d = 0; d < 64; ++d) {
        const float w = __shfl(q[n], d);
#pragma unroll
        for (int e = 0; e < NE; ++e) o[e] += w * S[(64 * n + d) * E + 64 * e];
      }
#pragma unroll
    for (int e = 0; e < NE; ++e) o[e] *= pw[i + 1];
    if (lost()) return;
  }
  const float ksc = 1.f / sqrtf((float)D);
  for (int j = 0; j <= i; ++j) {
    float k[ND], p = 0.f;
    turned(x + j * a.ldx + HD + (int64_t)h * D, j, k);
#pragma unroll
    for (int n = 0; n < ND; ++n) p += q[n] * (k[n] * ksc);
    p = wave_sum(p) * pw[i - j];
#pragma unroll
    for (int e = 0; e < NE; ++e) o[e] += p * bf2f(x[j * a.ldx + 2 * HD + (int64_t)h * E + lane + 64 * e]);
    if (lost()) return;
  }
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < NE; ++e) ss += o[e] * o[e];
  const float rs = 1.f / sqrtf(wave_sum(ss) / (float)E + a.eps);
  uint16_t* y = reinterpret_cast<uint16_t*>(a.y) + (ch.x + i) * HE + (int64_t)h * E + lane;
#pragma unroll
  for (int e = 0; e < NE; ++e)
    y[64 * e] = f2bf(o[e] * rs * silu_t<uint16_t>(bf2f(x[i * a.ldx + 2 * HD + HE + (int64_t)h * E + lane + 64 * e])));
}

// A wave has 32 rows of a block of 128, transposed: scores are keys x rows and outputs channels x rows, so that a row is a lane, and
// the scores of a tile, split, are the next product's operand where they are.  The pieces of q stay in registers (of heads of 128 some
// in LDS: what was spilled waited, with the loads ahead of it, in every tile), k is split once for the workgroup.
// What bounds it: two waves a SIMD with 31 thousand cycles of matrix instructions and as many of others, splits foremost, at 1.8 GHz,
// which this load clocks down to; 70 % of the time that both take after each other.  A run's two blocks with their rows dealt out so
// that both have 18 of the 36 tiles lose to the order (50 -> 55): both then stage nearly all keys.
template <int D, int E>
__global__ void __launch_bounds__(256, 2) retention_out_mfma_kernel(RetentionChunks a) {
  constexpr int R = 32, KS = D / 16, EB = E / 32, KB = R * D * 2, VB = R * E * 2;
  constexpr int BUF = 3 * KB + VB > kRetBlock * E * 2 ? 3 * KB + VB : kRetBlock * E * 2, PAD = 32;
  static_assert(3 * VB <= BUF, "the state's pieces");
  __shared__ __attribute__((aligned(1024))) char sm[2 * BUF];
  // the smallest pieces of the first QL fragments of q, which have no registers
  constexpr int QL = D == 128 && E == 128 ? 3 : 0;
  __shared__ __attribute__((aligned(16))) u16x8 ql[QL ? QL : 1][256];
  __shared__ float pw[PAD + kRetRun + 1];  // powers of the decay, ahead of them zeros: keys past a row
  // a run's second block, which has twice the keys, and its first one after each other on one XCD, which fill a CU
  const int at = (blockIdx.x >> 4) * 8 + (blockIdx.x & 7), h = at % a.H, by = at / a.H * 2 + 1 - ((blockIdx.x >> 3) & 1);
  if (by >= a.nblocks) return;
  const int4 bl = reinterpret_cast<const int4*>(a.blocks)[by];  // (run, first row in it, -, -)
  const int4 ch = reinterpret_cast<const int4*>(a.chunks)[bl.x];
  const int i0 = bl.y, tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, g = lane >> 5, rows = min(kRetBlock, ch.y - i0);
  const int wr = 32 * ((i0 >> 7) & 1 ? 3 - w : w), top = i0 + wr;  // the wave's rows of the block; its first one of the run
  const int64_t HD = (int64_t)a.H * D, HE = (int64_t)a.H * E;
  const uint16_t* x = reinterpret_cast<const uint16_t*>(a.x) + ch.x * a.ldx;
  const uint16_t *xk = x + HD + (int64_t)h * D, *xv = x + 2 * HD + (int64_t)h * E;
  const uint32_t span = (uint32_t)(((ch.y - 1) * a.ldx + E) * 2);
  const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void*)xv, 0, span, 0x00020000);
  const __amdgpu_buffer_rsrc_t grs = __builtin_amdgcn_make_buffer_rsrc((void*)(xv + HE), 0, span, 0x00020000);
  for (int i = tid; i < PAD + kRetRun + 1; i += 256) pw[i] = i < PAD ? 0.f : a.pw[(int64_t)h * (kRetRun + 1) + i - PAD];
  const float ksc = 1.f / sqrtf((float)D);

  const int kr = tid / (D / 16), kd = tid % (D / 16) * 8;  // (a head of 64: half of the threads)
  const bool keys = R * D / 16 == 256 || tid < R * D / 16;
  RmKey<D> key;
  auto krow = [&](int j0) { return min(j0 + kr, ch.y - 1); };
  auto load = [&](int j0) __attribute__((always_inline)) {
    if (keys) key.load(xk + krow(j0) * a.ldx, kd);
  };
  auto turn = [&](int j0) __attribute__((always_inline)) {
    const int64_t f = (int64_t)(ch.z + krow(j0)) * (D / 2) + kd;
    if (keys) key.turn(a.cosb + f, a.sinb + f);
  };
  auto stage = [&](int j0, char* b) __attribute__((always_inline)) {
    if (!keys) return;
    u16x8 pl[3], ph[3];
    key.template pieces<false>(ksc, true, pl, ph);  // (keys past the run are past every row that is stored)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      *reinterpret_cast<u16x8*>(b + i * KB + rm_along<D>(kr, kd / 8)) = pl[i];
      *reinterpret_cast<u16x8*>(b + i * KB + rm_along<D>(kr, kd / 8 + D / 16)) = ph[i];
    }
  };

  u16x8 qp[KS][3];  // row c, dims 16 s + 8 g ..
  {
    const int qr = min(top + c, ch.y - 1);  // rows past the run are not stored
    const uint16_t* xq = x + qr * a.ldx + (int64_t)h * D + 8 * g;
    const int64_t f = (int64_t)(ch.z + qr) * (D / 2) + 8 * g;
#pragma unroll
    for (int s = 0; s < KS / 2; ++s) {
      RmKey<D> q;
      q.load(xq, 16 * s);
      q.turn(a.cosb + f + 16 * s, a.sinb + f + 16 * s);
      q.template pieces<false>(1.f, true, qp[s], qp[s + KS / 2]);
      if (s < QL) ql[s][tid] = qp[s][2];
    }
  }
  const uint32_t lds0 = lds_addr(sm), qa = lds_addr(ql) + tid * 16;
  f32x16 acc[EB] = {};  // channels 32 e + 8 (i >> 2) + 4 g + (i & 3) of row c
  if (ch.z > 0) {       // a state ahead of this run
    constexpr int PT = R * E / 8 / 256;  // groups of 8 channels of a thread
    const float* S = a.ws + ((int64_t)bl.x * a.H + h) * D * E;
    float sv[PT][8];
    auto sload = [&](int d0) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < PT; ++i) {
        ldv<4>(S + d0 * E + (i * 256 + tid) * 8, reinterpret_cast<float(&)[4]>(sv[i][0]));
        ldv<4>(S + d0 * E + (i * 256 + tid) * 8 + 4, reinterpret_cast<float(&)[4]>(sv[i][4]));
      }
    };
    auto sstage = [&](char* b) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < PT; ++i) {
        const int at = i * 256 + tid;
        u16x8 p[3];
        rm_split(sv[i], p);
#pragma unroll
        for (int j = 0; j < 3; ++j) *reinterpret_cast<u16x8*>(b + j * VB + rm_across<E>(at / (E / 8), at % (E / 8))) = p[j];
      }
    };
    sload(0);
    sstage(sm);
    rm_sync();
#pragma unroll
    for (int t = 0; t < D / R; ++t) {
      if (t + 1 < D / R) sload((t + 1) * R);
      else load(0), turn(0);
      __builtin_amdgcn_sched_barrier(0);
      u16x4 ts[2][3][2];
      u16x8 q2[2];
      if (2 * t < QL) q2[0] = rd128_off(qa, 2 * t * 4096);
      if (2 * t + 1 < QL) q2[1] = rd128_off(qa, (2 * t + 1) * 4096);
      auto read = [&](int n) __attribute__((always_inline)) {
        const uint32_t sa = lds0 + (t & 1) * BUF + rm_tr<E, 8>(lane, n >> 1);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          ts[n & 1][i][0] = trd_off(sa, i * VB + 16 * (n & 1) * 2 * E);
          ts[n & 1][i][1] = trd_off(sa, i * VB + (16 * (n & 1) + 4) * 2 * E);
        }
      };
      read(0);
      f32x16 low;
#pragma unroll
      for (int n = 0; n < 2 * EB; ++n) {
        const int e = n >> 1;
        lds_wait();
        u16x8 sp[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          pin(ts[n & 1][i][0]), pin(ts[n & 1][i][1]);
          sp[i] = rm_whole(ts[n & 1][i][0], ts[n & 1][i][1]);
        }
        if (n < 2 && 2 * t + n < QL) pin(q2[n]);
        if (n + 1 < 2 * EB) read(n + 1);
        __builtin_amdgcn_sched_barrier(0);
        const u16x8 q[3] = {qp[2 * t + (n & 1)][0], qp[2 * t + (n & 1)][1], 2 * t + (n & 1) < QL ? q2[n & 1] : qp[2 * t + (n & 1)][2]};
        // the smaller products of a tile add up by themselves
        low = rm_mfma(sp[2], q[0], n & 1 ? low : f32x16{});
        low = rm_mfma(sp[0], q[2], low);
        low = rm_mfma(sp[1], q[1], low);
        low = rm_mfma(sp[1], q[0], low);
        low = rm_mfma(sp[0], q[1], low);
        acc[e] = rm_mfma(sp[0], q[0], acc[e]);
        __builtin_amdgcn_sched_barrier(0);
        if (n & 1) acc[e] += low;
      }
      __builtin_amdgcn_sched_barrier(0);
      if (t + 1 < D / R) {
        sstage(sm + ((t + 1) & 1) * BUF);
        rm_sync();
      }
    }
    const float f = pw[PAD + min(top + c + 1, kRetRun)];
#pragma unroll
    for (int e = 0; e < EB; ++e) acc[e] *= f;
  } else {
    load(0), turn(0);
    rm_sync();  // (the powers)
  }
  // buffer 0: the last tile of the state was in 1
  rm_rows<E, R, 4, true>(vrs, a.ldx, 0, ch.y, w, lane, sm + 3 * KB);
  stage(0, sm);
  rm_sync();
  uint32_t va[EB];
#pragma unroll
  for (int e = 0; e < EB; ++e) va[e] = lds0 + 3 * KB + rm_tr<E, 4>(lane, e);
  const uint32_t ka = lds0 + rm_along<D>(c, g), pa = lds_addr(pw);
  const int last = min(i0 + kRetBlock, ch.y);
  int st = 0;
  for (int j0 = 0; j0 < last; j0 += R, st ^= 1) {
    const bool more = j0 + R < last;
    char* next = sm + (st ^ 1) * BUF;
    const bool on = j0 <= top + 31;  // keys past its last row count for none
    f32x16 sc = {};
    rm_f2 wt[8];
    const int back = top + c - j0 - 4 * g;  // of score i: back - 8 (i >> 2) - (i & 3)
    if (on) {
      // the smaller products first, of all dims, then the largest
      u16x8 kf[2][3], q2[2];
      auto read = [&](int s, int b, int n) __attribute__((always_inline)) {
        const uint32_t at = (ka ^ (32 * s)) + st * BUF;
#pragma unroll
        for (int i = 0; i < n; ++i) kf[b][i] = rd128_off(at, i * KB);
        if (n == 3 && s < QL) q2[b] = rd128_off(qa, s * 4096);
      };
      read(0, 0, 3);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int b = s & 1;
        lds_wait();
#pragma unroll
        for (int i = 0; i < 3; ++i) pin(kf[b][i]);
        if (s < QL) pin(q2[b]);
        if (s + 1 < KS) read(s + 1, b ^ 1, 3);
        else read(0, b ^ 1, 1);
        __builtin_amdgcn_sched_barrier(0);
        sc = rm_mfma(kf[b][2], qp[s][0], sc);
        sc = rm_mfma(kf[b][0], s < QL ? q2[b] : qp[s][2], sc);
        sc = rm_mfma(kf[b][1], qp[s][1], sc);
        sc = rm_mfma(kf[b][1], qp[s][0], sc);
        sc = rm_mfma(kf[b][0], qp[s][1], sc);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int b = s & 1;
        lds_wait();
        pin(kf[b][0]);
        if (s + 1 < KS) {
          read(s + 1, b ^ 1, 1);
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) wt[i] = rm_rd2(pa + 4 * (PAD + back - 27), 26 - 8 * (i >> 1) - 2 * (i & 1));
        }
        __builtin_amdgcn_sched_barrier(0);
        sc = rm_mfma(kf[b][0], qp[s][0], sc);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (more) {
      rm_rows<E, R, 4, true>(vrs, a.ldx, j0 + R, ch.y, w, lane, next + 3 * KB);
      load(j0 + R);
      turn(j0 + R);
    } else {  // this wave's gates
      rm_rows<E, 32, 1, false>(grs, a.ldx, top, ch.y, 0, lane, next + w * 32 * E * 2);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (on) {
      lds_wait();
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        asm volatile("" : "+v"(wt[i]));
        sc[2 * i] *= wt[i][1];
        sc[2 * i + 1] *= wt[i][0];
      }
      if (j0 == top) {  // (zeros already, unless a later key's score is not finite)
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] = back >= 8 * (i >> 2) + (i & 3) ? sc[i] : 0.f;
      }
      u16x4 tv[2][2];
      auto read = [&](int n) __attribute__((always_inline)) {  // channels n % EB, keys 16 (n / EB) ..
        tv[n & 1][0] = trd_off(va[n % EB] + st * BUF, 16 * (n / EB) * 2 * E);
        tv[n & 1][1] = trd_off(va[n % EB] + st * BUF, (16 * (n / EB) + 8) * 2 * E);
      };
      read(0);
      u16x8 pp[3];
#pragma unroll
      for (int n = 0; n < 2 * EB; ++n) {
        if (n % EB == 0) {
          float p[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) p[i] = sc[8 * (n / EB) + i];
          rm_split(p, pp);
        }
        lds_wait();
        pin(tv[n & 1][0]), pin(tv[n & 1][1]);
        const u16x8 v = rm_whole(tv[n & 1][0], tv[n & 1][1]);
        if (n + 1 < 2 * EB) read(n + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 2; i >= 0; --i) acc[n % EB] = rm_mfma(v, pp[i], acc[n % EB]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more) {
      stage(j0 + R, next);
      rm_sync();
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the gates
  char* gb = sm + st * BUF + w * 32 * E * 2;
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < EB; ++e)
#pragma unroll
    for (int i = 0; i < 16; ++i) ss += acc[e][i] * acc[e][i];
  ss += __shfl_xor(ss, 32);
  const float rs = 1.f / sqrtf(ss / (float)E + a.eps);
#pragma unroll
  for (int e = 0; e < EB; ++e)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u16x4* p = reinterpret_cast<u16x4*>(gb + rm_along<E>(c, 4 * e + i) + 8 * g);
      const u16x4 gt = *p;
      u16x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = f2bf(acc[e][4 * i + j] * rs * silu_t<uint16_t>(bf2f(gt[j])));
      *p = o;
    }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wave reads its own rows back, whole
  __builtin_amdgcn_wave_barrier();
  uint16_t* y = reinterpret_cast<uint16_t*>(a.y) + (ch.x + top) * HE + (int64_t)h * E;
#pragma unroll
  for (int i = 0; i < 32 * E / 512; ++i) {
    const int at = i * 64 + lane, r = at / (E / 8), cc = at % (E / 8);
    if (wr + r < rows) *reinterpret_cast<u16x8*>(y + r * HE + 8 * cc) = *reinterpret_cast<const u16x8*>(gb + rm_along<E>(r, cc));
  }
  const int ln = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));  // (lane: not kept through the kernel for this)
  uint32_t again = (uint32_t)__ballot(wr + (ln & 31) < rows && __builtin_isnan(ss));
  if (again) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // those rows are stored a second time
  for (; again; again &= again - 1) rm_row<D, E>(a, ch, bl.x, h, top + __builtin_ctz(again), pw + PAD, ln);
}

}  // namespace mx

using namespace mx;

// Whatever the length: 100 tokens of 32 heads of 128 take 25 us with carry and both launches, 50 with the f32 instruction, 1 + 700 +
// 32 tokens of 4 heads 33 and 69, 8192 of 32 heads of 64 120 and 221.
extern "C" int mx_retention_mfma_takes(const RetentionChunks* p, int f32) {
  const RetentionChunks& a = *p;
  return !f32 && (a.D == 64 || a.D == 128) && (a.E == 64 || a.E == 128) && a.rd == a.D && a.ldx % 8 == 0 && a.ldx < 1 << 22 &&
         (((uintptr_t)a.x | (uintptr_t)a.y | (uintptr_t)a.cosb | (uintptr_t)a.sinb | (uintptr_t)a.ws) & 15) == 0;
}

#define RM(K, ...)                                                                      \
  do {                                                                                  \
    if (a.D == 64) { if (a.E == 64) K<64, 64> __VA_ARGS__; else K<64, 128> __VA_ARGS__; } \
    else { if (a.E == 64) K<128, 64> __VA_ARGS__; else K<128, 128> __VA_ARGS__; }         \
  } while (0)

extern "C" void mx_retention_mfma_ends(const RetentionChunks* p, hipStream_t stream) {
  const RetentionChunks& a = *p;
  RM(retention_ends_mfma_kernel, <<<dim3(a.H, a.nchunks), 4 * a.D, 0, stream>>>(a));
}

extern "C" void mx_retention_mfma_out(const RetentionChunks* p, hipStream_t stream) {
  const RetentionChunks& a = *p;
  RM(retention_out_mfma_kernel, <<<((a.nblocks + 1) / 2 * a.H + 7) / 8 * 16, 256, 0, stream>>>(a));
}
