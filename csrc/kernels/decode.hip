// Inference-side kernels for gfx950:
//   * rope_append : decode-step q/k RoPE at per-sequence positions + KV-cache append
//   * decode_attn : single-token GQA attention over a per-slot KV cache,
//                   split over the sequence (flash-decoding), memory-bound:
//                   each workgroup streams 256 keys of one (seq, kv-head) once
//                   and serves all q-heads of that group (GQA reuse);
//   * decode_combine : merges the per-split (m, l, o) partials;
//   * sample : greedy argmax or exact temperature sampling via Gumbel-max with
//              a counter-based hash RNG (one pass, no softmax materialised).
// KV cache layout per layer: [slots, Hkv, max_seq, D] bf16 (contiguous per slot
// and head: one 256-B row per token for D = 128), or PAGED: a pool of blocks
// [blocks, Hkv, block, D] addressed through a per-slot block table (common.h
// kv_row; the block size is a multiple of the 256-key decode split, so every
// split reads one contiguous block).
#include "common.h"

namespace mx {

// qkv [B, (Hq+2Hkv)*D] -> q [B, Hq, D] (rotated), K/V cache rows at pos[b]
template <int D>
__global__ void __launch_bounds__(256) rope_append_kernel(const uint16_t* __restrict__ qkv,
                                                          const float* __restrict__ cosb,
                                                          const float* __restrict__ sinb,
                                                          const int32_t* __restrict__ pos,
                                                          const int32_t* __restrict__ slots,
                                                          uint16_t* __restrict__ q, uint16_t* __restrict__ kc,
                                                          uint16_t* __restrict__ vc, int B, int Hq, int Hkv,
                                                          int max_seq, const int32_t* __restrict__ bt, int maxb) {
  constexpr int HALF = D / 2, CPH = HALF / 8;
  const int NH = Hq + 2 * Hkv;
  const int64_t n = (int64_t)B * NH * CPH;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int cc = (int)(i % CPH);
    const int head = (int)((i / CPH) % NH);
    const int b = (int)(i / ((int64_t)CPH * NH));
    const int c = cc * 8;
    const int p = pos[b];
    const int slot = slots ? slots[b] : b;
    const uint16_t* src = qkv + (int64_t)b * NH * D + (int64_t)head * D;
    u16x8 x1 = *reinterpret_cast<const u16x8*>(src + c);
    u16x8 x2 = *reinterpret_cast<const u16x8*>(src + HALF + c);
    uint16_t* dst;
    if (head >= Hq + Hkv) {
      dst = vc + kv_row(bt, maxb, max_seq, slot, Hkv, head - Hq - Hkv, p) * D;
      *reinterpret_cast<u16x8*>(dst + c) = x1;
      *reinterpret_cast<u16x8*>(dst + HALF + c) = x2;
      continue;
    }
    dst = head < Hq ? q + ((int64_t)b * Hq + head) * D
                    : kc + kv_row(bt, maxb, max_seq, slot, Hkv, head - Hq, p) * D;
    const float* cp = cosb + (int64_t)p * HALF + c;
    const float* sp = sinb + (int64_t)p * HALF + c;
    u16x8 y1, y2;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float a = bf2f(x1[j]), bb = bf2f(x2[j]);
      y1[j] = f2bf(a * cp[j] - bb * sp[j]);
      y2[j] = f2bf(bb * cp[j] + a * sp[j]);
    }
    *reinterpret_cast<u16x8*>(dst + c) = y1;
    *reinterpret_cast<u16x8*>(dst + HALF + c) = y2;
  }
}

constexpr int kSplit = 256;  // keys per workgroup
constexpr int kMaxRep = 16;  // q-heads per kv-head supported

// ---------------------------------------------------------------------------
// Decode attention, heads of D = 128, 64 or 32.  Memory-bound: the
// whole point is to stream each (seq, kv-head)'s cached K/V rows once at HBM
// rate, so
//   * a workgroup = 4 waves = 256 keys of one (seq, kv-head); each wave owns 64
//     keys and keeps its own online-softmax state (no barrier in the key loop);
//   * scores for ALL q-heads of the GQA group at once with
//     v_mfma_f32_16x16x32_bf16: S^T[key][head] = K . Q^T, K rows loaded straight
//     from HBM into the A fragments (16 B per lane), Q^T (heads padded to 16)
//     as the B fragment;
//   * the S^T accumulator (head on the lane, keys in registers) converted to
//     bf16 IS the B operand of O^T[d][head] += V^T . P (keys permuted inside
//     each 32-key k-step to match the accumulator's row order).  D = 128: one
//     bf16 rounding of P.  D < 128: P as the sum of three bf16 (24 bits, what f32
//     holds) in three products, so the weights keep their f32 precision;
//   * V^T fragments come from a row-major V image in LDS through
//     ds_read_b64_tr_b16; the image is filled by LDS-DMA (global_load_lds,
//     source-swizzled so the transposed reads are conflict-free);
//   * the four waves' partials are merged through LDS (each wave reuses its own
//     V region) into one (m, l, o) partial per split, the format of
//     decode_combine_kernel; a single split is the output itself.
// D = 128: 64 KiB LDS and < 128 VGPRs: two workgroups (8 waves) per CU, 256 KiB of
// K/V in flight per CU.  D = 64, bound by latency at the few workgroups of a small
// batch: 32 q-heads of 8 kv-heads, one sequence of 700 keys 6.4 us; with one key a
// thread for the scores and a serial walk over the split's keys for the outputs 17.5.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(1))) const void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

__device__ __forceinline__ f32x4 mfma16(const u16x8& a, const u16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                 c, 0, 0, 0);
}

__device__ __forceinline__ u16x4 tr_read16(const char* p) {
  s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
  return __builtin_bit_cast(u16x4, v);
}

// 16-B chunk swizzle of a row of 2 D bytes: transposed reads take 32 B of each of 16 rows, and rows that start in
// the same bank take different pairs of chunks
template <int D>
__device__ __forceinline__ int dswz(int row) {
  if constexpr (D == 128) return ((row & 3) << 2) | ((row >> 2) & 3);
  else if constexpr (D == 64) return ((row >> 1) & 3) << 1;
  else return ((row >> 2) & 1) << 1;
}

// stores / loads of the split partials that another workgroup of the SAME launch merges:
// write-through (sc1, relaxed agent-scope atomic store), so no release fence (an L2
// write-back per workgroup) is needed, and loads that bypass this CU's L1 (guide
// §6 Guideline 16, the sc1 hand-off form)
// st: 0 = plain store, 1 = agent-scope relaxed atomic store (sc1 write-through),
// 2 = system-scope relaxed atomic store; ld: 0 = plain load, 1 = agent, 2 = system
__device__ __forceinline__ void st_part(float* p, float v, int st) {
  if (st == 1) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else if (st == 2) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  else *p = v;
}
__device__ __forceinline__ float ld_part(const float* p, int ld) {
  float* q = const_cast<float*>(p);
  if (ld == 1) return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (ld == 2) return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  return *p;
}

// one split of decode_attn_mfma_kernel: (m, l, o) partial of 256 keys for every
// q-head of the GQA group (see the kernel's header comment); out: the only split, and its output
template <int D>
__device__ __forceinline__ void decode_split_body(const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc,
                                                  const uint16_t* __restrict__ vc, float* __restrict__ part_o,
                                                  float* __restrict__ pml, char* smem, float (*mls)[2][16], int b,
                                                  int hk, int rep, int Hq, int split, int nsplit, int k_lo, int k_hi,
                                                  int slot, int max_seq, float sl, const int32_t* __restrict__ bt,
                                                  int maxb, int Hkv, int st, uint16_t* __restrict__ out) {
  constexpr int ROWB = 2 * D, CPR = D / 8, WKEYS = 64, WTILE = WKEYS * ROWB, KS = D / 32, DB = D / 16;
  constexpr int NP = D == 128 ? 1 : 3;  // bf16 parts of a weight
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int64_t kvb = (kv_row(bt, maxb, max_seq, slot, Hkv, hk, k_lo) - k_lo) * D;  // one block per split
  const uint16_t* kbase = kc + kvb;
  const uint16_t* vbase = vc + kvb;
  const int wk0 = k_lo + WKEYS * w;
  char* vs = smem + w * WTILE;

  // V rows of this wave -> LDS (D / 8 x 1-KiB lane-linear DMA pieces; swizzle by
  // permuting each lane's SOURCE chunk).  Rows past k_hi duplicate a valid row
  // (finite; their probabilities are exactly 0).
#pragma unroll
  for (int seg = 0; seg < CPR; ++seg) {
    const int row = seg * (64 / CPR) + lane / CPR, slt = lane % CPR;
    const int ch = slt ^ dswz<D>(row);
    const int key = min(wk0 + row, k_hi - 1);
    __builtin_amdgcn_global_load_lds((gptr_t)(vbase + (int64_t)key * D + ch * 8), (lptr_t)(vs + seg * 1024), 16, 0,
                                     0);
  }
  // Q^T fragments (B operand): lane (c, g) holds Q[head c][32 s + 8 g .. +7]
  u16x8 qf[KS];
  const uint16_t* qrow = q + ((int64_t)b * Hq + hk * rep + min(c, rep - 1)) * D;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    qf[s] = *reinterpret_cast<const u16x8*>(qrow + 32 * s + 8 * g);
    if (c >= rep) qf[s] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
  // K fragments (A operand), straight from HBM: block j, k-step s ->
  // K[wk0 + 16 j + c][32 s + 8 g .. +7]
  u16x8 kf[4][KS];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int key = min(wk0 + 16 * j + c, k_hi - 1);
#pragma unroll
    for (int s = 0; s < KS; ++s) kf[j][s] = *reinterpret_cast<const u16x8*>(kbase + (int64_t)key * D + 32 * s + 8 * g);
  }
  f32x4 sacc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    sacc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) sacc[j] = mfma16(kf[j][s], qf[s], sacc[j]);
  }
  // softmax over this wave's 64 keys, per head (= lane column c); lane (c, g)
  // holds keys wk0 + 16 j + 4 g + i
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = wk0 + 16 * j + 4 * g + i;
      const float x = key < k_hi ? sacc[j][i] * sl : -INFINITY;
      sacc[j][i] = x;
      mx = fmaxf(mx, x);
    }
  mx = lane_max<32>(lane_max<16>(mx));
  const float mref = mx == -INFINITY ? 0.f : mx;  // wave with no valid key: all p = 0
  float ls = 0.f;
  u16x8 pb[NP][2];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float p = __builtin_amdgcn_exp2f(sacc[j][i] - mref);
      ls += p;
#pragma unroll
      for (int n = 0; n < NP; ++n) {
        pb[n][j >> 1][4 * (j & 1) + i] = f2bf(p);
        p -= bf2f(pb[n][j >> 1][4 * (j & 1) + i]);
      }
    }
  ls = lane_sum<32>(lane_sum<16>(ls));

  // O^T[d][head] += V^T . P; k-step t covers keys 32 t + {16 h + 4 g + i}
  f32x4 oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) oacc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's V DMA has landed (only it reads vs)
  const int qq = c >> 2, pp = c & 3;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int r0 = 32 * t + 4 * g + qq, r1 = r0 + 16;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int ch = 2 * db + (pp >> 1);
      const u16x4 va = tr_read16(vs + r0 * ROWB + 16 * (ch ^ dswz<D>(r0)) + 8 * (pp & 1));
      const u16x4 vb = tr_read16(vs + r1 * ROWB + 16 * (ch ^ dswz<D>(r1)) + 8 * (pp & 1));
      const u16x8 a = u16x8{va[0], va[1], va[2], va[3], vb[0], vb[1], vb[2], vb[3]};
#pragma unroll
      for (int n = NP - 1; n >= 0; --n) oacc[db] = mfma16(a, pb[n][t], oacc[db]);  // the smallest parts first
    }
  }
  // merge the four waves: each wave parks (m, l, O^T) in its own V region
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's transposed reads retired
  float* so = reinterpret_cast<float*>(vs);  // [d][16 heads]
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 4; ++i) so[(16 * db + 4 * g + i) * 16 + c] = oacc[db][i];
  if (g == 0) {
    mls[w][0][c] = mx;
    mls[w][1][c] = ls;
  }
  __syncthreads();
  for (int idx = tid; idx < rep * D; idx += 256) {
    const int h = idx / D, d = idx % D;
    float M = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) M = fmaxf(M, mls[ww][0][h]);
    float L = 0.f, acc = 0.f;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) {
      const float mw = mls[ww][0][h];
      const float f = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M);
      L += f * mls[ww][1][h];
      acc += f * reinterpret_cast<const float*>(smem + ww * WTILE)[d * 16 + h];
    }
    if (out) {  // as decode_combine_kernel writes one split
      out[((int64_t)b * Hq + hk * rep + h) * D + d] = f2bf(L > 0.f ? acc / L : 0.f);
      continue;
    }
    st_part(&part_o[(((int64_t)b * Hq + hk * rep + h) * nsplit + split) * D + d], acc, st);
    if (d == 0) {
      st_part(&pml[(int64_t)h * nsplit * 2], M, st);
      st_part(&pml[(int64_t)h * nsplit * 2 + 1], L, st);
    }
  }
}

// proto (fused split merge, cnt != nullptr; 0 = partials only / combine kernel):
//   1 = partials stored with agent-scope (sc1, write-through) atomic stores, read back with
//       agent-scope atomic loads, no fences;
//   2 = the same at system scope;
//   3 = agent-scope stores, an agent-scope acquire fence in the merger, plain loads;
//   4 = plain stores, one agent-scope release fence per workgroup (lane 0, after every wave's
//       vmcnt drain), acquire fence in the merger, plain loads (guide §5 in-launch split-K recipe).
template <int D>
__global__ void __launch_bounds__(256, 2) decode_attn_mfma_kernel(const uint16_t* __restrict__ q,
                                                                  const uint16_t* __restrict__ kc,
                                                                  const uint16_t* __restrict__ vc,
                                                                  const int32_t* __restrict__ lens, int len_off,
                                                                  const int32_t* __restrict__ slots,
                                                                  float* __restrict__ part_ml,
                                                                  float* __restrict__ part_o, int Hq, int Hkv,
                                                                  int max_seq, int nsplit, float sl,
                                                                  const int32_t* __restrict__ bt, int maxb,
                                                                  uint16_t* __restrict__ out,
                                                                  unsigned int* __restrict__ cnt, int proto) {
  constexpr int WTILE = 64 * 2 * D;  // 16 KiB per wave at D = 128
  __shared__ __attribute__((aligned(16))) char smem[4 * WTILE];
  __shared__ float mls[4][2][16];
  __shared__ int s_last;
  const int split = blockIdx.x, hk = blockIdx.y, b = blockIdx.z;
  const int rep = Hq / Hkv;
  const int len = lens[b] + len_off;
  const int slot = slots ? slots[b] : b;
  const int k_lo = split * kSplit;
  const int k_hi = min(len, k_lo + kSplit);
  const int tid = threadIdx.x;
  const bool fused = cnt != nullptr;
  const int st = !fused ? 0 : proto == 2 ? 2 : proto == 4 ? 0 : 1;  // store mode of the partials
  float* pml = part_ml + (((int64_t)b * Hq + hk * rep) * nsplit + split) * 2;
  uint16_t* const only = out && nsplit == 1 ? out : nullptr;
  if (k_lo >= k_hi) {  // empty split (workgroup-uniform): neutral partial
    if (only) {
      for (int i = tid; i < rep * D; i += 256) only[((int64_t)b * Hq + hk * rep) * D + i] = 0;
      return;
    }
    if (tid < rep) {
      st_part(&pml[(int64_t)tid * nsplit * 2], -INFINITY, st);
      st_part(&pml[(int64_t)tid * nsplit * 2 + 1], 0.f, st);
    }
  } else {
    decode_split_body<D>(q, kc, vc, part_o, pml, smem, mls, b, hk, rep, Hq, split, nsplit, k_lo, k_hi, slot, max_seq,
                         sl, bt, maxb, Hkv, st, only);
  }
  if (!fused || only) return;
  // In-launch combine: the last of the nsplit workgroups of this (seq, kv-head) to arrive
  // merges the partials and resets the counter (zero again for the next call).
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every wave: its partial stores done
  __syncthreads();
  if (tid == 0) {
    unsigned int* c = cnt + (int64_t)b * Hkv + hk;
    if (proto == 4) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    const unsigned prev = proto == 2 ? __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM)
                                     : __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int last = prev == (unsigned)(nsplit - 1);
    if (last) {
      __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (proto >= 3) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
    }
    s_last = last;
  }
  __syncthreads();
  if (!s_last) return;
  const int ld = proto == 1 ? 1 : proto == 2 ? 2 : 0;
  // the same arithmetic, in the same order, as decode_combine_kernel
  for (int idx = tid; idx < rep * D; idx += 256) {
    const int h = idx / D, d = idx % D;
    const int64_t bh = (int64_t)b * Hq + hk * rep + h;
    const float* ml = part_ml + bh * nsplit * 2;
    float M = -INFINITY;
    for (int sp = 0; sp < nsplit; ++sp) M = fmaxf(M, ld_part(ml + 2 * sp, ld));
    float L = 0.f, acc = 0.f;
    for (int sp = 0; sp < nsplit; ++sp) {
      const float m = ld_part(ml + 2 * sp, ld);
      if (m == -INFINITY) continue;
      const float wgt = __builtin_amdgcn_exp2f(m - M);
      L += wgt * ld_part(ml + 2 * sp + 1, ld);
      acc += wgt * ld_part(part_o + (bh * nsplit + sp) * D + d, ld);
    }
    out[bh * D + d] = f2bf(L > 0.f ? acc / L : 0.f);
  }
}

// merge splits: out[b, h, :] = sum_s exp2(m_s - M) o_s / sum_s exp2(m_s - M) l_s
template <int D>
__global__ void __launch_bounds__(D) decode_combine_kernel(const float* __restrict__ part_ml,
                                                           const float* __restrict__ part_o,
                                                           uint16_t* __restrict__ out, int nsplit) {
  const int64_t bh = blockIdx.x;
  const float* ml = part_ml + bh * nsplit * 2;
  const int d = threadIdx.x;
  if (nsplit <= 8) {
    // every partial load issued at once (one memory round trip instead of two: the outputs'
    // loads do not wait for the maxima); same arithmetic order as the loop below
    float mv[8], lv[8], ov[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const bool on = s < nsplit;
      mv[s] = on ? ml[2 * s] : -INFINITY;
      lv[s] = on ? ml[2 * s + 1] : 0.f;
      ov[s] = on ? part_o[(bh * nsplit + s) * D + d] : 0.f;
    }
    float M = -INFINITY;
#pragma unroll
    for (int s = 0; s < 8; ++s) M = fmaxf(M, mv[s]);
    float L = 0.f, acc = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      if (mv[s] == -INFINITY) continue;
      const float wgt = __builtin_amdgcn_exp2f(mv[s] - M);
      L += wgt * lv[s];
      acc += wgt * ov[s];
    }
    out[bh * D + d] = f2bf(L > 0.f ? acc / L : 0.f);
    return;
  }
  float M = -INFINITY;
  for (int s = 0; s < nsplit; ++s) M = fmaxf(M, ml[2 * s]);
  float L = 0.f, acc = 0.f;
  for (int s = 0; s < nsplit; ++s) {
    const float m = ml[2 * s];
    if (m == -INFINITY) continue;
    const float wgt = __builtin_amdgcn_exp2f(m - M);
    L += wgt * ml[2 * s + 1];
    acc += wgt * part_o[(bh * nsplit + s) * D + d];
  }
  out[bh * D + d] = f2bf(L > 0.f ? acc / L : 0.f);
}

// ---------------------------------------------------------------------------
// Decode attention, heads of 128, of more 256-key splits than the CUs have places for (kEvenPlaces): the
// keys of all sequences, in units of 16, are dealt evenly to one turn of workgroups.
//
// decode_attn_mfma_kernel gives every 256 keys of a sequence a workgroup.  16 sequences of 100 to 2,000 keys
// are 540 of them on 512 places, and the 28 of the second turn cost nearly what the 512 of the first do.
// Here a workgroup walks its equal share of the row of sequences of one KV head, segment by segment; a
// segment's keys are shared by its four waves.  K and V both come straight into registers (a lane takes 8
// neighbouring channels of 8 keys, and puts halves of its words together to the operand that the product
// reads), so no LDS holds a tile and three workgroups fit a CU, whose loads hide each other's products.  Loads of
// the next 32 keys issued ahead of the products of the last lose (29 us: 220 registers, two workgroups a CU), and
// so do more than two shares a CU (more segments, and parts to merge).
//
// Time alone, 32 heads of 8 (merge apart, 4.7 us as before), us: 16 sequences of 100 to 2,000 keys 26.4 -> 23.9,
// 48 of 60 to 600 21.4 -> 18.8, 32 of 100 to 1,000 25.5 -> 20.6, 7 of 2,500 21.7 -> 18.8.  Heads of 64, at
// half the bytes a key, do not gain (14.1 -> 14.1, 11.4 -> 13.6) and keep their splits.
//
// Level or slower where the sequences are alike and end with a split, over four turns and more, where nothing is uneven: 64 of 1,024
// keys 60.5 -> 64.2, of 2,048 116 -> 127, 128 of 1,024 117 -> 126; but 32 of 2,080 67 -> 61, 64 of 1,000 to 2,048 105 -> 96.  Long
// ones gain most, whose merge is then of as many parts as shares (1 of 32,768 78 -> 42, 8 of 16,384 144 -> 111).
//
// Scores, weights and sums are those of decode_split_body; a wave keeps a running maximum.  Where a row is cut follows from the
// lengths of all rows and its place among them, so the order of its sums, and with it the last bits of its outputs, may differ
// from batch to batch (the same call has the same bits; a row of fixed splits has its own whatever the others are).
constexpr int kEvenD = 128, kEvenPlaces = 512;  // two workgroups a CU
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

struct EvenState {  // of one wave
  float m, l;  // of head c; l: this lane's keys
  f32x4 o[8];  // [e][i]: channel 8 (4 g + i) + e of head c

  __device__ __forceinline__ void clear() {
    m = -INFINITY, l = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // keys key0 .. key0 + 31 below hi (key0 a multiple of 16); k0, v0 / k1, v1: rows of the first / second 16 keys,
  // l0, l1: the last row of them that is read
  __device__ __forceinline__ void take(const uint16_t* __restrict__ k0, const uint16_t* __restrict__ k1,
                                       const uint16_t* __restrict__ v0, const uint16_t* __restrict__ v1, int l0, int l1,
                                       const u16x8 (&qf)[4], int key0, int hi, float sl, int c, int g) {
    u32x4_t k[2][4], v[8];  // v: slot s is key 16 (s >> 2) + 4 g + (s & 3), channels 8 c ..
    const uint32_t r0 = min(c, l0) * kEvenD + 8 * g, r1 = min(c, l1) * kEvenD + 8 * g;
#pragma unroll
    for (int s = 0; s < 4; ++s) k[0][s] = *reinterpret_cast<const u32x4_t*>(k0 + (r0 + 32 * s));
#pragma unroll
    for (int s = 0; s < 4; ++s) k[1][s] = *reinterpret_cast<const u32x4_t*>(k1 + (r1 + 32 * s));
#pragma unroll
    for (int s = 0; s < 4; ++s)
      v[s] = *reinterpret_cast<const u32x4_t*>(v0 + (uint32_t)(min(4 * g + s, l0) * kEvenD + 8 * c));
#pragma unroll
    for (int s = 0; s < 4; ++s)
      v[4 + s] = *reinterpret_cast<const u32x4_t*>(v1 + (uint32_t)(min(4 * g + s, l1) * kEvenD + 8 * c));
    __builtin_amdgcn_sched_barrier(0);  // every load is in flight before the first product waits
    f32x4 sc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      sc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) sc[j] = mfma16(__builtin_bit_cast(u16x8, k[j][s]), qf[s], sc[j]);
    }
    float mx = m;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = key0 + 16 * j + 4 * g + i < hi ? sc[j][i] * sl : -INFINITY;
        sc[j][i] = x;
        mx = fmaxf(mx, x);
      }
    mx = lane_max<32>(lane_max<16>(mx));
    const float mref = mx == -INFINITY ? 0.f : mx, f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mref);
    m = mx;
    l *= f;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= f;
    u16x8 pb;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = __builtin_amdgcn_exp2f(sc[j][i] - mref);
        l += p;
        pb[4 * j + i] = f2bf(p);
      }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      u32x4_t a;  // channel e of the 8 keys: one half of a word of each
#pragma unroll
      for (int i = 0; i < 4; ++i)
        a[i] = __builtin_amdgcn_perm(v[2 * i + 1][e >> 1], v[2 * i][e >> 1], e & 1 ? 0x07060302u : 0x05040100u);
      o[e] = mfma16(__builtin_bit_cast(u16x8, a), pb, o[e]);
    }
  }
};

// What a row costs a workgroup beside its keys, in units of 16: its length, slot, block and q asked for one after another,
// the sums of its waves, and waves' turns of 32 keys that are not full.  Dealt by their keys alone, workgroups with the end
// of one row and the start of another ended 22 us into the launch, those within a row at 15 (16 sequences of 100 to 2,000
// keys).  A step of them, us, with 0 / 3 / 6 / 9 / 13: 4060 / 4008 / 4001 / 4013 / 4043; 32 of 250 to 1,000 4738 / 4710 /
// 4696 / 4753 / 4768; 24 of 225 to 900 4515 / 4497 / 4498 / 4510 / 4526; 8 of 750 to 3,000 3800 / 3791 / 3799 / 3844 / 3828.
// Short rows in a step built for long ones, the attention alone, us, with 0 / 6: 12 of 32 keys 14.6 / 7.0, 64 of 100 15.3 / 10.9, 128 of up
// to 256 26.3 / 22.1; rows that share by share were whole before are the worst, 40 of 128 9.7 / 11.0, 100 of 64 15.6 / 16.2.
constexpr int kEvenPad = 6;
// units that row b is dealt as, the first kEvenPad of which hold no keys; cap: positions that the buffers are sized for
__device__ __forceinline__ int even_units(const int32_t* lens, int len_off, int cap, int b) {
  const int n = (min(max(lens[b] + len_off, 0), cap) + 15) >> 4;
  return n ? n + kEvenPad : 0;
}
// units of a workgroup: an equal share of all, at least 8 (128 keys, or the first 32 of a row: with 14, so that a row's first 128 stay
// together, 64 rows of 100 keys 10.9 -> 14.0 us, 20 of up to 192 9.2 -> 12.3; alike only for rows of 128, 9.4 -> 8.3)
__device__ __forceinline__ int even_share(int total, int W) { return max((total + W - 1) / W, 8); }

__global__ void __launch_bounds__(256, 3)
    decode_even_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
                       const int32_t* __restrict__ lens, int len_off, const int32_t* __restrict__ slots,
                       float* __restrict__ part_ml, float* __restrict__ part_o, uint16_t* __restrict__ out, int B, int Hq,
                       int Hkv, int max_seq, int cap, int nparts, float sl, const int32_t* __restrict__ bt, int maxb) {
  constexpr int D = kEvenD;
  __shared__ float so[4][D][17];
  __shared__ float mls[4][2][16];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4, hk = blockIdx.y, rep = Hq / Hkv, x = blockIdx.x;
  int total = 0;
  for (int i = lane; i < B; i += 64) total += even_units(lens, len_off, cap, i);
  total = __builtin_amdgcn_readfirstlane(wave_sum(total));
  const int share = even_share(total, gridDim.x);
  int at = x * share;
  const int end = min(total, at + share);
  if (at >= end) return;
  int b = 0, start = 0;  // the row that holds unit `at`: start <= at < start + n
  for (int i0 = 0;; i0 += 64) {
    const int n = i0 + lane < B ? even_units(lens, len_off, cap, i0 + lane) : 0;
    const int upto = (int)wave_scan((uint32_t)n);
    const uint64_t past = __ballot(start + upto > at);
    if (past) {
      const int first = __ffsll((unsigned long long)past) - 1;
      b = __builtin_amdgcn_readfirstlane(i0 + first);
      start = __builtin_amdgcn_readlane(start + upto - n, first);
      break;
    }
    start = __builtin_amdgcn_readlane(start + upto, 63);
  }
  while (true) {
    const int len = min(max(lens[b] + len_off, 0), cap), n = (len + 15) >> 4;
    if (n == 0) {  // (units are left, so a later row has them)
      ++b;
      continue;
    }
    const int from = start + kEvenPad;  // of its keys
    const int u0 = max(at - from, 0), u1 = min(end - from, n), per = (u1 - u0 + 3) >> 2;
    if (u1 <= 0) return;  // its keys begin in the next share
    const int k_lo = 16 * (u0 + per * w), hi = min(len, 16 * min(u1, u0 + per * (w + 1)));
    const int slot = slots ? slots[b] : b;
    u16x8 qf[4];
    const uint16_t* qrow = q + ((int64_t)b * Hq + hk * rep + min(c, rep - 1)) * D;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      qf[s] = *reinterpret_cast<const u16x8*>(qrow + 32 * s + 8 * g);
      if (c >= rep) qf[s] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
    EvenState st;
    st.clear();
    const int past = (hi - 1) & ~15;  // the last 16 keys that have one
    for (int k = k_lo; k < hi; k += 32) {
      const int a1 = min(k + 16, past);  // 16 keys lie in one block: blocks are multiples of 256
      const int64_t b0 = kv_row(bt, maxb, max_seq, slot, Hkv, hk, k) * D, b1 = kv_row(bt, maxb, max_seq, slot, Hkv, hk, a1) * D;
      st.take(kc + b0, kc + b1, vc + b0, vc + b1, hi - 1 - k, hi - 1 - a1, qf, k, hi, sl, c, g);
    }
    st.l = lane_sum<32>(lane_sum<16>(st.l));
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int i = 0; i < 4; ++i) so[w][8 * (4 * g + i) + e][c] = st.o[e][i];
    if (g == 0) mls[w][0][c] = st.m, mls[w][1][c] = st.l;
    __syncthreads();
    const int part = x - from / share, last = (from + n - 1) / share - from / share;
    for (int idx = tid; idx < rep * D; idx += 256) {
      const int h = idx / D, d = idx % D;
      float M = -INFINITY, L = 0.f, acc = 0.f;
#pragma unroll
      for (int ww = 0; ww < 4; ++ww) M = fmaxf(M, mls[ww][0][h]);
#pragma unroll
      for (int ww = 0; ww < 4; ++ww) {
        const float mw = mls[ww][0][h], f = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M);
        L += f * mls[ww][1][h];
        acc += f * so[ww][d][h];
      }
      const int64_t bh = (int64_t)b * Hq + hk * rep + h;
      if (last == 0) {  // the row's only part is its output
        out[bh * D + d] = f2bf(L > 0.f ? acc / L : 0.f);
      } else {
        part_o[(bh * nparts + part) * D + d] = acc;
        if (d == 0) part_ml[(bh * nparts + part) * 2] = M, part_ml[(bh * nparts + part) * 2 + 1] = L;
      }
    }
    at = start = from + n;
    if (at >= end) return;
    ++b;
    __syncthreads();  // the sums are read
  }
}

// merge of decode_even_kernel's parts, of the rows that have several; W: its workgroups of a KV head
__global__ void __launch_bounds__(kEvenD)
    decode_even_merge_kernel(const float* __restrict__ part_ml, const float* __restrict__ part_o,
                             const int32_t* __restrict__ lens, int len_off, uint16_t* __restrict__ out, int B, int Hq,
                             int W, int cap, int nparts) {
  const int64_t bh = blockIdx.x;
  const int b = (int)(bh / Hq), d = threadIdx.x, lane = d & 63;
  const float* ml = part_ml + bh * nparts * 2;
  const float* po = part_o + bh * nparts * kEvenD + d;
  // the first parts' loads go out with those of the lengths; what is no part is not looked at
  float mv[8], lv[8], ov[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int p = min(s, nparts - 1);
    mv[s] = ml[2 * p], lv[s] = ml[2 * p + 1], ov[s] = po[(int64_t)p * kEvenD];
  }
  int total = 0, start = 0;
  const int n = even_units(lens, len_off, cap, b) - kEvenPad;
  for (int i = lane; i < B; i += 64) {
    const int u = even_units(lens, len_off, cap, i);
    total += u;
    if (i < b) start += u;
  }
  total = wave_sum(total), start = wave_sum(start);
  const int share = even_share(total, W), from = start + kEvenPad;
  const int parts = n > 0 ? (from + n - 1) / share - from / share + 1 : 0;
  if (parts == 1) return;  // written by its workgroup
  float M = -INFINITY, L = 0.f, acc = 0.f;
#pragma unroll
  for (int s = 0; s < 8; ++s) M = s < parts ? fmaxf(M, mv[s]) : M;
  for (int s = 8; s < parts; ++s) M = fmaxf(M, ml[2 * s]);
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    if (s >= parts || mv[s] == -INFINITY) continue;
    const float wgt = __builtin_amdgcn_exp2f(mv[s] - M);
    L += wgt * lv[s];
    acc += wgt * ov[s];
  }
#pragma unroll 4
  for (int s = 8; s < parts; ++s) {
    const float m = ml[2 * s], ls = ml[2 * s + 1], os = po[(int64_t)s * kEvenD];
    const float wgt = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - M);
    L += wgt * ls;
    acc += wgt * os;
  }
  out[bh * kEvenD + d] = f2bf(L > 0.f ? acc / L : 0.f);
}

// ---------------------------------------------------------------------------
// Decode attention of up to 512 keys: eight waves take a whole (sequence, KV head), 64 keys each, so that nothing is left
// to merge in a launch of its own.  K and V in registers as in EvenState; each wave leaves its maximum, sum and outputs
// in LDS, where they are added as decode_split_body adds four waves and decode_combine_kernel two splits, so the bits
// are those of the splits.
//
// Both launches against this one, 32 heads of 8, us: heads of 64, 1 / 4 / 32 sequences of up to 300 / 400 / 400 keys
// 6.5 / 7.1 / 11.0 -> 5.2 / 6.0 / 7.1; of 128, 8.6 / 9.0 / 15.7 -> 6.5 / 7.4 / 10.5.  Past 512 keys a CU to a sequence is too
// little (16 waves of 64 keys, one sequence of 700 keys, heads of 64: 7.2 in splits, 7.6 so; 2,048 keys 7.6, 16.9).
constexpr int kShortSplits = 2, kShortRep = 8;  // q-heads of a KV head: 34 KB of LDS at heads of 128

template <int D>
__global__ void __launch_bounds__(512)
    decode_short_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
                        const int32_t* __restrict__ lens, int len_off, const int32_t* __restrict__ slots,
                        uint16_t* __restrict__ out, int Hq, int Hkv, int max_seq, float sl,
                        const int32_t* __restrict__ bt, int maxb) {
  constexpr int KS = D / 32, E = D / 16, NP = D == 128 ? 1 : 3, TILES = 4 * kShortSplits;
  typedef uint32_t vrow_t __attribute__((ext_vector_type(E / 2)));
  typedef float orow_t __attribute__((ext_vector_type(E)));
  __shared__ float mls[TILES][2][16];
  __shared__ __attribute__((aligned(16))) float so[TILES * kShortRep * D];
  const int tid = threadIdx.x, lane = tid & 63, t = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4, hk = blockIdx.x, b = blockIdx.y, rep = Hq / Hkv;
  const int len = min(max(lens[b] + len_off, 0), kShortSplits * kSplit), slot = slots ? slots[b] : b;
  const int lim = len - 1 - 64 * t;  // the last row of the wave's tile that is read
  if (lim < 0) {
    if (g == 0) mls[t][0][c] = -INFINITY, mls[t][1][c] = 0.f;
  } else {
    u16x8 qf[KS];
    const uint16_t* qrow = q + ((int64_t)b * Hq + hk * rep + min(c, rep - 1)) * D;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      qf[s] = *reinterpret_cast<const u16x8*>(qrow + 32 * s + 8 * g);
      if (c >= rep) qf[s] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
    const int64_t base = kv_row(bt, maxb, max_seq, slot, Hkv, hk, 64 * t) * D;  // a tile lies in one block
    const uint16_t *kb = kc + base, *vb = vc + base;
    u32x4_t k[4][KS];
    vrow_t v[16];  // slot s: key 16 (s >> 2) + 4 g + (s & 3), channels E c ..
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t r = min(16 * j + c, lim) * D + 8 * g;
#pragma unroll
      for (int s = 0; s < KS; ++s) k[j][s] = *reinterpret_cast<const u32x4_t*>(kb + (r + 32 * s));
    }
#pragma unroll
    for (int s = 0; s < 16; ++s)
      v[s] = *reinterpret_cast<const vrow_t*>(vb + (uint32_t)(min(16 * (s >> 2) + 4 * g + (s & 3), lim) * D + E * c));
    __builtin_amdgcn_sched_barrier(0);  // every load is in flight before the first product waits
    f32x4 sc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      sc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) sc[j] = mfma16(__builtin_bit_cast(u16x8, k[j][s]), qf[s], sc[j]);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = 16 * j + 4 * g + i <= lim ? sc[j][i] * sl : -INFINITY;
        sc[j][i] = x;
        mx = fmaxf(mx, x);
      }
    mx = lane_max<32>(lane_max<16>(mx));
    const float mref = mx == -INFINITY ? 0.f : mx;
    float ls = 0.f;
    u16x8 pb[NP][2];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float p = __builtin_amdgcn_exp2f(sc[j][i] - mref);
        ls += p;
#pragma unroll
        for (int n = 0; n < NP; ++n) {
          pb[n][j >> 1][4 * (j & 1) + i] = f2bf(p);
          p -= bf2f(pb[n][j >> 1][4 * (j & 1) + i]);
        }
      }
    ls = lane_sum<32>(lane_sum<16>(ls));
    if (g == 0) mls[t][0][c] = mx, mls[t][1][c] = ls;
    f32x4 o[E];  // [e][i]: channel E (4 g + i) + e of head c
#pragma unroll
    for (int e = 0; e < E; ++e) {
      o[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        u32x4_t a;  // channel e of 8 keys: one half of a word of each
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t hi, lo;
          if constexpr (E == 2) hi = v[8 * h + 2 * i + 1][0], lo = v[8 * h + 2 * i][0];
          else hi = v[8 * h + 2 * i + 1][e >> 1], lo = v[8 * h + 2 * i][e >> 1];
          a[i] = __builtin_amdgcn_perm(hi, lo, e & 1 ? 0x07060302u : 0x05040100u);
        }
#pragma unroll
        for (int n = NP - 1; n >= 0; --n) o[e] = mfma16(__builtin_bit_cast(u16x8, a), pb[n][h], o[e]);
      }
    }
    if (c < rep) {
      float* const dst = so + (t * rep + c) * D + 4 * E * g;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        orow_t y;
#pragma unroll
        for (int e = 0; e < E; ++e) y[e] = o[e][i];
        *reinterpret_cast<orow_t*>(dst + E * i) = y;
      }
    }
  }
  __syncthreads();
  for (int idx = tid; idx < rep * D; idx += 512) {
    const int h = idx / D, d = idx % D;
    float M = -INFINITY, L = 0.f, acc = 0.f;
#pragma unroll
    for (int w = 0; w < TILES; ++w) M = fmaxf(M, mls[w][0][h]);
#pragma unroll
    for (int s = 0; s < kShortSplits; ++s) {
      float m = -INFINITY, lv = 0.f, ov = 0.f;
#pragma unroll
      for (int w = 4 * s; w < 4 * s + 4; ++w) m = fmaxf(m, mls[w][0][h]);
#pragma unroll
      for (int w = 4 * s; w < 4 * s + 4; ++w) {
        const float mw = mls[w][0][h];
        if (mw == -INFINITY) continue;  // (its outputs may not have been written)
        const float f = __builtin_amdgcn_exp2f(mw - m);
        lv += f * mls[w][1][h];
        ov += f * so[(w * rep + h) * D + d];
      }
      if (m == -INFINITY) continue;
      const float wgt = __builtin_amdgcn_exp2f(m - M);
      L += wgt * lv;
      acc += wgt * ov;
    }
    out[((int64_t)b * Hq + hk * rep + h) * D + d] = f2bf(L > 0.f ? acc / L : 0.f);
  }
}

__device__ __forceinline__ uint32_t hash3(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t h = a * 0x9E3779B1u ^ (b + 0x7F4A7C15u) * 0x85EBCA77u ^ (c + 0x165667B1u) * 0xC2B2AE3Du;
  h ^= h >> 15; h *= 0x2C1B3C6Du; h ^= h >> 12; h *= 0x297A2D39u; h ^= h >> 15;
  return h;
}

// logits [B, V] (bf16 or f32); temperature <= 0 -> greedy.  out ids [B] int64.
//
// Split over the vocabulary: grid (nchunks, B), each workgroup reduces `chunk`
// logits of one row to (max, smallest index); a second one-wave-per-row kernel
// combines the partials in chunk order.  One workgroup per row left a batch-1
// decode step with ONE CU streaming 256 KB of logits: 176 us of a 4.1 ms 8B
// step; split over ~63 workgroups it is a few microseconds.  (A last-arriver
// merge in the same kernel needed an agent-scope release fence per workgroup:
// 94 us at batch 64.)  The result (and the Gumbel noise of each (seed, row,
// step, index)) is the same as a single-pass argmax.  The partials live in a
// per-call workspace (allocated by the caller on its stream), so concurrent
// samplers on different streams of one device never share them.
constexpr int kSampMaxRows = 1024;   // rows per launch (more rows: several launches)
constexpr int kSampMaxChunks = 64;   // partials per row (= one wave in the final pass)

__device__ __forceinline__ void samp_pick(float& best, int& bi, float ov, int oi) {
  if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
}

template <typename T>
__global__ void __launch_bounds__(256) sample_kernel(const T* __restrict__ logits, int64_t* __restrict__ out, int V,
                                                     int chunk, float inv_temp, uint32_t seed, uint32_t step,
                                                     int row0, const float* __restrict__ temps,
                                                     const int64_t* __restrict__ seeds,
                                                     const int32_t* __restrict__ steps,
                                                     float* __restrict__ g_samp_val, int* __restrict__ g_samp_idx) {
  __shared__ float sv[4];
  __shared__ int si[4];
  const int lrow = blockIdx.y;
  const int64_t row = (int64_t)row0 + lrow;
  const T* x = logits + row * V;
  const int c0 = blockIdx.x * chunk, c1 = min(V, c0 + chunk);
  uint32_t nseed = seed + (uint32_t)row * 7919u;
  if (temps) {  // per-row parameters (mx_sample_temp_rows): noise of sampling.hip
    const float t = temps[row];
    inv_temp = t > 0.f ? 1.f / t : 0.f;
    nseed = (uint32_t)seeds[row];
    step = (uint32_t)steps[row];
  }
  float best = -INFINITY;
  int bi = c0 < V ? c0 : 0;
  for (int cb = c0 + (int)threadIdx.x; cb < c1; cb += 256 * 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {  // 8 independent loads in flight per thread
      const int c = cb + 256 * u;
      if constexpr (sizeof(T) == 2) v[u] = c < c1 ? bf2f(reinterpret_cast<const uint16_t*>(x)[c]) : -INFINITY;
      else v[u] = c < c1 ? reinterpret_cast<const float*>(x)[c] : -INFINITY;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = cb + 256 * u;
      if (c >= c1) break;
      float w = v[u];
      if (inv_temp > 0.f) {
        const uint32_t h = hash3(nseed, step, (uint32_t)c);
        const float uu = ((h >> 8) + 0.5f) * (1.0f / 16777216.0f);
        w = w * inv_temp - __logf(-__logf(uu));  // Gumbel-max
      }
      if (w > best) { best = w; bi = c; }
    }
  }
  wave_pick(best, bi);
  if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = best; si[threadIdx.x >> 6] = bi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) samp_pick(best, bi, sv[w], si[w]);
    g_samp_val[lrow * kSampMaxChunks + blockIdx.x] = best;
    g_samp_idx[lrow * kSampMaxChunks + blockIdx.x] = bi;
  }
}

// partials of one row (chunk order) -> out[row]; grid rows, one wave
__global__ void __launch_bounds__(64) sample_final_kernel(int64_t* __restrict__ out, int nch, int row0,
                                                          const float* __restrict__ g_samp_val,
                                                          const int* __restrict__ g_samp_idx) {
  const int lrow = blockIdx.x, l = threadIdx.x;
  float best = -INFINITY;
  int bi = 0x7fffffff;
  if (l < nch) {
    best = g_samp_val[lrow * kSampMaxChunks + l];
    bi = g_samp_idx[lrow * kSampMaxChunks + l];
  }
  wave_pick(best, bi);
  if (l == 0) out[(int64_t)row0 + lrow] = bi == 0x7fffffff ? 0 : bi;
}

}  // namespace mx

using namespace mx;

// bt / maxb: paged cache (block table [slots, maxb]; max_seq = the block size), nullptr: contiguous
extern "C" int mx_rope_append(const uint16_t* qkv, const float* cosb, const float* sinb, const int32_t* pos,
                              const int32_t* slots, uint16_t* q, uint16_t* kc, uint16_t* vc, int B, int Hq, int Hkv,
                              int D, int max_seq, const int32_t* bt, int maxb, hipStream_t stream) {
  const int64_t items = (int64_t)B * (Hq + 2 * Hkv) * (D / 16);
  if (items <= 0) return 0;
  const int grid = (int)std::min<int64_t>(1024, (items + 255) / 256);
#define RA(DD) \
  rope_append_kernel<DD><<<grid, 256, 0, stream>>>(qkv, cosb, sinb, pos, slots, q, kc, vc, B, Hq, Hkv, max_seq, bt, maxb)
  if (D == 128) RA(128); else if (D == 64) RA(64); else if (D == 32) RA(32); else return -1;
#undef RA
  return (int)hipGetLastError();
}

// workgroups of a KV head, and the most parts of a row, where the keys are dealt evenly: a row of n units touches at most
// (n + share - 2) / share + 1 shares of 8 units or more, and no more than there are
static int even_groups(int Hkv) { return std::max(1, kEvenPlaces / std::max(1, Hkv)); }
static int even_parts(int Hkv, int nsplit) { return std::min(2 * nsplit + 1, even_groups(Hkv)); }

// parts a row that the buffers of mx_decode_attn have room for
extern "C" int mx_decode_attn_parts(int Hkv, int nsplit) { return std::max(nsplit, even_parts(Hkv, nsplit)); }

extern "C" int mx_decode_attn(const uint16_t* q, const uint16_t* kc, const uint16_t* vc, const int32_t* lens,
                              int len_off, const int32_t* slots, float* part_ml, float* part_o, uint16_t* out, int B,
                              int Hq, int Hkv, int D, int max_seq, int nsplit, float scale, const int32_t* bt,
                              int maxb, unsigned int* cnt, hipStream_t stream) {
  if (B <= 0) return 0;
  if (Hq % Hkv || Hq / Hkv > kMaxRep) return -1;
  if (bt && max_seq % kSplit) return -1;  // a split must lie inside one block
  dim3 grid(nsplit, Hkv, B);
  const float sl = scale * 1.4426950408889634f;
  // out == nullptr: partials only, merged by the caller (skinny_gemm.hip MERGE, hybrid.hip attn_combine)
  // cnt (zeroed [B * Hkv] counters, owned by the caller; D = 128): the splits merge in-launch
  // MXLLM_DECODE_HANDOFF: hand-off protocol of the in-launch merge (see the kernel; read per call)
  const char* pe = getenv("MXLLM_DECODE_HANDOFF");
  const int proto = pe && *pe ? atoi(pe) : 4;
  const bool fused = out && cnt && D == 128 && proto >= 1 && proto <= 4;
  // up to 512 keys: one launch (B: the grid's second dimension)
  if (out && nsplit == kShortSplits && Hq / Hkv <= kShortRep && B <= 65535) {
#define DS(DD) \
  decode_short_kernel<DD><<<dim3(Hkv, B), 512, 0, stream>>>(q, kc, vc, lens, len_off, slots, out, Hq, Hkv, max_seq, sl, bt, maxb)
    if (D == 128) DS(128); else if (D == 64) DS(64); else if (D == 32) DS(32); else return -1;
#undef DS
    return (int)hipGetLastError();
  }
  // Heads of 128, more splits than places: dealt evenly.  What the caller's `nsplit` counts is the longest that the step
  // was built for; where the sequences of a call are shorter, the shares are (even_share).  Not of one split (no merge
  // to wait for: 32 heads of 8, us, split -> dealt: 80 sequences of 60 to 256 keys 16.0 -> 20.8, 256 36.3 -> 42.8; 72 of 10 to
  // 64 10.2 -> 19.0) nor of two where the kernel above does not take them (32 heads of 2, 256 of 20 to 200 keys 29.0 -> 31.5).
  if (out && D == kEvenD && nsplit > kShortSplits && (int64_t)nsplit * Hkv * B > kEvenPlaces) {
    const int W = even_groups(Hkv), cap = nsplit * kSplit, nparts = even_parts(Hkv, nsplit);
    decode_even_kernel<<<dim3(W, Hkv), 256, 0, stream>>>(q, kc, vc, lens, len_off, slots, part_ml, part_o, out, B, Hq, Hkv,
                                                         max_seq, cap, nparts, sl, bt, maxb);
    decode_even_merge_kernel<<<B * Hq, kEvenD, 0, stream>>>(part_ml, part_o, lens, len_off, out, B, Hq, W, cap, nparts);
    return (int)hipGetLastError();
  }
#define DA(DD)                                                                                                      \
  decode_attn_mfma_kernel<DD><<<grid, 256, 0, stream>>>(q, kc, vc, lens, len_off, slots, part_ml, part_o, Hq, Hkv, \
                                                        max_seq, nsplit, sl, bt, maxb, fused || nsplit == 1 ? out : nullptr, \
                                                        fused ? cnt : nullptr, proto);                              \
  if (out && !fused && nsplit > 1) decode_combine_kernel<DD><<<B * Hq, DD, 0, stream>>>(part_ml, part_o, out, nsplit)
  if (D == 128) { DA(128); } else if (D == 64) { DA(64); } else if (D == 32) { DA(32); } else return -1;
#undef DA
  return (int)hipGetLastError();
}

// ws: float workspace of mx_sample_ws_floats(B) elements
extern "C" int64_t mx_sample_ws_floats(int B) {
  return 2 * (int64_t)std::min(B, kSampMaxRows) * kSampMaxChunks;
}

static int sample_launch(const void* logits, int is_bf16, int64_t* out, int B, int V, float temperature,
                         uint32_t seed, uint32_t step, const float* temps, const int64_t* seeds,
                         const int32_t* steps, float* ws, hipStream_t stream) {
  if (B <= 0) return 0;
  if (V <= 0 || !ws) return -1;
  float* pv = ws;
  int* pi = reinterpret_cast<int*>(ws + (int64_t)std::min(B, kSampMaxRows) * kSampMaxChunks);
  const float it = temperature > 0.f ? 1.f / temperature : 0.f;
  int chunk = 2048, nch = (V + chunk - 1) / chunk;
  if (nch > kSampMaxChunks) {
    chunk = ((V + kSampMaxChunks - 1) / kSampMaxChunks + 255) / 256 * 256;
    nch = (V + chunk - 1) / chunk;
  }
  for (int r0 = 0; r0 < B; r0 += kSampMaxRows) {
    const dim3 grid(nch, std::min(kSampMaxRows, B - r0));
    if (is_bf16)
      sample_kernel<uint16_t><<<grid, 256, 0, stream>>>((const uint16_t*)logits, out, V, chunk, it, seed, step, r0,
                                                         temps, seeds, steps, pv, pi);
    else
      sample_kernel<float><<<grid, 256, 0, stream>>>((const float*)logits, out, V, chunk, it, seed, step, r0, temps,
                                                      seeds, steps, pv, pi);
    sample_final_kernel<<<grid.y, 64, 0, stream>>>(out, nch, r0, pv, pi);
  }
  return (int)hipGetLastError();
}

extern "C" int mx_sample(const void* logits, int is_bf16, int64_t* out, int B, int V, float temperature,
                         uint32_t seed, uint32_t step, float* ws, hipStream_t stream) {
  return sample_launch(logits, is_bf16, out, B, V, temperature, seed, step, nullptr, nullptr, nullptr, ws, stream);
}

// per-row temperature (<= 0: greedy), seed and step, no top-k / top-p: the draws of
// sampling.hip's sample_topkp_kernel for such rows (same noise), split over the vocabulary
extern "C" int mx_sample_temp_rows(const void* logits, int is_bf16, int64_t* out, int B, int V, const float* temps,
                                   const int64_t* seeds, const int32_t* steps, float* ws, hipStream_t stream) {
  return sample_launch(logits, is_bf16, out, B, V, 0.f, 0u, 0u, temps, seeds, steps, ws, stream);
}
