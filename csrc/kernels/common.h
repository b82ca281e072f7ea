// mxllm — shared device helpers for the gfx950 (CDNA4, MI355X) kernels.
//
// Conventions used by every kernel in csrc/kernels:
//  * bf16 tensors are passed as `const uint16_t*` (raw bits) so loads can be
//    vectorised as 16-byte `u16x8` (G13 of the CDNA HIP guide: hipcc never
//    auto-vectorises scalar bf16 loads).
//  * a wavefront is 64 lanes: every wave-level idiom here hard-codes 64.
//  * f32 -> bf16 goes through __float2bfloat16, which hipcc -O3 lowers to a
//    single v_cvt_pk_bf16_f32 on gfx950 (NaN-preserving, RNE).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>
#include <type_traits>

namespace mx {

constexpr int kWave = 64;

typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// Rotate-half RoPE of the pair (a, b) = (x[d], x[d + D/2]) by (c, s) = (cos, sin) of d's frequency,
// with the contraction pinned (one explicit fma each) so every kernel that applies it -- rope_split,
// the gemm8 RoPE epilogue and the tail-balanced sum pass -- produces the same bits.
__device__ __forceinline__ float rope_lo(float a, float b, float c, float s) { return __builtin_fmaf(a, c, -(b * s)); }
__device__ __forceinline__ float rope_hi(float a, float b, float c, float s) { return __builtin_fmaf(b, c, a * s); }
__device__ __forceinline__ float bf2f(uint16_t x) { return __uint_as_float(((uint32_t)x) << 16); }

__device__ __forceinline__ uint16_t f2bf(float f) {
  __hip_bfloat16 h = __float2bfloat16(f);
  return *reinterpret_cast<uint16_t*>(&h);
}

// SwiGLU gradient, s = sigmoid(g) by the hardware reciprocal:
//   dg = dm u s (1 + g (1 - s)),  du = dm g s.
// The one multiply-add is an explicit FMA and the rest are product chains, so
// -ffp-contract=fast has nothing left to contract.  Every kernel that produces
// dgu (elementwise.hip swiglu_bwd, lora.hip swiglu_lora, the gemm8 SwiGLU-backward
// epilogue) therefore gives the same bits.
__device__ __forceinline__ void swiglu_grad(float dm, float g, float u, float& dg, float& du) {
  const float s = __builtin_amdgcn_rcpf(1.f + __expf(-g));
  dg = dm * u * s * __builtin_fmaf(g, 1.f - s, 1.f);
  du = dm * g * s;
}

// two f32 -> packed bf16x2 in one u32 (lo in bits 0..15)
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  return (uint32_t)f2bf(lo) | ((uint32_t)f2bf(hi) << 16);
}

// LDS traffic of this wave done, then the workgroup's barrier: loads from memory stay in flight (__syncthreads waits
// for them)
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Folds over a wave's lanes in the vector ALU.  A shuffle (ds_bpermute) queues in the LDS pipe and its answer is waited
// for: the six dependent ones of a fold, by every wave of a workgroup at once, cost a launch of a decode step or of the
// sampler 0.3 to 1.2 us, where these take a tenth.  Same pairs in the same order as a butterfly of __shfl_xor (32, 16,
// .. 1), so sums keep their bits.  Every lane of the wave has to be on.
template <int CTRL>
__device__ __forceinline__ uint32_t lane_dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
struct LanePair {
  uint32_t a, b;
};
// The values of a lane and of lane ^ O, in either order.  O 4: where lanes i and i ^ 8 hold the same (after O 8).
// O 16, 32: a is that of the lower lane of the two.
template <int O>
__device__ __forceinline__ LanePair lane_pair(uint32_t v) {
  static_assert(O == 32 || O == 16 || O == 8 || O == 4 || O == 2 || O == 1, "a power of two");
  if constexpr (O == 32) {
    const auto s = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return {s[0], s[1]};
  } else if constexpr (O == 16) {
    const auto s = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return {s[0], s[1]};
  } else {
    // row_ror:8, row_ror:4, quad_perm [2, 3, 0, 1] and [1, 0, 3, 2]
    return {v, lane_dpp<O == 8 ? 0x128 : O == 4 ? 0x124 : O == 2 ? 0x4E : 0xB1>(v)};
  }
}
template <int O>
__device__ __forceinline__ float lane_sum(float v) {
  const LanePair p = lane_pair<O>(__float_as_uint(v));
  return __uint_as_float(p.a) + __uint_as_float(p.b);
}
template <int O>
__device__ __forceinline__ float lane_max(float v) {
  const LanePair p = lane_pair<O>(__float_as_uint(v));
  return fmaxf(__uint_as_float(p.a), __uint_as_float(p.b));
}
template <int O>
__device__ __forceinline__ int lane_sum(int v) {
  const LanePair p = lane_pair<O>((uint32_t)v);
  return (int)(p.a + p.b);
}
// the larger value, of equal ones the lower index (values are numbers)
template <int O>
__device__ __forceinline__ void lane_pick(float& v, int& i) {
  const LanePair p = lane_pair<O>(__float_as_uint(v)), q = lane_pair<O>((uint32_t)i);
  const float x = __uint_as_float(p.a), y = __uint_as_float(p.b);
  const bool other = y > x || (y == x && (int)q.b < (int)q.a);
  v = other ? y : x;
  i = (int)(other ? q.b : q.a);
}
// lanes 0 .. 15 of each sixteen
__device__ __forceinline__ float row_sum(float v) { return lane_sum<1>(lane_sum<2>(lane_sum<4>(lane_sum<8>(v)))); }
__device__ __forceinline__ float row_max(float v) { return lane_max<1>(lane_max<2>(lane_max<4>(lane_max<8>(v)))); }
__device__ __forceinline__ float wave_sum(float v) { return row_sum(lane_sum<16>(lane_sum<32>(v))); }
__device__ __forceinline__ float wave_max(float v) { return row_max(lane_max<16>(lane_max<32>(v))); }
__device__ __forceinline__ int wave_sum(int v) {
  return lane_sum<1>(lane_sum<2>(lane_sum<4>(lane_sum<8>(lane_sum<16>(lane_sum<32>(v))))));
}
__device__ __forceinline__ int row_min(int v) {
  v = min(v, (int)lane_pair<8>((uint32_t)v).b);
  v = min(v, (int)lane_pair<4>((uint32_t)v).b);
  v = min(v, (int)lane_pair<2>((uint32_t)v).b);
  return min(v, (int)lane_pair<1>((uint32_t)v).b);
}
__device__ __forceinline__ int wave_min(int v) {
  LanePair p = lane_pair<32>((uint32_t)v);
  p = lane_pair<16>((uint32_t)min((int)p.a, (int)p.b));
  return row_min(min((int)p.a, (int)p.b));
}
__device__ __forceinline__ void row_pick(float& v, int& i) {
  lane_pick<8>(v, i);
  lane_pick<4>(v, i);
  lane_pick<2>(v, i);
  lane_pick<1>(v, i);
}
__device__ __forceinline__ void wave_pick(float& v, int& i) {
  lane_pick<32>(v, i);
  lane_pick<16>(v, i);
  row_pick(v, i);
}
// what lane - n of a prefix sum's n-th step gives (zero where it has none): the steps 1, 2, 4, 8 within sixteen lanes,
// then the sums of the sixteen and the thirty-two ahead
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t lane_ahead(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false);
}
template <typename F>
__device__ __forceinline__ void wave_scan_steps(F&& f) {
  f(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xF>{});  // row_shr:1
  f(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xF>{});
  f(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xF>{});
  f(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xF>{});
  f(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xA>{});  // row_bcast:15
  f(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xC>{});  // row_bcast:31
}
// the value of lane l (the same l in every lane)
__device__ __forceinline__ unsigned long long lane_value(unsigned long long v, int l) {
  return ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), l) << 32) |
         (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
// sums over lanes 0 .. this one
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
  wave_scan_steps([&](auto c, auto r) { v += lane_ahead<c.value, r.value>(v); });
  return v;
}
__device__ __forceinline__ unsigned long long wave_scan(unsigned long long v) {
  wave_scan_steps([&](auto c, auto r) {
    const uint32_t lo = lane_ahead<c.value, r.value>((uint32_t)v), hi = lane_ahead<c.value, r.value>((uint32_t)(v >> 32));
    v += ((unsigned long long)hi << 32) | lo;
  });
  return v;
}

// Block-wide sum for blockDim.x <= 1024. `scratch` must hold >= 16 floats.
// Every thread receives the result.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = (blockDim.x + 63) >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  float r = 0.f;
  for (int i = 0; i < nw; i += 4) {  // (four on their way at once)
#pragma unroll
    for (int j = 0; j < 4; ++j) r += i + j < nw ? scratch[i + j] : 0.f;
  }
  return r;
}

__device__ __forceinline__ float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = (blockDim.x + 63) >> 6;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  float r = -INFINITY;
  for (int i = 0; i < nw; i += 4) {
#pragma unroll
    for (int j = 0; j < 4; ++j) r = fmaxf(r, i + j < nw ? scratch[i + j] : -INFINITY);
  }
  return r;
}

// XCD-aware, bijective remap of a 1-D workgroup id (guide §5, "XCD swizzle must
// be bijective"): consecutive logical tiles land on the same XCD (shared L2).
// Speed only — correctness never depends on placement.
__device__ __forceinline__ int xcd_remap(int orig, int nwg) {
  const int q = nwg >> 3, r = nwg & 7, xcd = orig & 7;
  return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
}

// Bijective remap for grids of (outer, bh) work items, bid = outer * BH + bh, whose cost
// varies with `outer` (causal attention: heaviest outer index first).  Workgroups are dealt
// round-robin over the 8 XCDs (MI355X_MICROARCH "Workgroup dispatch"): blocks b, b + 8, ...
// share one.  xcd_remap above gives each XCD a CONTIGUOUS bid range, i.e. a narrow band of
// outer indices, so one XCD ran all the heavy blocks while another idled (causal attention
// at B2 Hq64: 644 µs where the per-CU work is ~410).  Here XCD x takes the KV groups (G
// consecutive q-heads sharing one K/V head) {x, x + 8, ...} -> K / V stay in one L2 -- and
// walks them through every outer index in dispatch order, so every XCD sees the same
// heavy-to-light mix.  Falls back to identity (round-robin already balances) when BH is not
// a multiple of 8 G.
__device__ __forceinline__ int xcd_balance(int orig, int nwg, int BH, int G) {
  if ((nwg & 7) || G <= 0 || BH % (8 * G) || nwg % BH) return orig;
  const int x = orig & 7, j = orig >> 3, per = BH >> 3;
  const int outer = j / per, lb = j % per;
  const int bh = ((lb / G) * 8 + x) * G + lb % G;
  return outer * BH + bh;
}

// ---- KV cache addressing (decode kernels) ----
// Per layer the cache is [rows, Hkv, SEQ, D] bf16.  Contiguous (bt == nullptr): rows =
// slots, SEQ = max_seq.  Paged (bt = block table [slots, maxb] int32): rows = pool blocks,
// SEQ = the block size; token p of slot s lives in block bt[s][p / SEQ] at row p % SEQ.
// Returns the token-row index (multiply by D for the element offset).
__device__ __forceinline__ int64_t kv_row(const int32_t* __restrict__ bt, int maxb, int seq, int slot, int Hkv,
                                          int hk, int p) {
  if (!bt) return ((int64_t)slot * Hkv + hk) * seq + p;
  const int blk = bt[(int64_t)slot * maxb + p / seq];
  return ((int64_t)blk * Hkv + hk) * seq + (p % seq);
}

// ---- LDS-DMA-friendly transposed reads (used by the attention kernels) ----
// ds_read_b64_tr_b16 as inline asm with an immediate offset: invisible to hipcc's
// waitcnt pass, which otherwise drains every in-flight LDS-DMA (vmcnt(0)) before a
// builtin tr-read (it cannot tell that the read misses the DMA's buffer).  The caller
// waits with lds_wait() / lds_wait_le() and pins each result behind the wait with pin().
// LDS operations of a wave complete in order, so counted lgkmcnt waits are exact for
// the asm reads and conservative for anything the compiler interleaves.
template <int OFF>
__device__ __forceinline__ u16x4 trd_asm(uint32_t lds_addr) {
  u16x4 v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(lds_addr), "i"(OFF));
  return v;
}
// transposed read at base + off; `off` folds into the instruction's immediate when it
// is a compile-time constant < 64 KiB
__device__ __forceinline__ u16x4 trd_off(uint32_t base, int off) {
  u16x4 v;
  if (__builtin_constant_p(off) && off >= 0 && off < 65536)
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(base), "i"(off));
  else
    asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(v) : "v"(base + (uint32_t)off));
  return v;
}
// 16-B row read at base + off (immediate when constant), same waitcnt contract as trd_off
__device__ __forceinline__ u16x8 rd128_off(uint32_t base, int off) {
  u16x8 v;
  if (__builtin_constant_p(off) && off >= 0 && off < 65536)
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(base), "i"(off));
  else
    asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(base + (uint32_t)off));
  return v;
}
__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// at most n LDS operations of this wave still outstanding (n folds to a constant after unrolling)
__device__ __forceinline__ void lds_wait_le(int n) {
  switch (n) {
#define MX_LGKM(N) case N: asm volatile("s_waitcnt lgkmcnt(" #N ")" ::: "memory"); break;
    MX_LGKM(15) MX_LGKM(14) MX_LGKM(13) MX_LGKM(12) MX_LGKM(11) MX_LGKM(10) MX_LGKM(9) MX_LGKM(8)
    MX_LGKM(7) MX_LGKM(6) MX_LGKM(5) MX_LGKM(4) MX_LGKM(3) MX_LGKM(2) MX_LGKM(1)
#undef MX_LGKM
    default: asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); break;
  }
}
__device__ __forceinline__ void pin(u16x4& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void pin(u16x8& v) { asm volatile("" : "+v"(v)); }
// byte address of a __shared__ object in the LDS aperture
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(size_t)(__attribute__((address_space(3))) const char*)p;
}

}  // namespace mx

#define MX_CHECK_LAUNCH() (void)hipGetLastError()
