// Latent attention on the matrix cores (gfx950, bf16 storage, f32 scores and sums):
//   * latent_flash : prompt rows on expanded keys and values, heads up to 256 + 128 dims.  A workgroup takes
//                    128 query rows of one head and walks 64-key tiles, double-buffered in LDS by LDS-DMA; a
//                    key row's unrotated dims come from the expanded keys, the rotated ones from the
//                    latent rows that all heads share.  S^T = K Q^T with v_mfma_f32_32x32x16_bf16 (a
//                    lane owns one query column), O^T += V^T P^T with transposed LDS reads of V.  Windows
//                    skip the tiles ahead of them; the sink is the softmax's start value.
//   * latent_split : decode.  All heads attend to the same cached rows, so 16 or 32 heads are one side of
//                    the MFMA tile: S = K Q^T and O = P V on one 32-key image in LDS, whose rows are key
//                    and (first `rank` columns) value at once; split over the keys;
//   * latent_heads / latent_merge : decode queries taken onto the latent (with the new tokens' cache rows in the
//                    same launch), split partials merged, and the merged latents through W_uv.
#include "hybrid.h"
#include "latent_row.h"
#include "sublayer.h"

namespace mx {

typedef __bf16 bf16x8_l __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(1))) const void* lgptr_t;
typedef __attribute__((address_space(3))) void* llptr_t;

__device__ __forceinline__ f32x16 lm_mfma32(const u16x8& a, const u16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_l, a), __builtin_bit_cast(bf16x8_l, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 lm_mfma16(const u16x8& a, const u16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_l, a), __builtin_bit_cast(bf16x8_l, b), c, 0, 0, 0);
}
// 16-B chunk swizzle of a row image of `ch` chunks: rows spread over the chunks of the largest power of two
// (at most 16) that divides the row, so 16 rows at one logical chunk fall on 16 different bank groups
__host__ __device__ constexpr int lm_group(int ch) { return ch % 16 == 0 ? 16 : ch % 8 == 0 ? 8 : ch % 4 == 0 ? 4 : 2; }
__device__ __forceinline__ int lm_swz(int row, int grp) { return (row & 15) / (16 / grp); }
// the value image's: also conflict-free for transposed reads of 4 rows
template <int CH>
__device__ __forceinline__ int lm_vswz(int row) {
  return (((row & 3) << 2) | ((row >> 2) & 3)) & (CH - 1);
}

// ------------------------------------------------------------------ prompts
// What bounds it: a wave's own chain through a tile (products a quarter of the time, the softmax's instructions as much, LDS reads and
// their waits between), two waves a SIMD.  So a row image's fragments are asked for PF - 1 steps ahead of their products and a value's
// PV - 1 (more is level), and a tile's sources are pointers that move on by a tile, where all its rows are there, instead of 200 address
// instructions.  32 heads, causal / a window of 1024, us: 192 + 128 dims, 2048 rows 75.6 / 62.3 -> 67.5 / 57.3, 3000 125.7 / 90.6 ->
// 117.1 / 83.5, 1024 38.9 -> 33.8; 96 + 64 dims, 2048 rows 47.5 / 38.1 -> 41.4 / 35.2.  Row strides that spread a head's rows over the
// L2's channels are level.
template <int DK, int DV>
__global__ void __launch_bounds__(256, 2) latent_flash_kernel(LatentAttn a) {
  constexpr int BM = 128, BN = 64, CK = DK / 8, CV = DV / 8, KS = DK / 16, DB = DV / 32, G = lm_group(CK), PF = 3, PV = 4;
  constexpr int KT = BN * CK * 16, VT = BN * CV * 16, LK = CK / 4, LV = CV / 4;  // DMA pieces per wave
  __shared__ __attribute__((aligned(1024))) char smem[2 * (KT + VT)];
  // Blocks come longest first.  Where all workgroups are on the chip at once, two a CU, nothing is dealt as CUs become free: those of the
  // second round go shortest first, so that the longest shares its CU with the shortest (2048 rows of 32 heads, 192 + 128 dims, causal
  // 77.0 -> 75.6 us, 96 + 64 dims 49.1 -> 47.5; a window of 1024 is level).
  const int bid = blockIdx.x, h = bid % a.H, blk = bid / a.H, ahead = 256 / a.H;
  const int4 sg = reinterpret_cast<const int4*>(a.blocks)[(int)gridDim.x <= 512 && blk >= ahead ? ahead + a.nblocks - 1 - blk : blk];
  const int64_t row0 = sg.x;
  const int S = sg.y, q0 = sg.z * BM;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, hh = lane >> 5;
  const int qrow = q0 + 32 * w + r, qld = min(qrow, S - 1);
  const int DQ = a.D + a.R;

  u16x8 qf[KS];
  {
    const uint16_t* qp = reinterpret_cast<const uint16_t*>(a.q) + (row0 + qld) * a.ldq + (int64_t)h * DQ;
    const int half = a.R / 2;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int d = 16 * s + 8 * hh;
      u16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
      if (d < DQ) v = *reinterpret_cast<const u16x8*>(qp + d);
      if (d >= a.D && d < DQ) {  // interleaved pairs, position = row in its sequence
        const int64_t t = (int64_t)qld * half + (d - a.D) / 2;
        const f32x4 c = *reinterpret_cast<const f32x4*>(a.cosb + t), sn = *reinterpret_cast<const f32x4*>(a.sinb + t);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float x = bf2f(v[2 * j]), y = bf2f(v[2 * j + 1]);
          v[2 * j] = f2bf(x * c[j] - y * sn[j]);
          v[2 * j + 1] = f2bf(y * c[j] + x * sn[j]);
        }
      }
      qf[s] = v;
    }
  }

  const int kend = min(S, q0 + BM), ntiles = (kend + BN - 1) / BN;
  const int t0 = a.window > 0 ? max(0, q0 - a.window + 1) / BN : 0;
  // sources of this lane's pieces: byte address of row 0 of the sequence, and the row stride in bytes
  const char* kb = reinterpret_cast<const char*>(reinterpret_cast<const uint16_t*>(a.kv) + row0 * a.ldkv + (int64_t)h * a.D);
  const char* rb = reinterpret_cast<const char*>(reinterpret_cast<const uint16_t*>(a.lat) + row0 * a.ldl + a.rank);
  const char* vb = reinterpret_cast<const char*>(reinterpret_cast<const uint16_t*>(a.kv) + row0 * a.ldkv +
                                                 (int64_t)a.H * a.D + (int64_t)h * a.E);
  const int cd = a.D / 8, cr = DQ / 8, ce = a.E / 8;
  // this lane's sources in the next whole tile, and the bytes to the tile behind it
  const char* kp[LK];
  uint32_t vo[LV], rot = 0;  // rot, bit i: piece i is of the rotated dims
  const uint32_t kstep = (uint32_t)(BN * 2 * a.ldkv), rstep = (uint32_t)(BN * 2 * a.ldl);
  auto source = [&](int i, int ln, int64_t t) __attribute__((always_inline)) {
    const int idx = (w * LK + i) * 64 + ln, row = idx / CK, c = (idx % CK) ^ lm_swz(row, G);
    const int64_t kr = min(t + row, (int64_t)S - 1);
    // chunks past the head's dims repeat the first one (their query dims are zero)
    return c < cd ? kb + kr * (a.ldkv * 2) + 16 * c : c < cr ? rb + kr * (a.ldl * 2) + 16 * (c - cd) : kb + kr * (a.ldkv * 2);
  };
  auto vsource = [&](int i, int ln, int last) __attribute__((always_inline)) {
    const int idx = (w * LV + i) * 64 + ln, row = idx / CV, c = (idx % CV) ^ lm_vswz<CV>(row);
    return (uint32_t)(min(row, last) * (int)(a.ldkv * 2) + (c < ce ? 16 * c : 0));  // columns past E are not stored
  };
#pragma unroll
  for (int i = 0; i < LK; ++i) {
    const int idx = (w * LK + i) * 64 + lane, row = idx / CK, c = (idx % CK) ^ lm_swz(row, G);
    kp[i] = source(i, lane, (int64_t)t0 * BN);
    rot |= (uint32_t)(c >= cd && c < cr) << i;
  }
#pragma unroll
  for (int i = 0; i < LV; ++i) vo[i] = vsource(i, lane, BN - 1);
  auto issue = [&](int kt, int buf) __attribute__((always_inline)) {
    char* kd = smem + buf * (KT + VT) + w * (LK * 1024);
    char* vd = smem + buf * (KT + VT) + KT + w * (LV * 1024);
    const char* vt = vb + (int64_t)kt * (BN * 2) * a.ldkv;
    if (kt * BN + BN > S) {  // a tile that the sequence ends in: rows past it repeat the last one
      int ln = lane;
      asm volatile("" : "+v"(ln));  // (else what this takes is kept in registers through the loop)
#pragma unroll
      for (int i = 0; i < LK; ++i) kp[i] = source(i, ln, (int64_t)kt * BN);
#pragma unroll
      for (int i = 0; i < LV; ++i) vo[i] = vsource(i, ln, S - 1 - kt * BN);
    }
#pragma unroll
    for (int i = 0; i < LK; ++i) {
      __builtin_amdgcn_global_load_lds((lgptr_t)kp[i], (llptr_t)(kd + i * 1024), 16, 0, 0);
      kp[i] += rot >> i & 1 ? rstep : kstep;
    }
#pragma unroll
    for (int i = 0; i < LV; ++i) {
      __builtin_amdgcn_global_load_lds((lgptr_t)(vt + vo[i]), (llptr_t)(vd + i * 1024), 16, 0, 0);
    }
  };

  f32x16 o[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[d][j] = 0.f;
  const float sl = a.scale * 1.4426950408889634f;
  float m_i = a.sink ? a.sink[h] * 1.4426950408889634f : -1e30f, l_i = a.sink && hh == 0 ? 1.f : 0.f;

  const int gq = lane >> 4, li = lane & 15, tq = li >> 2, tp = li & 3;
  const uint32_t lds0 = lds_addr(smem);
  uint32_t va[DB][2];
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    const int chunk = (db * 32 + 16 * (gq & 1) + 4 * tp) >> 3;
    const int rA = 4 * hh + tq, rB = 8 + 4 * hh + tq;
    va[db][0] = lds0 + KT + rA * (CV * 16) + 16 * (chunk ^ lm_vswz<CV>(rA)) + 8 * (tp & 1);
    va[db][1] = lds0 + KT + rB * (CV * 16) + 16 * (chunk ^ lm_vswz<CV>(rB)) + 8 * (tp & 1);
  }
  const uint32_t kq = lds0 + r * (CK * 16) + 16 * (hh ^ lm_swz(r, G));
  issue(t0, 0);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), seen by the compiler: else it waits for the query loads in the loop
  __builtin_amdgcn_s_barrier();

  for (int kt = t0; kt < ntiles; ++kt) {
    const uint32_t bo = (uint32_t)((kt - t0) & 1) * (KT + VT);
    if (kt + 1 < ntiles) issue(kt + 1, (kt - t0 + 1) & 1);
    // this wave's rows see some key of the tile
    const bool active = kt * BN <= q0 + 32 * w + 31 && (a.window == 0 || kt * BN + BN - 1 > q0 + 32 * w - a.window);
    if (active) {
      f32x16 sacc[2];
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int j = 0; j < 16; ++j) sacc[n][j] = 0.f;
      u16x8 kf[PF][2];
      auto ld = [&](int st, u16x8(&x)[2]) __attribute__((always_inline)) {
        const int lo = (2 * st) & (G - 1), hi = (2 * st) & ~(G - 1);
        const uint32_t ad = (kq ^ (uint32_t)(16 * lo)) + bo;
        x[0] = rd128_off(ad, 16 * hi);
        x[1] = rd128_off(ad, 16 * hi + 32 * CK * 16);
      };
#pragma unroll
      for (int st = 0; st < PF - 1 && st < KS; ++st) ld(st, kf[st]);
#pragma unroll
      for (int st = 0; st < KS; ++st) {
        if (st + PF - 1 < KS) ld(st + PF - 1, kf[(st + PF - 1) % PF]);
        lds_wait_le(2 * (KS - 1 - st < PF - 1 ? KS - 1 - st : PF - 1));
        u16x8(&x)[2] = kf[st % PF];
        pin(x[0]);
        pin(x[1]);
        sacc[0] = lm_mfma32(x[0], qf[st], sacc[0]);
        sacc[1] = lm_mfma32(x[1], qf[st], sacc[1]);
      }
      float mp[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      const bool mask = kt * BN + BN - 1 > q0 + 32 * w || kt * BN + BN > S ||
                        (a.window > 0 && kt * BN <= q0 + 32 * w + 31 - a.window);
      if (mask) {
        const int lo = a.window > 0 ? qrow - a.window : -1;
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const int key = kt * BN + n * 32 + (j & 3) + 8 * (j >> 2) + 4 * hh;
            const float x = ((key > qrow) | (key <= lo) | (key >= S)) ? -INFINITY : sacc[n][j];
            sacc[n][j] = x;
            mp[j & 3] = fmaxf(mp[j & 3], x);
          }
      } else {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int j = 0; j < 16; ++j) mp[j & 3] = fmaxf(mp[j & 3], sacc[n][j]);
      }
      float mx = fmaxf(fmaxf(mp[0], mp[1]), fmaxf(mp[2], mp[3]));
      {  // the other half of this query's keys
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      }
      // rescale only when some row's maximum grows by more than 2^8
      const float mt = mx * sl;
      if (__any(mt > m_i + 8.f)) {
        const float mn = fmaxf(m_i, mt), al = __builtin_amdgcn_exp2f(m_i - mn);
        l_i *= al;
        m_i = mn;
#pragma unroll
        for (int d = 0; d < DB; ++d) o[d] *= al;
      }
      float lp[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[n][j], sl, -m_i));
          sacc[n][j] = p;
          lp[j & 3] += p;
        }
      l_i += (lp[0] + lp[1]) + (lp[2] + lp[3]);
      // (16 keys, 32 columns) of the values at a time, PV - 1 of them asked for ahead
      constexpr int NV = 4 * DB;
      u16x4 fv[PV][2];
      auto ldv = [&](int i) __attribute__((always_inline)) {
        fv[i % PV][0] = trd_off(va[i % DB][0] + bo, 16 * (i / DB) * (CV * 16));
        fv[i % PV][1] = trd_off(va[i % DB][1] + bo, 16 * (i / DB) * (CV * 16));
      };
#pragma unroll
      for (int i = 0; i < PV - 1; ++i) ldv(i);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        u16x8 pb;
#pragma unroll
        for (int j = 0; j < 8; ++j) pb[j] = f2bf(sacc[q >> 1][8 * (q & 1) + j]);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const int i = q * DB + db;
          if (i + PV - 1 < NV) ldv(i + PV - 1);
          lds_wait_le(2 * (NV - 1 - i < PV - 1 ? NV - 1 - i : PV - 1));
          u16x4(&f)[2] = fv[i % PV];
          pin(f[0]);
          pin(f[1]);
          o[db] = lm_mfma32(u16x8{f[0][0], f[0][1], f[0][2], f[0][3], f[1][0], f[1][1], f[1][2], f[1][3]}, pb, o[db]);
        }
      }
    }
    lds_wait();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the next tile landed
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_i), __float_as_uint(l_i), false, false);
  const float l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]), inv = l > 0.f ? 1.f / l : 0.f;
  if (qrow < S) {
    uint16_t* op = reinterpret_cast<uint16_t*>(a.out) + ((row0 + qrow) * a.H + h) * (int64_t)a.E;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int d = db * 32 + 8 * q4 + 4 * hh;
        if (d >= a.E) continue;
        u16x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = f2bf(o[db][4 * q4 + j] * inv);
        *reinterpret_cast<u16x4*>(op + d) = v;
      }
  }
}

// ------------------------------------------------------------------ decode
// LDS accesses as inline asm: the compiler would otherwise wait for the DMA in flight ahead of them
__device__ __forceinline__ float lm_rd32(uint32_t a) {
  float v;
  asm volatile("ds_read_b32 %0, %1" : "=v"(v) : "v"(a));
  return v;
}
__device__ __forceinline__ void lm_wr128(uint32_t a, const f32x4& v) { asm volatile("ds_write_b128 %0, %1" ::"v"(a), "v"(v) : "memory"); }
__device__ __forceinline__ void lm_wr64(uint32_t a, const u16x4& v) { asm volatile("ds_write_b64 %0, %1" ::"v"(a), "v"(v) : "memory"); }
__device__ __forceinline__ void lm_wr32(uint32_t a, float v) { asm volatile("ds_write_b32 %0, %1" ::"v"(a), "v"(v) : "memory"); }
template <int CTRL>
__device__ __forceinline__ float lm_dpp(float v) {
  return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ void lm_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

constexpr int kLsKeys = 32, kLsRow = 144;  // bytes of a head's scores (f32), then weights (bf16), and its rescale factor

// KS: 32-element steps of a cached row (rows are wc <= 32 KS wide); MB blocks of 16 heads.  LDS: two key
// images, the score rows.  4 waves: scores by (16 keys, head block), softmax 8 threads a head, value
// columns 16 (w + 4 j) by wave.
template <int KS, int MB>
__global__ void __launch_bounds__(256, KS <= 18 ? 2 : 1) latent_split_kernel(LatentDecode a) {
  constexpr int RB = (KS + 1) / 2;
  extern __shared__ __attribute__((aligned(1024))) char lsm[];
  const int split = blockIdx.x, h0 = blockIdx.y * 16 * MB, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int p = a.pos[b], slot = a.slots[b];
  const int vis = a.window > 0 ? min(p + 1, a.window) : p + 1, first = p + 1 - vis;
  const int k0 = split * a.span, n = min(a.span, vis - k0);
  if (n <= 0) {
    if (tid < 16 * MB && h0 + tid < a.H) {
      float* ml = a.ml + (((int64_t)b * a.H + h0 + tid) * a.nsplit + split) * 2;
      ml[0] = -INFINITY;
      ml[1] = 0.f;
    }
    return;
  }
  const int CK = a.wc / 8, rowb = a.wc * 2, grp = lm_group(CK), img = (kLsKeys * rowb + 1023) / 1024 * 1024;
  const uint32_t lds0 = lds_addr(lsm), sb = lds0 + 2 * img;
  const char* pool = reinterpret_cast<const char*>(a.pool);
  // wave w stages rows 8 w .. 8 w + 7 of a tile in pieces of 64 chunks: this lane's row and byte in it
  constexpr int PC = (KS + 1) / 2;
  int prow[PC], pcol[PC];
#pragma unroll
  for (int i = 0; i < PC; ++i) {
    const int idx = i * 64 + lane, row = idx / CK;
    prow[i] = row < 8 ? 8 * w + row : -1;
    pcol[i] = 16 * ((idx - row * CK) ^ lm_swz(8 * w + row, grp));
  }
  // the split's blocks (a split is at most 512 keys, a block at least 256), read once
  const int r0 = (first + k0) % a.ring, blk0 = a.bt ? r0 / a.seq : 0;
  int ba = slot, bb = slot, bc = slot;  // (one ring per slot: its rows are the slot's)
  const int ring = a.ring, seq = a.seq;
  const bool paged = a.bt != nullptr;
  if (paged) {
    const int32_t* row = a.bt + (int64_t)slot * a.maxb;
    ba = __builtin_amdgcn_readfirstlane(row[blk0]);
    bb = __builtin_amdgcn_readfirstlane(row[min(blk0 + 1, a.maxb - 1)]);
    bc = __builtin_amdgcn_readfirstlane(row[min(blk0 + 2, a.maxb - 1)]);
  }
  // a tile's rows are consecutive in the pool but for one cut (the ring's end, a block's edge)
  auto issue = [&](int t) __attribute__((always_inline)) {
    const int left = n - t * kLsKeys;  // rows past the last key repeat it
    int ra = r0 + t * kLsKeys;
    while (ra >= ring) ra -= ring;
    const int bi = ra / seq, in = ra - bi * seq, i = bi - blk0;
    const int cut = min(ring - ra, seq - in);
    const int x0 = ba, x1 = bb, x2 = bc;  // (selecting among the captures themselves goes through memory)
    const int ida = i == 0 ? x0 : i == 1 ? x1 : x2;
    const int rb = paged ? 0 : ra + cut == ring ? 0 : ra + cut;  // past the cut: the next block's first row, or the ring's
    const int idb = i == 0 ? x1 : x2;
    const char* pa = pool + ((int64_t)ida * seq + in) * rowb;
    const char* pb = pool + ((int64_t)idb * seq + rb) * rowb;
    char* dst = lsm + (t & 1) * img + 8 * w * rowb;
#pragma unroll
    for (int i = 0; i < PC; ++i) {
      const int row = min(prow[i], left - 1);
      const char* p = (row < cut ? pa : pb) + (row < cut ? row : row - cut) * rowb + pcol[i];
      if (prow[i] >= 0) __builtin_amdgcn_global_load_lds((lgptr_t)p, (llptr_t)(dst + i * 1024), 16, 0, 0);
    }
  };
  const int ntiles = (n + kLsKeys - 1) / kLsKeys;
  issue(0);

  const bool scorer = MB == 2 || w < 2;
  const int kblk = w & 1, hb = MB == 2 ? w >> 1 : 0;
  u16x8 qf[KS];
  {
    const int hq = min(h0 + 16 * hb + c, a.H - 1);
    const uint16_t* q = reinterpret_cast<const uint16_t*>(a.qa) + ((int64_t)b * a.H + hq) * a.wq;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int d = 32 * s + 8 * g;
      qf[s] = d < a.wq ? *reinterpret_cast<const u16x8*>(q + d) : u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  f32x4 acc[RB][MB];
#pragma unroll
  for (int j = 0; j < RB; ++j)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[j][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_i = -INFINITY, l_i = 0.f;  // of head tid / 8 (softmax threads)
  const float sl = a.scale * 1.4426950408889634f;
  const int krow = 16 * kblk + c, ksw = lm_swz(krow, grp);
  const int tq = c >> 2, tp = c & 3;

  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), seen by the compiler: else it waits for the query loads in the loop
  for (int t = 0; t < ntiles; ++t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lm_barrier();  // tile t staged; the other image and the score rows are free
    if (t + 1 < ntiles) issue(t + 1);
    const uint32_t kbuf = lds0 + (t & 1) * img;
    if (scorer) {
      f32x4 s4 = {0.f, 0.f, 0.f, 0.f};
      constexpr int U = 6;
#pragma unroll
      for (int s0 = 0; s0 < KS; s0 += U) {
        u16x8 kf[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (s0 + u < KS) {
            const int ch = min(4 * (s0 + u) + g, CK - 1);  // steps past the row meet zero queries
            kf[u] = rd128_off(kbuf + krow * rowb + 16 * (ch ^ ksw), 0);
          }
        lds_wait();
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (s0 + u < KS) {
            pin(kf[u]);
            s4 = lm_mfma16(kf[u], qf[s0 + u], s4);
          }
      }
      // (scaled here: the compiler places the wait between an MFMA and a VALU instruction, not ahead of inline asm)
      lm_wr128(sb + (16 * hb + c) * kLsRow + (16 * kblk + 4 * g) * 4, s4 * sl);  // keys 4 g .. of head c
    }
    lm_barrier();
    const int sh = tid >> 3, part = tid & 7;
    if (sh < 16 * MB) {
      u16x8 raw = rd128_off(sb + sh * kLsRow + part * 16, 0);
      lds_wait();
      pin(raw);
      f32x4 s = __builtin_bit_cast(f32x4, raw);
      float mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[i] = t * kLsKeys + 4 * part + i < n ? s[i] : -INFINITY;
        mx = fmaxf(mx, s[i]);
      }
      mx = fmaxf(mx, lm_dpp<0xB1>(mx));   // lane ^ 1
      mx = fmaxf(mx, lm_dpp<0x4E>(mx));   // lane ^ 2
      mx = fmaxf(mx, lm_dpp<0x141>(mx));  // the other four of eight
      const float mn = fmaxf(m_i, mx), al = __builtin_amdgcn_exp2f(m_i - mn);
      float sum = 0.f;
      u16x4 pb;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = __builtin_amdgcn_exp2f(s[i] - mn);
        sum += e;
        pb[i] = f2bf(e);
      }
      sum += lm_dpp<0xB1>(sum);
      sum += lm_dpp<0x4E>(sum);
      sum += lm_dpp<0x141>(sum);
      m_i = mn;
      l_i = l_i * al + sum;
      // the row's scores are in the registers of its 8 threads, all of this wave
      lm_wr64(sb + sh * kLsRow + part * 8, pb);
      if (part == 0) lm_wr32(sb + sh * kLsRow + 128, al);
    }
    lm_barrier();
    u16x8 pf[MB];
    float al[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      pf[mb] = rd128_off(sb + (16 * mb + c) * kLsRow + 16 * g, 0);
      al[mb] = lm_rd32(sb + (16 * mb + c) * kLsRow + 128);
    }
    lds_wait();
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      pin(pf[mb]);
      asm volatile("" : "+v"(al[mb]));
    }
#pragma unroll
    for (int j0 = 0; j0 < RB; j0 += 3) {
      u16x4 v[3][2];
#pragma unroll
      for (int u = 0; u < 3; ++u)
        if (j0 + u < RB) {
          const int ch = min(2 * (w + 4 * (j0 + u)) + (tp >> 1), CK - 1);  // blocks past the rank are not stored
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const int row = 8 * g + 4 * x + tq;
            v[u][x] = trd_off(kbuf + row * rowb + 16 * (ch ^ lm_swz(row, grp)) + 8 * (tp & 1), 0);
          }
        }
      lds_wait();
#pragma unroll
      for (int u = 0; u < 3; ++u)
        if (j0 + u < RB) {
          pin(v[u][0]);
          pin(v[u][1]);
          const u16x4 x = v[u][0], y = v[u][1];
          const u16x8 vf = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) acc[j0 + u][mb] = lm_mfma16(vf, pf[mb], acc[j0 + u][mb] * al[mb]);
        }
    }
  }
  if ((tid & 7) == 0 && (tid >> 3) < 16 * MB && h0 + (tid >> 3) < a.H) {
    float* ml = a.ml + (((int64_t)b * a.H + h0 + (tid >> 3)) * a.nsplit + split) * 2;
    ml[0] = m_i;
    ml[1] = l_i;
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int h = h0 + 16 * mb + c;
    if (h >= a.H) continue;
    float* po = a.po + (((int64_t)b * a.H + h) * a.nsplit + split) * a.rank;
#pragma unroll
    for (int j = 0; j < RB; ++j) {
      const int col = 16 * (w + 4 * j) + 4 * g;
      if (col < a.rank) *reinterpret_cast<f32x4*>(po + col) = acc[j][mb];  // rank is a multiple of 4
    }
  }
}

// ------------------------------------------------------------------ decode: products per head
// Y[b, h] = W[h] X[b, h] on 16 MB tokens, a wave 16 of the head's output channels.  QUERY: W_uk transposed
// ([H, rank, D]) on the unrotated query; one more workgroup per head rotates the rest of the query and stores
// the new tokens' latent rows (one wave a row).  Else: W_uv on the merged latents.
template <int MB, bool QUERY>
__global__ void __launch_bounds__(256) latent_heads_kernel(LatentDecode a, LatentRows rw) {
  const int N = QUERY ? a.rank : a.E, K = QUERY ? a.D : a.rank, h = blockIdx.y, b0 = blockIdx.z * 16 * MB;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int nb = min(16 * MB, a.B - b0);
  if constexpr (QUERY) {
    if (blockIdx.x == gridDim.x - 1) {
      const int half = a.R / 2, pad = a.wq - a.rank - a.R;
      const uint16_t* q = reinterpret_cast<const uint16_t*>(a.q) + (int64_t)h * (a.D + a.R) + a.D;
      uint16_t* qa = reinterpret_cast<uint16_t*>(a.qa) + (int64_t)h * a.wq + a.rank;
      for (int i = threadIdx.x; i < nb * half; i += 256) {
        const int b = b0 + i / half, k = i % half;
        float u = bf2f(q[b * a.ldq + 2 * k]), v = bf2f(q[b * a.ldq + 2 * k + 1]);
        latent_turn(a.cosb, a.sinb, half, a.pos[b], k, u, v);
        uint16_t* o = qa + (int64_t)b * a.H * a.wq + 2 * k;
        o[0] = f2bf(u);
        o[1] = f2bf(v);
      }
      for (int i = threadIdx.x; i < nb * pad; i += 256) qa[(int64_t)(b0 + i / pad) * a.H * a.wq + a.R + i % pad] = 0;
      if (rw.x)
        for (int i = h * 4 + w; i < nb; i += a.H * 4) {
          const int b = b0 + i;
          latent_row<uint16_t>(rw, b, a.pos[b], a.slots[b], a.pos[b] + 1, lane);
        }
      return;
    }
  }
  const int n0 = (blockIdx.x * 4 + w) * 16;
  if (n0 >= N) return;
  const uint16_t* wr = reinterpret_cast<const uint16_t*>(QUERY ? a.wuk_t : a.wuv) +
                       ((int64_t)h * N + min(n0 + c, N - 1)) * K;
  const uint16_t* xr[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int b = b0 + min(16 * mb + c, nb - 1);
    xr[mb] = QUERY ? reinterpret_cast<const uint16_t*>(a.q) + b * a.ldq + (int64_t)h * (a.D + a.R)
                   : reinterpret_cast<const uint16_t*>(a.om) + ((int64_t)b * a.H + h) * a.rank;
  }
  f32x4 acc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int U = MB == 1 ? 8 : 4;
  for (int kb = 0; kb < K; kb += 64 * U) {
    u16x8 fa[U][2], fb[U][MB][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = kb + 64 * u + 16 * g;
      const bool on = k < K;  // K is a multiple of 16
      const int kk = on ? k : 0;
      fa[u][0] = *reinterpret_cast<const u16x8*>(wr + kk);
      fa[u][1] = *reinterpret_cast<const u16x8*>(wr + kk + 8);
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
      for (int mb = 0; mb < MB; ++mb) {
        acc[mb] = lm_mfma16(fa[u][0], fb[u][mb][0], acc[mb]);
        acc[mb] = lm_mfma16(fa[u][1], fb[u][mb][1], acc[mb]);
      }
  }
  const int n = n0 + 4 * g;
  if (n >= N) return;  // N is a multiple of 4
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int b = b0 + 16 * mb + c;
    if (b - b0 >= nb) continue;
    uint16_t* y = QUERY ? reinterpret_cast<uint16_t*>(a.qa) + ((int64_t)b * a.H + h) * a.wq + n
                        : reinterpret_cast<uint16_t*>(a.out) + ((int64_t)b * a.H + h) * a.E + n;
    u16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = f2bf(acc[mb][i]);
    *reinterpret_cast<u16x4*>(y) = o;
  }
}

// split partials and the sink -> the head's latent om [B, H, rank]
constexpr int kLmSplits = 1024;
__global__ void __launch_bounds__(256) latent_merge_kernel(LatentDecode a) {
  __shared__ float ws[kLmSplits];
  __shared__ float scratch[16];
  const int h = blockIdx.x, b = blockIdx.y, t = threadIdx.x;
  const int64_t bh = (int64_t)b * a.H + h;
  const float* ml = a.ml + bh * a.nsplit * 2;
  const float sk = a.sink ? a.sink[h] * 1.4426950408889634f : -INFINITY;
  float m = sk;
  for (int s = t; s < a.nsplit; s += 256) m = fmaxf(m, ml[2 * s]);
  m = block_max(m, scratch);
  float l = a.sink && t == 0 ? exp2f(sk - m) : 0.f;
  for (int s = t; s < a.nsplit; s += 256) {
    const float x = ml[2 * s], e = x > -INFINITY ? exp2f(x - m) : 0.f;
    ws[s] = e;
    if (e > 0.f) l += e * ml[2 * s + 1];
  }
  l = block_sum(l, scratch);  // (its barriers publish ws)
  const float inv = 1.f / l;
  const float* po = a.po + bh * a.nsplit * a.rank;
  uint16_t* om = reinterpret_cast<uint16_t*>(a.om) + bh * a.rank;
  for (int c = 2 * t; c < a.rank; c += 512) {  // rank is even
    float x = 0.f, y = 0.f;
#pragma unroll 8
    for (int s = 0; s < a.nsplit; ++s) {
      const float2 v = *reinterpret_cast<const float2*>(po + (int64_t)s * a.rank + c);
      const float e = ws[s];
      x += e > 0.f ? e * v.x : 0.f;  // an empty split's rows were never written
      y += e > 0.f ? e * v.y : 0.f;
    }
    *reinterpret_cast<uint32_t*>(om + c) = pack_bf16x2(x * inv, y * inv);
  }
}

}  // namespace mx

using namespace mx;

// rows: the new tokens' latent rows (x nullptr: another layer's).  -1 (nothing launched): sizes it does not take
extern "C" int mx_latent_heads(const LatentDecode* pa, const LatentRows* rows, int query, hipStream_t stream) {
  const LatentDecode& a = *pa;
  if (a.B <= 0) return 0;
  if (a.H <= 0 || a.H > 65535 || a.D <= 0 || a.D % 16 || a.R < 0 || a.R % 2 || a.E <= 0 || a.E % 4 || a.rank <= 0 ||
      a.rank % 16 || a.wq < a.rank + a.R || a.wq % 4 || a.ldq % 8 || a.ldq < (int64_t)a.H * (a.D + a.R) || (a.D + a.R) % 8 ||
      (((uintptr_t)a.q | (uintptr_t)a.wuk_t | (uintptr_t)a.wuv | (uintptr_t)a.om | (uintptr_t)a.qa | (uintptr_t)a.out) & 15))
    return -1;
  const int N = query ? a.rank : a.E;
  const int mb = a.B <= 16 ? 1 : 2;
  const dim3 g((N + 63) / 64 + (query ? 1 : 0), a.H, (a.B + 16 * mb - 1) / (16 * mb));
  const LatentRows none = {};
  LatentRows rw = rows ? *rows : none;
  rw.vec = latent_row_vec(rw);
  if (query) {
    if (mb == 1) latent_heads_kernel<1, true><<<g, 256, 0, stream>>>(a, rw);
    else latent_heads_kernel<2, true><<<g, 256, 0, stream>>>(a, rw);
  } else {
    if (a.nsplit > kLmSplits || ((uintptr_t)a.po & 7)) return -1;
    latent_merge_kernel<<<dim3(a.H, a.B), 256, 0, stream>>>(a);
    if (mb == 1) latent_heads_kernel<1, false><<<g, 256, 0, stream>>>(a, none);
    else latent_heads_kernel<2, false><<<g, 256, 0, stream>>>(a, none);
  }
  return (int)hipGetLastError();
}

// -1 (nothing launched): sizes it does not take
extern "C" int mx_latent_flash(const LatentAttn* pa, hipStream_t stream) {
  const LatentAttn& a = *pa;
  if (a.T <= 0 || a.nblocks <= 0) return 0;
  const int DQ = a.D + a.R;
  if (a.H <= 0 || a.D <= 0 || a.D % 8 || a.R < 0 || a.R % 8 || a.E <= 0 || a.E % 8 || a.rank % 8 || DQ > 256 || a.E > 128 ||
      a.window < 0 || !(a.scale > 0.f) || a.ldq % 8 || a.ldkv % 8 || a.ldl % 8 || a.ldq < (int64_t)a.H * DQ ||
      a.ldkv < (int64_t)a.H * (a.D + a.E) || a.ldl < a.rank + a.R || (int64_t)a.nblocks * a.H > INT32_MAX ||
      (((uintptr_t)a.q | (uintptr_t)a.kv | (uintptr_t)a.lat | (uintptr_t)a.cosb | (uintptr_t)a.sinb | (uintptr_t)a.out) & 15))
    return -1;
  const unsigned g = (unsigned)(a.nblocks * a.H);
#define LF(DK, DV) latent_flash_kernel<DK, DV><<<g, 256, 0, stream>>>(a)
#define LFV(DK) do { if (a.E <= 32) LF(DK, 32); else if (a.E <= 64) LF(DK, 64); else LF(DK, 128); } while (0)
  if (DQ <= 32) LFV(32);
  else if (DQ <= 64) LFV(64);
  else if (DQ <= 96) LFV(96);
  else if (DQ <= 128) LFV(128);
  else if (DQ <= 192) LFV(192);
  else LFV(256);
#undef LFV
#undef LF
  return (int)hipGetLastError();
}

// heads: 16 or 32 a workgroup.  -1 (nothing launched): sizes it does not take
extern "C" int mx_latent_split(const LatentDecode* pa, int heads, hipStream_t stream) {
  const LatentDecode& a = *pa;
  if (a.B <= 0) return 0;
  if (a.H <= 0 || a.H > 65535 || a.B > 65535 || a.rank <= 0 || a.rank % 4 || a.wc <= 0 || a.wc % 32 || a.wc > 1024 ||
      a.wc < a.rank + a.R || a.wq != a.wc || a.seq <= 0 || a.ring <= 0 || a.nsplit <= 0 || a.span <= 0 || a.span > 512 ||
      a.window < 0 || (a.bt && (a.maxb <= 0 || a.seq < 256)) || (!a.bt && a.ring > a.seq) || (heads != 16 && heads != 32) || !(a.scale > 0.f) ||
      (((uintptr_t)a.qa | (uintptr_t)a.pool | (uintptr_t)a.po) & 15))
    return -1;
  const int img = (kLsKeys * a.wc * 2 + 1023) / 1024 * 1024;
  const size_t lds = 2 * (size_t)img + (size_t)heads * kLsRow;
#define LS(KS, MB)                                                                                                  \
  do {                                                                                                              \
    static bool set = hipFuncSetAttribute((const void*)latent_split_kernel<KS, MB>,                                 \
                                          hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess;    \
    if (!set) return -1;                                                                                            \
    latent_split_kernel<KS, MB><<<dim3(a.nsplit, (a.H + 16 * MB - 1) / (16 * MB), a.B), 256, lds, stream>>>(a);     \
  } while (0)
#define LSM(KS) do { if (heads == 32) LS(KS, 2); else LS(KS, 1); } while (0)
  const int ks = a.wc / 32;
  if (ks <= 4) LSM(4);
  else if (ks <= 9) LSM(9);
  else if (ks <= 12) LSM(12);
  else if (ks <= 18) LSM(18);
  else if (ks <= 24) LSM(24);
  else LS(32, 1);
#undef LSM
#undef LS
  return (int)hipGetLastError();
}
