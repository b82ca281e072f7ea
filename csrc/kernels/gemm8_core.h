// Core of the 8-phase bf16 GEMM for gfx950 (entry points: gemm8.hip; experts' products: moe_mfma.hip):
//
//   C[M, N] = alpha * op(A) op(B) (+ C when BETA),  fp32 accumulation, C fp32 or bf16,
//
// with each operand in either storage order, so the three GEMM forms of a Llama training step
// run without a transpose pass:
//   forward  y  = x W^T  : A = x  [T][in]  (k-contiguous), B = W [out][in] (k-contiguous)
//   input gr dX = dY W   : A = dY [T][out] (k-contiguous), B = W [out][in] = [k][n] (n-contiguous)
//   weight gr dW = dY^T X: A = dY [T][out] = [k][m] (m-contiguous), B = X [T][in] = [k][n]
// ("NN"-form dX ran at ~1.32 PF in hipBLASLt; token-major dW needed 6.8 / 73 ms of transposes
// per 8B / 70B-ZeRO-3 step, archive/profiles/r3o, r3p, r3d).
//
// Structure (CDNA guide §5 "The 256² 8-phase template", T1-T5, T10), designed here for the two
// operand orders:
//  * workgroup 512 threads = 8 waves as 2 (M) x 4 (N), output tile 256 x 256, each wave 128 x 64 =
//    8 x 4 blocks of v_mfma_f32_16x16x32_bf16 (16x16x32 rather than 32x32x16: the chip holds a
//    ~12-15 % higher clock on it on random data, MI355X_MICROARCH "DVFS give-back" item 7);
//  * the MFMA is issued with the operands swapped (B fragment as the A operand), so each lane's
//    4 accumulator registers are 4 CONSECUTIVE output columns of one row: 8-B (bf16) / 16-B (fp32)
//    epilogue stores instead of 2-B / 4-B ones;
//  * a K-tile (BK 64) is four 16-KiB half-tile images, A0 | A1 | B0 | B1, where A0 holds the rows
//    of output quadrant a = 0 of BOTH wave rows (and B0 the columns of quadrant b = 0 of all four
//    wave columns), so each image is read in exactly one phase;
//  * every image is filled by LDS-DMA (buffer_load ... lds, 16 B per lane, 2 per wave) into a
//    lane-linear layout; the XOR swizzle that makes the MFMA-operand reads bank-conflict free is
//    applied by permuting each lane's SOURCE address (guide rule 21):
//      - k-contiguous operand: [128 rows][64 k] (128-B rows), 16-B chunk c stored at c ^ ((r>>1)&7),
//        read with ds_read_b128 (lane: row l&15, k chunk l>>4);
//      - mn-contiguous operand: [64 k][128 cols] (256-B rows), chunk c stored at c ^ 2 t(k),
//        t(k) = (k&3) | ((k>>3)&1)<<2, read with two ds_read_b64_tr_b16 per 32-k step (T10);
//  * 8 phases per two K-tiles; phase p: {this phase's LDS reads, one half-tile prefetch,
//    s_barrier, lgkmcnt(0), 16 MFMAs (one 64x32 quadrant x K 64), s_barrier}; the two wave rows run
//    one barrier apart (ping-pong: one issues MFMAs while the other reads LDS); counted
//    vmcnt(6) (three half-tiles in flight across barriers) only in phases 4 and 8, raw s_barrier
//    (never __syncthreads: its fence would drain the DMA), all LDS in one __shared__ array, LDS
//    reads as inline asm (hipcc's waitcnt pass cannot see that they miss the in-flight DMA);
//  * read/restage order (why the schedule is race free): phase 1 reads B0 then A0 of the even
//    buffer and retires the B0 reads (counted lgkmcnt) before its first barrier, phase 2 B1,
//    phase 3 A1, phase 4 nothing; the next tile's images are restaged B0 @2, A0 @3, B1 @4, A1 @5,
//    i.e. >= 2 phases after an image's last read (1 for the early-retired B0), and read >= one
//    phase after the vmcnt that retires them (guide §5 "Read a staged buffer one phase AFTER the
//    wait", with the extra barrier of the staggered wave rows);
//  * workgroup -> tile: XCD-contiguous ranges (T1, bijective) of a grouped order (8 m-tiles x all
//    n-tiles) so one XCD's co-resident tiles share their A / B panels in its L2.
// Range-checked buffer descriptors read rows past K (mn-contiguous operands) as zeros, so the
// weight-gradient form takes any token count; M and N must be multiples of 256.
#pragma once

#include "hybrid.h"

namespace mx {

typedef __bf16 bf16x8_g __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void* g8lptr_t;

__device__ __forceinline__ f32x4 g8_mfma(const u16x8& a, const u16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_g, a), __builtin_bit_cast(bf16x8_g, b), c,
                                                 0, 0, 0);
}

constexpr int G8_HT = 16384;        // one half-tile image: 128 rows (cols) x 64 k x bf16
constexpr int G8_TILE = 4 * G8_HT;  // A0 | A1 | B0 | B1
constexpr int G8_BK = 64;

// image row r' (k-contiguous) / image column (mn-contiguous) -> row / column of the 256 tile
__device__ __forceinline__ int g8_map_b(int r, int h) { return (r >> 5) * 64 + h * 32 + (r & 31); }
__device__ __forceinline__ int g8_map_a(int r, int h) { return (r >> 6) * 128 + h * 64 + (r & 63); }

// ---- fused epilogues (forward projections, B = the weight [N][K], bf16 output) -----------------
// In the epilogue, lane l of wave (wr, wc) holds, per accumulator block j = 2 jh + jl, the 4
// consecutive VIRTUAL tile columns v = 64 wc + 32 jh + 16 jl + 4 (l >> 4) + [0, 4).  A fused epilogue
// picks which WEIGHT ROW feeds each virtual column (the B images are DMA-loaded from those rows), so
// the two operands of its elementwise op land in the SAME lane and register -- no LDS exchange:
//  G8_EPI_ROPE  (qkv projection, head dim 128: a tile = 2 heads): virtual (wc, jh, jl, q) -> head
//               column d = 32 (wc & 1) + 64 jh + 16 jl + q, so blocks jh = 0 / 1 hold the rotate-half
//               pair (d, d + 64); outputs written HEAD-MAJOR q [B,Hq,S,D], k / v [B,Hkv,S,D] (the
//               layout the attention kernels read; csrc/kernels/rope.hip rope_split, fused away)
//  G8_EPI_SWIGLU (gate-up projection, W = [gate; up], F rows each): tile pn covers gate columns
//               [128 pn, 128 pn + 128) and the same up columns: jh = 0 -> gate row 128 pn + 32 wc +
//               16 jl + q, jh = 1 -> the up row F further; outputs gu [T, 2F] (standard layout, saved
//               for the backward) AND m = silu(g) u [T, F] (elementwise.hip swiglu_fwd, fused away)
//  G8_EPI_SWIGLU_BWD (NN form: the down projection's dX GEMM dm = dy W_down, F = N columns): the
//               lane's 8 dm columns (after the bf16 swap) meet the saved gu [T, 2F] at the same
//               columns -> writes dgu [T, 2F] (and, with ep.m set, the recomputed m = silu(g) u) in
//               place of dm (elementwise.hip swiglu_bwd / swiglu_bwd_m, fused away)
// All round the GEMM result to bf16 first and then apply the exact expression of the kernel they
// replace: bitwise equal to GEMM -> rope_split / swiglu_fwd / swiglu_bwd on the same kernel's output.
//  G8_EPI_MOE / G8_EPI_MOE_GLU (expert mixtures, A = token rows, B = [experts][rows][K]): an output tile is up
//               to 256 rows of one expert out of a table; A's rows are gathered through it, rows, columns and
//               K past the end read as zeros and are not stored (K, F and the strides are multiples of 8).
//               GLU: columns as SWIGLU (gate and up of one channel in one lane), output [rows, F]
//  G8_EPI_ROWS / G8_EPI_ROWS_SWIGLU: any number of rows (A k-contiguous; the last tile's rows past M read as zeros
//               through the descriptor's range and are not stored).  SWIGLU: only m = silu(g) u is stored, the
//               projection itself never leaves the registers
//  G8_EPI_PART  one of k0 parts of K, as fp32 into image `part` (cpart elements on) of C; any number of rows
constexpr int G8_EPI_NONE = 0, G8_EPI_ROPE = 1, G8_EPI_SWIGLU = 2, G8_EPI_SWIGLU_BWD = 3, G8_EPI_MOE = 4,
              G8_EPI_MOE_GLU = 5, G8_EPI_ROWS = 6, G8_EPI_ROWS_SWIGLU = 7, G8_EPI_PART = 8;
constexpr bool g8_moe(int epi) { return epi == G8_EPI_MOE || epi == G8_EPI_MOE_GLU; }
constexpr bool g8_rows(int epi) { return epi >= G8_EPI_ROWS && epi <= G8_EPI_PART; }
constexpr bool g8_pairs(int epi) { return epi == G8_EPI_SWIGLU || epi == G8_EPI_ROWS_SWIGLU; }
constexpr uint32_t G8_OOB = 0x80000000u;  // past every descriptor's range: reads as zeros

struct G8Epi {
  uint16_t* q;        // ROPE: [B, Hq, S, 128]
  uint16_t* k;        //       [B, Hkv, S, 128]
  uint16_t* v;        //       [B, Hkv, S, 128]
  const float* cosb;  //       [>= S, 64] f32 (host table, mxllm/ops/reference.py rope_tables)
  const float* sinb;
  int S, Hq, Hkv;
  uint16_t* m;        // SWIGLU: [T, F] with row stride ldm (SWIGLU_BWD: optional recomputed m)
  int64_t ldm;
  int F;
  const uint16_t* gu; // SWIGLU_BWD: the forward's [T, 2F] with row stride ldg
  int64_t ldg;
  float* sq;          // plain bf16 beta-0 output: per-tile sum of squares of the stored values
};

// MOE / MOE_GLU
struct G8Moe {
  const int4* tiles;   // (expert, first sorted row, rows, number of tiles) of each 256-row tile, the unused ones last
  const int32_t* src;  // row of A of each sorted row (nullptr: the row itself)
  uint32_t arec;       // bytes of A
  int F;               // output columns
  float limit;         // MOE_GLU
};

// weight row feeding virtual tile column v (0..255) of output tile pn (G8_EPI_SWIGLU: absolute row)
template <int EPI>
__device__ __forceinline__ int g8_epi_row(int v, int pn, int F) {
  if constexpr (EPI == G8_EPI_ROPE) {
    return (v & ~127) + ((v >> 6) & 1) * 32 + ((v >> 5) & 1) * 64 + (v & 31);
  } else if constexpr (g8_pairs(EPI) || EPI == G8_EPI_MOE_GLU) {
    return (((v >> 5) & 1) ? F : 0) + 128 * pn + (v >> 6) * 32 + (v & 31);
  } else {
    return v;
  }
}
__device__ __forceinline__ int g8_t(int k) { return (k & 3) | (((k >> 3) & 1) << 2); }

// per-lane byte offsets of this wave's two LDS-DMA pieces of half-tile image h of one operand
template <bool KC, bool IS_A, int EPI = G8_EPI_NONE>
__device__ __forceinline__ void g8_src_offsets(int w, int lane, int64_t ld, int h, uint32_t (&off)[2], int pn = 0,
                                               int F = 0) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int pc = 2 * w + j;
    if constexpr (KC) {
      const int r = 8 * pc + (lane >> 3);
      const int c = (lane & 7) ^ ((r >> 1) & 7);
      const int row = IS_A ? g8_map_a(r, h) : g8_epi_row<EPI>(g8_map_b(r, h), pn, F);
      off[j] = (uint32_t)(((int64_t)row * ld + 8 * c) * 2);
    } else {
      const int k = 4 * pc + (lane >> 4);
      const int c = (lane & 15) ^ (2 * g8_t(k));
      const int col = IS_A ? g8_map_a(8 * c, h) : g8_map_b(8 * c, h);
      off[j] = (uint32_t)(((int64_t)k * ld + col) * 2);
    }
  }
}

// lane part of the LDS address of an MFMA-operand read
//  KC: block rows rb.. (rb % 16 == 0, folded into the immediate), k-step s
__device__ __forceinline__ uint32_t g8_kc_lane(int lane, int s) {
  const int i = lane & 15, g = lane >> 4;
  return (uint32_t)(i * 128 + 16 * ((4 * s + g) ^ ((i >> 1) & 7)));
}
//  MN: block columns cb..cb+15 (one base per cb; k-step s and read r are +8192 s + 1024 r)
__device__ __forceinline__ uint32_t g8_mn_lane(int lane, int cb) {
  const int g = lane >> 4, q = (lane & 15) >> 2, p = lane & 3;
  const int t = q | ((g & 1) << 2);
  return (uint32_t)((8 * g + q) * 256 + 16 * (((cb >> 3) ^ (2 * t)) + (p >> 1)) + 8 * (p & 1));
}

// In-kernel cycle stamps (diagnostic build V & 4; guide §7 "In-kernel stamps"): lane 0 of wave 0
// (wave row 0) and of wave 4 (wave row 1) record s_memtime at kernel start, after the prologue,
// at the top of every K-loop iteration (2 K-tiles) and after the loop / the epilogue, plus
// s_memrealtime at start and end (clock = d memtime / d realtime x 100 MHz).  Written with
// ordinary VECTOR global stores into a buffer nothing else reads; the normal build has none.
// The stamp buffer (1.3 MB of device memory) and the stamped / ablation variants exist only in a
// diagnostic build: MXLLM_FILE_FLAGS="gemm8.hip=-DMXLLM_GEMM8_DIAG" python -m mxllm._build.
constexpr int G8_NST = 80;
#ifdef MXLLM_GEMM8_DIAG
__device__ unsigned long long g8_stamps[1024 * 2 * G8_NST];
__device__ __forceinline__ void g8_stamp(int wg, int row, int k, unsigned long long v) {
  if (wg < 1024 && k < G8_NST) g8_stamps[((size_t)wg * 2 + row) * G8_NST + k] = v;
}
#else
__device__ __forceinline__ void g8_stamp(int, int, int, unsigned long long) {}
#endif

// sum of squares of the 8 bf16 values packed in `o` (what the plain epilogue stored), added to s
__device__ __forceinline__ float g8_sq8(const uint4& o, float s) {
  const uint32_t v[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float lo = __uint_as_float(v[i] << 16), hi = __uint_as_float(v[i] & 0xffff0000u);
    s = __builtin_fmaf(lo, lo, s);
    s = __builtin_fmaf(hi, hi, s);
  }
  return s;
}
__device__ __forceinline__ float g8_sigmoid(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
__device__ __forceinline__ float g8_rbf(float x) { return bf2f(f2bf(x)); }  // round through bf16

// 16-B pack / store of blocks (jl = 0, 1) of one jh: lanes l, l + 16 swap packed pairs (permlane16_swap) so
// every lane owns 8 consecutive columns (see the plain bf16 epilogue); `dst` = this lane's 8 columns
__device__ __forceinline__ uint4 g8_pack8(const f32x4& va, const f32x4& vb) {
  const auto s0 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(va[0], va[1]), pack_bf16x2(vb[0], vb[1]), false, false);
  const auto s1 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(va[2], va[3]), pack_bf16x2(vb[2], vb[3]), false, false);
  uint4 o;
  o.x = s0[0];
  o.y = s1[0];
  o.z = s0[1];
  o.w = s1[1];
  return o;
}
__device__ __forceinline__ void g8_store8(uint16_t* dst, const f32x4& va, const f32x4& vb) {
  *reinterpret_cast<uint4*>(dst) = g8_pack8(va, vb);
}

template <int EPI>
__device__ __forceinline__ void g8_epilogue_fused(f32x4 (&acc)[8][4], float alpha, int ml, int pn, int wc, int lane,
                                                  int M, int N, const G8Epi& ep, void* C, int64_t ldc, const G8Moe& mo, const int4& tl) {
  // this lane's 8 stored columns start at offset u8 inside a 32-column group (after the swap)
  const int u8 = 16 * ((lane >> 4) & 1) + 8 * (lane >> 5);
  if constexpr (g8_moe(EPI)) {
    uint16_t* out = reinterpret_cast<uint16_t*>(C);
#pragma unroll
    for (int qa = 0; qa < 2; ++qa)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int rl = ml + qa * 64 + 16 * i;
        f32x4(&x)[4] = acc[4 * qa + i];
        if constexpr (EPI == G8_EPI_MOE_GLU) {
#pragma unroll
          for (int jl = 0; jl < 2; ++jl)
#pragma unroll
            for (int c = 0; c < 4; ++c) x[jl][c] = clipped_glu<uint16_t>(x[jl][c], x[2 + jl][c], mo.limit);
        }
#pragma unroll
        for (int jp = 0; jp < (EPI == G8_EPI_MOE_GLU ? 1 : 2); ++jp) {
          const uint4 o = g8_pack8(x[2 * jp], x[2 * jp + 1]);
          const int col = (EPI == G8_EPI_MOE_GLU ? 128 * pn + 32 * wc : 256 * pn + 64 * wc + 32 * jp) + u8;
          if (rl < tl.z && col < mo.F) *reinterpret_cast<uint4*>(out + (int64_t)(tl.y + rl) * ldc + col) = o;
        }
      }
  } else if constexpr (EPI == G8_EPI_ROPE) {
    const int head = pn * 2 + (wc >> 1);  // 128-column heads: two per tile
    uint16_t* dst;
    int Hd, hh;
    if (head < ep.Hq) {
      dst = ep.q, Hd = ep.Hq, hh = head;
    } else if (head < ep.Hq + ep.Hkv) {
      dst = ep.k, Hd = ep.Hkv, hh = head - ep.Hq;
    } else {
      dst = ep.v, Hd = ep.Hkv, hh = head - ep.Hq - ep.Hkv;
    }
    const bool rot = head < ep.Hq + ep.Hkv;
    const int d0 = 32 * (wc & 1);  // head column of block (jh 0, jl 0, lane group 0)
#pragma unroll
    for (int qa = 0; qa < 2; ++qa)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = ml + qa * 64 + 16 * i;
        const int b = m / ep.S, sq = m - b * ep.S;
        f32x4 x0[2], x1[2];  // [jl]: head columns d (jh 0) and d + 64 (jh 1)
#pragma unroll
        for (int jl = 0; jl < 2; ++jl) {
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            x0[jl][c] = g8_rbf(acc[4 * qa + i][jl][c] * alpha);
            x1[jl][c] = g8_rbf(acc[4 * qa + i][2 + jl][c] * alpha);
          }
        }
        if (rot) {
#pragma unroll
          for (int jl = 0; jl < 2; ++jl) {
            const int f = d0 + 16 * jl + 4 * (lane >> 4);  // frequency index of x0[jl][0]
            const f32x4 cs = *reinterpret_cast<const f32x4*>(ep.cosb + (int64_t)sq * 64 + f);
            const f32x4 sn = *reinterpret_cast<const f32x4*>(ep.sinb + (int64_t)sq * 64 + f);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              const float a = x0[jl][c], bb = x1[jl][c];
              x0[jl][c] = rope_lo(a, bb, cs[c], sn[c]);
              x1[jl][c] = rope_hi(a, bb, cs[c], sn[c]);
            }
          }
        }
        uint16_t* row = dst + (((int64_t)b * Hd + hh) * ep.S + sq) * 128;
        g8_store8(row + d0 + u8, x0[0], x0[1]);
        g8_store8(row + d0 + 64 + u8, x1[0], x1[1]);
      }
  } else if constexpr (EPI == G8_EPI_SWIGLU_BWD) {
    const int F = N;
    const int cb = 256 * pn + 64 * wc + 16 * ((lane >> 4) & 1) + 8 * (lane >> 5);  // + 32 jp
#pragma unroll
    for (int qa = 0; qa < 2; ++qa) {
      // all 16 gu loads of this half first (64 VGPRs): one memory round trip per half, not per row
      u16x8 g8[4][2], u8v[4][2];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint16_t* gr = ep.gu + (int64_t)(ml + qa * 64 + 16 * i) * ep.ldg;
#pragma unroll
        for (int jp = 0; jp < 2; ++jp) {
          g8[i][jp] = *reinterpret_cast<const u16x8*>(gr + cb + 32 * jp);
          u8v[i][jp] = *reinterpret_cast<const u16x8*>(gr + F + cb + 32 * jp);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t m = ml + qa * 64 + 16 * i;
        u16x8 d8[2];
#pragma unroll
        for (int jp = 0; jp < 2; ++jp) {  // dm rounded to bf16 and swapped exactly as the plain store
          const f32x4 va = acc[4 * qa + i][2 * jp] * alpha, vb = acc[4 * qa + i][2 * jp + 1] * alpha;
          const auto s0 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(va[0], va[1]), pack_bf16x2(vb[0], vb[1]),
                                                          false, false);
          const auto s1 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(va[2], va[3]), pack_bf16x2(vb[2], vb[3]),
                                                          false, false);
          uint4 o;
          o.x = s0[0];
          o.y = s1[0];
          o.z = s0[1];
          o.w = s1[1];
          d8[jp] = __builtin_bit_cast(u16x8, o);
        }
        uint16_t* dr = reinterpret_cast<uint16_t*>(C) + m * ldc;
#pragma unroll
        for (int jp = 0; jp < 2; ++jp) {
          u16x8 og, ou;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            float dg, du;
            swiglu_grad(bf2f(d8[jp][j]), bf2f(g8[i][jp][j]), bf2f(u8v[i][jp][j]), dg, du);
            og[j] = f2bf(dg);
            ou[j] = f2bf(du);
          }
          *reinterpret_cast<u16x8*>(dr + cb + 32 * jp) = og;
          *reinterpret_cast<u16x8*>(dr + F + cb + 32 * jp) = ou;
          if (ep.m) {
            u16x8 om;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const float gf = bf2f(g8[i][jp][j]);
              om[j] = f2bf(gf * __builtin_amdgcn_rcpf(1.f + __expf(-gf)) * bf2f(u8v[i][jp][j]));
            }
            *reinterpret_cast<u16x8*>(ep.m + m * ep.ldm + cb + 32 * jp) = om;
          }
        }
      }
    }
  } else if constexpr (EPI == G8_EPI_ROWS) {
#pragma unroll
    for (int qa = 0; qa < 2; ++qa)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = ml + qa * 64 + 16 * i;
#pragma unroll
        for (int jp = 0; jp < 2; ++jp) {
          const f32x4 va = acc[4 * qa + i][2 * jp] * alpha, vb = acc[4 * qa + i][2 * jp + 1] * alpha;
          const uint4 o = g8_pack8(va, vb);  // lanes exchange: outside the row test
          if (m < M)
            *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(C) + m * ldc + 256 * pn + 64 * wc + 32 * jp + u8) = o;
        }
      }
  } else if constexpr (EPI == G8_EPI_PART) {
    const int n = 256 * pn + 64 * wc + 4 * (lane >> 4);
#pragma unroll
    for (int qa = 0; qa < 2; ++qa)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = ml + qa * 64 + 16 * i;
        float* row = reinterpret_cast<float*>(C) + m * ldc + n;
        if (m < M) {
#pragma unroll
          for (int j = 0; j < 4; ++j) *reinterpret_cast<f32x4*>(row + 32 * (j >> 1) + 16 * (j & 1)) = acc[4 * qa + i][j];
        }
      }
  } else if constexpr (EPI == G8_EPI_ROWS_SWIGLU) {
    const int col = 128 * pn + 32 * wc + u8;
#pragma unroll
    for (int qa = 0; qa < 2; ++qa)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = ml + qa * 64 + 16 * i;
        f32x4 mm[2];
#pragma unroll
        for (int jl = 0; jl < 2; ++jl)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const float g = g8_rbf(acc[4 * qa + i][jl][c] * alpha), u = g8_rbf(acc[4 * qa + i][2 + jl][c] * alpha);
            mm[jl][c] = g * g8_sigmoid(g) * u;
          }
        const uint4 o = g8_pack8(mm[0], mm[1]);
        if (m < M) *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(C) + m * ldc + col) = o;
      }
  } else {  // G8_EPI_SWIGLU
    const int F = N / 2;
    const int col = 128 * pn + 32 * wc + u8;  // gate column (up: + F; m: the same column)
#pragma unroll
    for (int qa = 0; qa < 2; ++qa)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t m = ml + qa * 64 + 16 * i;
        f32x4 g[2], u[2], mm[2];
#pragma unroll
        for (int jl = 0; jl < 2; ++jl)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            g[jl][c] = g8_rbf(acc[4 * qa + i][jl][c] * alpha);
            u[jl][c] = g8_rbf(acc[4 * qa + i][2 + jl][c] * alpha);
            mm[jl][c] = g[jl][c] * g8_sigmoid(g[jl][c]) * u[jl][c];
          }
        uint16_t* gu = reinterpret_cast<uint16_t*>(C) + m * ldc;
        g8_store8(gu + col, g[0], g[1]);
        g8_store8(gu + F + col, u[0], u[1]);
        g8_store8(ep.m + m * ep.ldm + col, mm[0], mm[1]);
      }
  }
}

// V != 0: timing-only ablation builds (bench/gemm8_probe.py --ablate; results are WRONG):
//   V & 1: every phase issues its 16 MFMAs twice (MFMA time per barrier doubled)
//   V & 2: no barriers in the K loop and no wave-row stagger (no LDS ordering at all)
//   V & 4: stamps only (results correct)
// PH = 4: the same images and registers on a 4-phase schedule (two quadrants = 32 MFMAs per phase,
// half the barriers; every phase retires its LDS reads before its first barrier so each image is
// restaged one phase after its last read; two half-tiles in flight across barriers, vmcnt(4))
template <bool A_KC, bool B_KC, bool OUT_F32, bool BETA, int V = 0, int PH = 8, int EPI = G8_EPI_NONE>
__global__ void __launch_bounds__(512, 1)
gemm8_kernel(const uint16_t* __restrict__ A, int64_t lda, const uint16_t* __restrict__ B, int64_t ldb,
             void* __restrict__ C, int64_t ldc, int M, int N, int K, const float* __restrict__ alpha_t,
             float alpha_f, int k0 = 0, int64_t cpart = 0, G8Epi ep = G8Epi{}, G8Moe mo = G8Moe{}) {
  static_assert(EPI == G8_EPI_NONE || EPI == G8_EPI_PART || (!OUT_F32 && !BETA && (EPI == G8_EPI_ROWS ? A_KC : EPI == G8_EPI_SWIGLU_BWD ? A_KC && !B_KC : A_KC && B_KC)),
                "fused epilogues: bf16, beta 0; TN-form forwards, NN-form SwiGLU backward");
  // K split in two (gridDim.y == 2, k0 = K of part 0): part 1 covers K rows / columns k0 .. K-1 of
  // both operands and writes its own output image C + cpart (mx_gemm8_tail: the last, partial wave
  // of tiles of a GEMM runs as twice as many half-K workgroups; the images are summed after)
  if (EPI != G8_EPI_PART && gridDim.y > 1) {
    const int kp = blockIdx.y;
    const int64_t koff = kp ? k0 : 0;
    A += A_KC ? koff : koff * lda;
    B += B_KC ? koff : koff * ldb;
    if (kp) C = reinterpret_cast<char*>(C) + cpart * (OUT_F32 ? 4 : 2);
    K = kp ? K - k0 : k0;
  }
  // ONE __shared__ array (a second LDS object makes hipcc drain vmcnt before LDS reads: guide §5 item 4a)
  __shared__ __attribute__((aligned(1024))) char smem[2 * G8_TILE];
  const int nN = N >> 8;
  int nM = (g8_rows(EPI) ? M + 255 : M) >> 8, pm, pn;
  {
    // MOE: the grid is as large as any choice of experts may need.  The tiles there are, over all XCDs: by the
    // grid's size the last XCDs had none while the first ones' 36 tiles took their 32 CUs two turns (2048 tokens, 4
    // of 16 experts of 768, K 4096: 240 tiles of a grid of 288, 158 us; 93 by the tiles' number)
    int grid = gridDim.x;
    if constexpr (g8_moe(EPI)) {
      nM = mo.tiles[0].w;
      grid = nM * nN;
      if ((int)blockIdx.x >= grid) return;
    }
    int L = xcd_remap(blockIdx.x, grid);
    if constexpr (EPI == G8_EPI_PART) {  // parts after each other: an XCD's tiles share the panels of one part of K
      const int tiles = nM * nN, kp = L / tiles, nkt = (K + G8_BK - 1) / G8_BK;
      const int t0 = nkt * kp / k0, t1 = nkt * (kp + 1) / k0;
      L -= kp * tiles;
      A += A_KC ? (int64_t)t0 * G8_BK : (int64_t)t0 * G8_BK * lda;
      B += B_KC ? (int64_t)t0 * G8_BK : (int64_t)t0 * G8_BK * ldb;
      C = reinterpret_cast<float*>(C) + kp * cpart;
      K = (kp + 1 == k0 ? K : t1 * G8_BK) - t0 * G8_BK;
    }
    constexpr int GM = 8;
    const int per = GM * nN, grp = L / per, first = grp * GM;
    const int rows = min(GM, nM - first), in = L - grp * per;
    pm = first + in % rows;
    pn = in / rows;
  }
  int4 tl = {0, 0, 0, 0};
  if constexpr (g8_moe(EPI)) {
    tl = mo.tiles[pm];
    B += (int64_t)tl.x * (EPI == G8_EPI_MOE_GLU ? 2 : 1) * mo.F * ldb;
  }
  // (MOE: rows are taken from the table, m0 = 0)
  const int m0 = g8_moe(EPI) ? 0 : pm << 8, n0 = pn << 8;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = w >> 2, wc = w & 3;
  const int nk = (K + G8_BK - 1) / G8_BK;
  constexpr bool ST = (V & 4) != 0;
  const bool stw = ST && (tid == 0 || tid == 256);  // lane 0 of waves 0 and 4
  const int strow = tid >= 256;
  int sti = 0;
  if constexpr (ST) {
    if (stw) {
      g8_stamp(blockIdx.x, strow, sti++, __builtin_amdgcn_s_memtime());
      g8_stamp(blockIdx.x, strow, sti++, __builtin_amdgcn_s_memrealtime());
    }
  }

  // ---- operand descriptors (range-checked: mn-contiguous rows past K read as zeros)
  const uint16_t* abase = A_KC ? A + (int64_t)m0 * lda : A + m0;
  // SWIGLU: gate and up rows are F apart -> absolute weight rows off the start of B
  const uint16_t* bbase = B_KC ? B + (int64_t)(g8_pairs(EPI) || g8_moe(EPI) ? 0 : n0) * ldb : B + n0;
  const uint32_t arec = g8_moe(EPI) ? mo.arec : A_KC ? (uint32_t)(((g8_rows(EPI) ? min(255, M - 1 - m0) : 255) * lda + (int64_t)nk * G8_BK) * 2) : (uint32_t)(((int64_t)K * lda - m0) * 2);
  const uint32_t brec = g8_moe(EPI) ? (uint32_t)((int64_t)(EPI == G8_EPI_MOE_GLU ? 2 : 1) * mo.F * ldb * 2)
                        : g8_pairs(EPI) ? (uint32_t)(((int64_t)(N - 1) * ldb + (int64_t)nk * G8_BK) * 2)
                        : B_KC ? (uint32_t)((255 * ldb + (int64_t)nk * G8_BK) * 2)
                               : (uint32_t)(((int64_t)K * ldb - n0) * 2);
  const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc((void*)abase, 0, arec, 0x00020000);
  const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc((void*)bbase, 0, brec, 0x00020000);
  const uint32_t astep = A_KC ? G8_BK * 2 : (uint32_t)(G8_BK * lda * 2);  // bytes per K-tile
  const uint32_t bstep = B_KC ? G8_BK * 2 : (uint32_t)(G8_BK * ldb * 2);
  uint32_t aoff[2][2], boff[2][2];
  int kcol[2] = {0, 0};  // MOE: first k of this lane's chunk in either piece
  if constexpr (g8_moe(EPI)) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int r = 8 * (2 * w + j) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        kcol[j] = 8 * c;
        const int ar = g8_map_a(r, h), bv = g8_map_b(r, h);
        const int64_t arow = ar < tl.z ? (mo.src ? mo.src[tl.y + ar] : tl.y + ar) : -1;
        const int brow = g8_epi_row<EPI>(bv, pn, mo.F) + (EPI == G8_EPI_MOE_GLU ? 0 : 256 * pn);
        const bool bon = EPI == G8_EPI_MOE_GLU ? brow - (((bv >> 5) & 1) ? mo.F : 0) < mo.F : brow < mo.F;
        aoff[h][j] = arow >= 0 ? (uint32_t)((arow * lda + 8 * c) * 2) : G8_OOB;
        boff[h][j] = bon ? (uint32_t)(((int64_t)brow * ldb + 8 * c) * 2) : G8_OOB;
      }
  } else {
    g8_src_offsets<A_KC, true>(w, lane, lda, 0, aoff[0]);
    g8_src_offsets<A_KC, true>(w, lane, lda, 1, aoff[1]);
    g8_src_offsets<B_KC, false, EPI>(w, lane, ldb, 0, boff[0], pn, N / 2);
    g8_src_offsets<B_KC, false, EPI>(w, lane, ldb, 1, boff[1], pn, N / 2);
  }

  // issue half-tile image `img` (0 A0, 1 A1, 2 B0, 3 B1) of K-tile kt into buffer kt & 1
  auto issue = [&](int kt, int img) __attribute__((always_inline)) {
    char* dst = smem + (kt & 1) * G8_TILE + img * G8_HT + (2 * w) * 1024;
    // the K-tile offset rides in voffset: the range check covers voffset + immediate only
    if constexpr (g8_moe(EPI)) {
      const uint32_t so = (uint32_t)kt * (G8_BK * 2);
      const uint32_t o0 = kt * G8_BK + kcol[0] < K ? (img < 2 ? aoff[img & 1][0] : boff[img & 1][0]) + so : G8_OOB;
      const uint32_t o1 = kt * G8_BK + kcol[1] < K ? (img < 2 ? aoff[img & 1][1] : boff[img & 1][1]) + so : G8_OOB;
      if (img < 2) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ars, (g8lptr_t)dst, 16, o0, 0, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ars, (g8lptr_t)(dst + 1024), 16, o1, 0, 0, 0);
      } else {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(brs, (g8lptr_t)dst, 16, o0, 0, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(brs, (g8lptr_t)(dst + 1024), 16, o1, 0, 0, 0);
      }
    } else if (img < 2) {
      const uint32_t so = (uint32_t)kt * astep;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ars, (g8lptr_t)dst, 16, aoff[img][0] + so, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ars, (g8lptr_t)(dst + 1024), 16, aoff[img][1] + so, 0, 0, 0);
    } else {
      const uint32_t so = (uint32_t)kt * bstep;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(brs, (g8lptr_t)dst, 16, boff[img - 2][0] + so, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(brs, (g8lptr_t)(dst + 1024), 16, boff[img - 2][1] + so, 0, 0, 0);
    }
  };

  // ---- LDS read bases (lane parts; + buffer / image offsets at the read)
  const uint32_t lds0 = lds_addr(smem);
  uint32_t akc[2], amn[4], bmn[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) akc[s] = g8_kc_lane(lane, s);
#pragma unroll
  for (int i = 0; i < 4; ++i) amn[i] = g8_mn_lane(lane, wr * 64 + 16 * i);
#pragma unroll
  for (int j = 0; j < 2; ++j) bmn[j] = g8_mn_lane(lane, wc * 32 + 16 * j);

  u16x8 fa[4][2], fb0[2][2], fb1[2][2];  // [block][k-step]
  f32x4 acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // A image `img` (0/1) of buffer `buf` -> fa;  KC: ds_read_b128, MN: 2 x ds_read_b64_tr_b16 per block and k-step
  auto read_a = [&](int buf, int img) __attribute__((always_inline)) {
    const uint32_t ib = lds0 + buf * G8_TILE + img * G8_HT;
    if constexpr (A_KC) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const uint32_t b = ib + akc[s];
#pragma unroll
        for (int i = 0; i < 4; ++i) fa[i][s] = rd128_off(b, (wr * 64 + 16 * i) * 128);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t b = ib + amn[i];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const u16x4 lo = trd_off(b, 8192 * s), hi = trd_off(b, 8192 * s + 1024);
          fa[i][s] = u16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
      }
    }
  };
  auto read_b = [&](int buf, int img, u16x8(&fb)[2][2]) __attribute__((always_inline)) {
    const uint32_t ib = lds0 + buf * G8_TILE + (2 + img) * G8_HT;
    if constexpr (B_KC) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const uint32_t b = ib + akc[s];
#pragma unroll
        for (int j = 0; j < 2; ++j) fb[j][s] = rd128_off(b, (wc * 32 + 16 * j) * 128);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint32_t b = ib + bmn[j];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const u16x4 lo = trd_off(b, 8192 * s), hi = trd_off(b, 8192 * s + 1024);
          fb[j][s] = u16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
      }
    }
  };
  auto pin_a = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      pin(fa[i][0]);
      pin(fa[i][1]);
    }
  };
  auto pin_b = [&](u16x8(&fb)[2][2]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      pin(fb[j][0]);
      pin(fb[j][1]);
    }
  };
  // quadrant (a, b): 16 MFMAs; swapped operands -> acc holds C^T blocks (4 consecutive columns per lane)
  auto mma = [&](int qa, int qb, u16x8(&fb)[2][2]) __attribute__((always_inline)) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[4 * qa + i][2 * qb + j] = g8_mfma(fb[j][s], fa[i][s], acc[4 * qa + i][2 * qb + j]);
    __builtin_amdgcn_s_setprio(0);
  };
  constexpr int NA = A_KC ? 8 : 16;  // LDS reads of one A image
  auto vm6 = []() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(6)" ::: "memory"); };
  auto vm0 = []() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };

  auto vm4 = []() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); };
  // ---- prologue: K-tile 0 (all four images) + K-tile 1's B0, A0, B1 (PH 4: B0, B1); retire tile 0
  issue(0, 2);
  issue(0, 0);
  issue(0, 3);
  issue(0, 1);
  if (nk > 1) {
    issue(1, 2);
    if constexpr (PH == 8) issue(1, 0);
    issue(1, 3);
    if constexpr (PH == 8) vm6(); else vm4();
  } else {
    vm0();
  }
  __builtin_amdgcn_s_barrier();
  if (!(V & 2) && wr == 1) __builtin_amdgcn_s_barrier();  // stagger the wave rows by one barrier
  if constexpr (ST) {
    if (stw) g8_stamp(blockIdx.x, strow, sti++, __builtin_amdgcn_s_memtime());
  }

  // one phase: reads -> prefetch -> [wait] -> barrier -> lgkmcnt(0) -> MFMA -> barrier
#define G8_SYNC_MMA(QA, QB, FB)                   \
  if constexpr (!(V & 2)) __builtin_amdgcn_s_barrier(); \
  lds_wait();                                     \
  pin_a();                                        \
  pin_b(FB);                                      \
  mma(QA, QB, FB);                                \
  if constexpr (V & 1) mma(QA, QB, FB);           \
  if constexpr (!(V & 2)) __builtin_amdgcn_s_barrier();

  if constexpr (PH == 4) {
#define G8_SYNC_MMA2(QA, QB0, FB0, QB1, FB1)              \
  __builtin_amdgcn_s_barrier();                           \
  pin_a();                                                \
  pin_b(FB0);                                             \
  pin_b(FB1);                                             \
  mma(QA, QB0, FB0);                                      \
  mma(QA, QB1, FB1);                                      \
  __builtin_amdgcn_s_barrier();
    for (int kt = 0;; kt += 2) {
      if constexpr (ST) {
        if (stw) g8_stamp(blockIdx.x, strow, sti++, __builtin_amdgcn_s_memtime());
      }
      // phase 1: buffer 0 (tile kt) B0, B1, A0; tile kt + 1's A0, A1 -> buffer 1
      read_b(0, 0, fb0);
      read_b(0, 1, fb1);
      read_a(0, 0);
      if (kt + 1 < nk) {
        issue(kt + 1, 0);
        issue(kt + 1, 1);
      }
      lds_wait();  // retired before the barrier: these images are restageable next phase
      G8_SYNC_MMA2(0, 0, fb0, 1, fb1)
      // phase 2: buffer 0 A1; tile kt + 2's B0, B1 -> buffer 0; retire tile kt + 1
      read_a(0, 1);
      if (kt + 2 < nk) {
        issue(kt + 2, 2);
        issue(kt + 2, 3);
        vm4();
      } else {
        vm0();
      }
      lds_wait();
      G8_SYNC_MMA2(1, 1, fb1, 0, fb0)
      if (kt + 1 >= nk) break;
      // phase 3: buffer 1 (tile kt + 1) B0, B1, A0; tile kt + 2's A0, A1 -> buffer 0
      read_b(1, 0, fb0);
      read_b(1, 1, fb1);
      read_a(1, 0);
      if (kt + 2 < nk) {
        issue(kt + 2, 0);
        issue(kt + 2, 1);
      }
      lds_wait();
      G8_SYNC_MMA2(0, 0, fb0, 1, fb1)
      // phase 4: buffer 1 A1; tile kt + 3's B0, B1 -> buffer 1; retire tile kt + 2
      read_a(1, 1);
      if (kt + 3 < nk) {
        issue(kt + 3, 2);
        issue(kt + 3, 3);
        vm4();
      } else {
        vm0();
      }
      lds_wait();
      G8_SYNC_MMA2(1, 1, fb1, 0, fb0)
      if (kt + 2 >= nk) break;
    }
#undef G8_SYNC_MMA2
  } else
  for (int kt = 0;; kt += 2) {
    if constexpr (ST) {
      if (stw) g8_stamp(blockIdx.x, strow, sti++, __builtin_amdgcn_s_memtime());
    }
    // phases 1-4: tile kt in buffer 0
    read_b(0, 0, fb0);
    read_a(0, 0);
    if (kt + 1 < nk) issue(kt + 1, 1);
    lds_wait_le(NA < 15 ? NA : 15);  // B0 reads retired before the barrier: B0 restageable in phase 2
    G8_SYNC_MMA(0, 0, fb0)
    read_b(0, 1, fb1);
    if (kt + 2 < nk) issue(kt + 2, 2);
    G8_SYNC_MMA(0, 1, fb1)
    read_a(0, 1);
    if (kt + 2 < nk) issue(kt + 2, 0);
    G8_SYNC_MMA(1, 1, fb1)
    if (kt + 2 < nk) {
      issue(kt + 2, 3);
      vm6();
    } else {
      vm0();
    }
    G8_SYNC_MMA(1, 0, fb0)
    if (kt + 1 >= nk) break;
    // phases 5-8: tile kt + 1 in buffer 1
    read_b(1, 0, fb0);
    read_a(1, 0);
    if (kt + 2 < nk) issue(kt + 2, 1);
    lds_wait_le(NA < 15 ? NA : 15);
    G8_SYNC_MMA(0, 0, fb0)
    read_b(1, 1, fb1);
    if (kt + 3 < nk) issue(kt + 3, 2);
    G8_SYNC_MMA(0, 1, fb1)
    read_a(1, 1);
    if (kt + 3 < nk) issue(kt + 3, 0);
    G8_SYNC_MMA(1, 1, fb1)
    if (kt + 3 < nk) {
      issue(kt + 3, 3);
      vm6();
    } else {
      vm0();
    }
    G8_SYNC_MMA(1, 0, fb0)
    if (kt + 2 >= nk) break;
  }
#undef G8_SYNC_MMA
  if (!(V & 2) && wr == 0) __builtin_amdgcn_s_barrier();  // match the stagger barrier
  if constexpr (ST) {
    if (stw) g8_stamp(blockIdx.x, strow, G8_NST - 3, __builtin_amdgcn_s_memtime());
  }

  // ---- epilogue: lane holds C[m][n .. n+3] per block
  const float alpha = alpha_f * (alpha_t ? alpha_t[0] : 1.f);
  float sqs = 0.f;  // ep.sq: this lane's sum of squares of the bf16 values it stores
  const int ml = m0 + wr * 128 + (lane & 15);
  const int nl = n0 + wc * 64 + 4 * (lane >> 4);
  if constexpr (EPI != G8_EPI_NONE) {
    g8_epilogue_fused<EPI>(acc, alpha, ml, pn, wc, lane, M, N, ep, C, ldc, mo, tl);
    return;
  }
#pragma unroll
  for (int qa = 0; qa < 2; ++qa) {
    f32x4 old[4][4];
    if constexpr (BETA) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int64_t m = ml + qa * 64 + 16 * i;
          const int n = nl + 32 * (j >> 1) + 16 * (j & 1);
          if constexpr (OUT_F32) {
            old[i][j] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(C) + m * ldc + n);
          } else {
            const uint2 v = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(C) + m * ldc + n);
            old[i][j] = f32x4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u),
                              __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u)};
          }
        }
    }
    if constexpr (OUT_F32) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int64_t m = ml + qa * 64 + 16 * i;
          const int n = nl + 32 * (j >> 1) + 16 * (j & 1);
          f32x4 v = acc[4 * qa + i][j] * alpha;
          if constexpr (BETA) v += old[i][j];
          *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(C) + m * ldc + n) = v;
        }
    } else {
      // bf16: blocks j, j + 1 are 16 columns apart and lanes l, l + 16 hold adjacent 4-column groups
      // of one row, so one v_permlane16_swap per packed dword pair gives every lane 8 consecutive
      // columns -> ONE 16-B store per block pair (guide T21, with the 16-lane swap) instead of two 8-B
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int jp = 0; jp < 2; ++jp) {
          f32x4 va = acc[4 * qa + i][2 * jp] * alpha, vb = acc[4 * qa + i][2 * jp + 1] * alpha;
          if constexpr (BETA) {
            va += old[i][2 * jp];
            vb += old[i][2 * jp + 1];
          }
          const auto s0 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(va[0], va[1]), pack_bf16x2(vb[0], vb[1]),
                                                          false, false);
          const auto s1 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(va[2], va[3]), pack_bf16x2(vb[2], vb[3]),
                                                          false, false);
          const int64_t m = ml + qa * 64 + 16 * i;
          const int n = n0 + wc * 64 + 32 * jp + 16 * ((lane >> 4) & 1) + 8 * (lane >> 5);
          uint4 o;
          o.x = s0[0];
          o.y = s1[0];
          o.z = s0[1];
          o.w = s1[1];
          *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(C) + m * ldc + n) = o;
          if (!BETA && ep.sq) sqs = g8_sq8(o, sqs);
        }
    }
  }
  if constexpr (!OUT_F32 && !BETA) {
    if (ep.sq) {  // workgroup-uniform: one fixed-order partial per output tile (deterministic)
      sqs = wave_sum(sqs);
      __syncthreads();  // every wave is past the K loop's LDS reads (its DMA drained at the last tile)
      float* red = reinterpret_cast<float*>(smem);
      if (lane == 0) red[w] = sqs;
      __syncthreads();
      if (tid == 0) {
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) t += red[i];
        ep.sq[pm * nN + pn] = t;
      }
    }
  }
  if constexpr (ST) {
    if (stw) {
      g8_stamp(blockIdx.x, strow, G8_NST - 2, __builtin_amdgcn_s_memtime());
      g8_stamp(blockIdx.x, strow, G8_NST - 1, __builtin_amdgcn_s_memrealtime());
    }
  }
}

// Sum of the S fp32 part images [M][N] of P in their order -> bf16 C [M][N]; GLU: N = 2F, C [M][F] = silu(gate) up of
// the sums rounded to bf16.  Bound by the images' bytes (the last level cache holds them: at most one 256 x 256 tile a CU).
template <bool GLU>
__global__ void __launch_bounds__(256) g8_parts_kernel(const float* __restrict__ P, int64_t part, int S, int N,
                                                       uint16_t* __restrict__ C, int64_t ldc, int64_t units) {
  const int F = GLU ? N / 2 : N, per = F / 8;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < units; i += (int64_t)gridDim.x * 256) {
    const int64_t m = i / per;
    const int n = (int)(i - m * per) * 8;
    const float* p = P + m * N + n;
    f32x4 a[GLU ? 4 : 2];
#pragma unroll
    for (int h = 0; h < (GLU ? 4 : 2); ++h) a[h] = *reinterpret_cast<const f32x4*>(p + 4 * (h & 1) + (h >> 1) * F);
#pragma unroll 4
    for (int s = 1; s < S; ++s) {
#pragma unroll
      for (int h = 0; h < (GLU ? 4 : 2); ++h)
        a[h] += *reinterpret_cast<const f32x4*>(p + s * part + 4 * (h & 1) + (h >> 1) * F);
    }
    u16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float v = a[j >> 2][j & 3];
      if constexpr (GLU) {
        const float g = g8_rbf(v);
        v = g * g8_sigmoid(g) * g8_rbf(a[2 + (j >> 2)][j & 3]);
      }
      o[j] = f2bf(v);
    }
    *reinterpret_cast<u16x8*>(C + m * ldc + n) = o;
  }
}

}  // namespace mx
