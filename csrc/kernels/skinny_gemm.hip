// bf16 weight-streaming GEMM for decode on gfx950: Y[M, N] = X[M, K] . W[N, K]^T with M <= 32
// tokens (serving path).  A decode step reads every weight once;
// for the small projections of an 8B model (34-117 MB) hipBLASLt's skinny solutions stream at
// 1.7-4.5 TB/s (archive/profiles/r2x_skinny_gemm.md), latency-bound: too few bytes in flight per CU.
//
// Same structure as the fp8 weight kernel (fp8_gemm.hip) without the dequantisation:
//  * workgroup = 8 waves = 16 output channels, N/16 workgroups; the waves split K (skinny_core.h) and meet in LDS;
//  * v_mfma_f32_16x16x32_bf16 with the WEIGHTS as the A operand and X^T as the B operand;
//  * 8 chunks' loads are issued before the first is used: 256 B of weights per lane in flight, 128 KB per workgroup.
//  * SWO (SwiGLU output, the decode MLP's gate|up projection, W = [gate; up] [2F, K]): a
//    workgroup's 16 channels are 8 gate rows n..n+7 and the matching 8 up rows F+n..F+n+7, so
//    the epilogue holds both halves of its 8 outputs and writes silu(g) * u [M, F] directly
//    (g, u rounded to bf16 first, as the separate GEMM + SwiGLU kernels round them: same bits).
//    Same weight stream as the plain kernel; one launch and the [M, 2F] round trip less.
//  * NORM (decode, M <= 4 rows): the RMSNorm (with the residual add) that produces X runs in
//    the prologue: every workgroup rebuilds the normalised rows in LDS from the residual h
//    (and the sub-block output `delta`), with the thread mapping, summation order and
//    rounding of rmsnorm.hip's forward kernel (same bits); workgroup 0 stores h + delta.
//    The X fragments then come from LDS.  Saves the two RMSNorm launches of every layer.
//  * ROPE (decode QKV projection, head_dim 128): a workgroup's 16 channels are 8 first-half
//    channels i..i+7 of one head and the matching second-half channels 64+i..64+i+7, so the
//    epilogue holds both halves of each rotation pair and does decode.hip rope_append's work:
//    rotated q rows -> q, rotated k and plain v rows -> the KV cache at (slot, pos).  Saves the
//    rope_append launch of every layer.
#include <cstdlib>

#include "common.h"
#include "decode_fuse.h"
#include "skinny_core.h"

namespace mx {

// TB: 8-token blocks (1, 2 or 4); X rows >= M are clamped to M-1 and discarded.
// NC: 16-channel groups per workgroup: each X fragment then feeds NC MFMAs, so X traffic per
// streamed weight byte drops NC-fold (it equals the weight traffic at 16 tokens with NC = 1).
// KP: K parts (sk_parts).  HALF: 8 channels a workgroup, 8 K parts, M <= 8.  WIDE: 16-row fragments and TB blocks of 16 tokens
// (sk_wide).  WHOLE: chunks of a wave's K part, loaded together.
template <int TB, int NC, int KP, bool SWO = false, bool NORM = false, bool ROPE = false, bool MERGE = false,
          bool HALF = false, bool WIDE = false, bool DEEP = false, int WHOLE = 0>
__global__ void __launch_bounds__(512) skinny_gemm_kernel(const uint16_t* __restrict__ X, int64_t ldx,
                                                          const uint16_t* __restrict__ W, int64_t ldw,
                                                          uint16_t* __restrict__ Y, int64_t ldy, int M, int K,
                                                          int F = 0, SkNorm na = {}, SkRope rp = {},
                                                          SkMerge mg = {}) {
  static_assert(!SWO || NC == 1, "SwiGLU epilogue: one channel group");
  static_assert(!ROPE || (NC == 1 && !SWO), "RoPE epilogue: one channel group");
  static_assert(!NORM || (TB == 1 && NC == 1), "fused RMSNorm: <= 8 rows, one channel group");
  static_assert(!MERGE || (TB == 1 && NC == 1 && !NORM && !SWO && !ROPE), "fused split merge: plain GEMM rows");
  static_assert(!HALF || (TB == 1 && NC == 1 && KP == 8 && !SWO && !NORM && !ROPE && !MERGE), "half groups: plain GEMM rows");
  constexpr bool LDSX = NORM || MERGE;  // X rows built in LDS by the prologue
  static_assert(!WIDE || (NC == 1 && KP == 8 && !NORM && !ROPE && !MERGE && !HALF), "16-row fragments: plain rows, SwiGLU");
  constexpr int UNR = sk_unr(NC), RB = HALF ? 1 : kSkBlocks<KP, NC>, BT = WIDE ? 16 : 8;  // tokens of a block
  typedef SkSum<TB, NC, KP> Sum;
  __shared__ f32x4 red[HALF ? kSkWaves * 16 : WIDE ? kSkWaves * TB * 64 : Sum::PLACES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (HALF ? 8 : 16 * NC);
  const int kq = K / KP;  // this wave's K part
  const int64_t k0 = (int64_t)sk_part<KP>(w) * kq + (WIDE ? 8 * g : sk_lane_k(c, g));
  const uint16_t* wrow[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int ch = WIDE ? c : (HALF ? 0 : 8 * sk_half<KP>(w, rb)) + (c & 7), j = KP == 8 ? rb >> 1 : rb;
    // SWO: channels 0 .. 7: gate rows blockIdx.x * 8 + ch, 8 .. 15: the matching up rows
    // ROPE: head blockIdx.x / 8, pair base 8 (blockIdx.x % 8); channels 8 .. 15: the second-half rows
    const int64_t wr = (SWO || ROPE) ? dfuse_row<SWO>(blockIdx.x, ch, F) : (int64_t)(n0 + 16 * j + ch);
    wrow[rb] = W + wr * ldw + k0 + (WIDE ? 32 * rb : 0);
  }
  const uint16_t* xr[TB];
  const int nit = kq / 64;
  // NORM: the first UNR chunks' weight loads go out before the prologue, so the weight stream's
  // latency overlaps the RMSNorm instead of following it
  u16x8 apre[UNR][RB];
  if constexpr (LDSX) sk_prefetch<NC>(wrow, nit, apre);
  if constexpr (LDSX) {
    extern __shared__ __attribute__((aligned(16))) uint16_t xs[];  // [M, K] normalised / merged rows
    if constexpr (NORM) {
      __shared__ float nscr[2][4];
      __shared__ float nrs[4];
      dfuse_norm_rows(X, ldx, M, K, na, xs, K, nscr, nrs);
    } else {
      dfuse_merge_rows(M, K, mg, xs);
    }
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) xr[tb] = xs + (int64_t)min(tb * 8 + (c & 7), M - 1) * K + k0;
  } else {
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) xr[tb] = X + (int64_t)min(tb * BT + (c & (BT - 1)), M - 1) * ldx + k0;
  }

  f32x4 acc[RB][TB];
  sk_stream<TB, NC, LDSX, WIDE, DEEP, WHOLE>(wrow, xr, nit, apre, acc);
  if constexpr (HALF) {
    const f32x4 part = sk_both_halves(acc[0][0]);
    if (c < 8 && g < 2) red[w * 16 + 8 * g + c] = part;
    __syncthreads();
    if (w == 0 && g < 2 && c < M) {
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ww = 0; ww < kSkWaves; ++ww) s += red[ww * 16 + 8 * g + c];
      u16x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = f2bf(s[i]);
      *reinterpret_cast<u16x4*>(Y + (int64_t)c * ldy + n0 + 4 * g) = o;
    }
  } else {
    const Sum sum{red};
    if constexpr (WIDE) {
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) red[(w * TB + tb) * 64 + lane] = acc[0][tb];
    } else {
      sum.put(w, c, g, acc);
    }
    __syncthreads();
    if (w == 0) {
#pragma unroll
      for (int j = 0; j < NC; ++j)
#pragma unroll
        for (int mb = 0; mb < (WIDE ? TB : (TB + 1) / 2); ++mb) {
          f32x4 s = {0.f, 0.f, 0.f, 0.f};
          if constexpr (WIDE) {
#pragma unroll
            for (int ww = 0; ww < kSkWaves; ++ww) s += red[(ww * TB + mb) * 64 + lane];
          } else {
            s = sum.get(c, g, j, mb);
          }
          const int m = mb * 16 + c;
          if constexpr (ROPE) {
            dfuse_rope_store(s, g, m, M, blockIdx.x, rp);
          } else if constexpr (SWO) {
            dfuse_swiglu_store(s, g, m, M, Y, ldy, blockIdx.x);
          } else if (m < M) {
            u16x4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = f2bf(s[i]);
            *reinterpret_cast<u16x4*>(Y + (int64_t)m * ldy + n0 + 16 * j + 4 * g) = o;
          }
        }
    }
  }
}

}  // namespace mx

// Where the kernel whose workgroups stay (stream_gemm.hip: X in LDS once a CU) takes less time, with the same bits but for its
// 16-row fragments of a K of 4096 and up to 3072 channels, which go there as long as the addresses allow (us, here ->
// there: K 2048, 3 / 8 / 32 rows: 3072 channels 5.2 / 6.1 / 8.8 -> 5.1 / 5.3 / 8.5, 16384 13.8 / 17.0 / 29.7 -> 13.0 / 13.4 / 18.6,
// 2 rows 12.8 -> 13.0; K 4096, 16 rows: 1024 channels 9.7 -> 9.1, 4096, one group a CU, 10.2 -> 10.5).
extern "C" int mx_stream_gemm(const uint16_t* x, int64_t ldx, const void* w, int64_t ldw, const float* scale, uint16_t* y,
                              int64_t ldy, int M, int N, int K, int epi, const uint16_t* delta, int64_t ldd,
                              const uint16_t* gamma, float eps, uint16_t* h_out, const float* cosb, const float* sinb,
                              const int32_t* pos, const int32_t* slots, uint16_t* q, uint16_t* kc, uint16_t* vc, int Hq,
                              int Hkv, int max_seq, const int32_t* bt, int maxb, hipStream_t stream);
extern "C" int mx_stream_ok(int M, int K, int norm);
// whether mx_skinny_gemm and mx_skinny_gemm_swiglu (N = 2 F) hand rows of these sizes on to it
extern "C" int mx_skinny_stays(int M, int N, int K) {
  return mx_stream_ok(M, K, 0) && (K == 2048 ? M > 2 : K == 4096 && M > 8 && M <= 16 && !(N > 3072 && N <= 4096));
}
// epi 0: plain, 1: SwiGLU (N = 2 F); -1: not taken
static int sk_stream_gemm(const uint16_t* x, int64_t ldx, const uint16_t* w, int64_t ldw, uint16_t* y, int64_t ldy, int M, int N,
                          int K, int epi, hipStream_t stream) {
  if (!mx_skinny_stays(M, N, K)) return -1;
  return mx_stream_gemm(x, ldx, w, ldw, nullptr, y, ldy, M, N, K, epi, nullptr, 0, nullptr, 0.f, nullptr, nullptr, nullptr,
                        nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, nullptr, 0, stream);
}

// the kernel of the sizes' K parts: KERNEL(4) or KERNEL(8)
#define SK_PARTS(KERNEL) \
  if (sk_parts(M, K) == 4) KERNEL(4); \
  else KERNEL(8)

using namespace mx;

// y = rmsnorm(h [+ delta]) . W^T (or with the SwiGLU epilogue: W = [gate; up], y [M, N/2]) for
// M <= 4 decode rows: the RMSNorm in the GEMM prologue (see NORM above).  h [M, K] (row stride
// ldh), delta [M, K] (row stride ldd) or nullptr, gamma [K]; h_out [M, K] (row stride K) gets
// h + delta when delta is given.  Requires M * K <= 32768 (64 KiB of LDS), K % 512 == 0.
// Decode QKV projection with the RoPE / KV-cache append in the epilogue (see ROPE above), and
// optionally the RMSNorm in the prologue (h, delta, gamma as mx_skinny_norm_gemm; norm = 0: X = h
// as is, any M <= 16).  w [(Hq + 2 Hkv) * 128, K]; q out [M, Hq, 128].
extern "C" int mx_skinny_rope_gemm(const uint16_t* h, int64_t ldh, int norm, const uint16_t* delta, int64_t ldd,
                                   const uint16_t* gamma, float eps, uint16_t* h_out, const uint16_t* w, int64_t ldw,
                                   const float* cosb, const float* sinb, const int32_t* pos, const int32_t* slots,
                                   uint16_t* q, uint16_t* kc, uint16_t* vc, int Hq, int Hkv, int max_seq,
                                   const int32_t* bt, int maxb, int M, int K, hipStream_t stream) {
  if (M <= 0) return 0;
  const int N = (Hq + 2 * Hkv) * 128;
  if (M > (norm ? 4 : 16) || (norm && (int64_t)M * K > 32768) || K % 512 || ldh % 8 || ldd % 8 || ldw % 8 ||
      ldh < K || ldw < K || (norm && delta && (ldd < K || !h_out)))
    return -1;
  // Past 4 rows of 2048 X is in LDS (us, 3072 channels, 6 / 8 rows 6.2 / 6.6 -> 5.9 / 6.1; 4 rows 5.9), with the same bits.
  if (!norm && K == 2048 && M > 4 &&
      mx_stream_gemm(h, ldh, w, ldw, nullptr, nullptr, 0, M, N, K, 2, nullptr, 0, nullptr, 0.f, nullptr, cosb, sinb, pos, slots, q,
                     kc, vc, Hq, Hkv, max_seq, bt, maxb, stream) == 0)
    return 0;
  const SkRope rp{cosb, sinb, pos, slots, q, kc, vc, Hq, Hkv, max_seq, bt, maxb};
  if (norm) {
    const SkNorm na{delta, ldd, gamma, h_out, eps};
#define SKR(KP) skinny_gemm_kernel<1, 1, KP, false, true, true><<<N / 16, 512, (size_t)M * K * 2, stream>>>( \
      h, ldh, w, ldw, nullptr, 0, M, K, 0, na, rp)
    SK_PARTS(SKR);
#undef SKR
  } else {
#define SKR(KP) skinny_gemm_kernel<1, 1, KP, false, false, true><<<N / 16, 512, 0, stream>>>(h, ldh, w, ldw, nullptr, 0, M, K, \
                                                                                            0, SkNorm{}, rp)
#define SKR2(KP) skinny_gemm_kernel<2, 1, KP, false, false, true><<<N / 16, 512, 0, stream>>>(h, ldh, w, ldw, nullptr, 0, M, K, \
                                                                                             0, SkNorm{}, rp)
    if (M <= 8) {
      SK_PARTS(SKR);
    } else {
      SK_PARTS(SKR2);
    }
#undef SKR
#undef SKR2
  }
  return (int)hipGetLastError();
}

// y[M, N] = merge(split partials) . W^T: the decode o-projection with decode.hip's split-K
// attention merge (decode_combine_kernel) in its prologue -- every workgroup rebuilds the
// attention output rows [M, Hq * 128] in LDS from part_ml [M, Hq, nsplit, 2] / part_o
// [M, Hq, nsplit, 128] (same bits as the combine kernel).  Saves the combine launch of every
// layer.  M <= 4, M * K <= 32768, K = Hq * 128 (% 512), N % 16 == 0.
extern "C" int mx_skinny_merge_gemm(const float* ml, const float* po, int nsplit, const uint16_t* w, int64_t ldw,
                                    uint16_t* y, int64_t ldy, int M, int N, int K, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 4 || (int64_t)M * K > 32768 || N % 16 || K % 512 || ldw % 8 || ldy % 4 || ldw < K || ldy < N ||
      nsplit < 1)
    return -1;
  const SkMerge mg{ml, po, nsplit};
#define SKM(KP) skinny_gemm_kernel<1, 1, KP, false, false, false, true><<<N / 16, 512, (size_t)M * K * 2, stream>>>( \
      nullptr, 0, w, ldw, y, ldy, M, K, 0, SkNorm{}, SkRope{}, mg)
  SK_PARTS(SKM);
#undef SKM
  return (int)hipGetLastError();
}

extern "C" int mx_skinny_norm_gemm(const uint16_t* h, int64_t ldh, const uint16_t* delta, int64_t ldd,
                                   const uint16_t* gamma, float eps, uint16_t* h_out, const uint16_t* w,
                                   int64_t ldw, uint16_t* y, int64_t ldy, int M, int N, int K, int swiglu,
                                   hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 4 || (int64_t)M * K > 32768 || N % 16 || K % 512 || ldh % 8 || ldd % 8 || ldw % 8 || ldy % 4 ||
      ldh < K || ldw < K || (delta && (ldd < K || !h_out)))
    return -1;
  const SkNorm na{delta, ldd, gamma, h_out, eps};
  const size_t lds = (size_t)M * K * 2;
  if (swiglu) {
    const int Fh = N / 2;
    if (Fh % 8 || ldy < Fh) return -1;
#define SKN(KP) skinny_gemm_kernel<1, 1, KP, true, true><<<Fh / 8, 512, lds, stream>>>(h, ldh, w, ldw, y, ldy, M, K, Fh, na)
    SK_PARTS(SKN);
#undef SKN
  } else {
    if (ldy < N) return -1;
#define SKN(KP) skinny_gemm_kernel<1, 1, KP, false, true><<<N / 16, 512, lds, stream>>>(h, ldh, w, ldw, y, ldy, M, K, 0, na)
    SK_PARTS(SKN);
#undef SKN
  }
  return (int)hipGetLastError();
}

// X [M, K] bf16 (row stride ldx), W [N, K] bf16 (row stride ldw), Y [M, N] bf16 (row stride
// ldy).  Requires M in 1..32, N % 16 == 0, K % 512 == 0, ldx / ldw multiples of 8, ldy of 4.
extern "C" int mx_skinny_gemm(const uint16_t* x, int64_t ldx, const uint16_t* w, int64_t ldw, uint16_t* y,
                              int64_t ldy, int M, int N, int K, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 32 || N % 16 || K % 512 || ldx % 8 || ldw % 8 || ldy % 4 || ldx < K || ldw < K || ldy < N) return -1;
  // MXLLM_SKINNY_NC: channel groups per workgroup (1, 2 or 4; default 1).  Two or four groups
  // cut the X traffic but halve / quarter the workgroups; measured at the Llama 8B / 70B decode
  // shapes they won only on the 8B qkv projection (archive/profiles/r2x_skinny_gemm.md)
  static const int nc_env = [] {
    const char* e = getenv("MXLLM_SKINNY_NC");
    return e && *e ? atoi(e) : 0;
  }();
  if (!nc_env && sk_stream_gemm(x, ldx, w, ldw, y, ldy, M, N, K, 0, stream) == 0) return 0;
  int nc = nc_env ? nc_env : 1;
  while (nc > 1 && (N % (16 * nc) || N / (16 * nc) < 128)) nc >>= 1;
#define SKG(TBV, NCV, KPV) \
  skinny_gemm_kernel<TBV, NCV, KPV><<<N / (16 * NCV), 512, 0, stream>>>(x, ldx, w, ldw, y, ldy, M, K)
#define SKT(NCV, KPV) /* 4 K parts: up to 16 rows */ \
  do { \
    if (M <= 8) SKG(1, NCV, KPV); else if (M <= 16) SKG(2, NCV, KPV); else SKG(KPV == 4 ? 2 : 4, NCV, KPV); \
  } while (0)
  // up to two workgroups a CU (us, compiler's order -> DEEP, one row: 4096 x 4096 7.7 -> 7.6, 4096 x 14336 23.1 -> 21.9; 128256 x
  // 2048 82 -> 88)
  if (M <= 8 && nc == 1 && N <= 16 * 512) {
#define SKD(KPV) \
  skinny_gemm_kernel<1, 1, KPV, false, false, false, false, false, false, true><<<N / 16, 512, 0, stream>>>(x, ldx, w, ldw, y, ldy, M, K)
    SK_PARTS(SKD);
#undef SKD
    return (int)hipGetLastError();
  }
#define SKC(KPV) \
  do { \
    if (nc >= 4) SKT(4, KPV); else if (nc == 2) SKT(2, KPV); else if (M <= 8) SKG(1, 1, KPV); else SKG(2, 1, KPV); \
  } while (0)
  if (sk_wide(M, K) && nc == 1) {
    if (M <= 16) skinny_gemm_kernel<1, 1, 8, false, false, false, false, false, true><<<N / 16, 512, 0, stream>>>(x, ldx, w, ldw, y, ldy, M, K);
    else skinny_gemm_kernel<2, 1, 8, false, false, false, false, false, true><<<N / 16, 512, 0, stream>>>(x, ldx, w, ldw, y, ldy, M, K);
    return (int)hipGetLastError();
  }
  SK_PARTS(SKC);
#undef SKC
#undef SKT
#undef SKG
  return (int)hipGetLastError();
}

// The same for up to 8 rows by groups of 8 channels (HALF): twice the workgroups, where 16 channels each leave CUs
// without one.  2048 channels, one row: K 8192 10.5 -> 8.0 us, K 12288 14.5 -> 11.0, K 2048 4.5 -> 3.7 (8 rows:
// 13.1 -> 9.9, 18.5 -> 14.0, 5.8 -> 4.4).  Always 8 K parts: for a K of 2048 other bits than above.
// K % 1024 == 0, N % 8 == 0.
extern "C" int mx_skinny_gemm_half(const uint16_t* x, int64_t ldx, const uint16_t* w, int64_t ldw, uint16_t* y,
                                   int64_t ldy, int M, int N, int K, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 8 || N % 8 || K % 1024 || ldx % 8 || ldw % 8 || ldy % 4 || ldx < K || ldw < K || ldy < N) return -1;
  // DEEP up to where the waves that it leaves are busy (2048 x 2048, one row 3.9 -> 3.7 us, 4096 x 4096 7.7 -> 7.5, 2048 x 8192 8.0 -> 8.4)
  if (K <= 4096)
    skinny_gemm_kernel<1, 1, 8, false, false, false, false, true, false, true><<<N / 8, 512, 0, stream>>>(x, ldx, w, ldw, y, ldy, M, K);
  // One workgroup a CU has the registers for a whole K part of up to 30 chunks in flight (231; scratch at 32), and nothing
  // beside it to hide its turns of 8 chunks.  Weights from memory, 1 / 4 / 8 rows, turns -> whole, us: 2048 x 9216 8.9 / 10.0 / 10.9 -> 7.9 /
  // 9.0 / 10.4, x 11264 11.4 / 12.6 / 13.1 -> 10.0 / 11.4 / 12.2, x 12288 12.0 / 13.6 / 14.0 -> 10.8 / 12.2 / 13.2, x 15360 14.6 / 16.3 / 16.8 ->
  // 12.7 / 14.9 / 16.0; 1024 x 10240 8.9 / 10.2 / 11.9 -> 7.8 / 9.5 / 11.1.  2048 x 12288 in a step of revesun-1b with 1 / 2 / 4 / 8 rows
  // 758 / 791 / 838 / 966 -> 740 / 771 / 823 / 953.  Rows ahead of the weights or behind them: as good or worse.  Two turns are level or
  // better left (2048 x 8192, a step of llama3.2-1b of one row 684 -> 684, beside other processes 686 -> 697).
#define SKH(U) \
  else if (N <= 8 * 256 && K == 512 * U) \
    skinny_gemm_kernel<1, 1, 8, false, false, false, false, true, false, false, U><<<N / 8, 512, 0, stream>>>(x, ldx, w, ldw, y, ldy, M, K);
  SKH(18) SKH(20) SKH(22) SKH(24) SKH(26) SKH(28) SKH(30)
#undef SKH
  else
    skinny_gemm_kernel<1, 1, 8, false, false, false, false, true><<<N / 8, 512, 0, stream>>>(x, ldx, w, ldw, y, ldy, M, K);
  return (int)hipGetLastError();
}

// y[M, F] = silu(g) * u with [g | u] = x[M, K] . W[2F, K]^T, W = [gate; up] rows: the decode
// MLP's gate|up projection with the SwiGLU in its epilogue.  Same contract as mx_skinny_gemm
// with N = 2F, plus F % 8 == 0.
extern "C" int mx_skinny_gemm_swiglu(const uint16_t* x, int64_t ldx, const uint16_t* w, int64_t ldw, uint16_t* y,
                                     int64_t ldy, int M, int F, int K, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 32 || F % 8 || K % 512 || ldx % 8 || ldw % 8 || ldy % 4 || ldx < K || ldw < K || ldy < F) return -1;
  if (sk_stream_gemm(x, ldx, w, ldw, y, ldy, M, 2 * F, K, 1, stream) == 0) return 0;
#define SKS(TBV, KPV) skinny_gemm_kernel<TBV, 1, KPV, true><<<F / 8, 512, 0, stream>>>(x, ldx, w, ldw, y, ldy, M, K, F)
#define SKT(KPV) \
  do { \
    if (M <= 8) SKS(1, KPV); else SKS(2, KPV); \
  } while (0)
  if (sk_wide(M, K)) {
    if (M <= 16) skinny_gemm_kernel<1, 1, 8, true, false, false, false, false, true><<<F / 8, 512, 0, stream>>>(x, ldx, w, ldw, y, ldy, M, K, F);
    else skinny_gemm_kernel<2, 1, 8, true, false, false, false, false, true><<<F / 8, 512, 0, stream>>>(x, ldx, w, ldw, y, ldy, M, K, F);
    return (int)hipGetLastError();
  }
  SK_PARTS(SKT);
#undef SKT
#undef SKS
  return (int)hipGetLastError();
}
