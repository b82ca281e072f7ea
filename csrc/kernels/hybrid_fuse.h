// Operands and epilogues of the fused decode GEMMs of the recurrent / chunked-attention decoders (hybrid_skinny.hip).
#pragma once

#include "conv_rope.h"
#include "hybrid.h"

namespace mx {

struct HsNorm {
  const uint16_t* delta;  // [M, K] or nullptr
  int64_t ldd;
  const float* h;         // [M, K] f32 residual
  const float* gamma;     // [K]
  float* h_out;           // [M, K]: h + delta (when delta)
  int groups;
  float eps;
};
struct HsPoly {
  const float* coef;
  float eps;
};
struct HsGru {
  const float* bias;      // [2 W]: z | u
  const int32_t* slots;
  float* state;           // [slots, W]
  int W;
};
struct HsConv {
  ConvRope a;             // x unused; q [M, H, Dp]
  const int32_t* pos;
  const int32_t* slots;
  uint16_t* gate;         // [M, H E]
};

// weight row of channel ch of a group: 4 channels each of z, u and the gate, the last quarter idle (the gate's again)
__device__ __forceinline__ int64_t hs_gru_row(int blk, int ch, int W) {
  return (int64_t)min(ch >> 2, 2) * W + blk * 4 + (ch & 3);
}

// lane (c, g): v[i] = projection g (z, u, gate) of channel 4 blk + i for token c
__device__ __forceinline__ void hs_gru_store(const f32x4& v, int lane, int M, int blk, const HsGru& gr, uint16_t* Y) {
  f32x4 u, gt;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    u[i] = __uint_as_float(lane_pair<16>(__float_as_uint(v[i])).b);  // lanes 0 .. 15: of lane + 16, of lane + 32
    gt[i] = __uint_as_float(lane_pair<32>(__float_as_uint(v[i])).b);
  }
  const int m = lane & 15, c = blk * 4;
  if (lane < 16 && m < M) {
    float* sp = gr.state + (int64_t)gr.slots[m] * gr.W + c;
    float bz[4], bu[4], s[4], o[4];
    ldv<4>(gr.bias + c, bz);
    ldv<4>(gr.bias + gr.W + c, bu);
    ldv<4>(sp, s);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float keep, add;
      mingru_gate<uint16_t>(v[i] + bz[i], u[i] + bu[i], keep, add);
      s[i] = keep * s[i] + add;
      o[i] = s[i] * (gt[i] * sigmoid_t<uint16_t>(gt[i]));
    }
    stv<4>(sp, s);
    stv<4>(Y + (int64_t)m * gr.W + c, o);
  }
}

// v: channels [ch, ch + 4) of token m, all of one section and head
__device__ __forceinline__ void hs_conv_store(const f32x4& v, int ch, int m, int M, const HsConv& cv) {
  if (m >= M) return;
  const ConvRope& a = cv.a;
  const int qk = (a.H + a.G) * a.D, C = qk + a.G * a.E;
  float u[4], y[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) u[i] = bf2f(f2bf(v[i]));  // the projection as the ring stores it
  if (ch >= C) {
    stv<4>(cv.gate + (int64_t)m * a.H * a.E + (ch - C), u);
    return;
  }
  const int p = cv.pos[m], slot = cv.slots[m];
  uint16_t* ring = reinterpret_cast<uint16_t*>(a.ring) + (int64_t)slot * a.taps * C + ch;
  float wv[4];
  ldv<4>(a.w + (int64_t)(a.taps - 1) * C + ch, wv);
#pragma unroll
  for (int i = 0; i < 4; ++i) y[i] = wv[i] * u[i];
  for (int back = 1; back < a.taps && back <= p; ++back) {
    float o[4];
    ldv<4>(ring + (int64_t)((p - back) % a.taps) * C, o);
    ldv<4>(a.w + (int64_t)(a.taps - 1 - back) * C + ch, wv);
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] += wv[i] * o[i];
  }
  stv<4>(ring + (int64_t)(p % a.taps) * C, u);
  const int sec = ch < a.H * a.D ? 0 : ch < qk ? 1 : 2;
  const int rel = sec == 0 ? ch : sec == 1 ? ch - a.H * a.D : ch - qk;
  const int dim = sec < 2 ? a.D : a.E, Wp = sec < 2 ? a.Dp : a.Ep;
  const int head = rel / dim, d0 = rel % dim;
  if (sec < 2) {
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      if (d0 + i + 1 < a.rd) {
        const int64_t t = (int64_t)p * (a.rd >> 1) + ((d0 + i) >> 1);
        const float c = a.cosb[t], s = a.sinb[t], e = y[i], f = y[i + 1];
        y[i] = e * c - f * s;
        y[i + 1] = f * c + e * s;
      }
    }
  }
  if (sec == 0) {
    uint16_t* q = reinterpret_cast<uint16_t*>(a.q) + head * a.qh + (int64_t)m * a.qt;
    stv<4>(q + d0, y);
    if (d0 + 4 >= dim)
      for (int d = dim; d < Wp; ++d) q[d] = 0;
  } else {
    uint16_t* cache = reinterpret_cast<uint16_t*>(sec == 1 ? a.kc : a.vc);
    stv<4>(cache + kv_row(a.bt, a.maxb, a.block, slot, a.G, head, p % a.chunk) * Wp + d0, y);
  }
}

// weight rows of the convolved projection, in whole groups of 16; 0: sizes that hs_conv_store does not take
static inline int hs_conv_rows(const ConvRope& a) {
  const int N = (a.H + a.G) * a.D + a.G * a.E + a.H * a.E;
  if (N % 16 || a.D % 4 || a.E % 4 || a.Dp % 4 || a.Ep % 4 || a.rd % 2 || a.rd > a.D || a.H <= 0 || a.G <= 0 ||
      a.H % a.G || a.taps < 1 || a.chunk <= 0 || a.block <= 0 || !a.ring || !a.kc || !a.vc || !a.bt || a.Dp < a.D ||
      a.Ep < a.E)
    return 0;
  return N;
}

}  // namespace mx
