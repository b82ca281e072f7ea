// The second embedding's gate in prompt passes (sigusun, mxllm/models/sigusun.py): gelu_tanh(x w^T) times the token's row of that
// embedding, w of few channels (64 of 4096).
#include "gemm8_core.h"
#include "hybrid.h"

namespace mx {

template <int N>
__device__ __forceinline__ void sg_vm_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// What bounds it: 64 k of a wave, which wait for their DMA, their LDS reads and their products behind one another; the bytes (2048
// rows of 4096: 16 MB, 2.7 us from memory) come by the side.  The library's product, which has 128 tiles there, takes 19.9 us in a
// prompt pass, and side_act 4.8 (this one 13.5).  So tiles are as small as a wave's block, one wave each: nothing is shared, there is no barrier,
// and S stages of 64 k (a row's 128 bytes are a line) are on their way.  K stays in order, as the library has it: the bits are the
// same wherever that does not cut K.  With side_act, replayed, 65 / 512 / 2048 / 4096 / 8192 rows of 64 x 4096, us: 12.7 / 13.2 /
// 18.0 / 19.3 / 19.8 -> 7.9 / 8.6 / 9.3 / 12.0 / 15.5; 64 x 2048 9.7 / 10.5 / 11.4 / 11.9 / 11.5 -> 5.0 / 5.6 / 6.3 / 7.8 / 10.3; 8
// stages are the same.  Blocks of 32 rows lose below 8192 rows (2048: 11.3), 64 channels a wave everywhere (16.7).  Fragments
// loaded straight from memory, 16 rows x 64 B a load, have half the rate (2048 rows 17.0).
template <int BJ, int S>
__global__ void __launch_bounds__(64) side_gate_kernel(const uint16_t* __restrict__ x, int64_t ldx, const uint16_t* __restrict__ w,
                                                       int64_t ldw, const uint16_t* __restrict__ emb, int64_t lde,
                                                       const int64_t* __restrict__ ids, int V, uint16_t* __restrict__ y, int T,
                                                       int N, int K) {
  constexpr int P = 2 + 2 * BJ, STG = P * 1024;  // pieces of 8 rows of a stage
  static_assert((S - 1) * P <= 63, "vmcnt");
  __shared__ __attribute__((aligned(1024))) char smem[S * STG];
  const int lane = threadIdx.x, c = lane & 15, g = lane >> 4;
  // the channels' waves of a row block on one XCD, so that its L2 has the rows once
  const int nc = (N + 16 * BJ - 1) / (16 * BJ), x8 = blockIdx.x & 7, q = blockIdx.x >> 3;
  const int t0 = (q / nc * 8 + x8) * 16, n0 = q % nc * 16 * BJ;
  if (t0 >= T) return;
  const int row = t0 + c;
  int64_t id = ids[min(row, T - 1)];
  const uint16_t *xb = x + (int64_t)t0 * ldx, *wb = w + (int64_t)n0 * ldw;
  const int xrows = min(T - t0, 16), wrows = min(N - n0, 16 * BJ);
  const __amdgpu_buffer_rsrc_t xrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)xb, 0, (uint32_t)(((xrows - 1) * ldx + K) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t wrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)wb, 0, (uint32_t)(((wrows - 1) * ldw + K) * 2), 0x00020000);
  uint32_t off[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int r = 8 * (p < 2 ? p : p - 2) + (lane >> 3), ch = (lane & 7) ^ ((r >> 1) & 7);
    off[p] = (uint32_t)(((p < 2 ? min(r, xrows - 1) * ldx : min(r, wrows - 1) * ldw) + 8 * ch) * 2);
  }
  const int nk = K / 64;
  auto piece = [&](int p, uint32_t k, char* d) __attribute__((always_inline)) {
    const uint32_t so = off[p] + k;
    if (p < 2) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (g8lptr_t)d, 16, so, 0, 0, 0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (g8lptr_t)d, 16, so, 0, 0, 0);
    }
  };
  auto stage = [&](int t, int st) __attribute__((always_inline)) {
    const uint32_t so = t < nk ? 128 * t : G8_OOB;
#pragma unroll
    for (int p = 0; p < P; ++p) piece(p, so, smem + st * STG + p * 1024);
  };
#pragma unroll
  for (int t = 0; t < S; ++t) stage(t, t);
  id = id < 0 ? 0 : (id >= V ? V - 1 : id);
  u16x4 e[BJ];
#pragma unroll
  for (int j = 0; j < BJ; ++j) e[j] = *reinterpret_cast<const u16x4*>(emb + id * lde + min(n0 + 16 * j + 4 * g, N - 4));
  f32x4 acc[BJ] = {};
  u16x8 fx[2][2], fw[2][BJ][2];
  const uint32_t lds0 = lds_addr(smem), l0 = lds0 + g8_kc_lane(lane, 0), l1 = lds0 + g8_kc_lane(lane, 1);
  auto read = [&](int b, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < BJ; ++j) {
      fw[b][j][0] = rd128_off(l0 + st * STG, (1 + j) * 2048);
      fw[b][j][1] = rd128_off(l1 + st * STG, (1 + j) * 2048);
    }
    fx[b][0] = rd128_off(l0 + st * STG, 0);
    fx[b][1] = rd128_off(l1 + st * STG, 0);
  };
  auto have = [&](int b) __attribute__((always_inline)) {
    lds_wait();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int j = 0; j < BJ; ++j) pin(fw[b][j][h]);
      pin(fx[b][h]);
    }
  };
  sg_vm_wait<(S - 1) * P>();
  read(0, 0);
  have(0);
  int st = 0;  // stage of tile t
  auto step = [&](int t, int b) __attribute__((always_inline)) {
    stage(t + S, st);  // its reads are done
    st = st + 1 == S ? 0 : st + 1;
    sg_vm_wait<(S - 1) * P>();
    read(b ^ 1, st);  // (behind the last tile: bytes that are not multiplied)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < BJ; ++j) acc[j] = g8_mfma(fw[b][j][h], fx[b][h], acc[j]);
    __builtin_amdgcn_sched_barrier(0);
    have(b ^ 1);
  };
  int t = 0;
  for (; t + 2 <= nk; t += 2) {
    step(t, 0);
    step(t + 1, 1);
  }
  if (t < nk) step(t, 0);
  sg_vm_wait<0>();  // no DMA into LDS outlives the wave
#pragma unroll
  for (int j = 0; j < BJ; ++j) {
    const int n = n0 + 16 * j + 4 * g;
    u16x4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = f2bf(gelu_tanh_t<uint16_t>(bf2f(f2bf(acc[j][r]))) * bf2f(e[j][r]));
    if (row < T && n < N) *reinterpret_cast<u16x4*>(y + (int64_t)row * N + n) = o;
  }
}

}  // namespace mx

using namespace mx;

// y [T, N] (contiguous) = gelu_tanh(x w^T) emb[ids]; -1 (nothing launched) for shapes, strides and addresses that are not taken.
// Two blocks of channels a wave where there are more than four waves of one a CU.
extern "C" int mx_side_gate(const uint16_t* x, int64_t ldx, const uint16_t* w, int64_t ldw, const uint16_t* emb, int64_t lde,
                            const int64_t* ids, int V, uint16_t* y, int T, int N, int K, hipStream_t stream) {
  if (T <= 0 || N <= 0 || N % 16 || K <= 0 || K % 64 || V <= 0 || ldx < K || ldw < K || lde < N || ldx % 8 || ldw % 8 || lde % 4 ||
      ldx >= 1 << 23 || ldw >= 1 << 23 || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) || ((uintptr_t)emb & 7))
    return -1;
  const int64_t rows = ((int64_t)T + 15) / 16, bj = rows * (N / 16) > 1024 ? 2 : 1;
  const int64_t grid = (rows + 7) / 8 * 8 * ((N / 16 + bj - 1) / bj);
  if (grid > INT32_MAX) return -1;
  if (bj == 1) side_gate_kernel<1, 4><<<(unsigned)grid, 64, 0, stream>>>(x, ldx, w, ldw, emb, lde, ids, V, y, T, N, K);
  else side_gate_kernel<2, 3><<<(unsigned)grid, 64, 0, stream>>>(x, ldx, w, ldw, emb, lde, ids, V, y, T, N, K);
  return (int)hipGetLastError();
}
