// Arguments of the kernels of latent attention, retention, expert mixtures and post-normed
// sublayers (postnorm.hip, latent.hip, latent_mfma.hip, retention.hip, retention_chunk.hip, moe.hip, moe_mfma.hip), shared with the op
// bindings.  Activations are bf16 or f32 (the f32 flag of each entry point); norms, tables, state and the
// residual stream are f32.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mx {

// h (+)= rms(src) * w, and the activation copy y of the new h
struct PostNorm {
  enum { kRows, kEmbed, kMix };
  int mode;
  const void* src;       // kRows [T, W]; kEmbed the table [V, W]; kMix expert outputs [T top, W]
  int64_t lds;
  const int64_t* ids;    // kEmbed: table row of each token
  int V;
  const int32_t* inv;    // kMix: [T, top] row of src of each choice (nullptr: t top + k)
  const float* wts;      // kMix: [T, top]
  int top;
  const void* shared;    // kMix: [T, W] added, or nullptr
  int64_t ldsh;
  float* h;              // [T, W]; kEmbed writes it, the others add
  const float* w;        // [W]
  void* y;               // [T, W] or nullptr
  float eps;
  int64_t T;
  int W;
};

// decode rows: the residual step, and dot products of the new h's bf16 copy with rows of a matrix
struct PostDots {
  PostNorm p;            // kRows or kMix (rows in pair order); y may be nullptr
  float* ho;             // [T, W]: the new h (p.h is only read)
  const uint16_t* m;     // [R, W]
  int R;
  float* logits;         // [T, R], or:
  uint16_t* side;        // [T, R]: gelu_tanh(dot) times columns of the tokens' rows of emb
  const uint16_t* emb;
  int64_t lde;
  const int64_t* ids;
  int V;
};

// prompt rows: the residual step behind the mixer and the router's choices on the new rows
struct PostRoute {
  PostNorm p;            // kRows; y: the copy
  const uint16_t* m;     // [E, W]
  int E, top;
  int32_t* ids;          // [T, top]
  float* wts;
};

// the shared latent and rotated key part of latent attention: rows = (position, slot or -1, sequence length, -)
struct LatentRows {
  const void* x;         // [T, rank + rot] projections
  int64_t ldx;
  const float* w;        // [rank]
  const float *cosb, *sinb;  // [positions, rot / 2]
  const int32_t* rows;
  int T, rank, rot;
  float eps;
  void* lat;             // [T, ldl]: latent | rotated part | zeros, or nullptr
  int64_t ldl;
  void* pool;            // cache [blocks (or slots), seq, wc], nullptr: none
  const int32_t* bt;     // nullptr: pool rows by slot
  int maxb, seq, ring, wc;  // position p is kept at row p % ring
  int vec;               // set by the launch
};

// attention of prompt rows on expanded keys and values
struct LatentAttn {
  const void* q;         // [T, H (D + R)] unrotated
  int64_t ldq;
  const void* kv;        // [T, H D + H E]
  int64_t ldkv;
  const void* lat;       // rotated key part at column rank
  int64_t ldl;
  const float *cosb, *sinb;
  const int32_t* rows;   // generic kernel: (position, -, -, -) of each row
  const int32_t* blocks; // MFMA kernel: (first row of the sequence, its rows, query block, -)
  int nblocks;
  const float* sink;     // [H] or nullptr
  void* out;             // [T, H E]
  int T, H, D, R, E, rank, window;  // window 0: all earlier keys
  float scale;
};

// one query per sequence against the cached latent
struct LatentDecode {
  const void* q;         // [B, H (D + R)] unrotated
  int64_t ldq;
  const void* wuk;       // [H D, rank]
  const void* wuk_t;     // [H, rank, D] (latent_heads) or nullptr
  const void* wuv;       // [H E, rank]
  const float *cosb, *sinb;
  const int32_t *pos, *slots;
  const void* pool;
  const int32_t* bt;
  int maxb, seq, ring, wc;
  const float* sink;
  void* qa;              // [B, H, wq]: latent query | rotated part | zeros
  int wq;
  float* ml;             // [B, H, nsplit, 2] running maximum (log2 units) and sum
  float* po;             // [B, H, nsplit, rank] unnormalised
  int nsplit, span;      // keys of a split
  void* om;              // [B, H, rank]: merged latents (latent_merge)
  void* out;             // [B, H E]
  int B, H, D, R, E, rank, window;
  float scale;
};

struct Retention {
  const void* x;         // [T, ldx]: q | k | v | gate projections
  int64_t ldx;
  const float *cosb, *sinb;  // [positions, rd / 2]
  const float* decay;    // [H], stride ldd
  int64_t ldd;
  const int32_t* seqs;   // prompts [n, 4]: (first row, rows, slot or -1, -); nullptr: one token a row
  int nseq;
  const int32_t *pos, *slots;  // tokens
  float* state;          // [slots, H, D, E] or nullptr
  void* y;               // [T, H E]
  int T, H, D, E, rd;
  float eps;
};

// prompts in runs of up to 256 rows of one sequence
struct RetentionChunks {
  const void* x;         // [T, ldx]: q | k | v | gate projections
  int64_t ldx;
  const float *cosb, *sinb;  // [positions, rd / 2]
  const float* pw;       // [H, 257]: powers of the decays
  const int32_t* chunks; // [nchunks, 4]: (first row, rows, position of the first, -)
  const int32_t* seqs;   // [nseq, 4]: (first run, runs, slot or -1, -)
  const int32_t* blocks; // [nblocks, 4]: (run, first row in it, -, -), 128 rows each
  int nchunks, nseq, nblocks;
  int carry;             // 0: no run has one ahead and no state is kept
  float* ws;             // [nchunks, H, D, E]
  float* state;          // [slots, H, D, E] or nullptr
  void* y;               // [T, H E]
  int H, D, E, rd;
  float eps;
  int v4;                // set by the launch
};

// the experts of a mixture applied to rows sorted by expert
struct MoeGemm {
  const void* x;         // [*, K]
  int64_t ldx;
  const int32_t* src;    // row of x of each sorted row (nullptr: the row itself)
  const int32_t* tiles;  // [ntiles, 4]: (expert, first sorted row, rows, tiles in use), the unused ones last with rows 0
  int ntiles;
  const void* w;         // [experts, N, K], GLU: [experts, 2 N, K] (gate rows, then up rows)
  void* y;               // [rows, N]
  int N, K, glu;
  float limit;
};

// the same for up to 64 tokens: pairs (token, choice) in order, the shared expert (sw) beside them
struct MoeFew {
  const uint16_t* x;     // up: [T, K] tokens; down: [T top, K] pairs
  int64_t ldx;
  const int32_t* ids;    // [T, top]
  const uint16_t* w;     // up: [E, gate | up, K]; down: [E, N, K]
  uint16_t* y;           // [T top, N]
  const uint16_t* sw;    // shared expert's weights, or nullptr
  const uint16_t* sx;    // down: [T, sK] (up reads x)
  uint16_t* sy;          // [T, sN]
  int T, top, E, N, K, sN, sK;
  float limit, slimit;
  const float* logits;   // up: [T, E] or nullptr (then ids are given)
  int32_t* ids_out;      // [T, top], with logits
  float* wts_out;
};

}  // namespace mx
