"""Ops of decoders that mix recurrent and chunked-attention layers: grouped RMS norm on an f32
residual, the minGRU recurrence, convolved + pair-rotated attention with a softmax sink and an
output gate, PolyNorm; and the row layouts they run on.

``PromptRows``: the concatenated tokens of several sequences from their first token on.
``TokenRows``: one token for each of several sequences (a decode step, graph-capturable).
Both carry where a layer's cached rows and state live (``SeqCaches``), so a model's layer loop is
the same for both.

GPU: csrc/kernels/hybrid.hip, mingru.hip, chunk_attn.hip, attn_fwd.hip (SEG) and decode.hip.
CPU tensors: plain PyTorch (the CPU test suite).
"""
from __future__ import annotations

import os
from dataclasses import dataclass

import numpy as np
import torch

from ._ext import native, use_native
from .linear import NORM_M, SKINNY_M, _DECODE_M, _NORM_STREAM_M, _SKINNY_SMALL_W, _near

MFMA_MAX_DIM = 128  # widest head of the MFMA attention kernels
MFMA_MAX_REP = 16   # query heads per key head in the split-K decode kernels


@dataclass(frozen=True)
class AttnShape:
    """One attention layer's constants.  ``chunk``: position i sees only keys of its own run of
    ``chunk`` positions; ``rot_dims`` of ``dim`` are rotated (interleaved pairs)."""

    heads: int
    kv_heads: int
    dim: int
    vdim: int
    taps: int
    chunk: int
    rot_dims: int
    scale: float

    @property
    def conv_channels(self) -> int:
        return (self.heads + self.kv_heads) * self.dim + self.kv_heads * self.vdim

    def mfma(self, dtype: torch.dtype) -> bool:
        """bf16 heads the matrix-core attention kernels take; the rest runs on chunk_attn.hip."""
        return (dtype == torch.bfloat16 and max(self.dim, self.vdim) <= MFMA_MAX_DIM
                and self.heads // self.kv_heads <= MFMA_MAX_REP)

    def row_dims(self, dtype: torch.dtype) -> tuple[int, int]:
        """Stored width of a key and of a value row: the MFMA kernels take one width of 32, 64 or
        128 for both (unused dims zero), the others whole 16-byte pieces."""
        if self.mfma(dtype):
            w = next(x for x in (32, 64, 128) if x >= max(self.dim, self.vdim))
            return w, w
        a = 16 // dtype.itemsize
        return (self.dim + a - 1) // a * a, (self.vdim + a - 1) // a * a


@dataclass
class SeqCaches:
    """What sequences keep between steps.  ``k`` / ``v``: per attention layer, paged pools
    [blocks, kv_heads, block, width]; a layer keeps position p at row p % chunk, so a slot's
    blocks cover at most one chunk.  ``conv``: per attention layer [slots, taps, channels], the
    projected values of position p at p % taps.  ``rec``: per recurrent layer f32 [slots, width]."""

    k: list
    v: list
    bt: torch.Tensor
    conv: list
    rec: list
    latent: dict | None = None  # layer -> its latents (mxllm/ops/latent.py LatentCache)


def pair_rope_tables(n: int, dims: int, base: float, device=None) -> tuple[torch.Tensor, torch.Tensor]:
    """cos / sin f32 [n, dims / 2] of position * base^(-2i / dims) (angles in f64, rounded once)."""
    i = torch.arange(dims // 2, dtype=torch.float64, device=device)
    f = torch.pow(torch.tensor(float(base), dtype=torch.float64, device=device), -2.0 * i / max(dims, 1))
    a = torch.arange(n, dtype=torch.float64, device=device)[:, None] * f[None]
    return a.cos().float().contiguous(), a.sin().float().contiguous()


class RopeTables:
    """A model's rotation tables by (dims, base), shared by layers alike."""

    def __init__(self, device):
        self.device = device
        self._have: dict = {}
        self._kept: list = []

    def get(self, dims: int, base: float, n: int) -> tuple[torch.Tensor, torch.Tensor]:
        """Tables of at least ``n`` positions."""
        key = (dims, base)
        have = self._have.get(key)
        if have is None or have[0].shape[0] < n:
            self._kept.append(have)  # captured decode graphs may still read the shorter tables
            have = self._have[key] = pair_rope_tables(max(n, 256), *key, device=self.device)
        return have


# ------------------------------------------------------------------ row layouts
class PromptRows:
    """Rows of several prompts, each from position 0; ``slots`` None: nothing is kept."""

    decode = False

    def __init__(self, lens: list[int], device, slots: list[int] | None = None, caches: SeqCaches | None = None):
        self.lens, self.device, self.caches = list(lens), device, caches if slots is not None else None
        self.slots = list(slots) if slots is not None else [-1] * len(lens)
        self.offs = np.concatenate([[0], np.cumsum(self.lens)]).astype(np.int64)
        self.T = int(self.offs[-1])
        self._tables: dict = {}
        # every row's (position, slot, sequence length, -)
        info = np.zeros((self.T, 4), dtype=np.int32)
        info[:, 0] = np.concatenate([np.arange(n) for n in self.lens])
        info[:, 1] = np.repeat(self.slots, self.lens)
        info[:, 2] = np.repeat(self.lens, self.lens)
        self.rowinfo = self._up(info)

    def _up(self, a: np.ndarray) -> torch.Tensor:
        return torch.from_numpy(np.ascontiguousarray(a)).to(self.device)

    def attn_blocks(self, chunk: int) -> torch.Tensor:
        """int32 [n, 4] query blocks of 128 rows of every (sequence, chunk) segment, longest first."""
        key = ("attn", chunk)
        if key not in self._tables:
            rows = []
            for o, n in zip(self.offs, self.lens):
                for s in range(0, n, chunk):
                    m = min(chunk, n - s)
                    rows += [(int(o) + s, m, qb, 0) for qb in range((m + 127) // 128)]
            rows.sort(key=lambda r: -r[2])
            self._tables[key] = self._up(np.array(rows, dtype=np.int32))
        return self._tables[key]

    def seqs(self) -> torch.Tensor:
        """int32 [n, 4] (first row, rows, slot or -1, -) of every sequence."""
        if "seqs" not in self._tables:
            self._tables["seqs"] = self._up(np.array([(int(o), n, s, 0) for o, n, s in
                                                      zip(self.offs, self.lens, self.slots)], dtype=np.int32))
        return self._tables["seqs"]

    def run_tables(self, n: int):
        """Runs of at most ``n`` rows of one sequence: (runs int32 [r, 4] = first row, rows, position of the
        first, -; sequences [s, 4] = first run, runs, slot or -1, -; blocks of 128 rows [b, 4] = run, first row
        in it, -, - ; whether any sequence has several runs)."""
        key = ("runs", n)
        if key not in self._tables:
            runs, seqs, blocks = [], [], []
            for o, m, s in zip(self.offs, self.lens, self.slots):
                seqs.append((len(runs), (m + n - 1) // n, s, 0))
                for p in range(0, m, n):
                    k = min(n, m - p)
                    blocks += [(len(runs), i, 0, 0) for i in range(0, k, 128)]
                    runs.append((int(o) + p, k, p, 0))
            blocks.sort(key=lambda b: -b[1])  # the longest look-back first
            self._tables[key] = (*(self._up(np.array(t, dtype=np.int32)) for t in (runs, seqs, blocks)),
                                 any(s[1] > 1 for s in seqs))
        return self._tables[key]

    def scan_tables(self, width: int):
        """(chunks int32 [n, 4] = first row, rows, sequence, last-of-sequence; seqs int32 [m, 3] =
        slot, first chunk, chunks; whether any sequence has several) for a scan of ``width`` channels:
        chunks short enough to fill the GPU with waves."""
        L = max(16, min(128, self.T * width // (256 * 2048)))
        L = 1 << (L.bit_length() - 1)
        key = ("scan", L)
        if key not in self._tables:
            ch, sq = [], []
            for i, (o, n) in enumerate(zip(self.offs, self.lens)):
                c0 = len(ch)
                for s in range(0, n, L):
                    ch.append((int(o) + s, min(L, n - s), i, int(s + L >= n)))
                sq.append((self.slots[i], c0, len(ch) - c0))
            self._tables[key] = (self._up(np.array(ch, dtype=np.int32)), self._up(np.array(sq, dtype=np.int32)),
                                 any(s[2] > 1 for s in sq))
        return self._tables[key]


class TokenRows:
    """One token per sequence: ``pos`` / ``slots`` int32 [B] on the device, ``max_len`` a host bound
    on the keys a step looks back over (pos + 1, or the longest chunk)."""

    decode = True

    def __init__(self, pos: torch.Tensor, slots: torch.Tensor, max_len: int, caches: SeqCaches):
        self.pos, self.slots, self.max_len, self.caches = pos, slots, max_len, caches
        self._local: dict = {}

    @property
    def rowinfo(self) -> torch.Tensor:
        """Every row's (position, slot, sequence length, -), as ``PromptRows`` has it."""
        if "info" not in self._local:
            self._local["info"] = torch.stack([self.pos, self.slots, self.pos + 1, self.pos], 1).contiguous()
        return self._local["info"]

    def chunk_pos(self, chunk: int) -> torch.Tensor:
        """Position inside the chunk = index of the newest cached row."""
        if chunk not in self._local:
            self._local[chunk] = torch.remainder(self.pos, chunk)
        return self._local[chunk]


# ------------------------------------------------------------------ ops
def embed_rows(ids: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """Token rows of the embedding table as the f32 residual stream."""
    if use_native(w):
        return native().embed_rows(ids.contiguous(), w)
    return w[ids].float()


def group_norm(delta: torch.Tensor | None, h: torch.Tensor, w: torch.Tensor, groups: int, eps: float,
               dtype: torch.dtype) -> torch.Tensor:
    """h (f32, in place) += delta; returns the RMS norm of h in ``groups`` equal parts, times w.  ``delta`` f32 [S, T, W]:
    the sums of S segments of a projection (``linear_parts``), added and rounded to bf16 first."""
    if use_native(h):
        if delta is not None and delta.dim() == 3:
            return native().group_norm_parts(delta, h, w, groups, eps)
        return native().group_norm(delta, h, w, groups, eps, dtype == torch.float32)
    if delta is not None:
        h += delta.float()
    p = h.view(h.shape[0], groups, -1)
    return ((p * torch.rsqrt(p.pow(2).mean(-1, keepdim=True) + eps)).view_as(h) * w).to(dtype)


def poly_norm(z: torch.Tensor, coef: torch.Tensor, eps: float) -> torch.Tensor:
    """a N(z) + b N(z^2) + c N(z^3) + e with N the RMS norm over the row; coef = (a, b, c, e)."""
    if use_native(z):
        return native().poly_norm(z, coef, eps)
    x = z.float()
    y = coef[3]
    for i in range(3):
        p = x ** (i + 1)
        y = y + coef[i] * p * torch.rsqrt(p.pow(2).mean(-1, keepdim=True) + eps)
    return y.to(z.dtype)


def min_gru(x: torch.Tensor, bias: torch.Tensor, rows, layer: int) -> torch.Tensor:
    """Gated recurrence over the rows of ``rows``: x [T, 3W] = z | u | g projections, bias f32 [2W]
    (z | u); recurrent layer ``layer``'s state is read and written in ``rows.caches``."""
    W = x.shape[1] // 3
    state = rows.caches.rec[layer] if rows.caches is not None else None
    if use_native(x):
        if rows.decode:
            return native().mingru_step(x, bias, rows.slots, state)
        chunks, seqs, multi = rows.scan_tables(W)
        return native().mingru_scan(x, bias, chunks, seqs, multi, state)
    z, u, g = x.float().split(W, 1)
    z = torch.sigmoid(z + bias[:W])
    u = u + bias[W:]
    add, keep = z * torch.where(u >= 0, u + 0.5, torch.sigmoid(u)), 1 - z
    s = torch.empty_like(z)
    if rows.decode:
        idx = rows.slots.long()
        s = keep * state[idx] + add
        state[idx] = s
    else:
        for i, n in enumerate(rows.lens):
            cur = torch.zeros(W)
            for t in range(int(rows.offs[i]), int(rows.offs[i]) + n):
                cur = keep[t] * cur + add[t]
                s[t] = cur
            if state is not None:
                state[rows.slots[i]] = cur
    return (s * torch.nn.functional.silu(g)).to(x.dtype)


def sink_attention(x: torch.Tensor, conv: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, sh: AttnShape, rows,
                   layer: int) -> torch.Tensor:
    """x [T, q | k | v | gate] projections -> gated attention output [T, heads * vdim]: causal
    convolution of q, k, v over time, rotation of q and k, attention inside chunks with one added to
    the softmax's denominator, times sigmoid(gate).  ``conv`` f32 [taps, channels]."""
    C = sh.conv_channels
    gate = x[:, C:]
    H, G, D, E = sh.heads, sh.kv_heads, sh.dim, sh.vdim
    c = rows.caches
    if not use_native(x):
        return _sink_attention_ref(x, conv, cos, sin, sh, rows, layer)
    ops = native()
    Dp, Ep = sh.row_dims(x.dtype)
    args = (x, conv, cos, sin, sh.rot_dims, H, G, D, E)
    if not rows.decode:
        keep = (c.k[layer], c.v[layer], c.bt, c.conv[layer]) if c is not None else ()
        q, k, v = ops.conv_rope_prefill(*args, Dp, Ep, rows.rowinfo, sh.chunk, *keep)
        if sh.mfma(x.dtype):
            return ops.attn_seg(q, k, v, rows.attn_blocks(sh.chunk), gate, E, sh.scale)
        return ops.chunk_attn(q, k, v, rows.rowinfo[:, 0].contiguous(), gate, D, E, sh.chunk, sh.scale)
    q = ops.conv_rope_decode(*args, rows.pos, rows.slots, sh.chunk, c.k[layer], c.v[layer], c.bt, c.conv[layer])
    return decode_sink_attention(q, gate, sh, rows, layer)


def decode_sink_attention(q: torch.Tensor, gate: torch.Tensor, sh: AttnShape, rows: TokenRows,
                          layer: int) -> torch.Tensor:
    """One query per sequence over the cached rows of its chunk (the new token's already stored)."""
    ops, c = native(), rows.caches
    if sh.mfma(q.dtype):
        ml, po = ops.decode_attn_partials(q, c.k[layer], c.v[layer], rows.chunk_pos(sh.chunk), rows.slots,
                                          min(rows.max_len, sh.chunk), sh.scale, 1, c.bt)
        return ops.attn_combine(ml, po, gate, sh.vdim)
    return ops.chunk_attn(q, c.k[layer], c.v[layer], rows.pos, gate, sh.dim, sh.vdim, sh.chunk, sh.scale, rows.slots,
                          c.bt)


# ------------------------------------------------------------------ fused decode steps
# csrc/kernels/hybrid_skinny.hip: the projections of up to SKINNY_M decode rows with the work after them
# in the GEMM's epilogue, and for up to NORM_M rows the norm or activation ahead of them in its
# prologue.  Each returns None where the kernel does not take the call (the caller runs the parts).
# MXLLM_HYBRID_FUSED=0: always the parts (A/B).
FUSED = os.environ.get("MXLLM_HYBRID_FUSED", "1") != "0"
_NORM_MAX, _POLY_MAX = 16384, 32768  # rows x width held in LDS by a prologue


def _fusable(t: torch.Tensor, w: torch.Tensor | None, mult: int = 16, rows: int | None = None) -> bool:
    """``rows``: the most that the kernel is for (SKINNY_M)."""
    M, K = t.shape
    rows = SKINNY_M if rows is None else rows
    return bool(FUSED and w is not None and use_native(t) and w.dtype == torch.bfloat16 and 0 < M <= min(rows, 16)
                and K % 512 == 0 and w.shape[0] % mult == 0 and w.stride(1) == 1 and w.stride(0) % 8 == 0
                and (M == 1 or w.numel() <= _SKINNY_SMALL_W))


def _norm_fits(h: torch.Tensor, groups: int) -> bool:
    M, K = h.shape
    return M <= NORM_M and M * K <= _NORM_MAX and (K // groups) % 8 == 0 and M * groups <= 512


def norm_linear(delta, h, gamma, groups: int, eps: float, w):
    """(group_norm(h + delta) w^T, h + delta) in one launch.  csrc/kernels/stream_gemm.hip where it has the sizes: a part of the norm
    to each of 8 waves, rows of 512 threads x 4 or 8 elements, up to 4 rows; from 6144 channels, those of the up projections it
    was measured for (us, norm and product apart -> here, 1 / 4 rows: 6144 x 2048 9.8 / 10.7 -> 7.9 / 9.6; 6144 x 4096 15.6 / 16.0 ->
    14.0 / 17.0, 8192 x 4096 16.8 / 17.3 -> 15.4 / 17.5; fewer would gain as well, 2048 x 2048 6.3 / 6.6 -> 4.9 / 6.1)."""
    if not _fusable(h, w):
        return None
    if w.shape[0] >= 6144 and _norm_stays(delta, h, gamma, groups, w):
        return native().stream_group_norm(delta, h, gamma, eps, w)
    if not _norm_fits(h, groups):
        return None
    return native().hs_norm_linear(delta, h, gamma, groups, eps, w)


def poly_linear(z, coef, eps: float, w):
    """poly_norm(z) w^T in one launch: one row and 4096 channels (us, the norm apart -> here: 4096 x 21504 34.5 -> 33.7, x 12288
    22.1 -> 21.6).  Every 16 channels do the norm again, and fewer channels' product by itself takes 8 a workgroup: 2048 x 12288,
    1 / 2 rows 14.7 / 15.2 -> 16.9 / 19.3; 4096 x 12288, 2 rows 22.2 -> 24.2."""
    if not (_fusable(z, w) and z.shape[0] <= min(NORM_M, 1) and z.numel() <= _POLY_MAX and w.shape[0] >= 4096):
        return None
    return native().hs_poly_linear(z, coef, eps, w)


def _norm_stays(delta, h, gamma, groups: int, w) -> bool:
    """Whether the workgroups that stay do the norm: 8 parts, one to each of their waves, rows of 512 threads x 4 or 8 elements, up to 4
    rows (csrc/kernels/stream_groups.h)."""
    return bool(h.shape[0] <= min(4, _NORM_STREAM_M) and groups == 8 and h.shape[1] in (2048, 4096) and _near(w)
                and all(t.data_ptr() % 16 == 0 for t in (h, gamma, w))
                and (delta is None or (delta.dim() == 2 and delta.stride(0) % 8 == 0 and delta.data_ptr() % 16 == 0)))


def _mixer_rows(h: torch.Tensor, width: int = 0) -> int:
    """Rows up to which a mixer's projection runs with its epilogue: past SKINNY_M for a width of 2048 (csrc/kernels/stream_hybrid.hip;
    steps of 9 / 12 / 16 sequences of the 1B size 998 / 1034 / 1057 us apart, 959 / 995 / 1021 so; of 4096, 8B size, 3945 / 4088 /
    4181 apart, 3960 / 4117 / 4214).  A minGRU's up to a state of 2048 (``width``; norm and projection, 9 / 16 rows: 2048 14.0 / 14.7 ->
    12.3 / 12.8, 2560 14.1 / 14.9 -> 14.9 / 15.7, 4096 16.8 / 18.0 -> 17.6 / 18.6); the convolution's at any size (640 / 768 / 1024 groups of
    channels, 16 rows: 26.5 / 27.3 / 32.7 -> 24.4 / 25.2 / 31.6)."""
    return _DECODE_M if h.shape[1] == 2048 and width <= 2048 else SKINNY_M


def _normed(delta, h, gamma, groups, eps, w):
    """(delta, x, gamma) of a fused projection: the norm in its prologue, or run ahead of it (a delta in parts is added there)."""
    if (_norm_stays(delta, h, gamma, groups, w) or _norm_fits(h, groups)) and (delta is None or delta.dim() == 2):
        return delta, h, gamma
    return None, group_norm(delta, h, gamma, groups, eps, torch.bfloat16), None


def gru_linear(delta, h, gamma, groups: int, eps: float, w, bias, rows, layer: int):
    """Decode: (minGRU output of the normed rows, new residual), state advanced; w = [z; u; gate]."""
    if not (rows.decode and _fusable(h, w, 12, _mixer_rows(h, bias.numel() // 2))):
        return None
    d, x, g = _normed(delta, h, gamma, groups, eps, w)
    y, hn = native().hs_gru_linear(d, x, g, groups, eps, w, bias, rows.slots, rows.caches.rec[layer])
    return y, (hn if g is not None else h)


def conv_linear(delta, h, gamma, groups: int, eps: float, w, conv, cos, sin, sh: AttnShape, rows, layer: int):
    """Decode: (gated attention output of the normed rows, new residual); w = [q; k; v; gate]."""
    if not (rows.decode and _fusable(h, w, 16, _mixer_rows(h)) and sh.dim % 4 == 0 and sh.vdim % 4 == 0):
        return None
    d, x, g = _normed(delta, h, gamma, groups, eps, w)
    c = rows.caches
    q, gate, hn = native().hs_conv_linear(d, x, g, groups, eps, w, conv, cos, sin, sh.rot_dims, sh.heads, sh.kv_heads,
                                          sh.dim, sh.vdim, rows.pos, rows.slots, sh.chunk, c.k[layer], c.v[layer],
                                          c.bt, c.conv[layer])
    return decode_sink_attention(q, gate, sh, rows, layer), (hn if g is not None else h)


# ------------------------------------------------------------------ CPU attention
def _sink_attention_ref(x, conv, cos, sin, sh: AttnShape, rows, layer: int) -> torch.Tensor:
    H, G, D, E, C, n = sh.heads, sh.kv_heads, sh.dim, sh.vdim, sh.conv_channels, sh.taps
    c = rows.caches
    bt = c.bt.tolist() if c is not None else None

    def place(slot, p):  # cache block and row of position p
        r = p % sh.chunk
        blk = c.k[layer].shape[2]
        return bt[slot][r // blk], r % blk

    def rot(t, p):  # [heads, D] at position p
        t = t.clone()
        k = sh.rot_dims
        a, b = t[:, 0:k:2].clone(), t[:, 1:k:2].clone()
        t[:, 0:k:2], t[:, 1:k:2] = a * cos[p] - b * sin[p], b * cos[p] + a * sin[p]
        return t

    def attend(q, ks, vs):  # q [H, D], ks [L, G, D], vs [L, G, E]
        ks, vs = ks.repeat_interleave(H // G, 1), vs.repeat_interleave(H // G, 1)
        s = torch.matmul(ks.transpose(0, 1), q[:, :, None])[..., 0] * sh.scale  # [H, L]
        m = s.amax(1, keepdim=True).clamp_min(0)
        e = torch.exp(s - m)
        w = e / (e.sum(1, keepdim=True) + torch.exp(-m))
        return torch.matmul(w[:, None], vs.transpose(0, 1))[:, 0].reshape(-1)

    def token(u, hist, p):  # newest value u [C], hist: earlier ones newest first
        y = conv[n - 1] * u
        for back, o in enumerate(hist[:n - 1], 1):
            y = y + conv[n - 1 - back] * o
        return (rot(y[:H * D].view(H, D), p).to(x.dtype).float(), rot(y[H * D:(H + G) * D].view(G, D), p),
                y[(H + G) * D:].view(G, E))

    out = torch.empty(x.shape[0], H * E)
    u = x[:, :C].float()
    if rows.decode:
        for b, (p, s) in enumerate(zip(rows.pos.tolist(), rows.slots.tolist())):
            hist = [c.conv[layer][s, (p - j) % n].float() for j in range(1, n) if p >= j]
            q, k, v = token(u[b], hist, p)
            c.conv[layer][s, p % n] = x[b, :C]
            blk, r = place(s, p)
            c.k[layer][blk, :, r, :D], c.v[layer][blk, :, r, :E] = k.to(x.dtype), v.to(x.dtype)
            at = [place(s, j) for j in range(p // sh.chunk * sh.chunk, p + 1)]
            out[b] = attend(q, torch.stack([c.k[layer][i, :, j, :D] for i, j in at]).float(),
                            torch.stack([c.v[layer][i, :, j, :E] for i, j in at]).float())
    else:
        for i, L in enumerate(rows.lens):
            o, s = int(rows.offs[i]), rows.slots[i]
            ks, vs = [], []
            for p in range(L):
                q, k, v = token(u[o + p], [u[o + p - j] for j in range(1, n) if p >= j], p)
                ks.append(k.to(x.dtype).float())
                vs.append(v.to(x.dtype).float())
                lo = p // sh.chunk * sh.chunk
                out[o + p] = attend(q, torch.stack(ks[lo:]), torch.stack(vs[lo:]))
                if c is not None:
                    if p >= L - n:
                        c.conv[layer][s, p % n] = x[o + p, :C]
                    if p >= L // sh.chunk * sh.chunk:
                        blk, r = place(s, p)
                        c.k[layer][blk, :, r, :D], c.v[layer][blk, :, r, :E] = k.to(x.dtype), v.to(x.dtype)
    return (out * torch.sigmoid(x[:, C:].float())).to(x.dtype)
