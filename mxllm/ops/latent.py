"""Latent attention: keys and values are projections of one normed latent per token, which (with a shared
rotated key part) is all the cache holds.

Prompts expand the latent to keys and values; decode steps take the query through W_uk onto the latent
and attend to the cache as it is.  A layer may use another layer's latent (``LatentCache`` is then the
other layer's).

GPU: csrc/kernels/latent_mfma.hip (bf16) and latent.hip.  CPU tensors: plain PyTorch (the CPU test suite).
"""
from __future__ import annotations

from dataclasses import dataclass

import torch

from ._ext import native, use_native
from .linear import linear


@dataclass(frozen=True)
class LatentShape:
    """``dim`` unrotated and ``rot_dim`` rotated query / key dimensions a head (interleaved pairs), values of
    ``vdim``, latents of ``rank``.  ``window`` 0: a query sees all earlier positions, else the last
    ``window`` up to its own."""

    heads: int
    dim: int
    rot_dim: int
    vdim: int
    rank: int
    scale: float
    window: int = 0

    @property
    def q_width(self) -> int:
        return self.heads * (self.dim + self.rot_dim)

    @property
    def row(self) -> int:
        """Width of a cached row: latent and rotated part in whole 32-element steps (the rest is zero)."""
        return (self.rank + self.rot_dim + 31) // 32 * 32


@dataclass
class LatentCache:
    """``pool`` [blocks, 1, block, row] with block table ``bt``, or [slots, 1, ring, row] (``bt`` None);
    position p of a sequence is kept at row p % ``ring``."""

    pool: torch.Tensor
    bt: torch.Tensor | None
    ring: int


def latent_rows(x: torch.Tensor, w: torch.Tensor, eps: float, cos: torch.Tensor, sin: torch.Tensor, sh: LatentShape,
                rows, cache: LatentCache | None) -> torch.Tensor:
    """x [T, rank + rot_dim] projections -> [T, row]: the RMS-normed latent times ``w`` and the rotated key
    part; kept in ``cache``."""
    if use_native(x):
        keep = (cache.pool, cache.bt, cache.ring) if cache is not None else ()
        return native().latent_rows(x, w, eps, cos, sin, sh.rot_dim, rows.rowinfo, sh.row, *keep)
    info = rows.rowinfo.tolist()
    c = x[:, :sh.rank].float()
    c = c * torch.rsqrt(c.pow(2).mean(-1, keepdim=True) + eps) * w
    kr = rotate_pairs(x[:, None, sh.rank:].float(), [r[0] for r in info], cos, sin)[:, 0]
    lat = torch.zeros(x.shape[0], sh.row, dtype=x.dtype)
    lat[:, :sh.rank + sh.rot_dim] = torch.cat([c, kr], 1).to(x.dtype)
    if cache is not None:
        for t, (p, slot, n, _) in enumerate(info):
            if slot >= 0 and p >= n - cache.ring:
                blk, r = cache_place(cache, slot, p)
                cache.pool[blk, 0, r] = lat[t]
    return lat


def latent_attention(q: torch.Tensor, lat: torch.Tensor, wkv: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                     sink: torch.Tensor | None, sh: LatentShape, rows, cache: LatentCache | None) -> torch.Tensor:
    """q [T, heads x (dim | rot_dim)] before rotation, wkv [heads x dim + heads x vdim, rank] -> [T, heads x
    vdim].  Prompt rows attend to ``lat`` (the rows' own latents), tokens to ``cache`` (:func:`latent_step`)."""
    if rows.decode:
        return latent_step(q, None, wkv, None, None, 0.0, cos, sin, sink, sh, rows, cache)
    if not use_native(q):
        return _attention_ref(q, lat, wkv, cos, sin, sink, sh, rows, cache)
    sizes = (sh.heads, sh.dim, sh.rot_dim, sh.vdim, sh.rank, sh.window, sh.scale)
    kv = linear(lat[:, :sh.rank], wkv)
    return native().latent_attn(q, kv, lat, cos, sin, rows.rowinfo, rows.attn_blocks(max(rows.lens)), sink, *sizes)


def latent_step(q: torch.Tensor, x: torch.Tensor | None, wkv: torch.Tensor, wuk_t: torch.Tensor | None,
                w: torch.Tensor | None, eps: float, cos: torch.Tensor, sin: torch.Tensor, sink: torch.Tensor | None,
                sh: LatentShape, rows, cache: LatentCache) -> torch.Tensor:
    """One token per sequence: its latent (projections ``x``, norm ``w``; None: stored already) into the cache,
    its query over the cached rows.  ``wuk_t``: :func:`key_weight` or None."""
    if use_native(q):
        return native().latent_decode(q, wkv, cos, sin, rows.pos, rows.slots, cache.pool, cache.bt, cache.ring, sink,
                                      sh.heads, sh.dim, sh.rot_dim, sh.vdim, sh.rank, sh.window, sh.scale, rows.max_len,
                                      x, w, eps, wuk_t)
    if x is not None:
        latent_rows(x, w, eps, cos, sin, sh, rows, cache)
    return _attention_ref(q, None, wkv, cos, sin, sink, sh, rows, cache)


def key_weight(wkv: torch.Tensor, sh: LatentShape) -> torch.Tensor:
    """[heads, rank, dim]: every head's W_uk transposed, as decode queries go through it."""
    return wkv[:sh.heads * sh.dim].view(sh.heads, sh.dim, sh.rank).transpose(1, 2).contiguous()


# ------------------------------------------------------------------ CPU
def rotate_pairs(x: torch.Tensor, pos: list[int], cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """x [T, heads, R] by interleaved pairs."""
    c, s = cos[pos][:, None], sin[pos][:, None]
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)


def cache_place(cache: LatentCache, slot: int, p: int) -> tuple[int, int]:
    r, blk = p % cache.ring, cache.pool.shape[2]
    return (slot, r) if cache.bt is None else (int(cache.bt[slot, r // blk]), r % blk)


def _attention_ref(q, lat, wkv, cos, sin, sink, sh: LatentShape, rows, cache):
    H, D, R, E = sh.heads, sh.dim, sh.rot_dim, sh.vdim
    info = rows.rowinfo.tolist()
    q = q.float().view(-1, H, D + R)
    q = torch.cat([q[..., :D], rotate_pairs(q[..., D:], [r[0] for r in info], cos, sin)], -1)
    out = torch.empty(q.shape[0], H * E)
    for t, (p, slot, _, _) in enumerate(info):
        n = min(p + 1, sh.window) if sh.window else p + 1
        if rows.decode:
            at = [cache_place(cache, slot, j) for j in range(p + 1 - n, p + 1)]
            rl = torch.stack([cache.pool[b, 0, r] for b, r in at]).float()
        else:
            rl = lat[t + 1 - n:t + 1].float()
        kv = rl[:, :sh.rank] @ wkv.float().t()
        kr = rl[:, None, sh.rank:sh.rank + R].expand(n, H, R)
        s = (torch.cat([kv[:, :H * D].view(n, H, D), kr], -1) * q[t]).sum(-1) * sh.scale  # [n, H]
        m = s.amax(0) if sink is None else torch.maximum(s.amax(0), sink)
        e = torch.exp(s - m)
        den = e.sum(0) + (0 if sink is None else torch.exp(sink - m))
        out[t] = ((e / den)[..., None] * kv[:, H * D:].view(n, H, E)).sum(0).reshape(-1)
    return out.to(lat.dtype if lat is not None else wkv.dtype)
