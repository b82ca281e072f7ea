"""Mixture of experts: routing, grouping of (token, choice) pairs by expert, and the experts' gated
feed-forwards on grouped rows.  Nothing of it needs the host, so it is graph-capturable.

GPU: csrc/kernels/moe_mfma.hip (bf16) and moe.hip.  CPU tensors: plain PyTorch (the CPU test suite).
"""
from __future__ import annotations

import torch

from . import sublayer
from ._ext import native, use_native
from .linear import linear, linear_clipped
from .sublayer import clipped_glu

GENERIC_ROWS = 64  # row tile of the products of any size
MFMA_ROWS = 256    # and of the matrix-core ones
FEW_TOKENS, FEW_PAIRS = 64, 1024  # what the decode kernel takes


def route(x: torch.Tensor, router: torch.Tensor, top: int) -> tuple[torch.Tensor, torch.Tensor]:
    """(experts int32 [T, top], weights f32 [T, top]): the largest router logits (computed in f32) and the
    softmax over them alone."""
    if use_native(x):
        return native().moe_route(x, router, top)
    val, idx = torch.topk(x.float() @ router.float().t(), top, dim=-1)
    return idx.int(), torch.softmax(val, -1)


def experts(x: torch.Tensor, ids: torch.Tensor, wgu: torch.Tensor, wdown: torch.Tensor, limit: float,
            sgu: torch.Tensor | None = None, sdown: torch.Tensor | None = None, slimit: float = 0.0):
    """(rows [T * top, W] of the chosen experts' outputs, the row of each (token, choice) pair or None where
    they are in that order, the shared expert's rows [T, W] or None).  wgu [E, gate | up, W], wdown
    [E, W, ff]; the shared expert sgu [gate | up, W], sdown [W, ff']."""
    if use_native(x) and few(x, ids.shape[1], wgu, sgu):
        y, _, sh = _run_few(x, ids, None, ids.shape[1], wgu, wdown, limit, sgu, sdown, slimit)
        return y, None, sh
    sh = None
    if sgu is not None:
        mid = linear_clipped(x, sgu, slimit) if sublayer.FUSED else None
        sh = linear(clipped_glu(linear(x, sgu), slimit) if mid is None else mid, sdown)
    if use_native(x):
        bm = MFMA_ROWS if _grouped(x, wgu) else GENERIC_ROWS
        src, inv, tiles = native().moe_group(ids, wgu.shape[0], bm)
        mid = native().moe_gemm(x, src, tiles, wgu, ids.numel(), True, limit, bm)
        return native().moe_gemm(mid, None, tiles, wdown, ids.numel(), False, 0.0, bm), inv, sh
    flat = ids.view(-1).long()
    out = torch.empty(flat.numel(), wdown.shape[1], dtype=x.dtype)
    rows = torch.arange(x.shape[0]).repeat_interleave(ids.shape[1])
    for e in flat.unique().tolist():
        at = (flat == e).nonzero()[:, 0]
        z = (x[rows[at]].float() @ wgu[e].float().t()).to(x.dtype)
        out[at] = (clipped_glu(z, limit).float() @ wdown[e].float().t()).to(x.dtype)
    return out, None, sh


def experts_of(x: torch.Tensor, logits: torch.Tensor, top: int, wgu: torch.Tensor, wdown: torch.Tensor, limit: float,
               sgu: torch.Tensor | None = None, sdown: torch.Tensor | None = None, slimit: float = 0.0):
    """:func:`experts` of the ``top`` largest router ``logits`` (f32 [T, E <= 64]), chosen in the same launch, where
    :func:`few` holds: (rows in pair order, weights, the shared expert's rows or None)."""
    return _run_few(x, None, logits, top, wgu, wdown, limit, sgu, sdown, slimit)


def _run_few(x, ids, logits, top, wgu, wdown, limit, sgu, sdown, slimit):
    ops = native()
    mid, smid, ids, wts = ops.moe_few(x, ids, logits, top, wgu, True, limit, sgu, None, slimit)
    y, sh, _, _ = ops.moe_few(mid, ids, None, top, wdown, False, 0.0, sdown, smid if sgu is not None else None, 0.0)
    return y, wts, sh if sgu is not None else None


def few(x: torch.Tensor, top: int, wgu: torch.Tensor, sgu: torch.Tensor | None) -> bool:
    """Decode steps: the kernel that streams each chosen expert's weights past its rows."""
    T = x.shape[0]
    dims = [x.shape[1], wgu.shape[1] // 2] + ([sgu.shape[0] // 2] if sgu is not None else [])
    return (x.dtype == torch.bfloat16 and T <= FEW_TOKENS and T * top <= FEW_PAIRS and all(d % 16 == 0 for d in dims)
            and x.stride(0) % 8 == 0)


def _grouped(x, wgu) -> bool:
    """Sizes the matrix-core products of sorted rows take."""
    return (x.dtype == torch.bfloat16 and x.shape[1] % 8 == 0 and wgu.shape[1] % 16 == 0 and x.stride(0) % 8 == 0
            and x.shape[0] * x.stride(0) < 1 << 29 and wgu[0].numel() < 1 << 29)
