"""Ops of decoders whose sublayers are normed at their output, on an f32 residual stream ``h``: every
residual step returns the activation copy of the new ``h`` (bf16; in f32 ``h`` itself) that the next
sublayer's projections read.

GPU: csrc/kernels/postnorm.hip.  CPU tensors: plain PyTorch (the CPU test suite).
"""
from __future__ import annotations

import os

import torch

from . import gemm
from ._ext import native, use_native
from .linear import _DECODE_M, SKINNY_M, _plain


def _rms(x: torch.Tensor, eps: float) -> torch.Tensor:
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _copy(h: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    return h if dtype == torch.float32 else h.to(dtype)


def embed_norm(ids: torch.Tensor, table: torch.Tensor, w: torch.Tensor, eps: float):
    """(h, its activation copy): the normed embedding rows."""
    if use_native(table):
        h, y = native().embed_norm(ids.contiguous(), table, w, eps)
        return h, h if table.dtype == torch.float32 else y
    h = _rms(table[ids].float(), eps) * w
    return h, _copy(h, table.dtype)


def post_norm(src: torch.Tensor, h: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    """h (f32, in place) += rms(src) * w."""
    if use_native(h):
        y = native().post_norm(src, h, w, eps)
        return h if src.dtype == torch.float32 else y
    h += _rms(src.float(), eps) * w
    return _copy(h, src.dtype)


def post_route(src: torch.Tensor, h: torch.Tensor, w: torch.Tensor, eps: float, router: torch.Tensor, top: int):
    """Prompt rows, one launch (csrc/kernels/post_route.hip): (:func:`post_norm`, the experts of each row and their weights as
    ``moe.route`` has them); None, and nothing done, for calls that it does not take."""
    T, W = h.shape
    if (not FUSED or not use_native(h) or src.dtype != torch.bfloat16 or router.dtype != torch.bfloat16 or T <= _DECODE_M or W % 1024
            or W > 4096 or router.shape[0] > 16 or not all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in (h, w, router))
            or src.stride(0) % 4 or src.data_ptr() % 8 or not _plain(src, h, router)):
        return None
    return native().post_route(src, h, w, eps, router, top)


DECODE_ROWS = 64  # rows up to which the fused decode kernels run
FUSED = os.environ.get("MXLLM_SUBLAYER_FUSED", "1") != "0"  # 0: always the parts, of prompts too (A/B)


def fusable(x: torch.Tensor, *mats: torch.Tensor | None) -> bool:
    """Whether :func:`post_dots` takes decode rows like ``x`` and these matrices."""
    return (FUSED and use_native(x) and x.dim() == 2 and x.dtype == torch.bfloat16 and x.shape[0] <= DECODE_ROWS
            and all(w is not None and w.dtype == torch.bfloat16 and w.is_contiguous() and w.shape[1] <= 4096
                    and w.shape[1] % 8 == 0 for w in mats))


def post_dots(src: torch.Tensor, h: torch.Tensor, w: torch.Tensor, eps: float, m: torch.Tensor,
              wts: torch.Tensor | None = None, shared: torch.Tensor | None = None, emb: torch.Tensor | None = None,
              ids: torch.Tensor | None = None, off: int = 0):
    """Decode rows, one launch: the residual step (:func:`post_norm`, or with ``wts`` :func:`mix_post_norm` of
    rows in pair order) and the products of the new h's copy with the rows of ``m``: (new h, copy, f32
    products), or with ``emb`` their :func:`side_act` in place of the products (and no copy).  ``h`` stays as
    it is."""
    return native().post_dots(src, h, w, eps, m, wts, shared, emb, ids, off)


def side_post(g: torch.Tensor, p: torch.Tensor | None, h: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor | None:
    """Decode rows, one launch: ``post_norm(g p^T, h, w, eps)`` of the few columns of a second embedding; None: sizes
    or types that it does not take.  A workgroup a row reads all of ``p``: 256 KB are worth the launch (steps of the 1B size, 8 / 16 /
    32 sequences 1242 / 1333 / 1572 -> 1216 / 1314 / 1556 us, 1 to 4 as before), 512 KB are not (8B, 1 / 8 sequences 3386 / 4549 ->
    3458 / 4608)."""
    W = h.shape[1]
    if not (p is not None and p.numel() <= 1 << 17 and FUSED and use_native(g) and g.dtype == p.dtype == torch.bfloat16
            and g.shape[0] <= DECODE_ROWS and g.shape[1] in (32, 64, 128) and W <= 4096 and W % (16 * 512 // g.shape[1]) == 0
            and g.is_contiguous() and p.is_contiguous() and all(t.data_ptr() % 16 == 0 for t in (g, p, h, w))):
        return None
    return native().post_side(g, p, h, w, eps)


def mix_post_norm(src: torch.Tensor, inv: torch.Tensor | None, wts: torch.Tensor, shared: torch.Tensor | None,
                  h: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    """h += rms(m) * w, m the sum of a token's expert rows by their weights ``wts`` [T, top] (row ``inv`` of
    ``src``; None: rows in (token, choice) order) and the ``shared`` expert's row."""
    if use_native(h):
        y = native().mix_post_norm(src, inv, wts, shared, h, w, eps)
        return h if src.dtype == torch.float32 else y
    rows = src.float() if inv is None else src.float()[inv.view(-1).long()]
    m = (rows.view(*wts.shape, -1) * wts[..., None]).sum(1)
    if shared is not None:
        m = m + shared.float()
    h += _rms(m, eps) * w
    return _copy(h, src.dtype)


def side_act(z: torch.Tensor, emb: torch.Tensor, ids: torch.Tensor, off: int) -> torch.Tensor:
    """gelu_tanh(z) times columns [off, off + dim) of the tokens' rows of ``emb``."""
    if use_native(z):
        return native().side_act(z, emb, ids, off)
    e = emb[ids, off:off + z.shape[1]].float()
    return (torch.nn.functional.gelu(z.float(), approximate="tanh") * e).to(z.dtype)


def side_gate(x: torch.Tensor, w: torch.Tensor, emb: torch.Tensor, ids: torch.Tensor, off: int) -> torch.Tensor | None:
    """:func:`side_act` of ``x w^T`` in one launch (csrc/kernels/side_gate.hip); None where it does not take the call."""
    # One wave a block of 16 rows x 16 channels: past 2,048 of them the library's larger tiles are the quicker ones (with side_act,
    # us, 64 x 4096 at 8192 / 16384 rows 19.8 / 26.7 -> 15.5 / 28.5, 64 x 2048 11.5 / 16.1 -> 10.3 / 17.7; 256 x 2048 at 2048 / 3000
    # 11.3 / 11.9 -> 9.2 / 13.5).  A decode step has it behind post_dots.
    if not FUSED or not use_native(x) or x.dim() != 2 or x.shape[0] <= _DECODE_M or SKINNY_M <= 0:
        return None
    (T, K), N = x.shape, w.shape[0]
    if (N % 16 or K % 64 or off % 4 or (T + 15) // 16 * (N // 16) > 2048 or emb.dtype != torch.bfloat16 or emb.shape[1] % 4
            or emb.data_ptr() % 8 or not _plain(x, w, emb) or not gemm.rows_ok(x, w, True, cols=16)):
        return None
    return native().side_gate(x, w, emb, ids, off)


def clipped_glu(z: torch.Tensor, limit: float) -> torch.Tensor:
    """z = gate | up: g = min(gate, limit), u = up clipped to +-limit; g sigmoid(1.702 g) (u + 1)."""
    if use_native(z):
        return native().clipped_glu(z, limit)
    g, u = z.float().chunk(2, -1)
    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return (g * torch.sigmoid(1.702 * g) * (u + 1)).to(z.dtype)
