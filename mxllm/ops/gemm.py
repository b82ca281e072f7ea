"""GEMM dispatch between the hand-written 8-phase MFMA kernel (csrc/kernels/gemm8.hip) and
hipBLASLt / rocBLAS (``torch.mm`` with the tuned solution table, mxllm/utils/gemm_tuning.py).

Every training GEMM of a Llama step is one of four operand orders over row-major bf16 storage:

  form  A stored   B stored   computes          used for
  tn    [M][K]     [N][K]     A @ B^T           forward  y = x W^T
  nn    [M][K]     [K][N]     A @ B             input gradient  dX = dY W
  tt    [K][M]     [K][N]     A^T @ B           weight gradient dW = dY^T X (token-major operands)
  nt    [K][M]     [N][K]     A^T @ B^T         (unused; for completeness)

``gemm8`` is selected only where it was measured faster: per (form, M, N, K, output dtype) from a
table (``mxllm/tuning/gemm8_gfx950.json``, written from ``bench/gemm8_probe.py`` runs; entries with
``tail``: the tail-balanced launch, ``mx_gemm8_tail`` -- a last wave of at most half the CUs runs as
twice as many half-K workgroups, e.g. the 16 x 40-tile 70B qkv forward), by the rule of ``_gains``
for the sizes that the table does not hold, or for every shape it takes in deterministic mode
(``MXLLM_DETERMINISTIC=1``: one workgroup per output tile, a fixed K order, no split-K or atomics —
the step is bitwise reproducible; vendor stream-K solutions are not, archive/profiles/r3aa).
``MXLLM_GEMM8=0`` disables it, ``=all`` forces it wherever it takes the shape (A/B runs).  Gradients whose output is one turn
of smaller tiles go to csrc/kernels/gemm_tile_forms.hip ahead of both (:func:`form_plan`; one workgroup a tile, K in order).
"""
from __future__ import annotations

import functools
import json
import os

import torch

from ._ext import native, untransformed, use_native

_TABLE_PATH = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tuning",
                           "gemm8_gfx950.json")
_TABLE: dict | None = None


def deterministic() -> bool:
    return os.environ.get("MXLLM_DETERMINISTIC", "0") == "1"


_TAIL: dict = {}


def _table() -> dict:
    global _TABLE
    if _TABLE is None:
        _TABLE = {}
        try:
            with open(_TABLE_PATH) as f:
                for e in json.load(f).get("wins", []):
                    key = (e["form"], e["M"], e["N"], e["K"], e["out"])
                    _TABLE[key] = int(e.get("ph", 8))
                    if e.get("tail"):
                        _TAIL[key] = int(e["tail"])
        except (OSError, ValueError, KeyError):
            pass
    return _TABLE


CUS = 256  # MI355X compute units: one gemm8 workgroup (256 x 256 tile) per CU at a time


def tail_split(M: int, N: int, K: int) -> int:
    """Split of the tail-balanced launch (mx_gemm8_tail), 0 if it does not apply: the tile grid leaves
    a last wave of at most half the CUs.  > 0: split at that COLUMN (whole waves of tiles in columns
    [0, N1)); < 0: split at ROW -value (when no column split gives whole waves)."""
    if M % 256 or N % 256 or K < 128:
        return 0
    nM, nN = M // 256, N // 256
    r = (nM * nN) % CUS
    if r == 0 or r > CUS // 2:
        return 0
    full = nM * nN - r
    if full % nM == 0 and 0 < full // nM < nN:
        return full // nM * 256
    if full % nN == 0 and 0 < full // nN < nM:
        return -(full // nN * 256)
    return 0


def _multi_rank() -> bool:
    """True in a process group of more than one rank.  The persistent gemm8 (table ``ph`` 5) gives
    each of its one-per-CU workgroups a FIXED share of the tiles; a collective kernel that holds CUs
    for its whole duration (RCCL's channels, the peer collectives) then delays the workgroups that
    cannot start, and with them the whole GEMM -- under ZeRO-3's reduce-scatters overlapped with the
    dW GEMMs that costs far more than the persistence wins (0.7 % of the world-1 config-4 proxy,
    profiles/r5e).  The one-tile-per-workgroup launch lets the hardware rebalance around them."""
    import torch.distributed as dist

    # asked only for ph-5 shapes (a few fp32 dW GEMMs per layer): not cached, so a process that
    # brings a group up or down later is still answered right
    return dist.is_available() and dist.is_initialized() and dist.get_world_size() > 1


def _policy() -> str:
    return os.environ.get("MXLLM_GEMM8", "table")


def takes(form: str, M: int, N: int, K: int) -> bool:
    """Shape constraints of the kernel (mirrors mx_gemm8)."""
    if M % 256 or N % 256 or K <= 0:
        return False
    return K % 64 == 0 or form == "tt"


def schedule(form: str, M: int, N: int, K: int, out_dtype: torch.dtype, rules: bool = True) -> int:
    """0 = not on gemm8; else its phase schedule (8 or 4) for this shape (``rules`` False: by the table alone)."""
    pol = _policy()
    if pol == "0" or not takes(form, M, N, K):
        return 0
    ph = _table().get((form, M, N, K, "f32" if out_dtype == torch.float32 else "bf16"), 0)
    if ph == 5 and _multi_rank():
        ph = 4  # persistent kernel: world 1 only (see _multi_rank)
    if ph:
        return ph
    if rules and out_dtype == torch.bfloat16 and _gains(form, M, N, K):
        return 4
    return DEFAULT_PH if (pol == "all" or deterministic()) else 0


def _gains(form: str, M: int, N: int, K: int) -> bool:
    """bf16-output shapes outside the table that gemm8 (4-phase, one 256 x 256 tile a CU) runs faster.

    ``tt``: what it saves is the two transposes and their launches; what it loses to hipBLASLt is the split of
    a long K when the tiles leave CUs idle.  (us: transposes + hipBLASLt -> gemm8; M x N, K tokens)
      * a short K, at any number of tiles: 512 x 512, 1000: 40 -> 23; 2048 x 2048, 300: 41 -> 14
        (4 to 64 tiles at 2048: 37 -> 38..41, at 4096: 36..56 -> 70..75);
      * a K that is no multiple of 64, which hipBLASLt reads slowly: 16384 x 2048, 3606: 271 -> 179;
      * else a last wave that is full enough.  One wave: 144 tiles 4096: 89 -> 77, 8192: 161 -> 146 (128 tiles 77 ->
        78 and 144 -> 154).  More: 256 tiles 118 -> 98, 512 237 -> 200, 384 172 -> 167 (288 tiles 149 -> 160).
    But not where there is little to save: a long K in multiples of 8 on 64 tiles (2048 x 2048, 3608 75 -> 74, 5160 93 -> 97,
    5600 93 -> 104), and round token counts of very many tiles, whose transposes are small beside the product or whose
    time is the output's (57344 x 8192, 256 520 -> 595, 416 662 -> 694, 1536 1270 -> 1355, but 1544 1293 -> 1165; 8192 x
    28672, 2304 840 -> 880; 128256 x 2048, 256 320 -> 355, but 768 553 -> 528 and 5120 2542 -> 2054).
    ``nn``: :func:`_gains_nn`."""
    tiles = (M // 256) * (N // 256)
    # past the kernel's 32-bit offsets (it would decline: the caller's other path stays)
    if K < 128 or (K + 63) // 64 * 64 * max(M if form == "tt" else 0, N) >= 1 << 30:
        return False
    if form == "tt":
        full = _wave_fill(tiles)
        if K % 32 == 0 and tiles >= 3584 and (min(M, N) >= 8192 or K <= 512):
            return False
        if K % 8 == 0 and K > 4096 and tiles < 96:
            return False
        return K <= 1536 or (K % 64 != 0 and tiles >= 64) or (tiles >= 144 and full >= (0.56 if tiles <= CUS else 0.7))
    return form == "nn" and _gains_nn(tiles)


def _wave_fill(tiles: int) -> float:
    """Part of the CUs' turns that ``tiles`` of one workgroup a CU use."""
    return tiles / (max(-(-tiles // CUS), 1) * CUS)


def _gains_nn(tiles: int) -> bool:
    """Input gradients: both kernels read the operands as they are; gemm8 where its tiles fill their waves (us,
    library -> gemm8): 176 tiles, 28672 -> 4096 at 2600 rows 830 -> 536, 6144 -> 4096 115 -> 109; 192, 8192 -> 8192 at
    1300 149 -> 142; 352 at 2600 300 -> 300; 784, 4096 -> 14336 at 3606 417 -> 336; but 160 tiles 176 -> 182, 280
    133 -> 152, 320 at 5000 219 -> 228."""
    return _wave_fill(tiles) >= 0.68


def rows_ok(a: torch.Tensor, b: torch.Tensor, b_kc: bool, swiglu: bool = False, cols: int = 256) -> bool:
    """What mx_gemm8_rows (csrc/kernels/gemm8_rows.hip) takes: any number of rows of ``a`` [M, K].  ``cols`` 16: what
    mx_gemm_tile (csrc/kernels/gemm_tile.hip) does (``b_kc``)."""
    if not (use_native(a) and a.is_cuda and a.device == b.device and a.dtype == b.dtype == torch.bfloat16):
        return False
    K, N = a.shape[1], b.shape[0 if b_kc else 1]
    ldb = b.stride(0)
    return bool(a.shape[0] > 0 and K % 64 == 0 and K > 0 and N % cols == 0 and N > 0
                and a.stride(1) == 1 and b.stride(1) == 1 and a.stride(0) % 8 == 0 and ldb % 8 == 0
                and a.stride(0) >= K and ldb >= (K if b_kc else N)
                and a.data_ptr() % 16 == 0 and b.data_ptr() % 16 == 0
                and 256 * a.stride(0) < 1 << 30 and (N if swiglu else 256 if b_kc else K) * ldb < 1 << 30)


@functools.lru_cache(maxsize=4096)  # (of sizes alone)
def _tile_plan(M: int, N: int, K: int, swiglu: bool) -> tuple[int, int] | None:
    plan = native().gemm_tile_plan(M, N, K, swiglu)
    return None if plan < 0 else divmod(plan, 64)


def tile_plan(M: int, N: int, K: int, swiglu: bool = False) -> tuple[int, int] | None:
    """(tile, parts of K) of a projection that csrc/kernels/gemm_tile.hip has faster than the library and gemm8 (the rule is
    beside the kernel: mx_gemm_tile_plan); None: not."""
    return None if _policy() == "0" else _tile_plan(M, N, K, swiglu)


@functools.lru_cache(maxsize=4096)
def _rows_head(M: int, N: int, K: int) -> tuple[int, int] | None:
    rows, cols = -(-M // 256), N // 256
    turns = rows * cols // CUS
    head = turns * CUS // max(cols, 1)
    rest = M - 256 * head
    if K > 2048 or not turns or head >= rows or (rows - head) * cols > CUS // 2 or head * cols < 0.9 * turns * CUS:
        return None
    plan = _tile_plan(rest, N, K, True)
    return (256 * head, plan[0]) if plan and plan[1] == 1 else None


def rows_head(M: int, N: int, K: int) -> tuple[int, int] | None:
    """Of a gate-up projection with SwiGLU that :func:`rows_gain` gives to gemm8 whole: (rows of its whole turns, the tile of
    csrc/kernels/gemm_tile.hip for the rows behind them), None: all rows gemm8.  Its last turn takes as long with a few tiles as with
    256; smaller tiles share those rows among all CUs.  Replayed, us: 16384 x 2048 at 1100 / 1300 /
    1500 / 2300 / 3300 / 4400 rows 88 / 88 / 90 / 137 / 188 / 240 -> 67 / 79 / 83 / 123 / 172 / 228; 16384 x 1024 at 1030 / 2560 47 / 76
    -> 36 / 72; 10240 x 2048 at 3584 129 -> 112.  Past half a turn of tiles it is level or loses (16384 x 2048 at 1800 99 -> 105, 2709
    146 -> 153), as past a K of 2048 (28672 x 4096 at 1300 / 1500 254 / 264 -> 259 / 275)."""
    return None if _policy() == "0" else _rows_head(M, N, K)


@functools.lru_cache(maxsize=4096)
def _form_plan(tt: bool, M: int, N: int, K: int) -> int:
    return native().gemm_tile_form_plan(tt, M, N, K)


def form_plan(form: str, M: int, N: int, K: int) -> int:
    """Tile of a gradient's product ("nn", "tt") that csrc/kernels/gemm_tile_forms.hip has faster than the library and gemm8
    (the rule is beside the kernel: mx_gemm_tile_form_plan); -1: not, or MXLLM_GEMM8 asks for one of those."""
    return _form_plan(form == "tt", M, N, K) if _policy() == "table" else -1


def form_mm(form: str, a: torch.Tensor, b: torch.Tensor, out: torch.Tensor | None = None, beta: float = 0.0):
    """``out = beta * out + op(a) b`` (bf16; ``out`` None: new) by that kernel; None: it does not take the call, or the
    backward that asks is one of many at once (``is_grads_batched``), traced or recorded."""
    if not (use_native(a) and a.is_cuda and a.device == b.device and a.dtype == b.dtype == torch.bfloat16 and a.numel() and b.numel()
            and (out is None or out.dtype == torch.bfloat16)) or asks_grad(a, b):
        return None
    M, N, K = _dims(form, a, b)
    tile = form_plan(form, M, N, K)
    if tile < 0 or not untransformed(a, b):
        return None
    if out is None:
        out, beta = torch.empty(M, N, dtype=a.dtype, device=a.device), 0.0
    return out if native().gemm_tile_form(a, b, out, form == "tt", float(beta), tile) else None


def rows_gain(M: int, N: int, K: int, b_kc: bool, swiglu: bool = False) -> int:
    """Parts of K (1: whole) in which the rows kernel is the faster one, else 0.

    In parts where the tiles leave half the CUs without one and K is long; each part costs its fp32 image's trip (us,
    library -> gemm8; K x N at rows):
      * projections (``b_kc``): K of 12,288 and 64 rows on.  14336 x 4096 at 64 35 -> 31, 128 59 -> 36, 400 80 -> 57,
        1000 122 -> 97, 2048 191 -> 171; 28672 x 8192 at 200 312 -> 122, 512 327 -> 192 (14336 x 4096 at 48 28 -> 30; 8192 x
        2048 at 512 29 -> 37, 2048 69 -> 67); in two or three parts not past a K of 24,576 (28672 x 8192 at 559 277 -> 315,
        768 304 -> 321);
      * input gradients: K of 6144 on.  16384 x 2048 at 1000 124 -> 68, 4096 237 -> 211; 6144 x 4096 at 512 53 -> 43
        (3072 x 2048 at 512 26 -> 30); in two or three parts of a K over 24,576 with the last tile's rows not mostly
        padding (57344 x 8192 at 560 524 -> 576, 700 595 -> 591, 1000 738 -> 656).
    Whole, where the library, which is tuned for round numbers of rows, falls behind between them:
      * projections (``b_kc``) of a K of 256 to 512 and 1,024 rows on, from five eighths of the CUs to two turns: 8192 x 512 at 1400 /
        1536 / 2048 / 2709 33 / 28 / 23.0 / 47 -> 19 / 19 / 20.7 / 34, 4096 x 256 at 2816 23 -> 15, 6144 x 384 at 1900 24 -> 17; .83 over
        118 random sizes (worst 5888 x 448 at 1599 17.3 -> 18.7; profiles/gemm_routes/short_k.txt).  With fewer tiles 4096 x 256 at 2500 13.1 ->
        14.4; with two turns and more 16384 x 256 at 2048 / 4096 31 / 57 -> 33 / 70; with fewer rows, which are wide outputs' or
        padding, 65536 x 256 at 33 / 64 10.6 / 10.8 -> 12.4 / 13.0, 32768 x 512 at 300 19.5 -> 20.4;
      * projections of K 8192 and more from 500 tiles on: 8192 x 57344 at 700 559 -> 530, 2600 1916 -> 1740;
        8192 x 10240 at 3100 537 -> 456 (at 2600, 440 tiles: 317 -> 321), up to 4096 tiles and from 128 rows on (8192 x
        128256 at 64 414 -> 394 to 454, 158 540 -> 450, 1700 2650 -> 2550, 2210 3378 -> 3555, 4445 6338 -> 6656).  With a
        shorter K the library is up to 27 % slower at some row counts and 3 to 6 % faster at others (4096 x 28672 at 2700 543
        -> 441, 4003 600 -> 634);
      * input gradients: :func:`_gains_nn`, with the last tile's rows not mostly padding (8192 -> 28672 at
        300 175 -> 184, 371 180 -> 190, 408 0.92);
      * gate-up with SwiGLU, which saves the projection's trip through HBM at any size: where the last tile's rows are
        not mostly padding and five eighths of the CUs have a tile.  2048 x 16384 at 700 48 -> 42, 2600 205 -> 142, 4096
        236 -> 198 (512, 128 tiles: 38 -> 40); 4096 x 28672 at 450 109 -> 97 (300: 77 -> 85), 4096 706 -> 640.  The longer K,
        the less the trip counts beside CUs that wait in the last turn or multiply padding: of a K of 4096 three fifths of
        the turns' places have to be outputs (10240 at 1792 rows, .55: 156 -> 163; 6144 at 3328, .61: 0.90), of a longer one .63
        (8192 x 8192 at 1105, .54: 143 -> 153; 1377, .67: 0.88), from three turns on .7
        (8192 x 10240 at 3328, .68: 447 -> 479; 3693, .75: 0.71), and past 8192 N at least as large (21504 x 4096 at 4013,
        .98: 465 -> 487, at 5120, .62: 724 -> 844)."""
    rows = -(-M // 256)
    tiles = rows * (N // 256)
    turns = -(-tiles // CUS)
    dense = 4 * M >= 3 * 256 * rows  # the last tile's missing rows are a quarter of the tiles at most
    useful = M * N / (max(turns, 1) * CUS * 65536)  # outputs of the places that the turns have
    if 0 < tiles <= CUS // 2 and not swiglu and (M >= 64 and K >= 12288 if b_kc else K >= 6144):
        parts = min(CUS // tiles, 16)
        if parts < 4 and K > 24576 and (b_kc or not dense):
            parts = 0
    elif swiglu:
        fill = 0.0 if K <= 2048 else 0.7 if turns > 2 else 0.6 if K <= 4096 else 0.63
        parts = int(tiles >= CUS * 5 // 8 and dense and useful >= fill and (K <= 8192 or N >= K))
    elif b_kc:
        parts = int(M >= 128 and M % 256 != 0 and K >= 8192 and 500 <= tiles <= 4096
                    or M >= 1024 and 256 <= K <= 512 and CUS * 5 // 8 < tiles < 2 * CUS)
    else:
        parts = int(M % 256 != 0 and K >= 128 and _gains_nn(tiles) and dense)
    return parts if parts and _policy() != "0" else 0


DEFAULT_PH = int(os.environ.get("MXLLM_GEMM8_DEFAULT_PH", "4"))


def want(form: str, M: int, N: int, K: int, out_dtype: torch.dtype, rules: bool = True) -> bool:
    return schedule(form, M, N, K, out_dtype, rules) > 0


def asks_grad(a: torch.Tensor, b: torch.Tensor) -> bool:
    """A backward pass that is itself to be differentiated (``create_graph``).  The sizes that go to a kernel by rule
    then stay with torch, which refuses what it cannot differentiate; a kernel would leave the gradient out."""
    return torch.is_grad_enabled() and (a.requires_grad or b.requires_grad)


# (A k-contiguous, B k-contiguous) per form
_KC = {"tn": (True, True), "nn": (True, False), "tt": (False, False), "nt": (False, True)}


def _dims(form, a, b):
    if form == "tn":
        return a.shape[0], b.shape[0], a.shape[1]
    if form == "nn":
        return a.shape[0], b.shape[1], a.shape[1]
    if form == "tt":
        return a.shape[1], b.shape[1], a.shape[0]
    return a.shape[1], b.shape[0], a.shape[0]


def mm(form: str, a: torch.Tensor, b: torch.Tensor, out: torch.Tensor | None = None, beta: float = 0.0,
       alpha_t: torch.Tensor | None = None, out_dtype: torch.dtype | None = None) -> torch.Tensor:
    """``out = beta * out + alpha_t * op(a) op(b)`` in operand order ``form`` (module doc).
    ``out`` None: a new [M, N] tensor of ``out_dtype`` (default: a's dtype) and beta is 0.
    ``alpha_t``: optional 1-element f32 device scalar (no host sync)."""
    M, N, K = _dims(form, a, b)
    odt = out.dtype if out is not None else (out_dtype or a.dtype)
    asked = asks_grad(a, b)
    if form in ("nn", "tt") and alpha_t is None and odt == torch.bfloat16 and (form == "tt" or beta == 0.0):
        y = form_mm(form, a, b, out, beta)
        if y is not None:
            return y
    if out is None and not asked and form in ("tn", "nn") and alpha_t is None and odt == torch.bfloat16:
        parts = rows_gain(M, N, K, form == "tn")
        if parts and rows_ok(a, b, form == "tn"):
            return native().gemm8_rows(a, b, form == "tn", False, parts)
    if out is None:
        out = torch.empty(M, N, dtype=odt, device=a.device)
        beta = 0.0
    ph = (schedule(form, M, N, K, odt, not asked) if use_native(a) and a.dtype == torch.bfloat16 and b.dtype == torch.bfloat16
          and odt in (torch.bfloat16, torch.float32) else 0)
    if ph:
        a_kc, b_kc = _KC[form]
        t = _TAIL.get((form, M, N, K, "f32" if odt == torch.float32 else "bf16"), 0)
        if (t and beta == 0.0 and alpha_t is None and odt == torch.bfloat16
                and native().gemm8_tail(a, a_kc, b, b_kc, out, abs(t), t < 0, ph)):
            return out
        if native().gemm8(a, a_kc, b, b_kc, out, float(beta), alpha_t, 1.0, ph):
            return out
    A = a if form in ("tn", "nn") else a.t()
    B = b.t() if form in ("tn", "nt") else b
    if alpha_t is not None:
        A = A * alpha_t.to(A.dtype)
    if odt == a.dtype:
        if beta == 0.0:
            return torch.mm(A, B, out=out)
        return out.addmm_(A, B, beta=beta)
    if a.is_cuda:  # bf16 operands, fp32 output (hipBLASLt D = C in fp32)
        return torch.ops.aten.addmm.dtype_out(out, A, B, odt, beta=beta, out=out)
    return out.mul_(beta).add_(A.float() @ B.float()) if beta != 0.0 else out.copy_(A.float() @ B.float())


def mm_sq(form: str, a: torch.Tensor, b: torch.Tensor, out: torch.Tensor, sq: torch.Tensor,
          alpha_t: torch.Tensor | None = None) -> bool:
    """``out = alpha_t * op(a) op(b)`` (bf16, beta 0) on gemm8 that also writes one fp32 sum of squares of
    the stored values per 256 x 256 output tile into ``sq`` (row-major tile order).  Only where the
    dispatch puts this shape on the plain 4-phase gemm8 anyway (same kernel, same bits in ``out``);
    False: nothing launched, the caller takes ``mm``."""
    M, N, K = _dims(form, a, b)
    if not (use_native(a) and a.dtype == b.dtype == out.dtype == torch.bfloat16 and M % 256 == 0 and N % 256 == 0):
        return False
    if schedule(form, M, N, K, torch.bfloat16) != 4 or (alpha_t is None and form_plan(form, M, N, K) >= 0):
        return False
    a_kc, b_kc = _KC[form]
    t = _TAIL.get((form, M, N, K, "bf16"), 0)
    if t and alpha_t is None:  # the tail-balanced launch, as ``mm`` takes it (its split part sums per tile)
        return bool(native().gemm8_tail(a, a_kc, b, b_kc, out, abs(t), t < 0, 4, sq))
    return bool(native().gemm8_sq(a, a_kc, b, b_kc, out, sq, alpha_t, 1.0))
