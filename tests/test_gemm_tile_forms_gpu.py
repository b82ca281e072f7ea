"""Gradients by one turn of tiles (csrc/kernels/gemm_tile_forms.hip) at the edges of their tiles and of K, against 64-bit sums of
the same bf16 operands."""
import pytest
import torch

from mxllm.ops import gemm
from mxllm.ops.linear import linear, weight_grad_

pytestmark = pytest.mark.gpu
TILES = [(64, 64), (64, 128), (128, 128), (128, 192), (192, 128), (256, 128), (192, 192)]


def _operands(gpu, tt, M, N, K, pad):
    torch.manual_seed(M + 3 * N + 7 * K)
    a = torch.randn(K, M + pad, device=gpu).bfloat16()[:, :M] if tt else torch.randn(M, K + pad, device=gpu).bfloat16()[:, :K]
    b = torch.randn(K, N + pad, device=gpu).bfloat16()[:, :N]
    x = a.double().t().contiguous() if tt else a.double()
    return a, b, x @ b.double()


def _close(got, want, K):
    # f32 sums of K products of unit operands (K 2^-24 of their sizes' sum at most, far less as seen) and one rounding to bf16
    assert float((got.double() - want).abs().max()) <= 2.0 ** -8 * float(want.abs().max()) + 2.0 ** -23 * K
    assert float((got.double() - want).norm()) <= 2.0 ** -8 * float(want.norm())


@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("K,pad", [(64, 0), (128, 8), (192, 0), (448, 64)])
def test_input_gradients(gpu, tile, K, pad):
    from mxllm.ops import native

    tm, tn = TILES[tile]
    for M, N in [(1, 16), (tm, tn), (tm + 1, tn + 16), (2 * tm - 1, 3 * tn - 48), (10 * tm - 15, 2 * tn)]:  # (bands of 8 tiles down)
        a, b, want = _operands(gpu, False, M, N, K, pad)
        out = torch.full((M, N + 8), 7.0, device=gpu).bfloat16()
        assert native().gemm_tile_form(a, b, out[:, :N], False, 0.0, tile)
        _close(out[:, :N], want, K)
        assert bool((out[:, N:] == 7).all())


@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("K,pad", [(1, 0), (63, 8), (64, 0), (65, 0), (200, 16), (449, 0)])
def test_weight_gradients(gpu, tile, K, pad):
    from mxllm.ops import native

    tm, tn = TILES[tile]
    for M, N in [(16, 16), (tm, tn), (tm + 16, tn + 48), (2 * tm - 16, 3 * tn - 16), (10 * tm - 16, 2 * tn)]:  # (bands of 8 tiles down)
        a, b, want = _operands(gpu, True, M, N, K, pad)
        out = torch.full((M, N), float("nan"), device=gpu).bfloat16()
        assert native().gemm_tile_form(a, b, out, True, 0.0, tile)
        _close(out, want, K)
        old = torch.randn(M, N, device=gpu).bfloat16()
        out = old.clone()
        assert native().gemm_tile_form(a, b, out, True, 1.0, tile)
        _close(out, want + old.double(), K)


class _Seen:
    """The native library, noting the tiles that gemm_tile_form ran."""

    def __init__(self, ops):
        self.ops, self.tiles = ops, []

    def __getattr__(self, name):
        return getattr(self.ops, name)

    def gemm_tile_form(self, *args):
        done = self.ops.gemm_tile_form(*args)
        self.tiles += [args[-1]] if done else []
        return done


@pytest.mark.parametrize("form,M,N,K", [("tt", 2048, 512, 1003), ("tt", 768, 768, 256), ("tt", 336, 1040, 777), ("nn", 333, 1024, 512), ("nn", 1000, 512, 4032)])
def test_route(gpu, form, M, N, K, monkeypatch):
    """``gemm.mm`` and, of weights, ``weight_grad_`` take the kernel for the sizes of its rule, and leave others and unaligned
    operands alone."""
    from mxllm.ops import native

    a, b, want = _operands(gpu, form == "tt", M, N, K, 0)
    tile = gemm.form_plan(form, M, N, K)
    assert tile >= 0 and gemm.form_plan("nn", M, N, 4096) < 0
    out = torch.empty(M, N, device=gpu, dtype=torch.bfloat16)
    assert native().gemm_tile_form(a, b, out, form == "tt", 0.0, tile)
    _close(out, want, K)
    seen = _Seen(native())
    monkeypatch.setattr(gemm, "native", lambda: seen)
    assert torch.equal(gemm.mm(form, a, b), out) and seen.tiles == [tile]
    if form == "tt":
        assert torch.equal(weight_grad_(None, a, b), out) and seen.tiles == [tile] * 2
        grad = torch.ones_like(out)
        _close(weight_grad_(grad, a, b, beta=1.0), want + 1, K)
        assert seen.tiles == [tile] * 3
    seen.tiles.clear()
    shifted = torch.empty(b.numel() + 4, device=gpu, dtype=torch.bfloat16)[4:].view_as(b).copy_(b)
    assert gemm.form_mm(form, a, shifted) is None
    _close(gemm.mm(form, a, shifted), want, K)
    assert not seen.tiles


def test_few_channels_stay():
    """Input gradients of 16 channels leave a K of 1024 and more to the library (the rule beside the kernel)."""
    for M in (81, 775, 2634, 8000):
        assert gemm.form_plan("nn", M, 16, 960) >= 0 and gemm.form_plan("tt", M // 16 * 16, 16, M) >= 0
        assert all(gemm.form_plan("nn", M, 16, K) < 0 for K in (1024, 1088, 3584))
    assert gemm.form_plan("nn", 2634, 32, 3584) >= 0


@pytest.mark.parametrize("T,N,K", [(2048, 2048, 2048), (64, 64, 64)])
def test_many_backwards_at_once(gpu, T, N, K):
    """``is_grads_batched`` runs a backward under vmap, for which the kernel has no rule: such a call goes elsewhere."""
    torch.manual_seed(T)
    w = torch.randn(N, K, device=gpu).bfloat16().requires_grad_()
    x, dy = torch.randn(T, K, device=gpu).bfloat16(), torch.randn(2, T, N, device=gpu).bfloat16()
    y = linear(x, w)
    assert gemm.form_plan("tt", N, K, T) >= 0
    (got,) = torch.autograd.grad(y, [w], dy, is_grads_batched=True, retain_graph=True)
    for i in range(2):
        _close(got[i], dy[i].double().t().contiguous() @ x.double(), T)
