"""Products of prompt passes that end in their activation, against the two launches."""
import pytest
import torch

from mxllm.ops import gemm, moe, sublayer
from mxllm.ops._ext import native
from mxllm.ops.linear import _DECODE_M, linear, linear_clipped

pytestmark = pytest.mark.gpu


def _rand(*shape, scale=1.0):
    return (torch.randn(*shape, device="cuda") * scale).bfloat16()


@pytest.mark.parametrize("tile", range(7))
@pytest.mark.parametrize("M,F,K", [(1, 8, 64), (33, 40, 128), (193, 200, 64), (257, 264, 320)])
def test_clipped_epilogue_is_the_two_launches(tile, M, F, K):
    """K in order in either: the product's bits are those of the same tile, the unit's those of clipped_glu."""
    torch.manual_seed(M)
    x, w = _rand(M, K), _rand(2 * F, K, scale=4 / K**0.5)
    x[0, 0] = float("inf")  # gates and ups of infinity and, with a zero weight, NaN
    w[F // 2, 0] = 0
    two = native().clipped_glu(native().gemm_tile(x, w, False, tile, 1), 2.5)
    one = native().gemm_tile_clipped(x, w, 2.5, tile)
    torch.testing.assert_close(one, two, rtol=0, atol=0, equal_nan=True)


def test_clipped_epilogue_in_the_experts():
    """Where the plan is one part the shared expert takes it, and its rows are those of the two launches."""
    torch.manual_seed(0)
    M, W, F = 300, 256, 2048
    x, w, down = _rand(M, W), _rand(2 * F, W, scale=4 / 16), _rand(W, F, scale=1 / 45)
    plan = gemm.tile_plan(M, 2 * F, W, True)
    assert plan and plan[1] == 1
    with torch.no_grad():
        mid = linear_clipped(x, w, 3.0)
        ref = sublayer.clipped_glu(native().gemm_tile(x, w, False, *plan), 3.0)
        assert torch.equal(mid, ref)
        wgu, wdown = _rand(4, 128, W, scale=0.1), _rand(4, W, 64, scale=0.1)
        ids = torch.randint(0, 4, (M, 2), device="cuda", dtype=torch.int32)
        assert torch.equal(moe.experts(x, ids, wgu, wdown, 7.0, w, down, 3.0)[2], linear(ref, down))
    w.requires_grad_()  # a gradient is asked: the two ops
    assert linear_clipped(x, w, 3.0) is None


@pytest.mark.parametrize("T,N,K", [(_DECODE_M + 1, 16, 64), (47, 64, 128), (300, 48, 192), (2048, 64, 4096), (4099, 64, 320), (8192, 64, 64),
                                   (700, 256, 256)])
def test_side_gate(T, N, K):
    """One launch against the product and its activation, over ragged rows, a second block of channels that is not there, K of fewer
    stages than are in flight, strided rows and ids past the table."""
    torch.manual_seed(T)
    x, w = _rand(T, K + 8)[:, :K], _rand(N, K, scale=1 / K**0.5)
    emb = _rand(100, 4 + N + 12)
    ids = torch.randint(0, 100, (T,), device="cuda")
    ids[0], ids[1] = -3, 1000
    with torch.no_grad():
        y = sublayer.side_gate(x, w, emb, ids, 4)
    z = x.double() @ w.double().t()
    e = emb[ids.clamp(0, 99), 4:4 + N].double()
    ref = torch.nn.functional.gelu(z, approximate="tanh") * e
    # the product and the result are rounded to bf16 (2^-9 each; gelu's slope is below 1.13, f32 sums are far below that)
    bound = 2.0**-8 * (1.2 * z.abs() * e.abs() + ref.abs()) + 2.0**-16 * (1 + e.abs())
    assert bool(((y.double() - ref).abs() <= bound).all())


def test_side_gate_refusals():
    x, w, emb = _rand(64, 64), _rand(64, 64), _rand(10, 128)
    ids = torch.zeros(64, device="cuda", dtype=torch.long)
    with torch.no_grad():
        assert sublayer.side_gate(x, w, emb, ids, 64) is not None
        assert sublayer.side_gate(x[:_DECODE_M], w, emb, ids[:_DECODE_M], 64) is None  # a decode step's
        assert sublayer.side_gate(x, w[:24], emb, ids, 0) is None
        assert sublayer.side_gate(x, w, emb, ids, 2) is None  # (its columns are not on 8 bytes)
        assert sublayer.side_gate(x.float(), w.float(), emb.float(), ids, 0) is None
        assert sublayer.side_gate(x[:, 1:33], w[:, :32], emb, ids, 0) is None
    assert sublayer.side_gate(x, w.requires_grad_(), emb, ids, 0) is None


def test_switched_off(monkeypatch):
    """MXLLM_SUBLAYER_FUSED=0 is the parts in prompts too: none of the launches that join two."""
    torch.manual_seed(0)
    x, w, emb = _rand(128, 1024), _rand(64, 1024, scale=1 / 32), _rand(10, 64)
    ids = torch.zeros(128, device="cuda", dtype=torch.long)
    sgu, sdown, wgu, wdown = _rand(4096, 1024, scale=1 / 32), _rand(1024, 2048, scale=1 / 45), _rand(4, 128, 1024, scale=0.1), _rand(4, 1024, 64)
    pick = torch.randint(0, 4, (128, 2), device="cuda", dtype=torch.int32)
    taken = []
    monkeypatch.setattr(moe, "linear_clipped", lambda *a: taken.append("unit") or linear_clipped(*a))
    with torch.no_grad():
        for fused in (True, False):
            monkeypatch.setattr(sublayer, "FUSED", fused)
            for name, r in (("gate", sublayer.side_gate(x, w, emb, ids, 0)),
                            ("route", sublayer.post_route(x, x.float(), x[0].float(), 1e-6, _rand(4, 1024), 2))):
                if r is not None:
                    taken.append(name)
            moe.experts(x, pick, wgu, wdown, 7.0, sgu, sdown, 3.0)
            assert taken == (["gate", "route", "unit"] if fused else [])
            taken.clear()
