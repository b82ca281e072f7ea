"""Products of prompt passes that end in their activation, against the two launches."""
import pytest
import torch

from mxllm.ops import gemm, moe, sublayer
from mxllm.ops._ext import native
from mxllm.ops.linear import linear, linear_clipped

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
