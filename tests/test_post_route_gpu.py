"""The residual step behind a prompt's mixer with the router's choices, against the two launches."""
import pytest
import torch

from mxllm.ops import moe, sublayer
from mxllm.ops._ext import native
from mxllm.ops.linear import _DECODE_M

pytestmark = pytest.mark.gpu


def _case(T, W, E):
    g = torch.Generator(device="cuda")
    g.manual_seed(T + W)

    def rand(*shape):
        return torch.randn(*shape, device="cuda", generator=g)

    return rand(T, W + 4).bfloat16()[:, :W], rand(T, W), 1 + 0.1 * rand(W), (rand(E, W) * W**-0.5).bfloat16()


@pytest.mark.parametrize("T,W,E,top", [(_DECODE_M + 1, 1024, 16, 4), (47, 3072, 7, 7), (300, 2048, 16, 1), (2048, 4096, 16, 4), (2709, 2048, 16, 4),
                                       (41, 4096, 1, 1), (5001, 4096, 13, 3)])
def test_post_route_is_the_two_launches(T, W, E, top):
    """Ragged rows, every width, fewer experts than a tile, all of them chosen, strided rows, infinities and NaN: the same bits."""
    src, h, w, router = _case(T, W, E)
    src[3, 5], h[9, 0], h[T - 1, W - 1] = float("inf"), float("nan"), float("-inf")
    h2 = h.clone()
    with torch.no_grad():
        x = native().post_norm(src, h2, w, 1e-5)
        ids, wts = moe.route(x, router, top)
        got = sublayer.post_route(src, h, w, 1e-5, router, top)
    for a, b in zip((*got, h), (x, ids, wts, h2)):
        torch.testing.assert_close(a, b, rtol=0, atol=0, equal_nan=True)


def test_post_route_refusals():
    src, h, w, router = _case(40, 1024, 8)
    kept = h.clone()
    with torch.no_grad():
        assert sublayer.post_route(src[:_DECODE_M], h[:_DECODE_M], w, 1e-5, router, 2) is None
        assert sublayer.post_route(src.float(), h, w, 1e-5, router, 2) is None
        assert sublayer.post_route(src, h, w, 1e-5, torch.cat([router] * 3), 2) is None  # (24 experts)
        assert sublayer.post_route(_case(40, 1025, 8)[0][:, 1:], h, w, 1e-5, router, 2) is None
        for W in (512, 1536, 5120):
            assert sublayer.post_route(*_case(40, W, 8)[:3], 1e-5, _case(40, W, 8)[3], 2) is None
    assert sublayer.post_route(src, h, w, 1e-5, router.requires_grad_(), 2) is None
    assert torch.equal(h, kept)
