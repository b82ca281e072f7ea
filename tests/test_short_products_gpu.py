"""Projections of a short K: both sides of the line to gemm8."""
import pytest
import torch

from mxllm.ops import gemm
from mxllm.ops._ext import native
from mxllm.ops.linear import linear


def test_lines():
    on = [(1400, 8192, 512), (2709, 8192, 512), (2709, 4096, 256)]
    off = [(1280, 8192, 512), (2709, 8192, 576), (2709, 8192, 192), (2500, 4096, 256)]
    assert all(gemm.rows_gain(*s, True) == 1 for s in on) and not any(gemm.rows_gain(*s, True) for s in off)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1281, 8192, 512), (2709, 4096, 256), (1700, 6144, 384)])
def test_short_products(M, N, K):
    """K in order in either kernel."""
    torch.manual_seed(M)
    x, w = torch.randn(M, K + 64, device="cuda").bfloat16()[:, :K], (torch.randn(N, K, device="cuda") * K**-0.5).bfloat16()
    with torch.no_grad():
        assert torch.equal(linear(x, w), native().gemm_tile(x, w, False, 4, 1))
