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


def test_short_products_stay_where_measured():
    """1,024 rows on, less than two turns; there gemm_tile has no plan that a caller would have to ask for first."""
    off = [(33, 128256, 512), (64, 65536, 256), (127, 65536, 384), (300, 32768, 512), (1023, 16384, 512), (1024, 32768, 256),
           (4096, 8192, 512), (2048, 16384, 256), (4096, 16384, 384)]
    assert not any(gemm.rows_gain(*s, True) for s in off)
    on = [(M, N, K) for M in (1024, 1100, 1700, 2500, 4090, 5900) for N in range(2048, 20000, 768) for K in (256, 320, 512)
          if gemm.rows_gain(M, N, K, True)]
    assert len(on) > 50 and not any(gemm.tile_plan(*s) for s in on)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1281, 8192, 512), (2709, 4096, 256), (1700, 6144, 384)])
def test_short_products(M, N, K):
    """K in order in either kernel."""
    torch.manual_seed(M)
    x, w = torch.randn(M, K + 64, device="cuda").bfloat16()[:, :K], (torch.randn(N, K, device="cuda") * K**-0.5).bfloat16()
    with torch.no_grad():
        assert torch.equal(linear(x, w), native().gemm_tile(x, w, False, 4, 1))
