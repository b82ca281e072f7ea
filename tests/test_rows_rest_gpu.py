"""Gate-up projections of prompts whose last turn of tiles is mostly empty."""
import pytest
import torch

from mxllm.ops import gemm
from mxllm.ops._ext import native
from mxllm.ops.linear import linear_swiglu


def test_lines():
    on = [(1025, 16384, 2048), (1536, 16384, 2048), (2300, 16384, 2048), (4400, 16384, 2048), (1100, 16384, 1024)]
    off = [(1024, 16384, 2048), (1537, 16384, 2048), (2709, 16384, 2048), (2048, 16384, 2048), (700, 16384, 2048), (2300, 16384, 2112),
           (4400, 28672, 4096), (5000, 16384, 1024)]  # (the last: five turns, the last of them ragged)
    assert all(gemm.rows_head(*s) for s in on) and not any(gemm.rows_head(*s) for s in off)


def test_lines_follow_the_switch(monkeypatch):
    """MXLLM_GEMM8 is read at each call: what one answer was under it does not stay for the next."""
    monkeypatch.setenv("MXLLM_GEMM8", "0")
    assert gemm.rows_head(1309, 16384, 2048) is None
    monkeypatch.setenv("MXLLM_GEMM8", "table")
    assert gemm.rows_head(1309, 16384, 2048)
    monkeypatch.setenv("MXLLM_GEMM8", "0")
    assert gemm.rows_head(1309, 16384, 2048) is None


@pytest.mark.gpu
@pytest.mark.parametrize("M,F,K", [(1025, 8192, 128), (1300, 8192, 256), (1536, 8192, 64), (2050, 8192, 192), (3073, 4096, 128), (1700, 5120, 128)])
def test_rest_is_whole(M, F, K):
    """K in order in either kernel: the bits are those of one launch, the last row's and the first's behind the cut among them."""
    torch.manual_seed(M)
    x, w = torch.randn(M, K + 8, device="cuda").bfloat16()[:, :K], (torch.randn(2 * F, K, device="cuda") * K**-0.5).bfloat16()
    whole = native().gemm8_rows(x, w, True, True, 1)
    for head, tile in [gemm.rows_head(M, 2 * F, K) or (256, 0), (M // 256 * 256 if M % 256 else M - 256, 3), (256, 4)]:
        assert torch.equal(native().gemm8_rows_rest(x, w, head, tile), whole)
    with torch.no_grad():
        assert torch.equal(linear_swiglu(x, w), whole)
