"""csrc/kernels/gemm_tile.hip: every tile at its edges, K of fewer tiles than stages, K in parts, SwiGLU, strided operands."""
import pytest
import torch

from mxllm import ops

pytestmark = pytest.mark.gpu

TILES = [(64, 64), (64, 128), (128, 128), (128, 192), (128, 256), (160, 192), (192, 192)]  # kGtTiles


def _operand(gpu, rows, K, seed):
    """Rows of a wider buffer whose other values are NaN: what is read beside them shows."""
    g = torch.Generator(device=gpu).manual_seed(seed)
    buf = torch.full((rows + 3, K + 72), float("nan"), device=gpu, dtype=torch.bfloat16)
    t = buf[1:1 + rows, 64:64 + K]
    t.copy_(torch.empty(rows, K, device=gpu).normal_(generator=g))
    return t


def _check(y, want, slack):
    """f32 sums of K products in some order are within K 2^-24 of the sum of their sizes (``slack``), and are rounded to bf16."""
    bound = 2.0 ** -8 * want.abs() + slack + 1e-30
    assert bool(((y.double() - want).abs() <= bound).all()), float(((y.double() - want).abs() / bound).max())


@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("K,parts", [(64, 1), (128, 1), (192, 1), (320, 1), (1088, 1), (1088, 3), (1088, 16)])
def test_tiles_at_their_edges(gpu, tile, K, parts):
    tm, tn = TILES[tile]
    for M, N in ((1, 16), (tm - 1, tn + 16), (tm, tn), (tm + 1, 2 * tn - 16)):
        a, b = _operand(gpu, M, K, 1), _operand(gpu, N, K, 2)
        want, size = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
        _check(ops.native().gemm_tile(a, b, False, tile, parts), want, K * 2.0 ** -24 * size)


@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("K,parts", [(128, 1), (576, 1), (576, 2)])
def test_swiglu_has_the_bits_of_two_passes(gpu, tile, K, parts):
    tm, tn = TILES[tile]
    for M, F in ((1, 8), (tm - 1, tn // 2 + 8), (tm + 1, tn)):
        a, b = _operand(gpu, M, K, 3), _operand(gpu, 2 * F, K, 4)
        y = ops.native().gemm_tile(a, b, True, tile, parts)
        assert torch.equal(y, ops.swiglu(ops.native().gemm_tile(a, b, False, tile, parts)))


@pytest.mark.parametrize("M", [9, 17, 33, 40, 300, 1030])
@pytest.mark.parametrize("N,K", [(64, 4096), (3360, 2048), (2048, 8192), (4096, 64)])
def test_linear_takes_any_rows(gpu, M, N, K):
    """Through ops.linear: prompt-sized rows beside each line, and the same bits in replays of a graph between eager calls."""
    a, b = _operand(gpu, M, K, 5), _operand(gpu, N, K, 6)
    want, size = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    y = ops.linear(a, b)
    _check(y, want, K * 2.0 ** -24 * size)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        z = ops.linear(a, b)
    for _ in range(3):
        z.zero_()
        g.replay()
        assert torch.equal(z, y) and torch.equal(ops.linear(a, b), y)


def test_refuses(gpu):
    a, b = _operand(gpu, 40, 128, 7), _operand(gpu, 32, 128, 8)
    f = ops.native().gemm_tile
    for args in ((a, b, False, 7, 1), (a, b, False, -1, 1), (a, b, False, 0, 3), (a, b, False, 0, 0), (a, b[:24], False, 0, 1),
                 (a[:, :96], b[:, :96], False, 0, 1), (a[:, 1:65], b[:, :64], False, 0, 1), (a, b[:, :64], False, 0, 1)):
        with pytest.raises(RuntimeError):
            f(*args)
