"""csrc/kernels/stream_hybrid.hip (through ``hybrid.gru_linear`` / ``conv_linear``): the mixers' projections on the workgroups that
stay, on both sides of their limits in rows, widths and norm parts, against the norm, the product and the step one after the other."""
import pytest
import torch

from mxllm import ops
from mxllm.ops import hybrid as hops

pytestmark = pytest.mark.gpu

# two roundings to bf16 of either side's f32 sums, which are in another order: 2 * 2^-8
TOL = 2 ** -7


def _near(a, b):
    err = float((a.double() - b.double()).norm() / b.double().norm())
    assert err < TOL, err


def _rows(gpu, M, K, groups, parts, add):
    g = torch.Generator(device=gpu).manual_seed(M + K)
    # parts of unlike size: a wave that took its neighbour's would show
    h = torch.empty(M, K, device=gpu).normal_(generator=g) * torch.logspace(-2, 2, groups, device=gpu).repeat_interleave(K // groups)
    gamma = torch.empty(K, device=gpu).uniform_(0.5, 1.5, generator=g)
    delta = torch.empty(M, K + 8, device=gpu).normal_(generator=g).bfloat16()[:, :K] if add else None
    if parts and add:
        delta = torch.empty(3, M, K, device=gpu).normal_(generator=g)
    return delta, h, gamma


CASES = [(M, K, groups, False, add) for M in (1, 2, 3, 4, 5, 8, 9, 10, 16) for K in (2048, 4096) for groups, add in ((8, True), (8, False))]
CASES += [(2, 2048, 4, False, True), (4, 1024, 8, False, True), (9, 2048, 8, True, True), (17, 2048, 8, False, True)]


@pytest.mark.parametrize("M,K,groups,parts,add", CASES)
@pytest.mark.parametrize("W", [36, 2048])
def test_gru(gpu, M, K, groups, parts, add, W):
    delta, h, gamma = _rows(gpu, M, K, groups, parts, add)
    g = torch.Generator(device=gpu).manual_seed(W)
    w = (torch.empty(3 * W, K, device=gpu).normal_(generator=g) * K ** -0.5).bfloat16()
    bias, state = torch.empty(2 * W, device=gpu).normal_(generator=g), torch.empty(M + 2, W, device=gpu).normal_(generator=g)
    slots = torch.arange(M + 1, 1, -1, device=gpu, dtype=torch.int32)
    pos = torch.full((M,), 5, device=gpu, dtype=torch.int32)
    outs = []
    for fused in (True, False):
        hh, s = h.clone(), state.clone()
        rows = hops.TokenRows(pos, slots, 64, hops.SeqCaches([], [], None, [], [s]))
        if fused:
            r = hops.gru_linear(delta, hh, gamma, groups, 1e-3, w, bias, rows, 0)
            if r is None:
                assert M > (16 if K == 2048 else 8)
                return
            y, hn = r
        else:
            y, hn = hops.min_gru(ops.linear(hops.group_norm(delta, hh, gamma, groups, 1e-3, torch.bfloat16), w), bias, rows, 0), hh
        outs.append((y, hn, s))
    (y, hn, s), (y2, hn2, s2) = outs
    assert torch.equal(hn, hn2) and torch.equal(s[:2], state[:2])
    _near(y, y2)
    _near(s[2:], s2[2:])


@pytest.mark.parametrize("M,K,groups,parts,add", CASES)
@pytest.mark.parametrize("H,G,D", [(4, 2, 32), (32, 8, 64)])
def test_conv(gpu, M, K, groups, parts, add, H, G, D):
    delta, h, gamma = _rows(gpu, M, K, groups, parts, add)
    g = torch.Generator(device=gpu).manual_seed(H)
    sh = hops.AttnShape(H, G, D, D, 4, 64, D // 2, D ** -0.5)
    C = sh.conv_channels
    w = (torch.empty(C + H * D, K, device=gpu).normal_(generator=g) * K ** -0.5).bfloat16()
    conv = torch.empty(4, C, device=gpu).normal_(generator=g)
    ang = torch.empty(80, D // 4, device=gpu).uniform_(0, 6, generator=g)
    kv = torch.empty(2, M + 2, G, 256, D, device=gpu).normal_(generator=g).bfloat16()
    ring = torch.empty(M + 2, 4, C, device=gpu).normal_(generator=g).bfloat16()
    bt = torch.arange(M + 2, device=gpu, dtype=torch.int32).flip(0)[:, None].contiguous()
    slots = torch.arange(M + 1, 1, -1, device=gpu, dtype=torch.int32)
    pos = (torch.arange(M, device=gpu, dtype=torch.int32) * 7) % 70  # from 0: fewer earlier values than taps; past a chunk
    outs = []
    for fused in (True, False):
        hh, c, r = h.clone(), kv.clone(), ring.clone()
        rows = hops.TokenRows(pos, slots, 64, hops.SeqCaches([c[0]], [c[1]], bt, [r], []))
        if fused:
            out = hops.conv_linear(delta, hh, gamma, groups, 1e-3, w, conv, ang.cos(), ang.sin(), sh, rows, 0)
            if out is None:
                assert M > (16 if K == 2048 else 8)
                return
            y, hn = out
        else:
            x = ops.linear(hops.group_norm(delta, hh, gamma, groups, 1e-3, torch.bfloat16), w)
            y, hn = hops.sink_attention(x, conv, ang.cos(), ang.sin(), sh, rows, 0), hh
        outs.append((y, hn, c, r))
    (y, hn, c, r), (y2, hn2, c2, r2) = outs
    assert torch.equal(hn, hn2) and torch.equal(r[:2], ring[:2])
    for a, b in ((y, y2), (c, c2), (r, r2)):
        _near(a, b)
    # what no row wrote is as it was
    assert int((c != kv).any(-1).sum()) <= 2 * M * G and int((r != ring).any(-1).sum()) <= M


@pytest.mark.parametrize("M", [8, 9, 16])
def test_rows_past_the_kernels_of_a_width(gpu, monkeypatch, M):
    """A limit of 16 rows of a width of 4096: what the workgroups that stay leave to csrc/kernels/hybrid_skinny.hip."""
    monkeypatch.setattr(hops, "SKINNY_M", 16)
    test_gru(gpu, M, 4096, 8, False, True, 36)
    test_conv(gpu, M, 4096, 8, False, True, 4, 2, 32)
