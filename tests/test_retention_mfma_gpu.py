"""Retention of prompts on the bf16 matrix cores (csrc/kernels/retention_mfma.hip): against 64-bit sums of the same operands, next to
the f32 matrix cores' (csrc/kernels/retention_chunk.hip, which takes rows that are not 16 bytes apart)."""
import pytest
import torch

from mxllm.ops import hybrid as hops
from mxllm.ops import retention as rops

pytestmark = pytest.mark.gpu
EPS = 1e-5


class _Caches:
    def __init__(self, n, width, fill):
        self.rec = [torch.full((n, width), fill, device="cuda")]


def _inputs(H, D, E, lens, seed=0):
    torch.manual_seed(seed)
    x = torch.randn(sum(lens), 2 * H * (D + E), device="cuda").bfloat16()
    decay = [1 - 2.0 ** (-5 - 7 * j / max(H - 1, 1)) for j in range(H)]
    ang = torch.arange(max(lens)).double()[:, None] * 1e4 ** (-torch.arange(D // 2).double() / (D // 2))
    return x, decay, ang.cos().float().cuda(), ang.sin().float().cuda()


def _exact(x, decay, cos, sin, H, D, E, lens):
    """Outputs ahead of the gate, gates and last states, all in f64."""
    q, k, v, gate = x.double().split([H * D] * 2 + [H * E] * 2, 1)
    d = torch.tensor(decay, dtype=torch.float64, device="cuda")
    outs, states, off = [], [], 0
    for n in lens:
        c, s = cos[:n].double()[:, None], sin[:n].double()[:, None]

        def rot(t):
            u, w = t[off:off + n].reshape(n, H, D).chunk(2, -1)
            return torch.cat([u * c - w * s, w * c + u * s], -1).transpose(0, 1).contiguous()

        Q, K, V = rot(q), rot(k) * D ** -0.5, v[off:off + n].reshape(n, H, E).transpose(0, 1).contiguous()
        i = torch.arange(n, device="cuda")
        back = i[:, None] - i[None]
        P = (Q @ K.transpose(1, 2).contiguous()) * torch.where(back >= 0, d[:, None, None] ** back.clamp(min=0), 0.0)
        outs.append((P @ V).transpose(0, 1))
        states.append((K * (d[:, None] ** (n - 1 - i))[..., None]).transpose(1, 2).contiguous() @ V)
        off += n
    o = torch.cat(outs)
    o = o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + EPS)
    return (o.reshape(sum(lens), H * E) * torch.nn.functional.silu(gate)), torch.stack(states)


def _run(x, decay, cos, sin, H, D, E, lens, keep=True):
    caches = _Caches(len(lens) + 1, H * D * E, 7.0)
    rows = hops.PromptRows(lens, "cuda", list(range(len(lens))), caches) if keep else hops.PromptRows(lens, "cuda")
    y = rops.retention(x, rops.decay_table(decay, "cuda"), cos, sin, rops.RetentionShape(H, D, E, D), EPS, rows, 0)
    assert bool((caches.rec[0][-1] == 7).all())
    return y, caches.rec[0][:-1].view(len(lens), H, D, E)


@pytest.mark.parametrize("D,E", [(64, 64), (64, 128), (128, 64), (128, 128)])
@pytest.mark.parametrize("lens", [[1], [31, 1, 33], [128, 129, 127], [256, 255, 257], [225, 700], [1300]])
def test_against_64_bits(D, E, lens):
    H = 3
    x, decay, cos, sin = _inputs(H, D, E, lens)
    ref, state = _exact(x, decay, cos, sin, H, D, E, lens)
    wide = torch.nn.functional.pad(x, (0, 4))[:, :-4]  # rows 8 bytes off: the f32 matrix cores
    y, S = _run(x, decay, cos, sin, H, D, E, lens)
    y0, S0 = _run(wide, decay, cos, sin, H, D, E, lens)
    # A run's sums have 32 roundings of f32 and more (rotations, scores, powers of the decay), 2^-24 each of the terms' sizes;
    # outputs one of bf16, 2^-9 of theirs, behind a norm that leaves their relative error.
    assert float((S - state).norm()) <= 2.0 ** -20 * float(state.norm())
    assert float((y.double() - ref).norm()) <= 2.0 ** -9 * float(ref.norm())
    off, off0 = ((t != ref.bfloat16()).double().mean().item() for t in (y, y0))  # not the nearest bf16 of the exact value
    err, err0 = (float((t - state).norm() / state.norm()) for t in (S, S0))
    assert err <= 1.1 * err0 + 2.0 ** -26 and off <= 1.25 * off0 + 4 / y.numel()
    alone, _ = _run(x, decay, cos, sin, H, D, E, lens, keep=False)  # no state is kept: the same outputs
    assert torch.equal(alone, y)


def test_rows_do_not_see_later_ones():
    H, D, E, n = 2, 128, 128, 300
    x, decay, cos, sin = _inputs(H, D, E, [n])
    y, _ = _run(x, decay, cos, sin, H, D, E, [n])
    z = x.clone()
    z[200:] = float("inf")
    w, _ = _run(z, decay, cos, sin, H, D, E, [n])
    assert torch.equal(w[:192], y[:192])  # (rows of one tile of 32 keys share its products of zero scores)


@pytest.mark.parametrize("D,E", [(64, 64), (64, 128), (128, 64), (128, 128)])
@pytest.mark.parametrize("what", ["v", "-v", "k", "q", "nan"])
def test_not_finite(D, E, what):
    """What is not finite in a row's outputs and in the states, and what is zero or untouched beside it, is as with the f32
    matrix cores (whose waves take zero products of later keys too: it starts where a tile of 32 keys does)."""
    H, lens = 3, [300, 40, 700]
    x, decay, cos, sin = _inputs(H, D, E, lens)
    bad = float(what.replace("-v", "-inf").replace("v", "inf").replace("k", "inf").replace("q", "inf"))
    col = {"q": D + 5, "k": H * D + D + 5, "nan": H * D + D + 5}.get(what, 2 * H * D + E + 5)
    for row in (64, 340 + 352):  # of the first sequence, and of the last one's second run
        x[row, col] = bad
    wide = torch.nn.functional.pad(x, (0, 4))[:, :-4]
    (y, S), (y0, S0) = _run(x, decay, cos, sin, H, D, E, lens), _run(wide, decay, cos, sin, H, D, E, lens)
    assert 0 < int((~y0.isfinite()).sum()) and int((~y0[:, :E].isfinite()).sum()) == 0  # head 1 alone
    for a, b in ((y, y0), (S, S0)):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a == 0, b == 0)
        assert torch.equal(a.isinf(), b.isinf()) and torch.equal(a[a.isinf()], b[b.isinf()])
        a, b = a[a.isfinite()].double(), b[b.isfinite()].double()
        assert float((a - b).norm()) <= 2.0 ** -8 * float(b.norm())
