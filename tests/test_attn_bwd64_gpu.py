"""The attention backward for heads of 64 (csrc/kernels/attn_bwd64.hip) at the edges of its tiles (32 rows a wave, 64 a tile,
128 a workgroup), with masks that start and end inside them, against 64-bit sums of the same bf16 inputs."""
import math

import pytest
import torch

from mxllm.ops import reference as ref

pytestmark = pytest.mark.gpu
D = 64
# P and dS are rounded to bf16 (2^-9 of each at most, in both products and, through O, in delta): three such errors in a row
# are 6e-3 of a gradient's norm where none cancel; 1.6e-3 to 2.2e-3 were seen
REL = 6e-3


def _inputs(gpu, B, Hq, Hkv, S, Sk):
    torch.manual_seed(S * 7 + Sk)
    q, do = (torch.randn(B, Hq, S, D, device=gpu).bfloat16() for _ in range(2))
    k, v = (torch.randn(B, Hkv, Sk, D, device=gpu).bfloat16() for _ in range(2))
    return q, k, v, do.transpose(1, 2).reshape(B, S, Hq * D)


@pytest.mark.parametrize("B,Hq,Hkv,S,Sk,causal", [
    (1, 4, 2, 2, 2, True), (2, 4, 1, 31, 31, True), (1, 8, 2, 64, 64, True), (1, 4, 4, 65, 65, True), (2, 8, 2, 128, 128, True),
    (1, 16, 2, 129, 129, True), (1, 8, 8, 300, 300, True), (1, 4, 2, 33, 65, True), (1, 8, 2, 64, 320, True),
    (1, 4, 2, 1, 200, True), (1, 4, 2, 300, 100, True), (1, 4, 2, 100, 300, False), (2, 4, 2, 257, 63, False)])
def test_gradients(gpu, B, Hq, Hkv, S, Sk, causal):
    from mxllm.ops import native

    q, k, v, do = _inputs(gpu, B, Hq, Hkv, S, Sk)
    scale = 1.0 / math.sqrt(D)
    o, lse = native().attn_fwd(q, k, v, causal, scale)
    got = native().attn_bwd(do, q, k, v, o, lse, causal, scale, 3)
    qd = q.double()
    kd, vd = (t.double().repeat_interleave(Hq // Hkv, 1) for t in (k, v))
    s = qd @ kd.transpose(-1, -2).contiguous() * scale
    if causal:
        s = s.masked_fill(torch.ones(S, Sk, device=gpu).triu(Sk - S + 1).bool(), float("-inf"))
    p = torch.softmax(s, -1).nan_to_num(0.0)  # (rows that see no key)
    dod = do.view(B, S, Hq, D).transpose(1, 2).double()
    dp = dod @ vd.transpose(-1, -2).contiguous()
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * scale

    def per_kv(t):
        return t.reshape(B, Hkv, -1, Sk, D).sum(2)

    want = (ds @ kd, per_kv(ds.transpose(-1, -2).contiguous() @ qd), per_kv(p.transpose(-1, -2).contiguous() @ dod))
    for g, w in zip((got[0], per_kv(got[1]), per_kv(got[2])), want):
        assert float((g.double() - w).norm()) <= REL * float(w.norm())
    again = native().attn_bwd(do, q, k, v, o, lse, causal, scale, 3)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


@pytest.mark.parametrize("S,pad", [(96, 0), (129, 64)])
def test_into_dqkv(gpu, S, pad):
    """Gradients written straight into d(qkv) have the bits of f32 ones turned back by rope_merge_bwd."""
    from mxllm.ops import native

    B, Hq, Hkv, scale = 2, 8, 2, 1.0 / math.sqrt(D)
    q, k, v, do = _inputs(gpu, B, Hq, Hkv, S, S)
    cos, sin = ref.rope_tables(S, D, 500000.0, None, gpu)
    o, lse = native().attn_fwd(q, k, v, True, scale)
    dq, dk, dv = native().attn_bwd(do, q, k, v, o, lse, True, scale, 3)
    want = native().rope_merge_bwd(dq, dk, dv, cos, sin, B, S, Hq, Hkv, D, pad)
    got = native().attn_bwd_rope(do, q, k, v, o, lse, True, scale, cos, sin, pad)
    n = (Hq + 2 * Hkv) * D
    assert got.stride() == want.stride() and torch.equal(got[:, :n], want[:, :n])


def test_long_rows_of_many_heads(gpu):
    """dO of one sequence past 4 GiB, which no byte offset of 32 bits reaches: the bits of calls of 32 heads each."""
    from mxllm.ops import native

    Hq, S, Sk = 128, 262_209, 40
    torch.manual_seed(1)
    q, o, do = (torch.randn(s, device=gpu, dtype=torch.bfloat16) for s in ((1, Hq, S, D), (1, S, Hq * D), (1, S, Hq * D)))
    k, v = (torch.randn(1, Hq // 32, Sk, D, device=gpu, dtype=torch.bfloat16) for _ in range(2))
    lse = torch.full((1, Hq, S), math.log2(Sk) + 1, device=gpu)
    assert (S - 1) * Hq * D * 2 > 2**32
    got = native().attn_bwd(do, q, k, v, o, lse, False, 0.125, 3)
    for i in range(0, Hq, 32):
        part = [t.view(1, S, Hq, D)[:, :, i:i + 32].reshape(1, S, 32 * D).contiguous() for t in (do, o)]
        want = native().attn_bwd(part[0], q[:, i:i + 32], k[:, i // 32:i // 32 + 1], v[:, i // 32:i // 32 + 1], part[1],
                                 lse[:, i:i + 32], False, 0.125, 3)
        assert all(torch.equal(g[:, i:i + 32], w) and bool(torch.isfinite(w).all()) for g, w in zip(got, want))
