"""HIP kernel numerics vs plain-PyTorch fp32 references.

Random (never zero) data, odd shapes where the kernel supports them.
"""
import math

import pytest
import torch

from mxllm.ops import reference as ref

pytestmark = pytest.mark.gpu


def _ops():
    from mxllm.ops import native

    return native()


def rel_err(a, b):
    a, b = a.float(), b.float()
    return ((a - b).norm() / (b.norm() + 1e-12)).item()


@pytest.mark.parametrize("T,H", [(1, 64), (37, 512), (512, 4096), (64, 8192), (3, 16384)])
def test_rmsnorm_fwd_bwd(gpu, T, H):
    torch.manual_seed(0)
    x = torch.randn(T, H, device=gpu, dtype=torch.bfloat16)
    w = (1 + 0.1 * torch.randn(H, device=gpu)).to(torch.bfloat16)
    y, rstd, _ = _ops().rmsnorm_fwd(x, None, w, 1e-5)
    xf = x.float().requires_grad_(True)
    wf = w.float().requires_grad_(True)
    yr = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-5) * wf
    assert rel_err(y, yr) < 1e-2
    dy = torch.randn_like(x)
    yr.backward(dy.float())
    dres = torch.randn_like(x)
    dx, dw = _ops().rmsnorm_bwd(dy, x, w, rstd, dres, True)
    assert rel_err(dx, xf.grad + dres.float()) < 1e-2
    assert rel_err(dw, wf.grad) < 1e-3


@pytest.mark.parametrize("T,H", [(1, 8), (33, 1000), (700, 2048), (20000, 72)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rmsnorm_backward_into_slot(gpu, T, H, dtype):
    """The weight's gradient over or onto what an owner's slot held, rounded once."""
    x, dy = torch.randn(2, T, H, device=gpu).to(torch.bfloat16)
    w = torch.ones(H, device=gpu, dtype=torch.bfloat16)
    _, rstd, _ = _ops().rmsnorm_fwd(x, None, w, 1e-5)
    dx, dw = _ops().rmsnorm_bwd(dy, x, w, rstd, None, True)
    old = torch.randn(H, device=gpu).to(dtype)
    for add in (False, True):
        buf = torch.cat([old, old.new_full((8,), 3.0)])
        slot = buf[:H]
        dx2, none = _ops().rmsnorm_bwd(dy, x, w, rstd, None, True, 0, slot, add)
        assert none is None and torch.equal(dx, dx2) and (buf[H:] == 3.0).all()
        assert torch.equal(slot, (old.float() + dw if add else dw).to(dtype))  # the same sum, one rounding


def test_add_rmsnorm(gpu):
    torch.manual_seed(1)
    x = torch.randn(300, 1024, device=gpu, dtype=torch.bfloat16)
    r = torch.randn_like(x)
    w = torch.randn(1024, device=gpu, dtype=torch.bfloat16)
    y, rstd, h = _ops().rmsnorm_fwd(x, r, w, 1e-5)
    href = (x.float() + r.float()).to(torch.bfloat16)
    assert torch.equal(h, href)
    assert rel_err(y, ref.rms_norm(href, w, 1e-5).float()) < 1e-2


@pytest.mark.parametrize("T,F", [(1, 8), (129, 1024), (1024, 14336)])
def test_swiglu(gpu, T, F):
    torch.manual_seed(2)
    gu = torch.randn(T, 2 * F, device=gpu, dtype=torch.bfloat16)
    m = _ops().swiglu_fwd(gu)
    guf = gu.float().requires_grad_(True)
    mr = torch.nn.functional.silu(guf[:, :F]) * guf[:, F:]
    assert rel_err(m, mr) < 1e-2
    dm = torch.randn_like(m)
    mr.backward(dm.float())
    dgu = _ops().swiglu_bwd(dm, gu)
    assert rel_err(dgu, guf.grad) < 1e-2
    # the recompute backward: same dgu and bitwise the forward's m from one pass over gu
    dgu2, m2 = _ops().swiglu_bwd_m(dm, gu)
    assert torch.equal(dgu2, dgu) and torch.equal(m2, m)


@pytest.mark.parametrize("rbw", ["1", "2", "4"])
@pytest.mark.parametrize("bwd", [False, True])
@pytest.mark.parametrize("T,F,R", [(16, 128, 16), (48, 384, 32), (1024, 1536, 48), (256, 256, 64), (4096, 28672, 16)])
def test_swiglu_lora_tail(gpu, T, F, R, bwd, rbw, monkeypatch):
    """SwiGLU fused with the neighbour's LoRA tail (csrc/kernels/lora.hip swiglu_lora_kernel):
    the SwiGLU output is bitwise the plain kernel's, the tail is s out V[:R]^T against fp32,
    zeros past R (V rows past R deliberately non-zero), bit-reproducible."""
    from mxllm.ops.linear import _padded_rows

    monkeypatch.setenv("MXLLM_SWIGLU_LORA_RBW", rbw)  # 16-row blocks per workgroup (clamped to T)
    torch.manual_seed(4)
    pad, s = 64, 2.0
    gu = torch.randn(T, 2 * F, device=gpu, dtype=torch.bfloat16)
    W = 2 * F if bwd else F
    V = torch.randn(pad, W + 24, device=gpu, dtype=torch.bfloat16)[:, :W]  # padded row stride
    dm = torch.randn(T, F, device=gpu, dtype=torch.bfloat16) if bwd else None
    out = _ops().swiglu_lora(dm, gu, pad, V, R // 16, s)
    plain = _ops().swiglu_bwd(dm, gu) if bwd else _ops().swiglu_fwd(gu)
    assert torch.equal(out, plain)
    full = _padded_rows(out, pad)
    assert full is not None
    tail = full[:, W:]
    ref_tail = s * (out.float() @ V[:R].float().t())
    assert rel_err(tail[:, :R], ref_tail) < 1e-2
    assert not tail[:, R:].any()
    again = _padded_rows(_ops().swiglu_lora(dm, gu, pad, V, R // 16, s), pad)
    assert torch.equal(again[:, W:], tail)


def test_attention_bwd_bounded_ds_image(gpu, monkeypatch):
    """Long-context memory bound: with the split-mode dS^T image over budget, the backward runs per
    (sequence, KV-group chunk) and gives the one-call dQ, and per-KV-head dK / dV (partials summed),
    to fp32 rounding."""
    from mxllm.ops import attention as A

    torch.manual_seed(11)
    B, Hq, Hkv, S, D = 2, 8, 2, 512, 128
    q = torch.randn(B, Hq, S, D, device=gpu, dtype=torch.bfloat16)
    k = torch.randn(B, Hkv, S, D, device=gpu, dtype=torch.bfloat16)
    v = torch.randn(B, Hkv, S, D, device=gpu, dtype=torch.bfloat16)
    sc = 1 / math.sqrt(D)
    o, lse = _ops().attn_fwd(q, k, v, True, sc)
    do = torch.randn(B * S, Hq * D, device=gpu, dtype=torch.bfloat16)
    ref_dq, ref_dk, ref_dv = _ops().attn_bwd(do, q, k, v, o, lse, True, sc, 3)
    monkeypatch.setattr(A, "_DS_BUDGET", 1.5 * 2**20)  # < one KV group's image: 4 chunks of 4 heads
    dq, dk, dv = A.attn_bwd(do, q, k, v, o, lse, True, sc, 3)
    assert dq.shape == ref_dq.shape
    assert rel_err(dq, ref_dq) < 1e-5

    def per_kv(t):
        return t.view(B, Hkv, -1, S, D).sum(2)

    assert rel_err(per_kv(dk), per_kv(ref_dk)) < 1e-5
    assert rel_err(per_kv(dv), per_kv(ref_dv)) < 1e-5


@pytest.mark.parametrize("T,V", [(5, 1000), (256, 128256)])
def test_cross_entropy(gpu, T, V):
    torch.manual_seed(3)
    logits = (3 * torch.randn(T, V, device=gpu)).to(torch.bfloat16)
    labels = torch.randint(0, V, (T,), device=gpu)
    labels[1] = -100
    lf = logits.float().requires_grad_(True)
    lr_ = torch.nn.functional.cross_entropy(lf, labels, ignore_index=-100)
    lr_.backward()
    work = logits.clone()
    loss, _ = _ops().ce_fwd_bwd(work, labels, -100)
    assert abs(loss.item() - lr_.item()) < 1e-3 * max(1.0, abs(lr_.item()))
    assert rel_err(work, lf.grad) < 1e-2
    assert work[1].abs().max().item() == 0.0


@pytest.mark.parametrize("gdt", [torch.float32, torch.bfloat16])
def test_adamw(gpu, gdt):
    torch.manual_seed(4)
    n = 10000 * 4
    p = torch.randn(n, device=gpu)
    g = torch.randn(n, device=gpu).to(gdt)
    m = torch.randn(n, device=gpu).abs() * 0.1
    v = torch.randn(n, device=gpu).abs() * 0.1
    pr, mr, vr = p.clone(), m.clone(), v.clone()
    lowp = torch.empty(n, device=gpu, dtype=torch.bfloat16)
    kw = dict(lr=1e-3, beta1=0.9, beta2=0.95, eps=1e-8, weight_decay=0.1, step=3)
    ref.adamw_(pr, g, mr, vr, grad_scale=0.5, **kw)
    from mxllm.ops import adamw_step_

    g0 = g.clone()
    adamw_step_(p, g, m, v, lowp, grad_scale=torch.tensor([0.5], device=gpu), **kw)
    assert rel_err(p, pr) < 1e-6 and rel_err(m, mr) < 1e-6 and rel_err(v, vr) < 1e-6
    assert torch.equal(lowp, p.to(torch.bfloat16))
    assert torch.equal(g, g0)  # untouched without zero_grad
    # fused gradient clearing: same update, gradient zeroed in the same pass
    p2, m2, v2 = p.clone(), m.clone(), v.clone()
    p3, m3, v3 = p.clone(), m.clone(), v.clone()
    adamw_step_(p2, g, m2, v2, None, grad_scale=0.5, **kw)
    adamw_step_(p3, g, m3, v3, None, grad_scale=0.5, zero_grad=True, **kw)
    assert torch.equal(p2, p3) and torch.equal(m2, m3) and torch.equal(v2, v3)
    assert g.abs().max().item() == 0.0


def test_embedding(gpu):
    torch.manual_seed(5)
    V, H, T = 1000, 512, 333
    w = torch.randn(V, H, device=gpu, dtype=torch.bfloat16)
    ids = torch.randint(0, V, (T,), device=gpu)
    out = _ops().embedding_fwd(ids, w)
    assert torch.equal(out, w[ids])
    dy = torch.randn(T, H, device=gpu, dtype=torch.bfloat16)
    dw = _ops().embedding_bwd(dy, ids, V)
    dref = torch.zeros(V, H, device=gpu).index_add_(0, ids, dy.float())
    assert rel_err(dw, dref) < 1e-5


@pytest.mark.parametrize("D", [32, 64, 128])
def test_rope_split_merge(gpu, D):
    torch.manual_seed(6)
    B, S, Hq, Hkv = 2, 70, 8, 2
    cos, sin = ref.rope_tables(256, D, 500000.0, {"factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                                                    "original_max_position_embeddings": 8192}, gpu)
    qkv = torch.randn(B * S, (Hq + 2 * Hkv) * D, device=gpu, dtype=torch.bfloat16)
    q, k, v = _ops().rope_split(qkv, cos, sin, B, S, Hq, Hkv, D)
    x = qkv.view(B, S, Hq + 2 * Hkv, D)
    qr = ref.apply_rope(x[:, :, :Hq], cos, sin).transpose(1, 2)
    kr = ref.apply_rope(x[:, :, Hq:Hq + Hkv], cos, sin).transpose(1, 2)
    assert rel_err(q, qr) < 1e-2 and rel_err(k, kr) < 1e-2
    assert torch.equal(v, x[:, :, Hq + Hkv:].transpose(1, 2).contiguous())
    # backward: merge(dq, dk partials per q head, dv partials) == autograd of split+rope+GQA-repeat
    xf = qkv.float().view(B, S, Hq + 2 * Hkv, D).requires_grad_(True)
    qf = ref.apply_rope(xf[:, :, :Hq], cos, sin).transpose(1, 2)
    kf = ref.apply_rope(xf[:, :, Hq:Hq + Hkv], cos, sin).transpose(1, 2).repeat_interleave(Hq // Hkv, 1)
    vf = xf[:, :, Hq + Hkv:].transpose(1, 2).repeat_interleave(Hq // Hkv, 1)
    dq = torch.randn(B, Hq, S, D, device=gpu)
    dkp = torch.randn(B, Hq, S, D, device=gpu)
    dvp = torch.randn(B, Hq, S, D, device=gpu)
    (qf * dq + kf * dkp + vf * dvp).sum().backward()
    dqkv = _ops().rope_merge_bwd(dq, dkp, dvp, cos, sin, B, S, Hq, Hkv, D)
    assert rel_err(dqkv, xf.grad.view(B * S, -1)) < 1e-2


ATTN_SHAPES = [
    (1, 4, 1, 128, 128, 128, True),
    (2, 8, 2, 200, 200, 128, True),
    (1, 8, 8, 256, 256, 64, False),
    (1, 4, 2, 77, 77, 32, True),
    (2, 16, 2, 512, 512, 128, True),
    (1, 8, 2, 64, 320, 128, True),   # prefill with a cached prefix (bottom-right causal)
    (1, 4, 2, 100, 300, 128, False),  # non-causal, key tail past the last full 64-key tile
    (1, 4, 1, 700, 700, 128, True),   # several 256-row query blocks, partial last block
]


@pytest.mark.parametrize("B,Hq,Hkv,S,Sk,D,causal", ATTN_SHAPES)
def test_attention_fwd_bwd(gpu, B, Hq, Hkv, S, Sk, D, causal):
    torch.manual_seed(7)
    q = torch.randn(B, Hq, S, D, device=gpu, dtype=torch.bfloat16)
    k = torch.randn(B, Hkv, Sk, D, device=gpu, dtype=torch.bfloat16)
    v = torch.randn(B, Hkv, Sk, D, device=gpu, dtype=torch.bfloat16)
    scale = 1.0 / math.sqrt(D)
    o, lse = _ops().attn_fwd(q, k, v, causal, scale)
    qf, kf, vf = [t.float().requires_grad_(True) for t in (q, k, v)]
    orf = ref.attention(qf.transpose(1, 2), kf.transpose(1, 2), vf.transpose(1, 2), causal=causal)  # [B,S,Hq,D]
    assert rel_err(o.view(B, S, Hq, D), orf) < 2e-2
    # lse (log2 domain) vs reference
    s = torch.matmul(qf, kf.repeat_interleave(Hq // Hkv, 1).transpose(-1, -2)) * scale
    if causal:
        i = torch.arange(S, device=gpu).view(S, 1)
        j = torch.arange(Sk, device=gpu).view(1, Sk)
        s = s.masked_fill(j > i + (Sk - S), float("-inf"))
    lse_ref = torch.logsumexp(s, -1) / math.log(2)
    assert (lse - lse_ref).abs().max().item() < 2e-2
    do = torch.randn(B, S, Hq, D, device=gpu, dtype=torch.bfloat16)
    orf.backward(do.float())
    dq, dkp, dvp = _ops().attn_bwd(do.view(B, S, Hq * D), q, k, v, o, lse, causal, scale)
    rep = Hq // Hkv
    dk = dkp.view(B, Hkv, -1, Sk, D).sum(2)  # partials: per q-head or per q-head group
    dv = dvp.view(B, Hkv, -1, Sk, D).sum(2)
    assert rel_err(dq, qf.grad) < 3e-2
    assert rel_err(dk, kf.grad) < 3e-2
    assert rel_err(dv, vf.grad) < 3e-2


@pytest.mark.parametrize("causal", [True, False])
def test_attention_fwd_growing_max(gpu, causal):
    """Exercise the forward's deferred-rescale branch (rescale only when a row's
    tile max exceeds its running max by > 2^8): scores grow with the key index,
    steeply for some rows (a rescale on nearly every 64-key tile, max jumps of
    tens of log2 units) and gently for others (growth below the threshold, so
    probabilities > 1 are carried), mixed inside every wave."""
    torch.manual_seed(3)
    B, Hq, Hkv, S, D = 1, 4, 1, 640, 128
    keypos = torch.arange(S, device=gpu, dtype=torch.float32) / S
    k = torch.randn(B, Hkv, S, D, device=gpu) * 0.3
    k[..., 0] = keypos * 8.0  # a key feature that grows along the sequence
    q = torch.randn(B, Hq, S, D, device=gpu) * 0.3
    # per row: steep (~20 log2 units of max growth per tile: rescale every tile),
    # medium (~4 per tile: deferred max lags by up to 8) and flat rows
    slope = torch.tensor([200.0, 40.0, 3.0], device=gpu)[torch.arange(S, device=gpu) % 3]
    q[..., 0] = slope
    q, k = q.to(torch.bfloat16), k.to(torch.bfloat16)
    v = torch.randn(B, Hkv, S, D, device=gpu, dtype=torch.bfloat16)
    scale = 1.0 / math.sqrt(D)
    o, lse = _ops().attn_fwd(q, k, v, causal, scale)
    qf, kf, vf = q.float(), k.float(), v.float()
    orf = ref.attention(qf.transpose(1, 2), kf.transpose(1, 2), vf.transpose(1, 2), causal=causal)
    assert rel_err(o.view(B, S, Hq, D), orf) < 2e-2
    s = torch.matmul(qf, kf.repeat_interleave(Hq // Hkv, 1).transpose(-1, -2)) * scale
    if causal:
        i = torch.arange(S, device=gpu).view(S, 1)
        j = torch.arange(S, device=gpu).view(1, S)
        s = s.masked_fill(j > i, float("-inf"))
    lse_ref = torch.logsumexp(s, -1) / math.log(2)
    assert (lse - lse_ref).abs().max().item() < 2e-2


@pytest.mark.parametrize("causal,S", [(True, 2048), (True, 200), (False, 333)])
def test_attention_bwd_deterministic(gpu, causal, S):
    """Deterministic dQ modes (2: per-key-block partials + ordered reduction,
    3: dS^T through HBM + dQ kernel): bitwise identical across runs, equal to
    the atomic path up to f32 summation order."""
    torch.manual_seed(21)
    B, Hq, Hkv, D = 1, 8, 2, 128
    q = torch.randn(B, Hq, S, D, device=gpu, dtype=torch.bfloat16)
    k = torch.randn(B, Hkv, S, D, device=gpu, dtype=torch.bfloat16)
    v = torch.randn(B, Hkv, S, D, device=gpu, dtype=torch.bfloat16)
    sc = 1 / math.sqrt(D)
    o, lse = _ops().attn_fwd(q, k, v, causal, sc)
    do = torch.randn(B, S, Hq * D, device=gpu, dtype=torch.bfloat16)
    ra = _ops().attn_bwd(do, q, k, v, o, lse, causal, sc, 1)  # f32 atomics
    for mode in (2, 3):
        r1 = _ops().attn_bwd(do, q, k, v, o, lse, causal, sc, mode)
        r2 = _ops().attn_bwd(do, q, k, v, o, lse, causal, sc, mode)
        for a, b in zip(r1, r2):
            assert torch.equal(a, b), mode
        # mode 3 rounds dS to bf16 before the dQ GEMM (as the atomic path does in LDS)
        torch.testing.assert_close(r1[0], ra[0], rtol=1e-3, atol=1e-3)
        if mode == 2:  # same key-block kernel: dK / dV summed in the same order
            assert torch.equal(r1[1], ra[1]) and torch.equal(r1[2], ra[2])
        else:  # D=128 split mode: the 8-wave kernel sums its q halves (and q-heads) in its own order
            def g(t):
                return t.view(B, Hkv, -1, S, D).sum(2)
            torch.testing.assert_close(g(r1[1]), g(ra[1]), rtol=1e-4, atol=1e-4)
            torch.testing.assert_close(g(r1[2]), g(ra[2]), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("mode", [3, 1])
def test_attention_training_shape_vs_fp32(gpu, mode):
    """The exact Llama-3.1-70B training attention shape (S=2048, Hq=64, Hkv=8,
    D=128, causal; one sequence) against an fp32 PyTorch reference: forward
    output and every gradient, through the default split backward (3) and the
    f32-atomic dQ path (1)."""
    torch.manual_seed(5)
    B, Hq, Hkv, S, D = 1, 64, 8, 2048, 128
    q = torch.randn(B, Hq, S, D, device=gpu, dtype=torch.bfloat16)
    k = torch.randn(B, Hkv, S, D, device=gpu, dtype=torch.bfloat16)
    v = torch.randn(B, Hkv, S, D, device=gpu, dtype=torch.bfloat16)
    sc = 1.0 / math.sqrt(D)
    o, lse = _ops().attn_fwd(q, k, v, True, sc)
    do = torch.randn(B, S, Hq, D, device=gpu, dtype=torch.bfloat16)
    dq, dkp, dvp = _ops().attn_bwd(do.view(B, S, Hq * D), q, k, v, o, lse, True, sc, mode)
    rep = Hq // Hkv
    dk = dkp.view(B, Hkv, -1, S, D).sum(2)
    dv = dvp.view(B, Hkv, -1, S, D).sum(2)
    qf, kf, vf = [t.float().requires_grad_(True) for t in (q, k, v)]
    orf = ref.attention(qf.transpose(1, 2), kf.transpose(1, 2), vf.transpose(1, 2), causal=True)
    assert rel_err(o.view(B, S, Hq, D), orf) < 2e-2
    orf.backward(do.float())
    assert rel_err(dq, qf.grad) < 3e-2
    assert rel_err(dk, kf.grad) < 3e-2
    assert rel_err(dv, vf.grad) < 3e-2


@pytest.mark.parametrize("hpw", [2, 4, 8])
def test_attention_bwd_heads_per_workgroup(gpu, hpw, monkeypatch):
    """The 8-wave backward with `hpw` q-heads of one KV group per workgroup (dK / dV summed over
    them in registers): [B, Hq / hpw, Sk, D] partials whose per-KV-head sums equal the one-head-
    per-workgroup result, and the same dQ (it does not depend on the grouping)."""
    torch.manual_seed(9)
    B, Hq, Hkv, S, D = 1, 16, 2, 640, 128
    q = torch.randn(B, Hq, S, D, device=gpu, dtype=torch.bfloat16)
    k = torch.randn(B, Hkv, S, D, device=gpu, dtype=torch.bfloat16)
    v = torch.randn(B, Hkv, S, D, device=gpu, dtype=torch.bfloat16)
    sc = 1.0 / math.sqrt(D)
    o, lse = _ops().attn_fwd(q, k, v, True, sc)
    do = torch.randn(B, S, Hq * D, device=gpu, dtype=torch.bfloat16)
    monkeypatch.setenv("MXLLM_ATTN_BWD8_HPW", "1")
    dq1, dk1, dv1 = _ops().attn_bwd(do, q, k, v, o, lse, True, sc, 3)
    monkeypatch.setenv("MXLLM_ATTN_BWD8_HPW", str(hpw))
    dq, dkp, dvp = _ops().attn_bwd(do, q, k, v, o, lse, True, sc, 3)
    assert dkp.shape == (B, Hq // hpw, S, D) and dk1.shape == (B, Hq, S, D)
    assert torch.equal(dq, dq1)

    def g(t):
        return t.view(B, Hkv, -1, S, D).sum(2)
    torch.testing.assert_close(g(dkp), g(dk1), rtol=1e-4, atol=1e-4)
    torch.testing.assert_close(g(dvp), g(dv1), rtol=1e-4, atol=1e-4)


def test_attention_block_autograd(gpu):
    """Full split+rope+attention autograd node vs the reference path."""
    from mxllm.ops.attention import attention_block

    torch.manual_seed(8)
    B, S, Hq, Hkv, D = 2, 192, 8, 2, 128
    cos, sin = ref.rope_tables(S, D, 500000.0, None, gpu)
    qkv = torch.randn(B * S, (Hq + 2 * Hkv) * D, device=gpu, dtype=torch.bfloat16, requires_grad=True)
    o = attention_block(qkv, cos, sin, B, S, Hq, Hkv, D)
    go = torch.randn_like(o)
    o.backward(go)
    x = qkv.detach().float().requires_grad_(True)
    from mxllm.ops.attention import split_heads_ref

    qq, kk, vv = split_heads_ref(x, B, S, Hq, Hkv, D)
    orf = ref.attention(ref.apply_rope(qq, cos, sin), ref.apply_rope(kk, cos, sin), vv).reshape(B * S, -1)
    orf.backward(go.float())
    assert rel_err(o, orf) < 2e-2
    assert rel_err(qkv.grad, x.grad) < 3e-2


def test_segmented_mean(gpu):
    texts = ["test", "hello world", "é漢字", "x" * 5000]
    codes = torch.tensor([ord(c) for t in texts for c in t], dtype=torch.int32, device=gpu)
    offs = torch.tensor([0] + list(torch.tensor([len(t) for t in texts]).cumsum(0)), dtype=torch.int64, device=gpu)
    out = _ops().segmented_mean(codes, offs).cpu()
    for i, t in enumerate(texts):
        assert abs(out[i].item() - torch.tensor([ord(c) for c in t], dtype=torch.float32).mean().item()) < 1e-3


@pytest.mark.parametrize("dtype,n", [(torch.float32, 1_000_003), (torch.bfloat16, 3_000_001), (torch.bfloat16, 7)])
def test_sq_norm_deterministic(gpu, dtype, n):
    """sum(x^2) for f32 and bf16 (one read, fixed-order reduction): matches fp64,
    and is bitwise identical across calls (DDP replicas must agree on the clip)."""
    from mxllm.ops import sq_norm

    x = torch.randn(n, device=gpu).to(dtype)
    a, b = sq_norm(x), sq_norm(x)
    assert torch.equal(a, b)
    ref = x.double().pow(2).sum().item()
    assert abs(a.item() - ref) / ref < 1e-5


@pytest.mark.parametrize("M,K", [(1, 1024), (5, 1024), (16, 1536), (17, 1024), (32, 2048), (33, 1024),
                                 (64, 1024), (100, 1024), (5, 768)])
def test_w8_linear(gpu, M, K):
    """FP8-weight GEMM (decode kernel for M <= 32 and K % 512 == 0, dequantise +
    hipBLASLt otherwise) vs an fp32 matmul with the reference-decoded weights."""
    from mxllm.serve.quant import dequantize_e4m3, quantize_e4m3

    torch.manual_seed(11)
    N = 96
    w = torch.randn(N, K, device=gpu) * 0.02
    q, s = quantize_e4m3(w)
    x = torch.randn(M, K + 64, device=gpu, dtype=torch.bfloat16)[:, :K]  # strided rows (padded producer buffers)
    y = _ops().w8_linear(x, q, s)
    yr = x.float() @ dequantize_e4m3(q, s).t()
    assert y.shape == (M, N) and rel_err(y, yr) < 1e-2
    assert rel_err(_ops().w8_dequant(q, s), dequantize_e4m3(q, s)) < 5e-3


@pytest.mark.parametrize("nc", ["", "4"])
@pytest.mark.parametrize("M,K", [(1, 1536), (4, 1536), (8, 1536), (16, 1536), (8, 8192), (16, 8192),
                                 (8, 4608), (4, 16384), (5, 16384)])
def test_w8_linear_wide(gpu, M, K, nc, monkeypatch):
    """FP8-weight decode GEMM at a projection-sized N (>= 8192: the two-channel-group
    variant for 6..16 tokens, and for 4..5 at K >= 16384; MXLLM_W8_NC=4 the four-group one)
    vs an fp32 matmul with the reference-decoded weights.
    K = 8192 / 4608 give every wave enough k-chunks for the unrolled batch loop
    (and, at 4608, a remainder for its tail loop)."""
    monkeypatch.setenv("MXLLM_W8_NC", nc)
    from mxllm.serve.quant import dequantize_e4m3, quantize_e4m3

    torch.manual_seed(12)
    N = 8192
    w = torch.randn(N, K, device=gpu) * 0.02
    q, s = quantize_e4m3(w)
    x = torch.randn(M, K + 64, device=gpu, dtype=torch.bfloat16)[:, :K]
    y = _ops().w8_linear(x, q, s)
    yr = x.float() @ dequantize_e4m3(q, s).t()
    assert y.shape == (M, N) and rel_err(y, yr) < 1e-2


def test_quant_rows_e4m3(gpu):
    """Per-token activation quantisation kernel == torch's e4m3fn conversion of
    x / (amax / 448), and its decode reproduces x to e4m3 precision."""
    torch.manual_seed(12)
    x = (torch.randn(37, 1024 + 64, device=gpu) * 3).to(torch.bfloat16)[:, :1024]
    q, s = _ops().quant_rows_e4m3(x)
    xf = x.float()
    s_ref = xf.abs().amax(1, keepdim=True) / 448.0
    assert torch.allclose(s, s_ref, rtol=1e-6)
    ref = (xf / s).to(torch.float8_e4m3fn)
    mism = (q.view(torch.float8_e4m3fn).float() != ref.float()).float().mean().item()
    assert mism < 1e-3, mism  # RNE on both sides; only 1/s rounding can flip a tie
    assert rel_err(q.view(torch.float8_e4m3fn).float() * s, xf) < 0.04


@pytest.mark.parametrize("rows", [16, 32, 48, 64])
@pytest.mark.parametrize("T,K", [(16, 128), (48, 384), (96, 1024), (4096, 8192), (4096, 28672), (4096, 10240)])
def test_lora_xwt_tile(gpu, T, K, rows, monkeypatch):
    """Row-tiled lora_xwt (MXLLM_LORA_XWT=tile): only the first `rows` rows of V are the adapter ->
    out[:, :rows] = alpha x V[:rows]^T, zeros in the rest of the 64-column pad (V's padding rows
    are deliberately non-zero here), columns past the pad untouched, bit-reproducible; row counts
    that select 1, 2 and 4 row blocks per workgroup."""
    monkeypatch.setenv("MXLLM_LORA_XWT", "tile")
    torch.manual_seed(5)
    pad = 64
    buf = torch.randn(T, K + pad + 8, device=gpu, dtype=torch.bfloat16)
    x = buf[:, :K]
    v = torch.randn(pad, K + 16, device=gpu, dtype=torch.bfloat16)[:, :K]
    sentinel = buf[:, K + pad:].clone()
    _ops().lora_xwt(x, v, buf[:, K:K + pad], 2.0, rows)
    want = 2.0 * x.float() @ v[:rows].float().t()
    assert rel_err(buf[:, K:K + rows], want) < 1e-2
    assert not buf[:, K + rows:K + pad].any()
    assert torch.equal(buf[:, K + pad:], sentinel)
    first = buf[:, K:K + pad].clone()
    _ops().lora_xwt(x, v, buf[:, K:K + pad], 2.0, rows)
    assert torch.equal(buf[:, K:K + pad], first)


@pytest.mark.parametrize("kern", ["lds", "reg"])
@pytest.mark.parametrize("T,K,vrows", [(256, 512, 64), (256, 4096, 64), (4096, 1024, 128), (64, 192, 64),
                                       (4096, 8192, 64)])
def test_lora_xwt(gpu, T, K, vrows, kern, monkeypatch):
    """out[:, :vrows] = alpha x V^T into the tail of a padded buffer (S = 1 and the
    ordered split reduction), columns past the tail untouched; both kernels: the
    LDS-DMA-staged one (default) and the register-fragment one (MXLLM_LORA_XWT=reg)."""
    monkeypatch.setenv("MXLLM_LORA_XWT", kern)
    torch.manual_seed(3)
    buf = torch.randn(T, K + vrows + 8, device=gpu, dtype=torch.bfloat16)
    x = buf[:, :K]
    vb = torch.randn(vrows, K + 8, device=gpu, dtype=torch.bfloat16)
    v = vb[:, :K]
    sentinel = buf[:, K + vrows:].clone()
    _ops().lora_xwt(x, v, buf[:, K:K + vrows], 2.0)
    want = 2.0 * x.float() @ v.float().t()
    assert rel_err(buf[:, K:K + vrows], want) < 1e-2
    assert torch.equal(buf[:, K + vrows:], sentinel)
    first = buf[:, K:K + vrows].clone()
    _ops().lora_xwt(x, v, buf[:, K:K + vrows], 2.0)
    assert torch.equal(buf[:, K:K + vrows], first)  # bit-reproducible
    if kern == "lds":  # split partials merged in-launch (sc1 hand-off): same bits, counters reset
        monkeypatch.setenv("MXLLM_LORA_FUSED_RED", "1")
        for _ in range(2):
            buf[:, K:K + vrows] = 0
            _ops().lora_xwt(x, v, buf[:, K:K + vrows], 2.0)
            assert torch.equal(buf[:, K:K + vrows], first)


@pytest.mark.parametrize("T,K,splits,r,acc", [(256, 512, [512, 128, 128], 16, False),
                                              (4096, 1024, [1024, 256, 256], 16, True),
                                              (512, 256, [1024, 1024], 16, True),
                                              (256, 320, [192], 16, False),
                                              (256, 512, [512, 256, 256], 32, True)])
def test_lora_grads(gpu, T, K, splits, r, acc, monkeypatch):
    """dA = g^T x and the diagonal blocks dB_i = dy_i^T st_i in one launch,
    accumulated into bf16 grads or written fresh; off-diagonal blocks untouched;
    the in-launch split merge (MXLLM_LORA_FUSED_RED=1) gives the same bits."""
    torch.manual_seed(4)
    n, N = len(splits), sum(splits)
    R = n * r
    pad = (R + 63) // 64 * 64
    xa = torch.randn(T, K + pad, device=gpu, dtype=torch.bfloat16)
    dya = torch.randn(T, N + pad, device=gpu, dtype=torch.bfloat16)
    ga = torch.randn(R, K, device=gpu, dtype=torch.bfloat16) if acc else torch.zeros(R, K, device=gpu,
                                                                                       dtype=torch.bfloat16)
    gb = torch.randn(N, R, device=gpu, dtype=torch.bfloat16) if acc else torch.zeros(N, R, device=gpu,
                                                                                       dtype=torch.bfloat16)
    ga0, gb0 = ga.clone(), gb.clone()
    x2, dy2, g, st = xa[:, :K], dya[:, :N], dya[:, N:], xa[:, K:]
    _ops().lora_grads(x2, dy2, g, st, ga, gb, splits, r, acc)
    want_a = g[:, :R].float().t() @ x2.float() + (ga0.float() if acc else 0)
    assert rel_err(ga, want_a) < 1e-2
    want_b = gb0.float().clone()
    off = 0
    for i, ni in enumerate(splits):
        blk = dy2[:, off:off + ni].float().t() @ st[:, i * r:(i + 1) * r].float()
        want_b[off:off + ni, i * r:(i + 1) * r] = blk + (want_b[off:off + ni, i * r:(i + 1) * r] if acc else 0)
        off += ni
    assert rel_err(gb, want_b) < 1e-2
    mask = torch.ones_like(gb, dtype=torch.bool)
    off = 0
    for i, ni in enumerate(splits):
        mask[off:off + ni, i * r:(i + 1) * r] = False
        off += ni
    assert torch.equal(gb[mask], gb0[mask])  # off-diagonal blocks untouched
    ga1, gb1 = ga0.clone(), gb0.clone()
    _ops().lora_grads(x2, dy2, g, st, ga1, gb1, splits, r, acc)
    assert torch.equal(ga1, ga) and torch.equal(gb1, gb)  # bit-reproducible
    monkeypatch.setenv("MXLLM_LORA_FUSED_RED", "1")
    monkeypatch.setenv("MXLLM_LORA_XTG_WT", "0")
    for _ in range(2):
        ga1, gb1 = ga0.clone(), gb0.clone()
        _ops().lora_grads(x2, dy2, g, st, ga1, gb1, splits, r, acc)
        assert torch.equal(ga1, ga) and torch.equal(gb1, gb)
    # one 64-col tile per wave over all rows (MXLLM_LORA_XTG_WT=1; the tile threshold lowered so
    # these shapes qualify): same products to fp32 rounding, off-diagonal blocks untouched, reproducible
    monkeypatch.setenv("MXLLM_LORA_XTG_WT", "1")
    monkeypatch.setenv("MXLLM_LORA_XTG_WT_MIN", "16")
    outs = []
    for _ in range(2):
        ga1, gb1 = ga0.clone(), gb0.clone()
        _ops().lora_grads(x2, dy2, g, st, ga1, gb1, splits, r, acc)
        assert rel_err(ga1, want_a) < 1e-2 and rel_err(gb1, want_b) < 1e-2
        assert torch.equal(gb1[mask], gb0[mask])
        outs.append((ga1, gb1))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("R,C,ld", [(4096, 8192, None), (64, 64, None), (37, 130, None), (130, 4096, 4160),
                                    (4096, 1, None)])
def test_transpose2d(gpu, R, C, ld):
    """LDS-tiled 16-bit transpose (full fine-tuning dW operand images): exact,
    row-strided inputs and ragged edge tiles included."""
    torch.manual_seed(0)
    base = torch.randn(R, ld or C, device=gpu, dtype=torch.bfloat16)
    x = base[:, :C]
    y = _ops().transpose2d(x)
    assert y.shape == (C, R) and y.is_contiguous()
    assert torch.equal(y, x.t())
    # with a device-scalar scale (the CE upstream gradient folded into dlogits' image)
    sc = torch.tensor([0.3], device=gpu)
    ys = _ops().transpose2d(x, sc)
    assert torch.equal(ys, (x.float() * 0.3).bfloat16().t())


@pytest.mark.parametrize("T,N,K", [(4096, 1024, 512), (300, 130, 72)])
def test_weight_grad_tn(gpu, T, N, K):
    """Full fine-tuning dW through transposed token-contiguous images equals
    dy^T x (fp32 reference), with and without beta=1 accumulation."""
    from mxllm.ops.linear import weight_grad_

    torch.manual_seed(0)
    dy = torch.randn(T, N, device=gpu, dtype=torch.bfloat16)
    x = torch.randn(T, K, device=gpu, dtype=torch.bfloat16)
    want = dy.float().t() @ x.float()
    assert rel_err(weight_grad_(None, dy, x), want) < 1e-2
    acc = torch.randn(N, K, device=gpu, dtype=torch.bfloat16)
    want2 = acc.float() + want
    weight_grad_(acc, dy, x)
    assert rel_err(acc, want2) < 1e-2


@pytest.mark.parametrize("M,N,K", [(1, 6144, 4096), (5, 4096, 14336), (16, 1040, 512), (17, 2048, 1024),
                                   (32, 96, 4608)])
def test_skinny_linear_vs_fp32(gpu, M, N, K):
    """Decode GEMM (csrc/kernels/skinny_gemm.hip) against fp32 torch, incl. a row-strided x
    (the view a producer leaves) and both token-block variants (<= 16 and 17..32 rows)."""
    torch.manual_seed(M + N)
    xb = torch.randn(M, K + 64, device=gpu, dtype=torch.bfloat16)
    x = xb[:, :K]
    w = torch.randn(N, K, device=gpu, dtype=torch.bfloat16) * 0.05
    y = _ops().skinny_linear(x, w)
    ref = x.float() @ w.float().t()
    assert y.shape == (M, N) and rel_err(y, ref) < 1e-2


@pytest.mark.gpu
@pytest.mark.parametrize("M,F,K", [(1, 14336, 4096), (5, 520, 512), (8, 1024, 1536), (17, 256, 1024),
                                   (32, 512, 2048)])
def test_skinny_linear_swiglu(gpu, M, F, K):
    """Decode gate|up projection with SwiGLU in the epilogue: bit-identical to the decode
    GEMM + SwiGLU kernel, and close to fp32 silu(x Wg^T) * (x Wu^T).  x is row-strided."""
    import sys

    from mxllm import ops

    torch.manual_seed(M * 7 + K)
    xb = torch.randn(M, K + 64, device=gpu, dtype=torch.bfloat16)
    x = xb[:, :K]
    w = torch.randn(2 * F, K, device=gpu, dtype=torch.bfloat16) * 0.05
    y = _ops().skinny_linear_swiglu(x, w)
    two = ops.swiglu(_ops().skinny_linear(x, w))
    assert y.shape == (M, F) and torch.equal(y, two)
    gu = x.float() @ w.float().t()
    ref = torch.nn.functional.silu(gu[:, :F]) * gu[:, F:]
    assert rel_err(y, ref) < 1e-2
    if M <= sys.modules["mxllm.ops.linear"].SKINNY_M:  # the routed entry point takes it
        assert torch.equal(ops.linear_swiglu(x, w), y)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,resid,swiglu", [(1, 6144, 4096, False, False), (1, 1024, 4096, True, False),
                                                (3, 512, 8192, True, False), (4, 2048, 4096, True, True),
                                                (1, 28672 // 8, 8192, True, True), (2, 1040, 1536, False, True)])
def test_skinny_norm_linear(gpu, M, N, K, resid, swiglu):
    """Decode projection with the (residual-add +) RMSNorm in the GEMM prologue: bit-identical to
    the RMSNorm kernel followed by the decode GEMM (or the SwiGLU-epilogue GEMM), same new
    residual, and close to the fp32 reference."""
    from mxllm import ops

    torch.manual_seed(M + N + K)
    h = torch.randn(M, K, device=gpu, dtype=torch.bfloat16)
    d = torch.randn(M, K, device=gpu, dtype=torch.bfloat16) if resid else None
    gamma = (1.0 + 0.1 * torch.randn(K, device=gpu)).to(torch.bfloat16)
    w = torch.randn(N, K, device=gpu, dtype=torch.bfloat16) * 0.05
    y, h2 = _ops().skinny_norm_linear(h, d, gamma, 1e-5, w, swiglu)
    if resid:
        xn, hn = ops.add_rms_norm(d, h, gamma, 1e-5)
        assert torch.equal(h2, hn)
    else:
        xn, hn = ops.rms_norm(h, gamma, 1e-5), h
        assert h2.data_ptr() == h.data_ptr()
    two = _ops().skinny_linear_swiglu(xn, w) if swiglu else _ops().skinny_linear(xn, w)
    assert torch.equal(y, two)
    hf = hn.float()
    xr = hf * torch.rsqrt(hf.pow(2).mean(-1, keepdim=True) + 1e-5) * gamma.float()
    gu = xr @ w.float().t()
    ref = torch.nn.functional.silu(gu[:, :N // 2]) * gu[:, N // 2:] if swiglu else gu
    assert rel_err(y, ref) < 2e-2
    import sys

    if M <= sys.modules["mxllm.ops.linear"].NORM_M:  # the routed entry point takes it
        got = ops.norm_linear(d, h, gamma, 1e-5, w, swiglu)
        assert got is not None and torch.equal(got[0], y)


@pytest.mark.gpu
@pytest.mark.parametrize("M,Hq,Hkv,K,norm,resid", [(1, 32, 8, 4096, True, True), (2, 8, 2, 1024, True, False),
                                                   (2, 64, 8, 8192, True, True), (5, 16, 4, 2048, False, False),
                                                   (4, 16, 4, 2048, False, False)])
def test_skinny_qkv_rope(gpu, M, Hq, Hkv, K, norm, resid):
    """Decode QKV projection with RoPE + KV-cache append in the GEMM epilogue (and the RMSNorm
    in its prologue): the same q, cache rows and residual as RMSNorm + decode GEMM + rope_append."""
    from mxllm import ops

    torch.manual_seed(M * 3 + Hq)
    D, max_seq, nslots = 128, 300, M + 2
    N = (Hq + 2 * Hkv) * D
    h = torch.randn(M, K, device=gpu, dtype=torch.bfloat16)
    d = torch.randn(M, K, device=gpu, dtype=torch.bfloat16) if resid else None
    gamma = (1.0 + 0.1 * torch.randn(K, device=gpu)).to(torch.bfloat16) if norm else None
    w = torch.randn(N, K, device=gpu, dtype=torch.bfloat16) * 0.05
    cos, sin = ref.rope_tables(1024, D, 500000.0, None, gpu)
    pos = torch.tensor([17, 299, 0, 5, 123][:M], dtype=torch.int32, device=gpu)
    slots = torch.tensor([3, 0, 2, 1, 4][:M], dtype=torch.int32, device=gpu) % nslots
    kc = torch.randn(nslots, Hkv, max_seq, D, device=gpu, dtype=torch.bfloat16)
    vc = torch.randn_like(kc)
    kc2, vc2 = kc.clone(), vc.clone()
    q, h2 = _ops().skinny_qkv_rope(h, d, gamma, 1e-5, w, cos, sin, pos, slots, kc, vc, Hq, Hkv)
    if norm:
        if resid:
            xn, hn = ops.add_rms_norm(d, h, gamma, 1e-5)
        else:
            xn, hn = ops.rms_norm(h, gamma, 1e-5), h
        assert torch.equal(h2, hn)
    else:
        xn = h
    qkv = _ops().skinny_linear(xn, w)
    q_ref = _ops().rope_append(qkv, cos, sin, pos, slots, kc2, vc2, Hq, Hkv, D)
    assert torch.equal(q.view(M, -1), q_ref.reshape(M, -1))
    assert torch.equal(kc, kc2) and torch.equal(vc, vc2)


@pytest.mark.parametrize("target", ["bf16", "fp32"])
@pytest.mark.parametrize("fresh", [True, False])
def test_embedding_sparse_backward(gpu, target, fresh):
    """Embedding backward into the owner's gradient buffer (sorted ids, one workgroup per
    distinct id, touched rows only) vs an fp32 index_add reference: repeated ids, first
    write of the step (fresh: stale buffer contents ignored) or accumulation."""
    from mxllm.ops.embedding import embedding

    torch.manual_seed(7)
    V, H = 3000, 512
    w = torch.nn.Parameter(torch.randn(V, H, device=gpu).bfloat16())
    ids = torch.randint(0, 40, (1200,), device=gpu)  # heavy repetition
    ids[:5] = 2999
    dy = torch.randn(1200, H, device=gpu).bfloat16()
    init = torch.randn(V, H, device=gpu)
    if target == "fp32":
        w._mx_grad32 = init.clone()
    else:
        w.grad = init.bfloat16().clone()
    w._mx_grad_fresh = fresh
    embedding(ids, w).backward(dy)
    ref = torch.zeros(V, H, device=gpu).index_add_(0, ids.reshape(-1), dy.reshape(-1, H).float())
    base = 0 if fresh else (init if target == "fp32" else init.bfloat16().float())
    got = w._mx_grad32 if target == "fp32" else w.grad.float()
    tol = 1e-5 if target == "fp32" else 1e-2
    assert ((got - (base + ref)).abs().max() / (base + ref).abs().max()).item() < tol
    # deterministic: the same call again gives the same bits
    first = got.clone()
    if target == "fp32":
        w._mx_grad32.copy_(init)
    else:
        w.grad.copy_(init.bfloat16())
    w._mx_grad_fresh = fresh
    embedding(ids, w).backward(dy)
    again = w._mx_grad32 if target == "fp32" else w.grad.float()
    assert torch.equal(again, first)


def test_embedding_backward_tied_is_deterministic(gpu):
    """No owner buffer (tied embeddings: autograd sums the embedding and head gradients): the
    embedding gradient comes from the same sorted, fixed-order kernel into a zeroed fp32 [V, H]
    -- equal to an fp32 index_add reference and bitwise the same on every call (the atomic
    accumulator it replaces made tied-embedding training differ run to run)."""
    from mxllm.ops.embedding import embedding

    torch.manual_seed(3)
    V, H = 5000, 512
    ids = torch.randint(0, 64, (2048,), device=gpu)  # flat token ids (as the model passes them), heavy repetition
    dy = torch.randn(2048, H, device=gpu).bfloat16()
    grads = []
    for _ in range(3):
        w = torch.nn.Parameter(torch.zeros(V, H, device=gpu).bfloat16())
        w._mx_no_direct = True
        embedding(ids, w).backward(dy)
        grads.append(w.grad.float().clone())
    ref = torch.zeros(V, H, device=gpu).index_add_(0, ids.reshape(-1), dy.reshape(-1, H).float())
    assert rel_err(grads[0], ref) < 1e-2
    assert torch.equal(grads[0], grads[1]) and torch.equal(grads[0], grads[2])


def test_chunked_lm_head_ce_matches_unchunked_gpu(gpu):
    """Long-sequence LM head + CE walked in token chunks (ce_inv_count + ce_chunk_f32 kernels: the
    loss from fp32 logits, dh / dW formed per chunk) vs the one-piece fused path (bf16 logits) and an
    fp32 PyTorch reference: loss and gradients."""
    import torch.nn.functional as F

    from mxllm.ops.loss import linear_cross_entropy

    torch.manual_seed(11)
    T, H, V = 1000, 256, 4096
    h = (torch.randn(T, H, device=gpu) * 0.5).to(torch.bfloat16).requires_grad_(True)
    w = (torch.randn(V, H, device=gpu) * 0.05).to(torch.bfloat16).requires_grad_(True)
    lab = torch.randint(0, V, (T,), device=gpu)
    lab[::17] = -100
    res = []
    for chunk in (None, 256):
        loss = linear_cross_entropy(h, w, lab) if chunk is None else linear_cross_entropy(h, w, lab, chunk=chunk)
        (loss * 0.5).backward()
        res.append((float(loss.detach()), h.grad.float().clone(), w.grad.float().clone()))
        h.grad = w.grad = None
    hf, wf = h.detach().float().requires_grad_(True), w.detach().float().requires_grad_(True)
    lr = F.cross_entropy(hf @ wf.t(), lab, ignore_index=-100)
    (lr * 0.5).backward()
    (l0, gh0, gw0), (l1, gh1, gw1) = res
    assert abs(l1 - float(lr)) < 2e-6 * abs(float(lr))  # fp32 logits: the loss of the fp32 reference
    assert abs(l0 - float(lr)) < 2e-3 * abs(float(lr))  # bf16 logits
    for g, r in ((gh0, hf.grad), (gh1, hf.grad), (gw0, wf.grad), (gw1, wf.grad)):
        assert rel_err(g, r) < 2e-2


@pytest.mark.parametrize("S", [8192])
def test_attention_long_context_vs_fp32(gpu, S):
    """Long context: causal GQA attention at S=8192 through the training
    kernels (forward + the default split backward) against an fp32 PyTorch reference —
    output, dQ, dK, dV."""
    torch.manual_seed(9)
    B, Hq, Hkv, D = 1, 8, 2, 128
    q = torch.randn(B, Hq, S, D, device=gpu, dtype=torch.bfloat16)
    k = torch.randn(B, Hkv, S, D, device=gpu, dtype=torch.bfloat16)
    v = torch.randn(B, Hkv, S, D, device=gpu, dtype=torch.bfloat16)
    sc = 1.0 / math.sqrt(D)
    o, lse = _ops().attn_fwd(q, k, v, True, sc)
    do = torch.randn(B, S, Hq, D, device=gpu, dtype=torch.bfloat16)
    dq, dkp, dvp = _ops().attn_bwd(do.view(B, S, Hq * D), q, k, v, o, lse, True, sc, 3)
    dk = dkp.view(B, Hkv, -1, S, D).sum(2)
    dv = dvp.view(B, Hkv, -1, S, D).sum(2)
    qf, kf, vf = [t.float().requires_grad_(True) for t in (q, k, v)]
    orf = ref.attention(qf.transpose(1, 2), kf.transpose(1, 2), vf.transpose(1, 2), causal=True)
    assert rel_err(o.view(B, S, Hq, D), orf) < 2e-2
    orf.backward(do.float())
    assert rel_err(dq, qf.grad) < 3e-2
    assert rel_err(dk, kf.grad) < 3e-2
    assert rel_err(dv, vf.grad) < 3e-2


@pytest.mark.parametrize("f32", [True, False])
def test_embedding_bwd_sorted_dominant_id(gpu, f32):
    """Sorted, chunked embedding backward: a dominant id (here 80 % of 5,000 tokens, as
    pad / EOS in packed batches) is split over 64-row chunks whose partials are combined in chunk
    order -- the sums match an fp64 reference and repeat bitwise."""
    torch.manual_seed(13)
    T, H, V = 5000, 512, 300
    ids = torch.randint(0, V, (T,), device=gpu)
    ids[torch.rand(T, device=gpu) < 0.8] = 7
    dy = torch.randn(T, H, device=gpu, dtype=torch.bfloat16)
    sid, perm = torch.sort(ids, stable=True)
    outs = []
    for _ in range(2):
        out = torch.zeros(V, H, device=gpu, dtype=torch.float32 if f32 else torch.bfloat16)
        _ops().embedding_bwd_sorted(dy, sid, perm, out)
        outs.append(out)
    ref = torch.zeros(V, H, device=gpu, dtype=torch.float64).index_add_(0, ids, dy.double())
    assert rel_err(outs[0], ref) < (1e-5 if f32 else 5e-3)
    assert torch.equal(outs[0], outs[1])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 2048, 8192), (8, 8, 1024), (5, 2056, 3072), (3, 40, 12288), (7, 4080, 2048)])
def test_skinny_linear_half(gpu, M, N, K):
    """Decode GEMM by groups of 8 channels against fp64: one group, odd row counts, K parts of one to twelve chunks."""
    torch.manual_seed(M + N)
    x = torch.randn(M, K + 64, device=gpu, dtype=torch.bfloat16)[:, :K]
    w = torch.randn(N, K, device=gpu, dtype=torch.bfloat16) * 0.05
    y = _ops().skinny_linear_half(x, w)
    assert y.shape == (M, N) and rel_err(y, x.double() @ w.double().t()) < 2 ** -8  # one bf16 rounding


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 8, 6144), (8, 2048, 8192), (3, 72, 10240), (5, 2048, 12288), (2, 1024, 14336), (8, 64, 16384),
                                   (2, 2048, 9216), (1, 1024, 11264), (8, 2048, 13312), (4, 8, 15360), (8, 2048, 15360), (8, 2056, 13312)])
def test_skinny_linear_half_whole_parts(gpu, M, N, K):
    """A wave's whole K part in flight (18 to 30 chunks) and the sizes beside them."""
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device=gpu, dtype=torch.bfloat16)
    w = torch.randn(N, K + 8, device=gpu, dtype=torch.bfloat16)[:, :K] * 0.05
    assert rel_err(_ops().skinny_linear_half(x, w), x.double() @ w.double().t()) < 2 ** -8  # one bf16 rounding


def _stream_weight(w, f8):
    from mxllm.serve.quant import quantize_e4m3

    return quantize_e4m3(w) if f8 else (w, None)


@pytest.mark.gpu
@pytest.mark.parametrize("f8", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 16, 2048), (3, 16 * 513, 4096), (16, 16 * 257, 4096), (17, 8192, 2048),
                                   (32, 16 * 600, 2048), (9, 48, 6144), (4, 96, 16384), (2, 16 * 1025, 8192)])
def test_stream_linear(gpu, M, N, K, f8):
    """Decode GEMM of workgroups that stay (csrc/kernels/stream_gemm.hip): the bits of the one-group kernels, with
    fewer, as many and more groups than workgroups, one and two workgroups a CU, both block sizes; row-strided x."""
    torch.manual_seed(M + N)
    x = torch.randn(M, K + 64, device=gpu, dtype=torch.bfloat16)[:, :K]
    w, s = _stream_weight(torch.randn(N, K, device=gpu, dtype=torch.bfloat16) * 0.05, f8)
    y = _ops().stream_linear(x, None, None, 0.0, w, s, False)[0]
    assert torch.equal(y, _ops().w8_linear(x, w, s) if f8 else _ops().skinny_linear(x, w))
    wd = w.view(torch.float8_e4m3fn).double() * s.double()[:, None] if f8 else w.double()
    assert rel_err(y, x.double() @ wd.t()) < 2 ** -8  # one bf16 rounding
    from mxllm import ops

    two = ops.swiglu(y)
    assert torch.equal(_ops().stream_linear(x, None, None, 0.0, w, s, True)[0], two)
    if M <= 4:
        for resid in (False, True):
            d = torch.randn(M, K, device=gpu, dtype=torch.bfloat16) if resid else None
            gamma = (1.0 + 0.1 * torch.randn(K, device=gpu)).to(torch.bfloat16)
            xn, hn = ops.add_rms_norm(d, x, gamma, 1e-5) if resid else (ops.rms_norm(x, gamma, 1e-5), x)
            for sw in (False, True):
                got, h2 = _ops().stream_linear(x, d, gamma, 1e-5, w, s, sw)
                assert torch.equal(h2, hn)
                assert torch.equal(got, _ops().stream_linear(xn, None, None, 0.0, w, s, sw)[0])


@pytest.mark.gpu
@pytest.mark.parametrize("f8", [False, True])
@pytest.mark.parametrize("M", [1, 4, 7, 8, 9, 16])
@pytest.mark.parametrize("groups", [257, 300, 384])
def test_stream_group_and_half(gpu, groups, M, f8):
    """257 to 384 groups of a K of 4096: a workgroup's group and half of another, one of them to every CU; plain, SwiGLU and
    QKV epilogues (a half has both channels of a pair), with the norm up to 4 rows."""
    from mxllm import ops

    torch.manual_seed(M + groups)
    K, N, D = 4096, 16 * groups, 128
    x = torch.randn(M, K, device=gpu, dtype=torch.bfloat16)
    w, s = _stream_weight(torch.randn(N, K, device=gpu, dtype=torch.bfloat16) * 0.05, f8)
    y = _ops().stream_linear(x, None, None, 0.0, w, s, False)[0]
    wd = w.view(torch.float8_e4m3fn).double() * s.double()[:, None] if f8 else w.double()
    assert rel_err(y, x.double() @ wd.t()) < 2 ** -8  # one bf16 rounding
    assert torch.equal(y, _ops().w8_linear(x, w, s) if f8 else _ops().skinny_linear(x, w))
    assert torch.equal(_ops().stream_linear(x, None, None, 0.0, w, s, True)[0], ops.swiglu(y))
    d, gamma = torch.randn_like(x), (1.0 + 0.1 * torch.randn(K, device=gpu)).to(torch.bfloat16)
    if M <= 4:
        xn, hn = ops.add_rms_norm(d, x, gamma, 1e-5)
        got, h2 = _ops().stream_linear(x, d, gamma, 1e-5, w, s, False)
        y = _ops().stream_linear(xn, None, None, 0.0, w, s, False)[0]
        assert torch.equal(h2, hn) and torch.equal(got, y)
    if groups == 384:
        Hq, Hkv, norm = 32, 8, M <= 4
        cos, sin = ref.rope_tables(64, D, 500000.0, None, gpu)
        slots, pos = torch.randperm(M, device=gpu).to(torch.int32), torch.randint(0, 64, (M,), device=gpu, dtype=torch.int32)
        kc, vc = (torch.randn(M, Hkv, 64, D, device=gpu, dtype=torch.bfloat16) for _ in range(2))
        kc2, vc2 = kc.clone(), vc.clone()
        q, _ = _ops().stream_qkv_rope(x, d if norm else None, gamma if norm else None, 1e-5, w, s, cos, sin, pos, slots, kc, vc,
                                      Hq, Hkv, None)
        q_ref = _ops().rope_append(y, cos, sin, pos, slots, kc2, vc2, Hq, Hkv, D, None)
        assert torch.equal(q.view(M, -1), q_ref.reshape(M, -1)) and torch.equal(kc, kc2) and torch.equal(vc, vc2)


@pytest.mark.gpu
@pytest.mark.parametrize("f8", [False, True])
@pytest.mark.parametrize("M,Hq,Hkv,D,K,norm", [(1, 32, 8, 64, 2048, True), (16, 32, 8, 128, 4096, False),
                                               (32, 5, 1, 64, 2048, False), (4, 64, 8, 128, 8192, True)])
def test_stream_qkv_rope(gpu, M, Hq, Hkv, D, K, norm, f8):
    """The QKV projection with RoPE and the cache append in the epilogue, heads of 64 and 128, contiguous and paged
    caches: q, cache rows and residual of RMSNorm + projection + rope_append."""
    from mxllm import ops

    torch.manual_seed(M * 3 + Hq)
    max_seq, nslots = 256, M + 2
    h = torch.randn(M, K, device=gpu, dtype=torch.bfloat16)
    d = torch.randn(M, K, device=gpu, dtype=torch.bfloat16) if norm else None
    gamma = (1.0 + 0.1 * torch.randn(K, device=gpu)).to(torch.bfloat16) if norm else None
    w, s = _stream_weight(torch.randn((Hq + 2 * Hkv) * D, K, device=gpu, dtype=torch.bfloat16) * 0.05, f8)
    cos, sin = ref.rope_tables(1024, D, 500000.0, None, gpu)
    slots = torch.randperm(nslots, device=gpu)[:M].to(torch.int32)
    xn, hn = ops.add_rms_norm(d, h, gamma, 1e-5) if norm else (h, h)
    qkv = _ops().stream_linear(xn, None, None, 0.0, w, s, False)[0]
    for bt in (None, torch.randperm(4 * nslots, device=gpu).to(torch.int32).view(nslots, 4)):
        pos = torch.randint(0, max_seq if bt is None else 1024, (M,), device=gpu, dtype=torch.int32)
        kc = torch.randn(nslots if bt is None else 4 * nslots, Hkv, max_seq, D, device=gpu, dtype=torch.bfloat16)
        vc = torch.randn_like(kc)
        kc2, vc2 = kc.clone(), vc.clone()
        q, h2 = _ops().stream_qkv_rope(h, d, gamma, 1e-5, w, s, cos, sin, pos, slots, kc, vc, Hq, Hkv, bt)
        q_ref = _ops().rope_append(qkv, cos, sin, pos, slots, kc2, vc2, Hq, Hkv, D, bt)
        assert torch.equal(h2, hn) and torch.equal(q.view(M, -1), q_ref.reshape(M, -1))
        assert torch.equal(kc, kc2) and torch.equal(vc, vc2)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Hq,Hkv,lens", [(8, 2, [1, 255, 256, 257]), (4, 4, [64, 65, 700]), (16, 1, [1300, 3]),
                                         (6, 2, [31, 256])])
def test_decode_attn_partials_precision(gpu, D, Hq, Hkv, lens):
    """Split-K decode attention on paged caches with stale rows (NaN past a sequence's end), every group size up to
    16: merged partials against f64.  Heads of 64 and 32 keep f32 softmax weights (an f32 sum of up to 1300 terms);
    heads of 128 round them to bf16.  The output of a single split equals the merge of its partials."""
    torch.manual_seed(D + Hq)
    B, blk = len(lens), 256
    maxb = (max(lens) + blk - 1) // blk
    bt = torch.randperm(B * maxb, device=gpu).to(torch.int32).view(B, maxb)
    kc = torch.full((B * maxb, Hkv, blk, D), float("nan"), device=gpu, dtype=torch.bfloat16)
    vc = kc.clone()
    q = torch.randn(B, Hq, D, device=gpu, dtype=torch.bfloat16)
    want = torch.empty(B, Hq, D, dtype=torch.float64, device=gpu)
    for b, n in enumerate(lens):
        k, v = (torch.randn(Hkv, n, D, device=gpu, dtype=torch.bfloat16) for _ in range(2))
        for j in range(0, n, blk):
            kc[int(bt[b, j // blk]), :, :min(blk, n - j)] = k[:, j:j + blk]
            vc[int(bt[b, j // blk]), :, :min(blk, n - j)] = v[:, j:j + blk]
        for h in range(Hq):
            s = k[h * Hkv // Hq].double() @ q[b, h].double() * D ** -0.5
            want[b, h] = torch.softmax(s, 0) @ v[h * Hkv // Hq].double()
    pos = torch.tensor(lens, dtype=torch.int32, device=gpu) - 1
    slots = torch.arange(B, dtype=torch.int32, device=gpu)
    ml, po = _ops().decode_attn_partials(q, kc, vc, pos, slots, max(lens), D ** -0.5, 1, bt)
    m, l = ml[..., 0].double(), ml[..., 1].double()
    w = torch.where(m > float("-inf"), torch.exp2(m - m.amax(-1, keepdim=True)), 0.0)
    o = torch.where(w[..., None] > 0, po.double(), 0.0)
    got = (w[..., None] * o).sum(2) / (w * l).sum(-1, keepdim=True)
    err = float((got - want).norm() / want.norm())
    assert err < (2 ** -8 if D == 128 else 2e-6), err
    out = _ops().decode_attn(q, kc, vc, pos, slots, max(lens), D ** -0.5, 1, bt, None).view(B, Hq, D)
    assert rel_err(out, want) < 2 ** -7
    one = [b for b, n in enumerate(lens) if n <= blk]
    if one:
        i = torch.tensor(one, device=gpu)
        y = _ops().decode_attn(q[i], kc, vc, pos[i], slots[i], blk, D ** -0.5, 1, bt, None).view(-1, Hq, D)
        assert torch.equal(y, out[i])


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 3, 4])
@pytest.mark.parametrize("N,K", [(16, 2048), (8208, 2048), (12288, 4096)])
@pytest.mark.parametrize("add", [False, True])
def test_stream_group_norm(gpu, M, N, K, add):
    """The grouped norm in the prologue of the GEMM that stays against the norm and the product one after the other: the
    residual's bits, and the product to two roundings to bf16 (the norm's sum is in another order); parts of unlike size."""
    torch.manual_seed(N + M)
    h = torch.randn(M, K, device=gpu) * torch.logspace(-2, 2, 8, device=gpu).repeat_interleave(K // 8)
    g = torch.randn(K, device=gpu)
    delta = torch.randn(M, K + 8, device=gpu).bfloat16()[:, :K] if add else None
    w = (torch.randn(N, K, device=gpu) * K ** -0.5).bfloat16()
    keep = h.clone()
    y, h2 = _ops().stream_group_norm(delta, h, g, 1e-3, w)
    assert torch.equal(h, keep)
    want_h = h + delta.float() if add else h
    assert torch.equal(h2, want_h)
    p = want_h.double().view(M, 8, -1)
    x = (p * torch.rsqrt(p.pow(2).mean(-1, keepdim=True) + 1e-3)).view(M, K) * g.double()
    assert rel_err(y, x @ w.double().t()) < 2 ** -7


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 4, 5, 8])
@pytest.mark.parametrize("K", [2048, 4096])
@pytest.mark.parametrize("limit", [None, 3, 8])
def test_group_norm_prologue_by_the_rows_asked_for(gpu, monkeypatch, M, K, limit):
    """MXLLM_NORM_FUSED_M past what the GEMM that stays takes (4 rows): the other prologue or the parts, never an error."""
    from mxllm.ops import hybrid as hops

    if limit is not None:
        monkeypatch.setattr(hops, "NORM_M", limit)
        monkeypatch.setattr(hops, "_NORM_STREAM_M", limit)
    torch.manual_seed(M)
    h, delta, g = torch.randn(M, K, device=gpu), torch.randn(M, K, device=gpu).bfloat16(), torch.rand(K, device=gpu) + 0.5
    w = (torch.randn(6144, K, device=gpu) * K ** -0.5).bfloat16()
    r = hops.norm_linear(delta, h, g, 8, 1e-5, w)
    want = h.double() + delta.double()
    if r is None:
        assert M > (limit or 4) or M * K > 16384
        h2 = h.clone()
        r = hops.group_norm(delta, h2, g, 8, 1e-5, torch.bfloat16) @ w.t(), h2
    p = want.view(M, 8, -1)
    x = (p * torch.rsqrt(p.pow(2).mean(-1, keepdim=True) + 1e-5)).view(M, K) * g.double()
    assert rel_err(r[1], want) < 1e-6 and rel_err(r[0], x @ w.double().t()) < 2 ** -7  # the norm's rounding and the product's


def _off16(t):
    """t in storage that starts between two 16-byte pieces."""
    room = torch.empty(t.numel() + 8, device=t.device, dtype=t.dtype)
    room[1:t.numel() + 1].copy_(t.flatten())
    return room[1:t.numel() + 1].view(t.shape)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3])
@pytest.mark.parametrize("odd", ["gamma", "h", "delta"])
def test_group_norm_prologue_leaves_operands_that_are_not_aligned(gpu, M, odd):
    """A norm weight off 16 bytes goes to the other prologue; past its rows everything goes to the parts, without an error."""
    from mxllm.ops import hybrid as hops

    K = 2048
    torch.manual_seed(M)
    t = dict(delta=torch.randn(M, K, device=gpu).bfloat16(), h=torch.randn(M, K, device=gpu), gamma=torch.rand(K, device=gpu) + 0.5)
    w = (torch.randn(6144, K, device=gpu) * K ** -0.5).bfloat16()
    if odd != "gamma" and M <= hops.NORM_M:
        return  # that prologue reads rows in 16-byte pieces and says so
    t[odd] = _off16(t[odd])
    r = hops.norm_linear(t["delta"], t["h"], t["gamma"], 8, 1e-5, w)
    assert (r is None) == (M > hops.NORM_M)
    if r is not None:
        h2 = t["h"].clone()
        y = hops.group_norm(t["delta"], h2, t["gamma"], 8, 1e-5, torch.bfloat16)
        assert torch.equal(r[1], h2) and rel_err(r[0], y.double() @ w.double().t()) < 2 ** -7


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 9, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(16, 1536), (48, 8192), (4112, 3584), (2048, 12288), (4096, 14336), (272, 21504), (8192, 4096)])
def test_stream_parts(gpu, M, N, K):
    """Products in segments of K (every length of block; few and uneven channel groups; strided rows): the sum is x w^T to f32
    (K products of f32 sums: 2^-24 sqrt(K) < 1e-5), and the norms that add it do what they do behind its rounding to
    bf16, to one rounding of a sum in another order (2^-8)."""
    torch.manual_seed(N + K + M)
    x = torch.randn(M, K + 8, device=gpu).bfloat16()[:, :K]
    w = (torch.randn(N, K, device=gpu) * K ** -0.5).bfloat16()
    if not _ops().stream_parts_segments(M, N, K):  # no segment fits LDS
        assert (M, K) == (32, 3584)
        with pytest.raises(RuntimeError):
            _ops().stream_parts(x, w)
        return
    parts = _ops().stream_parts(x, w)
    assert parts.shape == (_ops().stream_parts_segments(M, N, K), M, N)
    want = x.double() @ w.double().t()
    assert rel_err(parts.double().sum(0), want) < 1e-5
    h, g = torch.randn(M, N, device=gpu).bfloat16(), torch.randn(N, device=gpu).bfloat16()
    y, h2 = _ops().parts_norm(parts, h, g, 1e-5)
    hw = (h.double() + want.bfloat16().double())
    yw = hw * torch.rsqrt(hw.pow(2).mean(-1, keepdim=True) + 1e-5) * g.double()
    assert rel_err(h2, hw) < 2 ** -8 and rel_err(y, yw) < 2 ** -7
    r, gf = torch.randn(M, N, device=gpu), torch.randn(N, device=gpu)
    r2 = r.double() + want.bfloat16().double()
    y = _ops().group_norm_parts(parts, r, gf, 4, 1e-5)
    assert rel_err(r, r2) < 2 ** -8
    p = r2.view(M, 4, -1)
    assert rel_err(y, (p * torch.rsqrt(p.pow(2).mean(-1, keepdim=True) + 1e-5)).view(M, N) * gf.double()) < 2 ** -7


@pytest.mark.gpu
@pytest.mark.parametrize("odd", ["gamma", "h"])
def test_parts_norm_of_operands_that_are_not_aligned(gpu, odd):
    """They go to the norm that takes them, behind the parts' sum: the residual's bits, the norm to two roundings to bf16."""
    from mxllm import ops

    torch.manual_seed(3)
    M, N, K = 12, 2048, 8192
    t = dict(h=torch.randn(M, N, device=gpu).bfloat16(), gamma=torch.randn(N, device=gpu).bfloat16())
    parts = ops.linear_parts(torch.randn(M, K, device=gpu).bfloat16(), (torch.randn(N, K, device=gpu) * K ** -0.5).bfloat16())
    want = ops.parts_norm(parts, t["h"], t["gamma"], 1e-5)
    t[odd] = _off16(t[odd])
    y, h = ops.parts_norm(parts, t["h"], t["gamma"], 1e-5)
    assert torch.equal(h, want[1]) and rel_err(y, want[0]) < 2 ** -8


@pytest.mark.gpu
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Hq,Hkv", [(16, 2), (4, 4), (7, 1), (9, 1)])
def test_decode_attn_up_to_512_keys(gpu, D, Hq, Hkv):
    """Both splits of a sequence in one workgroup (up to 8 query heads of a KV head; 9 take two launches): lengths at the
    edges of waves and splits, none (zeros); stale rows are NaN.  Softmax weights of heads of 128 and every output are rounded to
    bf16 (2^-9 each): within 2^-7 of f64."""
    lens = [512, 0, 1, 63, 64, 65, 255, 256, 257, 320, 321, 511]
    B = len(lens)
    torch.manual_seed(D + Hq)
    kc = torch.full((B, Hkv, 600, D), float("nan"), device=gpu, dtype=torch.bfloat16)
    vc = kc.clone()
    q = torch.randn(B, Hq, D, device=gpu, dtype=torch.bfloat16)
    slots = torch.randperm(B, device=gpu).to(torch.int32)
    want = torch.zeros(B, Hq, D, dtype=torch.float64, device=gpu)
    for b, n in enumerate(lens):
        k, v = (torch.randn(Hkv, n, D, device=gpu, dtype=torch.bfloat16) for _ in range(2))
        kc[int(slots[b]), :, :n], vc[int(slots[b]), :, :n] = k, v
        if n:
            s = (q[b].double().view(Hkv, Hq // Hkv, 1, D) * k.double()[:, None]).sum(-1) * D ** -0.5
            want[b] = (torch.softmax(s, -1)[..., None] * v.double()[:, None]).sum(2).view(Hq, D)
    pos = torch.tensor(lens, dtype=torch.int32, device=gpu) - 1
    out = _ops().decode_attn(q, kc, vc, pos, slots, 512, D ** -0.5, 1, None, None).view(B, Hq, D)
    for b, n in enumerate(lens):
        if n == 0:
            assert not out[b].any()
        else:
            assert rel_err(out[b], want[b]) < 2 ** -7, (b, n)


@pytest.mark.gpu
def test_decode_attn_dealt_evenly_among_other_rows(gpu):
    """A row's cuts depend on the rows beside it: moved among them, and with others of other lengths, its output differs by
    the rounding of the softmax weights to bf16 against another maximum (2^-9 of each) and the output's own (2^-9), and
    the same call has the same bits."""
    torch.manual_seed(11)
    Hq, Hkv, D, B, room = 32, 8, 128, 24, 2048
    kc, vc = (torch.randn(B, Hkv, room, D, device=gpu, dtype=torch.bfloat16) for _ in range(2))
    q = torch.randn(B, Hq, D, device=gpu, dtype=torch.bfloat16)
    lens = torch.randint(200, room + 1, (B,), device=gpu).to(torch.int32)

    def run(rows, n):
        r = rows.long()
        return _ops().decode_attn(q[r], kc, vc, n[r].contiguous(), rows, room, D ** -0.5, 0, None, None).view(-1, Hq, D)

    rows = torch.arange(B, device=gpu, dtype=torch.int32)
    want = run(rows, lens)
    assert torch.equal(run(rows, lens), want)
    moved = rows[torch.randperm(B, device=gpu)]
    other = lens.clone()
    other[::2] = torch.randint(1, room + 1, (B // 2,), device=gpu).to(torch.int32)
    assert rel_err(run(moved, lens), want[moved.long()]) < 2 ** -7
    assert rel_err(run(rows, other)[1::2], want[1::2]) < 2 ** -7


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,room", [(32, 8, 256), (16, 1, 512)])
def test_decode_attn_of_few_splits_is_not_dealt(gpu, Hq, Hkv, room):
    """Many sequences of one split, or of two past 8 heads of a KV head, keep a workgroup a split (dealt evenly they took up to
    twice as long): a row's bits are those it has alone."""
    D, B = 128, 80 if room == 256 else 300
    torch.manual_seed(B)
    kc, vc = (torch.randn(B, Hkv, room, D, device=gpu, dtype=torch.bfloat16) for _ in range(2))
    q = torch.randn(B, Hq, D, device=gpu, dtype=torch.bfloat16)
    pos = torch.randint(40, room + 1, (B,), device=gpu).to(torch.int32)
    out = _ops().decode_attn(q, kc, vc, pos, None, room, D ** -0.5, 0, None, None)
    for b in range(0, B, 9):
        one = _ops().decode_attn(q[b:b + 1], kc[b:b + 1], vc[b:b + 1], pos[b:b + 1], None, room, D ** -0.5, 0, None, None)
        assert torch.equal(out[b], one[0])


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,lens,room", [(32, 8, [1, 15, 16, 17, 255, 256, 257, 0] + [1, 33, 700, 90] * 6, 700),
                                              (16, 1, [3000, 0, 1, 2600], 65536), (8, 8, [4000, 4096], 8448),
                                              (6, 2, [5] * 300, 256), (6, 2, [5] * 300, 700), (64, 8, [2000, 64, 65, 1999, 1, 1900], 3000)])
@pytest.mark.parametrize("paged", [False, True])
def test_decode_attn_dealt_evenly(gpu, Hq, Hkv, lens, room, paged):
    """More splits than the chip has places for: workgroups that take several sequences, sequences of many parts, of none
    (zeros) and of one, shares that end inside a block, more rows than a wave has lanes; stale rows are NaN.  Softmax
    weights are rounded to bf16 (2^-9 each) and so is the output: within 2^-7 of f64."""
    D, B, blk = 128, len(lens), 256
    torch.manual_seed(B + Hq)
    assert -(-room // blk) * Hkv * B > 512
    n_max = max(lens)
    nb = -(-n_max // blk)
    if paged:
        bt = torch.randperm(B * nb, device=gpu).to(torch.int32).view(B, nb)
        bt = torch.nn.functional.pad(bt, (0, -(-room // blk) - nb))  # blocks past a sequence's end are not read
        kc = torch.full((B * nb, Hkv, blk, D), float("nan"), device=gpu, dtype=torch.bfloat16)
    else:
        bt = None
        kc = torch.full((B, Hkv, room, D), float("nan"), device=gpu, dtype=torch.bfloat16)
    vc = kc.clone()
    q = torch.randn(B, Hq, D, device=gpu, dtype=torch.bfloat16)
    want = torch.zeros(B, Hq, D, dtype=torch.float64, device=gpu)
    for b, n in enumerate(lens):
        k, v = (torch.randn(Hkv, n, D, device=gpu, dtype=torch.bfloat16) for _ in range(2))
        if paged:
            for j in range(0, n, blk):
                kc[int(bt[b, j // blk]), :, :min(blk, n - j)] = k[:, j:j + blk]
                vc[int(bt[b, j // blk]), :, :min(blk, n - j)] = v[:, j:j + blk]
        else:
            kc[b, :, :n], vc[b, :, :n] = k, v
        if n:
            qd = q[b].double().view(Hkv, Hq // Hkv, D)
            s = (qd[:, :, None] * k.double()[:, None]).sum(-1) * D ** -0.5
            want[b] = (torch.softmax(s, -1)[..., None] * v.double()[:, None]).sum(2).view(Hq, D)
    pos = torch.tensor(lens, dtype=torch.int32, device=gpu)
    out = _ops().decode_attn(q, kc, vc, pos, None, room, D ** -0.5, 0, bt, None).view(B, Hq, D)
    for b, n in enumerate(lens):
        if n == 0:
            assert not out[b].any()
        else:
            assert rel_err(out[b], want[b]) < 2 ** -7, (b, n)


@pytest.mark.gpu
@pytest.mark.parametrize("filler", [[], [700] * 5])
def test_decode_attn_dealt_evenly_at_the_edges_of_shares(gpu, filler):
    """A row is dealt as six units without keys and one for every 16: the first row's length moves the second's keys past the end of
    a share (of 8 units, and of more where the others are long), one unit at a time: shares that end ahead of a row's keys, at
    them and behind their first unit, empty rows between, and the parts that the merge counts.  Within 2^-7 of f64, as above."""
    Hq, Hkv, D, room = 32, 8, 128, 2048
    for units in range(1, 30):
        lens = [16 * units, 0, 40, 0, 0, 16 * (units % 5) + 1, 129, 0, 15, 300, *filler]
        B = len(lens)
        assert room // 256 * Hkv * B > 512
        torch.manual_seed(units)
        kc, vc = (torch.full((B, Hkv, room, D), float("nan"), device=gpu, dtype=torch.bfloat16) for _ in range(2))
        q = torch.randn(B, Hq, D, device=gpu, dtype=torch.bfloat16)
        for b, n in enumerate(lens):
            kc[b, :, :n], vc[b, :, :n] = (torch.randn(Hkv, n, D, device=gpu, dtype=torch.bfloat16) for _ in range(2))
        out = _ops().decode_attn(q, kc, vc, torch.tensor(lens, dtype=torch.int32, device=gpu), None, room, D ** -0.5, 0, None, None).view(B, Hq, D)
        for b, n in enumerate(lens):
            if n == 0:
                assert not out[b].any()
                continue
            s = (q[b].double().view(Hkv, -1, 1, D) * kc[b, :, None, :n].double()).sum(-1) * D ** -0.5
            want = (torch.softmax(s, -1)[..., None] * vc[b, :, None, :n].double()).sum(2).view(Hq, D)
            assert rel_err(out[b], want) < 2 ** -7, (units, b, n)


@pytest.mark.gpu
@pytest.mark.parametrize("D,Hq,Hkv", [(32, 4, 2), (64, 32, 8), (128, 8, 1)])
@pytest.mark.parametrize("lens", [[1], [127, 1, 129], [256, 65, 700, 128, 3]])
def test_prompt_attention(gpu, D, Hq, Hkv, lens):
    """Prompts of several sequences in two launches: the bits of RoPE split, cache copies and attention sequence by
    sequence; cache rows that no prompt owns stay as they are."""
    from mxllm.ops.hybrid import PromptRows

    torch.manual_seed(D + len(lens))
    T, nslots, blk = sum(lens), len(lens) + 1, 256
    maxb = (max(lens) + blk - 1) // blk
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, device=gpu, dtype=torch.bfloat16)
    cos, sin = ref.rope_tables(max(lens), D, 500000.0, None, gpu)
    bt = torch.randperm(nslots * maxb, device=gpu).to(torch.int32).view(nslots, maxb)
    slots = torch.randperm(nslots)[:len(lens)].tolist()
    kc = torch.randn(nslots * maxb, Hkv, blk, D, device=gpu, dtype=torch.bfloat16)
    vc = torch.randn_like(kc)
    kc2, vc2 = kc.clone(), vc.clone()
    rows = PromptRows(lens, gpu, slots)
    o = _ops().prompt_attention(qkv, cos, sin, rows.rowinfo, rows.attn_blocks(max(lens)), max(lens), Hq, Hkv, kc, vc, bt,
                                D ** -0.5)
    at = 0
    for n, slot in zip(lens, slots):
        q, k, v = _ops().rope_split(qkv[at:at + n].contiguous(), cos, sin, 1, n, Hq, Hkv, D, None)
        assert torch.equal(o[at:at + n], _ops().attn_fwd(q, k, v, True, D ** -0.5)[0].view(n, Hq * D))
        for j in range(0, n, blk):
            m = min(blk, n - j)
            kc2[int(bt[slot, j // blk]), :, :m] = k[0, :, j:j + m]
            vc2[int(bt[slot, j // blk]), :, :m] = v[0, :, j:j + m]
        at += n
    assert torch.equal(kc, kc2) and torch.equal(vc, vc2)


@pytest.mark.gpu
@pytest.mark.parametrize("D,Hq,Hkv,S", [(32, 4, 2, 1), (64, 8, 2, 300), (128, 8, 8, 129)])
def test_prefill_attention_runs_the_kernels(gpu, D, Hq, Hkv, S):
    """One sequence on the GPU: the bits of RoPE split and flash attention, K and V handed out as [Hkv, S, D]."""
    from mxllm.ops.decode import prefill_attention

    torch.manual_seed(D + S)
    qkv = torch.randn(S, (Hq + 2 * Hkv) * D, device=gpu, dtype=torch.bfloat16)
    cos, sin = ref.rope_tables(S, D, 500000.0, None, gpu)
    kept = []
    o = prefill_attention(qkv, cos, sin, lambda k, v: kept.extend((k, v)), S, Hq, Hkv, D)
    q, k, v = _ops().rope_split(qkv, cos, sin, 1, S, Hq, Hkv, D, None)
    assert torch.equal(kept[0], k[0]) and torch.equal(kept[1], v[0])
    assert torch.equal(o, _ops().attn_fwd(q, k, v, True, D ** -0.5)[0].view(S, Hq * D))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 48, 2048), (2, 8208, 2048), (3, 48, 2048), (8, 8208, 3072), (7, 16, 512), (9, 32, 1536),
                                   (12, 1040, 3072), (16, 3088, 4096), (16, 48, 2048), (17, 48, 2560), (31, 16, 512), (9, 48, 2560),
                                   (9, 16, 3072), (13, 2064, 3584), (16, 48, 4608), (13, 48, 4096), (16, 3072, 4096), (9, 4112, 4096)])
def test_skinny_linear_fragments(gpu, M, N, K):
    """The decode GEMM's ways to read (4 and 8 K parts, all loads of a block ahead or not, blocks of 8 and of 16 rows and tokens,
    the kernel that stays) against fp64, plain and with SwiGLU; row-strided x, rows and groups at their edges."""
    from mxllm import ops

    torch.manual_seed(M + N + K)
    x = torch.randn(M, K + 64, device=gpu, dtype=torch.bfloat16)[:, :K]
    w = torch.randn(N, K, device=gpu, dtype=torch.bfloat16) * 0.05
    y = _ops().skinny_linear(x, w)
    assert rel_err(y, x.double() @ w.double().t()) < 2 ** -8  # one bf16 rounding
    assert torch.equal(_ops().skinny_linear_swiglu(x, w), ops.swiglu(y))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 16, 512), (2, 48, 4608), (2, 4112, 4096), (3, 48, 2048), (8, 4112, 4096), (8, 48, 14336),
                                   (5, 16, 1024), (9, 48, 4096)])
def test_w8_linear_fragments(gpu, M, N, K):
    """The e4m3 decode GEMM's ways to read (blocks of 8 and of 16 rows, K's rest by smaller blocks, the kernel that stays)
    against fp64 on the same codes: one bf16 rounding."""
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K + 64, device=gpu, dtype=torch.bfloat16)[:, :K]
    q, s = _stream_weight(torch.randn(N, K, device=gpu, dtype=torch.bfloat16) * 0.05, True)
    ref = x.double() @ (q.view(torch.float8_e4m3fn).double() * s.double()[:, None]).t()
    assert rel_err(_ops().w8_linear(x, q, s), ref) < 2 ** -8
