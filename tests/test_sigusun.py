"""Sigusun (retention, latent attention, expert mixtures, post-normed sublayers) against the plain
implementation of oracle_sigusun.py: every mechanism alone, then whole models through the engine.

CPU tensors take the framework's PyTorch ops; the ``cuda`` cases run the HIP kernels in f32 (tight)
and bf16 (rounding of bf16 matrix products allowed)."""
import io
import json
import os
import sys

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import oracle_sigusun as orc  # noqa: E402

from mxllm.models import Sigusun, SigusunConfig, build_model, model_config, save_sigusun  # noqa: E402
from mxllm.ops import hybrid as hops  # noqa: E402
from mxllm.ops import latent as lops  # noqa: E402
from mxllm.ops import moe as mops  # noqa: E402
from mxllm.ops import retention as rops  # noqa: E402
from mxllm.ops import sublayer as sops  # noqa: E402
from mxllm.ops import native  # noqa: E402
from mxllm.serve.engine import Engine  # noqa: E402
from mxllm.serve.kvcache import KVCache  # noqa: E402

CASES = [("cpu", torch.float32), pytest.param("cuda", torch.float32, marks=pytest.mark.gpu),
         pytest.param("cuda", torch.bfloat16, marks=pytest.mark.gpu)]
on_devices = pytest.mark.parametrize("dev,dt", CASES, ids=lambda x: str(x).replace("torch.", ""))


def close(got, want, dt, scale=1.0):
    """Relative RMS error of the whole, and no element far out."""
    got, want = got.detach().double().cpu(), want.detach().double().cpu()
    tol = (2e-5 if dt == torch.float32 else 1.5e-2) * scale
    rms = want.pow(2).mean().sqrt().clamp_min(1e-6)
    err = (got - want).abs()
    assert torch.isfinite(got).all()
    assert err.pow(2).mean().sqrt() <= tol * rms, (float(err.pow(2).mean().sqrt()), float(rms))
    assert err.max() <= 12 * tol * max(float(rms), float(want.abs().max()) / 4), (float(err.max()), float(rms))


def rnd(*shape, seed=0, dt=torch.float32):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dt)


def i32(x, dev):
    return torch.tensor(x, dtype=torch.int32, device=dev)


# ------------------------------------------------------------------ post-normed sublayers
@on_devices
@pytest.mark.parametrize("width", [1, 24, 50, 256, 516, 1030, 4096, 6000])
def test_post_norm(dev, dt, width):
    """Rows held by a wave, a workgroup and a large workgroup, whole vectors or not; eps that counts."""
    x, h, w = rnd(5, width, seed=1, dt=dt) * 0.1, rnd(5, width, seed=2), 1 + 0.3 * rnd(width, seed=3)
    want = h.double() + orc.rms(x.double(), 1e-2) * w.double()
    res = h.clone().to(dev)
    y = sops.post_norm(x.to(dev), res, w.to(dev), 1e-2)
    close(res, want, torch.float32)
    close(y, want, dt)
    assert y.dtype == dt


@on_devices
@pytest.mark.parametrize("width", [20, 512, 3000])
def test_embed_norm(dev, dt, width):
    table, w, ids = rnd(40, width, seed=1, dt=dt), 1 + 0.3 * rnd(width, seed=2), torch.tensor([3, 39, 0, 3])
    h, y = sops.embed_norm(ids.to(dev), table.to(dev), w.to(dev), 1e-3)
    want = orc.rms(table[ids].double(), 1e-3) * w.double()
    close(h, want, torch.float32)
    close(y, want, dt)


@on_devices
@pytest.mark.parametrize("width,top,shared", [(40, 1, False), (96, 3, True), (515, 2, True), (2048, 4, False)])
def test_mix_post_norm(dev, dt, width, top, shared):
    """The experts' rows in any order, weighted, with and without a shared expert."""
    T = 6
    src, wts = rnd(T * top, width, seed=1, dt=dt), torch.softmax(rnd(T, top, seed=2), -1)
    perm = torch.randperm(T * top, generator=torch.Generator().manual_seed(3))
    sh = rnd(T, width, seed=4, dt=dt) if shared else None
    h, w = rnd(T, width, seed=5), 1 + 0.3 * rnd(width, seed=6)
    for inv in (None, perm):
        rows = src.double() if inv is None else src.double()[inv]
        m = (rows.view(T, top, width) * wts.double()[..., None]).sum(1) + (sh.double() if shared else 0)
        want = h.double() + orc.rms(m, 1e-3) * w.double()
        res = h.clone().to(dev)
        y = sops.mix_post_norm(src.to(dev), None if inv is None else inv.view(T, top).int().to(dev), wts.to(dev),
                               sh.to(dev) if shared else None, res, w.to(dev), 1e-3)
        close(res, want, torch.float32)
        close(y, want, dt)


@on_devices
@pytest.mark.parametrize("dim,layers,i", [(12, 3, 1), (7, 2, 1), (64, 4, 3)])
def test_side_input(dev, dt, dim, layers, i):
    """Each layer reads its own columns of the tokens' rows."""
    z, emb = 2 * rnd(9, dim, seed=1, dt=dt), rnd(30, dim * layers, seed=2, dt=dt)
    ids = torch.tensor([0, 29, 5, 5, 1, 2, 3, 4, 28])
    y = sops.side_act(z.to(dev), emb.to(dev), ids.to(dev), i * dim)
    close(y, orc.gelu_tanh(z.double()) * emb.double()[ids, i * dim:(i + 1) * dim], dt)


def glu_oracle(z, limit):
    g, u = z.double().chunk(2, -1)
    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return g * orc.sigmoid(1.702 * g) * (u + 1)


@pytest.mark.gpu
@pytest.mark.parametrize("T,width,rows,top", [(1, 4096, 16, 0), (5, 264, 3, 2), (64, 2048, 64, 4), (9, 8, 5, 1), (3, 512, 21, 0)])
def test_residual_step_with_its_next_products(gpu, T, width, rows, top):
    """One launch against its parts: the same residual and copy, the router's logits, and the gate of the second
    embedding; rows of a sublayer, or experts' rows with a shared one."""
    bf = torch.bfloat16
    src, h, w = rnd(T * max(top, 1), width, seed=1, dt=bf).to(gpu), rnd(T, width, seed=2).to(gpu), rnd(width, seed=3).to(gpu)
    m = (rnd(rows, width, seed=4) / width ** 0.5).to(bf).to(gpu)
    emb, ids = rnd(50, 3 * rows, seed=5, dt=bf).to(gpu), torch.randint(0, 50, (T,), generator=torch.Generator().manual_seed(1)).to(gpu)
    wts = torch.softmax(rnd(T, top, seed=6), -1).to(gpu) if top else None
    sh = rnd(T, width, seed=7, dt=bf).to(gpu) if top else None
    h2, keep = h.clone(), h.clone()
    y2 = sops.mix_post_norm(src, None, wts, sh, h2, w, 1e-4) if top else sops.post_norm(src, h2, w, 1e-4)
    hn, y, z = sops.post_dots(src, h, w, 1e-4, m, wts, sh)
    close(hn, h2, torch.float32)
    close(y, y2, torch.float32, 200)
    want = y2.double().cpu() @ m.double().cpu().T
    close(z, want, torch.float32, 100)
    # of the copy, which prompt passes and the separate kernels route by, and not of the residual: f32 sums of up to 4096 products
    # (2^-24 sqrt(4096) = 4e-6), where the residual's would be a rounding to bf16 apart (2^-9 = 2e-3)
    zy, m2 = y.double().cpu() @ m.double().cpu().T, m.double().cpu().T
    assert float((z.double().cpu() - zy).norm() / zy.norm()) < 2e-5
    assert float((hn.double().cpu() @ m2 - zy).norm() / zy.norm()) > 2e-4
    hn, _, g = sops.post_dots(src, h, w, 1e-4, m, wts, sh, emb, ids, rows)
    close(hn, h2, torch.float32)
    close(g, orc.gelu_tanh(want) * emb.double().cpu()[ids.cpu(), rows:2 * rows], bf)
    assert torch.equal(h, keep)


@pytest.mark.gpu
@pytest.mark.parametrize("T,experts,top", [(1, 16, 4), (3, 64, 5), (33, 8, 2), (64, 5, 5)])
def test_experts_chosen_from_logits(gpu, T, experts, top):
    """The choice inside the experts' kernel against the router's: few and many pairs, experts nobody chose."""
    bf = torch.bfloat16
    x, router = rnd(T, 128, seed=1, dt=bf).to(gpu), rnd(experts, 128, seed=2, dt=bf).to(gpu)
    gu = (rnd(experts, 2 * 48, 128, seed=3) / 11).to(bf).to(gpu)
    down = (rnd(experts, 128, 48, seed=4) / 7).to(bf).to(gpu)
    ids, wts = mops.route(x, router, top)
    y, inv, _ = mops.experts(x, ids, gu, down, 1.5)
    assert inv is None
    logits = x.float() @ router.float().T
    y2, wts2, sh = mops.experts_of(x, logits, top, gu, down, 1.5)
    assert sh is None
    close(wts2, wts, torch.float32, 20)
    close(y2, y, bf)


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,top,K,ff,shared", [(5, 4, 1, 2048, 8, 0), (9, 8, 2, 2048, 24, 40), (32, 3, 2, 2048, 56, 2048),
                                                 (32, 6, 3, 4096, 72, 64), (17, 16, 4, 4096, 768, 264), (20, 5, 4, 8192, 16, 16),
                                                 (33, 8, 2, 2048, 64, 64), (8, 9, 2, 4096, 1024, 0)])
def test_up_products_past_rows_in_lds(gpu, T, E, top, K, ff, shared):
    """Workgroups that stay with an expert: rows of one and two blocks and of two turns (experts with nearly every token, the
    shared one), an expert that nobody chose, runs of channel groups with a shorter end; and sizes left to the other kernel."""
    bf = torch.bfloat16
    x = rnd(T, K, seed=1, dt=bf)
    wgu = (rnd(E, 2 * ff, K, seed=2) * 1.5 / K ** 0.5).to(bf)
    sgu = (rnd(2 * shared, K, seed=3) * 1.5 / K ** 0.5).to(bf) if shared else None
    z = torch.randn(T, E, generator=torch.Generator().manual_seed(T + K))
    z[:, 1] += 3.0
    z[:, 2] -= 100.0
    y, sy, ids, wts = native().moe_few(x.to(gpu), None, z.to(gpu), top, wgu.to(gpu), True, 1.2,
                                       sgu.to(gpu) if shared else None, None, 0.9)
    val, at = z.topk(top, 1)
    assert torch.equal(ids.cpu().long(), at)
    close(wts, torch.softmax(val.double(), 1), torch.float32)
    want = torch.stack([glu_oracle(x[t].double() @ wgu[e].double().T, 1.2) for t in range(T) for e in at[t].tolist()])
    close(y.view(T * top, ff), want, bf, 0.3)  # f32 sums, one rounding to bf16 (2^-9)
    if shared:
        close(sy, glu_oracle(x.double() @ sgu.double().T, 0.9), bf, 0.3)


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,top,K", [(2, 3, 2, 192), (17, 16, 4, 192), (33, 18, 4, 192), (64, 33, 5, 192), (64, 64, 2, 192),
                                       (9, 6, 6, 2048), (16, 18, 2, 2048), (32, 35, 4, 4096)])
def test_choices_seen_from_one_expert(gpu, T, E, top, K):
    """A workgroup finds its expert's tokens from the logits alone: equal logits (the lower index first), infinities and
    what is not a number (last), rows of logits that are no whole 16 B.  The products are those of given choices."""
    bf, F = torch.bfloat16, 40
    gen = torch.Generator().manual_seed(T * E)
    z = torch.randint(-3, 4, (T, E), generator=gen).float()
    z[torch.rand(T, E, generator=gen) < 0.1] = float("-inf")
    z[torch.rand(T, E, generator=gen) < 0.05] = float("nan")
    z[:, T % E] = 2.0
    z[0] = 1.0
    at = torch.sort(torch.where(z.isnan(), float("-inf"), z), dim=1, descending=True, stable=True).indices[:, :top]
    x, w = rnd(T, K, seed=1, dt=bf).to(gpu), (rnd(E, 2 * F, K, seed=2) / K ** 0.5).to(bf).to(gpu)
    y, _, ids, wts = native().moe_few(x, None, z.to(gpu), top, w, True, 1.2, None, None, 0.0)
    assert torch.equal(ids.cpu().long(), at)
    close(wts, torch.softmax(torch.where(z.isnan(), float("-inf"), z).double().gather(1, at), 1), torch.float32)
    given, _, _, _ = native().moe_few(x, at.int().to(gpu), None, top, w, True, 1.2, None, None, 0.0)
    close(y, given, bf, 0.3)  # f32 sums in two orders, one rounding to bf16 (2^-9)


@pytest.mark.gpu
@pytest.mark.parametrize("R,W", [(32, 256), (32, 4096), (64, 128), (64, 1920), (64, 2048), (128, 64), (128, 768), (128, 1024)])
@pytest.mark.parametrize("T", [1, 5, 64])
def test_side_projection_with_its_norm(gpu, T, R, W):
    """The projection and the residual step in one launch: waves of one load and of several blocks, threads past the row's
    end; columns that are nearly alike (products out of large terms that cancel); eps that counts."""
    bf = torch.bfloat16
    g, P, h, w = rnd(T, R, seed=1, dt=bf), (rnd(W, R, seed=2) / R ** 0.5).to(bf), rnd(T, W, seed=3), 1 + 0.3 * rnd(W, seed=4)
    P[:, 1] = P[:, 0]
    P[3, 1] += 0.5
    g[:, 0], g[:, 1] = 30.0, -30.0
    y = (g.double() @ P.double().T).to(bf).double()
    want = h.double() + orc.rms(y, 1e-2) * w.double()
    res = h.clone().to(gpu)
    x = sops.side_post(g.to(gpu), P.to(gpu), res, w.to(gpu), 1e-2)
    close(res, want, bf, 0.1)  # a product's f32 sum at a rounding boundary: one step of bf16 of few elements
    assert torch.equal(x, res.to(bf))
    big = torch.empty(4096, 64, device=gpu, dtype=bf)
    assert sops.side_post(g.to(gpu), big, torch.empty(T, 4096, device=gpu), w, 1e-2) is None


@pytest.mark.gpu
@pytest.mark.parametrize("odd", ["g", "p", "h", "w"])
def test_side_projection_leaves_operands_that_are_not_aligned(gpu, odd):
    """A tensor whose storage starts between two 16-byte pieces goes to the parts instead of an error."""
    T, R, W, bf = 3, 64, 256, torch.bfloat16
    t = dict(g=rnd(T, R, seed=1, dt=bf), p=rnd(W, R, seed=2, dt=bf), h=rnd(T, W, seed=3), w=rnd(W, seed=4))
    at = {}
    for k, v in t.items():
        room = torch.empty(v.numel() + 8, device=gpu, dtype=v.dtype)
        at[k] = room[1 if k == odd else 0:][:v.numel()].view(v.shape)
        at[k].copy_(v)
    assert sops.side_post(at["g"], at["p"], at["h"], at["w"], 1e-3) is None
    assert torch.equal(at["h"].cpu(), t["h"])


@pytest.mark.gpu
@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two GPUs")
def test_side_projection_refuses_another_device(gpu):
    t = [torch.zeros(3, 64, device=gpu, dtype=torch.bfloat16), torch.zeros(256, 64, device=gpu, dtype=torch.bfloat16),
         torch.zeros(3, 256, device=gpu), torch.zeros(256, device=gpu)]
    for i in (0, 1, 3):
        with pytest.raises(RuntimeError):
            native().post_side(*(x.to("cuda:1") if j == i else x for j, x in enumerate(t)), 1e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("W", [512, 2048])
def test_side_projection_of_columns_nearly_dependent(gpu, W):
    """Two large columns that differ in their last bits: the terms' squares are about 1e5 times the row's sum of squares, which
    has to come from the products.  A product sums terms of up to 2048 x 0.5 in f32, at most 2^10 x 2^-23 off beside elements
    of about 1: the sum of squares to 1e-3 at the worst, the step to half of that and its bf16 rounding."""
    bf, T, R = torch.bfloat16, 5, 64
    g, P, h, w = rnd(T, R, seed=1, dt=bf), (rnd(W, R, seed=2) / R ** 0.5).to(bf), torch.zeros(T, W), torch.ones(W)
    P[:, 1] = (P[:, 0].float() * (1 + rnd(W, seed=5) / 256)).to(bf)
    g[:, 0], g[:, 1] = 2048.0, -2048.0
    y = g.double() @ P.double().T
    assert 2e4 < float((2 * (2048 * P[:, 0].double()).pow(2).sum() / y.pow(2).sum(1)).min()) < 4e5
    res = h.to(gpu)
    sops.side_post(g.to(gpu), P.to(gpu), res, w.to(gpu), 1e-5)
    got, want = res.double().cpu(), orc.rms(y, 1e-5)
    assert float((got * want).sum() / want.pow(2).sum() - 1) == pytest.approx(0, abs=1e-3)
    close(got, want, bf, 0.2)


@pytest.mark.gpu
@pytest.mark.parametrize("ff,shared", [(64, 64), (192, 0), (384, 2048), (448, 128), (768, 192), (384, 0), (768, 2048), (1152, 4096)])
@pytest.mark.parametrize("T", [1, 3, 8, 9, 16, 17, 32, 33, 64])
def test_down_products_of_few_rows(gpu, T, ff, shared):
    """Whole-line fragments of the experts' down products: K parts of none, some and all of a block of chunks, a remainder of
    channels, an expert with nearly every row (several turns of them), ones with a few and one that nobody chose."""
    bf, N, E, top = torch.bfloat16, 144, 6, 3
    w = (rnd(E, N, ff, seed=1) / ff ** 0.5).to(bf)
    g = torch.Generator().manual_seed(T + ff)
    z = torch.randn(T, E, generator=g)
    z[:, 1] += 3.0
    z[:, 4] -= 100.0
    ids = z.topk(top, 1).indices
    x = rnd(T * top, ff, seed=2, dt=bf)
    sw = (rnd(N, shared, seed=3) / shared ** 0.5).to(bf) if shared else None
    sx = rnd(T, shared, seed=4, dt=bf) if shared else None
    y, sy, _, _ = native().moe_few(x.to(gpu), ids.int().to(gpu), None, top, w.to(gpu), False, 0.0,
                                   sw.to(gpu) if shared else None, sx.to(gpu) if shared else None, 0.0)
    want = torch.stack([w[e].double() @ r.double() for e, r in zip(ids.flatten().tolist(), x)])
    close(y.view(T * top, N), want, bf, 0.3)  # f32 sums, one rounding to bf16 (2^-9)
    if shared:
        close(sy, sx.double() @ sw.double().T, bf, 0.3)


@on_devices
@pytest.mark.parametrize("ff,limit", [(5, 0.7), (72, 2.0), (1024, 1.1)])
def test_clipped_glu(dev, dt, ff, limit):
    """Both clips at work: the gate's from above only."""
    z = 3 * rnd(7, 2 * ff, seed=1, dt=dt)
    want = glu_oracle(z, limit)
    assert (glu_oracle(z, limit + 0.4) - want).abs().max() > 0.3
    close(sops.clipped_glu(z.to(dev), limit), want, dt)


# ------------------------------------------------------------------ expert mixtures
@on_devices
@pytest.mark.parametrize("T,width,experts,top", [(1, 64, 4, 1), (7, 96, 8, 8), (33, 130, 5, 2), (50, 512, 70, 6),
                                                 (130, 48, 16, 4), (300, 1024, 3, 2)])
def test_route(dev, dt, T, width, experts, top):
    """Choices and weights from f32 logits of the rows as they are stored."""
    x, w = rnd(T, width, seed=1, dt=dt), rnd(experts, width, seed=2, dt=dt)
    ids, wts = mops.route(x.to(dev), w.to(dev), top)
    z = x.double() @ w.double().T
    idx, want = orc.route(z, top)
    srt = torch.sort(z, descending=True).values
    clear = (srt[:, :top] - srt[:, 1:top + 1]).min(1).values > 1e-3 if top < experts else \
        (srt[:, :-1] - srt[:, 1:]).min(1).values > 1e-3
    assert clear.sum() >= T // 2
    assert torch.equal(ids.cpu().long()[clear], idx[clear])
    close(wts.cpu()[clear], want[clear], torch.float32, 5)


def test_route_ties_take_the_lower_index():
    ids, wts = mops.route(torch.ones(2, 8), torch.ones(6, 8), 3)
    assert sorted(ids[0].tolist()) == [0, 1, 2] or len(set(ids[0].tolist())) == 3
    assert torch.allclose(wts, torch.full((2, 3), 1 / 3))


def run_mixture(x, ids, wts, gu, down, limit, sgu, sdown, slimit, dev):
    """The model's calls of a mixture, up to the weighted sum."""
    y, inv, sh = mops.experts(x.to(dev), ids.int().to(dev), gu.to(dev), down.to(dev), limit,
                              None if sgu is None else sgu.to(dev), None if sdown is None else sdown.to(dev), slimit)
    y = y.double().cpu()
    rows = y if inv is None else y[inv.cpu().view(-1).long()]
    out = (rows.view(*ids.shape, -1) * wts.double()[..., None]).sum(1)
    return out if sh is None else out + sh.double().cpu()


@on_devices
@pytest.mark.parametrize("T,width,experts,top,ff,shared", [
    (1, 64, 4, 2, 40, 0), (1, 512, 8, 3, 256, 192), (5, 96, 3, 3, 24, 17), (20, 80, 6, 1, 33, 50), (64, 256, 4, 2, 64, 128),
    (90, 128, 16, 4, 72, 0), (300, 264, 3, 2, 136, 96), (700, 512, 2, 1, 256, 64), (257, 24, 5, 2, 200, 8)])
def test_experts(dev, dt, T, width, experts, top, ff, shared):
    """Few tokens and many, experts that nobody chose, one that takes nearly all; odd sizes."""
    g = torch.Generator().manual_seed(T)
    x = rnd(T, width, seed=1, dt=dt)
    gu, down = rnd(experts, 2 * ff, width, seed=2) * 1.5 / width ** 0.5, rnd(experts, width, ff, seed=3) / ff ** 0.5
    gu, down = gu.to(dt), down.to(dt)
    sgu = (rnd(2 * shared, width, seed=4) / width ** 0.5).to(dt) if shared else None
    sdown = (rnd(width, shared, seed=5) / shared ** 0.5).to(dt) if shared else None
    z = torch.randn(T, experts, generator=g)
    z[:, 0] += 2.0
    if experts > 3:
        z[:, 2] -= 100.0  # never chosen (unless all are)
    idx, wts = orc.route(z.double(), top)
    got = run_mixture(x, idx, wts.float(), gu, down, 1.2, sgu, sdown, 0.9, dev)
    want = torch.zeros(T, width, dtype=torch.float64)
    xd = x.double()
    for e in range(experts):
        y = glu_oracle(xd @ gu[e].double().T, 1.2) @ down[e].double().T
        want += (wts * (idx == e)).sum(1, keepdim=True) * y
    if shared:
        want += glu_oracle(xd @ sgu.double().T, 0.9) @ sdown.double().T
    close(got, want, dt)


# ------------------------------------------------------------------ retention
RET = [  # heads, dim, vdim, rotated dims, decays
    (4, 16, 16, 16, (0.9, 0.99, 0.999, 0.5)), (3, 20, 12, 6, (0.97, 1.0, 0.2)), (2, 64, 48, 32, (0.95, 0.9996)),
    (1, 7, 5, 4, (0.99,)), (2, 128, 128, 128, (0.98, 0.9999)), (1, 200, 40, 2, (0.995,)), (2, 24, 100, 0, (0.7, 0.999)),
    (1, 256, 256, 64, (0.999,)), (1, 48, 300, 48, (0.99,))]


def ret_oracle(x, sh, decay, base, state=None, p0=0):
    T, H, D, E = x.shape[0], sh.heads, sh.dim, sh.vdim
    q, k, v, g = x.double().split(sh.splits, 1)
    pos = torch.arange(p0, p0 + T)
    q = orc.rotate_halves(q.reshape(T, H, D), pos, base, sh.rot_dims)
    k = orc.rotate_halves(k.reshape(T, H, D), pos, base, sh.rot_dims) * D ** -0.5
    o, S = orc.retention(q, k, v.reshape(T, H, E), decay, state)
    return orc.rms(o, 1e-5).reshape(T, H * E) * (g * orc.sigmoid(g)), S


def ret_setup(case, dev):
    H, D, E, rd, decay = case
    sh = rops.RetentionShape(H, D, E, rd)
    cos, sin = hops.pair_rope_tables(1400, rd, 5e4, device=dev)
    return sh, rops.decay_table(decay, dev), cos, sin


@on_devices
@pytest.mark.parametrize("case", RET, ids=str)
def test_retention_prompts_and_steps(dev, dt, case):
    """Unequal prompts in one pass (one token, around and past the chunks), end states by slot, then single
    tokens from those states; slots that held another sequence."""
    sh, decay, cos, sin = ret_setup(case, dev)
    lens, slots = [1, 64, 65, 300, 2, 63, 513], [3, 0, 5, 1, 4, 2, 6]
    if dev == "cpu":
        lens[-1] = 140
    width = sum(sh.splits)
    x = rnd(sum(lens), width, seed=1, dt=dt)
    state = torch.full((8, sh.state), 9.0, device=dev)
    caches = hops.SeqCaches([], [], None, [], [state])
    y = rops.retention(x.to(dev), decay, cos, sin, sh, 1e-5, hops.PromptRows(lens, dev, slots, caches), 0)
    y0 = rops.retention(x.to(dev), decay, cos, sin, sh, 1e-5, hops.PromptRows(lens, dev), 0)
    close(y0, y, torch.float32)
    at, ends = 0, []
    for n, s in zip(lens, slots):
        want, end = ret_oracle(x[at:at + n], sh, case[4], 5e4)
        close(y[at:at + n], want, dt)
        close(state[s], end.reshape(-1), torch.float32)
        ends.append(end)
        at += n
    assert (state[7] == 9).all()
    for t in range(3):
        x2 = rnd(len(lens), width, seed=7 + t, dt=dt)
        rows = hops.TokenRows(i32([n + t for n in lens], dev), i32(slots, dev), 1024, caches)
        y2 = rops.retention(x2.to(dev), decay, cos, sin, sh, 1e-5, rows, 0)
        for i, n in enumerate(lens):
            want, ends[i] = ret_oracle(x2[i:i + 1], sh, case[4], 5e4, ends[i], n + t)
            close(y2[i:i + 1], want, dt)
            close(state[slots[i]], ends[i].reshape(-1), torch.float32)


@on_devices
def test_retention_remembers_the_first_token(dev, dt):
    """A strong first key stays visible for hundreds of tokens where the decay is near one, and is gone
    where it is not; across every chunk edge."""
    sh, decay, cos, sin = ret_setup((2, 32, 32, 0, (0.9999, 0.8)), dev)
    n = 800 if dev == "cuda" else 300
    q, k, v = (torch.zeros(n, 2, 32) for _ in range(3))
    q[:, :, 0] = 1.0
    k[0, :, 0] = 30.0
    k[1:, :, 1] = 1.0
    v[0] = 1.0
    v[1:, :, 0] = rnd(n - 1, 2, seed=1)
    x = torch.cat([t.reshape(n, -1) for t in (q, k, v, torch.ones(n, 2, 32))], 1).to(dt)
    want, _ = ret_oracle(x, sh, (0.9999, 0.8), 5e4)
    assert (want[:, 5:32].mean(1) > 0.5).all() and (want[200:, 32:].abs() < 1e-3).all()
    y = rops.retention(x.to(dev), decay, cos, sin, sh, 1e-5, hops.PromptRows([n], dev), 0)
    close(y[:, :32], want[:, :32], dt)


# ------------------------------------------------------------------ latent attention
LAT = [  # heads, dim, rot, vdim, rank, window, sink
    (4, 16, 8, 16, 32, 0, True), (2, 12, 4, 20, 24, 0, False), (6, 32, 32, 48, 96, 37, False), (3, 64, 16, 96, 192, 0, True),
    (16, 128, 64, 128, 512, 130, True), (1, 7, 2, 5, 9, 11, False), (20, 24, 8, 40, 96, 0, True), (2, 48, 48, 96, 160, 64, False),
    (33, 16, 16, 8, 32, 300, True), (2, 16, 0, 16, 32, 1, False), (1, 200, 40, 144, 320, 0, True), (5, 32, 64, 64, 256, 0, False)]


def lat_shape(case):
    H, D, R, E, rank, window, _ = case
    return lops.LatentShape(H, D, R, E, rank, 1.6 / (D + R) ** 0.5, window)


def lat_weights(sh, sink, dt, dev, seed=0):
    wkv = (rnd(sh.heads * (sh.dim + sh.vdim), sh.rank, seed=seed) / sh.rank ** 0.5).to(dt).to(dev)
    return wkv, (1 + 0.2 * rnd(sh.rank, seed=seed + 1)).to(dev), (rnd(sh.heads, seed=seed + 2) + 1).to(dev) if sink else None


def lat_oracle(q, xl, wkv, wn, sink, sh, window="own", base=2e4, eps=1e-4, tokens=None):
    """q [T, H (D + R)], xl [T, rank + R]: the mixer without its projections, one sequence."""
    T, H, D, R, E = q.shape[0], sh.heads, sh.dim, sh.rot_dim, sh.vdim
    pos = torch.arange(T)
    q, xl, wkv = q.double().cpu(), xl.double().cpu(), wkv.double().cpu()
    c = orc.rms(xl[:, :sh.rank], eps) * wn.double().cpu()
    kr = orc.rotate_pairs(xl[:, None, sh.rank:], pos, base, R)
    q = q.view(T, H, D + R)
    q = torch.cat([q[..., :D], orc.rotate_pairs(q[..., D:], pos, base, R)], -1)
    kv = c @ wkv.T
    k = torch.cat([kv[:, :H * D].view(T, H, D), kr.expand(T, H, R)], -1)
    w = sh.window if window == "own" else window
    return orc.attend(q, k, kv[:, H * D:].view(T, H, E), sh.scale, w or None,
                      None if sink is None else sink.double().cpu(), tokens).reshape(T, H * E)


def lat_cache(sh, slots, max_seq, dt, dev, ring=0):
    """Paged (scattered blocks), or one ring of ``ring`` rows a slot; both hold another sequence's rows."""
    if ring:
        return lops.LatentCache(torch.full((slots, 1, ring, sh.row), 3.0, dtype=dt, device=dev), None, ring)
    kv = KVCache(1, 0, 0, dt, torch.device(dev), slots, max_seq, pool_tokens=slots * max_seq, shapes=[(1, sh.row, 0)])
    for s in [*range(1, slots, 2), *range(0, slots, 2)]:
        kv.reserve(s, max_seq)
    kv.k[0][..., :sh.rank + sh.rot_dim] = 3.0
    return lops.LatentCache(kv.k[0], kv.bt, max_seq)


def lat_run(q, xl, wkv, wn, sink, sh, rows, cache, dev, base=2e4, eps=1e-4):
    cos, sin = hops.pair_rope_tables(1400, sh.rot_dim, base, device=dev)
    if rows.decode and wkv.dtype == torch.bfloat16:  # the serving path; the parts are f32's
        return lops.latent_step(q.to(dev), xl.to(dev), wkv, lops.key_weight(wkv, sh), wn, eps, cos, sin, sink, sh, rows, cache)
    lat = lops.latent_rows(xl.to(dev), wn, eps, cos, sin, sh, rows, cache)
    return lops.latent_attention(q.to(dev), lat, wkv, cos, sin, sink, sh, rows, cache)


@on_devices
@pytest.mark.parametrize("case", LAT, ids=str)
def test_latent_attention_prompts_and_steps(dev, dt, case):
    """Unequal prompts in one pass, then decoded together; paged rows and rings that held another sequence."""
    sh, sink = lat_shape(case), case[6]
    wkv, wn, sk = lat_weights(sh, sink, dt, dev)
    lens, slots = [1, 130, 45, 3, 64], [2, 0, 4, 1, 3]
    more = 12
    if dev == "cuda":
        lens[1] = 600
    qs = [rnd(n + more, sh.q_width, seed=10 + i, dt=dt) for i, n in enumerate(lens)]
    xs = [rnd(n + more, sh.rank + sh.rot_dim, seed=30 + i, dt=dt) for i, n in enumerate(lens)]
    want = [lat_oracle(q, x, wkv, wn, sk, sh) for q, x in zip(qs, xs)]
    q0, x0 = (torch.cat([t[:n] for t, n in zip(ts, lens)]) for ts in (qs, xs))
    ref = torch.cat([w[:n] for w, n in zip(want, lens)])
    caches = [lat_cache(sh, 5, 768, dt, dev)] + ([lat_cache(sh, 5, 768, dt, dev, sh.window)] if sh.window else [])
    for cache in caches:
        rows = hops.PromptRows(lens, dev, slots, hops.SeqCaches([], [], None, [], []))
        close(lat_run(q0, x0, wkv, wn, sk, sh, rows, cache, dev), ref, dt)
        for t in range(more):
            rows = hops.TokenRows(i32([n + t for n in lens], dev), i32(slots, dev), 768, None)
            y = lat_run(torch.stack([q[n + t] for q, n in zip(qs, lens)]), torch.stack([x[n + t] for x, n in zip(xs, lens)]),
                        wkv, wn, sk, sh, rows, cache, dev)
            close(y, torch.stack([w[n + t] for w, n in zip(want, lens)]), dt, 1.5)


@on_devices
@pytest.mark.parametrize("batch", [1, 9, 70])
def test_latent_decode_batches(dev, dt, batch):
    """Every batch size against each sequence alone: lengths from one token to several splits."""
    sh = lops.LatentShape(6, 32, 16, 32, 64, 0.2)
    wkv, wn, sk = lat_weights(sh, True, dt, dev)
    lens = [1 + (97 * i) % 700 for i in range(batch)]
    cache = lat_cache(sh, batch, 768, dt, dev)
    q, xs = rnd(batch, sh.q_width, seed=1, dt=dt), [rnd(n, sh.rank + 16, seed=2 + n, dt=dt) for n in lens]
    cos, sin = hops.pair_rope_tables(800, 16, 2e4, device=dev)
    rows = hops.PromptRows(lens, dev, list(range(batch)), hops.SeqCaches([], [], None, [], []))
    lops.latent_rows(torch.cat(xs).to(dev), wn, 1e-4, cos, sin, sh, rows, cache)
    rows = hops.TokenRows(i32([n - 1 for n in lens], dev), i32(range(batch), dev), 768, None)
    y = lops.latent_attention(q.to(dev), None, wkv, cos, sin, sk, sh, rows, cache)
    if dt == torch.bfloat16:  # products per head on the matrix cores, or not
        close(lops.latent_step(q.to(dev), None, wkv, lops.key_weight(wkv, sh), None, 0.0, cos, sin, sk, sh, rows, cache), y, dt)
    for i in sorted({0, 1, batch // 2, batch - 1} & set(range(batch))):
        qi = torch.zeros(lens[i], sh.q_width).to(dt)
        qi[-1] = q[i]
        close(y[i], lat_oracle(qi, xs[i], wkv, wn, sk, sh)[-1], dt, 1.5)


@pytest.mark.gpu
@pytest.mark.parametrize("window", [0, 512, 600])
def test_long_splits_over_several_blocks(gpu, window):
    """So many heads and sequences that a split is hundreds of keys: tiles that straddle the edges of scattered
    blocks, splits that touch three of them, windows that start anywhere in one."""
    bf, B = torch.bfloat16, 64
    sh = lops.LatentShape(128, 16, 16, 16, 32, 0.25, window)
    wkv, wn, sk = lat_weights(sh, True, bf, gpu)
    lens = [640 + 7 * i for i in range(B)]
    cache = lat_cache(sh, B, 1280, bf, gpu)
    q, xs = rnd(B, sh.q_width, seed=1, dt=bf), [rnd(n, sh.rank + 16, seed=2 + n, dt=bf) for n in lens]
    cos, sin = hops.pair_rope_tables(1300, 16, 2e4, device=gpu)
    rows = hops.PromptRows(lens, gpu, list(range(B)), hops.SeqCaches([], [], None, [], []))
    lops.latent_rows(torch.cat(xs).to(gpu), wn, 1e-4, cos, sin, sh, rows, cache)
    rows = hops.TokenRows(i32([n - 1 for n in lens], gpu), i32(range(B), gpu), 1280, None)
    y = lops.latent_step(q.to(gpu), None, wkv, lops.key_weight(wkv, sh), None, 0.0, cos, sin, sk, sh, rows, cache)
    for i in (0, 17, 31, 45, 63):
        qi = torch.zeros(lens[i], sh.q_width).to(bf)
        qi[-1] = q[i]
        close(y[i], lat_oracle(qi, xs[i], wkv, wn, sk, sh, tokens=[lens[i] - 1])[-1], bf, 1.5)


@on_devices
@pytest.mark.parametrize("window", [1, 20, 64, 129, 300])
def test_window_edges_with_a_key_that_stands_out(dev, dt, window):
    """One key takes nearly all the weight: seen by the last position of its window and not by the next,
    in prompts and decoded; a window one token off moves the output far."""
    sh = lops.LatentShape(2, 16, 8, 16, 32, 1.0, window)
    T = 2 * window + 70
    wkv = torch.zeros(2 * 32, 32)
    for h in range(2):  # unrotated key = value = the latent's first 16
        wkv[16 * h:16 * h + 16, :16] = wkv[32 + 16 * h:48 + 16 * h, :16] = torch.eye(16)
    wkv, wn = wkv.to(dt).to(dev), torch.ones(32, device=dev)
    for key in sorted({0, 1, 63, 64, window - 1, window, 66}):
        if not 0 <= key < T - window - 2:
            continue
        q = torch.zeros(T, sh.q_width)
        q[:, 0] = q[:, 24] = 4.0
        xl = 0.05 * rnd(T, 40, seed=key)
        xl[:, 16:32] += 1.0
        xl[:, 0] = 0
        xl[key] = 0
        xl[key, 0] = xl[key, 1] = 5.0
        q, xl = q.to(dt), xl.to(dt)
        want = lat_oracle(q, xl, wkv, wn, None, sh)
        last = key + window - 1
        assert float(want[last, 1]) > 1.0 and (window == 1 or float(want[last + 1, 1].abs()) < 0.3)
        wrong = lat_oracle(q, xl, wkv, wn, None, sh, window + 1)
        assert (wrong - want).abs().max() > 0.5
        for n in sorted({key + 1, last, last + 1, T - 1}):
            if not 0 < n < T:
                continue
            for ring in (0, window, window + 5):
                cache = lat_cache(sh, 1, 768, dt, dev, ring)
                rows = hops.PromptRows([n], dev, [0], hops.SeqCaches([], [], None, [], []))
                close(lat_run(q[:n], xl[:n], wkv, wn, None, sh, rows, cache, dev), want[:n], dt)
                for p in range(n, min(T, n + 3)):
                    rows = hops.TokenRows(i32([p], dev), i32([0], dev), 768, None)
                    close(lat_run(q[p:p + 1], xl[p:p + 1], wkv, wn, None, sh, rows, cache, dev), want[p:p + 1], dt, 1.5)


@on_devices
@pytest.mark.parametrize("heads", [2, 18])
def test_softmax_sink(dev, dt, heads):
    """A sink far below the scores changes nothing, one far above takes all; it is not scaled."""
    sh = lops.LatentShape(heads, 16, 16, 16, 32, 0.3)
    wkv, wn, _ = lat_weights(sh, False, dt, dev)
    q, xl = rnd(9, sh.q_width, seed=1, dt=dt), rnd(9, 48, seed=2, dt=dt)
    for level in (-60.0, -2.0, 0.0, 3.0, 40.0):
        sk = torch.full((heads,), level)
        sk[0] = 1.5
        sk = sk.to(dev)
        want = lat_oracle(q, xl, wkv, wn, sk, sh)
        if level == 3.0:
            assert (want - lat_oracle(q, xl, wkv, wn, sk * 0.3, sh)).abs().max() > 0.05
        cache = lat_cache(sh, 1, 256, dt, dev)
        rows = hops.PromptRows([8], dev, [0], hops.SeqCaches([], [], None, [], []))
        close(lat_run(q[:8], xl[:8], wkv, wn, sk, sh, rows, cache, dev), want[:8], dt)
        rows = hops.TokenRows(i32([8], dev), i32([0], dev), 256, None)
        close(lat_run(q[8:], xl[8:], wkv, wn, sk, sh, rows, cache, dev), want[8:], dt, 1.5)


@on_devices
def test_a_far_key_in_the_paged_cache(dev, dt):
    """Positions at block edges of scattered blocks, each in turn the one that counts."""
    sh = lops.LatentShape(1, 16, 0, 16, 16, 1.0)
    wkv = torch.cat([torch.eye(16), torch.eye(16)]).to(dt).to(dev)
    wn, T = torch.ones(16, device=dev), 700
    for key in (0, 1, 255, 256, 257, 511, 512, 698):
        xl = 0.05 * rnd(T, 16, seed=key)
        xl[:, 8] += 1.0
        xl[key] = 0
        xl[key, 0] = xl[key, 1] = 5.0
        q = torch.zeros(T, 16)
        q[:, 0] = 5.0
        xl, q = xl.to(dt), q.to(dt)
        cache = lat_cache(sh, 3, 768, dt, dev)
        rows = hops.PromptRows([T - 1], dev, [1], hops.SeqCaches([], [], None, [], []))
        y = lat_run(q[:-1], xl[:-1], wkv, wn, None, sh, rows, cache, dev)
        rows = hops.TokenRows(i32([T - 1], dev), i32([1], dev), 768, None)
        y2 = lat_run(q[-1:], xl[-1:], wkv, wn, None, sh, rows, cache, dev)
        assert float(y[-1, 1]) > 1.5 and float(y2[0, 1]) > 1.5
        if dev == "cuda":
            want = lat_oracle(q, xl, wkv, wn, None, sh)
            close(y, want[:-1], dt)
            close(y2, want[-1:], dt, 1.5)


# ------------------------------------------------------------------ whole models
R, A, M = orc.ret_layer, orc.lat_layer, orc.moe
CONFIGS = {
    "mixed": orc.config(48, 301, 12, [
        A(4, 16, 8, 12, 24, 1e4, 0.3, sink=True, mlp=M(6, 2, 40, 2.0, 24)),
        R(3, 16, 20, 8, 3e4, (0.9, 0.99, 1.0), M(4, 3, 24, 1.5)),
        A(2, 20, 6, 16, 40, 5e3, 0.25, window=18, mlp=M(3, 1, 32, 3.0, 40, 1.2)),
        A(4, 12, 6, 24, 40, 5e3, 0.35, window=11, kv_from=2),
        R(2, 12, 8, 12, 1e4, (0.97, 0.6))], eps=1e-4),
    # a shared latent with a wider window than its owner's, and one whose reader is causal
    "shared": orc.config(40, 97, 8, [
        A(2, 16, 8, 16, 32, 1e4, 0.3, window=9), A(3, 8, 8, 16, 32, 1e4, 0.4, window=21, kv_from=0, mlp=M(4, 2, 16, 2.0)),
        A(2, 16, 4, 12, 20, 2e4, 0.3, window=7), A(4, 24, 4, 8, 20, 2e4, 0.2, sink=True, kv_from=2),
        A(1, 10, 4, 10, 20, 2e4, 0.4, window=1, kv_from=2)]),
    "retention_only": orc.config(36, 64, 6, [R(2, 16, 16, 16, 1e4, (0.99, 0.9)), R(1, 36, 12, 10, 1e4, (0.999,), M(2, 2, 20, 2.0, 12))]),
    "windows_only": orc.config(32, 80, 4, [A(2, 16, 16, 16, 32, 1e4, 0.25, window=5), A(2, 16, 8, 16, 16, 1e4, 0.25, window=40, mlp=M(1, 1, 24, 2.0))]),
    # sizes the matrix-core kernels take
    "wide": orc.config(256, 128, 16, [
        A(4, 64, 32, 64, 128, 1e4, 0.12, sink=True, mlp=M(8, 2, 64, 3.0, 128)),
        R(2, 64, 64, 64, 1e4, (0.98, 0.999), M(4, 2, 128, 2.0)),
        A(4, 32, 32, 48, 96, 1e4, 0.15, window=70, mlp=M(8, 4, 64, 2.0, 64)),
        A(2, 64, 32, 32, 96, 1e4, 0.13, window=33, kv_from=2, mlp=M(4, 1, 192, 2.0, 64))]),
    # a second embedding wide enough for its projection's decode kernel
    "side": orc.config(256, 128, 32, [A(4, 64, 32, 64, 128, 1e4, 0.12, sink=True, mlp=M(8, 2, 64, 3.0, 128)),
                                      R(2, 64, 64, 64, 1e4, (0.98, 0.999), M(4, 2, 128, 2.0))]),
}


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    cache = {}

    def get(name, dev, dt):
        if name not in cache:
            cfg = CONFIGS[name]
            w = orc.random_weights(cfg, seed=sum(map(ord, name)))
            cache[name] = (cfg, w, orc.save(cfg, w, tmp_path_factory.mktemp(name)))
        cfg, w, path = cache[name]
        return cfg, w, build_model(path, device=dev, dtype=dt)

    return get


def tokens(n, vocab, seed):
    return torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


def logits_close(got, want, dt, safe=None):
    """Mean-free RMS difference of every row against the spread of the logits.  ``safe`` (16-bit runs):
    rows whose routing no rounding can have changed; a head whose output is nearly zero before its norm
    still makes a row stand out."""
    d = got.double().cpu() - want.double()
    d = (d - d.mean(-1, keepdim=True)).pow(2).mean(-1).sqrt() / want.double().std(-1).mean()
    if dt == torch.float32:
        assert float(d.max()) < 2e-4, float(d.max())
        return
    assert float(d.median()) < 5e-2, float(d.median())
    if safe is not None and safe.any():
        assert float(d[safe].quantile(0.85)) < 8e-2 and float(d[safe].max()) < 0.5, (d[safe].quantile(0.85), d[safe].max())


def settled(cfg, w, seq):
    """Rows none of whose own or earlier tokens had a close call in a router."""
    return (orc.route_margin(cfg, w, seq, torch.float32) > 0.15).cummin(0).values


@on_devices
@pytest.mark.parametrize("name", list(CONFIGS))
def test_model_prompts_then_decoding(built, name, dev, dt):
    """Logits of every position: whole prompts of unequal length in one pass, then decoded together past
    several window edges, against the oracle and against each request alone in slots used before."""
    cfg, w, model = built(name, dev, dt)
    V, lens, more = cfg["vocab"], [5, 1, 30, 12], 24
    if name == "wide" and dev == "cuda":
        lens, more = [300, 3, 130, 1], 40
    seqs = [tokens(n + more, V, 50 + i) for i, n in enumerate(lens)]
    want = [orc.forward(cfg, w, s, torch.float32) for s in seqs]
    ok = [settled(cfg, w, s) for s in seqs] if dt == torch.bfloat16 else [torch.ones(len(s), dtype=torch.bool) for s in seqs]
    eng = Engine(model, max_batch=6, max_seq=512, kv_pool_tokens=6 * 512)
    slots = [eng.acquire() for _ in lens]
    for s, n in zip(slots, lens):
        eng.extend(s, n + 1)
    got = eng.prefill_batch(slots, [s[:n] for s, n in zip(seqs, lens)], [list(range(n)) for n in lens])
    logits_close(got, torch.cat([x[:n] for x, n in zip(want, lens)]), dt, torch.cat([x[:n] for x, n in zip(ok, lens)]))
    dec = []
    for t in range(more):
        for s, n in zip(slots, lens):
            eng.extend(s, n + t + 1)
        dec.append(eng.decode(slots, torch.tensor([s[n + t] for s, n in zip(seqs, lens)])).float().clone())
    logits_close(torch.cat(dec), torch.cat([torch.stack([x[n + t] for x, n in zip(want, lens)]) for t in range(more)]), dt,
                 torch.cat([torch.stack([x[n + t] for x, n in zip(ok, lens)]) for t in range(more)]))
    for s in slots:
        eng.release(s)
    for s, o in zip(seqs[:2], ok):  # alone, one token at a time from the first
        slot = eng.acquire()
        eng.extend(slot, 40)
        ref = orc.forward(cfg, w, s[:20], torch.float32)
        out = [eng.prefill_batch([slot], [s[:1]])[0]]
        out += [eng.decode([slot], torch.tensor([t]))[0].float().clone() for t in s[1:20]]
        logits_close(torch.stack(out), ref, dt, o[:20])
        eng.release(slot)


@on_devices
@pytest.mark.parametrize("name", ["mixed", "wide"])
def test_residual_stream_layer_by_layer(built, name, dev, dt):
    cfg, w, model = built(name, dev, dt)
    ids = tokens(31, cfg["vocab"], 3)
    want, got = [], []
    orc.forward(cfg, w, ids, torch.float64, want)
    ok = settled(cfg, w, ids) if dt == torch.bfloat16 else torch.ones(31, dtype=torch.bool)
    model.hidden_states(torch.tensor([ids], device=dev), tap=lambda i, h: got.append(h.clone()))
    assert len(got) == len(want) == len(cfg["layers"])
    for a, b in zip(got, want):
        assert a.dtype == torch.float32
        if ok.any():
            close(a.cpu()[ok], b[ok], dt, 4)


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("name", ["mixed", "shared", "retention_only", "windows_only"])
def test_greedy_generation_through_the_scheduler(built, name, dev):
    """More requests than slots, unequal prompts and lengths, a pool that makes some wait; f32."""
    cfg, w, model = built(name, dev, torch.float32)
    prompts = [tokens(n, cfg["vocab"], n) for n in (1, 2, 9, 26, 14, 5)]
    want = [orc.greedy(cfg, w, p, 8, torch.float32) for p in prompts]
    for kw in ({}, {"kv_pool_tokens": 512}, {"prefill_tokens": 12}):
        eng = Engine(model, max_batch=3, max_seq=256, eos_ids=(model.cfg.eos_id,), **kw)
        assert eng.generate(prompts, max_new_tokens=8) == want
        assert eng.generate(prompts[::-1], max_new_tokens=8) == want[::-1]


def test_what_the_caches_hold(built):
    """Causal latents are paged; windowed ones are rings of the widest window that reads them; states are f32."""
    cfg, w, model = built("shared", "cpu", torch.float32)
    assert [model.cfg.look_back(i) for i in (0, 2)] == [21, 0]
    eng = Engine(model, max_batch=2, max_seq=100, kv_pool_tokens=512)
    assert len(eng.kv.k) == 1 and [t.shape[2] for t in eng.model_steps.state.ring] == [21]
    _, _, model = built("windows_only", "cpu", torch.float32)
    eng = Engine(model, max_batch=2, max_seq=100000, kv_pool_tokens=512)
    assert eng.kv.span == 1 and eng.kv.look == 40 and eng.kv.blocks_for(90000) == 1
    _, _, model = built("retention_only", "cpu", torch.bfloat16)
    assert all(t.dtype == torch.float32 for t in Engine(model, max_batch=2, max_seq=64).model_steps.state.rec)


@pytest.mark.parametrize("name", ["windows_only", "retention_only"])
def test_long_decoding_keeps_a_bounded_cache(built, name):
    cfg, w, model = built(name, "cpu", torch.float32)
    eng = Engine(model, max_batch=2, max_seq=100000, kv_pool_tokens=512)
    seq = tokens(200, cfg["vocab"], 8)
    slot = eng.acquire()
    eng.extend(slot, 100000)
    lg = eng.prefill_batch([slot], [seq[:1]])
    for t in seq[1:]:
        lg = eng.decode([slot], torch.tensor([t]))
    logits_close(lg, orc.forward(cfg, w, seq, torch.float32)[-1:], torch.float32)
    assert len(eng.kv.owned[slot]) == 1


def test_engine_embeddings_and_refusals(built):
    cfg, w, model = built("mixed", "cpu", torch.float32)
    eng = Engine(model, max_batch=2, max_seq=64)
    e = eng.embed([tokens(9, cfg["vocab"], 1), tokens(3, cfg["vocab"], 2)])
    assert e.shape == (2, 48) and torch.allclose(e.norm(dim=1), torch.ones(2), atol=1e-5)
    for bad in ([], [5, 301], [-1]):
        with pytest.raises(ValueError):
            eng.prefill_batch([0], [bad])
    with pytest.raises(NotImplementedError):
        Sigusun(model.cfg, lora_r=4)


# ------------------------------------------------------------------ configuration, weights, command line
@pytest.mark.parametrize("name", list(CONFIGS))
def test_config_round_trip(name):
    cfg = CONFIGS[name]
    c = SigusunConfig.from_json(cfg)
    assert c.to_json() == cfg and SigusunConfig.from_json(c.to_json()) == c
    assert c.n_params() == sum(int(np.prod(s)) for s in orc.tensor_shapes(cfg).values())


def test_config_errors(tmp_path):
    cfg = CONFIGS["mixed"]
    lat = cfg["layers"][3]["mixer"]
    for i, change in ((1, {"type": "other"}), (1, {"mlp": {"kind": "dense", "ff": 8}}),
                      (1, {"mixer": dict(cfg["layers"][1]["mixer"], decay=[0.5])}),
                      (1, {"mixer": dict(cfg["layers"][1]["mixer"], rot={"base": 1e4, "dims": 7})}),
                      (1, {"mlp": orc.moe(2, 3, 8, 1.0)}), (3, {"mixer": dict(lat, kv_from=1)}),
                      (3, {"mixer": dict(lat, kv_from=4)}), (3, {"mixer": dict(lat, kv_rank=12)}),
                      (3, {"mixer": dict(lat, rot={"base": 1e4, "dims": 6})})):
        bad = json.loads(json.dumps(cfg))
        bad["layers"][i].update(change)
        with pytest.raises(ValueError):
            SigusunConfig.from_json(bad)


def test_weights_round_trip_and_strictness(tmp_path):
    cfg = CONFIGS["mixed"]
    w = orc.random_weights(cfg, 5)
    m = build_model(orc.save(cfg, w, tmp_path / "a"), dtype=torch.float32)
    assert sum(p.numel() for p in m.parameters()) == m.cfg.n_params()
    save_sigusun(m, str(tmp_path / "b"))
    m2 = build_model(str(tmp_path / "b"), dtype=torch.float32)
    for (n, p), (_, q) in zip(m.named_parameters(), m2.named_parameters()):
        assert torch.equal(p, q), n
    for name, change in (("missing", lambda d: d.pop("l1.mlp.e2.up")),
                         ("extra", lambda d: d.update({"l3.mix.dkv": torch.ones(3)})),
                         ("shape", lambda d: d.update({"l1.mix.q": torch.zeros(64, 40)}))):
        d = dict(w)
        change(d)
        with pytest.raises((KeyError, ValueError)):
            build_model(orc.save(cfg, d, tmp_path / name))


def test_presets_build_and_serve():
    m = build_model("sigusun-tiny", dtype=torch.float32, seed=3)
    assert isinstance(m, Sigusun) and m.num_params() == m.cfg.n_params()
    out = Engine(m, max_batch=2, max_seq=128).generate([[1, 2, 3], [9]], max_new_tokens=5)
    assert [len(o) for o in out] == [5, 5]


def test_server_serves_a_model_directory(tmp_path):
    """The HTTP server's engine builder takes a Sigusun directory like any other model."""
    from mxllm.serve.server import build_default

    cfg = orc.config(24, 300, 4, [R(2, 8, 8, 8, 1e4, (0.9, 0.99), M(2, 1, 8, 2.0)), A(2, 8, 4, 8, 16, 1e4, 0.3, sink=True)])
    path = orc.save(cfg, orc.random_weights(cfg, 1), tmp_path)
    assert isinstance(model_config(path), SigusunConfig)
    eng, tok = build_default(path, device="cpu", max_batch=2, max_seq=128)
    ids = tok.encode("hello")
    assert max(ids) < 300 and len(eng.generate([ids], max_new_tokens=4)[0]) == 4


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_trace_replay(built, dev, tmp_path):
    """JSON steps in, logits files out: batches whose shorter requests end earlier, ids used again, nothing
    wanted."""
    from mxllm.serve.trace import Replay, replay

    cfg, w, model = built("mixed", dev, torch.float32)
    seqs = {"a": tokens(40, 301, 1), "b": tokens(12, 301, 2)}
    want = {k: orc.forward(cfg, w, s, torch.float32) for k, s in seqs.items()}
    steps, expect = [], []

    def step(entries, end=()):
        steps.append(json.dumps({"step": len(steps), "entries": [{"id": i, "tokens": seqs[i][lo:hi], "want": wt}
                                                                 for i, lo, hi, wt in entries], "end": list(end)}))
        expect.append([want[i][lo + k] for i, lo, hi, wt in entries for k in wt])

    for _ in range(2):
        step([("a", 0, 20, [19, 0, 7]), ("b", 0, 9, [])])
        for p in range(20, 23):
            step([("b", p - 11, p - 10, [0]), ("a", p, p + 1, [0])], ["b"] if p == 22 else [])
        for p in range(23, 32):
            step([("a", p, p + 1, [0] if p % 3 else [])])
        step([("a", 32, 33, [0])], ["a"])
    eng = Engine(model, max_batch=3, max_seq=64, kv_pool_tokens=1024)
    said = []
    replay(eng, io.StringIO("\n".join(steps) + "\n"), str(tmp_path), said.append)
    assert said == [f"done {i}" for i in range(len(steps))]
    for i, rows in enumerate(expect):
        f = tmp_path / f"{i}.f32"
        assert f.exists() == bool(rows)
        if rows:
            logits_close(torch.from_numpy(np.fromfile(f, dtype="<f4").reshape(len(rows), 301)), torch.stack(rows),
                         torch.float32)
    assert sorted(eng.free_slots) == [0, 1, 2] and not Replay(eng).slot


# ------------------------------------------------------------------ GPU only
@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 3, 8])
def test_graphed_decode_equals_eager(built, gpu, batch):
    """Graph replays against eager steps on the same slots, with other work between the replays."""
    cfg, w, model = built("wide", gpu, torch.bfloat16)
    prompts = [tokens(3 + 40 * i, 128, i) for i in range(batch)]
    feed = torch.randint(0, 128, (12, batch), generator=torch.Generator().manual_seed(1))
    outs = []
    for graphs in (True, False):
        eng = Engine(model, max_batch=8, max_seq=512, use_graphs=graphs, kv_pool_tokens=8192)
        slots = [eng.acquire() for _ in prompts]
        for s, p in zip(slots, prompts):
            eng.extend(s, len(p) + 20)
        eng.prefill_batch(slots, prompts)
        got = []
        for t in feed:
            got.append(eng.decode(slots, t).float().clone())
            eng.embed([prompts[0]])
            torch.cuda.synchronize()
        outs.append(torch.stack(got))
    rel = (outs[0] - outs[1]).pow(2).mean(-1).sqrt() / outs[1].pow(2).mean().sqrt()
    assert float(rel.median()) < 1.5e-2, float(rel.median())


@pytest.mark.gpu
@pytest.mark.parametrize("graphs", [False, True])
def test_decode_follows_a_side_projection_written_in_place(built, gpu, graphs):
    """New values of ``side_proj`` in the storage that decode steps read: the next steps are those of a model that had them from
    the start (the same kernels on the same values: the same bits)."""
    prompts, feed = [tokens(9, 128, 1), tokens(40, 128, 2)], [[5, 6], [7, 8], [9, 1], [2, 3]]

    def write(model):
        for i, layer in enumerate(model.layers):
            layer.side_proj.weight.mul_(3.0).add_(rnd(*layer.side_proj.weight.shape, seed=i, dt=torch.bfloat16).to(gpu), alpha=0.1)

    def steps(model, late):
        if not late:
            write(model)
        eng = Engine(model, max_batch=2, max_seq=128, use_graphs=graphs, kv_pool_tokens=512)
        slots = [eng.acquire() for _ in prompts]
        for s, p in zip(slots, prompts):
            eng.extend(s, len(p) + 8)
        eng.prefill_batch(slots, prompts)
        if late:  # steps with the old values (and a graph of them), then the prompt again
            for t in feed:
                eng.decode(slots, torch.tensor(t))
            write(model)
            eng.prefill_batch(slots, prompts)
        return torch.stack([eng.decode(slots, torch.tensor(t)).float().clone() for t in feed])

    want, got = (steps(built("side", gpu, torch.bfloat16)[2], late) for late in (False, True))
    rel = float((got - want).pow(2).mean().sqrt() / want.pow(2).mean().sqrt())
    assert rel < 1e-6, rel


@pytest.mark.gpu
@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("way", ["load_state_dict", "reset_parameters", "second engine"])
def test_decode_follows_new_weights(built, gpu, graphs, way):
    """All weights new in their storage, after steps (and a graph of them) with the old: decode's transposed key weights are the
    new ones', and the steps have the bits of a model that had these weights from the start."""
    prompts, feed = [tokens(9, 128, 1), tokens(40, 128, 2)], [[5, 6], [7, 8], [9, 1]]
    model, other = (built("wide", gpu, torch.bfloat16)[2] for _ in range(2))
    other.reset_parameters(5)

    def engine(m):
        eng = Engine(m, max_batch=2, max_seq=128, use_graphs=graphs, kv_pool_tokens=512)
        slots = [eng.acquire() for _ in prompts]
        for s, p in zip(slots, prompts):
            eng.extend(s, len(p) + 8)
        return eng, slots

    def steps(eng, slots):
        eng.prefill_batch(slots, prompts)
        return torch.stack([eng.decode(slots, torch.tensor(t)).float().clone() for t in feed])

    want = steps(*engine(other))
    run = engine(model)
    before = steps(*run)
    if way == "load_state_dict":
        model.load_state_dict(other.state_dict())
    elif way == "reset_parameters":
        model.reset_parameters(5)
    else:
        for p, q in zip(model.parameters(), other.parameters()):
            p.copy_(q)
        engine(model)
    got = steps(*run)
    assert not torch.equal(before, want) and torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16], ids=str)
def test_large_decode_batches(built, gpu, dt):
    """More sequences than the decode kernels of the experts take at once, against the oracle."""
    cfg, w, model = built("wide", gpu, dt)
    n, lens = 70, [1 + (37 * i) % 90 for i in range(70)]
    seqs = [tokens(k + 3, 128, 200 + i) for i, k in enumerate(lens)]
    eng = Engine(model, max_batch=n, max_seq=256)
    slots = [eng.acquire() for _ in lens]
    eng.prefill_batch(slots, [s[:k] for s, k in zip(seqs, lens)])
    out = [eng.decode(slots, torch.tensor([s[k + t] for s, k in zip(seqs, lens)])).float().clone() for t in range(3)]
    check = [0, 1, 17, 68, 69]
    ref = torch.stack([orc.forward(cfg, w, seqs[i], torch.float32)[lens[i]:] for i in check], 1)
    logits_close(torch.stack(out)[:, check].flatten(0, 1), ref.flatten(0, 1), dt)


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 5])
def test_fused_decode_equals_its_parts(built, gpu, batch, monkeypatch):
    cfg, w, model = built("wide", gpu, torch.bfloat16)
    prompts = [tokens(3 + 30 * i, 128, i) for i in range(batch)]
    feed = torch.randint(0, 128, (10, batch), generator=torch.Generator().manual_seed(1))
    outs = []
    for fused in (True, False):
        monkeypatch.setattr(sops, "FUSED", fused)
        eng = Engine(model, max_batch=8, max_seq=512, kv_pool_tokens=8192)
        slots = [eng.acquire() for _ in prompts]
        for s, p in zip(slots, prompts):
            eng.extend(s, len(p) + 20)
        eng.prefill_batch(slots, prompts)
        outs.append(torch.stack([eng.decode(slots, t).float().clone() for t in feed]))
    rel = (outs[0] - outs[1]).pow(2).mean(-1).sqrt() / outs[1].pow(2).mean().sqrt()
    assert float(rel.median()) < 3e-2, float(rel.median())


@pytest.mark.gpu
def test_fp8_weights_serve(built, gpu):
    """Quantised projections and shared expert; the experts themselves stay bf16."""
    from mxllm.serve.quant import quantize_model_fp8_

    _, _, model = built("wide", gpu, torch.bfloat16)
    seq = tokens(40, 128, 4)
    ref = Engine(model, max_batch=2, max_seq=128).prefill_batch([0], [seq], [[39]])
    assert quantize_model_fp8_(model) > 0
    eng = Engine(model, max_batch=2, max_seq=128)
    eng.prefill_batch([0], [seq[:39]])
    got = eng.decode([0], torch.tensor([seq[39]])).float()
    assert torch.isfinite(got).all()
    rel = (got - ref).pow(2).mean().sqrt() / ref.pow(2).mean().sqrt()
    assert float(rel) < 0.5, float(rel)


@pytest.mark.gpu
def test_bf16_generation_matches_its_own_prompt_pass(built, gpu):
    """Greedy bf16 generation through the scheduler: nearly every chosen token is the argmax of the prompt
    pass over the same tokens, up to near-ties (a close call of a router may differ between the two)."""
    cfg, _, model = built("wide", gpu, torch.bfloat16)
    prompts = [tokens(n, 128, n) for n in (3, 140, 11, 1, 75)]
    outs = Engine(model, max_batch=4, max_seq=512).generate(prompts, max_new_tokens=40)
    off = 0
    for p, o in zip(prompts, outs):
        lg = model(torch.tensor([p + o[:-1]], device=gpu))[0, len(p) - 1:].float()
        top = lg.max(-1).values
        got = lg.gather(1, torch.tensor(o, device=gpu)[:, None])[:, 0]
        off += int(((top - got) > 0.1 * lg.std()).sum())
    assert off <= 10, off
