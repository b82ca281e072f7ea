"""Latent attention of prompts on the matrix cores: where tiles, windows and rounds of workgroups end."""
import pytest
import torch

from mxllm.ops import hybrid as hops
from mxllm.ops import latent as lops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,dim,rot,vdim,window,lens", [
    (32, 64, 32, 64, 0, [64, 65, 63, 128, 1]),        # whole tiles, one row more, one fewer
    (3, 128, 64, 128, 0, [513, 640]),                 # heads that do not divide a round of the CUs
    (32, 32, 16, 32, 100, [1100]),                    # a second round, shortest first; a window's edges in every block
    (40, 16, 16, 32, 0, [1700]),                      # more workgroups than places
    (300, 16, 16, 8, 0, [130]),                       # more heads than a round
    (2, 200, 40, 96, 64, [257, 300]), (5, 48, 0, 48, 0, [191, 2, 320])])
def test_latent_flash(heads, dim, rot, vdim, window, lens):
    torch.manual_seed(sum(lens))
    sh = lops.LatentShape(heads, dim, rot, vdim, 64, 1.6 / (dim + rot) ** 0.5, window)
    rows = hops.PromptRows(lens, torch.device("cuda"))
    T, D, R, E = rows.T, dim, rot, vdim
    q = torch.randn(T, sh.q_width + 8, device="cuda").bfloat16()[:, :sh.q_width]
    lat = torch.randn(T, sh.row, device="cuda").bfloat16()
    wkv = (torch.randn(heads * (D + E), 64, device="cuda") / 8).bfloat16()
    sink = torch.randn(heads, device="cuda")
    cos, sin = hops.pair_rope_tables(max(lens), R, 1e4, device="cuda")
    y = lops.latent_attention(q, lat, wkv, cos, sin, sink, sh, rows, None)
    # the same in f32, one sequence at a time
    kv = torch.nn.functional.linear(lat[:, :64], wkv).float()
    qf, o = q.float().view(T, heads, D + R).clone(), 0
    if R:
        pos = torch.cat([torch.arange(n) for n in lens]).cuda()
        c, s = cos[pos][:, None], sin[pos][:, None]
        a, b = qf[..., D::2].clone(), qf[..., D + 1::2].clone()
        qf[..., D::2], qf[..., D + 1::2] = a * c - b * s, b * c + a * s
        qf[..., D:] = qf[..., D:].bfloat16().float()
    for n in lens:
        k = torch.cat([kv[o:o + n, :heads * D].view(n, heads, D), lat[o:o + n, None, 64:64 + R].float().expand(n, heads, R)], -1)
        v = kv[o:o + n, heads * D:].view(n, heads, E).transpose(0, 1).contiguous()
        z = torch.matmul(qf[o:o + n].transpose(0, 1), k.permute(1, 2, 0).contiguous()) * sh.scale
        i = torch.arange(n, device="cuda")
        ok = (i[None] <= i[:, None]) & ((i[None] > i[:, None] - window) if window else True)
        z = torch.cat([z.masked_fill(~ok, float("-inf")), sink[:, None, None].expand(heads, n, 1)], -1)
        p = torch.softmax(z, -1)[..., :n]
        ref = torch.matmul(p, v)
        # weights and outputs are rounded to bf16: 2^-9 of sum |p v| and of the result, a weight's sum and its scale in f32
        bound = 2.0**-8 * (torch.matmul(p, v.abs()) + ref.abs()) + 1e-5
        got = y[o:o + n].float().view(n, heads, E).transpose(0, 1)
        assert bool(((got - ref).abs() <= bound).all())
        o += n
