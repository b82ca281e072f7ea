"""Whose hooks keep a parameter that is used twice with autograd (mxllm/parallel/grad_ready.py), on the CPU."""
import pytest
import torch

from mxllm.ops.linear import _LinearFn
from mxllm.parallel.grad_ready import callers_hook, own_hook, two_uses


def _both_uses(w):
    x = torch.arange(6.0).reshape(2, 3)
    (_LinearFn.apply(x, w).sum() + _LinearFn.apply(2 * x, w).square().sum()).backward()


def _want():
    w = torch.nn.Parameter(torch.ones(4, 3))
    _both_uses(w)
    return w.grad


@pytest.mark.parametrize("when", ["none", "before", "after", "exchanged"])
@pytest.mark.parametrize("post", [False, True])
def test_hooks_get_the_sum(when, post):
    seen = []

    def callers(w):
        if post:
            return w.register_post_accumulate_grad_hook(lambda p: (seen.append(p.grad.clone()), p.grad.mul_(3)) and None)
        return w.register_hook(lambda g: (seen.append(g.clone()), 3 * g)[1])

    w = torch.nn.Parameter(torch.ones(4, 3))
    w._mx_no_direct = True
    w.grad = torch.zeros(4, 3)
    early = callers(w) if when in ("before", "exchanged") else None
    mine = [own_hook(w, w.register_hook(lambda g: g)), own_hook(w, w.register_post_accumulate_grad_hook(lambda p: None))]
    if when == "exchanged":  # as many hooks as there were, another one
        early.remove()
    if when in ("after", "exchanged"):
        callers(w)
    with two_uses([w]):
        in_place = w._mx_two_uses if when == "none" else getattr(w, "_mx_two_uses", False)
        _both_uses(w)
    assert w._mx_no_direct and not getattr(w, "_mx_two_uses", False) and len(mine) == 2
    assert in_place == (when == "none")
    want = _want()
    assert torch.equal(w.grad, want if when == "none" else 3 * want)
    assert len(seen) == (when != "none") and all(torch.equal(s, want) for s in seen)


@pytest.mark.parametrize("grad_dtype", [None, "fp32"])
def test_owners_note_their_hooks(grad_dtype, monkeypatch):
    monkeypatch.setenv("MXLLM_FORCE_CPU", "1")
    from mxllm.models import Llama, get_config
    from mxllm.parallel.runtime import DistEnv
    from mxllm.train.trainer import OptimConfig, Trainer

    model = Llama(get_config("tiny").replace(n_layers=1, vocab_size=300), device="cpu", dtype=torch.bfloat16)
    tr = Trainer(model, DistEnv(device=torch.device("cpu")), OptimConfig(), grad_dtype=grad_dtype)
    tr.ddp.set_on_ready(lambda b: None)
    params = tr.flat.param_list
    assert all(p._post_accumulate_grad_hooks for p in params) and not any(callers_hook(p) for p in params)
    params[0].register_hook(lambda g: g)
    assert [callers_hook(p) for p in params] == [True] + [False] * (len(params) - 1)
