"""The gradient of a tied embedding and head, which a trainer's backward writes in place for both uses, against the sum that
autograd makes where the parameter has a hook of the caller's own."""
import pytest
import torch

from mxllm.models import get_config
from mxllm.models.llama import Llama
from mxllm.parallel.grad_ready import callers_hook
from mxllm.parallel.runtime import DistEnv
from mxllm.train.trainer import OptimConfig, Trainer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("accum", [1, 2])
@pytest.mark.parametrize("grad_dtype", [None, "fp32"])
def test_tied_gradient(gpu, accum, grad_dtype):
    cfg = get_config("llama3.2-1b").replace(n_layers=1, hidden=256, n_heads=4, n_kv_heads=2, ffn=512, vocab_size=1024)
    g = torch.Generator().manual_seed(5)
    steps = [[(torch.randint(0, 900, (2, 64), generator=g).to(gpu), torch.randint(0, 1024, (2, 64), generator=g).to(gpu))
              for _ in range(accum)] for _ in range(2)]
    grads, sums = [], []
    for hook in (False, True):
        model = Llama(cfg, device=gpu, dtype=torch.bfloat16, seed=3)
        tr = Trainer(model, DistEnv(device=gpu), OptimConfig(lr=0.0), grad_dtype=grad_dtype)
        if hook:
            model.tok_emb.register_hook(lambda t: sums.append(t.shape))
        out = []
        for s in steps:  # the second step finds the first one's gradients in the buffer
            tr.compute_grads(s)
            slot = next(x for x in tr.flat.slots if x.name == "tok_emb")
            out.append(tr.flat.grads[slot.offset:slot.offset + slot.numel].float().clone())
        assert model.tok_emb._mx_no_direct and not model.tok_emb._mx_two_uses if not hook else True
        grads.append(out)
    assert len(sums) == 2 * accum
    for a, b in zip(*grads):
        assert float(b.norm()) > 0
        # roundings to bf16 of either way: 2 a micro-batch and one of their sums, 2^-9 each
        assert float((a - b).norm()) <= (2 * accum + 1) * 2.0 ** -9 * float(b.norm())


def test_hook_ahead_of_the_trainer(gpu):
    """A mask that the caller put on the parameter before the trainer was there: it sees the sum, and what it returns is kept."""
    cfg = get_config("llama3.2-1b").replace(n_layers=1, hidden=256, n_heads=4, n_kv_heads=2, ffn=512, vocab_size=1024)
    g = torch.Generator().manual_seed(6)
    mb = (torch.randint(0, 900, (2, 64), generator=g).to(gpu), torch.randint(0, 1024, (2, 64), generator=g).to(gpu))
    mask = (torch.arange(1024, device=gpu) % 3 == 0).bfloat16()[:, None]
    grads, seen = [], []
    for hook in (False, True):
        model = Llama(cfg, device=gpu, dtype=torch.bfloat16, seed=3)
        if hook:
            model.tok_emb.register_hook(lambda t: (seen.append(t.clone()), t * mask)[1])
        tr = Trainer(model, DistEnv(device=gpu), OptimConfig(lr=0.0))
        assert callers_hook(model.tok_emb) == hook
        tr.compute_grads([mb])
        slot = next(x for x in tr.flat.slots if x.name == "tok_emb")
        grads.append(tr.flat.grads[slot.offset:slot.offset + slot.numel].view(slot.shape).clone())
    both, masked = grads
    assert len(seen) == 1 and torch.equal(masked, seen[0] * mask)
    # (bounds as above, one micro-batch)
    assert float((both.float() - seen[0].float()).norm()) <= 3 * 2.0 ** -9 * float(both.float().norm())
