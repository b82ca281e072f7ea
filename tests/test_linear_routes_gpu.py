"""What the inference kernels behind ``ops.linear`` and its fused forms must not take: they have neither derivatives nor
batching rules, and read whole 16-byte pieces of dense rows."""
import sys

import pytest
import torch

from mxllm import ops

pytestmark = pytest.mark.gpu


def _bf16(gpu, *shape, seed=0, std=1.0):
    g = torch.Generator(device=gpu).manual_seed(seed)
    return torch.empty(*shape, device=gpu).normal_(0, std, generator=g).bfloat16()


def _close(got, want, tol):
    err = float((got.double() - want.double()).norm() / want.double().norm())
    assert err < tol, err


# rows on each side of the decode GEMMs' limits (8, 16, 32) and of a prompt pass; 12,288: K in parts from 64 rows on
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 64])
@pytest.mark.parametrize("N,K", [(2048, 2048), (8192, 4096), (512, 12288)])
def test_frozen_weight_passes_gradients(gpu, M, N, K):
    """A frozen weight: the input's gradient is dy W, backward and forward mode (one bf16 rounding: 2^-8)."""
    x, w, dy = _bf16(gpu, M, K, seed=1).requires_grad_(), _bf16(gpu, N, K, seed=2, std=0.03), _bf16(gpu, M, N, seed=3)
    y = ops.linear(x, w)
    y.backward(dy)
    _close(x.grad, dy.double() @ w.double(), 2 ** -8)
    t = _bf16(gpu, M, K, seed=4)
    _, tan = torch.func.jvp(lambda a: ops.linear(a, w), (x.detach(),), (t,))
    _close(tan, t.double() @ w.double().t(), 2 ** -8)
    with torch.autograd.forward_ad.dual_level():  # a tangent of the weight alone
        dual = torch.autograd.forward_ad.make_dual(w, torch.ones_like(w))
        tan = torch.autograd.forward_ad.unpack_dual(ops.linear(x.detach(), dual)).tangent
    _close(tan, x.detach().double().sum(1, keepdim=True).expand(M, N), 2 ** -6)


@pytest.mark.parametrize("M", [1, 4, 16])
def test_fused_forms_decline_gradients(gpu, M):
    """The fused decode forms leave calls whose inputs ask for gradients to the caller's differentiable parts."""
    K, F, H, D = 4096, 4096, 4, 128
    x, w, gamma = _bf16(gpu, M, K), _bf16(gpu, 2 * F, K, seed=1, std=0.03), torch.ones(K, device=gpu).bfloat16()
    wq = _bf16(gpu, 3 * H * D, K, seed=2, std=0.03)
    cos = torch.ones(64, D // 2, device=gpu)
    pos = torch.zeros(M, dtype=torch.int32, device=gpu)
    kc, vc = torch.zeros(2, M, H, 64, D, device=gpu, dtype=torch.bfloat16)

    def forms(x, delta, gamma):
        a = ops.linear_swiglu(x, w), ops.qkv_rope_linear(None, x, None, 1e-5, wq, cos, cos, pos, None, kc, vc, H, H)
        return a + ((ops.norm_linear(delta, x, gamma, 1e-5, w, True),
                     ops.qkv_rope_linear(delta, x, gamma, 1e-5, wq, cos, cos, pos, None, kc, vc, H, H)) if M <= 4 else ())

    assert all(r is not None for r in forms(x, x, gamma))
    assert all(r is None for r in forms(x.clone().requires_grad_(), x, gamma))
    if M <= 4:
        for delta, g in ((x.clone().requires_grad_(), gamma), (x, gamma.clone().requires_grad_())):
            assert all(r is None for r in forms(x, delta, g)[2:])


@pytest.mark.parametrize("M", [4, 16, 64])
def test_transforms_and_tracers_take_the_library(gpu, M):
    """vmap, torch.func.grad, compilation, tracing and shape propagation of an inference call, on each side of the
    decode GEMMs' rows; a traced call is right at rows that it was not traced with."""
    from torch._subclasses import FakeTensorMode

    K, N = (2048, 4096) if M < 64 else (12288, 512)
    w, xs = _bf16(gpu, N, K, seed=1, std=0.03), _bf16(gpu, 3, M, K, seed=2)
    want = xs.double() @ w.double().t()
    _close(torch.func.vmap(lambda a: ops.linear(a, w))(xs), want, 2 ** -8)
    _close(torch.func.vmap(lambda b: ops.linear(xs[0], b))(torch.stack([w, 2 * w]))[1], 2 * want[0], 2 ** -8)
    dx = torch.func.grad(lambda a: ops.linear(a, w).double().sum())(xs[0])
    _close(dx, w.double().sum(0).expand(M, K), 2 ** -8)
    _close(torch.compile(lambda a: ops.linear(a, w), backend="eager", fullgraph=True)(xs[0]), want[0], 2 ** -8)
    traced = torch.jit.trace(lambda a: ops.linear(a, w), xs[0], check_trace=False)
    _close(traced(xs.reshape(-1, K)), want.reshape(-1, N), 2 ** -8)
    mode = FakeTensorMode()
    fakes = mode.from_tensor(xs[0]), mode.from_tensor(w)
    with mode:
        y = ops.linear(*fakes)
        assert y.shape == (M, N) and y.device == w.device


def _odd_rows(gpu, kind, M, K):
    """Rows whose layout the decode GEMMs do not read: overlapping, shorter apart than long, off 16-byte addresses."""
    if kind == "expanded":
        return _bf16(gpu, 1, K, seed=5).expand(M, K)
    if kind == "overlapping":
        return _bf16(gpu, M * 64 + K, seed=5).as_strided((M, K), (64, 1))
    buf = _bf16(gpu, M * (K + 8) + 8, seed=5)
    return buf[4:4 + M * (K + 8)].view(M, K + 8)[:, :K]


@pytest.mark.parametrize("M", [2, 8, 16, 32, 64])
@pytest.mark.parametrize("kind", ["expanded", "overlapping", "misaligned"])
def test_odd_layouts_take_the_library(gpu, kind, M):
    K, N = (2048, 4096) if M < 64 else (12288, 512)
    w, x = _bf16(gpu, N, K, seed=1, std=0.03), _odd_rows(gpu, kind, M, K)
    _close(ops.linear(x, w), x.double() @ w.double().t(), 2 ** -8)
    wk = _odd_rows(gpu, kind, N, K)
    _close(ops.linear(_bf16(gpu, M, K), wk), _bf16(gpu, M, K).double() @ wk.double().t(), 2 ** -8)
    gamma = torch.ones(K, device=gpu).bfloat16()
    for delta, h, v in ((x, _bf16(gpu, M, K), w), (None, x, w), (None, _bf16(gpu, M, K), wk)):
        assert ops.norm_linear(delta, h, gamma, 1e-5, v) is None
    if kind == "misaligned":
        odd = torch.ones(K + 4, device=gpu).bfloat16()[4:]
        assert ops.norm_linear(None, _bf16(gpu, M, K), odd, 1e-5, w) is None
        q, s = torch.zeros(N, K, device=gpu, dtype=torch.uint8), torch.ones(N + 1, device=gpu)[1:]
        assert ops.linear_swiglu(_bf16(gpu, M, K), q, s) is None


@pytest.mark.parametrize("M", [2, 12])
def test_weights_whose_rows_lie_far_apart(gpu, monkeypatch, M):
    """Rows past the 32-bit offsets of the workgroups that stay (every one of whose rules is made to ask for them): the kernel with
    64-bit addresses, or the parts; one bf16 rounding, with SwiGLU that of its two operands too."""
    lin = sys.modules["mxllm.ops.linear"]
    for rule in ("_stream_wins", "_norm_wins", "_parts_wins"):
        monkeypatch.setattr(lin, rule, lambda *a: True)
    N, gamma = 64, torch.ones(2048, device=gpu).bfloat16()

    def far(K, stride):
        w = torch.empty_strided((N, K), (stride, 1), device=gpu, dtype=torch.bfloat16)
        w.copy_(_bf16(gpu, N, K, seed=2, std=0.03))
        return w

    x, w = _bf16(gpu, M, 2048, seed=1), far(2048, 1 << 23)
    want = x.double() @ w.double().t()
    _close(ops.linear(x, w), want, 2 ** -8)
    assert ops.linear_parts(_bf16(gpu, 12, 8192), far(8192, 1 << 23)) is None
    assert M > 4 or ops.norm_linear(None, x, gamma, 1e-5, w) is None
    w = far(2048, 1 << 26)
    _close(ops.linear_swiglu(x, w), torch.nn.functional.silu(want[:, :32]) * want[:, 32:], 3 * 2 ** -8)


@pytest.mark.parametrize("M", [1, 16, 64])
def test_switch_off_is_the_library(gpu, M, monkeypatch):
    """MXLLM_SKINNY_M=0: no forward GEMM of inference runs on a kernel of ours."""
    lin = sys.modules["mxllm.ops.linear"]
    monkeypatch.setattr(lin, "SKINNY_M", 0)
    monkeypatch.setattr(lin, "_DECODE_M", 0)
    monkeypatch.setattr(lin, "native", lambda: pytest.fail("a kernel was asked for"))
    x, w = _bf16(gpu, M, 12288), _bf16(gpu, 512, 12288, seed=1, std=0.03)
    _close(ops.linear(x, w), x.double() @ w.double().t(), 2 ** -8)
    assert ops.linear_swiglu(x, w) is None and ops.norm_linear(None, x, x[0].contiguous(), 1e-5, w) is None


@pytest.mark.parametrize("M", [4, 16, 64])
def test_autocast_decides_the_type(gpu, M):
    x, w = _bf16(gpu, M, 12288), _bf16(gpu, 2048, 12288, seed=1, std=0.03)
    for dtype in (torch.float16, torch.bfloat16):
        with torch.autocast("cuda", dtype):
            y = ops.linear(x, w)
        assert y.dtype == dtype
        _close(y, x.double() @ w.double().t(), 2 ** -8)
