"""Sampling semantics (the reference's OpenAI-compatible
completion() at /root/reference/src/distributed_inference.py:37).

CPU: the fp32 oracle applies temperature BEFORE the top-k / nucleus cut.
GPU: the batched HIP sampler (csrc/kernels/sampling.hip) draws from exactly
that distribution (empirical frequencies vs the oracle), keeps greedy rows
greedy in a mixed batch, and reproduces the temperature-only kernel's draws.
"""
import math

import pytest
import torch

from mxllm.ops import decode as dops


def test_filter_probs_tempers_before_nucleus():
    x = torch.tensor([2.0, 1.0, 0.0, -1.0])
    cold = dops.filter_probs(x, 0.25, 0, 0.9)  # sharp: the top token alone reaches 0.9
    hot = dops.filter_probs(x, 4.0, 0, 0.9)    # flat: needs all four
    assert (cold > 0).sum() == 1 and (hot > 0).sum() == 4
    k2 = dops.filter_probs(x, 1.0, 2, 1.0)
    assert (k2 > 0).tolist() == [True, True, False, False]
    assert abs(float(k2.sum()) - 1.0) < 1e-6


def test_cpu_sample_rows_respects_support():
    g = torch.Generator().manual_seed(0)
    x = torch.randn(3, 64, generator=g)
    ids = dops.sample_rows(x, [0.0, 0.8, 1.5], [1.0, 0.5, 0.9], [0, 0, 5], [1, 2, 3], [0, 0, 0])
    assert ids[0] == x[0].argmax()
    assert dops.filter_probs(x[1], 0.8, 0, 0.5)[ids[1]] > 0
    assert dops.filter_probs(x[2], 1.5, 5, 0.9)[ids[2]] > 0


@pytest.mark.gpu
@pytest.mark.parametrize("V,temp,top_k,top_p", [(1000, 0.7, 50, 0.9), (1000, 1.3, 0, 0.8), (777, 1.0, 20, 1.0)])
def test_gpu_sampler_frequencies(gpu, V, temp, top_k, top_p):
    g = torch.Generator().manual_seed(V)
    row = (torch.randn(V, generator=g) * 2.0).to(torch.bfloat16)
    n = 20000
    logits = row.to(gpu).unsqueeze(0).expand(n, V).contiguous()
    ids = dops.sample_rows(logits, [temp] * n, [top_p] * n, [top_k] * n, [7] * n, list(range(n))).cpu()
    ref = dops.filter_probs(row.float(), temp, top_k, top_p)
    emp = torch.bincount(ids, minlength=V).float() / n
    assert (emp[ref == 0] == 0).all(), "drew a token outside the top-k / top-p set"
    tv = 0.5 * (emp - ref).abs().sum().item()
    assert tv < 0.04, tv


@pytest.mark.gpu
def test_gpu_sampler_mixed_batch_and_vocab_128k(gpu):
    V = 128256
    x = torch.randn(4, V, device=gpu).to(torch.bfloat16)
    ids = dops.sample_rows(x, [0.0, 0.9, 0.9, 1.0], [1.0, 1.0, 0.9, 0.5], [0, 0, 0, 40], [3, 3, 3, 3],
                           [5, 5, 5, 5]).cpu()
    assert ids[0] == x[0].float().argmax().item()
    # temperature-only rows draw exactly what the single-row Gumbel kernel draws
    from mxllm.ops import native

    one = native().sample(x[1:2].contiguous(), 0.9, 3, 5).cpu()
    assert ids[1] == one[0]
    assert dops.filter_probs(x[2].float().cpu(), 0.9, 0, 0.9)[ids[2]] > 0
    assert dops.filter_probs(x[3].float().cpu(), 1.0, 40, 0.5)[ids[3]] > 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 128256), (torch.float32, 50001)])
def test_gpu_temperature_rows_split_kernel_matches_topkp_kernel(gpu, dtype, V):
    """Rows without top-k / top-p: the draws of the temperature-only kernel (decode.hip, parameters in device
    arrays) equal the sampler's with thresholds (sampling.hip) for the same (seed, step) noise."""
    from mxllm.ops import native

    B = 6
    x = torch.randn(B, V, device=gpu).to(dtype)
    temps = torch.tensor([0.0, 0.7, 1.0, 1.3, 0.0, 0.2], device=gpu)
    seeds = torch.tensor([1, 2, 3, 4, 5, 123456789], device=gpu, dtype=torch.int64)
    steps = torch.tensor([0, 9, 17, 3, 1, 1000], device=gpu, dtype=torch.int32)
    ones = torch.ones(B, device=gpu)
    zeros = torch.zeros(B, device=gpu, dtype=torch.int32)
    for _ in range(3):
        a = native().sample_temp_rows(x, temps, seeds, steps)
        b = native().sample_rows(x, temps, ones, zeros, seeds, steps)
        assert torch.equal(a, b)
        steps += 1
    # routed entry point
    ids = dops.sample_rows(x, temps.tolist(), [1.0] * B, [0] * B, seeds.tolist(), steps.tolist())
    assert torch.equal(ids, native().sample_rows(x, temps, ones, zeros, seeds, steps))


def test_top_p_zero_is_greedy_cpu():
    """top_p <= 0 (an empty nucleus) samples greedily; NaN is rejected; SamplingParams
    validates its range (the kernel and the oracle used to disagree)."""
    from mxllm.serve.engine import SamplingParams

    x = torch.randn(3, 50, generator=torch.Generator().manual_seed(1))
    ids = dops.sample_rows(x, [1.0, 2.0, 0.5], [0.0, -1.0, 1e-9], [0, 0, 0], [1, 2, 3], [0, 0, 0])
    assert ids[0] == x[0].argmax() and ids[1] == x[1].argmax()
    with pytest.raises(ValueError):
        dops.sample_rows(x, [1.0] * 3, [float("nan")] * 3, [0] * 3, [0] * 3, [0] * 3)
    with pytest.raises(ValueError):
        SamplingParams(top_p=-0.5)
    SamplingParams(top_p=0.0)


@pytest.mark.gpu
def test_top_p_zero_is_greedy_gpu(gpu):
    x = torch.randn(4, 128256, device=gpu).bfloat16()
    ids = dops.sample_rows(x, [1.0, 0.7, 1.0, 0.0], [0.0, -2.0, 0.9, 0.5], [0, 0, 0, 0], [1, 2, 3, 4], [0, 0, 0, 0])
    want = x.float().argmax(-1)
    assert ids[0] == want[0] and ids[1] == want[1] and ids[3] == want[3]


@pytest.mark.gpu
def test_concurrent_samplers_on_two_streams(gpu):
    """The vocabulary-split sampler keeps its partials in a per-call workspace: two
    samplers running concurrently on different streams do not corrupt each other."""
    from mxllm.ops import native

    xs = [torch.randn(64, 128256, device=gpu).bfloat16() for _ in range(2)]
    want = [x.float().argmax(-1) for x in xs]
    streams = [torch.cuda.Stream(gpu) for _ in range(2)]
    torch.cuda.synchronize(gpu)
    outs = [[], []]
    for _ in range(20):
        for k in range(2):
            with torch.cuda.stream(streams[k]):
                outs[k].append(native().sample(xs[k], 0.0, 0, 0))
    torch.cuda.synchronize(gpu)
    for k in range(2):
        for o in outs[k]:
            assert torch.equal(o, want[k])


def _scores(V: int, seed: int, step: int):
    """The sampler's Gumbel noise of a row, and how far the hardware logarithm may be from it: its error of 2^-23
    weighs as much more as -log(u) is below one."""
    import numpy as np

    u32 = np.uint32
    with np.errstate(over="ignore"):
        a, b = u32(seed & 0xFFFFFFFF) * u32(0x9E3779B1), (u32(step) + u32(0x7F4A7C15)) * u32(0x85EBCA77)
        h = a ^ b ^ ((np.arange(V, dtype=u32) + u32(0x165667B1)) * u32(0xC2B2AE3D))
        h ^= h >> u32(15)
        h *= u32(0x2C1B3C6D)
        h ^= h >> u32(12)
        h *= u32(0x297A2D39)
        h ^= h >> u32(15)
    u = ((h >> u32(8)).astype(np.float32) + np.float32(0.5)).astype(np.float64) / 16777216.0  # rounded as on the device
    e = np.maximum(-np.log(u), 2.0 ** -25)
    return torch.from_numpy(-np.log(e)), torch.from_numpy(2.0 ** -22 / e + 1e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("V,dtype", [(16383, torch.float32), (16384, torch.bfloat16), (16385, torch.float32),
                                     (50257, torch.bfloat16), (128256, torch.float32), (128256, torch.bfloat16)])
@pytest.mark.parametrize("shape", ["normal", "flat", "equal", "masked", "peaked"])
def test_gpu_split_sampler_draws(gpu, V, dtype, shape):
    """The draw of every row is the best Gumbel score among the tokens that top-k and top-p keep, both computed in
    f64 (rows whose runner-up or boundary lies within rounding are left out; 70 rows: two launches)."""
    g = torch.Generator().manual_seed(V)
    B = 70
    x = torch.randn(B, V, generator=g) * {"normal": 2.5, "flat": 0.01, "equal": 0.0, "masked": 2.0, "peaked": 9.0}[shape]
    x += 1.5 * (shape == "equal")
    if shape == "masked":
        x[:, torch.rand(V, generator=g) < 0.7] = float("-inf")
    x = x.to(dtype)
    temps = [[0.8, 1.0, 0.0, 0.6, 1.7][i % 5] for i in range(B)]
    tops = [[0.9, 1.0, 0.5, 0.999, 0.02, 0.95, 0.7][i % 7] for i in range(B)]
    ks = [[0, 40, 1, 5000, 0, V, 3, 0, 900][i % 9] for i in range(B)]
    seeds, steps = [(i * 2654435761) % (1 << 40) for i in range(B)], [i * 3 for i in range(B)]
    got = dops.sample_rows(x.to(gpu), temps, tops, ks, seeds, steps).cpu()
    from mxllm.ops import native

    dev = [torch.tensor(t, dtype=d, device=gpu) for t, d in zip(
        (temps, tops, ks, seeds, steps), (torch.float32, torch.float32, torch.int32, torch.int64, torch.int32))]
    assert torch.equal(native().sample_rows(x.to(gpu), *dev).cpu(), got)
    checked = 0
    for i in range(B):
        row = x[i].double()
        if temps[i] <= 0:
            assert got[i] == row.argmax()
            continue
        t = float(torch.tensor(temps[i], dtype=torch.float32))
        keep = row > float("-inf")
        if 0 < ks[i] < V:
            keep &= row >= torch.topk(row, ks[i]).values[-1]
        w = torch.where(keep, torch.exp((row - row.max()) / t), 0.0)
        vals, inv = torch.unique(row, return_inverse=True)  # tokens of one value stay together
        mass = torch.zeros(len(vals), dtype=torch.float64).index_add_(0, inv, w)
        above = (mass.flip(0).cumsum(0).flip(0) - mass)[inv]
        if tops[i] < 1:
            p = float(torch.tensor(tops[i], dtype=torch.float32)) * w.sum()
            if (above[keep] - p).abs().min() < 1e-5 * w.sum():  # 2^17 masses of 2^-24 relative rounding, in f32
                continue
            keep &= above < p
        noise, err = _scores(V, seeds[i], steps[i])
        s = torch.where(keep, row / t + noise, float("-inf"))
        best = int((s - err).argmax())
        assert keep[got[i]], (i, temps[i], tops[i], ks[i])
        rest = s + err
        rest[best] = float("-inf")
        if (s - err)[best] > rest.max():
            assert got[i] == best, (i, temps[i], tops[i], ks[i])
            checked += 1
    assert checked > B // 5


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kept", [1, 63, 2047, 2048, 2049, 6000])
def test_gpu_split_sampler_kept_tokens_of_one_chunk(gpu, kept, dtype):
    """Kept tokens are gathered up to 2,048 a chunk, the rest scored where they lie: as many about that, all in the first
    8,192 of 16,384 (a chunk of a 64-row call) and in the histogram's first bin.  The cut of mass or count falls among 30 tokens
    131 bins lower, in the other chunk: what is ahead of them is scored and not listed.  The others lie in the last bin."""
    V, B, T, low = 16384, 64, 0.7, 30
    g = torch.Generator().manual_seed(kept)
    x = torch.full((B, V), -300.0)
    for i in range(B):
        x[i, torch.randperm(8192, generator=g)[:kept]] = 1.0
        x[i, 8192 + torch.randperm(8192, generator=g)[:low]] = 0.0
    x = x.to(dtype)
    below = low * math.exp(-1.0 / T)
    p, seeds = (kept + below / 2) / (kept + below), [7 * i for i in range(B)]
    wins = 0
    for step in (3, 4, 5, 6):
        got = dops.sample_rows(x.to(gpu), [T] * B, [p, 1.0] * (B // 2), [0, kept + low // 3] * (B // 2), seeds, [step] * B).tolist()
        for i in range(B):
            noise, err = _scores(V, seeds[i], step)
            s = torch.where(x[i] >= 0, x[i].double() / T + noise, float("-inf"))
            best = int((s - err).argmax())
            rest = s + err
            rest[best] = float("-inf")
            assert x[i, got[i]] >= 0 and (got[i] == best or (s - err)[best] <= rest.max()), (i, step)
            wins += got[i] < 8192
    assert wins > 3 * B if kept > 1 else 0 < wins < 4 * B  # the gathered ones hold most of the mass, or an eighth of it


@pytest.mark.gpu
@pytest.mark.parametrize("V", [1000, 16384, 50257])
@pytest.mark.parametrize("temp,p,k", [(0.8, 1.0, 0), (0.8, 0.9, 0), (0.8, 1.0, 40), (0.8, 0.9, 40), (0.0, 1.0, 0)])
def test_gpu_sampler_without_numbers(gpu, V, temp, p, k):
    """Rows that hold no number give token 0, never an id outside the vocabulary; tokens without a number are not
    drawn; an infinite logit is.  Both forms of the sampler, beside a row that needs neither."""
    g = torch.Generator().manual_seed(V)
    x = torch.randn(5, V, generator=g)
    x[0] = float("nan")
    x[1] = float("-inf")
    x[2, torch.rand(V, generator=g) < 0.1] = float("nan")
    x[3, V // 2] = float("inf")
    ids = dops.sample_rows(x.to(gpu), [temp] * 4 + [1.0], [p] * 5, [k] * 5, list(range(5)), [7] * 5).tolist()
    assert ids[:2] == [0, 0] and ids[3] == V // 2 and 0 <= ids[4] < V
    assert 0 <= ids[2] < V and not x[2, ids[2]].isnan()
    assert temp > 0 or ids[2] == x[2].nan_to_num(-1e9).argmax()


def test_split_sampler_masses_fit():
    """The split form takes no row whose masses, each up to 2^42, could sum to 2^64 (a total of zero restricts nothing);
    it alone has a workspace."""
    import ctypes

    from mxllm.ops import _ext

    if not _ext.available():
        pytest.skip("native library not built")
    ws = ctypes.CDLL(_ext.LIB).mx_sample_rows_ws
    ws.restype = ctypes.c_int64
    taken = [V for V in (1, 16383, 16384, (1 << 22) - 1, 1 << 22, 1 << 23) if ws(1, V) > 0]
    assert taken == [16384, (1 << 22) - 1] and max(taken) << 42 < 1 << 64


@pytest.mark.gpu
def test_concurrent_mixed_samplers_on_two_streams(gpu):
    """Two samplers of rows with their own temperature, top-k and top-p on different streams at once: every call has its
    own histograms, lists and counters, so the draws are those of the calls one by one."""
    B, V = 40, 128256
    g = torch.Generator(device=gpu).manual_seed(1)
    xs = [torch.empty(B, V, device=gpu).normal_(0, 2.5, generator=g).bfloat16() for _ in range(2)]
    ways = [(0.8, 0.9, 0), (0.7, 0.95, 50), (1.0, 1.0, 0), (0.0, 1.0, 0), (1.3, 1.0, 40)]
    temps, tops, ks = zip(*(ways[i % 5] for i in range(B)))

    def draw(k, step):
        return dops.sample_rows(xs[k], temps, tops, ks, [100 * k + i for i in range(B)], [step] * B)

    want = [[draw(k, step).clone() for step in range(10)] for k in range(2)]
    streams = [torch.cuda.Stream(gpu) for _ in range(2)]
    torch.cuda.synchronize(gpu)
    got = [[], []]
    for step in range(10):
        for k in range(2):
            with torch.cuda.stream(streams[k]):
                got[k].append(draw(k, step))
    torch.cuda.synchronize(gpu)
    assert all(torch.equal(a, b) for k in range(2) for a, b in zip(got[k], want[k]))


@pytest.mark.gpu
@pytest.mark.parametrize("V,dtype", [(16384, torch.bfloat16), (16389, torch.bfloat16), (50257, torch.float32)])
def test_gpu_split_sampler_does_not_depend_on_the_batch(gpu, V, dtype):
    """Rows by themselves, in sevens and all 70 at once (other chunks of a row, other alignments of its start): the masses
    are sums of integers, so every way draws the same tokens."""
    B = 70
    x = (torch.randn(B, V, generator=torch.Generator().manual_seed(V)) * 2.5).to(dtype).to(gpu)
    ways = [(0.8, 0.9, 0), (0.7, 0.95, 50), (1.0, 1.0, 0), (1.3, 0.999, 0), (0.0, 1.0, 0), (0.9, 1.0, 3000)]
    temps, tops, ks = zip(*(ways[i % 6] for i in range(B)))

    def draw(n):
        return torch.cat([dops.sample_rows(x[i:i + n], temps[i:i + n], tops[i:i + n], ks[i:i + n], range(i, min(B, i + n)),
                                           [9] * min(n, B - i)) for i in range(0, B, n)])

    want = draw(70)
    assert torch.equal(draw(1), want) and torch.equal(draw(7), want)
