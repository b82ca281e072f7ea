"""What a user of the framework has it do, as cases that can be timed and compared: serving steps of every
decoder it has (prompt passes and graphed decode steps through ``Engine``), token sampling, and optimizer steps
of ``Trainer``.

Kinds of case:
  * ``prefill``: one ``Engine.prefill_batch`` of ``prompts`` prompts of ``lo`` to ``hi`` tokens;
  * ``decode``: one ``Engine.decode`` step of ``batch`` sequences that hold ``lo`` to ``hi`` tokens;
  * ``sample``: one ``sample_rows`` of ``batch`` rows of logits, each with its own parameters;
  * ``train``: one ``Trainer.train_step``; ``layers`` 0 takes the model whole, else its first ones (a step of
    the 70B and 8B sizes costs the same a layer, and several replicas have to fit one card).
"""
from __future__ import annotations

import math
import random
import zlib

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

from mxllm.models import MODEL_CLASSES, get_config
from mxllm.ops.decode import sample_rows
from mxllm.parallel.runtime import DistEnv
from mxllm.serve.engine import Engine
from mxllm.serve.quant import quantize_model_fp8_
from mxllm.train.trainer import OptimConfig, Trainer

DEV = torch.device("cuda", 0)
LORA_R, LORA_ALPHA = 16, 32.0
LR, BETA1, BETA2, EPS, CLIP = 1e-4, 0.9, 0.95, 1e-8, 1.0
F64 = torch.float64


def _decode(name, model, batch, lo, hi, fp8=False):
    return {"name": name, "kind": "decode", "model": model, "batch": batch, "lo": lo, "hi": hi, "fp8": fp8}


def _prefill(name, model, prompts, lo, hi, fp8=False):
    return {"name": name, "kind": "prefill", "model": model, "prompts": prompts, "lo": lo, "hi": hi, "fp8": fp8}


def _train(name, model, layers, lora, batch, seq, accum=1):
    return {"name": name, "kind": "train", "model": model, "layers": layers, "lora": lora, "batch": batch, "seq": seq,
            "accum": accum}


def listed():
    return [
        # the draw at the end of a step of a full batch: requests with their own temperature, top-p and top-k
        {"name": "sample_b32", "kind": "sample", "batch": 32, "vocab": 128256},
        # one user of a small model: the least work a step can have, launches and latency
        _decode("llama1b_decode_b1", "llama3.2-1b", 1, 700, 700),
        # a busy server of the 8B size: requests of unlike lengths
        _decode("llama8b_decode_b16", "llama3.1-8b", 16, 100, 2000),
        # fp8 weights, which is how a latency-bound deployment is served
        _decode("llama8b_fp8_decode_b4", "llama3.1-8b", 4, 300, 1100, True),
        # a handful of short requests admitted together
        _prefill("llama1b_prefill_ragged", "llama3.2-1b", 6, 17, 901),
        # one long document
        _prefill("llama8b_prefill_4096", "llama3.1-8b", 1, 4096, 4096),
        _decode("revesun1b_decode_b4", "revesun-1b", 4, 200, 1500),
        _prefill("revesun8b_prefill_ragged", "revesun-8b", 3, 301, 1500),
        _decode("sigusun1b_decode_b32", "sigusun-1b", 32, 50, 1800),
        _prefill("sigusun8b_prefill_2048", "sigusun-8b", 1, 2048, 2048),
        # every weight of a small model
        _train("train_full_1b", "llama3.2-1b", 0, False, 2, 2048),
        # adapters on the 70B sizes, the benchmark's batch: the largest step
        _train("train_lora_70b_layers", "llama3.1-70b", 8, True, 2, 2048),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["decode", "prefill", "train", "sample"], [5, 4, 2, 1])[0]
    if kind == "sample":
        return {"kind": kind, "batch": _log(rng, 1, 64), "vocab": rng.choice([32000, 128256, 50257])}
    if kind == "train":
        model, layers, lora = rng.choice([("llama3.2-1b", 0, False), ("llama3.2-1b", 0, True), ("llama3.1-8b", 6, False),
                                          ("llama3.1-8b", 12, True), ("llama3.1-70b", 6, True)])
        accum, seq = rng.choice([1, 1, 2]), _log(rng, 150, 4096)
        c = _train("", model, layers, lora, max(1, min(4, 4096 // (seq * accum))), seq, accum if 2 * seq <= 4096 else 1)
    else:
        model = "%s-%s" % (rng.choice(["llama", "revesun", "sigusun"]), rng.choice(["1b", "8b"]))
        model = {"llama-1b": "llama3.2-1b", "llama-8b": "llama3.1-8b"}.get(model, model)
        fp8 = model.startswith("llama") and rng.random() < 0.25
        if kind == "decode":
            batch, hi = _log(rng, 1, 48), _log(rng, 30, 3500)
            hi = min(hi, 32000 // batch)
            c = _decode("", model, batch, rng.randint(max(1, hi // 8), hi), hi, fp8)
        else:
            n, hi = _log(rng, 1, 8), _log(rng, 16, 4096)
            hi = min(hi, 5000 // n)
            c = _prefill("", model, n, rng.randint(max(1, hi // 8), hi), hi, fp8)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs
def _config(case):
    cfg = get_config(case["model"])
    return cfg.replace(n_layers=case["layers"]) if case.get("layers") else cfg


def _lengths(case):
    """Tokens of each sequence: spread over lo .. hi, the first the longest."""
    r = random.Random(case["hi"] * 64 + case["lo"])
    n = case["batch"] if case["kind"] == "decode" else case["prompts"]
    return [case["hi"]] + [r.randint(case["lo"], case["hi"]) for _ in range(n - 1)]


def _prompts(case, vocab, seed):
    r = np.random.default_rng([seed, 1])
    return [r.integers(0, vocab, n).tolist() for n in _lengths(case)]


def _next_tokens(case, vocab, seed):
    return np.random.default_rng([seed, 2]).integers(0, vocab, case["batch"]).tolist()


def _weight(name, shape, dtype, seed, family):
    """The parameter ``name`` of a model: random weights that leave the residual stream as a trained model's is,
    many small steps from the token's own row (where every step replaces the stream, rounding is amplified layer by
    layer until it hides what a kernel does)."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1000003 + zlib.crc32(name.encode()))

    def normal(std, mean=0.0):
        return torch.empty(shape, dtype=dtype, device=DEV).normal_(mean, std, generator=g)

    last = name.split(".")[-1]
    if family == "sigusun" and last in ("norm1", "norm2", "side_norm"):
        return normal(0.01, 0.1)
    if "norm" in last:
        return normal(0.1, 1.0)
    if last == "bias":
        return normal(0.5)
    if last == "sink":
        return normal(1.0)
    if last == "conv":
        t = normal(0.2)
        t[:, -1] += 1.0
        return t
    if last == "act":
        return normal(0.03) + torch.tensor([0.5, 0.3, 0.2, 0.1], dtype=dtype, device=DEV)
    if last == "lora_b":
        return normal(0.001)
    if family == "llama" and name.endswith(("wo.weight", "wd.weight")):
        return normal(0.03 / math.sqrt(shape[-1]))
    if family == "llama" and last == "tok_emb":
        return normal(0.05)
    if family == "sigusun" and last in ("tok_emb", "side_emb"):
        return normal(1.0)
    return normal(1.0 / math.sqrt(shape[-1]))


def _family(model):
    return next(f for f in ("llama", "revesun", "sigusun") if model.startswith(f))


@torch.no_grad()
def _model(case, seed, **kw):
    cfg = _config(case)
    model = MODEL_CLASSES[type(cfg)](cfg, device=DEV, dtype=torch.bfloat16, init=False, **kw)
    family = _family(case["model"])
    for name, p in model.named_parameters():
        w = _weight(name, tuple(p.shape), p.dtype, seed, family)
        if name.endswith("lora_b"):  # one block a projection
            lin = model.get_submodule(name[:-len(".lora_b")])
            p.zero_()
            off = 0
            for i, n in enumerate(lin.splits):
                p[off:off + n, i * LORA_R:(i + 1) * LORA_R] = w[off:off + n, i * LORA_R:(i + 1) * LORA_R]
                off += n
        else:
            p.copy_(w)
    if kw.get("lora_r"):
        model.sync_adapters_()
        model.refresh_images_()
    return model


def _batches(case, vocab, seed):
    """(ids, labels) of each micro-batch; the first part of a sequence is its prompt and has no loss."""
    r = np.random.default_rng([seed, 3])
    B, S, out = case["batch"], case["seq"], []
    for _ in range(case["accum"]):
        t = torch.from_numpy(r.integers(0, vocab, (B, S + 1))).to(DEV)
        labels = t[:, 1:].clone()
        labels[:, :S // 4] = -100
        out.append((t[:, :-1].contiguous(), labels))
    return out


def _fill(eng, slots, prompts):
    """Prompt passes of a bounded number of tokens, as the scheduler makes them."""
    at = 0
    while at < len(slots):
        end, n = at + 1, len(prompts[at])
        while end < len(slots) and n + len(prompts[end]) <= 8192:
            n += len(prompts[end])
            end += 1
        eng.prefill_batch(slots[at:end], prompts[at:end])
        at = end


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sample":
        B, r = case["batch"], random.Random(seed)
        g = torch.Generator(device=DEV)
        g.manual_seed(seed)
        # most requests have a nucleus, some top-k as well, some are greedy
        ways = [r.choice([(0.8, 0.9, 0), (0.7, 0.95, 50), (1.0, 1.0, 0), (0.0, 1.0, 0), (0.6, 0.8, 0)]) for _ in range(B)]
        return {"kind": kind, "logits": torch.empty(B, case["vocab"], device=DEV).normal_(0, 2.5, generator=g).bfloat16(),
                "t": [w[0] for w in ways], "p": [w[1] for w in ways], "k": [w[2] for w in ways],
                "seeds": [r.randrange(1 << 31) for _ in range(B)], "steps": [r.randrange(500) for _ in range(B)]}
    if kind == "train":
        lora = {"lora_r": LORA_R, "lora_alpha": LORA_ALPHA} if case["lora"] else {}
        model = _model(case, seed, **lora)
        trainer = Trainer(model, DistEnv(device=DEV), OptimConfig(lr=LR, beta1=BETA1, beta2=BETA2, eps=EPS, grad_clip=CLIP))
        return {"kind": kind, "trainer": trainer, "batches": _batches(case, model.cfg.vocab_size, seed)}
    model = _model(case, seed)
    model.requires_grad_(False)
    if case["fp8"]:
        quantize_model_fp8_(model)
    vocab, lens = model.cfg.vocab_size, _lengths(case)
    eng = Engine(model, max_batch=len(lens), max_seq=max(lens) + 64)
    slots, prompts = [eng.acquire() for _ in lens], _prompts(case, vocab, seed)
    state = {"kind": kind, "engine": eng, "slots": slots}
    if kind == "prefill":
        return {**state, "prompts": prompts}
    _fill(eng, slots, prompts)
    state.update(lens=lens, tokens=torch.tensor(_next_tokens(case, vocab, seed)))
    eng.decode(slots, state["tokens"])  # a server has its step's graph
    _fill(eng, slots, prompts)          # what the step changed is made anew
    return state


def run(state):
    kind = state["kind"]
    if kind == "sample":
        return sample_rows(state["logits"], state["t"], state["p"], state["k"], state["seeds"], state["steps"])
    if kind == "train":
        tr = state["trainer"]
        loss = tr.train_step(state["batches"])
        return {"loss": loss, "grad_norm": tr.last_grad_norm, "weights": tr.flat.params, "m": tr.m, "v": tr.v}
    eng, slots = state["engine"], state["slots"]
    if kind == "prefill":
        return eng.prefill_batch(slots, state["prompts"])
    for s, n in zip(slots, state["lens"]):  # the step after the tokens that each sequence holds
        eng.lens[s] = n
    return eng.decode(slots, state["tokens"])


# ------------------------------------------------------------------ the least a pass moves and computes
def _mixed_params(case):
    """(parameters every token takes outside embedding and head, (experts, top, parameters of one) of all layers)."""
    cfg = _config(case)
    if _family(case["model"]) != "sigusun":
        return cfg.n_params() - cfg.vocab_size * cfg.hidden * (1 if getattr(cfg, "tie_embeddings", True) else 2), []
    dense = sum(s.n_params(cfg.hidden, cfg.side_dim) - s.moe.experts * 3 * cfg.hidden * s.moe.ff for s in cfg.layers)
    return dense, [(s.moe.experts, s.moe.top, 3 * cfg.hidden * s.moe.ff) for s in cfg.layers]


def _attended(case, n):
    """(flops, cached bytes) of the last of n positions: what its layers look back over."""
    cfg = _config(case)
    family = _family(case["model"])
    if family == "llama":
        return 4 * n * cfg.q_dim * cfg.n_layers, 4 * n * cfg.kv_dim * cfg.n_layers
    flops = held = 0
    for s in cfg.layers:
        if family == "revesun":
            if s.attn:
                a, k = s.attn, (n - 1) % s.attn.chunk + 1
                flops += 2 * k * a.heads * (a.dim + a.vdim)
                held += 2 * k * a.kv_heads * (a.dim + a.vdim)
            else:
                held += 8 * s.width
        elif s.lat:
            a, k = s.lat, min(n, s.lat.window or n)
            flops += 2 * k * a.heads * (a.dim + a.rot_dim + a.vdim)
            held += 2 * k * (a.rank + a.rot_dim)
        else:
            flops += 5 * s.ret.state
            held += 8 * s.ret.state
    return flops, held


def work(case):
    if case["kind"] == "sample":
        return {"bytes": 2 * case["batch"] * case["vocab"], "flops": 0}
    cfg = _config(case)
    dense, experts = _mixed_params(case)
    head = cfg.vocab_size * cfg.hidden
    if case["kind"] == "train":
        T = case["batch"] * case["seq"] * case["accum"]
        attn = 3.5 * _attended(case, case["seq"])[0] / 2
        if case["lora"]:
            lora = sum(LORA_R * (cfg.hidden + n) for n in (cfg.q_dim, cfg.kv_dim, cfg.kv_dim, cfg.ffn, cfg.ffn))
            lora = cfg.n_layers * (lora + LORA_R * (cfg.q_dim + cfg.ffn + 2 * cfg.hidden))
            return {"bytes": 2 * (dense + head) + 24 * lora, "flops": T * (4 * (dense + head) + 6 * lora + attn)}
        return {"bytes": 26 * (dense + head), "flops": T * (6 * (dense + head) + attn)}
    lens = _lengths(case)
    T = sum(lens) if case["kind"] == "prefill" else len(lens)
    flops = 2 * T * dense + 2 * len(lens) * head + sum(2 * T * top * n for _, top, n in experts)
    size = 1 if case["fp8"] else 2
    read = size * (dense + sum(e * n * (1 - (1 - top / e) ** T) for e, top, n in experts)) + 2 * head
    for n in lens:
        f, held = _attended(case, n if case["kind"] == "prefill" else n + 1)
        flops += f * n / 2 if case["kind"] == "prefill" else f
        read += held
    return {"bytes": int(read + 2 * len(lens) * cfg.vocab_size), "flops": int(flops)}


def tolerance(case):
    """Activations and products are rounded to bf16 (2^-9 each) through all layers."""
    if case["kind"] == "sample":
        return "exact"
    if case["kind"] == "train":
        return {"rel": 0.03, "max": 0.5}
    return {"rel": 0.03, "max": 0.3}


# ------------------------------------------------------------------ the same in 64 bits, in plain torch
class _Params:
    def __init__(self, case, seed):
        self.seed, self.family, self.fp8 = seed, _family(case["model"]), case.get("fp8", False)

    def __call__(self, name, *shape, dtype=torch.bfloat16):
        w = _weight(name, shape, dtype, self.seed, self.family).double()
        if self.fp8 and name.startswith("layers.") and name.endswith(".weight"):
            # e4m3 codes with a scale a row; codes below the normal range become its smallest
            s = (w.abs().amax(1, keepdim=True).float() / 448.0)
            q = (w.float() / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).double()
            q = torch.where(q.abs() < 2.0 ** -6, torch.copysign(torch.full_like(q, 2.0 ** -6), q), q)
            w = q * s.double()
        return w


def _rms(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


def _inv_freq(dims, base, scaling=None):
    inv = base ** (-torch.arange(0, dims, 2, dtype=F64, device=DEV) / dims)
    if not scaling:
        return inv
    f, old = scaling["factor"], scaling["original_max_position_embeddings"]
    lo, hi = scaling["low_freq_factor"], scaling["high_freq_factor"]
    turns = old * inv / (2 * math.pi)
    mix = ((turns - lo) / (hi - lo)).clamp(0, 1)
    return inv * (mix + (1 - mix) / f)


def _turn(x, inv, pairs):
    """x [T, heads, D] at positions 0 .. T - 1: its first 2 * len(inv) dimensions rotated, dimension 2i with
    2i + 1 (``pairs``) or i with i + len(inv)."""
    n = inv.numel()
    a = torch.arange(x.shape[0], dtype=F64, device=x.device)[:, None] * inv
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    r = x[..., :2 * n]
    u, v = (r[..., 0::2], r[..., 1::2]) if pairs else (r[..., :n], r[..., n:])
    p, q = u * c - v * s, v * c + u * s
    r = torch.stack([p, q], -1).flatten(-2) if pairs else torch.cat([p, q], -1)
    return torch.cat([r, x[..., 2 * n:]], -1)


def _attend(q, k, v, scale, sees, extra=None):
    """q [T, H, D], k [T, G, D], v [T, G, E], sees [T, T]; ``extra`` [H]: logits of a key without a value."""
    H, G, out = q.shape[1], k.shape[1], []
    for h in range(H):
        g = h * G // H
        s = (q[:, h] @ k[:, g].T * scale).masked_fill(~sees, float("-inf"))
        m = s.amax(1, keepdim=True)
        m = m if extra is None else torch.maximum(m, extra[h])
        e = torch.exp(s - m)
        d = e.sum(1, keepdim=True) + (0 if extra is None else torch.exp(extra[h] - m))
        out.append(e @ v[:, g] / d)
    return torch.stack(out, 1)


def _sees(n, window=0, chunk=0):
    i = torch.arange(n, device=DEV)[:, None]
    j = torch.arange(n, device=DEV)[None]
    m = j <= i
    if window:
        m &= j > i - window
    return m & (i // chunk == j // chunk) if chunk else m


def _by_sequence(lens, fn, *rows):
    return torch.cat([fn(*t) for t in zip(*(r.split(lens) for r in rows))])


def _llama_layer(P, cfg, i, x, lens, adapters, norms=None):
    """One layer; ``adapters(projection, input)`` adds what LoRA adds."""
    p, h = "layers.%d." % i, cfg.hidden
    inv = _inv_freq(cfg.head_dim, cfg.rope_theta, cfg.rope_scaling)

    def project(name, x, out):
        return x @ P(p + name + ".weight", out, x.shape[1]).T + adapters(p + name, x)

    def attend(z):
        q, k, v = z.view(z.shape[0], -1, cfg.head_dim).split([cfg.n_heads, cfg.n_kv_heads, cfg.n_kv_heads], 1)
        return _attend(_turn(q, inv, False), _turn(k, inv, False), v, cfg.head_dim ** -0.5, _sees(z.shape[0])).flatten(1)

    z = project("wqkv", _rms(x, P(p + "attn_norm", h), cfg.norm_eps), cfg.q_dim + 2 * cfg.kv_dim)
    x = x + project("wo", _by_sequence(lens, attend, z), h)
    g, u = project("wgu", _rms(x, P(p + "mlp_norm", h), cfg.norm_eps), 2 * cfg.ffn).chunk(2, 1)
    return x + project("wd", torch.nn.functional.silu(g) * u, h)


def _llama(P, cfg, ids, lens):
    x = P("tok_emb", cfg.vocab_size, cfg.hidden)[ids]
    for i in range(cfg.n_layers):
        x = _llama_layer(P, cfg, i, x, lens, lambda name, x: 0)
    return _rms(x, P("final_norm", cfg.hidden), cfg.norm_eps), "tok_emb" if cfg.tie_embeddings else "lm_head"


def _scan(a, b):
    """s_t = a_t s_(t-1) + b_t from nothing, by doubling."""
    n = 1
    while n < a.shape[0]:
        b = torch.cat([b[:n], b[n:] + a[n:] * b[:-n]])
        a = torch.cat([a[:n], a[n:] * a[:-n]])
        n *= 2
    return b


def _revesun(P, cfg, ids, lens):
    f32, h, eps = torch.float32, cfg.hidden, cfg.norm_eps

    def norm(x, name):
        parts = x.view(x.shape[0], cfg.norm_groups, -1)
        return _rms(parts, 1.0, eps).flatten(1) * P(name, h, dtype=f32)

    def unit(x):
        return _rms(x, 1.0, eps)

    x = P("tok_emb", cfg.vocab_size, h)[ids]
    for i, s in enumerate(cfg.layers):
        p = "layers.%d." % i
        y = norm(x, p + "norm1")
        if s.kind == "mingru":
            w = s.width
            z, u, g = (y @ P(p + "wx.weight", 3 * w, h).T).split(w, 1)
            bias = P(p + "bias", 2 * w, dtype=f32)
            z, u = torch.sigmoid(z + bias[:w]), u + bias[w:]
            c = torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
            o = _by_sequence(lens, _scan, 1 - z, z * c) * torch.nn.functional.silu(g)
        else:
            a = s.attn
            wide = [a.heads * a.dim, a.kv_heads * a.dim, a.kv_heads * a.vdim, a.heads * a.vdim]
            taps, inv = P(p + "conv", sum(wide[:3]), a.taps, dtype=f32), _inv_freq(a.rot_dims, s.rot_base)

            def attend(z):
                u, n = z[:, :sum(wide[:3])], z.shape[0]
                u = sum(taps[:, j] * torch.nn.functional.pad(u, (0, 0, a.taps - 1 - j, 0))[:n] for j in range(a.taps))
                q, k, v = u.split(wide[:3], 1)
                q, k = _turn(q.view(n, a.heads, a.dim), inv, True), _turn(k.view(n, a.kv_heads, a.dim), inv, True)
                o = _attend(q, k, v.view(n, a.kv_heads, a.vdim), a.scale, _sees(n, chunk=a.chunk),
                            torch.zeros(a.heads, dtype=F64, device=DEV))
                return o.flatten(1) * torch.sigmoid(z[:, sum(wide[:3]):])

            o = _by_sequence(lens, attend, y @ P(p + "wx.weight", sum(wide), h).T)
        x = x + o @ P(p + "wo.weight", h, o.shape[1]).T
        if s.ff:
            z = norm(x, p + "norm2") @ P(p + "wup.weight", s.ff, h).T
            c = P(p + "act", 4, dtype=f32)
            z = c[0] * unit(z) + c[1] * unit(z ** 2) + c[2] * unit(z ** 3) + c[3]
            x = x + z @ P(p + "wdown.weight", h, s.ff).T
    return norm(x, "final_norm"), "tok_emb"


def _clipped(z, limit):
    g, u = z.chunk(2, 1)
    g = g.clamp(max=limit)
    return g * torch.sigmoid(1.702 * g) * (u.clamp(-limit, limit) + 1)


def _sigusun(P, cfg, ids, lens):
    f32, h, eps, side = torch.float32, cfg.hidden, cfg.norm_eps, cfg.side_dim
    x = _rms(P("tok_emb", cfg.vocab_size, h)[ids], P("emb_norm", h, dtype=f32), eps)
    extra = _weight("side_emb", (cfg.vocab_size, cfg.n_layers * side), torch.bfloat16, P.seed, P.family)[ids].double()
    latents = {}
    for i, s in enumerate(cfg.layers):
        p = "layers.%d." % i
        inv = _inv_freq(s.rot[0], s.rot_base)
        if s.ret:
            H, D, E = s.ret.heads, s.ret.dim, s.ret.vdim
            z = x @ P(p + "wx.weight", sum(s.ret.splits), h).T

            def retain(z):
                n = z.shape[0]
                q, k, v, g = z.split(s.ret.splits, 1)
                q, k = _turn(q.view(n, H, D), inv, False), _turn(k.view(n, H, D), inv, False) * D ** -0.5
                t = torch.arange(n, dtype=F64, device=DEV)
                back, out = t[:, None] - t[None], []
                for j in range(H):
                    fade = torch.where(back >= 0, s.decay[j] ** back.clamp(min=0), 0.0)
                    out.append((q[:, j] @ k[:, j].T * fade) @ v.view(n, H, E)[:, j])
                return _rms(torch.stack(out, 1), 1.0, eps).flatten(1) * torch.nn.functional.silu(g)

            y = _by_sequence(lens, retain, z)
        else:
            a = s.lat
            H, D, R, E = a.heads, a.dim, a.rot_dim, a.vdim
            own = s.kv_from is None
            z = x @ P(p + "wx.weight", a.q_width + (a.rank + R if own else 0), h).T
            if own:
                c = _rms(z[:, a.q_width:a.q_width + a.rank], P(p + "lat_norm", a.rank, dtype=f32), eps)
                latents[i] = c, _by_sequence(lens, lambda r: _turn(r[:, None], inv, True)[:, 0], z[:, a.q_width + a.rank:])
            wkv = P(p + "wkv", H * (D + E), a.rank)
            sink = P(p + "sink", H, dtype=f32) if s.sink else None

            def attend(q, c, r):
                n = q.shape[0]
                q = q.view(n, H, D + R)
                q = torch.cat([q[..., :D], _turn(q[..., D:], inv, True)], -1)
                k, v = (c @ wkv.T).split([H * D, H * E], 1)
                k = torch.cat([k.view(n, H, D), r[:, None].expand(n, H, R)], -1)
                return _attend(q, k, v.view(n, H, E), a.scale, _sees(n, a.window), sink).flatten(1)

            y = _by_sequence(lens, attend, z[:, :a.q_width], *latents[i if own else s.kv_from])
        x = x + _rms(y @ P(p + "wo.weight", h, y.shape[1]).T, P(p + "norm1", h, dtype=f32), eps)
        m = s.moe
        val, at = torch.topk(x @ P(p + "router", m.experts, h).T, m.top, dim=1)
        wt = torch.softmax(val, 1)
        wgu, wdown = P(p + "wgu", m.experts, 2 * m.ff, h), P(p + "wdown", m.experts, h, m.ff)
        y = _clipped(x @ P(p + "sgu.weight", 2 * m.shared_ff, h).T, m.shared_limit) @ P(p + "sdown.weight", h, m.shared_ff).T
        for e in range(m.experts):
            row, j = (at == e).nonzero(as_tuple=True)
            y.index_add_(0, row, wt[row, j, None] * (_clipped(x[row] @ wgu[e].T, m.limit) @ wdown[e].T))
        x = x + _rms(y, P(p + "norm2", h, dtype=f32), eps)
        g = torch.nn.functional.gelu(x @ P(p + "side_gate.weight", side, h).T, approximate="tanh") * extra[:, i * side:(i + 1) * side]
        x = x + _rms(g @ P(p + "side_proj.weight", h, side).T, P(p + "side_norm", h, dtype=f32), eps)
    return _rms(x, P("final_norm", h, dtype=f32), eps), "head"


def _exact_train(case, seed):
    cfg, P, L = _config(case), _Params(case, seed), case["layers"] or get_config(case["model"]).n_layers
    h, q, kv, ff = cfg.hidden, cfg.q_dim, cfg.kv_dim, cfg.ffn
    splits = {"wqkv": (h, [q, kv, kv]), "wo": (q, [h]), "wgu": (h, [ff, ff]), "wd": (ff, [h])}
    leaves, blocks = {}, {}  # in the order of the optimizer's flat buffers: gradients as the backward makes them

    def leaf(name, *shape, block=1.0):
        leaves[name], blocks[name] = (P(name, *shape) * block).requires_grad_(), block

    if not case["lora"] and not cfg.tie_embeddings:
        leaf("lm_head", cfg.vocab_size, h)
    for i in reversed(range(L)):
        p = "layers.%d." % i
        if not case["lora"]:
            leaf("final_norm" if i + 1 == L else "layers.%d.attn_norm" % (i + 1), h)
        for name in ("wd", "wgu", "wo", "wqkv"):
            k, outs = splits[name]
            if case["lora"]:
                block = torch.block_diag(*[torch.ones(n, LORA_R, dtype=F64, device=DEV) for n in outs])
                leaf(p + name + ".lora_b", sum(outs), len(outs) * LORA_R, block=block)
                leaf(p + name + ".lora_a", len(outs) * LORA_R, k)
            else:
                leaf(p + name + ".weight", sum(outs), k)
        if not case["lora"]:
            leaf(p + "mlp_norm", h)
    if not case["lora"]:
        leaf("layers.0.attn_norm", h)
        leaf("tok_emb", cfg.vocab_size, h)

    def param(name, *shape, dtype=torch.bfloat16):
        return leaves[name] if name in leaves else P(name, *shape, dtype=dtype)

    def adapters(name, x):
        if not case["lora"]:
            return 0
        return x @ leaves[name + ".lora_a"].T @ leaves[name + ".lora_b"].T * (LORA_ALPHA / LORA_R)

    total = 0.0
    for ids, labels in _batches(case, cfg.vocab_size, seed):
        x = param("tok_emb", cfg.vocab_size, h)[ids.flatten()]
        for i in range(L):
            x = checkpoint(lambda x, i=i: _llama_layer(param, cfg, i, x, [case["seq"]] * case["batch"], adapters), x,
                           use_reentrant=False)
        x = _rms(x, param("final_norm", h), cfg.norm_eps)
        w = param("tok_emb" if cfg.tie_embeddings else "lm_head", cfg.vocab_size, h)
        loss = torch.nn.functional.cross_entropy(x @ w.T, labels.flatten())
        (loss / case["accum"]).backward()
        total += float(loss.detach())
    grads = {n: w.grad * blocks[n] for n, w in leaves.items()}
    norm = math.sqrt(sum(float(g.square().sum()) for g in grads.values()))
    coef = min(1.0, CLIP / (norm + 1e-6))

    def flat(fn):
        parts = [fn(leaves[n].detach(), g * coef).flatten() for n, g in grads.items()]
        return torch.cat([torch.nn.functional.pad(t, (0, -t.numel() % 64)) for t in parts])

    return {"loss": torch.tensor(total / case["accum"], dtype=F64), "grad_norm": torch.tensor([norm], dtype=F64),
            "weights": flat(lambda w, g: w - LR * g / (g.abs() + EPS)),
            "m": flat(lambda w, g: (1 - BETA1) * g), "v": flat(lambda w, g: (1 - BETA2) * g * g)}


def exact(case, seed):
    if case["kind"] == "sample":  # draws are random numbers of the framework's own
        return None
    if case["kind"] == "train":
        return _exact_train(case, seed)
    cfg, P = _config(case), _Params(case, seed)
    seqs = _prompts(case, cfg.vocab_size, seed)
    if case["kind"] == "decode":
        seqs = [s + [t] for s, t in zip(seqs, _next_tokens(case, cfg.vocab_size, seed))]
    lens = [len(s) for s in seqs]
    if 2 * sum(lens) * (_mixed_params(case)[0] + sum(t * n for _, t, n in _mixed_params(case)[1])) > 3e14:
        return None
    ids = torch.tensor([t for s in seqs for t in s], device=DEV)
    with torch.no_grad():
        x, head = {"llama": _llama, "revesun": _revesun, "sigusun": _sigusun}[P.family](P, cfg, ids, lens)
        last = torch.tensor(np.cumsum(lens) - 1, device=DEV)
        return x[last] @ P(head, cfg.vocab_size, cfg.hidden).T
