"""Sigusun: a decoder whose layers mix retention with latent attention (windowed or causal with a softmax
sink), expert mixtures for feed-forwards, and a second token embedding that every layer adds its part of
(MI355X serving layout).

Sublayers read the f32 residual stream itself and are RMS-normed at their output.  Every size and constant
comes from ``config.json`` (``SigusunConfig.from_json``); layers differ freely in kind and sizes.  The
projections that read a layer's input are one GEMM: q | k | v | gate of a retention layer, q | latent |
rotated key of a latent-attention layer.  ``rows`` runs the layer stack over a row layout of
mxllm/ops/hybrid.py: whole prompts of several sequences, or one token each.

Weights: projections, experts, router and embeddings in the model dtype (bf16, or f32 for a true-f32 run); norm
weights, sinks and decays in f32.
"""
from __future__ import annotations

import dataclasses
import json
import math
import os
from dataclasses import dataclass

import torch
import torch.nn as nn

from ..ops import hybrid as hops
from ..ops import latent as lops
from ..ops import linear
from ..ops import moe as mops
from ..ops import sublayer as sops
from ..ops.hybrid import PromptRows, RopeTables
from ..ops.latent import LatentShape
from ..ops.retention import RetentionShape, decay_table, retention
from .config import PRESETS
from .llama import FusedLinear, hooked, plain_weight

# latent-attention layer types -> whether the softmax has a sink
LATENT_TYPES = {"latent_attention": False, "latent_attention_2": True}


@dataclass(frozen=True)
class MoeShape:
    """``top`` of ``experts`` feed-forwards of width ``ff`` a token; ``shared_ff`` (0: none) of the one that
    every token takes.  ``limit`` clips an expert's inputs."""

    experts: int
    top: int
    ff: int
    limit: float
    shared_ff: int = 0
    shared_limit: float = 0.0

    def n_params(self, h: int) -> int:
        return h * (self.experts * (1 + 3 * self.ff) + 3 * self.shared_ff)


@dataclass(frozen=True)
class LayerSpec:
    """One layer: retention (``ret``, ``decay``) or latent attention (``lat``; ``sink``; ``kv_from``: the layer
    whose latent it uses, None: its own), and its feed-forward ``moe`` (None: none)."""

    rot_base: float
    ret: RetentionShape | None = None
    decay: tuple = ()
    lat: LatentShape | None = None
    sink: bool = False
    kv_from: int | None = None
    moe: MoeShape | None = None

    @property
    def rot(self) -> tuple[int, float]:
        return (self.ret.rot_dims if self.ret else self.lat.rot_dim), self.rot_base

    def n_params(self, h: int, side: int) -> int:
        n = 2 * h * side + 2 * h
        if self.ret:
            n += h * (sum(self.ret.splits) + self.ret.heads * self.ret.vdim)
        else:
            a = self.lat
            n += h * (a.q_width + a.heads * a.vdim) + a.rank * a.heads * (a.dim + a.vdim) + (a.heads if self.sink else 0)
            if self.kv_from is None:
                n += h * (a.rank + a.rot_dim) + a.rank
        return n + (h + self.moe.n_params(h) if self.moe else 0)


@dataclass(frozen=True)
class SigusunConfig:
    name: str
    vocab_size: int
    hidden: int
    layers: tuple
    side_dim: int
    norm_eps: float = 1e-5
    max_seq_len: int = 131072  # the design has no limit of its own: the longest the rotation tables go
    bos_id: int = 256
    eos_id: int = -1           # no end token: generation ends by length or a request's stop ids

    @property
    def n_layers(self) -> int:
        return len(self.layers)

    def n_params(self) -> int:
        return (sum(s.n_params(self.hidden, self.side_dim) for s in self.layers)
                + self.vocab_size * (2 * self.hidden + self.n_layers * self.side_dim) + 2 * self.hidden)

    def replace(self, **kw) -> "SigusunConfig":
        return dataclasses.replace(self, **kw)

    def latent_source(self, i: int) -> int:
        """The layer whose latent layer i attends to."""
        s = self.layers[i]
        return i if s.kv_from is None else s.kv_from

    def look_back(self, i: int) -> int:
        """Positions of layer i's latent that some layer still sees (0: all of them)."""
        w = [s.lat.window for j, s in enumerate(self.layers) if s.lat and self.latent_source(j) == i]
        return 0 if 0 in w else max(w)

    @staticmethod
    def from_json(d: dict, name: str = "sigusun") -> "SigusunConfig":
        specs: list[LayerSpec] = []
        for i, e in enumerate(d["layers"]):
            mx, rot = e["mixer"], e["mixer"]["rot"]
            moe = _moe_from(e.get("mlp"), i)
            if e["type"] == "retention":
                r = RetentionShape(heads=int(mx["heads"]), dim=int(mx["dim"]), vdim=int(mx["vdim"]), rot_dims=int(rot["dims"]))
                decay = tuple(float(x) for x in mx["decay"])
                if len(decay) != r.heads or r.rot_dims % 2 or r.rot_dims > r.dim:
                    raise ValueError(f"layer {i}: inconsistent retention sizes {r}, {len(decay)} decays")
                specs.append(LayerSpec(float(rot["base"]), ret=r, decay=decay, moe=moe))
            elif e["type"] in LATENT_TYPES:
                mask = mx.get("mask")
                a = LatentShape(heads=int(mx["heads"]), dim=int(mx["dim"]), rot_dim=int(mx["rot_dim"]), vdim=int(mx["vdim"]),
                                rank=int(mx["kv_rank"]), scale=float(mx["scale"]),
                                window=int(mask["size"]) if mask else 0)
                src = mx.get("kv_from")
                if a.rot_dim % 2 or int(rot["dims"]) != a.rot_dim or (mask and a.window < 1):
                    raise ValueError(f"layer {i}: inconsistent latent attention sizes {a}")
                spec = LayerSpec(float(rot["base"]), lat=a, sink=LATENT_TYPES[e["type"]],
                                 kv_from=None if src is None else int(src), moe=moe)
                if spec.kv_from is not None:
                    o = specs[spec.kv_from] if 0 <= spec.kv_from < i else None
                    if o is None or o.lat is None or o.kv_from is not None or (o.lat.rank, o.rot) != (a.rank, spec.rot):
                        raise ValueError(f"layer {i}: layer {src} has no latent that fits")
                specs.append(spec)
            else:
                raise ValueError(f"layer {i}: unknown layer type {e['type']!r}")
        return SigusunConfig(name=name, vocab_size=int(d["vocab"]), hidden=int(d["width"]), layers=tuple(specs),
                             side_dim=int(d["token_side"]["dim"]), norm_eps=float(d["norm"]["eps"]),
                             bos_id=256 if d["vocab"] > 256 else 0)

    def to_json(self) -> dict:
        layers = []
        for s in self.layers:
            rot = {"base": s.rot_base, "dims": s.rot[0]}
            if s.ret:
                mx = {"heads": s.ret.heads, "dim": s.ret.dim, "vdim": s.ret.vdim, "decay": list(s.decay), "rot": rot}
                kind = "retention"
            else:
                a = s.lat
                mx = {"heads": a.heads, "dim": a.dim, "rot_dim": a.rot_dim, "vdim": a.vdim, "kv_rank": a.rank,
                      "scale": a.scale, "rot": rot}
                if a.window:
                    mx["mask"] = {"size": a.window}
                if s.kv_from is not None:
                    mx["kv_from"] = s.kv_from
                kind = next(k for k, sink in LATENT_TYPES.items() if sink == s.sink)
            m = s.moe
            mlp = None if m is None else {
                "kind": "moe", "expert": {"ff": m.ff, "limit": m.limit}, "router": {"experts": m.experts, "top": m.top},
                "shared": {"ff": m.shared_ff, "limit": m.shared_limit} if m.shared_ff else None}
            layers.append({"type": kind, "mixer": mx, "mlp": mlp})
        return {"architecture": "Sigusun", "vocab": self.vocab_size, "width": self.hidden, "layers": layers,
                "norm": {"eps": self.norm_eps}, "token_side": {"dim": self.side_dim}}


def _moe_from(mlp: dict | None, i: int) -> MoeShape | None:
    if mlp is None:
        return None
    if mlp.get("kind", "moe") != "moe":
        raise ValueError(f"layer {i}: feed-forward kind {mlp['kind']!r} is not supported")
    r, e, sh = mlp["router"], mlp["expert"], mlp.get("shared")
    m = MoeShape(int(r["experts"]), int(r["top"]), int(e["ff"]), float(e["limit"]),
                 int(sh["ff"]) if sh else 0, float(sh["limit"]) if sh else 0.0)
    if not 0 < m.top <= m.experts:
        raise ValueError(f"layer {i}: {m.top} of {m.experts} experts")
    return m


class SigusunLayer(nn.Module):
    """``wx``: the projections of the layer's input; ``wkv``: keys and values of the latent [heads x dim +
    heads x vdim, rank]; ``wo``: the mixer's output; ``wgu`` / ``wdown``: the experts [experts, gate | up, W],
    [experts, W, ff]; ``sgu`` / ``sdown``: the shared one; ``side_gate`` / ``side_proj``: the token input."""

    def __init__(self, spec: LayerSpec, h: int, side: int, *, dtype, device):
        super().__init__()
        self.spec = spec
        kw = dict(dtype=dtype, device=device)

        def f32(*shape, value=0.0):
            return nn.Parameter(torch.full(shape, value, dtype=torch.float32, device=device))

        def param(*shape):
            return nn.Parameter(torch.empty(*shape, **kw))

        self.norm1 = f32(h, value=1.0)
        if spec.ret:
            r = spec.ret
            self.wx = FusedLinear(h, r.splits, **kw)
            self.wo = FusedLinear(r.heads * r.vdim, [h], **kw)
            self.register_buffer("decay", decay_table(spec.decay, device), persistent=False)
        else:
            a = spec.lat
            own = spec.kv_from is None
            self.wx = FusedLinear(h, [a.q_width] + ([a.rank + a.rot_dim] if own else []), **kw)
            if own:
                self.lat_norm = f32(a.rank, value=1.0)
            self.wkv = param(a.heads * (a.dim + a.vdim), a.rank)
            self.wuk_t = None  # key_weight(wkv), Sigusun.prepare
            self.sink = f32(a.heads) if spec.sink else None
            self.wo = FusedLinear(a.heads * a.vdim, [h], **kw)
        m = spec.moe
        if m:
            self.norm2 = f32(h, value=1.0)
            self.router = param(m.experts, h)
            self.wgu = param(m.experts, 2 * m.ff, h)
            self.wdown = param(m.experts, h, m.ff)
            if m.shared_ff:
                self.sgu = FusedLinear(h, [m.shared_ff] * 2, **kw)
                self.sdown = FusedLinear(m.shared_ff, [h], **kw)
        self.side_gate = FusedLinear(h, [side], **kw)
        self.side_proj = FusedLinear(side, [h], **kw)
        self.side_norm = f32(h, value=1.0)


def _refresh_loaded(model, incompatible) -> None:
    model.refresh()


class Sigusun(nn.Module):
    serves_float32 = True  # every kernel has an f32 form
    native_component = "serve"  # the part of the native library it needs (mxllm/_build.py)

    def __init__(self, cfg: SigusunConfig, *, device=None, dtype=torch.bfloat16, seed: int = 0, init: bool = True,
                 lora_r: int = 0, lora_alpha: float = 16.0):
        super().__init__()
        if lora_r:
            raise NotImplementedError("Sigusun has no LoRA adapters (serving only)")
        device = torch.device(device) if device is not None else torch.device("cpu")
        self.cfg = cfg
        self.dtype = dtype

        def param(*shape):
            return nn.Parameter(torch.empty(*shape, dtype=dtype, device=device))

        def ones():
            return nn.Parameter(torch.ones(cfg.hidden, dtype=torch.float32, device=device))

        self.tok_emb = param(cfg.vocab_size, cfg.hidden)
        self.side_emb = param(cfg.vocab_size, cfg.n_layers * cfg.side_dim)
        self.head = param(cfg.vocab_size, cfg.hidden)
        self.emb_norm, self.final_norm = ones(), ones()
        self.layers = nn.ModuleList([SigusunLayer(s, cfg.hidden, cfg.side_dim, dtype=dtype, device=device)
                                     for s in cfg.layers])
        self.tables = RopeTables(device)
        self.shared_latents = {s.kv_from for s in cfg.layers if s.kv_from is not None}
        # index of each retention layer among them (its state)
        self.state_index = [sum(1 for t in cfg.layers[:i] if t.ret) for i in range(cfg.n_layers)]
        if init:
            self.reset_parameters(seed)
        self.requires_grad_(False)
        self.register_load_state_dict_post_hook(_refresh_loaded)

    @torch.no_grad()
    def reset_parameters(self, seed: int = 0):
        """Random weights that keep activations near unit scale."""
        gen = torch.Generator(device=self.tok_emb.device)
        gen.manual_seed(seed)

        def fan_in(t: torch.Tensor):
            t.normal_(0.0, 1.0 / math.sqrt(t.shape[-1]), generator=gen)

        self.tok_emb.normal_(0.0, 1.0, generator=gen)
        self.side_emb.normal_(0.0, 1.0, generator=gen)
        fan_in(self.head)
        for layer in self.layers:
            for m in layer.children():
                fan_in(m.weight)
            for name in ("wkv", "router", "wgu", "wdown"):
                if getattr(layer, name, None) is not None:
                    fan_in(getattr(layer, name))
            if getattr(layer, "sink", None) is not None:
                layer.sink.normal_(0.0, 1.0, generator=gen)
        self.refresh()

    @property
    def head_weight(self) -> torch.Tensor:
        return self.head

    def prepare(self, max_seq: int) -> None:
        """Build what decoding derives once (its storage must not move under a captured graph): rotation tables,
        and in bf16 the key weights transposed."""
        for s in self.cfg.layers:
            self.tables.get(*s.rot, max_seq)
        self.refresh(True)

    @torch.no_grad()
    def refresh(self, make: bool = False) -> None:
        """Derive the transposed key weights again, in their storage: after the parameters were written (loading a state dict,
        ``reset_parameters`` and ``prepare`` do it themselves).  ``make``: those that are not there yet too."""
        for s, layer in zip(self.cfg.layers, self.layers):
            if not s.lat or not layer.wkv.is_cuda or self.dtype != torch.bfloat16 or (layer.wuk_t is None and not make):
                continue
            t = lops.key_weight(layer.wkv.data, s.lat)
            if layer.wuk_t is None or layer.wuk_t.device != t.device:
                layer.wuk_t = t
            else:
                layer.wuk_t.copy_(t)

    # ------------------------------------------------------------------ the layer stack
    def _mixer(self, i: int, x: torch.Tensor, rows, n: int, latents: dict) -> torch.Tensor:
        """Output of layer i's mixer for the rows ``x``."""
        layer, s = self.layers[i], self.layers[i].spec
        cos, sin = self.tables.get(*s.rot, n)
        z = layer.wx(x)
        if s.ret:
            return layer.wo(retention(z, layer.decay, cos, sin, s.ret, self.cfg.norm_eps, rows, self.state_index[i]))
        src, a = self.cfg.latent_source(i), s.lat
        if rows.decode:
            own = (z[:, a.q_width:], layer.lat_norm) if src == i else (None, None)
            return layer.wo(lops.latent_step(z[:, :a.q_width], own[0], layer.wkv, layer.wuk_t, own[1], self.cfg.norm_eps, cos,
                                             sin, layer.sink, a, rows, rows.caches.latent[src]))
        cache = rows.caches.latent[src] if rows.caches is not None else None
        if src == i:
            lat = lops.latent_rows(z[:, a.q_width:], layer.lat_norm, self.cfg.norm_eps, cos, sin, a, rows, cache)
            if i in self.shared_latents:
                latents[i] = lat
        else:
            lat = latents[src]
        return layer.wo(lops.latent_attention(z[:, :a.q_width], lat, layer.wkv, cos, sin, layer.sink, a, rows, cache))

    def _mixture(self, layer: SigusunLayer, y: torch.Tensor, h: torch.Tensor) -> torch.Tensor:
        """Residual steps of the mixer's output ``y`` and of the feed-forward behind it."""
        m, eps = layer.spec.moe, self.cfg.norm_eps
        r = sops.post_route(y, h, layer.norm1, eps, layer.router, m.top)
        if r is None:
            x = sops.post_norm(y, h, layer.norm1, eps)
            ids, wts = mops.route(x, layer.router, m.top)
        else:
            x, ids, wts = r
        shared = self._shared(layer)
        y, inv, sh = mops.experts(x, ids, layer.wgu, layer.wdown, m.limit, *(shared or ()))
        if m.shared_ff and shared is None:
            sh = layer.sdown(sops.clipped_glu(layer.sgu(x), m.shared_limit))
        return sops.mix_post_norm(y, inv, wts, sh, h, layer.norm2, eps)

    @staticmethod
    def _shared(layer: SigusunLayer):
        """(gate | up, down, limit) of the shared expert where there is one and it is not quantised."""
        m = layer.spec.moe
        if not m.shared_ff or plain_weight(layer.sgu) is None or plain_weight(layer.sdown) is None:
            return None
        return layer.sgu.weight, layer.sdown.weight, m.shared_limit

    def _fused(self, layer: SigusunLayer, y: torch.Tensor, h: torch.Tensor, ids: torch.Tensor, off: int):
        """Decode rows, from the mixer's output to the gated token input: (new h, gate), or None where the
        fused kernels do not take the layer."""
        m, eps, gate = layer.spec.moe, self.cfg.norm_eps, plain_weight(layer.side_gate)
        side = (self.side_emb, ids, off)
        if m is None:
            if not sops.fusable(y, gate):
                return None
            h, _, g = sops.post_dots(y, h, layer.norm1, eps, gate, None, None, *side)
            return h, g
        shared = self._shared(layer)
        if (not sops.fusable(y, gate, layer.router) or m.experts > 64 or (m.shared_ff and shared is None)
                or not mops.few(y, m.top, layer.wgu, shared[0] if shared else None)):
            return None
        h, x, logits = sops.post_dots(y, h, layer.norm1, eps, layer.router)
        e, wts, sh = mops.experts_of(x, logits, m.top, layer.wgu, layer.wdown, m.limit, *(shared or ()))
        h, _, g = sops.post_dots(e, h, layer.norm2, eps, gate, wts, sh, *side)
        return h, g

    def rows(self, ids: torch.Tensor, rows, tap=None) -> torch.Tensor:
        """Final normed hidden rows of token ``ids`` [T] laid out as ``rows``.  ``tap(i, h)``: the
        residual stream after layer i (diagnostics)."""
        c, eps = self.cfg, self.cfg.norm_eps
        n = 0 if rows.decode else max(rows.lens)  # decode: the tables prepare() sized
        h, x = sops.embed_norm(ids, self.tok_emb, self.emb_norm, eps)
        latents: dict = {}
        for i, layer in enumerate(self.layers):
            y, off = self._mixer(i, x, rows, n, latents), i * c.side_dim
            r = self._fused(layer, y, h, ids, off) if rows.decode else None
            if r is not None:
                h, g = r
            else:
                x = self._mixture(layer, y, h) if layer.spec.moe else sops.post_norm(y, h, layer.norm1, eps)
                w = plain_weight(layer.side_gate)
                g = None if w is None or hooked(layer.side_gate) else sops.side_gate(x, w, self.side_emb, ids, off)
                if g is None:
                    g = sops.side_act(layer.side_gate(x), self.side_emb, ids, off)
            x = sops.side_post(g, plain_weight(layer.side_proj), h, layer.side_norm, eps) if rows.decode else None
            if x is None:
                x = sops.post_norm(layer.side_proj(g), h, layer.side_norm, eps)
            if tap is not None:
                tap(i, h.clone())
        return hops.group_norm(None, h, self.final_norm, 1, eps, self.dtype)

    @torch.no_grad()
    def hidden_states(self, ids: torch.Tensor, tap=None) -> torch.Tensor:
        """ids [B, S] -> final normed hidden [B * S, H]; nothing is cached."""
        B, S = ids.shape
        return self.rows(ids.reshape(-1), PromptRows([S] * B, self.tok_emb.device), tap)

    @torch.no_grad()
    def forward(self, ids: torch.Tensor) -> torch.Tensor:
        """Logits [B, S, V] of whole sequences."""
        return linear(self.hidden_states(ids), self.head_weight).view(*ids.shape, -1)

    def num_params(self, trainable_only: bool = False) -> int:
        return 0 if trainable_only else sum(p.numel() for p in self.parameters())


# ------------------------------------------------------------------ checkpoints
def load_config(path: str) -> SigusunConfig:
    with open(os.path.join(path, "config.json")) as f:
        return SigusunConfig.from_json(json.load(f), name=os.path.basename(os.path.normpath(path)))


def name_map(cfg: SigusunConfig) -> dict[str, list[str]]:
    """mxllm parameter -> the checkpoint tensors whose rows it concatenates (the experts' 3-D parameters
    taken as rows)."""
    m = {"tok_emb": ["embed"], "emb_norm": ["embed.norm"], "side_emb": ["side.embed"], "final_norm": ["final.norm"],
         "head": ["head"]}
    for i, s in enumerate(cfg.layers):
        p, q = f"layers.{i}.", f"l{i}."
        mix, mlp = q + "mix.", q + "mlp."
        m[p + "norm1"] = [q + "norm1"]
        m[p + "wo.weight"] = [mix + "o"]
        if s.ret:
            m[p + "wx.weight"] = [mix + n for n in ("q", "k", "v", "g")]
        else:
            own = s.kv_from is None
            m[p + "wx.weight"] = [mix + "q"] + ([mix + "dkv"] if own else [])
            if own:
                m[p + "lat_norm"] = [mix + "dkv.norm"]
            m[p + "wkv"] = [mix + "uk", mix + "uv"]
            if s.sink:
                m[p + "sink"] = [mix + "sink"]
        if s.moe:
            ex = [f"{mlp}e{j}." for j in range(s.moe.experts)]
            m[p + "norm2"] = [q + "norm2"]
            m[p + "router"] = [mlp + "router"]
            m[p + "wgu"] = [e + n for e in ex for n in ("gate", "up")]
            m[p + "wdown"] = [e + "down" for e in ex]
            if s.moe.shared_ff:
                m[p + "sgu.weight"] = [mlp + "shared.gate", mlp + "shared.up"]
                m[p + "sdown.weight"] = [mlp + "shared.down"]
        m.update({p + "side_gate.weight": [q + "side.gate"], p + "side_proj.weight": [q + "side.proj"],
                  p + "side_norm": [q + "side.norm"]})
    return m


def _as_rows(t: torch.Tensor) -> torch.Tensor:
    return t.view(-1, t.shape[-1]) if t.dim() == 3 else t


@torch.no_grad()
def load_sigusun(path: str, *, device=None, dtype: torch.dtype = torch.bfloat16, **kw) -> Sigusun:
    """The model of a directory with ``config.json`` and safetensors (strict: every tensor present,
    fitting, and used)."""
    from .hf import HFReader

    cfg = load_config(path)
    kw.pop("seed", None)
    model = Sigusun(cfg, device=device, dtype=dtype, init=False, **kw)
    rd = HFReader(path)
    params = dict(model.named_parameters())
    for name, srcs in name_map(cfg).items():
        rd.fill_(_as_rows(params[name].data), srcs)
    rd.check_all_used(False)
    return model


@torch.no_grad()
def save_sigusun(model: Sigusun, path: str) -> str:
    """Write ``config.json`` + ``model.safetensors`` readable by :func:`load_sigusun` (bf16 tensors)."""
    from safetensors.torch import save_file

    os.makedirs(path, exist_ok=True)
    with open(os.path.join(path, "config.json"), "w") as f:
        json.dump(model.cfg.to_json(), f, indent=1)
    params, out = dict(model.named_parameters()), {}
    for name, srcs in name_map(model.cfg).items():
        t = _as_rows(params[name].detach().to("cpu", torch.bfloat16))
        for src, part in zip(srcs, t.split(_rows_of(model, name, len(srcs), t.shape[0]))):
            out[src] = part.contiguous()
    fn = os.path.join(path, "model.safetensors")
    save_file(out, fn)
    return fn


def _rows_of(model: Sigusun, name: str, n: int, rows: int) -> list[int]:
    """Row counts of the ``n`` checkpoint tensors stacked in parameter ``name``."""
    if n == 1:
        return [rows]
    layer = model.layers[int(name.split(".")[1])]
    if name.endswith("wx.weight"):
        return layer.wx.splits
    if name.endswith("wkv"):
        a = layer.spec.lat
        return [a.heads * a.dim, a.heads * a.vdim]
    return [rows // n] * n


# ------------------------------------------------------------------ presets
def _stack(n: int, heads: int, dim: int, rot: int, rank: int, window: int, moe: MoeShape, base: float) -> tuple:
    """n layers in fours: causal latent attention with a sink, retention, windowed latent attention, and the
    same on the latter's latent."""
    ret = RetentionShape(heads, dim, dim, dim)
    decay = tuple(1 - 2.0 ** (-5 - 7 * j / max(heads - 1, 1)) for j in range(heads))

    def layer(i: int) -> LayerSpec:
        if i % 4 == 1:
            return LayerSpec(base, ret=ret, decay=decay, moe=moe)
        lat = LatentShape(heads, dim, rot, dim, rank, 1.0 / math.sqrt(dim + rot), window if i % 4 else 0)
        return LayerSpec(base, lat=lat, sink=i % 4 == 0, kv_from=i - 1 if i % 4 == 3 else None, moe=moe)

    return tuple(layer(i) for i in range(n))


PRESETS["sigusun-tiny"] = SigusunConfig("sigusun-tiny", 320, 64, _stack(4, 4, 16, 8, 32, 20, MoeShape(4, 2, 40, 4.0, 56, 3.0), 1e4),
                                        side_dim=16)
# width, depth, heads and feed-forward parameters of the Llama presets of the same name
PRESETS["sigusun-1b"] = SigusunConfig("sigusun-1b", 128256, 2048,
                                      _stack(16, 32, 64, 32, 256, 1024, MoeShape(16, 4, 384, 7.0, 2048, 7.0), 5e5), side_dim=64)
PRESETS["sigusun-8b"] = SigusunConfig("sigusun-8b", 128256, 4096,
                                      _stack(32, 32, 128, 64, 512, 1024, MoeShape(16, 4, 768, 7.0, 2048, 7.0), 5e5), side_dim=64)
