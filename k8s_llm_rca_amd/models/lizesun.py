"""Lizesun decoder: pre-normed sublayers over an fp32 residual with the Dynamic Tanh norm
(``tanh(alpha x) w + b``: no statistics), three kinds of mixer and a dense squared-ReLU feed-forward.

    x <- x + mixer(dyt1(x));   x <- x + down(relu(up(dyt2(x)))^2)      # the second when the layer has a feed-forward

``attention``:     q / k / v with biases, RMS norm (plain weight) on every q and k head, no positions in the
                   scores, ``s = softcap tanh(scale q.k / softcap)``, a CHUNKED causal mask (i sees j <= i of its own
                   chunk of ``mask.size`` positions), values mixed with the first such layer's values of the same
                   token (``(1 - lam) v + lam v_first``, the mixed values are cached), one sigmoid gate per head.
``parallel``:      ``left_scale * left + right_scale * right`` of two mixers reading the same input:
                   left  -- rotary q / k (rotate-half pairs on the first ``rot.dims`` entries), then q and k divided
                            by their root mean square, sliding window that also keeps the sequence's first
                            ``mask.keep_first`` tokens, a learned sink per head in the softmax's denominator;
                   right -- a matrix memory with exponential input / forget gates (soft-capped, stabilised by a
                            running maximum), normaliser state, per-head unit norm, sigmoid gate.
``channel_delta``: short causal convolution + SiLU on q, k, v; unit-length q / k; the gated delta rule with one
                   decay per head and key channel (low-rank projection, softplus step size); per-head unit norm,
                   low-rank sigmoid gate.
Output:            the final Dynamic Tanh norm, then the head.

What a sequence carries from step to step: keys and values of the attention layers in cache pages
(:class:`~..engine.kv_cache.WindowKVPool`), and in its state slot the convolution tails, delta-rule states and
matrix memories with their normalisers and maxima (fp32).  Every size and every constant that can differ
between checkpoints comes from the configuration or from a tensor's shape.
"""
from __future__ import annotations

import json
import math
import os
from dataclasses import dataclass
from typing import Dict, List, Optional, Tuple

import torch

from ..ops import norm as N
from ..ops import row_step as R
from ..ops import seq_ops as S
from ..ops.linear import proj_f32out
from ..parallel.groups import ParallelContext, single


@dataclass(frozen=True)
class ChunkAttnSpec:
    heads: int
    kv_heads: int
    dim: int
    vdim: int
    chunk: int              # 0: plain causal
    scale: float
    softcap: float = 0.0    # 0: scores are not capped
    v_mix: bool = False


@dataclass(frozen=True)
class WindowSinkSpec:
    heads: int
    kv_heads: int
    dim: int
    vdim: int
    window: int             # 0: plain causal
    keep_first: int
    scale: float
    rot_dims: int = 0       # 0: no rotation
    rot_base: float = 10000.0


@dataclass(frozen=True)
class MemorySpec:
    heads: int
    dim: int
    vdim: int
    gate_cap: float


@dataclass(frozen=True)
class DeltaSpec:
    heads: int
    kv_heads: int
    dim: int
    vdim: int
    conv: int
    # ranks of the decay's and the gate's low-rank projections: a checkpoint's tensors give them
    # (config.json does not); these are what random initialisation uses
    a_rank: int = 16
    g_rank: int = 16


@dataclass(frozen=True)
class LayerSpec:
    kind: str                               # 'attention' | 'parallel' | 'channel_delta'
    attn: Optional[ChunkAttnSpec] = None
    left: Optional[WindowSinkSpec] = None
    right: Optional[MemorySpec] = None
    delta: Optional[DeltaSpec] = None
    left_scale: float = 1.0
    right_scale: float = 1.0
    ff: int = 0                             # 0: no feed-forward


@dataclass(frozen=True)
class LizesunConfig:
    name: str
    vocab_size: int
    hidden: int
    layers: Tuple[LayerSpec, ...]
    norm_eps: float = 1e-5
    embed_scale: float = 1.0
    max_position: int = 1 << 20    # no tabulated positions: any length the cache holds
    arch: str = "lizesun"

    @property
    def n_layers(self) -> int:
        return len(self.layers)

    @classmethod
    def from_json(cls, d: dict, name: str = "lizesun") -> "LizesunConfig":
        layers = []
        for L in d["layers"]:
            m = L.get("mixer") or {}
            f = L.get("mlp")
            ff = 0
            if f is not None:
                if f.get("kind", "dense") != "dense":
                    raise ValueError(f"unknown feed-forward kind {f.get('kind')!r}")
                ff = int(f["ff"])
            kind = L["type"]
            if kind == "attention":
                layers.append(LayerSpec(kind, attn=ChunkAttnSpec(
                    int(m["heads"]), int(m.get("kv_heads", m["heads"])), int(m["dim"]), int(m.get("vdim", m["dim"])),
                    int((m.get("mask") or {}).get("size", 0)), float(m["scale"]), float(m.get("softcap") or 0.0),
                    bool(m.get("v_mix", False))), ff=ff))
            elif kind == "parallel":
                a, b = m["left"], m["right"]
                mask, rot = a.get("mask") or {}, a.get("rot") or {}
                layers.append(LayerSpec(
                    kind,
                    left=WindowSinkSpec(int(a["heads"]), int(a.get("kv_heads", a["heads"])), int(a["dim"]),
                                        int(a.get("vdim", a["dim"])), int(mask.get("size", 0)),
                                        int(mask.get("keep_first", 0)), float(a["scale"]), int(rot.get("dims", 0)),
                                        float(rot.get("base", 10000.0))),
                    right=MemorySpec(int(b["heads"]), int(b["dim"]), int(b.get("vdim", b["dim"])),
                                     float(b["gate_cap"])),
                    left_scale=float(m.get("left_scale", 1.0)), right_scale=float(m.get("right_scale", 1.0)), ff=ff))
            elif kind == "channel_delta":
                layers.append(LayerSpec(kind, delta=DeltaSpec(
                    int(m["heads"]), int(m.get("kv_heads", m["heads"])), int(m["dim"]), int(m.get("vdim", m["dim"])),
                    int(m.get("conv", 1)), int(m.get("a_rank", 16)), int(m.get("g_rank", 16))), ff=ff))
            else:
                raise ValueError(f"unknown mixer type {kind!r}")
        return cls(name, int(d["vocab"]), int(d["width"]), tuple(layers), norm_eps=float(d["norm"]["eps"]),
                   embed_scale=float((d.get("embedding") or {}).get("scale", 1.0)))

    def to_json(self) -> dict:
        layers = []
        for L in self.layers:
            if L.kind == "attention":
                a = L.attn
                m = {"heads": a.heads, "kv_heads": a.kv_heads, "dim": a.dim, "vdim": a.vdim, "scale": a.scale,
                     "v_mix": a.v_mix}
                if a.chunk:
                    m["mask"] = {"size": a.chunk}
                if a.softcap:
                    m["softcap"] = a.softcap
            elif L.kind == "parallel":
                a, b = L.left, L.right
                left = {"heads": a.heads, "kv_heads": a.kv_heads, "dim": a.dim, "vdim": a.vdim, "scale": a.scale}
                if a.window:
                    left["mask"] = {"size": a.window, "keep_first": a.keep_first}
                if a.rot_dims:
                    left["rot"] = {"dims": a.rot_dims, "base": a.rot_base}
                m = {"left": left, "right": {"heads": b.heads, "dim": b.dim, "vdim": b.vdim, "gate_cap": b.gate_cap},
                     "left_scale": L.left_scale, "right_scale": L.right_scale}
            else:
                c = L.delta
                m = {"heads": c.heads, "kv_heads": c.kv_heads, "dim": c.dim, "vdim": c.vdim, "conv": c.conv,
                     "a_rank": c.a_rank, "g_rank": c.g_rank}
            layers.append({"type": L.kind, "mixer": m, "mlp": {"kind": "dense", "ff": L.ff} if L.ff else None})
        return {"architecture": "Lizesun", "vocab": self.vocab_size, "width": self.hidden,
                "embedding": {"scale": self.embed_scale}, "layers": layers, "norm": {"eps": self.norm_eps}}


def _stack(n_groups: int, W: int, heads: int, kv_heads: int, dim: int, chunk: int, window: int, ff: int):
    """Groups of (attention, parallel, channel_delta, attention), every layer with a feed-forward."""
    att = LayerSpec("attention", attn=ChunkAttnSpec(heads, kv_heads, dim, dim, chunk, 1.0 / math.sqrt(dim), 30.0,
                                                    True), ff=ff)
    par = LayerSpec("parallel",
                    left=WindowSinkSpec(heads, kv_heads, dim, dim, window, 4, 1.0 / math.sqrt(dim) * 8.0, dim // 2,
                                        50000.0),
                    right=MemorySpec(heads, dim // 2, dim, 15.0), left_scale=0.7, right_scale=0.9, ff=ff)
    dlt = LayerSpec("channel_delta", delta=DeltaSpec(heads, kv_heads, dim // 2, dim, 4, max(8, W // 32),
                                                     max(8, W // 32)), ff=ff)
    return tuple([att, par, dlt, att] * n_groups)


PRESETS: Dict[str, LizesunConfig] = {
    "tiny-lizesun": LizesunConfig("tiny-lizesun", 8192, 256, _stack(1, 256, 4, 2, 32, 40, 24, 512), embed_scale=4.0),
    # sizes of a ~1B-class decoder's layers (benchmarks; random weights)
    "lizesun-1b": LizesunConfig("lizesun-1b", 32768, 2048, _stack(3, 2048, 16, 2, 128, 1024, 1024, 8192),
                                embed_scale=8.0),
}


class LizesunModel:
    stateful = True            # per-sequence state slots besides cache pages: no rewinding, no page sharing
    step_layout = "segments"   # the engine packs steps as segments (ops.seq_ops.SegStepInputs)
    graph_capturable = False
    segment_graphs = True      # steps of single tokens replay HIP graphs (engine/graph_runner.py)
    loads = 0                  # times weights were loaded: a graph reads those it was captured with

    def __init__(self, cfg: LizesunConfig, device, dtype=torch.bfloat16, pc: Optional[ParallelContext] = None,
                 seed: int = 0, init: bool = True):
        self.cfg = cfg
        self.device = torch.device(device)
        if dtype not in (torch.bfloat16, torch.float32):
            raise ValueError("Lizesun runs in bfloat16 or float32")
        self.dtype = dtype
        self.pc = pc or single()
        if self.pc.tp_size != 1:
            raise ValueError("Lizesun runs on one device per replica (no tensor-parallel sharding of its mixers)")
        self.logits_f32 = True
        self.layers: List[Dict[str, object]] = []
        # layer -> index of its key / value pages, of its delta-rule state, of its matrix memory
        self.cache_of: List[Optional[int]] = []
        self.cache_dims: List[Tuple[int, int, int, int]] = []     # (H, G, D, V) per attention
        self.delta_of: List[Optional[int]] = []
        self.mem_of: List[Optional[int]] = []
        self.vmix_first: Optional[int] = None                     # the first layer that mixes values
        self.ropes: Dict[Tuple[int, float], S.Rope] = {}          # every distinct rotation of the stack
        n_delta = n_mem = 0
        vmix_width = None
        for i, L in enumerate(cfg.layers):
            a = L.attn if L.kind == "attention" else L.left
            if a is not None:
                if a.heads % a.kv_heads:
                    raise ValueError(f"layer {i}: heads must be a multiple of kv_heads")
                self.cache_of.append(len(self.cache_dims))
                self.cache_dims.append((a.heads, a.kv_heads, a.dim, a.vdim))
            else:
                self.cache_of.append(None)
            if L.kind == "attention" and a.v_mix:
                if self.vmix_first is None:
                    self.vmix_first, vmix_width = i, (a.kv_heads, a.vdim)
                elif (a.kv_heads, a.vdim) != vmix_width:
                    raise ValueError(f"layer {i}: layers that mix values must have values of one size")
            if L.kind == "parallel":
                if L.left.rot_dims % 2 or L.left.rot_dims > L.left.dim:
                    raise ValueError(f"layer {i}: an even rot.dims <= dim")
                key = (L.left.rot_dims, L.left.rot_base)
                if key[0] and key not in self.ropes:
                    self.ropes[key] = S.make_rope(*key, self.device)
                self.mem_of.append(n_mem)
                n_mem += 1
            else:
                self.mem_of.append(None)
            if L.kind == "channel_delta":
                c = L.delta
                if c.heads % c.kv_heads or not 1 <= c.conv <= 16:
                    raise ValueError(f"layer {i}: heads must be a multiple of kv_heads, conv 1..16")
                self.delta_of.append(n_delta)
                n_delta += 1
            else:
                self.delta_of.append(None)
        if init:
            self._random_init(seed)

    # ------------------------------------------------------- what the engine allocates for this model
    def _twins(self) -> List[bool]:
        """Per attention: whether the matrix-core kernel runs it (then its values are also cached transposed)."""
        return [S.masked_mfma_ok(H, G, D, V, self.dtype, self.device) for H, G, D, V in self.cache_dims]

    def _widths(self) -> List[Tuple[int, int]]:
        return [(G * D, G * V) for _, G, D, V in self.cache_dims]

    def cache_bytes_per_block(self, block_size: int) -> int:
        per = sum(a + (2 * b if tw else b) for (a, b), tw in zip(self._widths(), self._twins()))
        return max(1, per) * block_size * (2 if self.dtype == torch.bfloat16 else 4)

    def make_cache(self, num_blocks: int, block_size: int):
        from ..engine.kv_cache import WindowKVPool
        return WindowKVPool(self._widths(), num_blocks, block_size, self.device, self.dtype, self._twins())

    def state_spec(self) -> Dict[str, Tuple[int, ...]]:
        """Per-slot fp32 state tensors: name -> shape behind the slot dimension."""
        spec: Dict[str, Tuple[int, ...]] = {}
        for i, L in enumerate(self.cfg.layers):
            if L.kind == "channel_delta":
                j, c = self.delta_of[i], L.delta
                spec[f"dconv{j}"] = (c.conv - 1, 2 * c.kv_heads * c.dim + c.heads * c.vdim)
                spec[f"delta{j}"] = (c.heads, c.dim, c.vdim)
            elif L.kind == "parallel":
                j, b = self.mem_of[i], L.right
                spec[f"mem{j}"] = (b.heads, b.dim, b.vdim)
                spec[f"memn{j}"] = (b.heads, b.dim)
                spec[f"memm{j}"] = (b.heads,)
        return spec

    def workspace_bytes(self, tokens: int) -> int:
        w = self.cfg.hidden
        widest = w
        for L in self.cfg.layers:
            for a in (L.attn, L.left):
                if a is not None:
                    widest = max(widest, 2 * (a.heads * (a.dim + a.vdim) + a.kv_heads * (a.dim + a.vdim)))
            if L.right is not None:
                widest = max(widest, 3 * L.right.heads * (L.right.dim + L.right.vdim))
            if L.delta is not None:
                widest = max(widest, 3 * L.delta.heads * (L.delta.dim + L.delta.vdim))
            widest = max(widest, 2 * L.ff)
        return int(tokens * (3 * w * 4 + widest * 8) + (2 << 30))

    # --------------------------------------------------------------- weights
    def _random_init(self, seed: int) -> None:
        t = random_tensors(self.cfg, seed, self.device)
        self.load_tensors(t.__getitem__)

    def load_tensors(self, get, has=None) -> None:
        """Build the fused device layout from checkpoint tensors (``get(name)`` -> tensor; names of the
        safetensors file: ``embed``, ``l<i>.norm1``, ``l<i>.mix.left.q`` ...)."""
        cfg, dev, dt = self.cfg, self.device, self.dtype
        self.loads += 1

        def put(*names, dtype=dt):
            ts = [get(n) for n in names]
            t = ts[0] if len(ts) == 1 else torch.cat([x.reshape(x.shape[0], -1) if x.dim() > 1 else x for x in ts], 0)
            return t.to(device=dev, dtype=dtype).contiguous()

        def f32(*names):
            return put(*names, dtype=torch.float32)

        def norm(name):   # (alpha, w, b)
            return float(get(name + ".alpha").float().item()), f32(name), f32(name + ".b")

        self.embed = put("embed")
        self.final_norm = norm("final.norm")
        self.lm_head = put("head")
        self.layers = []
        for i, spec in enumerate(cfg.layers):
            p = f"l{i}.mix."
            L: Dict[str, object] = {"norm1": norm(f"l{i}.norm1")}
            if spec.kind == "attention":
                a = spec.attn
                L["w_in"] = put(p + "q", p + "k", p + "v", p + "g")            # one fp32-out GEMM: q | k | v | gate
                L["bias"] = f32(p + "q.b", p + "k.b", p + "v.b")
                L["q_w"], L["k_w"] = f32(p + "q.norm"), f32(p + "k.norm")
                L["lam"] = float(get(p + "vmix").float().item()) if a.v_mix and i != self.vmix_first else 0.0
                L["wo"] = put(p + "o")
            elif spec.kind == "parallel":
                a, b = p + "left.", p + "right."
                L["w_in"] = put(a + "q", a + "k", a + "v", b + "q", b + "k", b + "v", b + "g", b + "i", b + "f")
                L["sink"] = f32(a + "sink")
                L["wo_l"] = put(a + "o")
                L["gate_bias"] = f32(b + "i.b", b + "f.b")
                L["mem_norm"] = f32(b + "norm")
                L["wo_r"] = put(b + "o")
            else:
                # q | k | v, then the inputs of the decays and of the gate, beta (fp32 out)
                L["w_in"] = put(p + "q", p + "k", p + "v", p + "a1", p + "g1", p + "b")
                L["conv_w"] = f32(p + "q.conv", p + "k.conv", p + "v.conv")
                L["w_a2"], L["w_g2"] = put(p + "a2"), put(p + "g2")
                L["rate"] = torch.exp(f32(p + "A_log")).contiguous()
                L["dt_bias"] = f32(p + "dt_bias")
                L["delta_norm"] = f32(p + "norm")
                L["wo"] = put(p + "o")
            if spec.ff:
                L["norm2"] = norm(f"l{i}.norm2")
                L["w_up"], L["w_down"] = put(f"l{i}.mlp.up"), put(f"l{i}.mlp.down")
            self.layers.append(L)

    def weight_bytes(self) -> int:
        def size(v):
            if isinstance(v, tuple):
                return sum(size(t) for t in v)
            return v.numel() * v.element_size() if isinstance(v, torch.Tensor) else 0
        n = sum(size(t) for L in self.layers for t in L.values())
        return n + sum(size(t) for t in (self.embed, self.lm_head, self.final_norm))

    # -------------------------------------------------------------- forward
    def _chunk_attention(self, li: int, h, inp: S.SegStepInputs, kcs, vcs, vts, vmix: dict) -> torch.Tensor:
        L, a = self.layers[li], self.cfg.layers[li].attn
        ci = self.cache_of[li]
        H, G, D, V = a.heads, a.kv_heads, a.dim, a.vdim
        keep = other = None
        if a.v_mix:
            if li == self.vmix_first:
                keep = vmix["v"] = torch.empty(inp.input_ids.shape[0], G * V, dtype=torch.float32, device=self.device)
            else:
                other = vmix["v"]
        n = H * D + G * (D + V)
        prep = dict(norm=True, q_w=L["q_w"], k_w=L["k_w"], eps=self.cfg.norm_eps, lam=L["lam"], v_other=other, v_keep=keep)
        made = S.proj_prep(h, L["w_in"], L["bias"], H, G, D, V, inp.slots, kcs[ci], vcs[ci], vts[ci], inp.seg, **prep)
        if made is not None:
            return S.masked_attention(made[0], H, G, D, V, kcs[ci], vcs[ci], inp.seg, a.scale, vt=vts[ci], softcap=a.softcap,
                                      chunk=a.chunk, gate=made[1])
        x = R.proj_f32out(h, L["w_in"])                                # [T, H D + G D + G V + H] fp32
        return S.prep_attention(x[:, :n], L["bias"], H, G, D, V, inp.positions, inp.slots, kcs[ci], vcs[ci], vts[ci], inp.seg,
                                self.dtype, a.scale, prep, dict(softcap=a.softcap, chunk=a.chunk, gate=x[:, n:]))

    def _parallel(self, li: int, h, inp: S.SegStepInputs, kcs, vcs, vts, states, tables: S.RopeTables):
        L, spec = self.layers[li], self.cfg.layers[li]
        a, b = spec.left, spec.right
        ci, j = self.cache_of[li], self.mem_of[li]
        H, G, D, V = a.heads, a.kv_heads, a.dim, a.vdim
        nl = H * D + G * (D + V)
        rope = self.ropes.get((a.rot_dims, a.rot_base))
        prep = dict(norm=True, eps=self.cfg.norm_eps, rope=rope, rope_cs=tables.of(rope))
        mask = dict(window=a.window, keep_first=a.keep_first, sink=L["sink"])
        made = S.proj_prep(h, L["w_in"], None, H, G, D, V, inp.slots, kcs[ci], vcs[ci], vts[ci], inp.seg, **prep)
        if made is not None:
            o = S.masked_attention(made[0], H, G, D, V, kcs[ci], vcs[ci], inp.seg, a.scale, vt=vts[ci], **mask)
            return o, S.memory_layer(made[1], b.heads, b.dim, b.vdim, L["gate_bias"], b.gate_cap, states[f"mem{j}"], states[f"memn{j}"],
                                     states[f"memm{j}"], inp.seg, L["mem_norm"], self.cfg.norm_eps, self.dtype)
        x = R.proj_f32out(h, L["w_in"])                                # left q | k | v, right q | k | v | g | i | f
        return S.attention_and_memory(x[:, :nl], H, G, D, V, inp.positions, inp.slots, kcs[ci], vcs[ci], vts[ci], inp.seg,
                                      self.dtype, a.scale, prep, mask, x[:, nl:], b.heads, b.dim, b.vdim, L["gate_bias"],
                                      b.gate_cap, states[f"mem{j}"], states[f"memn{j}"], states[f"memm{j}"], inp.seg,
                                      L["mem_norm"], self.cfg.norm_eps, self.dtype)

    def _delta(self, li: int, h, inp: S.SegStepInputs, states) -> torch.Tensor:
        L, c = self.layers[li], self.cfg.layers[li].delta
        j = self.delta_of[li]
        qkv, agb = R.conv_proj(h, L["w_in"], L["conv_w"], states[f"dconv{j}"], inp.seg)      # [T, 2 G D + H V], [T, ra + rg + H]
        return S.delta_low_rank(qkv, c.heads, c.kv_heads, c.dim, c.vdim, agb, L["w_a2"], L["w_g2"], L["rate"], L["dt_bias"],
                                states[f"delta{j}"], inp.seg, L["delta_norm"], self.cfg.norm_eps, self.dtype)

    def forward(self, inp: S.SegStepInputs, kcs: List[torch.Tensor], vcs: List[torch.Tensor],
                vts: List[Optional[torch.Tensor]], states: Dict[str, torch.Tensor],
                layers_out: Optional[list] = None, head: bool = True):
        """Logits [len(logits_idx), vocab] fp32.  ``kcs`` / ``vcs``: the paged keys and values of every
        attention (``vts``: the values' transposed twins, or None); ``states``: the per-slot tensors of
        :meth:`state_spec`.  ``layers_out`` (debugging): receives a copy of the residual after every layer.
        Without ``head``: what :meth:`logits` makes them of."""
        cfg, dt = self.cfg, self.dtype
        T, W, nl = inp.input_ids.shape[0], cfg.hidden, cfg.n_layers
        idx = S.wanted_rows(inp)
        few = nl > 0 and (idx is None or T <= R.INTO_ROWS)   # (few rows: the same products whichever of them are wanted)
        x = torch.empty(T, W, dtype=torch.float32, device=self.device)
        first = self.layers[0]["norm1"] if nl else (1.0, None, None)
        tables = S.RopeTables(inp.positions, self.ropes.values())      # cos | sin of the step's positions, made once
        h = N.embed_scale_dyt(inp.input_ids, self.embed, cfg.embed_scale, x, *first, out_dtype=dt, tables=tables)
        vmix: dict = {}
        for li, (spec, L) in enumerate(zip(cfg.layers, self.layers)):
            # (the final norm reads the wanted rows only, or with the last layer where every row is wanted or there are few)
            nxt = self.layers[li + 1]["norm1"] if li + 1 < nl else self.final_norm if few else (1.0, None, None)
            after = L["norm2"] if spec.ff else nxt
            if spec.kind == "parallel":
                ol, orr = self._parallel(li, h, inp, kcs, vcs, vts, states, tables)
                x = R.residual(h, x)
                h = R.dyt_product(x, ol, L["wo_l"], spec.left_scale, orr, L["wo_r"], spec.right_scale, *after, out_dtype=dt)
            else:
                o = (self._chunk_attention(li, h, inp, kcs, vcs, vts, vmix) if spec.kind == "attention"
                     else self._delta(li, h, inp, states))
                x = R.residual(h, x)
                h = R.dyt_product(x, o, L["wo"], 1.0, None, None, 1.0, *after, out_dtype=dt)
            if spec.ff:
                u = R.relu_sq_proj(h, L["w_up"])
                x = R.residual(h, x)
                h = R.dyt_product(x, u, L["w_down"], 1.0, None, None, 1.0, *nxt, out_dtype=dt)
            if layers_out is not None:
                if isinstance(h, R.RowStep):
                    h = h.read()                                       # the residual as it is behind this layer
                layers_out.append(x.clone())
        if few:
            h = R.rows(h, idx)
        else:
            xr = x.index_select(0, idx).contiguous() if idx is not None else x
            h = N.add_dyt(xr, None, 1.0, None, 1.0, *self.final_norm, out_dtype=dt)
        return self.logits(h) if head else h

    def logits(self, h) -> torch.Tensor:
        return R.proj_f32out(h, self.lm_head)


def random_tensors(cfg: LizesunConfig, seed: int = 0, device="cpu") -> Dict[str, torch.Tensor]:
    """Seeded random weights under the checkpoint's names, bfloat16 (so a bfloat16 and a float32 model
    built from them hold the same numbers)."""
    dev = torch.device(device)
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    W = cfg.hidden

    def rnd(*shape, std=0.02, mean=0.0):
        return torch.empty(*shape, dtype=torch.float32, device=dev).normal_(mean, std, generator=g).to(torch.bfloat16)

    def lin(n_out, n_in, gain=1.0):
        return rnd(n_out, n_in, std=gain / math.sqrt(n_in))

    t: Dict[str, torch.Tensor] = {"embed": rnd(cfg.vocab_size, W, std=1.0 / max(cfg.embed_scale, 1e-6)),
                                  "head": lin(cfg.vocab_size, W)}

    def norm(name):
        t[name] = rnd(W, std=0.1, mean=1.0)
        t[name + ".b"] = rnd(W, std=0.05)
        t[name + ".alpha"] = rnd((), std=0.05, mean=0.7)

    norm("final.norm")
    for i, L in enumerate(cfg.layers):
        p = f"l{i}.mix."
        norm(f"l{i}.norm1")
        if L.kind == "attention":
            a = L.attn
            t[p + "q"], t[p + "k"] = lin(a.heads * a.dim, W), lin(a.kv_heads * a.dim, W)
            t[p + "v"], t[p + "o"] = lin(a.kv_heads * a.vdim, W), lin(W, a.heads * a.vdim)
            t[p + "q.b"], t[p + "k.b"] = rnd(a.heads * a.dim, std=0.1), rnd(a.kv_heads * a.dim, std=0.1)
            t[p + "v.b"] = rnd(a.kv_heads * a.vdim, std=0.1)
            t[p + "q.norm"], t[p + "k.norm"] = rnd(a.dim, std=0.2, mean=1.5), rnd(a.dim, std=0.2, mean=1.5)
            t[p + "vmix"] = rnd((), std=0.05, mean=0.3)
            t[p + "g"] = lin(a.heads, W)
        elif L.kind == "parallel":
            a, b = L.left, L.right
            q, m = p + "left.", p + "right."
            t[q + "q"], t[q + "k"] = lin(a.heads * a.dim, W), lin(a.kv_heads * a.dim, W)
            t[q + "v"], t[q + "o"] = lin(a.kv_heads * a.vdim, W), lin(W, a.heads * a.vdim)
            t[q + "sink"] = rnd(a.heads, std=1.0)
            t[m + "q"], t[m + "k"] = lin(b.heads * b.dim, W), lin(b.heads * b.dim, W)
            t[m + "v"], t[m + "g"] = lin(b.heads * b.vdim, W), lin(b.heads * b.vdim, W)
            t[m + "o"] = lin(W, b.heads * b.vdim)
            t[m + "norm"] = rnd(b.heads * b.vdim, std=0.1, mean=1.0)
            t[m + "i"], t[m + "f"] = lin(b.heads, W, 2.0), lin(b.heads, W, 2.0)
            t[m + "i.b"], t[m + "f.b"] = rnd(b.heads, std=0.5), rnd(b.heads, std=0.5, mean=2.0)
        else:
            c = L.delta
            t[p + "q"], t[p + "k"] = lin(c.kv_heads * c.dim, W), lin(c.kv_heads * c.dim, W)
            t[p + "v"], t[p + "o"] = lin(c.heads * c.vdim, W), lin(W, c.heads * c.vdim)
            for n_, ch in (("q", c.kv_heads * c.dim), ("k", c.kv_heads * c.dim), ("v", c.heads * c.vdim)):
                t[p + n_ + ".conv"] = rnd(ch, c.conv, std=0.5)
            t[p + "b"] = lin(c.heads, W)
            t[p + "A_log"] = rnd(c.heads, std=0.5, mean=-1.0)
            t[p + "norm"] = rnd(c.vdim, std=0.1, mean=1.0)
            t[p + "a1"], t[p + "a2"] = lin(c.a_rank, W), lin(c.heads * c.dim, c.a_rank)
            t[p + "dt_bias"] = rnd(c.heads * c.dim, std=0.5, mean=-1.0)
            t[p + "g1"], t[p + "g2"] = lin(c.g_rank, W), lin(c.heads * c.vdim, c.g_rank)
        if L.ff:
            norm(f"l{i}.norm2")
            t[f"l{i}.mlp.up"], t[f"l{i}.mlp.down"] = lin(L.ff, W), lin(W, L.ff, 0.5)
    return t


def load_checkpoint(path: str, device, dtype, pc=None) -> LizesunModel:
    """A folder with config.json and model.safetensors (bfloat16 weights) -> the model on ``device``."""
    from safetensors import safe_open
    with open(os.path.join(path, "config.json")) as f:
        cfg = LizesunConfig.from_json(json.load(f), name=os.path.basename(os.path.normpath(path)) or "lizesun")
    model = LizesunModel(cfg, device, dtype, pc, init=False)
    with safe_open(os.path.join(path, "model.safetensors"), framework="pt", device="cpu") as h:
        model.load_tensors(h.get_tensor, set(h.keys()).__contains__)
    return model


def save_checkpoint(cfg: LizesunConfig, tensors: Dict[str, torch.Tensor], path: str) -> None:
    """Write config.json + model.safetensors (bfloat16) in the layout :func:`load_checkpoint` reads."""
    from safetensors.torch import save_file
    os.makedirs(path, exist_ok=True)
    with open(os.path.join(path, "config.json"), "w") as f:
        json.dump(cfg.to_json(), f, indent=1)
    save_file({k: v.to(torch.bfloat16).contiguous() for k, v in tensors.items()},
              os.path.join(path, "model.safetensors"))
