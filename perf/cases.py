"""The work that is timed: engine steps with given tokens (``LLMEngine.feed``), as a replayed conversation.

One pass is what a request costs a user: new sequences are opened, each turn's prompt is fed as one portion, its reply is fed
token by token, and the sequences are released.  Logits come back as a recorded schedule asks for them: of eight tokens
spread over every portion, its last among them, and of every reply token.

Three models, which between them hold the framework's kinds of token mixer at the presets' own sizes:

* ``llama3-8b``  -- the backend of the headline benchmark: full attention over paged keys and values, dense gated unit;
* ``fikerax-1b`` -- linear attention with a fixed decay, windowed attention, windowed latent attention, repeated layers;
* ``lizesun-1b`` -- chunked and windowed attention with a sink, a matrix memory, the gated delta rule, squared ReLU.
"""
import math
import random
from dataclasses import replace

import torch

from k8s_llm_rca_amd.engine.engine import EngineConfig, LLMEngine
from k8s_llm_rca_amd.models import fikerax, lizesun
from k8s_llm_rca_amd.models.llama import LlamaModel
from k8s_llm_rca_amd.models.registry import get_any_config

BLOCK = 64
WANTED = 8      # rows of a portion whose logits come back
F64 = torch.float64
#: tokens of one portion over all sequences, at most
MOST_TOKENS = {"llama3-8b": 8192, "fikerax-1b": 32768, "lizesun-1b": 32768}


def _overrides(model):
    """What differs from the preset.  The layers of a model repeat, so a part of them is timed: through more of them random
    weights turn bfloat16's rounding into differences in which a wrong result would not be seen (relative error against
    64 bits through 4 / 8 / 32 layers of llama3-8b: 2.0e-2 / 2.8e-2 / 4.7e-2)."""
    cfg = get_any_config(model)
    if model == "llama3-8b":
        return {"n_layers": 4}
    if model == "lizesun-1b":
        return {"layers": cfg.layers[:8]}
    # unit-size heads times the preset's scale make scores of some hundreds, as no trained weights do: every softmax would
    # pick one key, and another one after each change of rounding
    return {"layers": tuple(replace(L, mix=replace(L.mix, scale=L.mix.dim ** -0.5)) if L.kind == "attention" else L
                            for L in cfg.layers)}


def _config(case):
    return get_any_config(case["model"], **_overrides(case["model"]))


def _case(model, batch, prompt, turns, steps, dtype="bfloat16"):
    return {"model": model, "batch": batch, "prompt": prompt, "turns": turns, "steps": steps, "dtype": dtype}


def listed():
    return [
        # one operator's question to an idle server: a short prompt, then token after token (latency, launches)
        {"name": "llama-question", **_case("llama3-8b", 1, 100, 1, 12)},
        # many pipelines at once, prompts of different lengths, then a shared reply
        {"name": "llama-threads", **_case("llama3-8b", 16, 450, 1, 8)},
        # reading long event logs, one token of an answer
        {"name": "llama-logs", **_case("llama3-8b", 2, 4000, 1, 1)},
        # the smallest call: a few words and a few tokens back
        {"name": "fikerax-question", **_case("fikerax-1b", 1, 17, 1, 12)},
        # a handful of threads that go on for a second turn, odd lengths
        {"name": "fikerax-threads", **_case("fikerax-1b", 7, 701, 2, 8)},
        # the throughput benchmark's prompts, and its largest batch with a reply
        {"name": "fikerax-prompts", **_case("fikerax-1b", 8, 2048, 1, 1)},
        {"name": "fikerax-batch", **_case("fikerax-1b", 64, 512, 1, 8)},
        # a recorded schedule replayed in float32 to look into a difference
        {"name": "fikerax-replay-f32", **_case("fikerax-1b", 2, 333, 1, 4, "float32")},
        # the same uses of the recurrent design
        {"name": "lizesun-question", **_case("lizesun-1b", 1, 40, 1, 12)},
        {"name": "lizesun-threads", **_case("lizesun-1b", 5, 1100, 2, 8)},
        {"name": "lizesun-prompts", **_case("lizesun-1b", 8, 2048, 1, 1)},
        {"name": "lizesun-batch", **_case("lizesun-1b", 64, 512, 1, 8)},
    ]


def draw(rng):
    model = rng.choice(sorted(MOST_TOKENS))
    dtype = "float32" if model == "fikerax-1b" and rng.random() < 0.2 else "bfloat16"
    most = 1024 if dtype == "float32" else MOST_TOKENS[model]

    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    batch = spread(1, min(64, most // 64))
    prompt = min(spread(16, 4096), most // batch)
    turns = 2 if rng.random() < 0.3 and prompt <= 2048 else 1
    return _case(model, batch, prompt, turns, rng.randint(0, 12), dtype)


def _portions(case):
    """[turn][sequence] -> tokens of the prompt portion: the longest has ``prompt``, the others down to half of that (a batch
    of prompts with at most one reply token: all the same, as the throughput benchmark has them)."""
    r = random.Random(case["prompt"] * 64 + case["batch"])
    n, b = case["prompt"], case["batch"]
    return [[n] + [n if case["steps"] <= 1 else r.randint(max(1, n // 2), n) for _ in range(b - 1)] for _ in range(case["turns"])]


def _tokens(case, seed):
    """[sequence] -> all its tokens: portion, reply, portion, reply ..."""
    vocab = get_any_config(case["model"]).vocab_size
    r = random.Random(seed)
    return [[r.randrange(vocab) for _ in range(sum(t[i] + case["steps"] for t in _portions(case)))]
            for i in range(case["batch"])]


def _wanted(n):
    """Offsets of the wanted rows of a portion of n >= WANTED tokens."""
    return [n * (k + 1) // WANTED - 1 for k in range(WANTED)]


def prepare(case, seed):
    portions, tokens = _portions(case), _tokens(case, seed)
    blocks = sum(-(-len(t) // BLOCK) + 1 for t in tokens)
    engine = LLMEngine(EngineConfig(model=case["model"], model_overrides=_overrides(case["model"]), device="cuda",
                                    dtype=getattr(torch, case["dtype"]), seed=seed, num_blocks=blocks + 16, block_size=BLOCK,
                                    max_context=8192, state_slots=case["batch"]))
    return {"engine": engine, "tokens": tokens, "portions": portions, "steps": case["steps"]}


def run(state):
    engine, tokens, turns = state["engine"], state["tokens"], len(state["portions"])
    sids = [engine.new_sequence() for _ in tokens]
    at = [0] * len(sids)
    # what feed() returns may be the next feed's buffer too, so that it is copied out
    read = torch.empty(turns, len(sids) * WANTED, engine.mc.vocab_size, device="cuda")
    said = torch.empty(turns, state["steps"], len(sids), engine.mc.vocab_size, device="cuda")
    for turn, portion in enumerate(state["portions"]):
        read[turn].copy_(engine.feed([(s, t[a:a + n], _wanted(n)) for s, t, a, n in zip(sids, tokens, at, portion)]))
        at = [a + n for a, n in zip(at, portion)]
        for step in range(state["steps"]):
            said[turn, step].copy_(engine.feed([(s, [t[a]], [0]) for s, t, a in zip(sids, tokens, at)]))
            at = [a + 1 for a in at]
    for s in sids:
        engine.release_sequence(s)
    return {"read": read, "said": said}


def _cost(cfg):
    """(numbers in the layers' matrices, multiply-adds of a token through them, the attentions' (heads, multiply-adds of a
    query and a key, window, cached numbers of a token), the recurrent states' sizes) -- the last two per layer run."""
    W, once, attn, state = cfg.hidden, 0, [], []
    if cfg.arch == "llama":
        once = cfg.n_layers * (2 * W * cfg.q_size + 2 * W * cfg.kv_size + 3 * W * cfg.intermediate)
        return once, once, [(cfg.n_heads, 2 * cfg.head_dim, 0, 2 * cfg.kv_size)] * cfg.n_layers, []
    sizes = []
    if cfg.arch == "fikerax":
        for L in cfg.layers:
            c = L.mix
            if L.kind == "lightning":
                n = W * c.heads * (2 * c.dim + 3 * c.vdim)
            elif L.kind == "attention":
                n = W * (c.heads + c.kv_heads) * (c.dim + c.vdim)
            else:
                n = W * (c.q_rank + c.kv_rank + c.rot_dim + c.heads * c.vdim) + c.heads * (
                    c.q_rank * (c.dim + c.rot_dim) + c.kv_rank * (c.dim + c.vdim))
            sizes.append(n + 3 * W * L.ff)
        for i, _ in cfg.runs:
            L, c = cfg.layers[i], cfg.layers[i].mix
            if L.kind == "lightning":
                state.append(c.heads * c.dim * c.vdim)
            elif L.kind == "attention":
                attn.append((c.heads, c.dim + c.vdim, c.window, c.kv_heads * (c.dim + c.vdim)))
            else:
                attn.append((c.heads, 2 * c.kv_rank + c.rot_dim, c.window, c.kv_rank + c.rot_dim))
        return sum(sizes), sum(sizes[i] for i, _ in cfg.runs), attn, state
    for L in cfg.layers:
        a = L.attn or L.left
        n = 2 * W * L.ff
        if a is not None:
            n += W * (a.heads + a.kv_heads) * (a.dim + a.vdim)
            attn.append((a.heads, a.dim + a.vdim, L.attn.chunk if L.attn else a.window, a.kv_heads * (a.dim + a.vdim)))
        if L.right is not None:
            b = L.right
            n += W * b.heads * (2 * b.dim + 3 * b.vdim)
            state.append(b.heads * b.dim * b.vdim)
        if L.delta is not None:
            c = L.delta
            n += W * (2 * c.kv_heads * c.dim + 2 * c.heads * c.vdim + c.a_rank + c.g_rank)
            n += c.a_rank * c.heads * c.dim + c.g_rank * c.heads * c.vdim
            state.append(c.heads * c.dim * c.vdim)
        once += n
    return once, once, attn, state


def work(case):
    """Every feed reads each matrix once (the reply's feeds follow one another), the keys and values its rows see and the
    states; multiply-adds count two operations."""
    cfg, B = _config(case), case["batch"]
    once, runs, attn, state = _cost(cfg)
    size = 4 if case["dtype"] == "float32" else 2
    head = cfg.vocab_size * cfg.hidden
    total = {"bytes": 0.0, "flops": 0.0}
    at = [0] * B
    for portion in _portions(case):
        for rows in [portion] + [[1] * B] * case["steps"]:
            wanted = B * (WANTED if rows is portion else 1)
            total["bytes"] += size * (once + head + sum(rows) * cfg.hidden) + 4 * wanted * cfg.vocab_size
            total["flops"] += 2.0 * (runs * sum(rows) + head * wanted)
            for heads, dims, window, cached in attn:
                for a, n in zip(at, rows):
                    if window:
                        pairs = sum(min(a + i + 1, window) for i in range(n))
                        seen = min(a, window)
                    else:
                        pairs, seen = n * a + n * (n + 1) / 2, a
                    total["flops"] += 2.0 * pairs * heads * dims
                    total["bytes"] += size * cached * (seen + n)
            total["bytes"] += sum(8.0 * B * s for s in state)
            total["flops"] += sum(4.0 * sum(rows) * s for s in state)
            at = [a + n for a, n in zip(at, rows)]
    return total


def tolerance(case):
    """About four times the differences from 64 bits that were measured (relative 2.0e-2, 3.3e-3, 1.1e-2 and, in float32,
    1.0e-6; of single logits 1.2e-1, 2.0e-2, 1.2e-1 and 6.5e-6), the two largest cut to 3e-2."""
    if case["dtype"] == "float32":
        return {"rel": 5e-6, "max": 5e-5}
    return {"llama3-8b": {"rel": 0.03, "max": 0.5}, "fikerax-1b": {"rel": 0.013, "max": 0.1},
            "lizesun-1b": {"rel": 0.03, "max": 0.5}}[case["model"]]


# ------------------------------------------------------------------------------------------ in 64 bits, plain torch
def _d(t):
    return t.to(F64)


def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _softmax_over(s, visible, sink=None):
    """Weights over the keys of scores [b, h, i, j]; a sink [h] is one more score without a value."""
    s = s.masked_fill_(~visible, -math.inf)
    m = s.amax(-1, keepdim=True)
    if sink is not None:
        m = torch.maximum(m, sink[None, :, None, None])
    e = s.sub_(m).exp_()
    z = e.sum(-1, keepdim=True)
    return e.div_(z if sink is None else z + torch.exp(sink[None, :, None, None] - m))


def _attend(q, k, v, scale, visible, sink=None, cap=0.0):
    """q [b, t, h, d], k and v [b, t, g, ...] -> [b, t, h * v], one sequence and key head at a time."""
    b, t, h, _ = q.shape
    g = k.shape[2]
    out = torch.empty(b, t, h, v.shape[-1], dtype=F64, device=q.device)
    for i in range(b):
        for j in range(g):
            hs = slice(j * (h // g), (j + 1) * (h // g))
            s = torch.matmul(q[i, :, hs].transpose(0, 1), k[i, :, j].T)[None] * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            p = _softmax_over(s, visible, None if sink is None else sink[hs])
            out[i, :, hs] = torch.matmul(p[0], v[i, :, j]).transpose(0, 1)
    return out.reshape(b, t, -1)


def _turn(x, freqs, amp=1.0, pairs=False):
    """x [b, t, h, d] with its first 2 len(freqs) entries turned: halves, or neighbours with ``pairs``."""
    n = len(freqs)
    f = torch.tensor(freqs, dtype=F64, device=x.device)
    a = torch.arange(x.shape[1], dtype=F64, device=x.device)[:, None] * f
    c, s = (a.cos() * amp)[None, :, None], (a.sin() * amp)[None, :, None]
    u, v = (x[..., 0:2 * n:2], x[..., 1:2 * n:2]) if pairs else (x[..., :n], x[..., n:2 * n])
    y = [u * c - v * s, v * c + u * s]
    y = torch.stack(y, -1).flatten(-2) if pairs else torch.cat(y, -1)
    return torch.cat([y, x[..., 2 * n:]], -1)


def _freqs(dims, base):
    return [base ** (-2.0 * i / dims) for i in range(dims // 2)]


def _llama(cfg, seed, ids):
    m = LlamaModel(cfg, "cuda", torch.bfloat16, seed=seed)          # the seeded random weights
    b, t = ids.shape
    H, G, D, I, eps = cfg.n_heads, cfg.n_kv_heads, cfg.head_dim, cfg.intermediate, cfg.rms_eps
    seen = torch.ones(t, t, dtype=torch.bool, device="cuda").tril()
    f = _freqs(D, cfg.rope_theta)
    x = _d(m.embed[ids])
    for L in m.layers:
        y = (_unit(x, eps) * _d(L["in_norm"])) @ _d(L["wqkv"]).T
        q, k, v = (z.view(b, t, -1, D) for z in y.split([H * D, G * D, G * D], -1))
        x = x + _attend(_turn(q, f), _turn(k, f), v, D ** -0.5, seen) @ _d(L["wo"]).T
        g, u = ((_unit(x, eps) * _d(L["post_norm"])) @ _d(L["w_gu"]).T).split(I, -1)
        x = x + (_silu(g).mul_(u)) @ _d(L["w_down"]).T
    return _unit(x, eps) * _d(m.final_norm), _d(m.lm_head)


def _stretched(dims, base, sc):
    out = []
    for f in _freqs(dims, base):
        factor, low, high, original = sc
        wave = 2.0 * math.pi / f
        if wave > original / low:
            f = f / factor
        elif wave >= original / high:
            s = (original / wave - low) / (high - low)
            f = (1.0 - s) * f / factor + s * f
        out.append(f)
    return out


def _yarn(dims, base, sc):
    factor, original, fast, slow = sc

    def pair(turns):
        return dims * math.log(original / (2.0 * math.pi * turns)) / (2.0 * math.log(base))

    lo, hi = max(math.floor(pair(fast)), 0), min(math.ceil(pair(slow)), dims - 1)
    out = []
    for i, f in enumerate(_freqs(dims, base)):
        r = min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0)
        out.append(f / factor * r + f * (1.0 - r))
    return out, 0.1 * math.log(factor) + 1.0


def _fikerax(cfg, seed, ids):
    w = {n: v for n, v in fikerax.random_tensors(cfg, seed, "cuda").items()}
    b, t = ids.shape
    eps, W = cfg.norm_eps, cfg.hidden
    far = torch.arange(t, device="cuda")[:, None] - torch.arange(t, device="cuda")[None]

    def lin(x, name):
        return x @ _d(w[name]).T

    def lightning(p, c, h):
        q, k = (_silu(lin(h, p + n)).view(b, t, c.heads, c.dim) for n in "qk")
        v = _silu(lin(h, p + "v")).view(b, t, c.heads, c.vdim)
        o = torch.empty_like(v)
        for j in range(c.heads):
            keep = torch.pow(torch.tensor(c.decay[j], dtype=torch.float32).item(), far.clamp_min(0).to(F64)).tril_()
            for i in range(b):
                o[i, :, j] = ((q[i, :, j] @ k[i, :, j].T) * keep) @ v[i, :, j]
        o = _unit(o.reshape(b, t, -1), eps) * _d(w[p + "norm"])
        return lin(o * torch.sigmoid(lin(h, p + "g")), p + "o")

    def attention(p, c, h):
        q, k, v = ((lin(h, p + n) + _d(w[p + n + ".b"])).view(b, t, -1, e) for n, e in (("q", c.dim), ("k", c.dim), ("v", c.vdim)))
        f = _stretched(c.rot_dims, c.rot_base, c.stretch)
        q, k = _unit(_turn(q, f), eps), _unit(_turn(k, f), eps)
        return lin(_attend(q, k, v, c.scale, (far >= 0) & (far < c.window)), p + "o")

    def latent(p, c, h):
        q = lin(_unit(lin(h, p + "dq"), eps) * _d(w[p + "dq.norm"]), p + "uq").view(b, t, c.heads, c.dim + c.rot_dim)
        kv = lin(h, p + "dkv")
        z = _unit(kv[..., :c.kv_rank], eps) * _d(w[p + "dkv.norm"])
        f, amp = _yarn(c.rot_dim, c.rot_base, c.yarn)
        kr = _turn(kv[:, :, None, c.kv_rank:], f, amp, True).expand(b, t, c.heads, c.rot_dim)
        q = torch.cat([q[..., :c.dim], _turn(q[..., c.dim:], f, amp, True)], -1)
        k = torch.cat([lin(z, p + "uk").view(b, t, c.heads, c.dim), kr], -1)
        v = lin(z, p + "uv").view(b, t, c.heads, c.vdim)
        return lin(_attend(q, k, v, c.scale, (far >= 0) & (far < c.window), _d(w[p + "sink"])), p + "o")

    kinds = {"lightning": lightning, "attention": attention, "latent_attention": latent}
    start = _d(w["embed"][ids]) * cfg.embed_scale
    x = start
    for i, again in cfg.runs:
        L = cfg.layers[i]
        x = x + start if again else x
        x = x + kinds[L.kind](f"l{i}.mix.", L.mix, _unit(x, eps) * (1.0 + _d(w[f"l{i}.norm1"])))
        if L.ff:
            h, p = _unit(x, eps) * (1.0 + _d(w[f"l{i}.norm2"])), f"l{i}.mlp."
            x = x + lin(_silu(lin(h, p + "gate")).mul_(lin(h, p + "up")), p + "down")
    return _unit(x, eps) * (1.0 + _d(w["final.norm"])), _d(w["head"])


def _lizesun(cfg, seed, ids):
    w = {n: v for n, v in lizesun.random_tensors(cfg, seed, "cuda").items()}
    b, t = ids.shape
    eps = cfg.norm_eps
    pos = torch.arange(t, device="cuda")
    far = pos[:, None] - pos[None]
    first = []

    def lin(x, name):
        return x @ _d(w[name]).T

    def dyt(x, name):
        return torch.tanh(_d(w[name + ".alpha"]) * x).mul_(_d(w[name])).add_(_d(w[name + ".b"]))

    def chunked(p, c, h):
        q, k, v = ((lin(h, p + n) + _d(w[p + n + ".b"])).view(b, t, -1, e) for n, e in (("q", c.dim), ("k", c.dim), ("v", c.vdim)))
        q, k = _unit(q, eps) * _d(w[p + "q.norm"]), _unit(k, eps) * _d(w[p + "k.norm"])
        if c.v_mix and not first:
            first.append(v)
        elif c.v_mix:
            lam = _d(w[p + "vmix"])
            v = (1.0 - lam) * v + lam * first[0]
        seen = (far >= 0) & (pos[:, None] // c.chunk == pos[None] // c.chunk)
        o = _attend(q, k, v, c.scale, seen, cap=c.softcap).view(b, t, c.heads, c.vdim)
        return lin((o * torch.sigmoid(lin(h, p + "g"))[..., None]).reshape(b, t, -1), p + "o")

    def window(p, c, h):
        f = _freqs(c.rot_dims, c.rot_base)
        q, k, v = (lin(h, p + n).view(b, t, -1, e) for n, e in (("q", c.dim), ("k", c.dim), ("v", c.vdim)))
        q, k = _unit(_turn(q, f), eps), _unit(_turn(k, f), eps)
        seen = (far >= 0) & ((far < c.window) | (pos[None] < c.keep_first))
        return lin(_attend(q, k, v, c.scale, seen, _d(w[p + "sink"])), p + "o")

    def memory(p, c, h):
        """The recurrence written out: row i weighs row j by exp(F_i - F_j + i_j - m_i), F the summed log forget gates."""
        q, k, v = (lin(h, p + n).view(b, t, c.heads, e) for n, e in (("q", c.dim), ("k", c.dim), ("v", c.vdim)))
        cap = c.gate_cap
        ig = cap * torch.tanh((lin(h, p + "i") + _d(w[p + "i.b"])) / cap)
        F = torch.nn.functional.logsigmoid(cap * torch.tanh((lin(h, p + "f") + _d(w[p + "f.b"])) / cap)).cumsum(1)
        m = F + torch.cummax(ig - F, 1)[0].clamp_min(0.0)
        o = torch.empty_like(v)
        for i in range(b):
            for j in range(c.heads):
                g = (F[i, :, j, None] - m[i, :, j, None] + (ig - F)[i, None, :, j]).masked_fill_(far < 0, -math.inf).exp_()
                s = (q[i, :, j] @ k[i, :, j].T).mul_(g) * c.dim ** -0.5
                o[i, :, j] = (s @ v[i, :, j]) / (torch.maximum(s.sum(1).abs(), torch.exp(-m[i, :, j])) + 1e-6)[:, None]
        o = _unit(o, eps).reshape(b, t, -1) * _d(w[p + "norm"]) * torch.sigmoid(lin(h, p + "g"))
        return lin(o, p + "o")

    def conv(x, taps):
        n = taps.shape[1]
        ext = torch.cat([torch.zeros(b, n - 1, x.shape[2], dtype=F64, device="cuda"), x], 1)
        return _silu(sum(taps[:, j] * ext[:, j:j + t] for j in range(n)))

    def delta(p, c, h):
        q, k, v = (conv(lin(h, p + n), _d(w[p + n + ".conv"])).view(b, t, -1, e) for n, e in (("q", c.dim), ("k", c.dim), ("v", c.vdim)))
        rep = c.heads // c.kv_heads
        q = (q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * c.dim ** -0.5).repeat_interleave(rep, 2)
        k = (k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(rep, 2)
        beta = torch.sigmoid(lin(h, p + "b"))
        lo = torch.nn.functional.softplus(lin(lin(h, p + "a1"), p + "a2") + _d(w[p + "dt_bias"]))
        g = torch.exp(-torch.exp(_d(w[p + "A_log"]))[:, None] * lo.view(b, t, c.heads, c.dim))
        S = torch.zeros(b, c.heads, c.dim, c.vdim, dtype=F64, device="cuda")
        o = torch.empty_like(v)
        for i in range(t):
            S *= g[:, i, :, :, None]
            u = beta[:, i, :, None] * (v[:, i] - (k[:, i, :, None] @ S)[:, :, 0])
            S += k[:, i, :, :, None] * u[:, :, None]
            o[:, i] = (q[:, i, :, None] @ S)[:, :, 0]
        gate = torch.sigmoid(lin(lin(h, p + "g1"), p + "g2")).view(b, t, c.heads, c.vdim)
        return lin((_unit(o, eps) * _d(w[p + "norm"]) * gate).reshape(b, t, -1), p + "o")

    x = _d(w["embed"][ids]) * cfg.embed_scale
    for i, L in enumerate(cfg.layers):
        p, h = f"l{i}.mix.", dyt(x, f"l{i}.norm1")
        if L.kind == "attention":
            x = x + chunked(p, L.attn, h)
        elif L.kind == "parallel":
            x = x + L.left_scale * window(p + "left.", L.left, h) + L.right_scale * memory(p + "right.", L.right, h)
        else:
            x = x + delta(p, L.delta, h)
        if L.ff:
            x = x + lin(torch.relu(lin(dyt(x, f"l{i}.norm2"), f"l{i}.mlp.up")).square_(), f"l{i}.mlp.down")
    return dyt(x, "final.norm"), _d(w["head"])


def exact(case, seed):
    """The whole sequences at once (no cache, no portions), shorter ones filled up behind their end."""
    cfg, tokens = _config(case), _tokens(case, seed)
    ids = torch.zeros(len(tokens), max(map(len, tokens)), dtype=torch.long)
    for i, seq in enumerate(tokens):
        ids[i, :len(seq)] = torch.tensor(seq)
    forward = {"llama": _llama, "fikerax": _fikerax, "lizesun": _lizesun}[cfg.arch]
    read, said = [], []                 # [turn][sequence] -> positions
    at = [0] * len(tokens)
    for portion in _portions(case):
        read.append([[a + w for w in _wanted(n)] for a, n in zip(at, portion)])
        said.append([[a + n + j for j in range(case["steps"])] for a, n in zip(at, portion)])
        at = [a + n + case["steps"] for a, n in zip(at, portion)]
    step = max(1, 16384 // ids.shape[1])
    parts = []
    for i in range(0, len(tokens), step):
        x, head = forward(cfg, seed, ids[i:i + step].cuda())

        def logits(places):
            which = torch.tensor([p[i:i + step] for p in places], device="cuda", dtype=torch.long)
            return x[torch.arange(x.shape[0], device="cuda")[None, :, None], which] @ head.T

        parts.append((logits(read).flatten(1, 2), logits(said).transpose(1, 2)))
    return {"read": torch.cat([p[0] for p in parts], 1), "said": torch.cat([p[1] for p in parts], 2)}
