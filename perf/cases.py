"""What the speed of this framework is measured on: single steps of the engine's model runner, the work that every request, chunk and token
that a user sends ends up as.

A case names a model directory of this repository, the type it is served in, and the sequences of ONE step: `decodes` running sequences that
bring one token each (contexts spread evenly over ctx_min..ctx_max), and `prompts` portions of prompts (lengths spread over new_min..new_max)
behind `cached` tokens that are in the cache already.  prepare() builds the runner as the engine does and runs everything that comes before
that step through it, so that caches and states hold what they hold in use; run() is the step: the logits of every sequence that is to be
sampled, on the device.  The caches' pages that the step writes and the recurrent states that it updates are returned with them.

Weights are the framework's synthetic ones with two changes, without which a rounding in the 16-bit products would grow to several percent of
the logits and the outputs would say nothing about the arithmetic.  Routers of mixture-of-experts layers are laid so that every token has clear
first choices and all experts about as many tokens, as trained ones do.  The Qwen3 models have an embedding table of unit scale, and the matrices
that write to the residual stream are scaled down by the depth, as is usual at the start of training.

exact() restates the models in float64 from their equations, whole sequences at once.
"""
from __future__ import annotations

import gc
import json
import math
import os
import random
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "nano-vllm-v1_amd"))

PAGE, CHUNK, MAX_LEN = 256, 1024, 4096
HYBRIDS = ("lamutar-hybrid-1k", "dinatar-mixed-1k", "lakatar-mixed-1k", "sokipel-mixed-1k", "mopalorn-mixed-1k", "tabedra-1k")


def _case(model, decodes=0, ctx=(0, 0), prompts=0, new=(0, 0), cached=0, dtype="bfloat16", name=None):
    c = {} if name is None else {"name": name}
    return dict(c, model=model, dtype=dtype, decodes=decodes, ctx_min=ctx[0], ctx_max=ctx[1], prompts=prompts, new_min=new[0], new_max=new[1], cached=cached)


def listed():
    return [
        # the reference's own model: one user's next token (nothing but latency) ...
        _case("qwen3-0.6b", decodes=1, ctx=(1037, 1037), name="0.6b one token"),
        # ... a server with a few users, contexts as in the offline workload (100..1024 in, 100..1024 out) ...
        _case("qwen3-0.6b", decodes=24, ctx=(100, 2047), name="0.6b 24 tokens"),
        # ... and the offline workload's full batch of 256
        _case("qwen3-0.6b", decodes=256, ctx=(100, 2047), name="0.6b 256 tokens"),
        # chunked prefill: the first chunk of a long prompt at the token budget of 1024
        _case("qwen3-0.6b", prompts=1, new=(1024, 1024), name="0.6b chunk"),
        # the step that a busy server with chunked prefill runs most: running sequences and a later portion of a prompt in what is left of the budget
        _case("qwen3-0.6b", decodes=100, ctx=(128, 1151), prompts=1, new=(924, 924), cached=1024, name="0.6b mixed"),
        # the large model of the serving script: a wave of new requests (128 tokens each on average)
        _case("qwen3-14b", prompts=8, new=(64, 191), name="14b 8 prompts"),
        # the hybrid families, each in one of the two directions (the other comes from draw): whole prompts, one at the budget and ragged ones ...
        _case("lamutar-hybrid-1k", prompts=1, new=(1024, 1024), name="lamutar chunk"),
        _case("lakatar-mixed-1k", prompts=3, new=(151, 521), name="lakatar 3 prompts"),
        _case("sokipel-mixed-1k", prompts=1, new=(1000, 1000), name="sokipel chunk"),
        # ... decoding at the batch that their comparison in bench.py takes ...
        _case("dinatar-mixed-1k", decodes=64, ctx=(512, 1535), name="dinatar 64 tokens"),
        _case("mopalorn-mixed-1k", decodes=64, ctx=(512, 1535), name="mopalorn 64 tokens"),
        # ... and served in full precision (scoring a short prompt)
        _case("tabedra-1k", prompts=1, new=(301, 301), dtype="float32", name="tabedra fp32 prompt"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    """Half of the cases on the reference's own architecture, half on the hybrids; decode, prefill (fresh or behind cached tokens) and mixed steps."""
    model = rng.choice(["qwen3-0.6b"] * 5 + ["qwen3-14b"] + list(HYBRIDS))
    dtype = "float32" if model in HYBRIDS and rng.random() < 0.15 else "bfloat16"
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "mixed"])
    most = 256 if model == "qwen3-0.6b" else 64
    decodes = ctx_min = ctx_max = prompts = new_min = new_max = cached = 0
    if kind != "prefill":
        decodes = _log_int(rng, 1, most if kind == "decode" else most // 2)
        ctx_max = _log_int(rng, 64, 2047)
        ctx_min = rng.randint(max(1, ctx_max // 8), ctx_max)
    if kind != "decode":
        room = CHUNK - decodes
        if dtype == "float32" or model == "qwen3-14b":       # (so that none costs more than the largest listed case)
            room = min(room, 512 if dtype == "float32" else 768)
        prompts = _log_int(rng, 1, 8) if kind == "prefill" else 1
        new_max = _log_int(rng, 24, room // prompts)
        new_min = rng.randint(max(1, new_max // 4), new_max)
        cached = rng.choice([0, 0, rng.randint(1, 1500)])
    return _case(model, decodes, (ctx_min, ctx_max), prompts, (new_min, new_max), cached, dtype)


# ------------------------------------------------------------------------------------------------ sizes of a step
def _spread(lo, hi, n):
    """n sizes from lo to hi, evenly spread, in an order of their own (the same for every seed)."""
    sizes = [lo + (hi - lo) * i // max(n - 1, 1) for i in range(n)] if n > 1 else [hi] * n
    random.Random(n).shuffle(sizes)
    return sizes


def _step_of(case):
    """(tokens in the cache, tokens of this step) per sequence, the running ones first as the scheduler orders them."""
    return ([(c - 1, 1) for c in _spread(case["ctx_min"], case["ctx_max"], case["decodes"])]
            + [(case["cached"], n) for n in _spread(case["new_min"], case["new_max"], case["prompts"])])


def _path(model):
    return os.path.join(ROOT, "nano-vllm-v1_amd", "model_configs", model)


def _config(model):
    with open(os.path.join(_path(model), "config.json")) as f:
        return json.load(f)


def _tokens(case, seed):
    g = torch.Generator().manual_seed(int(seed))
    vocab = 10000                                            # (as the reference's scripts draw their prompts)
    return [torch.randint(0, vocab, (c + n,), generator=g).tolist() for c, n in _step_of(case)]


# ------------------------------------------------------------------------------------------------ weights
def _weights(case):
    """(name, tensor) of every weight of the case's model in checkpoint naming."""
    from nanovllm.config import load_hf_config
    from nanovllm.models import get_model_class
    from nanovllm.utils.loader import synthetic_tensors
    cfg, hf = _config(case["model"]), load_hf_config(_path(case["model"]))
    make = getattr(get_model_class(hf), "synthetic_tensors", synthetic_tensors)
    tensors = make(hf, seed=0, device=torch.device("cuda", 0), dtype=getattr(torch, case["dtype"]))
    moe = [L["mlp"]["router"] for L in cfg.get("layers", ()) if (L.get("mlp") or {}).get("kind") == "moe"]
    if moe:
        experts, top = moe[0]["experts"], moe[0]["top"]
        g = torch.Generator().manual_seed(7)
        basis = torch.linalg.qr(torch.randn(cfg["width"], experts, generator=g))[0].t().to("cuda")         # [experts, width], orthonormal
        picks = torch.rand(cfg["vocab"], experts, generator=g).argsort(1)[:, :top].to("cuda")
    for name, t in tensors:
        if name == "model.embed_tokens.weight":
            t = t * 48.0
        elif name.endswith(("o_proj.weight", "down_proj.weight")):
            t = t / cfg["num_hidden_layers"]
        elif moe and name == "embed":
            t = (t.float() + sum((16.0 - (2.0 if top > 2 else 4.0) * j) * basis[picks[:, j]] for j in range(top))).to(t.dtype)
        elif name.endswith(".mlp.router"):
            t = (0.2 * basis.roll(5 * int(name[1:name.index(".")]), 0)).to(t.dtype)
        yield name, t


# ------------------------------------------------------------------------------------------------ the step
def prepare(case, seed):
    from nanovllm.config import Config
    from nanovllm.engine.model_runner import ModelRunner
    from nanovllm.engine.sequence import Sequence

    gc.collect()                                             # (a runner's captured graphs refer back to it)
    step, tokens = _step_of(case), _tokens(case, seed)
    # pages: those that the step writes first, then the rest of every sequence's
    written = [range(c // PAGE, (c + n - 1) // PAGE + 1) for c, n in step]
    tables = [[0] * (w.stop) for w in written]
    page = 0
    for table, w in zip(tables, written):
        for i in w:
            table[i], page = page, page + 1
    pages_written = page
    for table, w in zip(tables, written):
        for i in range(w.start):
            table[i], page = page, page + 1
    slots = max(16, -(-len(step) // 16) * 16)
    cfg = Config(_path(case["model"]), max_num_batched_tokens=CHUNK, max_num_seqs=slots, max_model_len=MAX_LEN, num_kvcache_blocks=page, chunked_prefill=True,
                 dtype=case["dtype"])
    runner = ModelRunner(cfg, 0, [])
    runner.load_weights(_weights(case))
    seqs = []
    for i, (ids, table) in enumerate(zip(tokens, tables)):
        s = Sequence(ids)
        s.block_table, s.state_slot = table, i
        seqs.append(s)
    _history(runner, seqs, [c for c, _ in step])
    for s, (c, n) in zip(seqs, step):
        s.num_cached_tokens, s.num_new_tokens = c, n
    return {"runner": runner, "seqs": seqs, "kept": _buffers(runner, pages_written, len(step))}


def _history(runner, seqs, cached):
    """Everything before the step, in steps of at most CHUNK tokens."""
    batch, room = [], CHUNK

    def flush():
        nonlocal batch, room
        if batch:
            runner.run([s for s, _ in batch])
            for s, n in batch:
                s.num_cached_tokens += n
        batch, room = [], CHUNK

    for s, c in zip(seqs, cached):
        while s.num_cached_tokens + sum(n for q, n in batch if q is s) < c:
            if any(q is s for q, _ in batch) or not room:
                flush()
                continue
            n = min(c - s.num_cached_tokens, room)
            s.num_new_tokens = n
            batch.append((s, n))
            room -= n
    flush()


def _buffers(runner, pages, slots):
    """The runner's buffers that a step leaves its keys, values and states in: the first `pages` pages, the first `slots` states."""
    if getattr(runner, "kv_cache", None) is not None:
        return {"kv": runner.kv_cache[:, :, :pages]}
    kept = {"kv": [], "states": []}
    for m in runner.model.modules():
        for cache in getattr(m, "k_caches", []) + getattr(m, "v_caches", []):
            kept["kv"].append(cache[:pages])
        for state in getattr(m, "states", []):
            if state is not None and state.dim() > 2:        # (a single number per sequence is a token id kept in such a pool)
                kept["states"].append(state[:slots])
    return kept


def run(state):
    logits, _, _ = state["runner"].forward_logits(state["seqs"])
    return dict(state["kept"], logits=logits)


# ------------------------------------------------------------------------------------------------ what a step cannot do without
def _linear(cfg):
    """(elements of the matrices every token passes, [(experts, chosen, elements of one)], elements of the output projection)."""
    if "hidden_size" in cfg:
        h, d = cfg["hidden_size"], cfg["head_dim"]
        layer = h * d * (2 * cfg["num_attention_heads"] + 2 * cfg["num_key_value_heads"]) + 3 * h * cfg["intermediate_size"]
        return cfg["num_hidden_layers"] * layer, [], cfg["vocab_size"] * h
    w, dense, experts = cfg["width"], 0, []
    times = _passes(cfg)
    for i, L in enumerate(cfg["layers"]):
        dense += times[i] * sum(_mixer_linear(kind, m, w) for kind, m in _parts(L))
        mlp = L.get("mlp")
        if not mlp:
            continue
        sides = 2 if cfg["architecture"] in ("Mopalorn", "Tabedra") or (cfg["architecture"] == "Dinatar" and mlp["kind"] == "dense") else 3
        if mlp["kind"] == "dense":
            dense += times[i] * sides * w * mlp["ff"]
            continue
        if mlp.get("shared"):
            dense += times[i] * sides * w * mlp["shared"]["ff"]
        experts += [(mlp["router"]["experts"], mlp["router"]["top"], sides * w * mlp["expert"]["ff"])] * times[i]
    return dense, experts, cfg["vocab"] * w


def _passes(cfg):
    loop = cfg.get("loop")
    return [loop["times"] if loop and loop["start"] <= i < loop["stop"] else 1 for i in range(len(cfg["layers"]))]


def _parts(L):
    """(kind, mixer) of a layer's mixers."""
    if L["type"] != "parallel":
        return [(L["type"], L["mixer"])]
    right = L["mixer"]["right"]
    return [("attention", L["mixer"]["left"]), ("mamba2" if "state" in right else "delta", right)]


def _mixer_linear(kind, m, w):
    H, G = m["heads"], m.get("kv_heads", m["heads"])
    d, dv = m.get("dim", 0), m.get("vdim", m.get("dim", 0))
    if kind in ("attention", "attention_2"):
        own = 0 if m.get("kv_from") is not None else G * (d + dv)
        return w * (H * d + own + H * dv) + (w * H * dv if "bias_max" in m else 0)
    if kind == "latent_attention":
        q = m["q_rank"] * (w + H * (d + m["rot_dim"])) if "q_rank" in m else w * H * (d + m["rot_dim"])
        return q + (0 if m.get("kv_from") is not None else w * (m["kv_rank"] + m["rot_dim"])) + m["kv_rank"] * H * (d + dv) + w * H * dv
    if kind == "mamba2":
        return w * (3 * H * dv + 2 * m["groups"] * m["state"] + H)
    if kind == "general_delta":
        return 6 * w * H * d
    if kind == "delta":
        return w * (2 * G * d + 3 * H * dv)
    return w * H * {"wkv": 5 * d, "hgrn2": 2 * d + 2 * dv}.get(kind, 2 * d + 3 * dv)


def _cached_row(kind, m):
    """(heads, key size, value size, cached elements of a token, window) of an attention mixer."""
    if kind == "latent_attention":
        row = m["kv_rank"] + m["rot_dim"]
        return m["heads"], row, m["kv_rank"], row, (m.get("mask") or {}).get("size", 0)
    d, dv = m["dim"], m.get("vdim", m["dim"])
    return m["heads"], d, dv, m.get("kv_heads", m["heads"]) * (d + dv), (m.get("mask") or {}).get("size", 0)


def work(case):
    cfg, step = _config(case["model"]), _step_of(case)
    size = 4 if case["dtype"] == "float32" else 2
    tokens, rows = sum(n for _, n in step), len(step)
    dense, experts, head = _linear(cfg)
    flops = 2.0 * tokens * dense + 2.0 * rows * head
    nbytes = size * (dense + head) + rows * head / (cfg.get("width") or cfg["hidden_size"]) * (2 if "hidden_size" in cfg else 4)
    for count, top, elements in experts:
        nbytes += size * elements * min(count, top * tokens)
        flops += 2.0 * tokens * top * elements
    mixers = []
    if "hidden_size" in cfg:
        m = {"heads": cfg["num_attention_heads"], "kv_heads": cfg["num_key_value_heads"], "dim": cfg["head_dim"]}
        mixers = [("attention", m)] * cfg["num_hidden_layers"]
    else:
        for times, L in zip(_passes(cfg), cfg["layers"]):
            mixers += _parts(L) * times
    for kind, m in mixers:
        if "attention" in kind:
            H, dk, dv, row, window = _cached_row(kind, m)
            for c, n in step:
                seen = [min(p + 1, window) if window else p + 1 for p in (c, c + n - 1)]
                flops += 2.0 * n * (seen[0] + seen[1]) / 2 * H * (dk + dv)
                nbytes += size * row * (min(c, window) + n if window else c + n)
        else:
            dk, dv = (m["state"], m["vdim"]) if kind == "mamba2" else (m["dim"], m.get("vdim", m["dim"]))
            flops += 2.0 * tokens * m["heads"] * dk * dv * (3 if "delta" in kind else 2)
            nbytes += 4.0 * m["heads"] * dk * dv * sum(2 if c else 1 for c, _ in step)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Measured against float64: fp32 0.8e-6 to 2e-6 off; bf16 0.002 to 0.005 over an fp32 residual stream (the hybrids), 0.010 to 0.016 over a bf16
    one of 28 and 40 layers."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5}
    return {"rel": 0.02 if case["model"] in HYBRIDS else 0.03}


# ------------------------------------------------------------------------------------------------ the models in float64
# x is [sequences, tokens, width], every sequence from its first token, padded at its end (nothing looks ahead).
F = torch.float64


class _Weights:
    """A checkpoint's tensors in float64, converted where they are used."""

    def __init__(self, tensors, prefix=""):
        self.tensors, self.prefix = tensors, prefix

    def __getitem__(self, name):
        return self.tensors[self.prefix + name].to(F)

    def __contains__(self, name):
        return self.prefix + name in self.tensors

    def at(self, more):
        return _Weights(self.tensors, self.prefix + more)

    def mul(self, name, x):
        return torch.matmul(x, self[name].t().contiguous())


def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, w, b, eps):
    x = x - x.mean(-1, keepdim=True)
    return _unit(x, eps) * w + b


def _silu(x):
    return x * torch.sigmoid(x)


def _heads(x, n):
    return x.view(*x.shape[:-1], n, -1)


def _flat(x):
    return x.reshape(*x.shape[:-2], -1)


def _conv(x, w, bias=None):
    """Causal convolution over time per channel, the last tap on the token itself."""
    taps = w.shape[1]
    pad = torch.cat([x.new_zeros(x.shape[0], taps - 1, x.shape[2]), x], 1)
    y = sum(pad[:, j:j + x.shape[1]] * w[:, j] for j in range(taps))
    return y if bias is None else y + bias


def _frequencies(rot, device):
    """Frequencies of the pairs and the factor on sine and cosine: plain, all divided by a factor, by turns over the original length (YaRN), or by wavelength."""
    dims, base, sc = rot["dims"], rot["base"], rot.get("scaling")
    f = torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=F, device=device)
    if not sc:
        return f, 1.0
    if "fast" in sc:
        def where(turns):
            return dims * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
        lo, hi = max(math.floor(where(sc["fast"])), 0), min(math.ceil(where(sc["slow"])), dims - 1)
        ramp = ((torch.arange(dims // 2, dtype=F, device=device) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        return f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1.0
    if "original" in sc:
        turns = sc["original"] * f / (2 * math.pi)
        mix = ((turns - sc["low"]) / (sc["high"] - sc["low"])).clamp(0.0, 1.0)
        return (1 - mix) * f / sc["factor"] + mix * f, 1.0
    return f / sc["factor"], 1.0


def _rotate(x, rot, interleaved=False, sign=1.0):
    if not rot:
        return x
    dims = rot["dims"]
    f, mag = _frequencies(rot, x.device)
    ang = sign * torch.arange(x.shape[1], dtype=F, device=x.device)[:, None, None] * f
    c, s = torch.cos(ang) * mag, torch.sin(ang) * mag
    out = x.clone()
    first, second = (slice(0, dims, 2), slice(1, dims, 2)) if interleaved else (slice(0, dims // 2), slice(dims // 2, dims))
    a, b = x[..., first], x[..., second]
    out[..., first], out[..., second] = a * c - b * s, b * c + a * s
    return out


def _attend(q, k, v, scale, visible, bias=None, sink=None, cap=0.0):
    """q [N, T, H, d], k [N, S, G, d], v [N, S, G, e], visible [T, S], bias [H, T, S] -> [N, T, H, e]."""
    N, T, H, _ = q.shape
    group = H // k.shape[2]
    out = q.new_empty(N, T, H, v.shape[3])
    for n in range(N):
        for h in range(H):
            s = torch.matmul(q[n, :, h].contiguous(), k[n, :, h // group].t().contiguous()) * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            if bias is not None:
                s = s + bias[h]
            s = s.masked_fill(~visible, -math.inf)
            top = s.amax(1, keepdim=True) if sink is None else torch.maximum(s.amax(1, keepdim=True), sink[h])
            e = torch.exp(s - top)
            den = e.sum(1, keepdim=True) + (0.0 if sink is None else torch.exp(sink[h] - top))
            out[n, :, h] = torch.matmul(e / den, v[n, :, h // group].contiguous())
    return out


def _causal(T, device, window=0, keep_first=0, chunk=0):
    i, j = torch.arange(T, device=device)[:, None], torch.arange(T, device=device)[None, :]
    seen = j <= i
    if window:
        seen = seen & ((i - j < window) | (j < keep_first))
    if chunk:
        seen = seen & (i // chunk == j // chunk)
    return seen


def _scan(q, k, w, v, read_first=False, bonus=None):
    """S <- diag(w) S + k v^T, o = S^T q; q, k, w [N, T, H, dk] (w's last axis may be 1), v [N, T, H, dv]."""
    N, T, H, dk = k.shape
    S, out = v.new_zeros(N, H, dk, v.shape[3]), torch.empty_like(v)
    for t in range(T):
        kv = k[:, t, :, :, None] * v[:, t, :, None, :]
        if read_first:
            out[:, t] = ((S + bonus[:, :, None] * kv) * q[:, t, :, :, None]).sum(2)
            S = w[:, t, :, :, None] * S + kv
        else:
            S = w[:, t, :, :, None] * S + kv
            out[:, t] = (S * q[:, t, :, :, None]).sum(2)
    return out


def _delta_scan(q, k, w, u, au, v):
    """S <- diag(w) S - au (u^T S) + k v^T, both terms from the old S; o = S^T q."""
    N, T, H, dk = k.shape
    S, out = v.new_zeros(N, H, dk, v.shape[3]), torch.empty_like(v)
    for t in range(T):
        uS = (u[:, t, :, :, None] * S).sum(2)
        S = w[:, t, :, :, None] * S - au[:, t, :, :, None] * uS[:, :, None, :] + k[:, t, :, :, None] * v[:, t, :, None, :]
        out[:, t] = (S * q[:, t, :, :, None]).sum(2)
    return out


def _softplus(x):
    return torch.nn.functional.softplus(x, threshold=50.0)


def _gated(W, x, act=_silu):
    return W.mul("down", act(W.mul("gate", x)) * W.mul("up", x))


def _squared(W, x):
    return W.mul("down", torch.relu(W.mul("up", x)) ** 2)


def _mixture(W, x, ids, weights, expert):
    """Sum over a token's chosen experts; expert(weights of one, rows, their routing weights)."""
    flat, out = x.reshape(-1, x.shape[-1]), torch.zeros_like(x).reshape(-1, x.shape[-1])
    ids, weights = ids.reshape(flat.shape[0], -1), weights.reshape(flat.shape[0], -1)
    for e in range(int(ids.max()) + 1):
        at, j = torch.nonzero(ids == e, as_tuple=True)
        if at.numel():
            out.index_add_(0, at, expert(W.at(f"e{e}."), flat[at], weights[at, j][:, None]))
    return out.view_as(x)


# Qwen3 (models/qwen3.py)
def _qwen3(cfg, W, tokens, last):
    eps, H, G = cfg["rms_norm_eps"], cfg["num_attention_heads"], cfg["num_key_value_heads"]
    x = W.tensors["model.embed_tokens.weight"][tokens].to(F)
    seen, rot = _causal(tokens.shape[1], x.device), {"dims": cfg["head_dim"], "base": float(cfg["rope_theta"])}
    for i in range(cfg["num_hidden_layers"]):
        L = W.at(f"model.layers.{i}.")
        h = _unit(x, eps) * L["input_layernorm.weight"]
        q, k, v = (_heads(L.mul(f"self_attn.{n}_proj.weight", h), c) for n, c in (("q", H), ("k", G), ("v", G)))
        q, k = _unit(q, eps) * L["self_attn.q_norm.weight"], _unit(k, eps) * L["self_attn.k_norm.weight"]
        o = _attend(_rotate(q, rot), _rotate(k, rot), v, cfg["head_dim"] ** -0.5, seen)
        x = x + L.mul("self_attn.o_proj.weight", _flat(o))
        h = _unit(x, eps) * L["post_attention_layernorm.weight"]
        x = x + L.mul("mlp.down_proj.weight", _silu(L.mul("mlp.gate_proj.weight", h)) * L.mul("mlp.up_proj.weight", h))
    x = _unit(x[torch.arange(x.shape[0]), last], eps) * W["model.norm.weight"]
    return W.mul("model.embed_tokens.weight" if cfg["tie_word_embeddings"] else "lm_head.weight", x)


# Lamutar (models/lamutar.py)
def _lamutar_attention(W, m, eps, h):
    H, G, dv = m["heads"], m["kv_heads"], m["vdim"]
    q, k, v = _unit(W.mul("q", h), eps) * W["q.norm"], _unit(W.mul("k", h), eps) * W["k.norm"], W.mul("v", h)
    turn = {"dims": dv, "base": m["rot"]["base"]}
    v = _rotate(_heads(v, G), turn)
    o = _attend(_rotate(_heads(q, H), m["rot"]), _rotate(_heads(k, G), m["rot"]), v, m["scale"], _causal(h.shape[1], h.device))
    o = _rotate(o, turn, sign=-1.0) * torch.sigmoid(W.mul("g", h))[..., None]
    return W.mul("o", _flat(o))


def _general_delta(W, m, eps, h):
    r, k, v = (_heads(W.mul(n, h), m["heads"]) for n in "rkv")
    z = torch.matmul(torch.tanh(W.mul("w1", h)), W["w2"].t().contiguous()) + W["w0"]
    w = _heads(torch.exp(-math.exp(-0.5) * torch.sigmoid(z)), m["heads"])
    a = _heads(torch.sigmoid(W.mul("a", h) + W["a.b"]), m["heads"])
    u = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    o = _flat(_unit(_delta_scan(r, k, w, u, a * u, v), eps)) * W["norm"]
    return W.mul("o", o * torch.sigmoid(W.mul("g", h)))


def _lamutar(cfg, W, tokens, last):
    eps, loop = cfg["norm"]["eps"], cfg["loop"]

    def dyt(L, name, x):
        return torch.tanh(L[name + ".alpha"] * x) * L[name] + L[name + ".b"]

    def gelu(z):
        return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))

    x = first = W.tensors["embed"][tokens].to(F)
    order = [(i, -1) for i in range(loop["start"])] + [(i, t) for t in range(loop["times"]) for i in range(loop["start"], loop["stop"])]
    for i, t in order + [(i, -1) for i in range(loop["stop"], len(cfg["layers"]))]:
        L, spec = W.at(f"l{i}."), cfg["layers"][i]
        if t >= 0 and i == loop["start"]:
            x = W.mul("loop.in", torch.cat([x, first], -1)) + W["loop.step"][t]
        mixer = _lamutar_attention if spec["type"] == "attention" else _general_delta
        x = x + dyt(L, "norm1b", mixer(L.at("mix."), spec["mixer"], eps, dyt(L, "norm1", x)))
        if spec.get("mlp"):
            x = x + dyt(L, "norm2b", _gated(L.at("mlp."), dyt(L, "norm2", x), gelu))
    z = W.mul("head", dyt(W, "final.norm", x[torch.arange(x.shape[0]), last]))
    return cfg["logit_softcap"] * torch.tanh(z / cfg["logit_softcap"])


# Dinatar (models/dinatar.py)
def _biased_attention(W, m, h):
    T, H, G = h.shape[1], m["heads"], m["kv_heads"]
    q, k, v = (_heads(W.mul(n, h) + W[n + ".b"], c) for n, c in (("q", H), ("k", G), ("v", G)))
    slope = torch.tensor([2.0 ** (-8.0 * (i + 1) / H) for i in range(H)], dtype=F, device=h.device)
    p = torch.arange(T, dtype=F, device=h.device)
    bias = -slope[:, None, None] * (p[:, None] - p[None, :])
    o = _attend(q, k, v, m["scale"], _causal(T, h.device, m["mask"]["size"], m["mask"]["keep_first"]), bias)
    return W.mul("o", _flat(o))


def _mamba2(W, m, eps, h):
    H, dv, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
    z, xbc, dt = W.mul("in", h).split([H * dv, H * dv + 2 * G * N, H], -1)
    x, B, C = _silu(_conv(xbc, W["conv"], W["conv.b"])).split([H * dv, G * N, G * N], -1)
    x, B, C = _heads(x, H), (_heads(B, G).repeat_interleave(H // G, 2)), _heads(C, G).repeat_interleave(H // G, 2)
    dt = _softplus(dt + W["dt_bias"])[..., None]
    y = _scan(C, dt * B, torch.exp(-torch.exp(W["A_log"])[:, None] * dt), x) + W["D"][:, None] * x
    y = _heads(_flat(y) * _silu(z), m["norm_groups"])
    return W.mul("o", _flat(_unit(y, eps)) * W["norm"])


def _hgrn2(W, m, eps, h):
    f = W["lower"] + (1.0 - W["lower"]) * torch.sigmoid(W.mul("f", h) + W["f.b"])
    q, f, v = (_heads(t, m["heads"]) for t in (_silu(W.mul("q", h)), f, W.mul("v", h)))
    return W.mul("o", _flat(_unit(_scan(q, 1.0 - f, f, v), eps) * W["norm"]))


def _gla(W, m, eps, h):
    q, k, v = (_heads(W.mul(n, h), m["heads"]) for n in "qkv")
    z = W.mul("a2", W.mul("a1", h)) + W["a2.b"]
    decay = _heads(torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]), m["heads"])
    o = _unit(_scan(q * m["dim"] ** -0.5, k, decay, v), eps) * W["norm"]
    return W.mul("o", _flat(o) * _silu(W.mul("g", h)))


def _dinatar(cfg, W, tokens, last):
    eps = cfg["norm"]["eps"]
    order = [i for i in range(len(cfg["layers"]))]
    if cfg.get("loop"):
        a, b = cfg["loop"]["start"], cfg["loop"]["stop"]
        order = order[:a] + order[a:b] * cfg["loop"]["times"] + order[b:]
    x = W.tensors["embed"][tokens].to(F) * cfg["embedding"]["scale"] + W["pos"][:tokens.shape[1]]
    for i in order:
        L, spec = W.at(f"l{i}."), cfg["layers"][i]
        M, m, mlp = L.at("mix."), spec["mixer"], spec.get("mlp")
        h = _layer_norm(x, L["norm1"], L["norm1.b"], eps)
        if spec["type"] == "parallel":
            left, right = _biased_attention(M.at("left."), m["left"], h), _mamba2(M.at("right."), m["right"], eps, h)
            x = x + 0.5 * (_unit(left, eps) * M["left.out"] + _unit(right, eps) * M["right.out"])
        else:
            x = x + (_hgrn2 if spec["type"] == "hgrn2" else _gla)(M, m, eps, h)
        E = L.at("mlp.")
        if mlp and mlp["kind"] == "dense":
            x = x + _squared(E, h)
        elif mlp:
            best, ids = (E.mul("router", h) + E["router.b"]).topk(mlp["router"]["top"], -1)
            x = x + _mixture(E, h, ids, torch.softmax(best, -1), lambda w, r, a: a * _gated(w, r))
            if mlp.get("shared"):
                x = x + _gated(E.at("shared."), h)
    x = _layer_norm(x[torch.arange(x.shape[0]), last], W["final.norm"], W["final.norm.b"], eps)
    return W.mul("embed", x) * cfg["logit_scale"]


# Lakatar (models/lakatar.py)
def _wkv(W, m, eps, h):
    before = torch.cat([torch.zeros_like(h[:, :1]), h[:, :-1]], 1)
    mixed = {n: h + (before - h) * W["mu." + n] for n in "rkvgw"}
    r, k, v = (_heads(W.mul(n, mixed[n]), m["heads"]) for n in "rkv")
    z = W.mul("w2", torch.tanh(W.mul("w1", mixed["w"]))) + W["w0"]
    o = _scan(r, k, _heads(torch.exp(-torch.exp(z)), m["heads"]), v, True, W["u"])
    return W.mul("o", _flat(_unit(o, eps)) * W["norm"] * _silu(W.mul("g", mixed["g"])))


def _retention(W, m, eps, h):
    q, k, v = (_heads(W.mul(n, h), m["heads"]) for n in "qkv")
    decay = torch.tensor(m["decay"], dtype=F, device=h.device)[:, None].expand(*q.shape[:3], 1)
    o = _scan(_rotate(q, m["rot"]), _rotate(k, m["rot"]) * m["dim"] ** -0.5, decay, v)
    return W.mul("o", _flat(_unit(o, eps)) * _silu(W.mul("g", h)))


def _latent_attention(W, m, eps, h, interleaved, latents, index):
    H, d, R = m["heads"], m["dim"], m["kv_rank"]
    q = W.mul("uq", _unit(W.mul("dq", h), eps) * W["dq.norm"]) if "dq" in W else W.mul("q", h)
    q = _heads(q, H)
    q = torch.cat([q[..., :d], _rotate(q[..., d:], m["rot"], interleaved)], -1)
    if m.get("kv_from") is None:
        down = W.mul("dkv", h)
        latents[index] = _unit(down[..., :R], eps) * W["dkv.norm"], _rotate(down[..., None, R:], m["rot"], interleaved)
    c, k_rot = latents[index if m.get("kv_from") is None else m["kv_from"]]
    k = torch.cat([_heads(W.mul("uk", c), H), k_rot.expand(*k_rot.shape[:2], H, -1)], -1)
    seen = _causal(h.shape[1], h.device, (m.get("mask") or {}).get("size", 0))
    return _attend(q, k, _heads(W.mul("uv", c), H), m["scale"], seen)


def _lakatar(cfg, W, tokens, last):
    eps, alpha, latents = cfg["norm"]["eps"], cfg["postln_alpha"], {}
    x = W.tensors["embed"][tokens].to(F)
    for i, spec in enumerate(cfg["layers"]):
        L, m, mlp = W.at(f"l{i}."), spec["mixer"], spec.get("mlp")
        M, E = L.at("mix."), L.at("mlp.")
        if spec["type"] == "latent_attention":
            o = _latent_attention(M, m, eps, x, True, latents, i) * torch.sigmoid(M.mul("g", x))[..., None]
            y = M.mul("o", _flat(o))
        else:
            y = (_wkv if spec["type"] == "wkv" else _retention)(M, m, eps, x)
        x = _unit(alpha * x + L["ls1"] * y, eps) * (1.0 + L["norm1"])
        if mlp:
            r = mlp["router"]
            s = torch.softmax(E.mul("router", x), -1)
            choice = s + E["correction"]
            grouped = choice.view(*choice.shape[:-1], r["groups"]["count"], -1)
            kept = grouped.amax(-1).topk(r["groups"]["keep"], -1).indices
            allowed = torch.zeros(grouped.shape[:-1], dtype=torch.bool, device=x.device).scatter_(-1, kept, True)
            ids = choice.masked_fill(~allowed.repeat_interleave(grouped.shape[-1], -1), -math.inf).topk(r["top"], -1).indices
            y = _mixture(E, x, ids, s.gather(-1, ids) * r["scale"], lambda w, rows, a: a * _gated(w, rows))
            y = y + torch.sigmoid(E.mul("shared.sg", x)) * _gated(E.at("shared."), x)
            x = _unit(alpha * x + L["ls2"] * y, eps) * (1.0 + L["norm2"])
    return W.mul("head", _unit(x[torch.arange(x.shape[0]), last], eps) * (1.0 + W["final.norm"]))


# Sokipel (models/sokipel.py)
def _sink_attention(W, m, eps, h, beside):
    H, G = m["heads"], m["kv_heads"]
    q, k, v = (W.mul(n, h) for n in "qkv")
    if beside:
        q, k, v = q + W["q.b"], k + W["k.b"], v + W["v.b"]
        q, k = _unit(_heads(q, H), eps) * W["q.norm"], _unit(_heads(k, G), eps) * W["k.norm"]
    else:
        q, k = _heads(_unit(q, eps) * W["q.norm"], H), _heads(_unit(k, eps) * W["k.norm"], G)
    seen = _causal(h.shape[1], h.device, chunk=(m.get("mask") or {}).get("size", 0))
    o = _attend(_rotate(q, m["rot"], not beside), _rotate(k, m["rot"], not beside), _heads(v, G), m["scale"], seen, sink=W["sink"])
    if beside:
        o = o * torch.sigmoid(W.mul("g", h))[..., None]
    return W.mul("o", _flat(o))


def _gated_delta(W, m, eps, h):
    H, G, d = m["heads"], m["kv_heads"], m["dim"]
    q, k, v = (_silu(_conv(W.mul(n, h), W[n + ".conv"])) for n in "qkv")
    q, k = ((t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 2) for t in (_heads(q, G), _heads(k, G)))
    beta = torch.sigmoid(W.mul("b", h))[..., None]
    g = torch.exp(-torch.exp(W["A_log"]) * _softplus(W.mul("a", h) + W["dt_bias"]))[..., None]
    o = _delta_scan(q / math.sqrt(d), beta * k, g, k, beta * g * k, _heads(v, H))
    return W.mul("o", _flat(_unit(o, eps) * W["norm"]) * _silu(W.mul("g", h)))


def _sokipel(cfg, W, tokens, last):
    eps, mult = cfg["norm"]["eps"], cfg["residual_mult"]
    x = W.tensors["embed"][tokens].to(F) * cfg["embedding"]["scale"]
    for i, spec in enumerate(cfg["layers"]):
        L, m, mlp = W.at(f"l{i}."), spec["mixer"], spec.get("mlp")
        M, E = L.at("mix."), L.at("mlp.")
        h = x + _conv(x, L["canon1"])
        if spec["type"] == "attention":
            y = _sink_attention(M, m, eps, h, False)
        elif spec["type"] == "delta":
            y = _gated_delta(M, m, eps, h)
        else:
            y = m["left_scale"] * _sink_attention(M.at("left."), m["left"], eps, h, True) + m["right_scale"] * _gated_delta(M.at("right."), m["right"], eps, h)
        x = x + mult * L["norm1"] * _unit(y, eps)
        if mlp:
            cap = mlp["expert"]["limit"]

            def expert(w, rows, a):
                gate, up = w.mul("gate", a * rows).clamp(max=cap), w.mul("up", a * rows).clamp(-cap, cap)
                return w.mul("down", gate * torch.sigmoid(1.702 * gate) * (up + 1.0))

            score, ids = torch.sigmoid(E.mul("router", x)).topk(mlp["router"]["top"], -1)
            x = x + mult * L["norm2"] * _unit(_mixture(E, x, ids, score, expert), eps)
    z = W.mul("head", W["final.norm"] * _unit(x[torch.arange(x.shape[0]), last], eps))
    return cfg["logit_softcap"] * torch.tanh(z / cfg["logit_softcap"])


# Mopalorn (models/mopalorn.py)
def _pooled_attention(W, m, h, v):
    H, G, T = m["heads"], m["kv_heads"], h.shape[1]
    size, pool = m["mask"]["size"], m["mask"]["pool"]
    q, k = _heads(W.mul("q", h), H), _heads(W.mul("k", h), G)
    blocks = T // pool
    means = [t[:, :blocks * pool].view(t.shape[0], blocks, pool, *t.shape[2:]).mean(2) for t in (k, v)]
    i = torch.arange(T, device=h.device)[:, None]
    whole = torch.arange(blocks, device=h.device)[None, :] < torch.div((i - size + 1).clamp(min=0), pool, rounding_mode="floor")
    seen = torch.cat([whole, _causal(T, h.device, size)], 1)
    return _attend(q, torch.cat([means[0], k], 1), torch.cat([means[1], v], 1), m["scale"], seen, sink=W["sink"])


def _mopalorn(cfg, W, tokens, last):
    eps, first = cfg["norm"]["eps"], None
    x = W.tensors["embed"][tokens].to(F)
    for i, spec in enumerate(cfg["layers"]):
        L, m = W.at(f"l{i}."), spec["mixer"]
        M, E = L.at("mix."), L.at("mlp.")
        h = _unit(x, eps) * L["norm1"]
        if spec["type"] == "latent_attention":
            o = _flat(_latent_attention(M, m, eps, h, False, {}, i)) * torch.sigmoid(M.mul("g", h))
        else:
            own = M.mul("v", h)
            v = own if first is None else (1.0 - M["vmix"]) * own + M["vmix"] * first
            first, v = own if first is None else first, _heads(v, m["kv_heads"])
            if spec["type"] == "attention":
                p = torch.arange(h.shape[1], device=h.device)
                warm = 1.0 + m["q_temp"]["coef"] * torch.log(torch.div(p + 1, m["q_temp"]["every"], rounding_mode="floor").to(F) + 1)
                q, k = _heads(M.mul("q", h), m["heads"]) * warm[:, None, None], _heads(M.mul("k", h), m["kv_heads"])
                o = _attend(q, k, v, m["scale"], _causal(h.shape[1], h.device), cap=m["softcap"])
            else:
                o = _pooled_attention(M, m, h, v)
            o = _flat(o)
        x = x + _unit(M.mul("o", o), eps) * L["norm1b"]
        z = E.mul("up", _unit(x, eps) * L["norm2"])
        p, q = _softplus(E["act"][0]), _softplus(E["act"][1])
        z = torch.where(z > 0, p * z * z + z / 2, (0.5 + q) * (torch.expm1(z.clamp(max=0.0)) - z) + z / 2)
        x = x + _unit(E.mul("down", z), eps) * L["norm2b"]
    return W.mul("embed", _unit(x[torch.arange(x.shape[0]), last], eps) * W["final.norm"]) * cfg["logit_scale"]


# Tabedra (models/tabedra.py)
def _distance_bias(rel, reach, T):
    rows = rel.shape[0]
    half = rows // 2

    def bucket(n):
        return n if n < half else min(rows - 1, half + math.floor(math.log(n / half) / math.log(reach / half) * (rows - half) + 1e-9))

    of = torch.tensor([bucket(n) for n in range(T)], device=rel.device)
    p = torch.arange(T, device=rel.device)
    return rel[of[(p[:, None] - p[None, :]).clamp(min=0)]].permute(2, 0, 1).contiguous()


def _tabedra(cfg, W, tokens, last):
    eps, T, kept = cfg["norm"]["eps"], tokens.shape[1], {}
    b = cfg["embedding"]["bigram"]
    pair = torch.cat([torch.full_like(tokens[:, :1], b["buckets"]), (tokens[:, :-1] * b["mul_prev"] + tokens[:, 1:] * b["mul_cur"]) % b["buckets"]], 1)
    x = W.tensors["embed"][tokens].to(F) + W.tensors["bigram"][pair].to(F) + W["pos"][:T]
    streams = [x] * cfg["streams"]

    def around(L, q, sublayer):
        into, out, mix = L[f"hc{q}.in"], L[f"hc{q}.out"], L[f"hc{q}.mix"]
        y = sublayer(_layer_norm(sum(into[s] * t for s, t in enumerate(streams)), L[f"norm{q}"], L[f"norm{q}.b"], eps))
        return [sum(mix[s, t] * z for s, z in enumerate(streams)) + out[t] * y for t in range(len(streams))]

    for i, spec in enumerate(cfg["layers"]):
        L, m, mlp = W.at(f"l{i}."), spec["mixer"], spec["mlp"]

        def mixer(h):
            M, H, G = L.at("mix."), m["heads"], m["kv_heads"]

            def part(leaf, n):
                return _heads(_conv(M.mul(leaf, h), M[leaf + ".conv"]), n)

            q = _unit(part("q", H), eps)
            if m.get("kv_from") is None:
                kept[i] = _unit(part("k", G), eps), part("v", G)
            k, v = kept[i if m.get("kv_from") is None else m["kv_from"]]
            o = _attend(q, k, v, m["scale"], _causal(T, h.device, m["mask"]["size"]), _distance_bias(M["rel"], m["bias_max"], T))
            return M.mul("o", _flat(o) * torch.sigmoid(M.mul("g", h)))

        def experts(h):
            E = L.at("mlp.")
            s = torch.softmax(E.mul("router", h), -1)
            ids = (s + E["correction"]).topk(mlp["router"]["top"], -1).indices
            w = s.gather(-1, ids)
            w = w / (w.sum(-1, keepdim=True) + 1e-20)
            return _mixture(E, h, ids, w, lambda e, rows, a: a * _squared(e, rows)) + _squared(E.at("shared."), h)

        streams = around(L, 1, mixer)
        streams = around(L, 2, experts)
    x = sum(streams)[torch.arange(tokens.shape[0]), last]
    return W.mul("head", _layer_norm(x, W["final.norm"], W["final.norm.b"], eps))


_FORWARD = {"Lamutar": _lamutar, "Dinatar": _dinatar, "Lakatar": _lakatar, "Sokipel": _sokipel, "Mopalorn": _mopalorn, "Tabedra": _tabedra}


@torch.inference_mode()
def exact(case, seed):
    """The logits; the caches and states lie in the framework's own layouts and have no plain counterpart."""
    cfg, tokens = _config(case["model"]), _tokens(case, seed)
    if sum(len(t) for t in tokens) > {"qwen3-0.6b": 280_000, "qwen3-14b": 18_000}.get(case["model"], 100_000):
        return None                                          # (20 s and more in float64)
    weights = dict(_weights(case))
    W, forward = _Weights(weights), _FORWARD.get(cfg.get("architecture"), _qwen3)
    order = sorted(range(len(tokens)), key=lambda i: len(tokens[i]))
    rows = [None] * len(tokens)
    while order:
        group, longest = [], 0
        while order and (not group or (len(group) + 1) * max(longest, len(tokens[order[-1]])) <= 32768):
            group.append(order.pop())
            longest = max(longest, len(tokens[group[-1]]))
        batch = torch.tensor([tokens[i] + [0] * (longest - len(tokens[i])) for i in group], device="cuda")
        last = torch.tensor([len(tokens[i]) - 1 for i in group], device="cuda")
        for i, z in zip(group, forward(cfg, W, batch, last)):
            rows[i] = z
    out = {"logits": torch.stack(rows), "kv": None}
    return out if "hidden_size" in cfg else dict(out, states=None)
