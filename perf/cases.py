"""Performance cases: the work that programs on this backend have it do.

A case names a kind of call, a model and its sizes:

* ``decode``: a session whose caches hold a prompt decodes ``steps`` greedy
  steps and returns the tokens and the last step's logits;
* ``prefill``: a session's empty caches take the prompts (of one length, or
  ragged) and the last rows' logits come back;
* ``forward``: the trainer's forward with its cross-entropy over every row;
* ``nodes``: one sequence through the per-shader launchers, as a graph
  builder drives them: the prompt's prefill graph, then captured decode steps;
* ``sample``: one token per row of device logits by the reference's sampler.

Models are ``hall`` (dim 768, 12 layers, 12 heads of 64), ``pidgeon``
(dim 320, 8 layers, 5 heads of 64) and ``scaled`` (dim 2048, 16 heads of 128,
bfloat16-valued weights) cut to two of its 24 layers, which keeps the layer's
kernels and the lm_head at their full sizes.  A program loads its weights once
and opens sessions on them, so the last models used are kept here; prompts,
caches and logits are made anew from the seed.
"""

import ctypes
import importlib
from collections import OrderedDict
from dataclasses import replace

import numpy as np
import torch

akasha = importlib.import_module("akasha-core_amd")
hip = akasha.hip

_backend = None
_models = OrderedDict()  # at most two of (name, bf16) -> Model
_weights = OrderedDict()  # at most one of name -> float32 host arrays


def listed():
    return [
        # One user's chat: a short prompt, then tokens one by one.  Launches
        # and latency count; the weights are read once per token.
        {"name": "chat_decode", "kind": "decode", "model": "hall", "batch": 1, "prompt": 64,
         "steps": 16, "kv16": False},
        # A full serving batch near the end of the 512-token context.
        {"name": "batch_decode", "kind": "decode", "model": "hall", "batch": 32, "prompt": 448,
         "steps": 16, "kv16": False},
        # The scaled model with 64 sequences at the end of a 2048-token
        # context: the KV cache's rows are what is read.
        {"name": "long_decode", "kind": "decode", "model": "scaled", "batch": 64, "prompt": 2040,
         "steps": 4, "kv16": False},
        # A chat's first prompt: the smallest prefill, few rows per matrix.
        {"name": "chat_prefill", "kind": "prefill", "model": "hall", "batch": 1, "prompt": 64,
         "ragged": False, "bf16": False},
        # Prompts of uneven, odd lengths arriving together.
        {"name": "ragged_prefill", "kind": "prefill", "model": "hall", "batch": 7, "prompt": 211,
         "ragged": True, "bf16": False},
        # A serving batch of full-context prompts.
        {"name": "batch_prefill", "kind": "prefill", "model": "hall", "batch": 16, "prompt": 512,
         "ragged": False, "bf16": False},
        # Long prompts on the scaled model, in fp32 accuracy.
        {"name": "long_prefill", "kind": "prefill", "model": "scaled", "batch": 8, "prompt": 2048,
         "ragged": False, "bf16": False},
        # The same on the optional bfloat16 kernels.
        {"name": "long_prefill_bf16", "kind": "prefill", "model": "scaled", "batch": 8,
         "prompt": 2048, "ragged": False, "bf16": True},
        # A training batch's forward: every row through the lm_head and the
        # cross-entropy.
        {"name": "train_forward", "kind": "forward", "model": "hall", "batch": 16, "prompt": 512},
        # A chat turn through the reference's graph of shaders.
        {"name": "nodes_chat", "kind": "nodes", "model": "hall", "prompt": 64, "steps": 8},
        # Sampling a batch with the chat command's parameters.
        {"name": "sample_chat", "kind": "sample", "rows": 32, "vocab": 50257, "seen": 480,
         "temperature": 0.8, "top_k": 40, "top_p": 0.95, "penalty": 1.15},
        # Sampling with no top_k: the nucleus of the whole vocabulary.
        {"name": "sample_nucleus", "kind": "sample", "rows": 32, "vocab": 50257, "seen": 0,
         "temperature": 0.8, "top_k": 0, "top_p": 0.95, "penalty": 1.0},
    ]


def _log(rng, low, high):
    """A whole number, uniform in its logarithm."""
    return min(high, max(low, round(low * (high / low) ** rng.random())))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "forward", "nodes",
                       "sample"])
    if kind == "decode":
        if rng.random() < 0.35:
            return {"kind": kind, "model": "scaled", "batch": _log(rng, 8, 64),
                    "prompt": _log(rng, 100, 2040), "steps": rng.randint(2, 4),
                    "kv16": rng.random() < 0.5}
        return {"kind": kind, "model": rng.choice(["hall", "hall", "pidgeon"]),
                "batch": _log(rng, 1, 32), "prompt": _log(rng, 16, 448),
                "steps": rng.randint(4, 16), "kv16": False}
    if kind == "prefill":
        if rng.random() < 0.4:
            return {"kind": kind, "model": "scaled", "batch": _log(rng, 1, 8),
                    "prompt": _log(rng, 100, 2048), "ragged": rng.random() < 0.3,
                    "bf16": rng.random() < 0.4}
        return {"kind": kind, "model": rng.choice(["hall", "hall", "pidgeon"]),
                "batch": _log(rng, 1, 16), "prompt": _log(rng, 16, 512),
                "ragged": rng.random() < 0.4, "bf16": False}
    if kind == "forward":
        return {"kind": kind, "model": rng.choice(["hall", "pidgeon"]), "batch": _log(rng, 1, 16),
                "prompt": _log(rng, 16, 512)}
    if kind == "nodes":
        return {"kind": kind, "model": rng.choice(["hall", "pidgeon"]),
                "prompt": _log(rng, 8, 200), "steps": rng.randint(4, 8)}
    return {"kind": kind, "rows": _log(rng, 1, 32), "vocab": _log(rng, 5000, 50257),
            "seen": rng.choice([0, rng.randint(1, 480)]),
            "temperature": rng.choice([0.0, 0.7, 0.8, 1.0]), "top_k": rng.choice([0, 0, 10, 40]),
            "top_p": rng.choice([0.9, 0.95, 1.0]), "penalty": rng.choice([1.0, 1.15])}


def _config(name):
    c = akasha.ModelConfig
    if name == "scaled":
        return replace(c.scaled(), num_layers=2)
    return c.pidgeon() if name == "pidgeon" else c.akasha_hall_1()


def _device_weights(name, dtype=torch.float32):
    """Matrices N(0, 0.02) and gains 1 + N(0, 0.02), in params() order; the
    scaled model's values are bfloat16."""
    g = torch.Generator(device="cuda").manual_seed(sum(map(ord, name)))
    out = []
    for shape in _config(name).param_shapes():
        a = torch.randn(shape, generator=g, device="cuda") * 0.02
        if len(shape) == 1:
            a += 1.0
        if name == "scaled":
            a = a.bfloat16().float()
        out.append(a.to(dtype))
    return out


def _host_weights(name):
    if name not in _weights:
        _weights.clear()
        _weights[name] = [a.cpu().numpy() for a in _device_weights(name)]
    return _weights[name]


def _the_backend():
    global _backend
    if _backend is None:
        _backend = hip.Backend(0)
    return _backend


def _model(name, bf16=False):
    key = (name, bf16)
    if key not in _models:
        while len(_models) >= 2:
            _models.popitem(last=False)
        m = hip.Model(_the_backend(), _config(name))
        m.upload(_host_weights(name))
        if bf16:
            m.set_prefill_bf16(True)
        _models[key] = m
    _models.move_to_end(key)
    return _models[key]


def _lengths(case):
    """The prompts' lengths: of ragged ones, from a fifth of the longest up,
    the same for every seed."""
    b, p = case["batch"], case["prompt"]
    if not case.get("ragged") or b == 1:
        return [p] * b
    low = max(1, p // 5)
    return [p - (i * 7919) % (p - low + 1) for i in range(b)]


def _tokens(case, seed, count):
    rng = np.random.default_rng([seed, 1])
    return rng.integers(0, _config(case["model"]).vocab_size, size=count, dtype=np.uint32)


def _prompts(case, seed):
    lens = _lengths(case)
    t = _tokens(case, seed, sum(lens))
    if case.get("ragged"):
        return np.split(t, np.cumsum(lens)[:-1])
    return t.reshape(case["batch"], -1)


def _sample_inputs(case, seed):
    """Logits N(0, 2^2), as an untrained or a well-spread model's, the history
    of ids already generated and one uniform draw per row."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    rows, n, h = case["rows"], case["vocab"], case["seen"]
    logits = torch.randn(rows, n, generator=g, device="cuda") * 2
    seen = torch.randint(0, n, (rows, max(h, 1)), generator=g, device="cuda").to(torch.int32)
    seen_len = torch.full((rows,), h, dtype=torch.int32, device="cuda")
    uni = torch.rand(rows, generator=g, device="cuda", dtype=torch.float64)
    return logits, seen, seen_len, uni


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sample":
        _the_backend()
        logits, seen, seen_len, uni = _sample_inputs(case, seed)
        out = torch.zeros(case["rows"], dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        return {"case": case, "logits": logits, "seen": seen, "seen_len": seen_len, "uni": uni,
                "out": out}
    cfg = _config(case["model"])
    if kind == "nodes":
        d = akasha.shader_graph.ShaderDecoder(hip, _the_backend(), cfg,
                                              _host_weights(case["model"]), cfg.seq_len)
        t = _tokens(case, seed, case["prompt"] + case["steps"])
        return {"case": case, "decoder": d, "prompt": t[:case["prompt"]].tolist(),
                "next": t[case["prompt"]:].tolist()}
    model = _model(case["model"], case.get("bf16", False))
    if kind == "forward":
        f = hip.Forward(model, case["batch"], case["prompt"])
        t = _tokens(case, seed, 2 * case["batch"] * case["prompt"])
        return {"case": case, "forward": f, "tokens": t[::2].copy(), "targets": t[1::2].copy()}
    prompts = _prompts(case, seed)
    s = hip.Session(model, cfg.seq_len, case["batch"])
    if kind == "decode":
        if case["kv16"]:
            s.set_kv_bf16(True)
        s.prefill(prompts, want_logits=False)
        s.decode_greedy(1, want_tokens=False)  # the step's graph
    return {"case": case, "session": s, "prompts": prompts}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        s = state["session"]
        s.truncate(case["prompt"])
        tokens = s.decode_greedy(case["steps"] - 1)
        logits, last = s.decode_step(None)
        return {"tokens": np.vstack([tokens, last[None]]).astype(np.int64), "logits": logits}
    if kind == "prefill":
        s = state["session"]
        s.reset()
        logits, tokens = s.prefill(state["prompts"])
        return {"tokens": tokens.astype(np.int64), "logits": logits}
    if kind == "forward":
        mean, losses = state["forward"].loss(state["tokens"], state["targets"])
        return {"mean": mean, "losses": losses}
    if kind == "nodes":
        d = state["decoder"]
        d.reset()
        return [d.prefill(state["prompt"])] + [d.decode_step(t) for t in state["next"]]
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    seen = case["seen"] > 0
    _backend.sample_rows(p(state["logits"]), case["rows"], case["vocab"], p(state["out"]),
                         temperature=case["temperature"], top_k=case["top_k"],
                         top_p=case["top_p"], repetition_penalty=case["penalty"],
                         seen=p(state["seen"]) if seen else None, seen_stride=case["seen"],
                         seen_len=p(state["seen_len"]) if seen else None, uniforms=p(state["uni"]))
    return state["out"]


def work(case):
    """Each weight, cached row, logit and token id once; two operations per
    multiply-add of the matrices and of the causal attention."""
    kind = case["kind"]
    if kind == "sample":
        n = case["rows"] * case["vocab"]
        return {"bytes": 4 * n + 4 * case["rows"] * (case["seen"] + 3), "flops": n}
    c = _config(case["model"])
    d, v, n_layers = c.dim, c.vocab_size, c.num_layers
    layers = n_layers * (4 * d * d + 2 * d * c.ffn_hidden)
    weight = 2 if case["model"] == "scaled" else 4
    kv = 2 if case.get("kv16") else 4

    def decode(batch, at, steps):
        rows = sum(at + i + 1 for i in range(steps))
        return {"bytes": steps * (weight * (layers + d * v) + 4 * batch * (d + v))
                + kv * 2 * n_layers * batch * d * (rows + steps),
                "flops": 2 * steps * batch * (layers + d * v) + 4 * n_layers * batch * d * rows}

    def rows_of(lens, heads):
        rows = sum(lens)
        return {"bytes": weight * (layers + d * v) + 4 * d * rows + 4 * 2 * n_layers * d * rows
                + 4 * heads * v,
                "flops": 2 * rows * layers + 2 * heads * d * v
                + 2 * n_layers * d * sum(x * (x + 1) for x in lens)}

    if kind == "decode":
        return decode(case["batch"], case["prompt"], case["steps"])
    if kind == "prefill":
        return rows_of(_lengths(case), case["batch"])
    if kind == "forward":
        w = rows_of([case["prompt"]] * case["batch"], case["batch"] * case["prompt"])
        # The loss needs neither the cache nor the logits in memory.
        rows = case["batch"] * case["prompt"]
        w["bytes"] = weight * (layers + d * v) + 4 * d * rows + 12 * rows
        return w
    a, b = rows_of([case["prompt"]], 1), decode(1, case["prompt"], case["steps"])
    return {k: a[k] + b[k] for k in a}


def tolerance(case):
    """About four times the error measured against exact(): 3.9e-3 with
    bfloat16 kernels, 1.8e-3 with a bfloat16 cache, 1e-6 in 32 bits, 1.6e-6
    for the mean loss, which is summed in order in 32 bits."""
    if case["kind"] == "sample":
        return "exact"
    if case.get("bf16"):
        return {"rel": 1.5e-2, "max": 8e-2, "differ": 0.01}
    if case.get("kv16"):
        return {"rel": 7e-3, "max": 4e-2, "differ": 0.01}
    if case["kind"] == "forward":
        return {"rel": 7e-6, "max": 5e-5}
    return {"rel": 5e-6, "max": 5e-5, "differ": 0.01}


def _norm64(x, gain, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * gain


def _rope64(x, at, head):
    """Adjacent pairs of each head turned by at * 10000^(-2i/head), the angle
    taken in 32 bits as the model defines it."""
    i = torch.arange(0, head, 2, dtype=torch.float64, device=x.device) / head
    inv = 1.0 / torch.pow(10000.0, i).float()
    pos = torch.arange(at, at + x.shape[-2], device=x.device).float()
    angle = (pos[:, None] * inv).double()
    cos, sin = angle.cos(), angle.sin()
    p = x.unflatten(-1, (-1, head // 2, 2))
    a, b = p[..., 0], p[..., 1]
    cos, sin = cos[:, None], sin[:, None]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-3)


def _rows64(c, w, tokens, cache, at):
    """Final normed rows [B, S, d] of tokens [B, S] at position `at`, with
    cache[l] = (K, V) of [B, ctx, d] written and attended to."""
    d, head, heads = c.dim, c.head_dim, c.num_heads
    s = tokens.shape[1]
    x = w[0][tokens]
    for layer in range(c.num_layers):
        n1, qkv, wo, n2, up, down = w[1 + 6 * layer:7 + 6 * layer]
        q, k, v = (_norm64(x, n1, c.norm_eps) @ qkv).split(d, -1)
        kc, vc = cache[layer]
        kc[:, at:at + s], vc[:, at:at + s] = _rope64(k, at, head), v
        split = lambda t: t.unflatten(-1, (heads, head)).transpose(1, 2)  # noqa: E731
        q, k, v = split(_rope64(q, at, head)), split(kc[:, :at + s]), split(vc[:, :at + s])
        score = (q @ k.transpose(-1, -2)) / head ** 0.5
        if s > 1:
            mask = torch.ones(s, at + s, dtype=torch.bool, device=x.device).tril(at)
            score = score.masked_fill(~mask, float("-inf"))
        x = x + (score.softmax(-1) @ v).transpose(1, 2).flatten(-2) @ wo
        h = _norm64(x, n2, c.norm_eps) @ up
        x = x + (h * torch.sigmoid(h)) @ down
    return _norm64(x, w[-2], c.norm_eps)


def _cache64(c, batch, rows):
    z = lambda: torch.zeros(batch, rows, c.dim, dtype=torch.float64, device="cuda")  # noqa: E731
    return [(z(), z()) for _ in range(c.num_layers)]


def _on_gpu(a):
    return torch.from_numpy(np.asarray(a, np.int64)).cuda()


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None
    c = _config(case["model"])
    w = _device_weights(case["model"], torch.float64)
    if kind == "forward":
        t = _tokens(case, seed, 2 * case["batch"] * case["prompt"])
        tokens = _on_gpu(t[::2]).reshape(case["batch"], -1)
        targets = _on_gpu(t[1::2]).reshape(case["batch"], -1)
        losses = []
        for b in range(case["batch"]):
            x = _rows64(c, w, tokens[b:b + 1], _cache64(c, 1, case["prompt"]), 0)[0] @ w[-1]
            losses.append(x.logsumexp(-1) - x.gather(-1, targets[b][:, None])[:, 0])
        losses = torch.cat(losses)
        return {"mean": float(losses.mean()), "losses": losses}
    if kind == "nodes":
        t = _on_gpu(_tokens(case, seed, case["prompt"] + case["steps"]))[None]
        x = _rows64(c, w, t, _cache64(c, 1, t.shape[1]), 0)[0]
        return list(x[case["prompt"] - 1:] @ w[-1])
    if kind == "prefill":
        rows = [_rows64(c, w, _on_gpu(p)[None], _cache64(c, 1, len(p)), 0)[0, -1]
                for p in _prompts(case, seed)]
        return {"tokens": None, "logits": torch.stack(rows) @ w[-1]}
    prompts, end = _on_gpu(_prompts(case, seed)), case["prompt"] + case["steps"]
    cache = _cache64(c, case["batch"], end)
    rows = [_rows64(c, w, prompts[b:b + 1], [(k[b:b + 1], v[b:b + 1]) for k, v in cache], 0)[0, -1]
            for b in range(case["batch"])]
    logits = torch.stack(rows) @ w[-1]
    for i in range(case["steps"]):
        token = logits.argmax(-1)
        logits = _rows64(c, w, token[:, None], cache, case["prompt"] + i)[:, 0] @ w[-1]
    return {"tokens": None, "logits": logits}
