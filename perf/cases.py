"""The work a program built on this framework has it do, as cases to time.

One Bonsai token or prompt chunk passes through five kinds of call, and each
kind is a case of its own:

* ``decode_attn``   the fused attention step of one token, layer after layer;
* ``decode_proj``   the four Q1_0 matvecs of each layer for one token;
* ``head``          final norm + LM head, top-k over the logits, its readback;
* ``prefill_attn``  the fused attention step of a prompt chunk, one layer;
* ``prefill_proj``  quantize + Q1_0 x Q8_0 matmuls of a layer for a chunk;

and ``decode_token`` is a whole decode token, all of the first three in order.
Attention shapes are Config's (32 query heads on 8 KV heads of 128, 36 layers),
the projections' sizes Bonsai-4B's (2560 / 9728 / 151936) or generic ones.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bonsai-pot_amd"))
from bonsai_pot_amd import Config, Model  # noqa: E402

HD, GROUP = 128, 4
CHUNK_ROWS = 16384   # cache rows written per call while a cache is filled


def listed():
    return [
        # The first tokens of a chat: every layer's attention over a short cache.
        {"name": "decode_attn_300", "kind": "decode_attn", "layers": 36, "n_kv": 8, "pos": 300},
        # The usual context: the benchmark's headline step.
        {"name": "decode_attn_4096", "kind": "decode_attn", "layers": 36, "n_kv": 8, "pos": 4096},
        # A long document; four layers' caches already exceed the on-chip caches.
        {"name": "decode_attn_32768", "kind": "decode_attn", "layers": 4, "n_kv": 8, "pos": 32768},
        # One decode token's projections, wider than 4B's, over eight layers.
        {"name": "decode_proj_wide", "kind": "decode_proj", "layers": 8, "hidden": 4096, "q": 4096, "kv": 1024,
         "ffn": 12288, "arith": "f16"},
        # The end of every decoded token: logits, top-k, values on the host.
        {"name": "head_151936", "kind": "head", "hidden": 2560, "vocab": 151936, "topk": 32, "arith": "f16"},
        # A whole token of Bonsai-4B at an ordinary position.
        {"name": "decode_token_4b", "kind": "decode_token", "layers": 36, "hidden": 2560, "q": 4096, "kv": 1024,
         "ffn": 9728, "vocab": 151936, "topk": 32, "pos": 1000},
        # The reference's longest prompt chunk, from an empty cache.
        {"name": "prefill_attn_512", "kind": "prefill_attn", "n_kv": 8, "m": 512, "pos": 0},
        # A long prompt in one chunk: the benchmark's prefill metric.
        {"name": "prefill_attn_2048", "kind": "prefill_attn", "n_kv": 8, "m": 2048, "pos": 0},
        # A later chunk of a prompt whose length no tile divides.
        {"name": "prefill_attn_777_on_1501", "kind": "prefill_attn", "n_kv": 8, "m": 777, "pos": 1501},
        # A chat turn: a few tokens over a long history.
        {"name": "prefill_attn_64_on_16384", "kind": "prefill_attn", "n_kv": 8, "m": 64, "pos": 16384},
        # All projections of one Bonsai-4B layer for a full chunk.
        {"name": "prefill_proj_512", "kind": "prefill_proj", "hidden": 2560, "q": 4096, "kv": 1024, "ffn": 9728,
         "m": 512},
        # The same for a chat turn of a few words.
        {"name": "prefill_proj_33", "kind": "prefill_proj", "hidden": 2560, "q": 4096, "kv": 1024, "ffn": 9728,
         "m": 33},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode_attn", "decode_attn", "decode_proj", "head", "prefill_attn", "prefill_attn",
                       "prefill_attn", "prefill_proj", "prefill_proj", "decode_token"])
    n_kv = rng.choice([8, 8, 8, 4, 12])
    if kind == "decode_attn":
        pos = _log_int(rng, 1, 40000)
        return {"kind": kind, "layers": max(1, min(36, 130000 // max(pos, 1))), "n_kv": n_kv, "pos": pos}
    if kind == "prefill_attn":
        m = _log_int(rng, 2, 2048)
        pos = rng.choice([0, 1]) * _log_int(rng, 1, min(20000, max(2, 4000000 // m - m // 2)))
        return {"kind": kind, "n_kv": n_kv, "m": m, "pos": pos}
    hidden = 128 * rng.randint(8, 32)
    ffn = 128 * rng.randint(2 * hidden // 128, 4 * hidden // 128)
    if kind == "head":
        return {"kind": kind, "hidden": hidden, "vocab": 16 * _log_int(rng, 500, 9500),
                "topk": rng.choice([1, 8, 20, 32]), "arith": rng.choice(["f16", "f16", "auto"])}
    if kind == "prefill_proj":
        hidden = 128 * rng.randint(8, 20)
        ffn = 128 * rng.randint(2 * hidden // 128, 76)
        return {"kind": kind, "hidden": hidden, "q": 512 * rng.randint(4, 8), "kv": 128 * rng.randint(2, 8),
                "ffn": ffn, "m": _log_int(rng, 2, 512)}
    if kind == "decode_proj":
        return {"kind": kind, "layers": rng.randint(2, 10), "hidden": hidden, "q": 512 * rng.randint(4, 8),
                "kv": 128 * rng.randint(2, 8), "ffn": min(ffn, 16384), "arith": rng.choice(["f16", "f16", "f16", "mfma"])}
    hidden = 128 * rng.randint(8, 20)
    return {"kind": kind, "layers": rng.randint(2, 24), "hidden": hidden, "q": 512 * 8, "kv": 128 * 8,
            "ffn": 128 * rng.randint(2 * hidden // 128, 76), "vocab": 16 * _log_int(rng, 2000, 9000), "topk": 32,
            "pos": _log_int(rng, 1, 8000)}


# ---- inputs, from the seed alone ------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(torch.float16)


def _norm_w(g, n):
    """Norm weights around 1, as trained ones are."""
    return (1.0 + 0.2 * torch.randn(n, generator=g, device="cuda")).to(torch.float16)


def _same_size_w(g, n):
    """Head-norm weights of one magnitude. The fused attention steps normalize
    q in place, so a pass repeated on the same state normalizes it again: with
    weights of one magnitude q keeps its distribution however often."""
    return torch.where(torch.rand(n, generator=g, device="cuda") < 0.5, -1.5, 1.5).to(torch.float16)


class _Weights:
    """Q1_0 tensors one after the other in one buffer: per tensor the f16 scales
    [n][k/128], then the sign bits [n][k/128][16 bytes]."""

    def __init__(self, g):
        self.g, self.parts, self.at = g, [], 0

    def _put(self, t):
        pad = -t.numel() % 64
        self.parts += [t, torch.zeros(pad, dtype=torch.uint8, device="cuda")]
        at, self.at = self.at, self.at + t.numel() + pad
        return at

    def tensor(self, n, k):
        size = (0.5 + torch.rand(n, k // 128, generator=self.g, device="cuda")) / math.sqrt(k)
        d = self._put(size.to(torch.float16).view(torch.uint8).reshape(-1))
        qs = self._put(torch.randint(0, 256, (n * k // 8,), generator=self.g, device="cuda", dtype=torch.uint8))
        return {"n": n, "k": k, "d": d, "qs": qs}

    def buffer(self):
        return torch.cat(self.parts)


def _layer_weights(w, c):
    t = w.tensor
    return {"q": t(c["q"], c["hidden"]), "k": t(c["kv"], c["hidden"]), "v": t(c["kv"], c["hidden"]),
            "o": t(c["hidden"], c["q"]), "gate": t(c["ffn"], c["hidden"]), "up": t(c["ffn"], c["hidden"]),
            "down": t(c["hidden"], c["ffn"])}


class _Regions:
    """Element offsets of named f16 regions of the activation buffer."""

    def __init__(self):
        self.at, self.size = {}, 0

    def add(self, name, n):
        self.at[name] = self.size
        self.size += (n + 63) // 64 * 64

    def of(self, act, name, *shape):
        return act[self.at[name]:self.at[name] + math.prod(shape)].view(*shape)


class _DeviceMemory:
    """Lets torch view memory that the model owns; the view keeps the model."""

    def __init__(self, model, ptr, nbytes):
        self.model = model
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1", "data": (ptr, False), "version": 2}


def _cache_rows(model, first, n):
    """Views of cache rows [first, first + n) of every layer: qs and d of K and V."""
    cfg, out = model.cfg, {}
    *buffers, nbytes = model.kv_buffers()
    for name, ptr in zip("kv", buffers):
        mem = torch.as_tensor(_DeviceMemory(model, ptr, nbytes), device="cuda")
        nd = cfg.n_layer * model.max_seq * (cfg.kv_dim // 32) * 4
        out[name + "_d"] = mem[:nd].view(torch.float32).view(cfg.n_layer, model.max_seq, -1)[:, first:first + n]
        out[name + "_qs"] = mem[nd:].view(torch.int8).view(cfg.n_layer, model.max_seq, -1)[:, first:first + n]
    return out


def _with_arith(arith, make):
    """Model options are read from the environment when a model is created."""
    was = os.environ.get("BP_MATVEC_ARITH")
    os.environ["BP_MATVEC_ARITH"] = arith
    try:
        return make()
    finally:
        if was is None:
            del os.environ["BP_MATVEC_ARITH"]
        else:
            os.environ["BP_MATVEC_ARITH"] = was


def _history(case, seed, layer, lo, n, kv_dim):
    """Raw f16 K and V of cached rows [lo, lo + n) of one layer."""
    g = _gen(seed * 1000003 + layer * 4099 + lo)
    kv = torch.randn(2, n, kv_dim, generator=g, device="cuda", dtype=torch.float32)
    return kv[0].to(torch.float16), kv[1].to(torch.float16)


def _fill_cache(model, case, seed, w_norms, w_k_off, layers, pos):
    kv_dim = model.cfg.kv_dim
    for il in range(layers):
        for lo in range(0, pos, CHUNK_ROWS):
            n = min(CHUNK_ROWS, pos - lo)
            both = torch.cat([t.reshape(-1) for t in _history(case, seed, il, lo, n, kv_dim)])
            model.dispatch_kv_writeback_fused(both.data_ptr(), w_norms.data_ptr(), 0, n * kv_dim, w_k_off, il, lo, n)
            torch.cuda.synchronize()


def _round64(n):
    return (n + 63) // 64 * 64


def _attn_inputs(case, seed):
    """(w_norms = [w_q | w_k], q, k, v) of the new tokens, [layers][m][...]."""
    layers, m = case.get("layers", 1), case.get("m", 1)
    g = _gen(seed)
    w = torch.cat([_same_size_w(g, HD), _norm_w(g, HD)])
    kv_dim = case["n_kv"] * HD
    return w, _randn(g, layers, m, GROUP * kv_dim), _randn(g, layers, m, kv_dim), _randn(g, layers, m, kv_dim)


def _prepare_attn(case, seed):
    layers, m, pos, n_kv = case.get("layers", 1), case.get("m", 1), case["pos"], case["n_kv"]
    w, q, k, v = _attn_inputs(case, seed)
    cfg = Config(n_layer=layers, n_head=GROUP * n_kv, n_kv_head=n_kv)
    r = _Regions()
    for name, t in (("q", q), ("k", k), ("v", v), ("out", q)):
        r.add(name, t.numel())
    act = torch.zeros(r.size, dtype=torch.float16, device="cuda")
    for name, t in (("q", q), ("k", k), ("v", v)):
        r.of(act, name, *t.shape).copy_(t)
    model = Model(cfg, _round64(pos + m))
    model.set_stream(torch.cuda.current_stream().cuda_stream)
    _fill_cache(model, case, seed, w, HD, layers, pos)
    out = {"out": r.of(act, "out", *q.shape), "q": r.of(act, "q", *q.shape), **_cache_rows(model, pos, m)}
    return {"case": case, "model": model, "act": act, "w": w, "r": r, "outputs": out}


def _run_attn(s):
    c, model, at = s["case"], s["model"], s["r"].at
    m, pos, kv = c.get("m", 1), c["pos"], model.cfg.kv_dim
    act, w = s["act"].data_ptr(), s["w"].data_ptr()
    for il in range(c.get("layers", 1)):
        q, k, v, out = at["q"] + il * m * GROUP * kv, at["k"] + il * m * kv, at["v"] + il * m * kv, at["out"] + il * m * GROUP * kv
        if c["kind"] == "decode_attn":
            model.dispatch_attention_decode_step(act, w, q, k, v, out, 0, HD, il, pos)
        else:
            model.dispatch_attention_prefill_step(act, w, q, k, v, out, 0, HD, il, pos, m)
    return s["outputs"]


# ---- projections, head and whole tokens ------------------------------------------
def _token_inputs(case, seed):
    """Everything a decode token's calls read, by kind."""
    g = _gen(seed)
    w = _Weights(g)
    s = {"layers": [_layer_weights(w, case) for _ in range(case.get("layers", 0))]}
    if "vocab" in case:
        s["head"] = w.tensor(case["vocab"], case["hidden"])
    s["weights"] = w.buffer()
    # per layer: attention norm, FFN norm, head norms of q and k; then the final norm
    h = case["hidden"]
    s["norms"] = _norm_w(g, (case.get("layers", 0) * (2 * h + 2 * HD)) + h)
    s["x"] = _randn(g, h)
    if case["kind"] == "decode_proj":
        s["attn_out"] = _randn(g, case["layers"], case["q"])
    return s


def _prepare_token(case, seed):
    s = _token_inputs(case, seed)
    h, layers = case["hidden"], case.get("layers", 0)
    r = _Regions()
    r.add("res", h)
    if layers:
        per = layers if case["kind"] == "decode_proj" else 1
        for name, n in (("q", case["q"]), ("k", case["kv"]), ("v", case["kv"]), ("attn", per * case["q"]),
                        ("gate", case["ffn"]), ("up", case["ffn"])):
            r.add(name, n)
    if "vocab" in case:
        r.add("logits", case["vocab"])
    act = torch.zeros(r.size, dtype=torch.float16, device="cuda")
    r.of(act, "res", h).copy_(s["x"])
    if case["kind"] == "decode_proj":
        r.of(act, "attn", layers, case["q"]).copy_(s["attn_out"])
    pos = case.get("pos", 0)
    n_kv = case.get("kv", 1024) // HD if case["kind"] == "decode_token" else 8
    cfg = Config(n_layer=max(1, layers if case["kind"] == "decode_token" else 1), n_head=GROUP * n_kv, n_kv_head=n_kv)
    model = _with_arith(case.get("arith", "f16"), lambda: Model(cfg, _round64(pos + 1)))
    model.set_stream(torch.cuda.current_stream().cuda_stream)
    if case["kind"] == "decode_token":
        _fill_cache(model, case, seed, s["norms"], 2 * h + HD, layers, pos)
    s.update(case=case, model=model, act=act, r=r, result=torch.zeros(64, dtype=torch.int32, device="cuda"))
    return s


def _matvec(s, t, src, dst, accumulate):
    s["model"].dispatch_matvec_q1_0(s["weights"].data_ptr(), s["act"].data_ptr(), t["k"], t["n"], t["d"], t["qs"], src,
                                    dst, accumulate)


def _normed(s, w_off, *to):
    at = s["r"].at
    s["model"].dispatch_matvec_q1_0_fused_normed(
        s["weights"].data_ptr(), s["act"].data_ptr(), s["norms"].data_ptr(), to[0][0]["k"], at["res"], w_off,
        [(t["d"], t["qs"], t["n"], at[dst]) for t, dst in to])


def _run_layers(s):
    c, model, at = s["case"], s["model"], s["r"].at
    h = c["hidden"]
    s["act"][at["res"]:at["res"] + h].copy_(s["x"])   # the token's embedding row
    for il, t in enumerate(s["layers"]):
        n = il * (2 * h + 2 * HD)
        _normed(s, n, (t["q"], "q"), (t["k"], "k"), (t["v"], "v"))
        attn = at["attn"]
        if c["kind"] == "decode_token":
            model.dispatch_attention_decode_step(s["act"].data_ptr(), s["norms"].data_ptr(), at["q"], at["k"], at["v"],
                                                 attn, n + 2 * h, n + 2 * h + HD, il, c["pos"])
        else:
            attn += il * c["q"]
        _matvec(s, t["o"], attn, at["res"], True)
        _normed(s, n + h, (t["gate"], "gate"), (t["up"], "up"))
        d = t["down"]
        model.dispatch_matvec_q1_0_silu(s["weights"].data_ptr(), s["act"].data_ptr(), d["k"], d["n"], d["d"], d["qs"],
                                        at["gate"], at["up"], at["res"], True)


def _run_head(s):
    c, model, at = s["case"], s["model"], s["r"].at
    _normed(s, len(s["layers"]) * (2 * c["hidden"] + 2 * HD), (s["head"], "logits"))
    model.dispatch_topk_reduce(s["act"].data_ptr(), s["result"].data_ptr(), c["vocab"], c["topk"], at["logits"], 0)
    return model.wait_topk_readback(s["result"].data_ptr(), 0, c["topk"])


def _run_token(s):
    c, r, act = s["case"], s["r"], s["act"]
    out = {}
    if c["kind"] != "head":
        _run_layers(s)
        for name, n in (("res", c["hidden"]), ("q", c["q"]), ("k", c["kv"]), ("v", c["kv"]), ("gate", c["ffn"]),
                        ("up", c["ffn"])):
            out[name] = r.of(act, name, n)
    if c["kind"] != "decode_proj":
        values, indices = _run_head(s)
        out["logits"] = r.of(act, "logits", c["vocab"])
        out["top_values"] = values
        if c["kind"] == "head":   # after 36 layers near ties may fall either way
            out["top_indices"] = indices.astype(np.int64)
    if c["kind"] == "decode_token":
        out["attn"] = r.of(act, "attn", c["q"])
    return out


def _prefill_inputs(case, seed):
    g = _gen(seed)
    w = _Weights(g)
    t = _layer_weights(w, case)
    m = case["m"]
    # the normed residual (twice), the attention output and silu(gate) * up
    return {"t": t, "weights": w.buffer(), "res": _randn(g, m, case["hidden"]), "xn": _randn(g, m, case["hidden"]),
            "attn": _randn(g, m, case["q"]), "xf": _randn(g, m, case["hidden"]),
            "ffn": _randn(g, m, case["ffn"]) * _randn(g, m, case["ffn"])}


def _prepare_prefill_proj(case, seed):
    s = _prefill_inputs(case, seed)
    m, r = case["m"], _Regions()
    for name in ("res", "xn", "attn", "xf", "ffn"):
        r.add(name, s[name].numel())
    for name in ("q", "k", "v", "gate", "up"):
        r.add(name, m * s["t"][name]["n"])
    act = torch.zeros(r.size, dtype=torch.float16, device="cuda")
    for name in ("res", "xn", "attn", "xf", "ffn"):
        r.of(act, name, *s[name].shape).copy_(s[name])
    model = Model(Config(n_layer=1), 64)
    model.set_stream(torch.cuda.current_stream().cuda_stream)
    k = max(case["hidden"], case["q"], case["ffn"])
    q8 = torch.zeros(m * k // 32 * 4 + m * k, dtype=torch.uint8, device="cuda")
    outputs = {n: r.of(act, n, m, s["t"][n]["n"]) for n in ("q", "k", "v", "gate", "up")}
    outputs["res"] = r.of(act, "res", m, case["hidden"])
    return {"case": case, "model": model, "act": act, "q8": q8, "r": r, "t": s["t"], "weights": s["weights"],
            "outputs": outputs}


def _run_prefill_proj(s):
    model, at, m = s["model"], s["r"].at, s["case"]["m"]
    act, q8, weights = s["act"].data_ptr(), s["q8"].data_ptr(), s["weights"].data_ptr()
    for src, to, accumulate in (("xn", "qkv", False), ("attn", "o", True), ("xf", ("gate", "up"), False),
                                ("ffn", ("down",), True)):
        k = s["t"][to[0]]["k"]
        model.dispatch_quantize_act(act, q8, k, m, at[src], 0, m * k // 32 * 4)
        for name in to:
            t = s["t"][name]
            model.dispatch_matmul_q1_0(weights, q8, act, k, t["n"], m, t["d"], t["qs"], 0, m * k // 32 * 4,
                                       at["res" if accumulate else name], accumulate)
    return s["outputs"]


# ---- the interface -----------------------------------------------------------------
def prepare(case, seed):
    if case["kind"].endswith("_attn"):
        return _prepare_attn(case, seed)
    if case["kind"] == "prefill_proj":
        return _prepare_prefill_proj(case, seed)
    return _prepare_token(case, seed)


def run(state):
    kind = state["case"]["kind"]
    if kind.endswith("_attn"):
        return _run_attn(state)
    if kind == "prefill_proj":
        return _run_prefill_proj(state)
    return _run_token(state)


def work(case):
    c, nbytes, flops = case, 0, 0

    def weights(n, k, m=1):
        return n * (k // 128) * 18, 2 * n * k * m

    if c["kind"].endswith("_attn") or c["kind"] == "decode_token":
        n_kv, m, layers = c.get("n_kv", c.get("kv", 0) // HD), c.get("m", 1), c.get("layers", 1)
        row = n_kv * (HD + 4 * HD // 32)   # one cache row of K or of V
        pairs = m * c["pos"] + m * (m + 1) // 2
        # cached rows read, new rows and q / k / v read, rows, q and out written
        nbytes += layers * (2 * c["pos"] * row + m * (2 * row + n_kv * HD * 2 * (3 * GROUP + 2)))
        flops += layers * 4 * HD * GROUP * n_kv * pairs
    if "ffn" in c:
        m = c.get("m", 1)
        h, q, kv, f = c["hidden"], c["q"], c["kv"], c["ffn"]
        for n, k in ((q + 2 * kv, h), (h, q), (2 * f, h), (h, f)):
            b, o = weights(n, k, m)
            nbytes += c.get("layers", 1) * (b + 2 * m * (n + k))
            flops += c.get("layers", 1) * o
    if "vocab" in c:
        b, o = weights(c["vocab"], c["hidden"])
        nbytes, flops = nbytes + b + 2 * (c["hidden"] + c["vocab"]) + 8 * c["topk"], flops + o
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"].endswith("_attn"):
        # q bits and cache rows are the same by contract; out is f16 of an f32 softmax
        return {"rel": 1.5e-3, "max": 0.02}
    if case["kind"] == "decode_token":
        # attention's roundings travel through the layers that follow
        return {"rel": 1e-2, "max": 0.2}
    if case.get("arith", "f16") != "f16":
        return {"rel": 1e-3, "max": 0.02, "differ": 0.01}
    return "exact"   # the order of every sum is part of these calls' contract


# ---- the same in 64 bits --------------------------------------------------------------
def _rope(x, pos0):
    """NEOX RoPE of x [m, heads, 128] at positions pos0 ..., f16 table."""
    j = torch.arange(HD // 2, dtype=torch.float64, device="cuda")
    angle = torch.arange(pos0, pos0 + x.shape[0], dtype=torch.float64, device="cuda")[:, None] * 1e6 ** (-2 * j / HD)
    c, s = (f(angle).float().half().double()[:, None] for f in (torch.cos, torch.sin))
    a, b = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w.double()


def _q8(x):
    """(dequantized, d) of x [..., n] in blocks of 32."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    q = torch.where(d > 0, torch.round(b / torch.where(d > 0, d, torch.ones_like(d))), torch.zeros_like(b))
    return (q * d).reshape(x.shape), d.squeeze(-1)


def _cache(case, seed, layer, n_kv, w_k, pos):
    """Dequantized K and V rows [0, pos) of a filled layer."""
    ks, vs = [], []
    for lo in range(0, pos, CHUNK_ROWS):
        n = min(CHUNK_ROWS, pos - lo)
        k, v = _history(case, seed, layer, lo, n, n_kv * HD)
        ks.append(_q8(_rope(_rms(k.double().view(n, n_kv, HD), w_k), lo))[0])
        vs.append(_q8(v.double().view(n, n_kv, HD))[0])
    empty = [torch.zeros(0, n_kv, HD, dtype=torch.float64, device="cuda")]
    return torch.cat(ks or empty), torch.cat(vs or empty)


def _exact_attn(case, seed, layer, q, k, v, w_q, w_k):
    """One layer's step in 64 bits: (out, q, k_d, v_d) of the m new tokens."""
    m, pos, n_kv = q.shape[0], case["pos"], k.shape[-1] // HD
    qn = _rope(_rms(q.double().view(m, GROUP * n_kv, HD), w_q), pos)
    kq, kd = _q8(_rope(_rms(k.double().view(m, n_kv, HD), w_k), pos))
    vq, vd = _q8(v.double().view(m, n_kv, HD))
    ck, cv = _cache(case, seed, layer, n_kv, w_k, pos)
    ck, cv = torch.cat([ck, kq]), torch.cat([cv, vq])
    mask = torch.arange(pos + m, device="cuda")[None] > pos + torch.arange(m, device="cuda")[:, None]
    out = torch.empty_like(qn)
    for h in range(GROUP * n_kv):
        p = qn[:, h] @ ck[:, h // GROUP].T / math.sqrt(HD)
        out[:, h] = torch.softmax(p.masked_fill(mask, -math.inf), -1) @ cv[:, h // GROUP]
    return out.reshape(m, -1), qn.reshape(m, -1), kd.reshape(m, -1), vd.reshape(m, -1)


def _dense(weights, t):
    n, k = t["n"], t["k"]
    d = weights[t["d"]:t["d"] + n * k // 64].view(torch.float16).double().view(n, k // 128, 1)
    qs = weights[t["qs"]:t["qs"] + n * k // 8].view(n, k // 128, 16, 1)
    bits = (qs >> torch.arange(8, dtype=torch.uint8, device="cuda")) & 1
    return ((2.0 * bits.view(n, k // 128, 128).double() - 1) * d).view(n, k)


def _exact_token(case, seed):
    s = _token_inputs(case, seed)
    h, x, out = case["hidden"], s["x"].double(), {}
    w, norms = s["weights"], s["norms"]
    for il, t in enumerate(s["layers"]):
        n = il * (2 * h + 2 * HD)
        xn = _rms(x, norms[n:n + h])
        out["q"], out["k"], out["v"] = (_dense(w, t[name]) @ xn for name in "qkv")
        if case["kind"] == "decode_token":
            w_q, w_k = norms[n + 2 * h:n + 2 * h + HD], norms[n + 2 * h + HD:n + 2 * h + 2 * HD]
            # every layer's cache was filled with the first layer's norm weights
            attn, q, _, _ = _exact_token_attn(case, seed, il, out, w_q, w_k, norms[2 * h + HD:2 * h + 2 * HD])
            out["q"], out["attn"] = q.view(-1), attn.view(-1)
            attn = out["attn"]
        else:
            attn = s["attn_out"][il].double()
        x = x + _dense(w, t["o"]) @ attn
        xn = _rms(x, norms[n + h:n + 2 * h])
        out["gate"], out["up"] = _dense(w, t["gate"]) @ xn, _dense(w, t["up"]) @ xn
        x = x + _dense(w, t["down"]) @ (out["gate"] * torch.sigmoid(out["gate"]) * out["up"])
        out["res"] = x
    if "head" in s:
        at = len(s["layers"]) * (2 * h + 2 * HD)
        xn = _rms(x, norms[at:at + h])
        out["logits"] = torch.cat([_dense(w, {**s["head"], "n": min(16384, case["vocab"] - lo),
                                              "d": s["head"]["d"] + lo * (h // 64),
                                              "qs": s["head"]["qs"] + lo * (h // 8)}) @ xn
                                   for lo in range(0, case["vocab"], 16384)])
        out["top_values"] = torch.topk(out["logits"], case["topk"]).values
    return out


def _exact_token_attn(case, seed, il, out, w_q, w_k, w_fill):
    n_kv, pos = case["kv"] // HD, case["pos"]
    q = _rope(_rms(out["q"].view(1, -1, HD), w_q), pos)
    kq, kd = _q8(_rope(_rms(out["k"].view(1, n_kv, HD), w_k), pos))
    vq, vd = _q8(out["v"].view(1, n_kv, HD))
    ck, cv = _cache(case, seed, il, n_kv, w_fill, pos)
    ck, cv = torch.cat([ck, kq]).transpose(0, 1), torch.cat([cv, vq]).transpose(0, 1)
    p = torch.softmax(q.view(n_kv, GROUP, HD) @ ck.transpose(1, 2).contiguous() / math.sqrt(HD), -1)
    return p @ cv.contiguous(), q, kd, vd


def exact(case, seed):
    if case["kind"].endswith("_attn"):
        w, q, k, v = _attn_inputs(case, seed)
        got = [_exact_attn(case, seed, il, q[il], k[il], v[il], w[:HD], w[HD:]) for il in range(case.get("layers", 1))]
        out, qn, kd, vd = (torch.stack(t) for t in zip(*got))
        return {"out": out, "q": qn, "k_d": kd, "k_qs": None, "v_d": vd, "v_qs": None}
    if case["kind"] == "prefill_proj":
        s = _prefill_inputs(case, seed)
        dense = {n: _dense(s["weights"], t) for n, t in s["t"].items()}
        x = {n: _q8(s[n].double())[0] for n in ("xn", "attn", "xf", "ffn")}
        out = {n: x["xn"] @ dense[n].T for n in "qkv"}
        out.update({n: x["xf"] @ dense[n].T for n in ("gate", "up")})
        out["res"] = s["res"].double() + x["attn"] @ dense["o"].T + x["ffn"] @ dense["down"].T
        return out
    return _exact_token(case, seed)
