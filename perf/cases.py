"""The performance cases of the attention path: what a program that serves models through gi_attn has it do.

A case is a dict of plain values:
  entry    "operator": attention() / attention_q4(), the operator of one layer over the reference's cache layout;
           "kernel": decode() / prefill() over head-major caches, what a program with its own layer loop calls;
           "layer": one layer's attention step as the engine runs it, qk_norm_rope and then the operator (and the
           rotation back for the 4-bit cache);
           "token": the same step of `layers` layers for one generated token, captured once into a HIP graph with the
           position in device memory and replayed, which is how a decode loop runs
  heads, kv_heads, hd, cache ("f16", "int8" or "q4")
  n        tokens of the call; pos: position of the first one (the keys before it are already in the cache)
  verify   the tokens are a speculative draft (the operator's exact flag)

listed() covers generated tokens over short and long contexts, a speculative block, a chat turn appended to a
conversation, chunks and whole prompts, in every cache format and in the head shapes of the models that the
repository's tests and benchmark use; draw() spreads sizes over the same ranges.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ghost-infer_amd"))
import gi_attn  # noqa: E402

BASE, EPS = 1e6, 1e-6
CAP_STEP = 4096  # sessions grow their caches in steps of 4096 positions


def _case(entry, heads, kv_heads, hd, cache, n, pos, name=None, verify=False, layers=1):
    c = dict(entry=entry, heads=heads, kv_heads=kv_heads, hd=hd, cache=cache, n=n, pos=pos, verify=verify, layers=layers)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one generated token of a 16-layer stretch of an 8B-class model over the default (int8) cache at an ordinary
        # chat length: many small launches in a row
        _case("token", 32, 8, 128, "int8", 1, 2900, "token_int8_3k", layers=16),
        # the smallest call: one token early in a conversation, issued call by call without a graph
        _case("operator", 32, 8, 128, "f16", 1, 700, "decode_f16_700"),
        # a long document: one token over 64K keys
        _case("kernel", 32, 4, 128, "f16", 1, 65535, "decode_f16_64k"),
        # the wide heads of hybrid models over the smallest cache format, long context
        _case("operator", 16, 2, 256, "q4", 1, 40000, "decode_h256_q4_40k"),
        # eight draft tokens checked at once over a long context
        _case("operator", 32, 4, 128, "int8", 8, 32768, "verify_int8_32k", verify=True),
        # a user's next message in a conversation: a few dozen tokens after some thousand
        _case("operator", 32, 8, 128, "int8", 57, 6100, "turn_int8_57_at_6k"),
        # a chunk of a long prompt, as chunked prefill issues it
        _case("kernel", 32, 4, 128, "f16", 512, 15872, "chunk_f16_512_at_16k"),
        # the longest whole prompt in one call
        _case("kernel", 32, 8, 128, "f16", 8192, 0, "prompt_f16_8k"),
        # an ordinary prompt through the whole step of a layer, default cache
        _case("layer", 32, 8, 128, "int8", 1500, 0, "layer_int8_1500"),
        # a longer prompt of a model with 256-wide heads over its 4-bit cache, the whole step with both rotations
        _case("layer", 16, 2, 256, "q4", 3000, 0, "layer_h256_q4_3000"),
        # a short prompt of a small model (3 query heads per kv head)
        _case("operator", 9, 3, 64, "f16", 300, 0, "prompt_h64_300"),
        # a follow-up of a model whose head size takes the f32 kernels
        _case("operator", 32, 32, 96, "f16", 200, 1800, "turn_h96_200_at_2k"),
    ]


#: (query heads, kv heads, head size, how often): the head shapes of the tests and the benchmark
SHAPES = [(32, 8, 128, 4), (32, 4, 128, 3), (16, 2, 256, 3), (32, 8, 64, 1), (9, 3, 64, 1), (32, 32, 80, 1), (32, 32, 96, 1)]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        heads, kv_heads, hd, _ = rng.choices(SHAPES, [s[3] for s in SHAPES])[0]
        cache = rng.choice(["f16", "int8"] + (["q4"] if hd == 256 else []))
        kind = rng.choice(["token", "decode", "verify", "turn", "chunk", "prompt"])
        layers, verify = 1, False
        if kind == "token":
            entry, n, pos, layers = "token", 1, _log(rng, 100, 32000), rng.choice([4, 8, 16])
        elif kind == "decode":
            entry, n, pos = rng.choice(["operator", "kernel"]), 1, _log(rng, 100, 65535)
        elif kind == "verify":
            entry, n, pos, verify = "operator", rng.randint(2, 12), _log(rng, 100, 40000), True
        elif kind == "turn":
            entry, n, pos = rng.choice(["operator", "layer"]), _log(rng, 16, 255), _log(rng, 200, 40000)
        elif kind == "chunk":
            entry, n, pos = rng.choice(["operator", "kernel", "layer"]), _log(rng, 256, 2048), _log(rng, 512, 32000)
        else:
            entry, n, pos = rng.choice(["operator", "kernel", "layer"]), _log(rng, 16, 8192), 0
        if entry == "kernel" and cache == "q4":
            entry = "operator"
        c = _case(entry, heads, kv_heads, hd, cache, n, pos, verify=verify, layers=layers)
        w = work(c)
        # no more than the largest listed case; the f32 kernels' matrix rate is a sixteenth
        if w["flops"] <= (3e10 if hd in (80, 96) else 5.5e11) and w["bytes"] <= 4.1e8:
            return c


def work(case):
    h, k, hd, n, pos = case["heads"], case["kv_heads"], case["hd"], case["n"], case["pos"]
    keys = n * pos + n * (n + 1) // 2
    row = hd * 2 if case["cache"] == "f16" else hd + 4 if case["cache"] == "int8" else hd // 2 + hd // 16
    qo = 4 if case["entry"] != "kernel" or n == 1 else 2  # bytes of a query and of an output value
    b = 2 * (pos + n) * k * row + 2 * n * h * hd * qo
    if case["entry"] in ("layer", "token"):
        b += n * (2 * (h + k) + k) * hd * 4 + 2 * n * k * row  # q | k | v rows read, q | k written, cache rows stored
    return {"bytes": case["layers"] * b, "flops": case["layers"] * 4 * h * hd * keys}


def tolerance(case):
    # Relative errors against 64 bits, measured, times about four. Decode keeps queries and probabilities to f32
    # (up to 1e-6), except at head size 256 over the int8 and 4-bit caches, which takes one f16 query and
    # probability as the prefill does (3e-4 to 5e-4); an f16 output adds its own rounding. The steps with RoPE carry
    # the f32 angle of their position (2e-5); a 4-bit value that falls to the other side of a rounding with it is a
    # whole step away (2e-3 over a prompt). So may stored bytes, which "differ" counts.
    one = case["n"] == 1 or case["verify"]
    f32 = case["hd"] in (80, 96) or one and (case["hd"] != 256 or case["cache"] == "f16")
    if case["entry"] in ("layer", "token"):
        return {"rel": 7e-3 if case["cache"] == "q4" else 1e-4 if f32 else 2e-3, "differ": 2e-3}
    f16_out = case["entry"] == "kernel" and not one
    return {"rel": 1e-5 if f32 and not f16_out else 1.5e-3}


def _cached(c):
    """Positions of the session's cache: whole growth steps."""
    return -(-(c["pos"] + c["n"]) // CAP_STEP) * CAP_STEP


def _quantise(x, cache):
    """Rows [..., hd] stored in the cache's format: (values, scales)."""
    if cache == "f16":
        return x.half(), None
    if cache == "int8":
        d = x.abs().amax(-1) / 127
        return (x / d[..., None]).round().to(torch.int8), d
    g = x.view(*x.shape[:-1], x.shape[-1] // 32, 32)
    d = (g.abs().amax(-1) / 7).half()
    q = ((g / d[..., None].float()).round().clamp(-7, 7) + 8).to(torch.uint8).view(*x.shape[:-1], x.shape[-1] // 2, 2)
    return (q[..., 0] | (q[..., 1] << 4)).contiguous(), d


def _widen(x, s, cache):
    """The 64-bit values that cache rows stand for."""
    if cache == "f16":
        return x.double()
    if cache == "int8":
        return x.double() * s.double()[..., None]
    q = torch.stack((x & 15, x >> 4), -1).view(*x.shape[:-1], -1, 32).float() - 8
    return (q * s.float()[..., None]).half().double().flatten(-2)


def prepare(case, seed):
    h, k, hd, n, pos, cache = (case[x] for x in ("heads", "kv_heads", "hd", "n", "pos", "cache"))
    L, dev, entry = case["layers"], torch.device("cuda"), case["entry"]
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)

    def randn(*shape):
        return torch.randn(shape, generator=gen, device=dev)

    cap = pos + n if entry == "kernel" else _cached(case)
    s = {"case": case}
    lay = (k, cap) if entry == "kernel" else (cap, k)  # head-major rows, or the reference's
    caches = [[_quantise(randn(*lay, hd), cache) for _ in "kv"] for _ in range(L)]
    s["kv"] = [(a[0], b[0]) for a, b in caches]
    s["scales"] = [(a[1], b[1]) for a, b in caches]
    if entry == "kernel":
        # queries as a rotary kernel of the program's own leaves them: f32 for one token, f16 for a prompt
        s["q"] = (2 * randn(n, h * hd)) if n == 1 else (2 * randn(n, h * hd)).half()
    else:
        # the layer's packed rows; queries a little peaked, as trained heads are
        s["qkv"] = [randn(n, (h + 2 * k) * hd) for _ in range(L)]
        if entry == "operator":
            s["qkv"][0][:, : h * hd] *= 2
    if entry in ("layer", "token"):
        s["qn"], s["kn"] = (torch.rand(hd, generator=gen, device=dev) * 1.5 + 0.5 for _ in "qk")
    if n == 1 or case["verify"]:  # a session keeps its decode workspace and rows
        s["ws"] = gi_attn.new_workspace(cap, n, h, k, hd, dev)
        s["out"] = [torch.empty((n, h * hd), device=dev) for _ in range(L)]
    if entry == "token":
        s["posp"] = torch.full((1,), pos, dtype=torch.int32, device=dev)
        s["rows"] = [r.clone() for r in s["qkv"]]  # stands for the projection that writes the step's rows

        def step():
            torch._foreach_copy_(s["qkv"], s["rows"])
            for i in range(L):
                _layer(s, i, posp=s["posp"], ctx_cap=cap)

        step()
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            step()
    return s


def _operator(s, i, **kw):
    c = s["case"]
    (kc, vc), (ks, vs) = s["kv"][i], s["scales"][i]
    if "out" in s:
        kw.update(out=s["out"][i], workspace=s["ws"])
    if c["cache"] == "q4":
        return gi_attn.attention_q4(s["qkv"][i], kc, vc, ks, vs, c["pos"], c["heads"], c["kv_heads"], exact=c["verify"], **kw)
    return gi_attn.attention(s["qkv"][i], kc, vc, c["pos"], c["heads"], c["kv_heads"], hd=c["hd"], exact=c["verify"],
                             k_scale=ks, v_scale=vs, **kw)


def _layer(s, i, **kw):
    c = s["case"]
    (kc, vc), (ks, vs) = s["kv"][i], s["scales"][i]
    rope = dict(base=BASE, qn=s["qn"], kn=s["kn"], eps=EPS, posp=kw.get("posp"))
    if c["cache"] == "q4":
        gi_attn.qk_norm_rope_q4(s["qkv"][i], kc, vc, ks, vs, c["pos"], c["heads"], c["kv_heads"], **rope)
        return gi_attn.hadamard_rows(_operator(s, i, **kw))
    gi_attn.qk_norm_rope(s["qkv"][i], kc, vc, c["pos"], c["heads"], c["kv_heads"], hd=c["hd"], k_scale=ks, v_scale=vs, **rope)
    return _operator(s, i, **kw)


def run(state):
    c = state["case"]
    if c["entry"] == "operator":
        return _operator(state, 0)
    if c["entry"] == "kernel":
        (kc, vc), (ks, vs) = state["kv"][0], state["scales"][0]
        kw = dict(hd=c["hd"], kv_layout="head_major", k_scale=ks, v_scale=vs)
        if c["n"] == 1:
            return gi_attn.decode(state["q"], kc, vc, c["pos"], c["heads"], c["kv_heads"], out=state["out"][0],
                                  workspace=state["ws"], **kw)
        return gi_attn.prefill(state["q"], kc, vc, c["pos"], c["heads"], c["kv_heads"], **kw)
    if c["entry"] == "token":
        state["graph"].replay()
        out = state["out"]
    else:
        out = [_layer(state, 0)]
    return {"out": out, "qkv": state["qkv"], "kv": [list(x) for x in state["kv"][:2]],
            "scales": [list(x) for x in state["scales"][:2] if x[0] is not None]}


def _attention64(q, k, v, pos, G):
    """q [n, heads, hd], k and v [kv_heads, keys, hd], all 64-bit -> [n, heads * hd]."""
    n, heads, hd = q.shape
    out = torch.empty_like(q)
    for h in range(heads):
        for r in range(0, n, 2048):
            e = min(n, r + 2048)
            last = pos + e
            s = q[r:e, h] @ k[h // G, :last].T / math.sqrt(hd)
            s.masked_fill_(torch.arange(last, device=q.device)[None] > torch.arange(pos + r, pos + e, device=q.device)[:, None], -math.inf)
            out[r:e, h] = torch.softmax(s, -1) @ v[h // G, :last]
    return out.view(n, -1)


def _hadamard64(x):
    m = torch.ones(1, 1, dtype=torch.float64, device=x.device)
    while m.shape[0] < x.shape[-1]:
        m = torch.cat((torch.cat((m, m), 1), torch.cat((m, -m), 1)))
    return x @ m / math.sqrt(m.shape[0])


def _rope64(x, w, pos):
    """x [n, heads, hd]: RMSNorm with weight w, then RoPE of the pairs (i, i + hd/2)."""
    n, _, hd = x.shape
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w
    i = torch.arange(hd // 2, dtype=torch.float64, device=x.device)
    a = torch.arange(pos, pos + n, dtype=torch.float64, device=x.device)[:, None] * BASE ** (-2 * i / hd)
    c, s = a.cos()[:, None], a.sin()[:, None]
    lo, hi = x[..., : hd // 2], x[..., hd // 2:]
    return torch.cat((lo * c - hi * s, lo * s + hi * c), -1)


def exact(case, seed):
    s = prepare(dict(case, entry="layer") if case["entry"] == "token" else case, seed)
    h, k, hd, n, pos, cache = (case[x] for x in ("heads", "kv_heads", "hd", "n", "pos", "cache"))
    G = h // k

    def wide(i, major):
        kv = [_widen(x, sc, cache) for x, sc in zip(s["kv"][i], s["scales"][i])]
        return [x if major else x.transpose(0, 1) for x in kv]

    if case["entry"] == "kernel":
        return _attention64(s["q"].double().view(n, h, hd), *wide(0, True), pos, G)
    if case["entry"] == "operator":
        return _attention64(s["qkv"][0][:, : h * hd].double().view(n, h, hd), *wide(0, False), pos, G)
    outs, rows, kvs, scales = [], [], [], []
    for i in range(case["layers"]):
        x = s["qkv"][i].double().view(n, h + 2 * k, hd)
        q, kk, v = _rope64(x[:, :h], s["qn"].double(), pos), _rope64(x[:, h: h + k], s["kn"].double(), pos), x[:, h + k:]
        if cache == "q4":
            q, kk = _hadamard64(q), _hadamard64(kk)
        rows.append(torch.cat((q, kk, v), 1).view(n, -1))
        stored, marks = [], []
        for t, sc, new in zip(s["kv"][i], s["scales"][i], (kk, _hadamard64(v) if cache == "q4" else v)):
            val, d = _quantise(new.float(), cache)
            w = t.double() if cache == "f16" else None
            if w is not None:
                w[pos: pos + n] = new
            t[pos: pos + n] = val
            if d is not None:
                sc[pos: pos + n] = d
            stored.append(w)
            marks.append(sc.double() if cache == "int8" else None)
        if i < 2:
            kvs.append(stored)
            scales.append(marks)
        o = _attention64(q, *wide(i, False), pos, G)
        outs.append(_hadamard64(o.view(n, h, hd)).view(n, -1) if cache == "q4" else o)
    return {"out": outs, "qkv": rows, "kv": kvs, "scales": scales if cache != "f16" else []}
