"""What a user of this framework has it do, as cases that can be timed and compared: single matrix-vector products,
batched products from a few tokens to a long prompt, a whole decoding step, a long list of independent products,
attention over a KV cache and the f32 matrix-vector product - each through the package's public entry points.

A case is a dict of plain values:
  op "gemv"       fmt, n, k                       y[n] = W[n x k] x, W in a k-quant format            (Q*KGemvKernel)
  op "gemm"       fmt, m, n, k                    C[m x n] = A[m x k] W^T                             (QuantizeKernel.ggml, Q5KKernel, Q6KKernel)
  op "list"       layers, hidden, ffn, vocab      the matrices of a decoder in one list               (GemvBatch)
  op "step"       the same, heads, kv_heads, dim, positions   one decoded token, attention included   (GemvBatch, IncrementalAttentionKernel)
  op "attention"  heads, kv_heads, dim, positions one query against the cache                         (IncrementalAttentionKernel)
  op "gemv_f32"   k, n                            y[n] = sum_k A[k][n] x[k]                           (CoalescedGemvKernel)
"""
from __future__ import annotations

import torch

import trueno_amd as t

SUPER_BLOCK = {"q4k": 144, "q5k": 176, "q6k": 210}      # bytes of 256 weights
GEMV = {"q4k": t.Q4KGemvKernel, "q5k": t.Q5KGemvKernel, "q6k": t.Q6KGemvKernel}
GEMM = {"q4k": t.QuantizeKernel.ggml, "q5k": t.Q5KKernel, "q6k": t.Q6KKernel}

_device = None


def _gpu():
    """The context and the stream of this program: made once, as a program that decodes makes them."""
    global _device
    if _device is None:
        ctx = t.CudaContext(0)
        _device = (ctx, t.CudaStream(ctx))
    return _device


def listed():
    return [
        # one token, the gate projection of a 7B model: a small call, mostly latency
        {"name": "gemv_q4k_11008x4096", "op": "gemv", "fmt": "q4k", "n": 11008, "k": 4096},
        # one token, the down projection in the 5-bit format: rows longer than one slab of 4096 columns
        {"name": "gemv_q5k_4096x11008", "op": "gemv", "fmt": "q5k", "n": 4096, "k": 11008},
        # one token, the vocabulary projection: the largest single matrix
        {"name": "gemv_q6k_32000x4096", "op": "gemv", "fmt": "q6k", "n": 32000, "k": 4096},
        # one token, an f32 projection that was left unquantised
        {"name": "gemv_f32_4096x11008", "op": "gemv_f32", "k": 4096, "n": 11008},
        # one query over a long cache with shared KV heads
        {"name": "attention_32x8_8192", "op": "attention", "heads": 32, "kv_heads": 8, "dim": 128, "positions": 8192},
        # every matrix of a 7B decoder in one list, activations of its own for every layer: the repository's benchmark
        {"name": "list_7b", "op": "list", "layers": 32, "hidden": 4096, "ffn": 11008, "vocab": 32000},
        # one decoded token of a 7B model with 2048 positions in its cache, norms, swiglu and residuals folded in
        {"name": "step_7b_2048", "op": "step", "layers": 32, "hidden": 4096, "ffn": 11008, "vocab": 32000, "heads": 32, "kv_heads": 32,
         "dim": 128, "positions": 2048},
        # a few sequences decoded together: 4 and 16 tokens against the two feed-forward shapes
        {"name": "gemm_q4k_14336x4096_m4", "op": "gemm", "fmt": "q4k", "m": 4, "n": 14336, "k": 4096},
        {"name": "gemm_q4k_4096x14336_m16", "op": "gemm", "fmt": "q4k", "m": 16, "n": 4096, "k": 14336},
        # a short prompt of odd length, the 5-bit format
        {"name": "gemm_q5k_11008x4096_m61", "op": "gemm", "fmt": "q5k", "m": 61, "n": 11008, "k": 4096},
        # a prompt of 512 tokens through the 6-bit down projection
        {"name": "gemm_q6k_4096x11008_m512", "op": "gemm", "fmt": "q6k", "m": 512, "n": 4096, "k": 11008},
        # a long prompt through the widest feed-forward matrix
        {"name": "gemm_q4k_14336x4096_m2048", "op": "gemm", "fmt": "q4k", "m": 2048, "n": 14336, "k": 4096},
    ]


def _log(rng, low, high):
    """An integer of low .. high, spread evenly over the logarithm."""
    return min(high, max(low, int(round(low * (high / low) ** rng.random()))))


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def draw(rng):
    least, most = 1.2e7, max(_cost(c) for c in listed())      # from a few microseconds on
    while True:
        op = rng.choice(["gemv", "gemv", "gemv", "gemm", "gemm", "gemm", "gemm", "attention", "gemv_f32", "list", "step"])
        fmt = rng.choice(["q4k", "q4k", "q5k", "q6k"])
        if op == "gemv":
            case = {"op": op, "fmt": fmt, "n": _log(rng, 512, 32000), "k": 256 * _log(rng, 4, 56)}
        elif op == "gemm":
            case = {"op": op, "fmt": fmt, "m": _log(rng, 2, 2048), "n": _log(rng, 512, 32000), "k": 256 * _log(rng, 4, 56)}
        elif op == "attention":
            kv_heads = rng.choice([4, 8, 16, 32])
            case = {"op": op, "heads": kv_heads * rng.choice([1, 2, 4]), "kv_heads": kv_heads, "dim": rng.choice([64, 128, 128, 256]),
                    "positions": _log(rng, 64, 16384)}
        elif op == "gemv_f32":
            case = {"op": op, "k": _log(rng, 512, 14336), "n": rng.choice([1, 4, 4]) * _log(rng, 512, 3584)}
        else:
            heads = 2 * rng.randint(8, 20)
            case = {"op": op, "layers": _log(rng, 2, 32), "hidden": 128 * heads, "ffn": 256 * rng.randint(20, 56), "vocab": _log(rng, 8000, 32000)}
            if op == "step":
                case.update(heads=heads, kv_heads=heads // rng.choice([1, 2]), dim=128, positions=_log(rng, 64, 4096))
        if least <= _cost(case) <= most:
            return case


# ---- inputs ---------------------------------------------------------------------------------------------------------
def _weights(gen, fmt, n, k):
    """Random blocks whose weights spread around zero with a standard deviation of about 0.02: uniform quants and block
    scales, one f16 scale per 256 weights (and for Q4_K and Q5_K the f16 minimum that centres them)."""
    size, blocks = SUPER_BLOCK[fmt], n * (k // 256)
    w = torch.randint(0, 256, (blocks, size), dtype=torch.uint8, device="cuda", generator=gen)
    d = (torch.rand(blocks, device="cuda", generator=gen) + 0.5) * {"q4k": 1.3e-4, "q5k": 6.5e-5, "q6k": 1.5e-5}[fmt]
    if fmt == "q6k":
        w[:, 208:210] = d.to(torch.float16).view(torch.uint8).view(blocks, 2)
    else:
        w[:, 0:2] = d.to(torch.float16).view(torch.uint8).view(blocks, 2)
        w[:, 2:4] = (d * {"q4k": 7.5, "q5k": 15.5}[fmt]).to(torch.float16).view(torch.uint8).view(blocks, 2)
    return w.view(-1)


def _activations(gen, *shape):
    """Normal values with the few channels of much larger size that a transformer's activations have."""
    x = torch.randn(shape, device="cuda", generator=gen)
    return x * (1.0 + 7.0 * (torch.rand(shape[-1], device="cuda", generator=gen) < 0.01))


def _new(*shape):
    return torch.zeros(shape, device="cuda")


def _layer_matrices(case):
    h, f = case["hidden"], case["ffn"]
    kv = h * case.get("kv_heads", 1) // case.get("heads", 1)
    return [("q", "q4k", h, h), ("k", "q4k", kv, h), ("v", "q4k", kv, h), ("o", "q4k", h, h), ("gate", "q4k", f, h), ("up", "q4k", f, h),
            ("down", "q6k", h, f)]


def prepare(case, seed):
    ctx, stream = _gpu()
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    op, s = case["op"], {"op": case["op"], "ctx": ctx, "stream": stream}
    if op == "gemv":
        s.update(w=_weights(gen, case["fmt"], case["n"], case["k"]), x=_activations(gen, case["k"]), y=_new(case["n"]),
                 kernel=GEMV[case["fmt"]](case["k"], case["n"]))
    elif op == "gemm":
        s.update(w=_weights(gen, case["fmt"], case["n"], case["k"]), x=_activations(gen, case["m"], case["k"]), y=_new(case["m"], case["n"]),
                 kernel=GEMM[case["fmt"]](case["m"], case["n"], case["k"]))
    elif op == "gemv_f32":
        s.update(w=torch.randn((case["k"], case["n"]), device="cuda", generator=gen) * 0.02, x=_activations(gen, case["k"]), y=_new(case["n"]),
                 kernel=t.CoalescedGemvKernel(case["k"], case["n"]))
    elif op == "attention":
        _attention(s, gen, case, 1)
        s["q"] = torch.randn((case["heads"], case["dim"]), device="cuda", generator=gen)
        s["y"] = _new(case["heads"], case["dim"])
    else:
        mats = _layer_matrices(case)
        s["w"] = [{name: _weights(gen, fmt, n, k) for name, fmt, n, k in mats} for _ in range(case["layers"])]
        s["head_w"] = _weights(gen, "q6k", case["vocab"], case["hidden"])
        s["logits"] = _new(case["vocab"])
        (_prepare_list if op == "list" else _prepare_step)(s, gen, case, mats)
    torch.cuda.synchronize()
    return s


def _attention(s, gen, case, layers):
    """The caches of `layers` layers, full up to the last position, and the kernel."""
    shape = (layers, case["kv_heads"], case["positions"], case["dim"])
    s["cache_k"] = torch.randn(shape, device="cuda", generator=gen)
    s["cache_v"] = torch.randn(shape, device="cuda", generator=gen)
    s["positions"] = case["positions"]
    s["kernel"] = t.IncrementalAttentionKernel.with_gqa(case["positions"], case["dim"], case["heads"], case["kv_heads"])


def _prepare_list(s, gen, case, mats):
    """q, k, v, gate and up of a layer read a vector of its own; o reads the normalised q, down the normalised gate, the
    head the normalised output of the last down: nothing else orders the entries."""
    norm, layers = t.GemvBatch.NORM_INPUT, case["layers"]
    s["x"] = _activations(gen, layers, case["hidden"])
    s["out"] = {name: _new(layers, n) for name, _, n, _ in mats}
    batch = t.GemvBatch()
    for l in range(layers):
        for name, fmt, n, k in mats:
            source = {"o": "q", "down": "gate"}.get(name)
            x = s["x"][l] if source is None else s["out"][source][l]
            batch.add(fmt, k, n, s["out"][name][l].data_ptr(), s["w"][l][name].data_ptr(), x.data_ptr(), 0 if source is None else norm)
    batch.add("q6k", case["hidden"], case["vocab"], s["logits"].data_ptr(), s["head_w"].data_ptr(), s["out"]["down"][layers - 1].data_ptr(), norm)
    s["batch"] = batch


def _prepare_step(s, gen, case, mats):
    """Per layer: q, k, v <- rmsnorm(h) * g1; attention; h1 = h + o(attention); gate, up <- rmsnorm(h1) * g2;
    h = h1 + down(silu(gate) * up); then the head on rmsnorm(h) * g1.  The layers share one set of activations; the
    first reads the token's embedding."""
    norm, layers = t.GemvBatch.NORM_INPUT, case["layers"]
    _attention(s, gen, case, layers)
    s["embedding"] = _activations(gen, case["hidden"])
    g1, g2 = (torch.rand(case["hidden"], device="cuda", generator=gen) + 0.5 for _ in range(2))
    act = {name: _new(n) for name, _, n, _ in mats}
    act["h"], act["h1"], act["attention"] = (_new(case["hidden"]) for _ in range(3))
    s.update(act=act, gammas=(g1, g2), before=[], after=[])
    shape = {name: (fmt, k, n) for name, fmt, n, k in mats}
    for l in range(layers):
        w, h = s["w"][l], s["embedding"] if l == 0 else act["h"]
        before, after = t.GemvBatch(), t.GemvBatch()
        for name in ("q", "k", "v"):
            before.add(*shape[name], act[name].data_ptr(), w[name].data_ptr(), h.data_ptr(), norm, gamma=g1.data_ptr(), norm_eps=1e-5)
        after.add(*shape["o"], act["h1"].data_ptr(), w["o"].data_ptr(), act["attention"].data_ptr(), residual=h.data_ptr())
        for name in ("gate", "up"):
            after.add(*shape[name], act[name].data_ptr(), w[name].data_ptr(), act["h1"].data_ptr(), norm, gamma=g2.data_ptr(), norm_eps=1e-5)
        after.add(*shape["down"], act["h"].data_ptr(), w["down"].data_ptr(), act["gate"].data_ptr(), x2=act["up"].data_ptr(),
                  residual=act["h1"].data_ptr())
        s["before"].append(before)
        s["after"].append(after)
    s["after"][-1].add("q6k", case["hidden"], case["vocab"], s["logits"].data_ptr(), s["head_w"].data_ptr(), act["h"].data_ptr(), norm,
                       gamma=g1.data_ptr(), norm_eps=1e-5)


# ---- one pass -------------------------------------------------------------------------------------------------------
def run(s):
    op, stream = s["op"], s["stream"]
    if op in ("gemv", "gemv_f32"):
        s["kernel"].launch(stream, s["y"].data_ptr(), s["w"].data_ptr(), s["x"].data_ptr())
        return s["y"]
    if op == "gemm":
        s["kernel"].launch(stream, s["x"].data_ptr(), s["w"].data_ptr(), s["y"].data_ptr())
        return s["y"]
    if op == "attention":
        s["kernel"].launch(stream, s["q"].data_ptr(), s["cache_k"].data_ptr(), s["cache_v"].data_ptr(), s["y"].data_ptr(), s["positions"])
        return s["y"]
    if op == "list":
        s["batch"].launch(stream)
        return {"logits": s["logits"], **s["out"]}
    act = s["act"]
    for l, (before, after) in enumerate(zip(s["before"], s["after"])):
        before.launch(stream)
        s["kernel"].launch(stream, act["q"].data_ptr(), s["cache_k"][l].data_ptr(), s["cache_v"][l].data_ptr(), act["attention"].data_ptr(),
                           s["positions"])
        after.launch(stream)
    return {"logits": s["logits"], **act}


# ---- the same functions in 64 bits -----------------------------------------------------------------------------------
def _dequantised(fmt, w, rows, k):
    """f64 [rows x k] of the raw blocks: Q4_K and Q6_K as GGML lays them out, Q5_K with eight contiguous 12-bit (scale, min)
    fields and value i's fifth bit in bit i % 8 of byte 144 + i // 8."""
    b = w.view(rows * (k // 256), SUPER_BLOCK[fmt])
    half = lambda at: b[:, at:at + 2].contiguous().view(torch.float16).double()
    if fmt == "q6k":
        i = torch.arange(256, device=w.device)
        h, g, l = i // 128, i % 128 // 32, i % 32
        low = (b[:, 64 * h + l + 32 * (g & 1)] >> (4 * (g >> 1))) & 15
        high = (b[:, 128 + 32 * h + l] >> (2 * g)) & 3
        scale = b[:, 192:208].contiguous().view(torch.int8).double()[:, 8 * h + l // 16 + 2 * g]
        return (half(208) * scale * ((low + 16 * high).double() - 32.0)).view(rows, k)
    quants = b[:, 16:144].view(-1, 4, 1, 32)
    q = torch.cat((quants & 15, quants >> 4), 2).reshape(-1, 256).double()
    f = b[:, 4:16].long()
    if fmt == "q4k":
        s = torch.cat((f[:, 0:4] & 63, (f[:, 8:12] & 15) | (f[:, 0:4] >> 6 << 4)), 1)
        m = torch.cat((f[:, 4:8] & 63, (f[:, 8:12] >> 4) | (f[:, 4:8] >> 6 << 4)), 1)
    else:
        even, odd = f[:, 0::3] | (f[:, 1::3] & 15) << 8, f[:, 1::3] >> 4 | f[:, 2::3] << 4
        fields = torch.stack((even, odd), 2).reshape(-1, 8)
        s, m = fields & 63, fields >> 6
        bits = torch.arange(8, device=w.device, dtype=torch.uint8)
        q += 16.0 * ((b[:, 144:176, None] >> bits) & 1).reshape(-1, 256)
    spread = lambda v: v.double().repeat_interleave(32, 1)
    return (half(0) * spread(s) * q - half(2) * spread(m)).view(rows, k)


def _exact_product(fmt, w, n, k, a):
    """f64 a [.. x k] times the matrix, in runs of rows that keep the dequantised part small."""
    step, size = max(1, (1 << 25) // k), (k // 256) * SUPER_BLOCK[fmt]
    return torch.cat([a @ _dequantised(fmt, w[r * size:min(r + step, n) * size], min(step, n - r), k).T for r in range(0, n, step)], -1)


def _exact_attention(q, k, v):
    """softmax(q . k / sqrt(dim)) v per head; the heads of a group share a KV head."""
    group = q.shape[0] // k.shape[0]
    out = []
    for h in range(q.shape[0]):
        p = torch.softmax(k[h // group].double() @ q[h] * q.shape[1] ** -0.5, 0)
        out.append(p @ v[h // group].double())
    return torch.stack(out)


def _normalised(x, eps, gamma=1.0):
    return x / torch.sqrt((x * x).mean() + eps) * gamma


def exact(case, seed):
    s, op = prepare(case, seed), case["op"]
    if op in ("gemv", "gemm"):
        return _exact_product(case["fmt"], s["w"], case["n"], case["k"], s["x"].double())
    if op == "gemv_f32":
        return s["x"].double() @ s["w"].double()
    if op == "attention":
        return _exact_attention(s["q"].double(), s["cache_k"][0], s["cache_v"][0])
    shape = {name: (fmt, n, k) for name, fmt, n, k in _layer_matrices(case)}
    product = lambda l, name, x: _exact_product(shape[name][0], s["w"][l][name], *shape[name][1:], x)
    head = lambda x: _exact_product("q6k", s["head_w"], case["vocab"], case["hidden"], x)
    if op == "list":
        out = {name: [] for name in shape}
        for l in range(case["layers"]):
            x, got = s["x"][l].double(), {}
            for name in shape:
                source = {"o": "q", "down": "gate"}.get(name)
                got[name] = product(l, name, x if source is None else _normalised(got[source], 1e-6))
                out[name].append(got[name])
        return {"logits": head(_normalised(out["down"][-1], 1e-6)), **{name: torch.stack(v) for name, v in out.items()}}
    h, (g1, g2), act = s["embedding"].double(), (g.double() for g in s["gammas"]), {}
    for l in range(case["layers"]):
        x = _normalised(h, 1e-5, g1)
        act.update({name: product(l, name, x) for name in ("q", "k", "v")})
        act["attention"] = _exact_attention(act["q"].view(case["heads"], case["dim"]), s["cache_k"][l], s["cache_v"][l]).view(-1)
        act["h1"] = h + product(l, "o", act["attention"])
        x = _normalised(act["h1"], 1e-5, g2)
        act.update({name: product(l, name, x) for name in ("gate", "up")})
        h = act["h"] = act["h1"] + product(l, "down", torch.nn.functional.silu(act["gate"]) * act["up"])
    return {"logits": head(_normalised(h, 1e-5, g1)), **{name: act.get(name) for name in s["act"]}}      # "o" and "down" go into h1 and h


# ---- what a pass cannot do without, and what it may be off by --------------------------------------------------------
def _product(fmt, m, n, k):
    return n * (k // 256) * SUPER_BLOCK[fmt] + 4 * m * k + 4 * m * n, 2 * m * n * k


def work(case):
    op = case["op"]
    if op in ("gemv", "gemm"):
        nbytes, flops = _product(case["fmt"], case.get("m", 1), case["n"], case["k"])
        return {"bytes": nbytes, "flops": flops}
    if op == "gemv_f32":
        return {"bytes": 4 * (case["k"] * case["n"] + case["k"] + case["n"]), "flops": 2 * case["k"] * case["n"]}
    nbytes = flops = 0
    if op in ("attention", "step"):
        cache, pairs = case["kv_heads"] * case["positions"] * case["dim"], case["heads"] * case["positions"] * case["dim"]
        nbytes, flops = 8 * cache + 8 * case["heads"] * case["dim"], 4 * pairs
        if op == "attention":
            return {"bytes": nbytes, "flops": flops}
    for _, fmt, n, k in _layer_matrices(case):
        b, f = _product(fmt, 1, n, k)
        nbytes, flops = nbytes + b, flops + f
    b, f = _product("q6k", 1, case["vocab"], case["hidden"])
    return {"bytes": case["layers"] * nbytes + b, "flops": case["layers"] * flops + f}


def tolerance(case):
    """About four times the largest error seen against the same function in f64: 1.6e-7 and 1.1e-6 for one product (f32
    sums over 1024 to 14336 terms), 3.1e-7 and 1.1e-6 for attention, 8e-7 and 2.8e-6 for a list (a layer's second product
    reads the first's results), 3.5e-6 and 2e-5 for a step (32 layers deep, a softmax in each)."""
    return {"attention": {"rel": 1.2e-6, "max": 5e-6}, "list": {"rel": 3e-6, "max": 1.2e-5},
            "step": {"rel": 1.4e-5, "max": 8e-5}}.get(case["op"], {"rel": 6e-7, "max": 5e-6})
