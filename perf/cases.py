"""The work that a user of this framework has it do, as measurable cases.

Each case is one pass through the public modules over packed GGUF weights: a projection
(`DevicePackedLinear`), the projections of a decoder layer with their fused producers
(`HipFusedOps`, `project_shared`), the expert FFN of a mixture-of-experts layer
(`HipPackedMoEExperts`) or a token lookup (`DevicePackedEmbedding`). Sizes are those of the
benchmark configurations (Llama-3-8B layer and head, the prefill chunks, the expert sets) and of
the ranges around them: one token to a prefill chunk of 2048, rows of 4 to 56 blocks, all four
packed types, bfloat16 layers (the GPU dtype) and float32 ones.

Weights are random quants with scales that give zero-mean values of standard deviation about 0.02,
as trained projections have; activations are N(0, 1), as a norm leaves them.
"""

import math

import torch
import torch.nn.functional as F

Q8_0, Q4_K, Q6_K, IQ4_XS = 8, 12, 14, 23
# (values per block, bytes per block)
GEOMETRY = {Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210), IQ4_XS: (256, 136)}
W_STD = 0.02
EPS = 1e-5
IQ4_GRID = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]

MAX_FLOPS = 2.0 * 1024 * 218103808  # the prefill layer's
MAX_WEIGHT_BYTES = 128256 * 3360  # the output head's


# ------------------------------------------------------------------------------------ the cases
def linear(name, type_, n, k, m, dtype="bf16"):
    return {"name": name, "kind": "linear", "type": type_, "n": n, "k": k, "m": m, "dtype": dtype}


def layer(name, m, embd=4096, kv=1024, ffn=14336):
    return {"name": name, "kind": "layer", "m": m, "embd": embd, "kv": kv, "ffn": ffn}


def moe(name, m, experts, top_k, embd, ffn):
    return {"name": name, "kind": "moe", "m": m, "experts": experts, "top_k": top_k, "embd": embd,
            "ffn": ffn}


def embed(name, type_, n, k, m):
    return {"name": name, "kind": "embed", "type": type_, "n": n, "k": k, "m": m}


def listed():
    return [
        # one attention projection of one token: the smallest call of a decode step
        linear("decode_q4k", Q4_K, 4096, 4096, 1),
        # the vocabulary head of one token: the largest single weight of a decode step
        linear("head_q6k", Q6_K, 128256, 4096, 1),
        # every projection of one decoder layer for one token, q|k|v and gate|up grouped
        layer("layer_decode_1", 1),
        # the same for sixteen concurrent replies
        layer("layer_decode_16", 16),
        # a gate projection for more concurrent replies than one decode tile, or a short prompt
        linear("short_prompt_q4k", Q4_K, 14336, 4096, 48),
        # a prompt of odd length through an 8-bit model's float32 projection
        linear("prompt_q8_0_f32", Q8_0, 4096, 4096, 333, "f32"),
        # a prefill chunk through an IQ4_XS model's float32 projection
        linear("prefill_iq4xs_f32", IQ4_XS, 4096, 4096, 512, "f32"),
        # a long prefill chunk through the widest projection
        linear("prefill_q4k", Q4_K, 14336, 4096, 2048),
        # every projection of one decoder layer for a prefill chunk
        layer("layer_prefill", 1024),
        # the expert FFN of few large experts for sixteen concurrent replies
        moe("moe_decode_16", 16, 8, 2, 4096, 14336),
        # the expert FFN of many small experts for a prefill chunk
        moe("moe_prefill", 512, 64, 8, 2048, 1024),
        # the token lookup of a prefill chunk
        embed("embedding", Q6_K, 128256, 4096, 512),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    while True:
        pick = rng.random()
        rows = _log(rng, 1, 16) if rng.random() < 0.4 else _log(rng, 17, 2048)
        if pick < 0.55:
            c = linear("", rng.choice([Q8_0, Q4_K, Q4_K, Q6_K, Q6_K, IQ4_XS]), _log(rng, 256, 32768),
                       256 * rng.choice([4, 5, 8, 11, 12, 14, 16, 16, 20, 32, 43, 56]), rows,
                       rng.choice(["bf16", "bf16", "bf16", "f32"]))
        elif pick < 0.7:
            c = layer("", rows, *rng.choice([(2048, 512, 8192), (3072, 1024, 8192),
                                             (4096, 1024, 14336), (5120, 1024, 13824),
                                             (4096, 4096, 11008)]))
        elif pick < 0.9:
            c = moe("", rows, *rng.choice([(8, 2, 4096, 14336), (40, 8, 1536, 512),
                                           (64, 8, 2048, 1024), (16, 4, 3072, 2048)]))
        else:
            c = embed("", rng.choice([Q8_0, Q4_K, Q6_K, IQ4_XS]), _log(rng, 8192, 128256),
                      256 * rng.choice([4, 8, 12, 16, 20]), rows)
        del c["name"]
        w = work(c)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= 4 * MAX_WEIGHT_BYTES:
            return c


# ---------------------------------------------------------------------------- weights and inputs
def _bytes(g, shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g)


def _half(v):
    return v.to(torch.float16).view(torch.uint8).reshape(*v.shape, 2)


def _spread(g, n):
    """Block scales: within a factor of about two of one another."""
    return torch.exp(0.4 * torch.randn(n, device="cuda", generator=g))


def packed(g, type_, n, k):
    """(n, row_bytes) packed rows on the GPU."""
    size, nbytes = GEOMETRY[type_]
    nb = n * (k // size)
    out = _bytes(g, (nb, nbytes))
    s = W_STD * _spread(g, nb)
    if type_ == Q8_0:  # d, 32 signed bytes
        out[:, 0:2] = _half(s / 73)
        out[:, 2:] = torch.where(out[:, 2:] == 128, 129, out[:, 2:])
    elif type_ == Q4_K:  # d, dmin, 8 six-bit scales and mins, 128 bytes of nibbles
        sc = torch.randint(24, 64, (nb, 8), dtype=torch.uint8, device="cuda", generator=g)
        mn = (sc.int() + torch.randint(-6, 7, (nb, 8), device="cuda", generator=g)).clamp(0, 63).to(torch.uint8)
        d = s / (45 * 4.6)
        out[:, 0:2], out[:, 2:4] = _half(d), _half(7.5 * d)
        out[:, 4:8] = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
        out[:, 8:12] = (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6)
        out[:, 12:16] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    elif type_ == Q6_K:  # low nibbles, high bits, 16 signed scales, d
        out[:, 208:210] = _half(s / (74 * 18.5))
    else:  # IQ4_XS: d, high and low scale bits, 128 bytes of grid indices
        out[:, 0:2] = _half(s / (18.5 * 70))
    return out.reshape(n, (k // size) * nbytes)


def _linear(g, type_, n, k, dtype=torch.bfloat16):
    from matricxon_amd.device_packed import DevicePackedLinear

    return DevicePackedLinear(packed(g, type_, n, k), k, type_, None, dtype, backend="native")


def _dtype(case):
    return torch.float32 if case.get("dtype") == "f32" else torch.bfloat16


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _x(g, m, k, dtype=torch.bfloat16):
    return torch.randn(m, k, device="cuda", generator=g).to(dtype)


LAYER = ("q", "k", "v", "o", "gate", "up", "down")


def _layer_shapes(c):
    e, kv, f = c["embd"], c["kv"], c["ffn"]
    return {"q": (Q4_K, e, e), "k": (Q4_K, kv, e), "v": (Q6_K, kv, e), "o": (Q4_K, e, e),
            "gate": (Q4_K, f, e), "up": (Q4_K, f, e), "down": (Q6_K, e, f)}


def _moe_shapes(c):
    e, f = c["embd"], c["ffn"]
    return {"gate": (Q4_K, f, e), "up": (Q4_K, f, e), "down": (Q6_K, e, f)}


def _routing(g, c):
    logits = torch.randn(c["m"], c["experts"], device="cuda", generator=g)
    w, idx = torch.topk(torch.softmax(logits, -1), c["top_k"])
    return w / w.sum(-1, keepdim=True), idx


def _raw(case, seed):
    """The packed weights and the inputs of a case, in the order in which `prepare` makes them."""
    g, kind, m = _gen(seed), case["kind"], case["m"]
    if kind == "linear":
        w = packed(g, case["type"], case["n"], case["k"])
        return w, _x(g, m, case["k"], _dtype(case))
    if kind == "embed":
        w = packed(g, case["type"], case["n"], case["k"])
        return w, torch.randint(0, case["n"], (m,), device="cuda", generator=g)
    if kind == "layer":
        ws = {name: packed(g, *t) for name, t in _layer_shapes(case).items()}
        norms = [(1 + 0.1 * torch.randn(case["embd"], device="cuda", generator=g)).to(torch.bfloat16)
                 for _ in range(2)]
        return ws, norms, _x(g, m, case["embd"])
    ws = {name: packed(g, t, case["experts"] * n, k).view(case["experts"], n, -1)
          for name, (t, n, k) in _moe_shapes(case).items()}
    w, idx = _routing(g, case)
    return ws, w, idx, _x(g, m, case["embd"])


def prepare(case, seed):
    from matricxon_amd.device_packed import DevicePackedEmbedding, DevicePackedLinear
    from matricxon_amd.fused_ops import HipFusedOps
    from matricxon_amd.moe import HipPackedMoEExperts

    kind, raw = case["kind"], _raw(case, seed)
    if kind == "linear":
        mod = DevicePackedLinear(raw[0], case["k"], case["type"], None, _dtype(case), backend="native")
        return {"kind": kind, "mod": mod, "x": raw[1]}
    if kind == "embed":
        mod = DevicePackedEmbedding(raw[0], case["k"], case["type"], torch.bfloat16)
        return {"kind": kind, "mod": mod, "x": raw[1]}
    if kind == "layer":
        owner = torch.nn.Module()
        for name, (t, _, k) in _layer_shapes(case).items():
            setattr(owner, name, DevicePackedLinear(raw[0][name], k, t, None, torch.bfloat16,
                                                    backend="native"))
        if HipFusedOps.active() is None:
            HipFusedOps.configure(True)
        return {"kind": kind, "mod": owner, "norms": raw[1], "x": raw[2]}
    types = tuple(t for t, _, _ in _moe_shapes(case).values())
    mod = HipPackedMoEExperts(*raw[0].values(), *types, case["embd"], case["ffn"], F.silu,
                              torch.bfloat16)
    return {"kind": kind, "mod": mod, "w": raw[1], "idx": raw[2], "x": raw[3]}


def run(s):
    if s["kind"] in ("linear", "embed"):
        return s["mod"](s["x"])
    if s["kind"] == "moe":
        return s["mod"](s["x"], s["w"], s["idx"])
    # a decoder layer's projections; attention itself is not this framework's, so the output
    # projection reads the queries
    from matricxon_amd.fused_ops import HipFusedOps, project_shared

    ops, mod, x = HipFusedOps.active(), s["mod"], s["x"]
    h = ops.rms_norm(x, s["norms"][0], EPS)
    q, k, v = project_shared(mod, ("q", "k", "v"), h)
    x = x + mod.o(q)
    h = ops.rms_norm(x, s["norms"][1], EPS)
    gate, up = project_shared(mod, ("gate", "up"), h)
    y = x + mod.down(ops.silu_mul(gate, up))
    return {"q": q, "k": k, "v": v, "gate": gate, "up": up, "y": y}


# ------------------------------------------------------------------------------------- the floor
def _row_bytes(type_, k):
    size, nbytes = GEOMETRY[type_]
    return (k // size) * nbytes


def work(case):
    kind, m = case["kind"], case["m"]
    if kind == "linear":
        n, k, e = case["n"], case["k"], 4 if case.get("dtype") == "f32" else 2
        return {"bytes": n * _row_bytes(case["type"], k) + e * m * (n + k), "flops": 2.0 * m * n * k}
    if kind == "embed":
        return {"bytes": m * (_row_bytes(case["type"], case["k"]) + 8 + 2 * case["k"]),
                "flops": 2.0 * m * case["k"]}
    if kind == "layer":
        shapes = _layer_shapes(case).values()
        weights = sum(n * _row_bytes(t, k) for t, n, k in shapes)
        outs = 3 * case["embd"] + 2 * case["kv"] + 2 * case["ffn"]  # x, q, y, k, v, gate, up
        return {"bytes": weights + 2 * m * outs, "flops": 2.0 * m * sum(n * k for _, n, k in shapes)}
    shapes, ne, tk = _moe_shapes(case).values(), case["experts"], case["top_k"]
    active = ne * (1 - (1 - tk / ne) ** m)  # experts that a routing of m tokens names
    weights = sum(n * _row_bytes(t, k) for t, n, k in shapes)
    return {"bytes": active * weights + m * (4 * case["embd"] + 12 * tk),
            "flops": 2.0 * m * tk * sum(n * k for _, n, k in shapes)}


# -------------------------------------------------------------------------------------- 64 bits
def _f16(b):
    return b.contiguous().view(torch.float16).double()


def dequantized(w, type_, k):
    """The (n, k) float64 values of packed rows, by the formats' definitions."""
    size, nbytes = GEOMETRY[type_]
    b = w.reshape(-1, nbytes)
    nb = b.shape[0]
    if type_ == Q8_0:
        v = _f16(b[:, 0:2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif type_ == Q4_K:
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, 16:].reshape(nb, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(nb, 8, 32).double()
        v = (_f16(b[:, 0:2]) * sc).unsqueeze(-1) * q - (_f16(b[:, 2:4]) * mn).unsqueeze(-1)
    elif type_ == Q6_K:
        ql, qh = b[:, :128].reshape(nb, 2, 2, 32), b[:, 128:192].reshape(nb, 2, 32)
        q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * _f16(b[:, 208:210])
        v = (q.reshape(nb, 16, 16).double() - 32) * sc.unsqueeze(-1)
    else:
        high = b[:, 2].int() | (b[:, 3].int() << 8)
        ib = torch.arange(8, device=b.device)
        ls = ((b[:, 4:8].int()[:, ib // 2] >> (4 * (ib % 2))) & 15) | (((high.unsqueeze(1) >> (2 * ib)) & 3) << 4)
        qs = b[:, 8:].reshape(nb, 8, 16)
        grid = torch.tensor(IQ4_GRID, dtype=torch.float64, device=b.device)
        v = grid[torch.cat([qs & 15, qs >> 4], 2).long()] * (_f16(b[:, 0:2]) * (ls - 32)).unsqueeze(-1)
    return v.reshape(-1, k)


def _q8k(x):
    """The values that the integer kernels multiply: x in blocks of 256, each rounded to 255 steps of
    its largest magnitude (the Q8_K activations of the path's definition), as float64."""
    b = x.float().reshape(x.shape[0], -1, 256)
    amax = b.abs().amax(-1, keepdim=True).double()
    # both quotients are float32 in the definition (torch's own float32 division by or of a number
    # multiplies by a reciprocal, which is another rounding)
    q = torch.round(b * torch.where(amax > 0, 127 / amax, 0).float()).clamp(-127, 127)
    return (q.double() * (amax / 127).float().double()).reshape(x.shape)


def _project(w, type_, k, x):
    """x @ W.T in float64, row blocks at a time (the head's weight in 64 bits is 4 GB)."""
    xq = x.double() if type_ == IQ4_XS else _q8k(x)
    step = max(1, (1 << 27) // k)
    return torch.cat([xq @ dequantized(w[i:i + step], type_, k).T for i in range(0, w.shape[0], step)], 1)


def _rms(x, w):
    x32 = x.double()
    n = (x32 * torch.rsqrt(x32.square().mean(-1, keepdim=True) + EPS)).to(torch.bfloat16)
    return (n.double() * w.double()).to(torch.bfloat16)


def _swiglu(gate, up):
    return (F.silu(gate.double()).to(torch.bfloat16).double() * up.double()).to(torch.bfloat16)


def exact(case, seed):
    """`run` with every product and sum in float64; tensors that go from one module to the next are
    in the layer's dtype, as the modules return them."""
    kind, raw = case["kind"], _raw(case, seed)
    if kind == "linear":
        return _project(raw[0], case["type"], case["k"], raw[1])
    if kind == "embed":
        return dequantized(raw[0][raw[1]], case["type"], case["k"])
    bf = torch.bfloat16
    if kind == "layer":
        ws, norms, x = raw
        shapes = _layer_shapes(case)

        def proj(name, v):
            return _project(ws[name], shapes[name][0], shapes[name][2], v)

        h = _rms(x, norms[0])
        q, k, v = proj("q", h), proj("k", h), proj("v", h)
        x = (x.double() + proj("o", q.to(bf)).to(bf).double()).to(bf)
        h = _rms(x, norms[1])
        gate, up = proj("gate", h), proj("up", h)
        y = x.double() + proj("down", _swiglu(gate.to(bf), up.to(bf))).to(bf).double()
        return {"q": q, "k": k, "v": v, "gate": gate, "up": up, "y": y}
    ws, tw, idx, x = raw
    shapes = _moe_shapes(case)
    out = torch.zeros(case["m"], case["embd"], dtype=torch.float64, device="cuda")
    for e in range(case["experts"]):
        tok, slot = (idx == e).nonzero(as_tuple=True)
        if tok.numel() == 0:
            continue
        gate, up = (_project(ws[n][e], shapes[n][0], shapes[n][2], x[tok]).to(bf) for n in ("gate", "up"))
        down = _project(ws["down"][e], shapes["down"][0], shapes["down"][2], _swiglu(gate, up))
        out.index_add_(0, tok, down.to(bf).double() * tw[tok, slot].double().unsqueeze(-1))
    return out


def tolerance(case):
    """Float32 results: about four times the error that their sums show against 64 bits. bfloat16
    results: a rounding step each way, and for several modules in a row what a last-bit change of an
    intermediate value makes of the activations' 8-bit rounding."""
    if case["kind"] == "linear" and case.get("dtype") == "f32":
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] in ("linear", "embed"):
        return {"rel": 7e-3, "max": 2e-2}
    return {"rel": 1e-2, "max": 0.1}
