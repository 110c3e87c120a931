"""The work a user of this framework has it do, as cases to time and compare.

Every case runs through the public binding (osm_hip) the way a serving or
generation program does: weights resident (or, for the capped cache, in a
pinned host store), inputs in torch tensors on the GPU, one call per step.
Kinds:

  decode   a step of `tokens` tokens through `layers` MoE sublayers (RMSNorm,
           router, top-k, experts, shared expert, residual), fp32 activations:
           token generation for one request (each layer on the output of the
           one before) or for a batch (each layer on its own input, as
           attention would give it)
  prefill  a bf16 prompt chunk of `tokens` tokens through `layers` MoE layers,
           each on its own input
  cached   `tokens` tokens, one after another, through chained sublayers whose
           experts live in a capped HBM cache over a pinned host store
  gemv     a row of q4 projections kept in HBM, applied to one vector

The default geometry is Qwen3-Next-80B-A3B's MoE layer (hidden 2048, expert
width 512, 512 experts, top-10 with a shared expert, groups of 64), the one
this repository benchmarks. Weights are the repository's synthetic ones (the
nibbles uniform, scales |N| * 0.02, biases -8 * scale + N * 0.002, router
N * 0.02), another model for each seed. A case runs over enough layers, and
the states in turn, that a pass reads its weights from HBM rather than from
the last-level cache.
"""

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "orbi-streammoe_amd"))

import osm_hip  # noqa: E402

SHAPE = {"hidden": 2048, "inter": 512, "experts": 512, "top_k": 10, "group": 64, "meta": "bf16", "router": "bf16"}
META = {"bf16": osm_hip.BF16, "f32": osm_hip.F32}
ROUTER = {"bf16": osm_hip.BF16, "f32": osm_hip.F32, "q8": osm_hip.AFFINE_Q8}
SHARED = 0xFFFFFFFF  # the shared expert's id in the synthetic generator
EPS = 1e-6
Q8_GROUP = 64


def listed():
    return [
        # One request generating: the whole 48-layer step, replayed as a graph. Latency and launches count.
        dict(SHAPE, name="decode_1", kind="decode", tokens=1, layers=48),
        # A few requests at once, with the 8-bit router that MLX checkpoints store.
        dict(SHAPE, name="decode_4_q8", kind="decode", tokens=4, layers=8, router="q8"),
        # A small serving batch.
        dict(SHAPE, name="decode_16", kind="decode", tokens=16, layers=4),
        # A ragged batch, as continuous batching forms it.
        dict(SHAPE, name="decode_37", kind="decode", tokens=37, layers=4),
        # A full serving batch.
        dict(SHAPE, name="decode_64", kind="decode", tokens=64, layers=4),
        # Experts with the f32 scales and biases that the reference's converter writes; a larger ragged batch.
        dict(SHAPE, name="decode_157_f32", kind="decode", tokens=157, layers=2, meta="f32"),
        # A prompt with fp32 activations through an 8-bit router, residuals and norms included.
        dict(SHAPE, name="decode_512_q8", kind="decode", tokens=512, layers=2, router="q8"),
        # A short prompt, or the ragged end of a chunked one.
        dict(SHAPE, name="prefill_77", kind="prefill", tokens=77, layers=2),
        # The benchmark's prompt chunk.
        dict(SHAPE, name="prefill_512", kind="prefill", tokens=512, layers=2),
        # A long prompt's chunk, the largest call.
        dict(SHAPE, name="prefill_4096", kind="prefill", tokens=4096, layers=2),
        # A model larger than its HBM budget: 24 tokens with about a third of the experts resident.
        dict(SHAPE, name="cached_24", kind="cached", tokens=24, layers=3, budget_mb=512),
        # The single operator over resident weights: a row of dense projections.
        dict(name="gemv_4096x2048", kind="gemv", rows=4096, cols=2048, group=64, meta="f32", count=24),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "cached", "gemv"])
    if kind == "gemv":
        cols = 128 * rng.randint(4, 40)
        return {"kind": kind, "rows": log(512, 16384), "cols": cols, "group": rng.choice([32, 64, 128]),
                "meta": rng.choice(["f32", "bf16"]), "count": rng.randint(8, 24)}
    c = {"kind": kind, "hidden": rng.choice([1024, 2048, 2048, 2048]), "inter": rng.choice([256, 512, 512, 768]),
         "experts": rng.choice([128, 256, 512, 512]), "top_k": rng.choice([4, 8, 10, 10]),
         "group": rng.choice([32, 64, 64, 64, 128]), "meta": rng.choice(["bf16", "bf16", "f32"]),
         "router": rng.choice(["bf16", "bf16", "q8", "f32"])}
    if kind == "decode":
        c["tokens"] = log(1, 600)
        c["layers"] = 24 if c["tokens"] == 1 else 8 if c["tokens"] < 8 else 4 if c["tokens"] < 100 else 2
    elif kind == "prefill":
        c["tokens"] = log(20, 4000)
        c["layers"] = 2
    else:
        c["tokens"] = rng.randint(8, 32)
        c["layers"] = 2
        stride = expert_bytes(c)
        c["budget_mb"] = max(64, int(rng.uniform(0.1, 0.4) * 2 * c["experts"] * stride / 2**20))
    return c


def chained(c):
    return c["kind"] == "cached" or c["kind"] == "decode" and c["tokens"] == 1


# ---- sizes ----------------------------------------------------------------------------
def expert_bytes(c):
    meta = 4 if c["meta"] == "f32" else 2
    return 3 * c["hidden"] * c["inter"] // 2 + 2 * 3 * (c["hidden"] * c["inter"] // c["group"]) * meta


def router_bytes(c):
    n = (c["experts"] + 1) * c["hidden"]
    return n * 2 if c["router"] == "bf16" else n * 4 if c["router"] == "f32" else n + 8 * n // Q8_GROUP


def work(case):
    c = case
    if c["kind"] == "gemv":
        meta = 4 if c["meta"] == "f32" else 2
        one = c["rows"] * c["cols"] // 2 + 2 * (c["rows"] * c["cols"] // c["group"]) * meta + 4 * c["rows"]
        return {"bytes": c["count"] * one + 4 * c["cols"], "flops": 2.0 * c["count"] * c["rows"] * c["cols"]}
    T, D, I, E, k = c["tokens"], c["hidden"], c["inter"], c["experts"], c["top_k"]
    flops = c["layers"] * (2.0 * T * (k + 1) * 3 * D * I + 2.0 * T * D * (E + 1))
    if c["kind"] == "cached":  # one token after another: every pick's weights are read for it
        per_layer = T * ((k + 1) * expert_bytes(c) + router_bytes(c) + 8 * D)
    else:  # the distinct experts of the tokens' picks, expected over uniform routing
        distinct = E * (1.0 - (1.0 - k / E) ** T)
        per_layer = (distinct + 1) * expert_bytes(c) + router_bytes(c) + T * D * (6 if c["kind"] == "prefill" else 8)
    return {"bytes": c["layers"] * per_layer, "flops": flops}


def tolerance(case):
    # Measured against exact(), times four. fp32 sums: 6e-7 for a layer of the per-token kernels (below 40 tokens),
    # 1.6e-7 for the GEMV, 3.5e-6 over 48 chained layers, 2.1e-5 at the worst of the cached chain's tokens. The grouped
    # GEMMs take fp32 activations as two bf16 terms, 16 significant bits: 4.4e-6 to 7.2e-6 a layer.
    if case["kind"] == "gemv":
        return {"rel": 7e-7, "max": 3e-5}
    if case["kind"] == "cached":
        return {"rel": 8e-5, "max": 3e-3}
    if case["kind"] == "decode" and case["tokens"] < 40:
        return {"rel": 1.4e-5, "max": 6e-4} if case["tokens"] == 1 else {"rel": 2.5e-6, "max": 1e-4}
    return {"rel": 3e-5, "max": 1.2e-3}


# ---- inputs ---------------------------------------------------------------------------
_context = None


def context():
    """The program's one context, kept for its life."""
    global _context
    if _context is None:
        _context = osm_hip.Context(0)
    return _context


def geometry(c):
    return osm_hip.geometry(c["hidden"], c["inter"], c["group"], META[c["meta"]])


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def quantize_q8(w):
    """MLX affine 8-bit: (packed words, scales, biases) of w [rows, cols], on the GPU."""
    rows, cols = w.shape
    g = w.view(rows, cols // Q8_GROUP, Q8_GROUP)
    lo, hi = g.amin(-1), g.amax(-1)
    scale = ((hi - lo) / 255.0).clamp_min(1e-8)
    q = ((g - lo[..., None]) / scale[..., None]).round().clamp(0, 255).to(torch.uint8)
    return q.view(rows, cols), scale, lo


def router_weights(c, seed, layer):
    """Router [E, D] and shared-gate vector [D], as fp32 values and as the layer takes them."""
    rows = torch.randn(c["experts"] + 1, c["hidden"], device="cuda", generator=generator(seed * 131 + 7 * layer + 3)) * 0.02
    if c["router"] == "f32":
        host = rows.cpu().numpy()
        return rows, host[:-1], host[-1]
    if c["router"] == "bf16":
        b = rows.to(torch.bfloat16)
        host = b.view(torch.int16).cpu().numpy().view(np.uint16)
        return b.float(), host[:-1], host[-1]
    q, s, b = quantize_q8(rows)
    value = (s[..., None] * q.view(*s.shape, Q8_GROUP).float() + b[..., None]).view(rows.shape)
    packed = q.cpu().numpy().view(np.uint32)
    sh, bh = s.cpu().numpy(), b.cpu().numpy()
    return value, (packed[:-1], sh[:-1], bh[:-1], Q8_GROUP), (packed[-1:], sh[-1:], bh[-1:], Q8_GROUP)


def norm_weight(c, seed, layer):
    return 1.0 + 0.02 * torch.randn(c["hidden"], device="cuda", generator=generator(seed * 131 + 7 * layer + 5))


def inputs(c, seed):
    g = generator(seed * 131 + 1)
    if chained(c):
        return torch.randn(c["tokens"], c["hidden"], device="cuda", generator=g)
    x = torch.randn(c["layers"], c["tokens"], c["hidden"], device="cuda", generator=g)
    return x.to(torch.bfloat16) if c["kind"] == "prefill" else x


def moe_layers(ctx, c, seed, max_tokens):
    out = []
    for l in range(c["layers"]):
        _, router, gate = router_weights(c, seed, l)
        shared = osm_hip.synth_expert_blob(ctx, seed, l, SHARED, geometry(c))
        out.append(osm_hip.MoeLayer(ctx, geometry(c), c["experts"], c["top_k"], router, ROUTER[c["router"]], gate,
                                    norm_weight(c, seed, l).cpu().numpy(), shared, max_tokens=max_tokens, rms_eps=EPS))
    return out


class _View:
    """A library buffer as torch sees it; the tensor made from it keeps the buffer."""

    def __init__(self, buffer):
        self.buffer = buffer
        ptr = osm_hip.load().osm_buffer_device_ptr(buffer.h)
        self.__cuda_array_interface__ = {"shape": (buffer.count,), "typestr": "<f4", "data": (ptr, False), "version": 3}


def projection(c, seed, i):
    g = generator(seed * 131 + 11 * i + 2)
    rows, cols, groups = c["rows"], c["cols"], c["cols"] // c["group"]
    words = torch.randint(-(2**31), 2**31, (rows, cols // 8), device="cuda", generator=g, dtype=torch.int64).to(torch.int32)
    scale = (torch.randn(rows, groups, device="cuda", generator=g).abs() * 0.02)
    bias = -8.0 * scale + 0.002 * torch.randn(rows, groups, device="cuda", generator=g)
    if c["meta"] == "bf16":
        scale, bias = scale.to(torch.bfloat16), bias.to(torch.bfloat16)
    return words, scale, bias


def prepare(case, seed):
    c, ctx = case, context()
    if c["kind"] == "gemv":
        as_numpy = (lambda t: t.view(torch.int16).cpu().numpy().view(np.uint16)) if c["meta"] == "bf16" else (lambda t: t.cpu().numpy())
        weights, outs, views = [], [], []
        for i in range(c["count"]):
            words, scale, bias = projection(c, seed, i)
            weights.append(osm_hip.Q4ProjectionWeights(ctx, words.cpu().numpy().view(np.uint32), c["rows"], c["cols"] // 8,
                                                       as_numpy(scale), as_numpy(bias), c["group"], META[c["meta"]]))
            y = osm_hip.FloatBuffer(ctx, c["rows"])
            outs.append(y)
            views.append(torch.as_tensor(_View(y), device="cuda"))
        x = osm_hip.FloatBuffer(ctx, c["cols"])
        x.upload(torch.randn(c["cols"], device="cuda", generator=generator(seed * 131 + 1)).cpu().numpy())
        return {"kind": "gemv", "weights": weights, "x": x, "outs": outs, "views": views}
    x = inputs(c, seed)
    g = geometry(c)
    if c["kind"] == "cached":
        store = osm_hip.ExpertStore(g, c["layers"], c["experts"])
        store.synthesize(ctx, seed)
        cache = osm_hip.ExpertCache(ctx, c["budget_mb"] * 2**20, store=store)
        return {"kind": "cached", "cache": cache, "store": store, "layers": moe_layers(ctx, c, seed, 1), "x": x.cpu().numpy()}
    slab = osm_hip.ExpertSlab(ctx, g, c["layers"], c["experts"])
    slab.synthesize(seed)
    s = {"kind": c["kind"], "slab": slab, "layers": moe_layers(ctx, c, seed, c["tokens"]), "x": x, "tokens": c["tokens"],
         "y": torch.empty(x.shape, dtype=torch.float32, device="cuda")}
    torch.cuda.synchronize()
    if chained(c):  # a generation loop replays its step
        s["scratch"] = torch.empty_like(x)
        s["graph"] = osm_hip.decode_graph(ctx, s["layers"], list(range(c["layers"])), slab, x.data_ptr(),
                                          s["y"].data_ptr(), s["scratch"].data_ptr(), c["tokens"], True)
    elif c["kind"] == "decode" and c["tokens"] <= 16:
        with ctx.capture() as cap:
            decode(s)
        s["graph"] = cap.graph
    return s


def decode(s):
    for l, layer in enumerate(s["layers"]):
        layer.decode_device(s["slab"], l, s["x"][l].data_ptr(), s["y"][l].data_ptr(), s["tokens"], sublayer=True)


# ---- one pass -------------------------------------------------------------------------
def run(state):
    s, ctx = state, context()
    if s["kind"] == "gemv":
        for w, y in zip(s["weights"], s["outs"]):
            osm_hip.run_q4_gemv_preloaded(ctx, w, s["x"], y)
        return s["views"]
    if s["kind"] == "cached":
        ids = list(range(len(s["layers"])))
        return [osm_hip.run_cached_layers(ctx, s["layers"], ids, s["cache"], s["x"][t:t + 1]) for t in range(len(s["x"]))]
    if s["kind"] == "prefill":
        for l, layer in enumerate(s["layers"]):
            layer.prefill_device(s["slab"], l, s["x"][l].data_ptr(), s["y"][l].data_ptr(), s["tokens"])
        return s["y"]
    if "graph" in s:
        s["graph"].launch()
    else:
        decode(s)
    return s["y"]


# ---- the same in 64 bits, in plain torch ------------------------------------------------
_M64 = (1 << 64) - 1


def _signed(v):
    v &= _M64
    return v - (1 << 64) if v >> 63 else v


def _shr(z, n):
    return (z >> n) & ((1 << (64 - n)) - 1)


def _mix(z):
    """The SplitMix64 finaliser, of a Python integer or an int64 tensor."""
    if isinstance(z, int):
        z = (z + 0x9E3779B97F4A7C15) & _M64
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _M64
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _M64
        return z ^ (z >> 31)
    z = z + _signed(0x9E3779B97F4A7C15)
    z = (z ^ _shr(z, 30)) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ _shr(z, 27)) * _signed(0x94D049BB133111EB)
    return z ^ _shr(z, 31)


def _stream(seed, a, b, t):
    return _mix(_mix(_mix(seed) ^ a) ^ ((b << 8) | t))


def _counter(stream, n):
    return torch.arange(n, device="cuda", dtype=torch.int64) + _signed(stream)


def _normal(stream, n):
    h0 = _mix(_counter(stream, n))
    h1 = _mix(h0)
    h2 = _mix(h1)
    s = sum((_shr(h, sh) & 0xFFFF) for h in (h0, h1, h2) for sh in (0, 16, 32, 48))
    return (s - 393210).float() * 2.0**-16


def _synth_matrix(seed, layer, expert, first, rows, cols, group):
    """One projection of a synthetic expert, dequantised to float64 [rows, cols]."""
    words = _mix(_counter(_stream(seed, layer, expert, first), rows * cols // 8))
    q = torch.stack([(words >> (4 * j)) & 0xF for j in range(8)], -1).view(rows, cols // group, group)
    n = rows * cols // group
    s = (_normal(_stream(seed, layer, expert, first + 1), n).abs() * 0.02).to(torch.bfloat16).float()
    b = (-8.0 * s + _normal(_stream(seed, layer, expert, first + 2), n) * 0.002).to(torch.bfloat16)
    s, b = s.double().view(rows, -1, 1), b.double().view(rows, -1, 1)
    return (q.double() * s + b).view(rows, cols)


def _expert(c, seed, layer, expert, x):
    D, I, G = c["hidden"], c["inter"], c["group"]
    gate = x @ _synth_matrix(seed, layer, expert, 0, I, D, G).t()
    up = x @ _synth_matrix(seed, layer, expert, 3, I, D, G).t()
    return (gate * torch.sigmoid(gate) * up) @ _synth_matrix(seed, layer, expert, 6, D, I, G).t()


def _moe(c, seed, layer, x):
    value, _, _ = router_weights(c, seed, layer)
    logits = x @ value.double().t()
    p = torch.softmax(logits[:, :-1], -1)
    w, ids = torch.topk(p, c["top_k"], dim=-1)
    w = w / w.sum(-1, keepdim=True)
    y = torch.sigmoid(logits[:, -1:]) * _expert(c, seed, layer, SHARED, x)
    for e in torch.unique(ids).tolist():
        t, j = (ids == e).nonzero(as_tuple=True)
        y.index_add_(0, t, w[t, j][:, None] * _expert(c, seed, layer, e, x[t]))
    return y


def _sublayer(c, seed, layer, x):
    scale = torch.rsqrt(x.square().mean(-1, keepdim=True) + float(np.float32(EPS)))
    return x + _moe(c, seed, layer, x * scale * norm_weight(c, seed, layer).double())


def exact(case, seed):
    c = case
    if c["kind"] == "gemv":
        x = torch.randn(c["cols"], device="cuda", generator=generator(seed * 131 + 1)).double()
        out = []
        for i in range(c["count"]):
            words, scale, bias = projection(c, seed, i)
            w = words.to(torch.int64)
            q = torch.stack([(w >> (4 * j)) & 0xF for j in range(8)], -1).view(c["rows"], -1, c["group"]).double()
            out.append((q * scale.double()[..., None] + bias.double()[..., None]).view(c["rows"], c["cols"]) @ x)
        return out
    x = inputs(c, seed).double()
    if c["kind"] == "prefill":
        return torch.stack([_moe(c, seed, l, x[l]) for l in range(c["layers"])])
    if not chained(c):
        return torch.stack([_sublayer(c, seed, l, x[l]) for l in range(c["layers"])])
    for l in range(c["layers"]):
        x = _sublayer(c, seed, l, x)
    return [r[None].cpu().numpy() for r in x] if c["kind"] == "cached" else x
