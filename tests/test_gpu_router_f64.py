"""Routers that are not bf16 through the fp64 router GEMM: every token's
picks against the oracle's, at the K ranges, token tiles and router rows
where the GEMM's edges lie."""

import math

import numpy as np
import pytest

import oracle as O
import osm_hip
from helpers import bf16_bits, bf16_to_f32, max_abs, rel_l2
from test_gpu_router_q8 import dequant, quantize_q8

pytestmark = pytest.mark.gpu


def layer(ctx, kind, D, E, k, T, seed, group=64, norm=None):
    rng = np.random.default_rng(seed)
    I, G = 128, 64
    g = osm_hip.geometry(D, I, G, osm_hip.BF16)
    slab = osm_hip.ExpertSlab(ctx, g, 1, E)
    slab.synthesize(seed)
    shared = O.synth_expert_blob(seed, 0, O.SHARED_EXPERT_ID, D, I, G)
    w = rng.normal(0, 0.9 / np.sqrt(D), (E + 1, D)).astype(np.float32)
    w[1] = w[0] * np.float32(1 + 2.0**-21)  # a pair whose logits the bounds cannot tell apart
    if kind == "q8":
        r, sg = quantize_q8(w[:-1], group, rng), quantize_q8(w[-1:], group, rng)
        value, gate = dequant(*r, group), dequant(*sg, group)
        moe = osm_hip.MoeLayer(ctx, g, E, k, r + (group,), osm_hip.AFFINE_Q8, sg + (group,), norm, shared, max_tokens=T)
    else:
        dt, code = (np.float16, osm_hip.F16) if kind == "f16" else (np.float32, osm_hip.F32)
        w = w.astype(dt)
        value, gate = w[:-1].astype(np.float32), w[-1:].astype(np.float32)
        moe = osm_hip.MoeLayer(ctx, g, E, k, w[:-1], code, w[-1], norm, shared, max_tokens=T)
    return slab, moe, value, gate


def check(moe, x, value, gate, E, k, normed=None):
    """x: the layer's input; normed: the reference's normalised input in the sublayer form."""
    r = moe.routing(len(x), normalized=normed is not None)
    ref = x if normed is None else normed
    if normed is not None:
        x = r["normalized"].reshape(ref.shape)
        # A sum of squares is within D roundings either side, halved by the root; four more operations.
        assert np.all(np.abs(x - ref) <= (x.shape[1] + 8) * 2.0**-24 * np.abs(ref))
    exact = x.astype(np.float64) @ value.astype(np.float64).T
    # Summed in fp64 (at most 2,048 roundings of 2^-53) and rounded to fp32 once.
    bound = 2.0**-24 * np.abs(exact) + 2.0**-40 * (np.abs(x).astype(np.float64) @ np.abs(value).astype(np.float64).T)
    assert np.all(np.abs(r["logits"] - exact) <= bound)
    for t in range(len(x)):
        ora = O.route_qwen_top_k(ref[t], value, x.shape[1], E, k, True)
        assert np.array_equal(r["ids"][t], ora["ids"]), t
        # The weights are the picks' softmax of the logits checked above, each exp, sum and quotient rounded.
        p = np.exp(r["logits"][t][ora["ids"]].astype(np.float64) - r["logits"][t].max())
        assert max_abs(r["weights"][t], p / p.sum()) <= 1e-6
    s = 1 / (1 + np.exp(-(x.astype(np.float64) @ gate[0].astype(np.float64))))
    assert max_abs(r["shared_gate"], s) <= 2e-6


# D 2048, 768 and 384: K ranges of 512, 256 and 128 columns. E + 1 rows fill a 64-row block, or leave one row in the
# next. 40 tokens are the fewest; 49 and 257 leave one in the last tile of 16. fp32 input takes the GEMM from 12,288
# products of tokens and rows on (hidden 2,048 and below), bf16 from a third: (768, 63, 40) takes the per-token router.
@pytest.mark.parametrize("D,E,T", [(2048, 128, 49), (768, 63, 40), (384, 64, 257), (2048, 512, 64), (2048, 256, 49),
                                   (768, 319, 40)])
@pytest.mark.parametrize("kind", ["q8", "f32", "f16"])
def test_router_f64(ctx, D, E, T, kind):
    k, seed = 6, 900 + D + T
    slab, moe, value, gate = layer(ctx, kind, D, E, k, T, seed)
    x = O.synth_tokens(seed, 0, T, D)
    xd, yd = ctx.alloc(T * D * 4), ctx.alloc(T * D * 4)
    xd.upload(x)
    moe.set_path(osm_hip.PATH_GROUPED)
    moe.routing_stats(reset=True)
    moe.decode_device(slab, 0, xd.ptr, yd.ptr, T)
    check(moe, x, value, gate, E, k)
    assert moe.routing_stats()["exact"] < T  # the bounds prove some of them
    bits = ((x.view(np.uint32) + 0x7FFF + ((x.view(np.uint32) >> 16) & 1)) >> 16).astype(np.uint16)
    xd.upload(bits)
    moe.prefill_device(slab, 0, xd.ptr, yd.ptr, T)
    check(moe, (bits.astype(np.uint32) << 16).view(np.float32).reshape(T, D), value, gate, E, k)


# The sublayer form: a word of 8 columns per thread with a part of the workgroup idle (384, 640), one (2,048), and up to
# two, three and four (2,176, 4,224, 6,400 and 8,192, the widest, in 16 K ranges); enough tokens for the GEMM. Affine q8 groups that hold whole
# 64-column runs (64, 128) and that do not.
@pytest.mark.parametrize("kind,D,E,group", [
    ("q8", 384, 64, 4), ("q8", 384, 63, 48), ("q8", 640, 64, 32), ("q8", 640, 64, 128), ("f32", 384, 64, 0),
    ("q8", 2048, 512, 64), ("f32", 2048, 128, 0), ("q8", 2176, 64, 64), ("f16", 4224, 64, 0), ("f32", 6400, 64, 0),
    ("q8", 8192, 64, 64)])
def test_router_f64_sublayer(ctx, kind, D, E, group):
    k, T, seed = 6, 201, 700 + D + group
    nw = (1 + np.random.default_rng(seed).normal(0, 0.02, D)).astype(np.float32)
    slab, moe, value, gate = layer(ctx, kind, D, E, k, T, seed, group, nw)
    x = O.synth_tokens(seed, 0, T, D) * np.float32(1.5)
    xd, yd = ctx.alloc(T * D * 4), ctx.alloc(T * D * 4)
    xd.upload(x)
    out = []
    for sublayer in (False, True):
        normed = O.rms_norm(x, T, D, nw, 1e-6).reshape(T, D) if sublayer else None
        for path in (osm_hip.PATH_PER_TOKEN, osm_hip.PATH_GROUPED):
            moe.set_path(path)
            moe.routing_stats(reset=True)
            moe.decode_device(slab, 0, xd.ptr, yd.ptr, T, sublayer=sublayer)
            check(moe, x, value, gate, E, k, normed)
            assert moe.routing_stats()["exact"] < T  # the bounds prove some of them
            out.append(yd.download(np.float32, T * D))
        assert rel_l2(out[-1], out[-2]) <= 2e-5  # the experts' GEMMs take the input as two bf16 terms


def test_partial_sums_in_fp64(ctx):
    # Five K ranges of 128 columns. Rows 0-31: 2^26 at the end of the first, taken off at the end of the second, the
    # rest multiples of 2^-24 below 1. Their sums are exact in fp64, and the logit is the exact sum rounded once; ranges
    # held in 48 bits would be off by up to 2^-22. Row 32: the second range's own sum is beyond fp32, the running sums
    # of the reference are not.
    rng = np.random.default_rng(1)
    D, E, k, T = 640, 64, 6, 200
    w = (rng.integers(-2**24, 2**24, (E, D)) * 2.0**-24).astype(np.float32)
    w[:32, 127], w[:32, 255] = 2.0**26, -(2.0**26)
    w[32] = 0
    w[32, [0, 128, 129, 256, 639]] = [-3e38, 3e38, 3e38, -3e38, 20]
    g = osm_hip.geometry(D, 128, 64, osm_hip.BF16)
    slab = osm_hip.ExpertSlab(ctx, g, 1, E)
    slab.synthesize(1)
    moe = osm_hip.MoeLayer(ctx, g, E, k, w, osm_hip.F32, None, None, None, max_tokens=T)
    want = np.array([math.fsum(row) for row in w.tolist()], np.float32)
    ids = O.route_qwen_top_k(np.ones(D, np.float32), w, D, E, k, True)["ids"]
    for path in (osm_hip.PATH_PER_TOKEN, osm_hip.PATH_GROUPED):
        moe.set_path(path)
        r = moe.run_slab(slab, 0, np.ones((T, D), np.float32))
        assert np.array_equal(r["logits"], np.tile(want, (T, 1))), path
        assert np.array_equal(r["ids"], np.tile(ids, (T, 1))), path


# Inputs whose squares are below fp32's smallest number, against a router large enough for logits of the usual size: the
# bounds have to know the products' size all the same. Each expert's columns are blocks of 16, eight values and their
# negatives in an order of its own, which leave nothing, and its logit in the last column; the reference's sums of them
# are off by a multiple of the gaps between the logits, token by token.
@pytest.mark.parametrize("kind", ["f32", "bf16"])
def test_bounds_of_tiny_inputs(ctx, kind):
    rng = np.random.default_rng(4)
    D, E, k, T = 384, 64, 6, 200
    a = np.abs(bf16_to_f32(bf16_bits(rng.normal(0, 1e4, (23, 8)))))
    w = np.zeros((E, D), np.float32)
    for e in range(E):
        for b in range(23):
            w[e, 16 * b:16 * b + 16] = rng.permutation(np.concatenate([a[b], -a[b]]))
        w[e, D - 1] = 1 + (37 * e % E) * 2.0**-7
    w *= np.float32(2.0**80)
    x = np.repeat((rng.uniform(0.5, 2, (T, 1)) * 2.0**-80).astype(np.float32), D, 1)
    g = osm_hip.geometry(D, 128, 64, osm_hip.BF16)
    slab = osm_hip.ExpertSlab(ctx, g, 1, E)
    slab.synthesize(1)
    r, code = (bf16_bits(w), osm_hip.BF16) if kind == "bf16" else (w, osm_hip.F32)
    moe = osm_hip.MoeLayer(ctx, g, E, k, r, code, None, None, None, max_tokens=T)
    moe.set_path(osm_hip.PATH_GROUPED)
    got = moe.run_slab(slab, 0, x)["ids"]
    for t in range(T):
        assert np.array_equal(got[t], O.route_qwen_top_k(x[t], w, D, E, k, True)["ids"]), t
