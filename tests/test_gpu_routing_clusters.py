"""Near ties in clusters of two to eight experts, inside the picks and across
their end, equal rows among them: every token's ids against the oracle's, for
widths on both sides of what the split chains take."""

import numpy as np
import pytest

import oracle as O
import osm_hip
from helpers import bf16_bits
from test_gpu_routing_exact import _libm_expf, _softmax_sum

pytestmark = pytest.mark.gpu


# 128 columns: one run of 16 per chunk. 2,048: the widest of the split chains; 2,176 and 192 are left to the general
# form, in the sublayer form too. Clusters of up to six open experts are settled apart, seven and eight go to the general
# form. More than 512 experts: four to a thread. Intermediate 1,088: more than 512 workgroups for one token, which then
# takes the general form too.
@pytest.mark.parametrize("D,E,I", [(128, 40, 64), (192, 40, 64), (1920, 40, 64), (2048, 40, 64), (2176, 40, 64),
                                   (384, 520, 64), (2176, 520, 64), (384, 40, 1088), (256, 520, 1088)])
@pytest.mark.parametrize("clusters", [(2,), (3, 2), (6,), (7,), (2, 2, 2), (8, 3)])
def test_routing_clusters(ctx, D, E, I, clusters):
    G, k, T = 64 if D % 64 == 0 else 32, 6, 24
    seed = 5000 + D + sum(c * 10**i for i, c in enumerate(clusters))
    rng = np.random.default_rng(seed)
    g = osm_hip.geometry(D, I, G, osm_hip.BF16)
    slab = osm_hip.ExpertSlab(ctx, g, 1, E)
    slab.synthesize(seed)
    router = rng.normal(0, 1.0 / np.sqrt(D), (E, D)).astype(np.float32)
    ids = rng.permutation(E)
    at = 0
    for m in clusters:
        base = router[ids[at]] * np.float32(rng.uniform(1.0, 2.5))
        for j in range(m):  # some rows equal, the others a few units in the last place apart
            router[ids[at + j]] = base * np.float32(1 + int(rng.integers(-3, 4)) * 2.0**-22)
        at += m
    nw = (1 + rng.normal(0, 0.02, D)).astype(np.float32)
    moe = osm_hip.MoeLayer(ctx, g, E, k, router, osm_hip.F32, None, nw, None, max_tokens=T, rms_eps=1e-6)
    moe.set_path(osm_hip.PATH_PER_TOKEN)
    x = rng.normal(0, 1, (T, D)).astype(np.float32)
    xd, yd = ctx.alloc(T * D * 4), ctx.alloc(T * D * 4)
    moe.routing_stats(reset=True)
    for sublayer in (False, True):
        xr = O.rms_norm(x, T, D, nw, 1e-6).reshape(T, D) if sublayer else x
        want = [O.route_qwen_top_k(xr[t], router, D, E, k, True)["ids"] for t in range(T)]
        xd.upload(x)
        moe.decode_device(slab, 0, xd.ptr, yd.ptr, T, sublayer=sublayer)  # the selection kernel
        got = moe.routing(T)["ids"]
        for t in range(T):
            assert np.array_equal(got[t], want[t]), (sublayer, t)
        for t in range(6):  # one token: gate/up selects
            xd.upload(x[t:t + 1])
            moe.decode_device(slab, 0, xd.ptr, yd.ptr, 1, sublayer=sublayer)
            assert np.array_equal(moe.routing(1)["ids"][0], want[t]), (sublayer, t)
    assert moe.routing_stats()["exact"] > 0


# ---------------------------------------------------------------------------
# Logits set exactly: the router's input is 1 in its first column and 0
# elsewhere, so expert e's logit is router[e, 0] in whatever order it is summed.
# In the sublayer form that input is 16 normalised at 256 columns (the mean of
# the squares is 1) times a norm weight of 1/16. The bounds do not know that
# the sums are exact: logits a few units in the last place apart are open.

EXACT_D = 256


def rows_for(logits):
    router = np.zeros((len(logits), EXACT_D), np.float32)
    router[:, 0] = logits
    return router


def encoded(router, kind):
    """The layer's router arguments for a router of whole numbers from -5 to 250 (kinds but f32)."""
    if kind == "f32":
        return router, osm_hip.F32
    if kind == "q8":  # value q - 5, groups of 32
        q = (router + 5).astype(np.uint32)
        packed = (q[:, 0::4] | (q[:, 1::4] << 8) | (q[:, 2::4] << 16) | (q[:, 3::4] << 24)).astype(np.uint32)
        one = np.ones((len(router), router.shape[1] // 32), np.float32)
        return (packed, one, -5 * one, 32), osm_hip.AFFINE_Q8
    return (router.astype(np.float16), osm_hip.F16) if kind == "f16" else (bf16_bits(router), osm_hip.BF16)


def every_selection(ctx, router, k, x, xin, nw, kind="f32"):
    """(label, ids, stats) of each kernel that selects for the router's input x (xin, normalised with nw): one token and
    four (inside gate/up), 16 (the selection kernel behind the per-token router), 48 and 320 (grouped, behind the router
    GEMM, of which routers that are not bf16 and of few rows take the second alone), with and without the norm, and 1,024
    bf16 tokens."""
    E, D = router.shape
    I, G = 128, 64
    g = osm_hip.geometry(D, I, G, osm_hip.BF16)
    slab = osm_hip.ExpertSlab(ctx, g, 1, E)
    slab.synthesize(1)
    moe = osm_hip.MoeLayer(ctx, g, E, k, *encoded(router, kind), None, nw, None, max_tokens=1024, rms_eps=1e-20)
    assert np.array_equal(O.rms_norm(xin, 1, D, nw, 1e-20), x)
    for sublayer in (False, True):
        for T, path in ((1, osm_hip.PATH_PER_TOKEN), (4, osm_hip.PATH_PER_TOKEN), (16, osm_hip.PATH_PER_TOKEN),
                        (48, osm_hip.PATH_GROUPED), (320, osm_hip.PATH_GROUPED)):
            moe.set_path(path)
            xd, yd = ctx.alloc(T * D * 4), ctx.alloc(T * D * 4)
            xd.upload(np.tile(xin if sublayer else x, (T, 1)))
            moe.routing_stats(reset=True)
            moe.decode_device(slab, 0, xd.ptr, yd.ptr, T, sublayer=sublayer)
            yield (T, sublayer), moe.routing(T)["ids"], moe.routing_stats()
    T = 1024
    xd, yd = ctx.alloc(T * D * 2), ctx.alloc(T * D * 4)
    xd.upload(np.tile((x.view(np.uint32) >> 16).astype(np.uint16), (T, 1)))  # x is bf16 already
    moe.routing_stats(reset=True)
    moe.prefill_device(slab, 0, xd.ptr, yd.ptr, T)
    yield (T, "prefill"), moe.routing(T)["ids"], moe.routing_stats()


def check_every_selection(ctx, logits, k):
    x = np.zeros(EXACT_D, np.float32)
    x[0] = 1.0
    return check_rows(ctx, rows_for(logits), k, x, 16 * x, 1 / 16)


def check_rows(ctx, router, k, x, xin, nw):
    want = O.route_qwen_top_k(x, router, EXACT_D, len(router), k, True)["ids"]
    for label, ids, _ in every_selection(ctx, router, k, x, xin, np.full(EXACT_D, nw, np.float32)):
        assert np.array_equal(ids, np.tile(want, (len(ids), 1))), (label, ids[0], want)
    return list(want)


def distant(E=40):
    return np.full(E, -5, np.float32)


# Three experts whose logits, 7 below the largest, differ by less than the rounding of that distance: one probability,
# so the reference takes id 10, the lowest logit of the three (or the three in id order). Ranked by the logit, 20 and
# 30 are the neighbours across the end of the picks, in id order themselves.
@pytest.mark.parametrize("k,want", [(2, [0, 10]), (3, [0, 10, 20]), (4, [0, 10, 20, 30])])
@pytest.mark.parametrize("l30", [1 + 2.0**-23, 1 + 2.0**-22])
def test_one_probability_across_the_picks(ctx, k, want, l30):
    logits = distant()
    logits[0], logits[20], logits[30], logits[10] = 8, 1 + 2.0**-22, l30, 1
    assert check_every_selection(ctx, logits, k) == want


def quotient_tie(extra):
    """(logits, want): 20 and 30 share a logit, 10's exp is one unit below theirs and divides by the softmax sum to the
    same probability; `extra` more experts are within the bounds' reach, too far for a tie."""
    expf = _libm_expf()
    rng = np.random.default_rng(3)
    E = 40 + extra
    f = np.float32
    while True:
        logits = (-1 - 2 * rng.random(E)).astype(np.float32)
        logits[0] = 1
        a = f(0.15 + 0.2 * rng.random())
        b = f(a - f(2.0**-24))
        ea, eb = expf(f(a - 1)), expf(f(b - 1))
        if eb == ea or np.nextafter(eb, f(1)) != ea:
            continue
        logits[20], logits[30], logits[10] = a, a, b
        for j in range(extra):
            logits[40 + j] = a - f(1e-6) * f(1 + j % 8)
        if f(ea / _softmax_sum(logits, expf)) == f(eb / _softmax_sum(logits, expf)):
            return logits


# The two of one exp are the neighbours across the end of the picks; the reference picks 10. Up to 64 candidates are
# ranked in one wavefront's registers, more in LDS.
@pytest.mark.parametrize("extra", [0, 70])
def test_quotient_tie_behind_an_equal_exp(ctx, extra):
    assert check_every_selection(ctx, quotient_tie(extra), 2) == [0, 10]


# Logits that the reference's fp32 sums move by tens (inputs of 1; a little over 2^26, then n columns of +-4, half a
# unit in its last place, which they drop, then the first taken off again; the rest in the last column). What the device's fp64 sums say of the distance to
# the largest logit is then no guide to the reference's exps.
def moved(row, n, step, ref):
    big = 2.0**26 + 16
    row[0], row[1:n + 1], row[n + 1], row[-1] = big, step, -big, ref


def distance_rows(case):
    router = np.zeros((40, EXACT_D), np.float32)
    router[:, -1] = -2000
    if case == "open":  # 100 and, by the device's sums, 30 and 28: for the reference 150 and more below, p = 0
        router[0, -1] = 100
        moved(router[33], 20, 4, -50)
        moved(router[36], 22, 4, -60)
    elif case == "proven":  # 0 and -79, apart by their bounds: for the reference -127, p = 0
        router[0, -1] = 0
        moved(router[36], 12, 4, -127)
    else:  # -1 for the device, 59 for the reference, 58.5 above three logits that round to one distance from it
        moved(router[5], 15, -4, 59)
        router[20, -1] = router[30, -1] = 0.5
        router[10, -1] = 0.5 - 13 * 2.0**-23
    return router


@pytest.mark.parametrize("case,want", [("open", [0, 1]), ("proven", [0, 1]), ("above", [5, 10])])
def test_distance_from_the_largest_logit(ctx, case, want):
    x = np.ones(EXACT_D, np.float32)
    assert check_rows(ctx, distance_rows(case), 2, x, x, 1.0) == want


# Chains whose running value leaves their exact sum by tens (as above), from column `at` on, so that a chunk of 32 columns
# starts from none of the values around its exact start and is run once more; their logits, in the opposite order to the
# device's, decide the picks. 0: every chunk but the first; 20: across a boundary, where the value is a few units off, and
# the rest; 200: the last chunk alone.
@pytest.mark.parametrize("at", [0, 20, 200])
def test_chunk_from_another_start(ctx, at):
    router = np.zeros((40, EXACT_D), np.float32)
    router[:, -1] = -2000
    moved(router[33, at:], 20, 4, 3)  # 83 by the device's sums
    moved(router[36, at:], 10, 4, 5)  # 45
    x = np.ones(EXACT_D, np.float32)
    want = O.route_qwen_top_k(x, router, EXACT_D, 40, 2, True)["ids"]
    assert list(want) == [36, 33]
    for label, ids, stats in every_selection(ctx, router, 2, x, x, x):
        assert np.array_equal(ids, np.tile(want, (len(ids), 1))), (label, ids[0])
        assert stats["exact"] == len(ids) and stats["exact_all"] == 0, (label, stats)


# Logits a + b s for a first column of 1 and one of s near the end (past column 2,048 at hidden 4,096), the router's
# values whole numbers that every dtype holds. 40 experts are two to a thread, 520 four.
SHAPES = [(256, 40), (1024, 520), (4096, 520)]


def two_columns(ctx, D, E, kind, k, s, logits):
    router = np.zeros((E, D), np.float32)
    router[:, 0] = -5
    for e, (a, b) in logits.items():
        router[e, 0], router[e, D - 2] = a, b
    x = np.zeros(D, np.float32)
    x[0], x[D - 2] = 1, s
    root = np.float32(D**0.5)
    want = O.route_qwen_top_k(x, router, D, E, k, True)["ids"]
    for label, ids, stats in every_selection(ctx, router, k, x, root * x, np.full(D, 1 / root, np.float32), kind):
        assert np.array_equal(ids, np.tile(want, (len(ids), 1))), (label, ids[0], want)
        assert stats["exact"] == len(ids), (label, stats)
        yield label, len(ids), stats, list(want)


# Two clusters that the bounds leave open, one across the end of the picks, every logit apart by more than the tie margin:
# no token needs the full recompute.
@pytest.mark.parametrize("D,E", SHAPES)
@pytest.mark.parametrize("kind", ["f32", "f16", "bf16", "q8"])
def test_open_clusters_every_router(ctx, D, E, kind):
    logits = {7: (8, 2), 30: (8, 0), 3: (8, 1), 12: (4, 0), 25: (4, 1)}
    for label, tokens, stats, want in two_columns(ctx, D, E, kind, 4, 2.0**-17, logits):
        assert want == [7, 3, 30, 25] and stats["exact_all"] == 0, (label, stats)


# Every pick but the first more than 80 below the largest logit: every token needs it, and the second column decides.
@pytest.mark.parametrize("D,E", SHAPES)
@pytest.mark.parametrize("kind", ["f32", "f16", "bf16", "q8"])
def test_full_recompute_every_router(ctx, D, E, kind):
    logits = {0: (100, 0), 20: (15, 200), 30: (15, 100), 10: (15, 0)}
    for label, tokens, stats, want in two_columns(ctx, D, E, kind, 3, 2.0**-13, logits):
        assert want == [0, 20, 30] and stats["exact_all"] == tokens, (label, stats)
