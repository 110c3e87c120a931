"""Near ties in clusters of two to eight experts, inside the picks and across
their end, equal rows among them: every token's ids against the oracle's, for
widths on both sides of what the split chains take."""

import numpy as np
import pytest

import oracle as O
import osm_hip

pytestmark = pytest.mark.gpu


# 128 columns: one run of 16 per chunk. 2,048: the widest of the split chains; 2,176 and 192 are left to the general
# form. Clusters of up to six open experts are settled apart, seven and eight go to the general form.
@pytest.mark.parametrize("D", [128, 192, 1920, 2048, 2176])
@pytest.mark.parametrize("clusters", [(2,), (3, 2), (6,), (7,), (2, 2, 2), (8, 3)])
def test_routing_clusters(ctx, D, clusters):
    I, G, E, k, T = 64, 64 if D % 64 == 0 else 32, 40, 6, 24
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
