"""The q4 GEMV over 16-byte chunks at the edges of its dispatch, against float64."""

import numpy as np
import pytest

import osm_hip
from helpers import bf16_bits, bf16_to_f32, pack_q4

pytestmark = pytest.mark.gpu


# out_dim, in_dim, group: 16, 32 and 64 lanes to a row; one, two and four rows per wavefront with a ragged last
# workgroup; a partial and a second pass over the columns; groups of 32 to 128 and one that is no power of two; the
# word-wise kernel on either side of the size limit and for a row that is no whole number of chunks.
@pytest.mark.parametrize("out_dim,in_dim,group", [
    (2049, 512, 32), (16401, 512, 64), (16401, 480, 96), (4097, 1024, 128), (1027, 1056, 32), (515, 2080, 32),
    (4099, 2048, 64), (8201, 2048, 64), (257, 4992, 128), (2047, 512, 64), (513, 2056, 8)])
@pytest.mark.parametrize("meta", [osm_hip.F32, osm_hip.BF16])
def test_gemv_chunks(ctx, out_dim, in_dim, group, meta):
    rng = np.random.default_rng(out_dim + in_dim + group)
    q = rng.integers(0, 16, (out_dim, in_dim), dtype=np.uint32)
    s = np.abs(rng.normal(0, 0.02, (out_dim, in_dim // group))).astype(np.float32)
    b = (-8 * s + rng.normal(0, 0.002, s.shape)).astype(np.float32)
    if meta == osm_hip.BF16:
        s, b = bf16_bits(s), bf16_bits(b)
    x = rng.normal(0, 1, in_dim).astype(np.float32)
    w = osm_hip.Q4ProjectionWeights(ctx, pack_q4(q), out_dim, in_dim // 8, s, b, group, meta)
    xb, yb = osm_hip.FloatBuffer(ctx, in_dim), osm_hip.FloatBuffer(ctx, out_dim)
    xb.upload(x)
    osm_hip.run_q4_gemv_preloaded(ctx, w, xb, yb)
    if meta == osm_hip.BF16:
        s, b = bf16_to_f32(s), bf16_to_f32(b)
    sq = np.repeat(s.astype(np.float64), group, 1) * q
    bx = np.repeat(b.astype(np.float64), group, 1)
    x = x.astype(np.float64)
    # No term meets more than 32 roundings: its word's chain and sums, the words of three passes, the lanes' six levels.
    bound = 32 * 2.0**-24 * ((np.abs(sq) + np.abs(bx)) @ np.abs(x))
    assert np.all(np.abs(yb.download() - (sq + bx) @ x) <= bound)
