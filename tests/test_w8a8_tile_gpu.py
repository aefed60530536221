"""W8A8 at the edges of its tiles: rows modulo 64, weight rows modulo 64 (and
counts that are no multiple of four, whose outputs take 4-byte stores), K
modulo 128, both sides of the tile kernel's first row counts.  Bit-exact:
integer sums, then the oracle's own float operations."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,b", [(1001, 1040, 77), (65, 16, 33), (130, 2064, 9), (64, 512, 17), (300, 528, 32),
                                   (257, 4112, 130), (4, 128, 512), (3, 1552, 16)])
@pytest.mark.parametrize("epi", ["none", "bias", "silu_bias"])
def test_w8a8_tile_edges(gpu, xe, m, k, b, epi):
    dev, ctx = gpu
    print("[case] w8a8 tile m=%d k=%d b=%d %s" % (m, k, b, epi), flush=True)
    rng = np.random.default_rng(m + k + b)
    q = rng.integers(-127, 128, (m, k)).astype(np.int8)
    s = rng.uniform(0.001, 0.02, m).astype(np.float32)
    bias = rng.standard_normal(m).astype(np.float32)
    x = rng.standard_normal((b, k)).astype(np.float32)
    x[b // 2, k // 3] = np.nan  # quantises to 0 and does not count in the scale
    w = ctx.register_weight_q8(q, s, bias)
    xq = rng.integers(-128, 128, (b, k)).astype(np.int8)
    acc = ctx.gemv_i8act(w, xq)
    assert np.array_equal(acc, xq.astype(np.int64) @ q.astype(np.int64).T)
    code = {"none": xe.XE_EPI_NONE, "bias": xe.XE_EPI_BIAS, "silu_bias": xe.XE_EPI_SILU_BIAS}[epi]
    xb, yb, sb = xe.Buf.from_array(dev, x), xe.Buf(dev, b * m * 4), xe.Buf(dev, 4)
    ctx.w8a8_linear_dev(w, xb, b, code, yb, sb)
    ctx.synchronize()
    got = yb.read(np.float32, b * m).reshape(b, m)
    want, sa = O.w8a8_linear(x, q, s, None if epi == "none" else bias, epi=code)
    assert np.array_equal(sb.read(np.float32, 1), np.float32([sa]))
    assert np.array_equal(got.view(np.uint32), np.asarray(want, np.float32).reshape(b, m).view(np.uint32))
    w.free()
    for buf in (xb, yb, sb):
        buf.free()
