"""Many rows at once: the plane GEMM of large op-layer batches.

Compared with a float64 product of the same stored weights (bar: rel-L2 1e-6,
an fp32 sum's rounding at these K: about 2^-24 sqrt(K) / 4), at sizes that
leave remainders in every tile: rows modulo 64 and 128, weight rows modulo 64
and 256, K modulo 64.
"""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wd", ["i8", "i4", "bf16", "bfp16"])
@pytest.mark.parametrize("m,k,b,norm", [(16401, 1040, 211, "ln"), (1153, 6928, 449, "rms1p"), (4100, 4096, 512, "none")])
def test_wide_linear(gpu, xe, wd, m, k, b, norm):
    _, ctx = gpu
    print("[case] wide linear %s m=%d k=%d b=%d %s" % (wd, m, k, b, norm), flush=True)
    rng = np.random.default_rng(m + k + b)
    w = rng.standard_normal((m, k)).astype(np.float32) * 0.02
    bias = rng.standard_normal(m).astype(np.float32)
    x = rng.standard_normal((b, k)).astype(np.float32)
    x[:, ::97] *= 50.0  # a few large channels, as a residual stream has
    x[3] = 0.0
    x[5] *= 1e-30
    gamma = rng.normal(1.0, 0.1, k).astype(np.float32)
    beta = rng.normal(0.0, 0.1, k).astype(np.float32)
    if wd == "i8":
        q, s = O.quant_rows_i8(w)
        h, val = ctx.register_weight_q8(q, s, bias), q.astype(np.float64) * s[:, None].astype(np.float64)
    elif wd == "i4":
        q, s = O.quant_rows_i4(w)
        h, val = ctx.register_weight_q4(q, s, bias), O.unpack_i4(q).astype(np.float64) * s[:, None].astype(np.float64)
    elif wd == "bf16":
        bits = O.bf16_bits(w)
        h, val = ctx.register_weight_bf16(bits, bias), O.bf16_to_f32(bits).astype(np.float64)
    else:
        mant, exps = O.bfp16_encode(w)
        h, val = ctx.register_weight_bfp16(mant, exps, bias), O.bfp16_decode(mant, exps).astype(np.float64)
    xd = x.astype(np.float64)
    if norm == "ln":
        ctx.set_norm(h, xe.Norm.Ln(gamma, beta, 1e-5))
        xd = xd - xd.mean(1, keepdims=True)
        xd = xd / np.sqrt((xd * xd).mean(1, keepdims=True) + np.float32(1e-5)) * gamma + beta
    elif norm == "rms1p":
        ctx.set_norm(h, xe.Norm.Rms1p(gamma, 1e-6))
        xd = xd / np.sqrt((xd * xd).mean(1, keepdims=True) + np.float32(1e-6)) * (1.0 + gamma.astype(np.float64))
    got = ctx.gemv(h, x) if norm == "none" else ctx.fused_norm_gemv(h, x)
    h.free()
    want = xd @ val.T + bias
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= 1e-6, "rel-L2 %g" % err
    # row by row: a row's exponent, padding or order mixed up shows here
    rows = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert rows.max() <= 2e-6, "row %d rel-L2 %g" % (rows.argmax(), rows.max())
