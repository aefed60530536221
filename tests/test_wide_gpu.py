"""Many rows at once: the plane GEMM of large op-layer batches, and prompts fed
in passes over all their tokens.

The GEMM is compared with a float64 product of the same stored weights
(bar: rel-L2 1e-6, an fp32 sum's rounding at these K: about 2^-24 sqrt(K) / 4),
at sizes that leave remainders in the tile that takes them (rows modulo 128 or
64, weight rows modulo 256 or 64, K modulo 64): test_wide_linear on the 128 x
256 tile (1153 x 6928 in bf16 / bfp16 on the GEMM without planes),
test_wide_linear_paths on each tile, split and not.  Prompts are compared with the oracle's
token-by-token logits (the bars of parity_util), at row counts either side of
the plane kernels' first one, over several key tiles and over more rows than
one pass takes.
"""
import numpy as np
import pytest

import oracle_lib as O
from parity_util import compare_logits, greedy_identity
from test_decoder_gpu import build, prompts, tiny

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


# (kernel, K splits) a shape has to run on: both tiles, split and not, odd
# weight counts, K beyond 8192 (512 threads a row), about the smallest product
PATHS = [
    (4590, 640, 475, "ln", "i8 i4", ("planes", 1)),
    (3387, 1888, 125, "ln", "i8 i4", ("planes", 2)),
    (1375, 8608, 127, "rms1p", "i8 i4", ("planes", 5)),
    (1063, 560, 451, "ln", "i8 i4", ("planes", 1)),
    (5327, 528, 97, "rms1p", "i8 i4 bf16 bfp16", ("planes", 1)),
    (7029, 560, 386, "ln", "i8 i4 bf16 bfp16", ("planes_big", 1)),
    (9969, 2192, 281, "rms1p", "i8 i4 bf16 bfp16", ("planes_big", 2)),
    (3519, 8640, 133, "ln", "i8 i4 bf16 bfp16", ("planes_big", 8)),
]


@pytest.mark.parametrize("wd,m,k,b,norm,path", [(wd,) + c[:4] + (c[5],) for c in PATHS for wd in c[4].split()])
def test_wide_linear_paths(gpu, xe, wd, m, k, b, norm, path):
    wdtype = {"i8": xe.XE_I8, "i4": xe.XE_I4, "bf16": xe.XE_BF16, "bfp16": xe.XE_BFP16}[wd]
    code = {"ln": xe.XE_NORM_LN, "rms1p": xe.XE_NORM_RMS1P}[norm]
    assert xe.linear_path(wdtype, m, k, b, norm=code) == path
    test_wide_linear(gpu, xe, wd, m, k, b, norm)


def prompt_cfg(xe, family, wd):
    wdtype = {"i8": xe.XE_I8, "bf16": xe.XE_BF16, "bfp16": xe.XE_BFP16}[wd]
    cfg = tiny(xe, {"opt": xe.XE_OPT, "whisper": xe.XE_WHISPER}.get(family, xe.XE_GEMMA3), wdtype)
    if family == "gemma_hd128":
        cfg = cfg.replace(n_heads=4, n_kv_heads=2, head_dim=128)
    return cfg


@pytest.mark.parametrize("family,wd,batch,n", [
    ("gemma", "i8", 1, 4), ("gemma", "i8", 1, 129), ("gemma", "i8", 1, 130), ("gemma", "bf16", 3, 50),
    ("gemma", "i8", 2, 3), ("gemma", "i8", 2, 330), ("gemma_hd128", "i8", 2, 70), ("gemma", "bfp16", 22, 4),
    ("opt", "i8", 1, 70), ("opt", "bfp16", 5, 40), ("opt", "i8", 20, 111),
    ("opt", "bf16", 3, 66), ("whisper", "i8", 1, 5), ("whisper", "bfp16", 7, 29), ("whisper", "bf16", 3, 80)])
def test_prompt_passes_logits(gpu, xe, family, wd, batch, n):
    cfg = prompt_cfg(xe, family, wd)
    print("[case] prompt %s %s batch %d, %d tokens" % (family, wd, batch, n), flush=True)
    dec, om = build(xe, gpu, cfg, seed=31, batch=batch)
    pr = prompts(cfg, batch, n, seed=n)
    dec.feed(pr[:, :-1])
    got, _ = dec.step(pr[:, -1], np.full(batch, n - 1, np.int32))
    for p in range(n):
        want = om.step(pr[:, p], np.full(batch, p, np.int32))
    compare_logits(got, want, "prompt-%s-%s-b%d-n%d" % (family, wd, batch, n))
    dec.close()
    om.close()


@pytest.mark.parametrize("step", ["ll", "graph"])
@pytest.mark.parametrize("family,batch", [("opt", 1), ("opt", 3), ("gemma", 1), ("gemma", 4), ("whisper", 2)])
def test_prompt_without_a_workspace(gpu, xe, monkeypatch, step, family, batch):
    """No room for a pass (a limit of nothing, as an allocation that fails):
    the prompt is fed token by token on the step executor -- the low-latency
    launch with its forced tokens, or the graph replayed -- and the streams go
    on from there."""
    monkeypatch.setenv("XE_STEP", step)
    monkeypatch.setenv("XE_PROMPT_MB", "0")
    cfg = prompt_cfg(xe, family, "i8")
    print("[case] prompt without a workspace %s batch %d %s" % (family, batch, step), flush=True)
    dec, om = build(xe, gpu, cfg, seed=37, batch=batch)
    n = 7
    assert dec.executor(batch) == step and dec.prompt_pass(batch, n) == 0
    pr = prompts(cfg, batch, n, seed=4)
    dec.feed(pr[:, :-1])
    got, _ = dec.step(pr[:, -1], np.full(batch, n - 1, np.int32))
    for p in range(n):
        want = om.step(pr[:, p], np.full(batch, p, np.int32))
    compare_logits(got, want, "prompt-steps-%s-b%d-%s" % (family, batch, step))
    om.reset()
    greedy_identity(dec.generate(pr, 12), om, pr, "prompt-steps-%s-b%d-%s" % (family, batch, step))
    dec.close()
    om.close()


@pytest.mark.parametrize("family,batch,n,mb", [("gemma", 1, 75, "34"), ("gemma", 2, 330, "36"), ("gemma_hd128", 3, 41, "34.5"),
                                               ("opt", 2, 90, "35"), ("whisper", 5, 31, "35")])
def test_prompt_in_smaller_passes(gpu, xe, monkeypatch, family, batch, n, mb):
    """A workspace limit that a pass over the whole prompt exceeds (as an
    allocation that fails): smaller passes, the later ones over cached keys."""
    monkeypatch.delenv("XE_STEP", raising=False)
    cfg = prompt_cfg(xe, family, "i8")
    print("[case] smaller passes %s batch %d, %d tokens, %s MB" % (family, batch, n, mb), flush=True)
    dec, om = build(xe, gpu, cfg, seed=41, batch=batch)
    assert dec.prompt_pass(batch, n - 1) == n - 1
    monkeypatch.setenv("XE_PROMPT_MB", mb)
    assert 2 <= dec.prompt_pass(batch, n - 1) < n - 1
    pr = prompts(cfg, batch, n, seed=n)
    dec.feed(pr[:, :-1])
    got, _ = dec.step(pr[:, -1], np.full(batch, n - 1, np.int32))
    for p in range(n):
        want = om.step(pr[:, p], np.full(batch, p, np.int32))
    compare_logits(got, want, "prompt-passes-%s-b%d-n%d" % (family, batch, n))
    dec.close()
    om.close()


@pytest.mark.parametrize("wd", ["i8", "i4"])
@pytest.mark.parametrize("m,k,b,path", [(4100, 4096, 509, ("planes_big", 3)), (4590, 640, 475, ("planes", 1)),
                                        (7029, 560, 386, ("planes_big", 1)), (3519, 8656, 389, ("planes_big", 4))])
def test_wide_linear_range_within_a_row(gpu, xe, wd, m, k, b, path):
    """Rows whose elements differ by up to the whole fp32 range: one large
    element under a zero weight column, magnitudes spread over 2^-100 .. 2^100
    under weights that are non-zero in 48 columns only, between ordinary rows
    and in tiles of ordinary rows.  Bars: dense rows as above (they sum K
    comparable products); an output of n = 48 products within (n + 8) 2^-24 of
    the sum of their magnitudes (n roundings of an fp32 sum, operands to
    2^-23 each, the scale)."""
    _, ctx = gpu
    assert xe.linear_path(xe.XE_I8 if wd == "i8" else xe.XE_I4, m, k, b) == path
    print("[case] wide range %s m=%d k=%d b=%d" % (wd, m, k, b), flush=True)
    rng = np.random.default_rng(m + b)
    x = rng.standard_normal((b, k)).astype(np.float32)
    few = np.sort(rng.choice(np.arange(8, k), 48, replace=False))
    w = rng.standard_normal((m, k)).astype(np.float32)
    w[:, :8] = 0.0
    w[-64:] = 0.0
    w[-64:, few] = rng.standard_normal((64, 48)).astype(np.float32)
    ratios = [2.0 ** e for e in (8, 16, 20, 24, 26, 27, 28, 29, 30, 31, 36, 43, 60, 100)] + [1e9, 1e13, 1e30]
    at = rng.permutation(130)[:len(ratios)].tolist() + list(range(b - len(ratios), b))
    for r, ratio in zip(at, ratios * 2):
        x[r, r % 8] = ratio
    for r in (130, 131, b - 20):
        x[r] *= np.exp2(rng.integers(-100, 101, k)).astype(np.float32)
    x[132] = 0.0
    x[133] *= np.float32(2.0 ** -120)  # a small row: nothing is out of its range
    x[134, few[:24]] *= np.float32(2.0 ** -90)
    if wd == "i8":
        q, s = O.quant_rows_i8(w)
        h, val = ctx.register_weight_q8(q, s), q.astype(np.float64) * s[:, None].astype(np.float64)
    else:
        q, s = O.quant_rows_i4(w)
        h, val = ctx.register_weight_q4(q, s), O.unpack_i4(q).astype(np.float64) * s[:, None].astype(np.float64)
    got = ctx.gemv(h, x)
    h.free()
    want = x.astype(np.float64) @ val.T
    size = np.abs(x).astype(np.float64) @ np.abs(val).T
    diff = np.abs(got - want)
    few_err = (diff[:, -64:] / np.maximum(size[:, -64:], 1e-300)).max(axis=1)
    assert few_err.max() <= 56 * 2.0 ** -24, "row %d: %g of its products" % (few_err.argmax(), few_err.max())
    dense = np.linalg.norm(got - want, axis=1) / np.maximum(np.linalg.norm(want, axis=1), 1e-300)
    dense[[130, 131, b - 20]] = 0.0  # of few dominant products: the bound above
    assert dense.max() <= 2e-6, "row %d rel-L2 %g" % (dense.argmax(), dense.max())
