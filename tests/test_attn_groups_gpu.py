"""Split attention whose partials merge in groups: split counts either side of
one group (16 splits), of groups of eight (up to 64) and of sixteen, streams
of one split beside streams of many, against the oracle; and the merge inside
the split kernel equal to the separate merge launch bit for bit."""
import math

import numpy as np
import pytest

import oracle_lib as O
from test_attn_gpu import close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,hd,ctxlen,b", [
    (4, 1, 256, 1024, 1), (4, 1, 256, 1088, 1), (4, 1, 256, 4096, 3), (4, 1, 256, 4160, 2), (4, 1, 256, 16384, 1),
    (2, 2, 64, 3000, 5), (8, 1, 128, 9000, 2), (12, 12, 64, 2100, 1)])
def test_grouped_merge(gpu, monkeypatch, hq, hkv, hd, ctxlen, b):
    _, ctx = gpu
    print("[case] grouped merge hq=%d hkv=%d hd=%d ctx=%d b=%d" % (hq, hkv, hd, ctxlen, b), flush=True)
    rng = np.random.default_rng(hq + hd + ctxlen + b)
    lens = rng.integers(1, ctxlen + 1, b).astype(np.int32)
    lens[0] = ctxlen
    if b > 1:
        lens[1] = 3
    q = rng.standard_normal((b, hq, hd)).astype(np.float32)
    kc = O.bf16_bits(rng.standard_normal((b, hkv, ctxlen, hd)).astype(np.float32))
    vc = O.bf16_bits(rng.standard_normal((b, hkv, ctxlen, hd)).astype(np.float32))
    scale = 1.0 / math.sqrt(hd)
    monkeypatch.setenv("XE_ATTN_MERGE", "block")
    first = ctx.attn(q, kc, vc, lens, scale)
    again = ctx.attn(q, kc, vc, lens, scale)  # the arrival counters are zero again
    monkeypatch.setenv("XE_ATTN_MERGE", "launch")
    launched = ctx.attn(q, kc, vc, lens, scale)
    monkeypatch.delenv("XE_ATTN_MERGE")
    bits = np.asarray(first, np.float32).view(np.uint32)
    assert np.array_equal(bits, np.asarray(again, np.float32).view(np.uint32))
    assert np.array_equal(bits, np.asarray(launched, np.float32).view(np.uint32))
    close(first, O.attn_decode(q, kc, vc, lens, scale))


@pytest.mark.parametrize("hq,hkv,hd,ctxlen", [(4, 1, 256, 1088), (4, 1, 256, 4160), (8, 2, 128, 1100), (2, 2, 64, 3000)])
def test_merge_of_infinite_values(gpu, monkeypatch, hq, hkv, hd, ctxlen):
    """An infinity in the last split's values, with a split count that leaves
    the last group short: infinite in that dimension, untouched in the others,
    the same from both merges."""
    _, ctx = gpu
    print("[case] infinite value hq=%d hkv=%d hd=%d ctx=%d" % (hq, hkv, hd, ctxlen), flush=True)
    rng = np.random.default_rng(hq + ctxlen)
    q = rng.standard_normal((1, hq, hd)).astype(np.float32)
    kc = O.bf16_bits(rng.standard_normal((1, hkv, ctxlen, hd)).astype(np.float32))
    vc = O.bf16_bits(rng.standard_normal((1, hkv, ctxlen, hd)).astype(np.float32))
    lens, scale = np.array([ctxlen], np.int32), 1.0 / math.sqrt(hd)
    finite = O.attn_decode(q, kc, vc, lens, scale).reshape(hq, hd)
    vc[0, :, ctxlen - 1, 5] = 0x7F80
    vc[0, :, ctxlen - 1, 9] = 0xFF80
    for merge in ("block", "launch"):
        monkeypatch.setenv("XE_ATTN_MERGE", merge)
        got = np.asarray(ctx.attn(q, kc, vc, lens, scale)).reshape(hq, hd)
        assert np.all(got[:, 5] == np.inf) and np.all(got[:, 9] == -np.inf), merge
        rest = np.delete(np.arange(hd), [5, 9])
        close(got[:, rest], finite[:, rest])


@pytest.mark.parametrize("hq,hkv,hd", [(4, 1, 256), (8, 1, 64), (16, 2, 64), (8, 1, 256), (8, 2, 128), (12, 12, 64)])
def test_splits_fit_the_chip(gpu, hq, hkv, hd):
    """More than 64 splits a stream only while all workgroups are resident: two
    a CU, one where 8 query heads share a key head (a second round of
    workgroups took 8 x 64 at 9000 keys of two streams from 28.5 to 34.5 us);
    512 outputs a key head merge in a launch beyond one group of splits."""
    _, ctx = gpu
    resident = 256 if hq // hkv == 8 else 512
    for b in (1, 2, 3, 5, 16, 64):
        for n in (1, 64, 65, 1024, 1025, 9000, 32768, 1 << 17):
            splits, launch = ctx.attn_splits(b, hq, hkv, hd, n)
            assert 1 <= splits <= min(256, -(-n // 64))
            assert splits <= 64 or splits * b * hkv <= resident
            outs = hq // hkv * hd
            assert launch == (splits > 1 and (outs > 512 or (outs == 512 and splits > 16)))
    print("[case] resident splits %d/%d x %d" % (hq, hkv, hd), flush=True)
    rng = np.random.default_rng(hq + hd)
    n = 9000
    q = rng.standard_normal((2, hq, hd)).astype(np.float32)
    kc = O.bf16_bits(rng.standard_normal((2, hkv, n, hd)).astype(np.float32))
    vc = O.bf16_bits(rng.standard_normal((2, hkv, n, hd)).astype(np.float32))
    lens = np.array([n, 5000], np.int32)
    close(ctx.attn(q, kc, vc, lens, 0.1), O.attn_decode(q, kc, vc, lens, 0.1))
