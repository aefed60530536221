"""The rule that says which kernel a linear runs on, over the whole range of
sizes (host code, no device): what each kernel accepts, and that the K splits
fit their workspace."""
import random

import pytest

from conftest import load_xe

WS_FLOATS = 8 << 20  # split-K partials


@pytest.fixture(scope="module")
def xe():
    return load_xe()


def test_few_rows_never_take_planes(xe):
    for wd in (xe.XE_I8, xe.XE_I4, xe.XE_BF16, xe.XE_BFP16):
        for m, k in ((16, 16), (3072, 768), (14336, 4096)):
            for b in range(1, 65):
                kernel, ks = xe.linear_path(wd, m, k, b, norm=xe.XE_NORM_LN)
                assert kernel == ("gemv" if b < 4 else "gemm") and ks == 0


def test_planes_within_their_limits(xe):
    rng = random.Random(7)
    seen = set()
    for _ in range(4000):
        wd = rng.choice((xe.XE_I8, xe.XE_I4, xe.XE_BF16, xe.XE_BFP16))
        m = int(2 ** rng.uniform(0, 17))
        k = 16 * int(2 ** rng.uniform(0, 11.5))
        b = rng.randint(65, 512)
        norm = rng.choice((xe.XE_NORM_NONE, xe.XE_NORM_LN, xe.XE_NORM_RMS))
        kernel, ks = xe.linear_path(wd, m, k, b, norm=norm, x_dtype=rng.choice((xe.XE_F32, xe.XE_BF16)))
        seen.add((kernel, ks > 1))
        if kernel.startswith("planes"):
            assert k <= 16384 and m * k * (2 if wd == xe.XE_BF16 else 1) < 2 ** 31
            assert 1 <= ks <= 8 and (ks == 1 or ks * m * b <= WS_FLOATS)
            steps = -(-k // 64)
            assert ks == 1 or -(-steps // ks) >= 4
        else:
            assert kernel == "gemm" and ks == 0
    assert {("planes", False), ("planes", True), ("planes_big", False), ("planes_big", True), ("gemm", False)} <= seen


def test_bad_arguments(xe):
    for args in ((0, 16, 100), (16, 8, 100), (16, 16, 0), (16, 16, 513)):
        with pytest.raises(xe.XdnaError):
            xe.linear_path(xe.XE_I8, args[0], args[1], args[2])
