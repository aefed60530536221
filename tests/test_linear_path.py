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


def test_products_slower_over_planes_stay(xe):
    """Measured slower over planes than on the GEMM without (us over planes /
    without: 21.8 / 17.0, 26.5 / 25.0, 48.8 / 45.0, 78 / 61, 66 / 61, 75 / 60,
    25.1 / 21.3, 27.8 / 25.3, 22.5 / 20.8): below 2^28 multiply-adds, of a short
    K, of a weight tile more than the XCDs, spilled stages, scalar partials."""
    ln, no = xe.XE_NORM_LN, xe.XE_NORM_NONE
    for wd, m, k, b, norm in ((xe.XE_BF16, 8243, 48, 200, ln), (xe.XE_BF16, 1536, 1152, 512, ln),
                              (xe.XE_I8, 3961, 5952, 128, no), (xe.XE_BF16, 2560, 5120, 384, no),
                              (xe.XE_I8, 2560, 5120, 384, no), (xe.XE_BF16, 2050, 4096, 384, ln),
                              (xe.XE_BF16, 3072, 768, 300, ln), (xe.XE_I8, 5281, 1152, 192, ln),
                              (xe.XE_BF16, 3799, 256, 450, ln)):
        assert xe.linear_path(wd, m, k, b, norm=norm) == ("gemm", 0), (wd, m, k, b)


def test_products_faster_over_planes_take_them(xe):
    for m, k, b in ((13824, 1152, 512), (4096, 4096, 512), (14336, 4096, 512), (4096, 14336, 512), (3072, 768, 512)):
        assert xe.linear_path(xe.XE_I8, m, k, b)[0].startswith("planes")
    for m, k, b in ((13824, 1152, 512), (4096, 4096, 512), (14336, 4096, 512)):
        assert xe.linear_path(xe.XE_BF16, m, k, b)[0].startswith("planes")


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
            assert 512 <= k <= 16384 and m * k * b >= 2 ** 28 and m * k * (2 if wd == xe.XE_BF16 else 1) < 2 ** 31
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
