"""The transforms that run as matrix products on the matrix cores (lengths
without a power-of-two FFT, and the kinds that never have one) against the
kinds' definitions (FFTW's, as fft.f90:96-149 uses them) in extended
precision: lengths at the edges of the 16-row tiles and of the mirror (odd,
even, one point), line counts that leave the last workgroup ragged, and
enough lines for two tiles per wavefront."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

KINDS = ("R2HC", "HC2R", "REDFT10", "REDFT01", "RODFT10", "RODFT01", "REDFT11", "RODFT11", "RODFT00")


def matrix(kind, n):
    """M[k, j] with the angles reduced in integers."""
    k, j = np.arange(n, dtype=np.int64)[:, None], np.arange(n, dtype=np.int64)[None, :]
    pi = np.longdouble("3.14159265358979323846264338327950288")
    cos = lambda p, q: np.cos(pi * (p % (2 * q)).astype(np.longdouble) / q)
    sin = lambda p, q: np.sin(pi * (p % (2 * q)).astype(np.longdouble) / q)
    if kind == "R2HC":
        return np.where(k <= n // 2, cos(2 * j * k, n), -sin(2 * j * (n - k), n))
    if kind == "HC2R":
        m = np.where(j <= n // 2, 2 * cos(2 * j * k, n), -2 * sin(2 * (n - j) * k, n))
        return np.where((j == 0) | (2 * j == n), m / 2, m)
    if kind == "REDFT10":
        return 2 * cos((2 * j + 1) * k, 2 * n)
    if kind == "REDFT01":
        return np.where(j == 0, 1, 2) * cos(j * (2 * k + 1), 2 * n)
    if kind == "RODFT10":
        return 2 * sin((2 * j + 1) * (k + 1), 2 * n)
    if kind == "RODFT01":
        return np.where(j == n - 1, 1, 2) * sin((j + 1) * (2 * k + 1), 2 * n)
    if kind == "REDFT11":
        return 2 * cos((2 * j + 1) * (2 * k + 1), 4 * n)
    if kind == "RODFT11":
        return 2 * sin((2 * j + 1) * (2 * k + 1), 4 * n)
    return 2 * sin((j + 1) * (k + 1), n + 1)


def check(ctx, kind, n, howmany, tile=0):
    M = matrix(kind, n)
    x = np.random.default_rng(n + howmany).uniform(-1, 1, (howmany, n))
    x[howmany // 2] = 0.0
    ref = (x.astype(np.longdouble) @ M.T) if howmany < 1000 else x @ M.astype(np.float64).T
    # a sum of n products in any order, and coefficients whose reduced angle
    # (below 2 pi) carries a few roundings; the float64 reference of the long
    # run errs as much again
    u = 2.0 ** -53
    tol = (n + 4) * u * (np.abs(x) @ np.abs(M).astype(np.float64).T) + 16 * u * np.abs(x).sum(1)[:, None]
    tol *= 1 if howmany < 1000 else 2
    for strided in (False, True):
        y = ctx.r2r_lines(kind, x, strided=strided, tile=tile)
        assert (np.abs(y - ref) <= tol).all(), (kind, n, strided, float(np.abs(y - ref).max()))
        assert not y[howmany // 2].any()


@pytest.fixture(scope="module")
def ctx(tmp_path_factory):
    import snac_amd
    d, b = cases.write_case(str(tmp_path_factory.mktemp("r2r")), [cases.channel_block((4, 4, 4))], 5600.0)
    with snac_amd.Context(d, b, 3) as c:
        yield c


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [1, 3, 5, 15, 17, 30, 31, 33, 63, 90, 97, 192, 255, 333, 600, 1100])
def test_matrix_lines(ctx, kind, n):
    check(ctx, kind, n, 37)


@pytest.mark.parametrize("kind", ["R2HC", "HC2R"])
@pytest.mark.parametrize("n", [48, 72, 80, 96, 120, 144, 160, 192, 240, 288, 320, 384, 480])
def test_mixed_radix_lines(ctx, kind, n):
    """The lengths with factors 3 and 5 that have an FFT, both tiles."""
    for tile in (0, 1):
        check(ctx, kind, n, 75, tile)


@pytest.mark.parametrize("kind", ["R2HC", "HC2R", "REDFT11"])
@pytest.mark.parametrize("n", [42, 2])
def test_many_lines(ctx, kind, n):
    check(ctx, kind, n, 16384 * 4 + 21)
