"""Odd periodic axes on the multigrid levels: the lines at the two ends are
neighbours and have one colour.  Each is relaxed from the other's value before
the sweep, so a solve gives the same bits every time, whichever line kernel
runs, and needs about the iterations of the even axis beside it: launched
levels and the coarse end, lines with and without factors (3 and 520 rows have
none), both precisions, the 3D hierarchy with one and with both periodic axes
odd, and the Helmholtz solves that stop at the finest level."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

INNER = (slice(1, -1),) * 3


def project(ctx):
    """pp and the CG count of one pressure solve of seeded velocities"""
    rng = np.random.default_rng(3)
    for f in ("u", "v", "w"):
        ctx.set(0, f, rng.uniform(-1, 1, ctx.shape(0, f)))
    ctx.bounduvw(False)
    ctx.fillps(1e-3)
    ctx.solve_pressure()
    pp = ctx.get(0, "pp")[INNER]
    return pp - pp.mean(), ctx.solver_stats()


def context(tmp_path, name, n, prec, solver, fft_axis):
    import snac_amd
    d, b = cases.write_case(str(tmp_path / name), [cases.channel_block(n)], 5600.0)
    ctx = snac_amd.Context(d, b, fft_axis)
    ctx.set_solver(solver)
    ctx.set_precision(prec)
    return ctx


def check(tmp_path, n, even, prec, fft_axis, variants):
    with context(tmp_path, "t", n, "fp64", "tensor", 3) as ctx:
        ref, _ = project(ctx)
    its = {}
    for name, size in (("even", even), ("odd", n)):
        with context(tmp_path, name, size, prec, "mg", fft_axis) as ctx:
            try:
                for v in variants:
                    print(f"{name} {size} {prec} variant {v}", flush=True)
                    ctx.set_mg_line_variant(v)
                    a, (it, relres) = project(ctx)
                    its[name, v] = it
                    assert relres <= 1e-13
                    if name == "odd":
                        b, _ = project(ctx)
                        np.testing.assert_array_equal(a, b)
                        # stops at 1e-13 of the right-hand side; the pressure's condition takes the rest
                        assert np.linalg.norm(a - ref) <= 1e-10 * np.linalg.norm(ref)
            finally:
                ctx.set_mg_line_variant(-1)
    print(its, flush=True)
    for v in variants:
        assert its["odd", v] <= its["even", v] + 5, its


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [(33, 24, 4), (90, 5, 4), (37, 3, 4), (69, 72, 4), (45, 520, 4), (11, 24, 4),
                               (35, 256, 4)])
def test_modes(tmp_path, n, prec):
    even = {90: 88}.get(n[0], n[0] - 1)
    check(tmp_path, n, (even,) + n[1:], prec, 3, (-1, 0, 1, 2, 3, 4))


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [(33, 12, 17), (32, 12, 17), (33, 12, 16)])
def test_coupled(tmp_path, n, prec):
    check(tmp_path, n, (32, 12, 16), prec, 0, (-1, 0, 1))


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_helmholtz(tmp_path, prec):
    out = []
    for name in ("a", "b"):
        with context(tmp_path, name, (33, 24, 8), prec, "mg", 3) as ctx:
            ctx.set_impdiff(True)
            rng = np.random.default_rng(4)
            for f in ("u", "v", "w"):
                ctx.set(0, f, rng.uniform(-1, 1, ctx.shape(0, f)))
            ctx.init_bounds()
            ctx.steps(1e-3, 2)
            out.append([ctx.get(0, f) for f in ("u", "v", "w")])
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, b)
