"""The multigrid sweeps and the fused coarse end from precomputed line factors
(the default where a level's columns fall into few classes; the FP32 ones in
the place of the kernels the timing chose, with their bits) against the
direct solver and against the unfactored kernels (forced variant 0), over
line lengths at the edges of the lane splits (32 lanes of 2..8 rows, 64 lanes
in FP64 from 193 rows and in both precisions from 257, unfactored past 512
and under 4), odd periodic axes at a launched level (90 -> 45 columns) and in
the coarse end, and a stretched axis whose finest level has too many classes."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

INNER = (slice(1, -1),) * 3


def solve(tmp_path, name, blk, prec, solver, variant=-1, fft_axis=3):
    """pp of one pressure solve of seeded velocities, with its CG count"""
    import snac_amd
    d, b = cases.write_case(str(tmp_path / name), [blk], 5600.0)
    with snac_amd.Context(d, b, fft_axis) as ctx:
        ctx.set_solver(solver)
        ctx.set_precision(prec)
        ctx.set_mg_line_variant(variant)
        try:
            rng = np.random.default_rng(3)
            for f in ("u", "v", "w"):
                ctx.set(0, f, rng.uniform(-1, 1, ctx.shape(0, f)))
            ctx.bounduvw(False)
            ctx.fillps(1e-3)
            ctx.solve_pressure()
            pp = ctx.get(0, "pp")[INNER]
            return pp - pp.mean(), ctx.solver_stats(), ctx.mg_line_choices()
        finally:
            ctx.set_mg_line_variant(-1)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [(90, 5, 4), (70, 3, 4), (34, 33, 4), (40, 64, 4), (40, 66, 4), (44, 97, 4), (34, 192, 4),
                               (36, 194, 4), (34, 256, 4), (36, 300, 4), (34, 512, 4), (34, 520, 4), (11, 24, 4)])
def test_factored_lines(tmp_path, n, prec):
    blk = cases.channel_block(n)
    ref, _, _ = solve(tmp_path, "t", blk, "fp64", "tensor")
    got, (it, relres), choices = solve(tmp_path, "f", blk, prec, "mg")
    old, (it0, _), _ = solve(tmp_path, "v", blk, prec, "mg", variant=0)
    if n[0] > 32 and prec == "fp64":
        assert all((v == 5) == (4 <= n[1] <= 512) for v in choices[0]), choices
    if prec == "mixed" and choices[1] and set(choices[1]) <= {choices[1][0]} and choices[1][0] <= 2:
        # the FP32 factors stand for the kernel chosen, bit for bit
        same, _, _ = solve(tmp_path, "s", blk, prec, "mg", variant=choices[1][0])
        np.testing.assert_array_equal(got, same)
    assert relres <= 1e-13
    # both stop at 1e-13 of the right-hand side; the pressure's condition takes the rest
    assert np.linalg.norm(got - ref) <= 1e-10 * np.linalg.norm(ref)
    assert np.linalg.norm(old - ref) <= 1e-10 * np.linalg.norm(ref)
    # the sweeps precondition as well as the unfactored ones (FP32: they are the unfactored ones, checked above)
    if prec == "fp64":
        assert it <= it0 + 1, (it, it0)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_many_classes(tmp_path, prec):
    blk = cases.cavity_block((40, 24, 8), lid=0.0, gr=(1.0, 1.2, 0.0))
    got, (it, relres), choices = solve(tmp_path, "f", blk, prec, "mg")
    old, (it0, _), _ = solve(tmp_path, "v", blk, prec, "mg", variant=0)
    assert 5 not in choices[0][:1], choices
    assert relres <= 1e-13
    if prec == "fp64":
        assert it <= it0 + 1, (it, it0)
    assert np.linalg.norm(got - old) <= 1e-10 * np.linalg.norm(old)
