"""The fused coarse end from precomputed line factors against the unfactored one
(any forced line variant): all levels in the coarse end, or under launched
ones; 2..8 rows per lane on 32 lanes, 4 on 64 (FP64; FP32 lines past 256 rows
have no factors), whole and ragged, an odd axis, the singular mode, several column classes, vectors
in LDS and in memory.  FP32: the same bits (its factors hold the unfactored
kernel's values); FP64: the same solution, the iterations of the unfactored
form."""
import numpy as np
import pytest

import cases
from test_gpu_mg_odd import INNER

pytestmark = pytest.mark.gpu


def solves(tmp_path, blk, prec, lds):
    """pp of one pressure solve and its CG count: factored, unfactored"""
    import snac_amd
    d, b = cases.write_case(str(tmp_path), [blk], 5600.0)
    out = []
    with snac_amd.Context(d, b, 3) as ctx:
        ctx.set_solver("mg")
        ctx.set_precision(prec)
        ctx.set_mg_fast_rcp(False)  # launched levels: the forced kernel and the factored one then divide alike
        ctx.set_mg_tail_lds(lds)
        try:
            # FP32 launched levels run as the kernel their set-up timing chose, which need not be kernel 0
            v32 = ctx.mg_line_choices()[1]
            for v in (-1, v32[0] if prec == "mixed" and v32 else 0):
                ctx.set_mg_line_variant(v)
                rng = np.random.default_rng(3)
                for f in ("u", "v", "w"):
                    ctx.set(0, f, rng.uniform(-1, 1, ctx.shape(0, f)))
                ctx.bounduvw(False)
                ctx.fillps(1e-3)
                ctx.solve_pressure()
                out.append((ctx.get(0, "pp")[INNER], ctx.solver_stats()))
        finally:
            ctx.set_mg_line_variant(-1)
            ctx.set_mg_fast_rcp(True)
            ctx.set_mg_tail_lds(True)
    return out


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("lds", [True, False])
@pytest.mark.parametrize("n", [(32, 64, 4), (16, 5, 4), (20, 33, 6), (32, 160, 4), (32, 250, 4), (28, 256, 4), (12, 24, 4),
                               (11, 24, 4), (31, 96, 4), (64, 128, 4)])
def test_coarse_end(tmp_path, n, lds, prec):
    (a, (it, ra)), (b, (it0, rb)) = solves(tmp_path, cases.channel_block(n), prec, lds)
    assert max(ra, rb) <= 1e-13
    if prec == "mixed":
        np.testing.assert_array_equal(a, b)
    else:
        assert abs(it - it0) <= 1, (it, it0)
        a, b = a - a.mean(), b - b.mean()
        # both stop at 1e-13 of the right-hand side; the pressure's condition takes the rest
        assert np.linalg.norm(a - b) <= 1e-10 * np.linalg.norm(b)
        assert (a != b).any()  # two kernels, not one twice


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_column_classes(tmp_path, prec):
    blk = cases.cavity_block((16, 24, 8), lid=0.0, gr=(1.0, 1.2, 0.0))
    (a, (it, _)), (b, (it0, _)) = solves(tmp_path, blk, prec, True)
    if prec == "mixed":
        np.testing.assert_array_equal(a, b)
    else:
        assert abs(it - it0) <= 1, (it, it0)
        a, b = a - a.mean(), b - b.mean()
        assert np.linalg.norm(a - b) <= 1e-10 * np.linalg.norm(b)
        assert (a != b).any()
