"""The CG passes' partial sums on either side of the count beyond which a launch
of its own adds them up (1024 a group): the 3D multigrid of a channel without
an FFT axis, whose one group has 990 and 1080 of them, and its singular mode,
against the direct solver."""
import numpy as np
import pytest

from test_gpu_mg_odd import context, project

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("nz", [132, 144])
def test_partial_sums(tmp_path, nz, prec):
    n = (160, 96, nz)
    with context(tmp_path, "t", n, "fp64", "tensor", 3) as ctx:
        ref, _ = project(ctx)
    with context(tmp_path, "m", n, prec, "mg", 0) as ctx:
        got, (it, relres) = project(ctx)
    assert relres <= 1e-13
    # stops at 1e-13 of the right-hand side; the pressure's condition takes the rest
    assert np.linalg.norm(got - ref) <= 1e-10 * np.linalg.norm(ref), it


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("nz", [8, 9, 1030])
def test_flags(tmp_path, nz, prec):
    """the convergence flags of as many modes as their workgroup adds up itself, of one more, and of two rounds"""
    n = (20, 12, nz)
    with context(tmp_path, "t", n, "fp64", "tensor", 3) as ctx:
        ref, _ = project(ctx)
    with context(tmp_path, "m", n, prec, "mg", 3) as ctx:
        got, (it, relres) = project(ctx)
    assert relres <= 1e-13
    assert np.linalg.norm(got - ref) <= 1e-10 * np.linalg.norm(ref), it
