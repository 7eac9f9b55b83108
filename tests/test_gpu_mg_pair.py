"""Both colours of a periodic multigrid level in one launch, over several line
pairs per lane segment: a last segment that is full, short or of one pair,
lines of 2..6 rows on 32 lanes and 4 on 64 in whole and ragged chunks, against the direct
solver and the unfactored kernels.  (One pair per segment and the edges of
the lane splits: the factored lines' test.)"""
import numpy as np
import pytest

import cases
from test_gpu_mg_factored import solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(512, 64, 32), (500, 12, 64), (258, 33, 128), (480, 130, 36), (136, 192, 128), (66, 20, 256),
                               (260, 256, 64), (264, 200, 36)])
def test_line_pairs(tmp_path, n):
    blk = cases.channel_block(n)
    ref, _, _ = solve(tmp_path, "t", blk, "fp64", "tensor")
    got, (it, relres), choices = solve(tmp_path, "f", blk, "fp64", "mg")
    old, (it0, _), _ = solve(tmp_path, "v", blk, "fp64", "mg", variant=0)
    assert choices[0] and all(v == 5 for v in choices[0]), choices
    assert relres <= 1e-13
    # all stop at 1e-13 of the right-hand side; the pressure's condition takes the rest
    assert np.linalg.norm(got - ref) <= 1e-10 * np.linalg.norm(ref)
    assert np.linalg.norm(old - ref) <= 1e-10 * np.linalg.norm(ref)
    assert it <= it0 + 1, (it, it0)
