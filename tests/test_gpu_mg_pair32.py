"""Both colours of an FP32 multigrid level in one launch, over several line pairs
per lane segment (3 or 4 a segment on the finest level, the last segment full,
of one pair or short), lines in whole and ragged chunks, against the unfactored
kernels bit for bit: the levels' kernel is forced while the plan is set up, 2
for the factors with refined reciprocals and 0 for those with IEEE quotients,
so that neither side depends on a timing."""
import numpy as np
import pytest

import cases
from test_gpu_mg_odd import project

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [0, 2])
@pytest.mark.parametrize("n", [(256, 64, 64), (258, 33, 64), (260, 100, 64), (264, 256, 64), (262, 250, 48)])
def test_same_bits(tmp_path, n, variant):
    import snac_amd
    d, b = cases.write_case(str(tmp_path), [cases.channel_block(n)], 5600.0)
    with snac_amd.Context(d, b, 3) as ctx:
        ctx.set_mg_line_variant(variant)
        try:
            ctx.set_solver("mg")
            ctx.set_precision("mixed")
            choices = ctx.mg_line_choices()
            assert choices[1] and all(v == variant for v in choices[1]), choices
            assert all(v == 5 for v in choices[0]), choices
            ctx.set_timing(True)
            out, launches = [], []
            for v in (-1, variant):
                ctx.set_mg_line_variant(v)
                ctx.get_timing()
                pp, (it, relres) = project(ctx)
                assert relres <= 1e-13
                out.append(pp)
                launches.append(ctx.get_timing()["mg_line0"][1] / it)
        finally:
            ctx.set_mg_line_variant(-1)
    # one descent a V-cycle, or three sweeps that read their neighbours
    assert launches == [1, 3]
    np.testing.assert_array_equal(out[0], out[1])


def test_forced_choice_is_not_kept(tmp_path):
    """a later plan of the same shape does not take over a forced choice"""
    import snac_amd
    d, b = cases.write_case(str(tmp_path), [cases.channel_block((82, 3, 4))], 5600.0)
    seen = []
    for v in (1, 0, -1):
        with snac_amd.Context(d, b, 3) as ctx:
            ctx.set_mg_line_variant(v)
            try:
                ctx.set_solver("mg")
                seen.append(ctx.mg_line_choices())
            finally:
                ctx.set_mg_line_variant(-1)
    for choices, v in zip(seen, (1, 0)):
        for prec in (0, 1):  # three rows have no factors in either precision
            assert choices[prec] and all(c == v for c in choices[prec]), seen
    assert seen[2][0] and all(0 <= c <= 4 for c in seen[2][0]), seen
