"""The velocity components' Helmholtz solves side by side (chunked line solves
2 and 3) against one component after the other (variant 1): the channel, whose
components share their transforms (64 FFT points, 90 and 96 matrix-product and
mixed-radix points along x), and two blocks along x."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


def blocks(n, nb):
    out = []
    for q in range(nb):
        B = cases.channel_block((n[0] // nb, n[1], n[2]), friend=q + 1)
        B["lmin"][0], B["lmax"][0] = 6.0 * q / nb, 6.0 * (q + 1) / nb
        if nb > 1:
            for side in range(2):
                for c in range(3):
                    B["bcvel"][c][0][side] = 2.0 - q
                B["bcpre"][0][side] = 2.0 - q
        out.append(B)
    return out


@pytest.mark.parametrize("n,nb", [((64, 24, 16), 1), ((90, 17, 8), 1), ((96, 33, 12), 1), ((64, 24, 16), 2)])
def test_together(tmp_path, n, nb):
    import snac_amd
    d, b = cases.write_case(str(tmp_path), blocks(n, nb), 100.0, bforce=(0.1, 0, 0))
    rng = np.random.default_rng(4)
    init = {(q, f): rng.uniform(-1, 1, (n[0] // nb + 2, n[1] + 2, n[2] + 2)) for q in range(nb) for f in "uvw"}
    out = []
    for v in (1, 2, 3):
        with snac_amd.Context(d, b, 3) as ctx:
            ctx.set_impdiff(True)
            ctx.set_tridiag_variant(v)
            for (q, f), a in init.items():
                ctx.set(q, f, a)
            ctx.init_bounds()
            ctx.steps(1e-3, 3)
            out.append({(q, f): ctx.get(q, f) for q in range(nb) for f in "uvw"})
    for k, a in out[0].items():
        for o in out[1:]:
            # a line solve errs by a few ulp of the unit fields, nine solves and their projections in a row
            assert np.abs(o[k] - a).max() <= 1e-12 * max(1.0, np.abs(a).max()), k
