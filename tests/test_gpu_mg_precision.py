"""The transforms of the mixed mode on the MG-PCG path, made when the mode is
first asked for: before the plan, after it, and after the Helmholtz plans of
implicit diffusion; 37 modes (a dense product) and 72 (a mixed-radix FFT in
FP64, a dense product in the mixed mode).  Switching back gives FP64's bits."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("impdiff", [False, True])
@pytest.mark.parametrize("nz", [37, 72])
def test_switch(tmp_path, nz, impdiff):
    import snac_amd
    d, b = cases.write_case(str(tmp_path), [cases.channel_block((16, 12, nz))], 500.0)
    rng = np.random.default_rng(6)

    def steps(ctx):
        for f in ("u", "v", "w"):
            ctx.set(0, f, init[f])
        for f in ("p", "dudtrko", "dvdtrko", "dwdtrko"):
            ctx.set(0, f, np.zeros(ctx.shape(0, f)))
        ctx.init_bounds()
        ctx.steps(1e-3, 2)
        return [ctx.get(0, f) for f in ("u", "v", "w", "p")]

    def context(first):
        ctx = snac_amd.Context(d, b, 3)
        if first == "precision":
            ctx.set_precision("mixed")
        ctx.set_solver("mg")
        ctx.set_impdiff(impdiff)
        return ctx

    with context("precision") as ctx:
        init = {f: rng.uniform(-1, 1, ctx.shape(0, f)) for f in ("u", "v", "w")}
        want = steps(ctx)
    with context("plan") as ctx:
        fp64 = steps(ctx)
        ctx.set_precision("mixed")
        got = steps(ctx)
        ctx.set_precision("fp64")
        again = steps(ctx)
    for a, g, f, x in zip(want, got, fp64, again):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, g)
        np.testing.assert_array_equal(f, x)
