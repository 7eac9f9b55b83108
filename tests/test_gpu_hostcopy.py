"""Field uploads and downloads in chunks of 131072 doubles: one chunk, a few
chunks with rows across their edges, and enough for several host threads.  A
copy moves bytes, so what comes back is what went up, and the other fields
stay as they were."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "p", "dudtrko", "dvdtrko", "s1", "dsdtrko1")


@pytest.mark.parametrize("n", [(2, 2, 3), (130, 64, 40), (254, 66, 62)])
def test_round_trip(tmp_path, n):
    import snac_amd
    blk = cases.channel_block(n)
    blk["cbcscal"] = [[["F", "F"], ["D", "D"], ["F", "F"]]]
    blk["bcscal"] = [[[1.0, 1.0], [0.0, 1.0], [1.0, 1.0]]]
    d, b = cases.write_case(str(tmp_path), [blk], 500.0, nscal=1,
                            scalar=dict(alphai=[700.0], beta=0.0, ssource=[0.0], is_sforced=[False], scalf=[0.0]))
    rng = np.random.default_rng(3)
    with snac_amd.Context(d, b, 3) as ctx:
        want = {f: np.asfortranarray(rng.uniform(-1, 1, ctx.shape(0, f))) for f in FIELDS}
        for f, a in want.items():
            ctx.set(0, f, a)
        for f, a in want.items():
            assert np.array_equal(ctx.get(0, f), a), f
