"""Cases of several grid blocks run their stencils and matrix transforms over
up to eight blocks per launch: a channel cut into ten blocks along x (two
launches, the second of two blocks) against the same channel as one block.
The transform along z (9 points) is a matrix product, run block by block in
one launch."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


def test_ten_blocks(tmp_path):
    import snac_amd
    nb, n, ny, nz = 10, 4, 12, 9
    one = cases.channel_block((nb * n, ny, nz))
    many = []
    for q in range(nb):
        B = cases.channel_block((n, ny, nz), lengths=(6.0 / nb, 1.0, 3.0), friend=q + 1)
        B["lmin"][0], B["lmax"][0] = 6.0 * q / nb, 6.0 * (q + 1) / nb
        link = ((q - 1) % nb + 1.0, (q + 1) % nb + 1.0)
        for side in range(2):
            for c in range(3):
                B["bcvel"][c][0][side] = link[side]
            B["bcpre"][0][side] = link[side]
        many.append(B)
    rng = np.random.default_rng(5)
    init = {f: rng.uniform(-1, 1, (nb * n, ny, nz)) for f in ("u", "v", "w")}
    out = []
    for name, blocks in (("one", [one]), ("many", many)):
        d, b = cases.write_case(str(tmp_path / name), blocks, 100.0, bforce=(0.1, 0, 0))
        with snac_amd.Context(d, b, 3) as ctx:
            ctx.set_rk_variant(0)
            w = nb * n // ctx.nblocks
            for q in range(ctx.nblocks):
                for f, a in init.items():
                    ctx.set(q, f, np.pad(a[q * w:(q + 1) * w], 1))
            ctx.init_bounds()
            ctx.steps(2e-3, 3)
            out.append({f: np.concatenate([ctx.get(q, f)[1:-1, 1:-1, 1:-1] for q in range(ctx.nblocks)])
                        for f in ("u", "v", "w", "p")})
    for f in out[0]:
        a, b = out[0][f], out[1][f]
        if f == "p":
            a, b = a - a.mean(), b - b.mean()
        # the blocks' spacings are rounded on their own: a few ulp of the metrics
        assert np.linalg.norm(a - b) <= 1e-11 * np.linalg.norm(a), f
