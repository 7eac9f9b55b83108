"""The work that users of this library have it do, as measurable cases.

A case is one simulation: a context made from dns.nml / blocks.nml, initial
fields uploaded, and then passes of `steps` RK3 time steps after which the
program takes the fields back to the host (a snapshot, a checkpoint, its own
statistics).  Fields cross the library's boundary only at upload and download,
so the download is part of a pass, as it is part of any such program; the
state goes on from pass to pass.

Geometries:
  cavity4  the lid-driven cavity of the reference's known-answer test: four
           blocks that tile a thin box, x periodic, walls and a lid around
  dhc      the differentially heated cavity: a scalar with fixed wall values
           driving the flow by buoyancy
  channel  the periodic channel (x, z periodic, y stretched between walls)
  cavity   the closed lid-driven box: cosine transforms, no periodic axis
  box      the triply periodic box
  bfs      the backward-facing step of three blocks (a Poiseuille inflow, an
           outflow): a union that is no box, so only MG-PCG solves it
Solvers: "auto" (direct on a box, MG-PCG elsewhere) or "mg"; precision "fp64"
or "mixed"; impdiff: implicit diffusion.
"""
import math
import os
import tempfile

import numpy as np
import torch

import snac_amd

# &hypre hypre_tol of the MG-PCG cases: the benchmark's default, and for the mixed form the tests' value -- its FP32
# right-hand sides turn whatever the solver leaves in the velocities into rounding flips of the next substage
TOL = {"fp64": 1e-10, "mixed": 1e-13}


def _case(name, geom, nx, ny, nz, steps, solver="auto", precision="fp64", impdiff=False):
    c = {"geom": geom, "nx": nx, "ny": ny, "nz": nz, "steps": steps, "solver": solver, "precision": precision,
         "impdiff": impdiff}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest programs in use: the two validation cases, where a step is a chain of tiny launches
        _case("cavity4_2x64x64", "cavity4", 2, 64, 64, 40),
        _case("dhc_32x2x32", "dhc", 32, 2, 32, 40),
        # a first test run on a coarse channel
        _case("channel_64x48x32", "channel", 64, 48, 32, 40),
        # a size taken from a resolution estimate, not from a power of two
        _case("channel_180x77x90", "channel", 180, 77, 90, 20),
        # a closed cavity: cosine transforms on both uniform axes
        _case("cavity_128x64x64", "cavity", 128, 64, 64, 40),
        # decaying turbulence in a periodic box, at multiples of 32 that are no powers of two
        _case("box_192x96x96", "box", 192, 96, 96, 10),
        # production channels on the direct solver, implicit and explicit diffusion; the second is the largest case
        _case("channel_256x64x64_impdiff", "channel", 256, 64, 64, 10, impdiff=True),
        _case("channel_512x128x128", "channel", 512, 128, 128, 40),
        # the batched MG-PCG solver: FP64, and the mixed form on the benchmark's lines of 256 rows
        _case("channel_512x128x64_mg", "channel", 512, 128, 64, 10, solver="mg"),
        _case("channel_256x256x64_mg_mixed", "channel", 256, 256, 64, 10, solver="mg", precision="mixed"),
        # the multi-block case that only MG-PCG solves
        _case("bfs_512x80x48", "bfs", 512, 80, 48, 10, solver="mg"),
    ]


def draw(rng):
    def size(lo, hi):
        # multiples of a small power of two half of the time, any integer otherwise
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        m = rng.choice([1, 1, 2, 8, 16])
        return max(lo, n // m * m)

    kind = rng.choice(["channel", "channel", "channel_mg", "channel_mg", "channel_impdiff", "cavity", "box", "dhc",
                       "cavity4", "bfs"])
    if kind == "channel":
        return _case(None, "channel", size(32, 400), size(24, 100), size(24, 100), 10)
    if kind == "channel_mg":
        return _case(None, "channel", size(32, 320), size(24, 256), size(16, 48), 6, solver="mg",
                     precision=rng.choice(["fp64", "mixed"]))
    if kind == "channel_impdiff":
        return _case(None, "channel", size(32, 400), size(24, 100), size(24, 80), 6, impdiff=True)
    if kind == "cavity":
        return _case(None, "cavity", size(24, 200), size(24, 90), size(24, 90), 10)
    if kind == "box":
        return _case(None, "box", size(32, 256), size(24, 90), size(24, 90), 10)
    if kind == "dhc":
        return _case(None, "dhc", size(24, 300), rng.choice([2, 4, 8]), size(24, 200), 30)
    if kind == "cavity4":
        return _case(None, "cavity4", 2, 2 * size(16, 48), 2 * size(16, 48), 30)
    # the step: nx and ny are split 3:5 and 2:3 between its blocks
    return _case(None, "bfs", 8 * size(12, 64), 5 * size(12, 28), size(16, 48), 4, solver="mg",
                 precision=rng.choice(["fp64", "mixed"]))


# ---- the namelists ----
RE = {"channel": 5600.0, "cavity": 1000.0, "cavity4": 1000.0, "box": 1600.0, "bfs": 1000.0, "dhc": 1186.78165819}
ALPHAI = 842.614977318  # the heated cavity's 1/diffusivity
BFORCE = 12.0 / 5600.0  # the channel's laminar driving force


def _blocks(c):
    """Blocks as dicts: n, lo, hi, gr, velocity walls (BC character or friend number per face), pressure, values."""
    nx, ny, nz, g = c["nx"], c["ny"], c["nz"], c["geom"]

    def block(n, lo, hi, faces, gr=(0.0, 0.0, 0.0), values=None, inflow=False):
        return {"n": n, "lo": lo, "hi": hi, "faces": faces, "gr": gr, "values": values or {}, "inflow": inflow}

    if g == "channel":
        return [block((nx, ny, nz), (0, 0, 0), (6.0, 1.0, 3.0), [1, 1, "D", "D", 1, 1], gr=(0.0, 1.8, 0.0))]
    if g == "box":
        return [block((nx, ny, nz), (0, 0, 0), (2 * math.pi,) * 3, [1] * 6)]
    if g == "cavity":
        return [block((nx, ny, nz), (0, 0, 0), (1.0, 1.0, 1.0), ["D"] * 6, values={(0, 2, 1): 1.0})]
    if g == "dhc":
        return [block((nx, ny, nz), (0, 0, 0), (1.0, 0.03125 * ny, 1.0), ["D", "D", 1, 1, "D", "D"])]
    if g == "cavity4":
        hy, hz, lx = ny // 2, nz // 2, 0.15625 * nx
        lid = {(1, 2, 1): 1.0}  # v = 1 on the lid z+
        return [block((nx, hy, hz), (0, 0, 0), (lx, .5, .5), [1, 1, "D", 2, "D", 3]),
                block((nx, hy, hz), (0, .5, 0), (lx, 1., .5), [2, 2, 1, "D", "D", 4]),
                block((nx, hy, hz), (0, 0, .5), (lx, .5, 1.), [3, 3, "D", 4, 1, "D"], values=lid),
                block((nx, hy, hz), (0, .5, .5), (lx, 1., 1.), [4, 4, 3, "D", 2, "D"], values=lid)]
    n1, h1 = 3 * nx // 8, 2 * ny // 5
    gr = (0.0, 1.2, 0.0)
    return [block((n1, h1, nz), (0, 0, 0), (3.0, 1.0, 2.0), ["I", 2, "D", "D", 1, 1], gr, {(0, 0, 0): 1.0}, True),
            block((nx - n1, h1, nz), (3.0, 0, 0), (8.0, 1.0, 2.0), [1, "O", "D", 3, 2, 2], gr),
            block((nx - n1, ny - h1, nz), (3.0, 1.0, 0), (8.0, 2.5, 2.0), ["D", "O", 2, "D", 3, 3], gr)]


FFT_AXIS = {"cavity4": 1, "dhc": 2}


def _write(c, path):
    vel = {"D": "D", "I": "D", "O": "N"}
    pre = {"D": "N", "I": "N", "O": "D"}
    blocks = _blocks(c)
    out = ["&blocks\nnblocks = %d\n" % len(blocks)]
    for b, B in enumerate(blocks, start=1):
        def put(key, v, dims="1:3,%d" % b):
            out.append("block_%s(%s) = %s\n" % (key, dims, ", ".join("'%s'" % x if isinstance(x, str) else repr(x)
                                                                     for x in v)))
        put("dims", (1, 1, 1))
        put("ng", B["n"])
        put("lmin", [float(x) for x in B["lo"]])
        put("lmax", [float(x) for x in B["hi"]])
        put("gt", (0, 0, 0))
        put("gr", B["gr"])
        link = [0.0 if isinstance(f, str) else float(f) for f in B["faces"]]
        for q in range(3):
            put("cbcvel", ["F" if not isinstance(f, str) else vel[f] for f in B["faces"]], "0:1,1:3,%d,%d" % (q + 1, b))
            put("bcvel", [B["values"].get((q, f // 2, f % 2), link[f]) for f in range(6)],
                "0:1,1:3,%d,%d" % (q + 1, b))
        put("cbcpre", ["F" if not isinstance(f, str) else pre[f] for f in B["faces"]], "0:1,1:3,%d" % b)
        put("bcpre", link, "0:1,1:3,%d" % b)
        if c["geom"] == "dhc":
            put("cbcscal", ["D", "D", "F", "F", "N", "N"], "0:1,1:3,1,%d" % b)
            put("bcscal", [-0.5, 0.5, 1.0, 1.0, 0.0, 0.0], "0:1,1:3,1,%d" % b)
        put("inflow_type", [1 if B["inflow"] and f == 0 else 0 for f in range(6)], "0:1,1:3,%d" % b)
        out.append("block_inivel(%d) = 'zer'\n" % b)
    out.append("/\n")
    with open(os.path.join(path, "blocks.nml"), "w") as f:
        f.write("".join(out))
    heat = c["geom"] == "dhc"
    with open(os.path.join(path, "dns.nml"), "w") as f:
        f.write("&dns\ncfl = 0.5, dtmax = 1.0e5, dt_f = -1.\nvisci = %r\nnstep = 1, time_max = 100., tw_max = 0.1\n"
                "stop_type(1:3) = T, F, F\nrestart = F, is_overwrite_save = T, nsaves_max = 0\n"
                "icheck = 10, iout0d = 0, iout1d = 0, iout2d = 0, iout3d = 0, isave = 0\n"
                "bforce(1:3) = %r, 0., 0.\ngacc(1:3) = 0., 0., %r\nnscal = %d\n/\n"
                "&hypre\nhypre_solver_i = 2, hypre_tol = %r, hypre_maxiter = 1000\n/\n"
                % (RE[c["geom"]], BFORCE if c["geom"] == "channel" else 0.0, -1.0 if heat else 0.0, int(heat), TOL[c["precision"]]))
        if heat:
            f.write("&scalar\niniscal(:) = 'zer'\nalphai(:) = %r\nbeta = 1.\nssource(:) = 0.\nis_sforced(:) = F\n"
                    "scalf(:) = 0.\n/\n" % ALPHAI)
    return os.path.join(path, "dns.nml"), os.path.join(path, "blocks.nml")


# ---- inputs ----
def _faces(n, lo, hi, gr):
    """Face positions of one axis: uniform, or clustered at both ends by a hyperbolic tangent."""
    r = np.arange(n + 1) / n
    if gr:
        r = 0.5 * (1.0 + np.tanh((r - 0.5) * gr) / np.tanh(gr / 2))
    return lo + r * (hi - lo)


def _dt(c):
    """A time step well inside the explicit scheme's limits, from the grid alone."""
    conv = diff = 0.0
    for a, speed in enumerate((1.6, 0.3, 0.3) if c["geom"] in ("channel", "bfs") else (1.2, 1.2, 1.2)):
        h = min(float(np.diff(_faces(B["n"][a], B["lo"][a], B["hi"][a], B["gr"][a])).min()) for B in _blocks(c))
        conv += speed / h
        diff += 1.0 / h ** 2
    dt = 0.4 / conv
    return dt if c["impdiff"] else min(dt, 0.3 * RE[c["geom"]] / diff)


def _fields(c, seed):
    """Interiors of u (and of the heated cavity's scalar) of each block, as (z, y, x) tensors: the geometry's base flow
    and seeded noise.  v and w start from rest; the first projection gives them their share of the noise."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    out = []
    for B in _blocks(c):
        nx, ny, nz = B["n"]
        u = 0.2 * torch.rand((nz, ny, nx), generator=gen, dtype=torch.float64, device=dev) - 0.1
        f = [_faces(B["n"][a], B["lo"][a], B["hi"][a], B["gr"][a]) for a in range(3)]
        x, y, z = (torch.tensor(0.5 * (v[1:] + v[:-1]), device=dev) for v in f)
        if c["geom"] == "channel" or (c["geom"] == "bfs" and float(y.max()) <= 1.0):
            u += (6.0 * y * (1.0 - y))[None, :, None]
        elif c["geom"] == "box":  # vortices: the projection adds the other components
            u += torch.sin(x)[None, None, :] * torch.cos(y)[None, :, None] * torch.cos(z)[:, None, None]
        out.append({"u": u})
        if c["geom"] == "dhc":
            out[-1]["s1"] = 0.1 * u + (x - 0.5)[None, None, :]
    return out


NAMES = ("u", "v", "w")


def _outputs(c):
    """The fields a program takes back: all of the state; with the mixed form the velocities that its statistics are
    made of (its pressure is only as good as the FP32 right-hand sides)."""
    return NAMES + (("p",) if c["precision"] == "fp64" else ()) + (("s1",) if c["geom"] == "dhc" else ())


def prepare(case, seed):
    with tempfile.TemporaryDirectory() as tmp:
        dns, blocks = _write(case, tmp)
        ctx = snac_amd.Context(dns, blocks, FFT_AXIS.get(case["geom"], 3), device=0)
    ctx.set_solver(case["solver"])
    ctx.set_precision(case["precision"])
    if case["impdiff"]:
        ctx.set_impdiff(True)
    if case["geom"] == "dhc":
        ctx.set_buoyancy(True)
    for b, fields in enumerate(_fields(case, seed)):
        for name, a in fields.items():
            ctx.set(b, name, torch.nn.functional.pad(a, (1, 1, 1, 1, 1, 1)).cpu().numpy().T)  # x fastest, ghosts zero
    ctx.init_bounds()
    return {"ctx": ctx, "dt": _dt(case), "steps": case["steps"], "names": _outputs(case)}


def run(state):
    ctx = state["ctx"]
    ctx.steps(state["dt"], state["steps"])
    return {"%s%d" % (name, b): ctx.get(b, name) for b in range(ctx.nblocks) for name in state["names"]}


def work(case):
    """Per cell and RK3 substage: the fields u, v, w, p and the three old tendencies (with a scalar two arrays more)
    read and written, and the pressure solve's right-hand side written, transformed there and back along the two other
    axes and solved along the line (16 bytes a pass); with implicit diffusion such a solve per component.  The fields'
    download at the end.  The arithmetic: some 200 operations in the stencils, 5 log2 n a transform."""
    cells = float(sum(np.prod(B["n"]) for B in _blocks(case)))
    solves = 4 if case["impdiff"] else 1
    fields = 9 if case["geom"] == "dhc" else 7
    logs = sum(math.log2(max(2, case[k])) for k in ("nx", "ny", "nz"))
    return {"bytes": cells * (case["steps"] * 3 * (16.0 * fields + solves * 88.0) + 16.0 * 4),
            "flops": cells * case["steps"] * 3 * (200.0 + solves * 10.0 * logs)}


# ---- the same discrete equations in plain torch, 64 bits ----
class _Box:
    """RK3 steps of one box (blocks that tile it included): second-order staggered differences, the pressure and
    Helmholtz problems solved by diagonalising each axis's one-dimensional operator."""

    RK = ((32.0 / 60.0, 0.0), (25.0 / 60.0, -17.0 / 60.0), (45.0 / 60.0, -25.0 / 60.0))

    def __init__(self, case):
        self.c = case
        B = _blocks(case)
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        four = case["geom"] == "cavity4"
        self.n = (case["nx"], case["ny"], case["nz"])
        last = B[-1] if four else B[0]
        self.per = [not isinstance(B[0]["faces"][2 * a], str) for a in range(3)]
        self.val = last["values"]
        self.visc = 1.0 / RE[case["geom"]]
        self.df, self.dc, self.h = [], [], []
        for a in range(3):
            d = np.diff(_faces(self.n[a], B[0]["lo"][a], last["hi"][a], B[0]["gr"][a]))
            df = np.concatenate([d[-1:], d, d[:1]] if self.per[a] else [d[:1], d, d[-1:]])
            dc = np.append(0.5 * (df[1:] + df[:-1]), 0.0)
            dc[-1] = dc[-2]
            self.h.append((df, dc))
            shape = [1, 1, 1]
            shape[a] = -1
            self.df.append(torch.tensor(df, device=self.dev).reshape(shape))
            self.dc.append(torch.tensor(dc, device=self.dev).reshape(shape))
        self.eig = {}

    # a field's interior shifted by one cell along some axes: {axis: -1 or 1}
    @staticmethod
    def at(f, **sh):
        return f[tuple(slice(1 + sh.get(k, 0), f.shape[a] - 1 + sh.get(k, 0)) for a, k in enumerate("xyz"))]

    def m(self, v, a, s=0):
        t = v[a]
        return t.narrow(a, 1 + s, t.shape[a] - 2)

    def axis(self, a, comp):
        """Eigenvectors and eigenvalues of axis a's second difference for a velocity component (own axis: faces), the
        pressure (-1) or the scalar (3), symmetrised by the cells' widths."""
        kind = "periodic" if self.per[a] else "face" if a == comp else "N" if comp < 0 else "D"
        key = (a, kind)
        if key not in self.eig:
            df, dc, n = self.h[a][0], self.h[a][1], self.n[a]
            face = a == comp
            w = dc[1:n + 1] if face else df[1:n + 1]
            lo = df[1:n + 1] if face else dc[0:n]
            hi = df[2:n + 2] if face else dc[1:n + 1]
            A = np.zeros((n, n))
            for i in range(n):
                A[i, i] -= 1 / lo[i] + 1 / hi[i]
                if i > 0 or kind == "periodic":
                    A[i, i - 1] += 1 / lo[i]
                if i < n - 1 or kind == "periodic":
                    A[i, (i + 1) % n] += 1 / hi[i]
            if kind == "N":
                A[0, 0] += 1 / lo[0]
                A[-1, -1] += 1 / hi[-1]
            if kind == "D":
                A[0, 0] -= 1 / lo[0]
                A[-1, -1] -= 1 / hi[-1]
            if kind == "face":  # the wall's face is no unknown
                A, w = A[:-1, :-1], w[:-1]
            s = 1 / np.sqrt(w)
            lam, V = np.linalg.eigh(s[:, None] * A * s[None, :])
            f = torch.tensor(V.T / s[None, :], device=self.dev)  # weighted: V^T sqrt(w)
            b = torch.tensor(s[:, None] * V, device=self.dev)
            self.eig[key] = (torch.tensor(lam, device=self.dev), f, b)
        return self.eig[key]

    def solve(self, rhs, comp, shift):
        """(Laplacian + shift) x = rhs; a singular pressure's constant is left for the caller."""
        lam = 0.0
        for a in range(3):
            l, f, _ = self.axis(a, comp)
            rhs = torch.movedim(torch.tensordot(f, rhs, dims=([1], [a])), 0, a)
            shape = [1, 1, 1]
            shape[a] = -1
            lam = lam + l.reshape(shape)
        lam = lam + shift
        if comp < 0:
            zero = lam.abs() < 1e-9 * lam.abs().max() / max(self.n) ** 2
            rhs = torch.where(zero, torch.zeros_like(rhs), rhs / torch.where(zero, torch.ones_like(lam), lam))
        else:
            rhs = rhs / lam
        for a in range(3):
            rhs = torch.movedim(torch.tensordot(self.axis(a, comp)[2], rhs, dims=([1], [a])), 0, a)
        return rhs

    def fill(self, f, comp, correc=False):
        """Ghost layers: wraps, then the walls in the order x, y, z."""
        for a in range(3):
            if self.per[a]:
                n = self.n[a]
                f.narrow(a, 0, 1).copy_(f.narrow(a, n, 1))
                f.narrow(a, n + 1, 1).copy_(f.narrow(a, 1, 1))
        for a in range(3):
            if self.per[a]:
                continue
            n = self.n[a]
            for side in range(2):
                g, i = (0, 1) if side == 0 else (n + 1, n)
                if comp < 0 or (comp == 3 and a == 2):
                    f.narrow(a, g, 1).copy_(f.narrow(a, i, 1))
                    continue
                v = (-0.5, 0.5)[side] if comp == 3 else self.val.get((comp, a, side), 0.0)
                if a != comp:
                    f.narrow(a, g, 1).copy_(2 * v - f.narrow(a, i, 1))
                elif not correc:
                    if side == 0:
                        f.narrow(a, 0, 1).fill_(v)
                    else:
                        f.narrow(a, n, 1).fill_(v)
                        f.narrow(a, n + 1, 1).copy_(f.narrow(a, n - 1, 1))

    def face(self, f, a):
        """f averaged onto the faces between each cell and the next along a."""
        n = f.shape[a]
        return 0.5 * (f.narrow(a, 0, n - 1) + f.narrow(a, 1, n - 1))

    def laplacian(self, f, comp):
        out = 0.0
        for a, k in enumerate("xyz"):
            g, w = (self.df, self.dc) if a == comp else (self.dc, self.df)
            up, lo = (self.m(g, a, 1), self.m(g, a)) if a == comp else (self.m(g, a), self.m(g, a, -1))
            c = self.at(f)
            out = out + ((self.at(f, **{k: 1}) - c) / up - (c - self.at(f, **{k: -1})) / lo) / self.m(w, a)
        return out

    def advection(self, vel, c):
        """Momentum flux differences of component c: fluxes through a face are cell-area averages of the carrying
        velocity times the plain average of the carried one."""
        q, out = vel[c], 0.0
        kc = "xyz"[c]
        for a, k in enumerate("xyz"):
            if a == c:
                r = self.at(q)
                fp, fm = self.at(q, **{k: 1}), self.at(q, **{k: -1})
                # (the carrying sum times the carried neighbour, as the scheme has it)
                d = 0.25 * ((r + fp) * fp - (r + fm) * fm)
            else:
                w0, w1 = self.m(self.df, c), self.m(self.df, c, 1)
                f = vel[a]
                hi = self.at(f) * w0 + self.at(f, **{kc: 1}) * w1
                lo = self.at(f, **{k: -1}) * w0 + self.at(f, **{k: -1, kc: 1}) * w1
                d = 0.25 * (hi * self.at(q, **{k: 1}) - lo * self.at(q, **{k: -1})) / w0
            out = out - d / (self.m(self.dc, a) if a == c else self.m(self.df, a)) * (
                self.m(self.df, c) / self.m(self.dc, c) if a != c else 1.0)
        return out

    def grad(self, p, a):
        return (self.at(p, **{"xyz"[a]: 1}) - self.at(p)) / self.m(self.dc, a)

    def steps(self, vel, p, s, dt, steps):
        imp, heat = self.c["impdiff"], s is not None
        inner = (slice(1, -1),) * 3
        old, sold = [0.0] * 3, 0.0
        for step in range(3 * steps):
            f1, f2 = (x * dt for x in self.RK[step % 3])
            f12 = f1 + f2
            if heat:
                al = 1.0 / ALPHAI
                d = 0.0
                for a, k in enumerate("xyz"):
                    c, up, lo = self.at(s), self.at(s, **{k: 1}), self.at(s, **{k: -1})
                    q = vel[a]
                    d = d + (al * ((up - c) / self.m(self.dc, a) - (c - lo) / self.m(self.dc, a, -1))
                             - 0.5 * (up + c) * self.at(q) + 0.5 * (lo + c) * self.at(q, **{k: -1})) / self.m(self.df, a)
                s = s.clone()
                s[inner] += f1 * d + f2 * sold
                sold = d
                self.fill(s, 3)
            new, rhs = [], []
            for c in range(3):
                adv, lap = self.advection(vel, c), self.visc * self.laplacian(vel[c], c)
                r = adv if imp else adv + lap
                f = -self.grad(p, c)
                if c == 0 and self.c["geom"] == "channel":
                    f = f + BFORCE
                if c == 2 and heat:
                    f = f + 0.5 * (self.at(s, z=1) + self.at(s))
                q = vel[c].clone()
                q[inner] += f1 * r + f2 * old[c] + f12 * f
                if imp:
                    q[inner] += 0.5 * f12 * lap
                new.append(q)
                rhs.append(r)
            vel, old = new, rhs
            al = -0.5 * self.visc * f12
            if imp:
                for c in range(3):
                    inn = tuple(slice(1, self.n[a] + (0 if a == c and not self.per[a] else 1)) for a in range(3))
                    vel[c][inn] = self.solve(vel[c][inn] / al, c, 1.0 / al)
            for c in range(3):
                self.fill(vel[c], c)
            div = 0.0
            for a, k in enumerate("xyz"):
                div = div + (self.at(vel[a]) - self.at(vel[a], **{k: -1})) / self.m(self.df, a)
            x = self.solve(div / f12, -1, 0.0)
            # the constant: zero mean for MG-PCG and the periodic box, else the last line cell's value
            line = 2 if self.c["geom"] == "cavity4" or self.c["geom"] == "dhc" else 1
            if self.c["solver"] == "mg" or all(self.per):
                x = x - x.mean()
            else:
                x = x - x.narrow(line, self.n[line] - 1, 1).mean()
            pp = torch.zeros_like(p)
            pp[inner] = x
            self.fill(pp, -1)
            for a in range(3):
                q = vel[a]
                g = (pp.narrow(a, 1, self.n[a] + 1) - pp.narrow(a, 0, self.n[a] + 1)) / self.dc[a].narrow(
                    a, 0, self.n[a] + 1)
                q.narrow(a, 0, self.n[a] + 1).sub_(f12 * g)
                self.fill(q, a, correc=True)
            p = p.clone()
            p[inner] += x
            if imp:
                p[inner] += al * self.laplacian(pp, -1)
            self.fill(p, -1)
        return vel, p, s


def exact(case, seed):
    if case["geom"] == "bfs":  # no box: a sparse solve per mode and substage takes minutes
        return None
    parts = [{k: a.permute(2, 1, 0) for k, a in f.items()} for f in _fields(case, seed)]
    if case["geom"] == "cavity4":
        low, high = (torch.cat([parts[b]["u"], parts[b + 1]["u"]], 1) for b in (0, 2))
        parts = [{"u": torch.cat([low, high], 2)}]
    box = _Box(case)
    start = {k: torch.nn.functional.pad(a, (1, 1, 1, 1, 1, 1)) for k, a in parts[0].items()}
    vel = [start["u"], torch.zeros_like(start["u"]), torch.zeros_like(start["u"])]
    for q, f in enumerate(vel + ([start["s1"]] if "s1" in start else [])):
        box.fill(f, q)
    vel, p, s = box.steps(vel, torch.zeros_like(vel[0]), start.get("s1"), _dt(case), case["steps"])
    fields = dict(zip(NAMES + ("p", "s1"), vel + [p, s]))
    fields = {k: fields[k] for k in _outputs(case)}
    if case["geom"] != "cavity4":
        return {"%s0" % k: v.contiguous() for k, v in fields.items()}
    hy, hz = case["ny"] // 2, case["nz"] // 2
    return {"%s%d" % (k, b): v[:, (b % 2) * hy:(b % 2) * hy + hy + 2, (b // 2) * hz:(b // 2) * hz + hz + 2].contiguous()
            for k, v in fields.items() for b in range(4)}
