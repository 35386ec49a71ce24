"""The work this framework is used for, as cases that can be timed and compared.

Three kinds of call, all through the public host API of radiant_hip:

* ``pass``: one transport pass of a group (T(z), A z or z - A z) on state vectors that stay on the
  GPU, as an external Krylov solver applies the operator (rt_problem_pass_device).
* ``solve``: one fixed-source multigroup solve of a resident problem, its flux moments collected
  into host memory, as ``compute_flux`` returns them to Radiant (with the flux at the cutoff energy
  for the slowing-down types).
* ``batch`` and ``serve``: many uneven problems solved together, and a stream of requests submitted
  to the server, every result collected.

Inputs are seeded synthetic problems in Radiant's array layouts (radiant_hip.problems): random
downscatter cross sections, random or checkerboard material maps, a box source.  What a user keeps
between calls (the uploaded problem, the batch, the server) is made by ``prepare``.

``exact`` restates the transport pass (cell closures as weak-form matrices, plane-by-plane sweep,
half-range boundary moments) and the group loop in plain torch FP64 on the same input arrays.
"""
import math
import os
import sys
import time

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "radiant.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from radiant_hip import _lib, problems, solver  # noqa: E402

DEV = "cuda:0"


# ------------------------------------------------------------------------------------------
# Cases
# ------------------------------------------------------------------------------------------
def listed():
    return [
        # Passes: the operator alone, from a launch-bound slab to what the pass's scratch holds.
        # The 1D slab of the benchmark suite (200 cells, P7, S16): the smallest call there is.
        dict(name="slab_pass", kind="pass", nd=1, nx=200, ny=1, nz=1, G=10, L=7, order=16, mode=2),
        # The 2D plane of the benchmark suite (128 x 128, P5, 128 directions), inhomogeneous pass.
        dict(name="plane_pass", kind="pass", nd=2, nx=128, ny=128, nz=1, G=4, L=5, order=8, mode=0),
        # A ragged 3D box with 80 directions: near the largest state the allocation-free pass takes.
        dict(name="box_pass", kind="pass", nd=3, nx=31, ny=29, nz=30, G=3, L=3, order=8, mode=2),
        # Solves, FP64 as Radiant computes them (all moments in the Krylov state).
        # The 1D slab of the benchmark suite: ten groups of a few iterations, bound by latency.
        dict(name="slab_solve", kind="solve", nd=1, nx=200, ny=1, nz=1, G=10, L=7, order=16, precision="fp64"),
        # Electrons in a slab: Boltzmann-Fokker-Planck with linear discontinuous cells in space and
        # energy, flux and cutoff flux.
        dict(name="slab_electrons", kind="solve", nd=1, nx=120, ny=1, nz=1, G=6, L=7, order=16, precision="fp64",
             electrons=True, closure="DG", k=2),
        # A reflected 2D cell with linear discontinuous closures and Anderson acceleration.
        dict(name="plane_dg_solve", kind="solve", nd=2, nx=36, ny=31, nz=1, G=3, L=3, order=8, precision="fp64",
             accel="anderson", closure="DG", k=2, reflect=True),
        # A 3D box in FP64 with the faithful GMRES state.
        dict(name="box_solve", kind="solve", nd=3, nx=40, ny=37, nz=42, G=3, L=3, order=8, precision="fp64"),
        # Solves, mixed precision (FP32 passes inside FP64 refinement): the production mode.
        # The 2D plane of the benchmark suite at a quarter of its groups.
        dict(name="plane_solve_mixed", kind="solve", nd=2, nx=128, ny=128, nz=1, G=5, L=5, order=8,
             precision="mixed-fp32"),
        # The benchmark's 64^3 cube with 168 directions at four groups: the largest case.
        dict(name="cube_solve_mixed", kind="solve", nd=3, nx=64, ny=64, nz=64, G=4, L=3, order=12,
             precision="mixed-fp32"),
        # Electrons in a 3D box (order-1 cells, angular Fokker-Planck on the Carlson set).
        dict(name="box_electrons", kind="solve", nd=3, nx=24, ny=26, nz=21, G=4, L=3, order=6, precision="mixed-fp32",
             electrons=True),
        # Many uneven 2D problems advanced together (32..96 cells per axis, 8 to 16 groups).
        dict(name="plane_batch", kind="batch", n=12, mix=1, nmin=32, nmax=96, gmin=8, gmax=16, precision="mixed-fp32"),
        # A burst of 3D requests to the server, every flux collected by its client.
        dict(name="box_requests", kind="serve", n=6, mix=2, nmin=20, nmax=36, gmin=3, gmax=6, precision="mixed-fp32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges: sizes log-uniform, ragged grids, the same options."""
    kind = rng.choice(["pass", "pass", "solve64", "solve64", "mixed", "mixed", "electrons", "closure", "batch", "serve"])
    if kind in ("pass", "solve64", "mixed"):
        nd = rng.choice([1, 2, 3])
        c = dict(kind="pass" if kind == "pass" else "solve", nd=nd)
        if nd == 1:
            c.update(nx=_log(rng, 40, 500), ny=1, nz=1, G=rng.randint(3, 12), L=rng.choice([3, 5, 7]),
                     order=rng.choice([8, 12, 16, 24]))
        elif nd == 2:
            top = 140 if kind == "pass" else 128
            c.update(nx=_log(rng, 16, top), ny=_log(rng, 16, top), nz=1, G=rng.randint(2, 5), L=rng.randint(1, 5),
                     order=rng.choice([4, 6, 8]))
        else:
            hi = 30 if kind == "pass" else (40 if kind == "solve64" else 64)
            orders = [4, 6, 8] if kind == "pass" else ([4, 6, 8] if kind == "solve64" else [4, 8, 10, 12])
            c.update(nx=_log(rng, 10, hi), ny=_log(rng, 10, hi), nz=_log(rng, 10, hi), G=rng.randint(2, 4),
                     L=rng.randint(1, 3), order=rng.choice(orders))
        if kind == "pass":
            c["mode"] = rng.choice([0, 1, 2])
            if rng.random() < 0.25:
                c["reflect"] = True
        else:
            c["precision"] = "fp64" if kind == "solve64" else rng.choice(["mixed-fp32", "mixed-fp32", "mixed-bf16"])
            if kind == "solve64":
                c["accel"] = rng.choice(["gmres", "gmres", "anderson", "bicgstab"])
                c["reflect"] = rng.random() < 0.25
        return c
    if kind == "electrons":
        if rng.random() < 0.5:
            return dict(kind="solve", nd=1, nx=_log(rng, 40, 300), ny=1, nz=1, G=rng.randint(3, 8), L=rng.choice([3, 7]),
                        order=rng.choice([8, 16]), precision="fp64", electrons=True, closure="DG", k=2)
        return dict(kind="solve", nd=3, nx=_log(rng, 10, 26), ny=_log(rng, 10, 26), nz=_log(rng, 10, 26),
                    G=rng.randint(2, 4), L=rng.randint(1, 3), order=rng.choice([4, 6]), precision="mixed-fp32",
                    electrons=True)
    if kind == "closure":
        return dict(kind=rng.choice(["pass", "solve"]), nd=2, nx=_log(rng, 12, 40), ny=_log(rng, 12, 40), nz=1,
                    G=rng.randint(2, 3), L=rng.randint(1, 3), order=rng.choice([4, 6, 8]), precision="fp64", mode=2,
                    accel=rng.choice(["gmres", "anderson"]), closure="DG", k=2, reflect=rng.random() < 0.5)
    if kind == "batch":
        return dict(kind="batch", n=rng.randint(4, 14), mix=rng.randint(10, 10 ** 6), nmin=24, nmax=rng.randint(60, 96),
                    gmin=6, gmax=rng.randint(10, 16), precision="mixed-fp32")
    return dict(kind="serve", n=rng.randint(3, 7), mix=rng.randint(10, 10 ** 6), nmin=16, nmax=rng.randint(24, 36),
                gmin=2, gmax=rng.randint(3, 6), precision="mixed-fp32")


# ------------------------------------------------------------------------------------------
# Inputs
# ------------------------------------------------------------------------------------------
def _problem(c, seed):
    nd, dims = c["nd"], (c["nx"], c["ny"], c["nz"])
    s = 20260000 + int(seed)
    opts = dict(G=c["G"], L=c["L"], quad_order=c["order"], seed=s)
    if nd == 1 and dims[0] == 200 and not c.get("electrons"):
        p = problems.config0(seed=s)
    elif nd == 2 and dims[0] == dims[1] and not c.get("closure"):
        p = problems.config_2d(N=dims[0], block=max(1, dims[0] // 8), **opts)
    elif nd == 3 and dims[0] == dims[1] == dims[2] and not c.get("electrons"):
        p = problems.config_3d(N=dims[0], width=0.1 * dims[0], **opts)
    else:  # ragged grids: cells of 0.05 cm (slab), 0.08 cm (plane) or 0.1 cm (box)
        p = problems.small_problem(nd, dims=dims, Nmat=3 if nd == 3 else 2, **opts)
        h = {1: 0.05, 2: 0.08, 3: 0.1}[nd]
        p.dx = p.dx * h
        if nd >= 2:
            p.dy = p.dy * h
        if nd >= 3:
            p.dz = p.dz * h
    p.tol = 1e-10
    p.accel = c.get("accel", "gmres")
    if c.get("reflect"):  # reflected on the low faces, void on the high ones
        p.bc = np.array([1, 0] * nd, np.int32)
    if c.get("closure"):
        p.scheme, p.scheme_order = c["closure"], c["k"]
        if nd >= 2:
            p.scheme_y, p.scheme_order_y = c["closure"], c["k"]
    if c.get("electrons"):
        r = np.random.default_rng(seed)
        p.csd, p.solver_type, p.fokker_planck = True, "BFP", "finite-difference"
        p.Sb = 0.7 * r.uniform(0.5, 2.0, (p.G + 1, p.Nmat))
        p.dE = r.uniform(0.5, 1.5, p.G)
        p.T = 0.25 * r.uniform(0.2, 1.0, (p.G, p.Nmat))
        if c.get("closure"):
            p.scheme_e, p.scheme_order_e = c["closure"], c["k"]
    return p


def _many(c, seed):
    """The problems of a batch or of a burst of requests: sizes from the case, values from the seed."""
    r = problems.SplitMix64(1000003 * c["mix"] + 17)
    out = []
    for i in range(c["n"]):
        N, G = r.randint(c["nmin"], c["nmax"]), r.randint(c["gmin"], c["gmax"])
        s = 7919 * (int(seed) + 1) + i
        if c["kind"] == "batch":
            L, qo = r.randint(1, 5), (6, 8)[r.randint(0, 1)]
            out.append(problems.config_2d(N=N, G=G, L=L, quad_order=qo, block=max(1, N // 8), seed=s))
        else:
            qo = (6, 8, 10)[r.randint(0, 2)]
            out.append(problems.config_3d(N=N, width=0.1 * N, G=G, L=3, quad_order=qo, Nmat=3, seed=s))
    return out


def _pass_inputs(c, seed, d, S):
    """State vector and out-of-group source of a pass: a positive scalar flux, higher moments that
    fall off with their Legendre order, boundary moments alike; the source only on the moments the
    cross sections reach."""
    g = torch.Generator(device=DEV)
    g.manual_seed(1 + int(seed))
    pl = torch.as_tensor(d.keep["pl"], device=DEV)
    fall = 0.5 ** pl.double()
    z = torch.randn(S, generator=g, device=DEV, dtype=torch.float64)
    n = d.Nc * d.Np
    m = z[:n].view(d.Nc, d.Np)
    m.mul_(0.1 * fall * fall)
    m[:, 0] += 1.0
    z[n:] *= 0.1
    q = torch.randn(d.Nc, d.Np, generator=g, device=DEV, dtype=torch.float64) * fall * (pl <= d.desc.Ls)
    return z, q


def _handle_kw(c):
    return dict(precision=c.get("precision", "fp64"), state="reduced" if c.get("precision", "fp64") != "fp64" else "faithful")


def prepare(case, seed):
    c = case
    if c["kind"] == "pass":
        h = solver.ResidentProblem(_problem(c, seed))
        z, q = _pass_inputs(c, seed, h.d, h.state_length())
        return dict(kind="pass", h=h, z=z, q=q, out=torch.empty_like(z), mode=c["mode"])
    if c["kind"] == "solve":
        return dict(kind="solve", h=solver.ResidentProblem(_problem(c, seed), **_handle_kw(c)), cutoff=bool(c.get("electrons")))
    if c["kind"] == "batch":
        return dict(kind="batch", h=solver.ResidentBatch(_many(c, seed), precision=c["precision"]))
    srv = solver.Server(64 << 30, max_active=4, precision=c["precision"])
    return dict(kind="serve", h=srv, descs=[srv.describe(p) for p in _many(c, seed)])


def run(state):
    h = state["h"]
    if state["kind"] == "pass":
        _lib.check(_lib.lib().rt_problem_pass_device(h.h, 1, state["mode"], state["q"].data_ptr(),
                                                     state["z"].data_ptr(), state["out"].data_ptr()))
        return {"state": state["out"]}
    if state["kind"] == "solve":
        h.solve()
        out = {"flux": h.flux().reshape(-1, order="F")}
        if state["cutoff"]:
            out["cutoff"] = h.flux_cutoff().reshape(-1, order="F")
        return out
    if state["kind"] == "batch":
        h.solve()
        return [h.flux(i).reshape(-1, order="F") for i in range(len(h.descs))]
    ids = [h.submit(d) for d in state["descs"]]
    got = {}
    while len(got) < len(ids):
        busy = True
        for r in ids:
            if r not in got:
                v = h.poll(r)
                if v is not None:
                    got[r] = v[0].reshape(-1, order="F")
                    busy = False
        if busy:
            time.sleep(0.0002)
    return [got[r] for r in ids]


# ------------------------------------------------------------------------------------------
# What a pass or solve cannot do without
# ------------------------------------------------------------------------------------------
_DIRS = {1: lambda n: n, 2: lambda n: 2 * n * n, 3: lambda n: n * (n + 2)}


def _sizes(c):
    nd = c["nd"]
    cells = c["nx"] * c["ny"] * c["nz"]
    K = 1
    if c.get("closure"):
        K = c["k"] ** (nd + (1 if c.get("electrons") else 0))
    N = _DIRS[nd](c["order"])
    if c.get("electrons"):
        act = N
    else:
        act = min(N, {1: c["L"] + 1, 2: (c["L"] + 1) ** 2, 3: (c["L"] + 1) ** 2}[nd])
    return cells, K, N, act


def _solve_work(cells, K, N, act, G):
    # at least an inhomogeneous pass, three iterations and the reconstruction per group
    col = cells * K
    flops = G * (4 * (2.0 * N * act * col * 2 + 10.0 * N * col) + 2.0 * N * N * col)
    return 8.0 * G * N * col + 8.0 * G * cells + 4.0 * cells, flops


def work(case):
    c = case
    if c["kind"] == "pass":
        cells, K, N, act = _sizes(c)
        col = cells * K
        src = act * col if c["mode"] == 0 else 0
        return {"bytes": 8.0 * (2 * N * col + src) + 4.0 * cells, "flops": 2.0 * N * (act + N) * col + 10.0 * N * col}
    if c["kind"] == "solve":
        b, f = _solve_work(*_sizes(c), c["G"])
        return {"bytes": b, "flops": f}
    B = F = 0.0
    for p in _many(c, 0):
        N = _DIRS[p.ndims](p.quad_order)
        b, f = _solve_work(p.Nc, 1, N, min(N, (p.Lxs + 1) ** 2), p.G)
        B, F = B + b, F + f
    return {"bytes": B, "flops": F}


def tolerance(case):
    # A pass is FP64 sums of at most a few hundred terms through the pair M, D (condition 2e5 for
    # the 2D product set: 2e-15 seen against exact(); below 1e-16 elsewhere).  Solves stop at a
    # relative residual of 1e-10, which leaves errors of 3e-12 to 5e-11 in the flux.
    if case["kind"] == "pass":
        return {"rel": 1e-14, "max": 1e-12}
    return {"rel": 2e-10, "max": 2e-8}


# ------------------------------------------------------------------------------------------
# The same results in plain torch FP64
# ------------------------------------------------------------------------------------------
class _Transport:
    """Passes and group solves of one problem from its input arrays (column-major, as Radiant
    passes them).  Cells hold the moments over (E, x, y, z), energy fastest, full coupling."""

    def __init__(self, p, d, dev):
        self.dev, k, q = dev, d.keep, d.desc
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev, dtype=torch.float64)
        self.nd, self.G, self.Nd, self.Np, self.Nps = q.ndims, q.G, q.Nd, q.Np, q.Nps
        self.N = N = [q.Nx, q.Ny, q.Nz]
        self.cells, self.csd = N[0] * N[1] * N[2], bool(q.csd)
        self.O = O = [max(1, q.order_e), max(1, q.order_x), max(1, q.order_y), max(1, q.order_z)]
        self.K = O[0] * O[1] * O[2] * O[3]
        dd = np.array([-1.0, 2.0])
        self.w = [k.get("omega_" + a, dd) for a in "exyz"]
        nmat, self.Ls = q.Nmat, q.Ls
        self.sigt = k["sigt"].reshape((self.G, nmat), order="F")
        self.sigs = k["sigs"].reshape((nmat, self.G, self.G, q.Ls + 1), order="F")
        self.mat = torch.as_tensor(k["mat"] - 1, device=dev)
        self.pl = k["pl"]
        M, D = k["M"].reshape((self.Nd, self.Np), order="F"), k["D"].reshape((self.Np, self.Nd), order="F")
        self.T = k["T"].reshape((self.G, nmat), order="F") if "T" in k else None
        self.act = [i for i in range(self.Np) if self.pl[i] <= q.Ls or self.T is not None]
        self.M, self.D, self.Dact = t(M[:, self.act]), t(D), t(D[self.act])
        self.Mfp = t(k["Mfp"].reshape((self.Np, self.Np), order="F")) if "Mfp" in k else None
        self.qvol = t(k["qvol"].reshape((self.G, self.cells), order="F"))
        if self.csd:
            self.Sb, self.dE = k["Sb"].reshape((self.G + 1, nmat), order="F"), k["dE"]
        self.cos = [k["mu"], k["eta"], k["xi"]]
        self.h = [k["dx"], k["dy"], k["dz"]]
        self._order()
        self._boundary(q, k, t)
        self.g = None

    # sweep order: cells sorted by plane kx + ky + kz, each direction's own cell index per entry
    def _order(self):
        Nx, Ny, Nz = self.N
        kz, ky, kx = (a.ravel() for a in np.meshgrid(np.arange(Nz), np.arange(Ny), np.arange(Nx), indexing="ij"))
        pl = kx + ky + kz
        o = np.argsort(pl, kind="stable")
        kx, ky, kz, pl = kx[o], ky[o], kz[o], pl[o]
        ends = np.searchsorted(pl, np.arange(pl[-1] + 2))
        self.planes = [(int(a), int(b)) for a, b in zip(ends[:-1], ends[1:])]
        i = lambda a: torch.as_tensor(a, device=self.dev)
        self.pos = [i(ky + Ny * kz), i(kx + Nx * kz), i(kx + Nx * ky)]
        fw = np.stack([np.asarray(c) >= 0 for c in self.cos], 1)
        self.ax = []       # true index along each axis, per direction and sweep entry
        for a, kk in enumerate((kx, ky, kz)):
            f = i(fw[:, a])[:, None]
            self.ax.append(torch.where(f, i(kk)[None], i(self.N[a] - 1 - kk)[None]))
        self.cidx = self.ax[0] + Nx * (self.ax[1] + Ny * self.ax[2])
        others = [(1, 2), (0, 2), (0, 1)]
        self.ppos = []     # face position in sweep order -> true position, per direction
        for a, (u, v) in enumerate(others):
            m = np.arange(self.N[u] * self.N[v])
            ku, kv = m % self.N[u], m // self.N[u]
            tu = torch.where(i(fw[:, u])[:, None], i(ku)[None], i(self.N[u] - 1 - ku)[None])
            tv = torch.where(i(fw[:, v])[:, None], i(kv)[None], i(self.N[v] - 1 - kv)[None])
            self.ppos.append(tu + self.N[u] * tv)
        self.fm = [self.K // self.O[a + 1] for a in range(3)]
        self.fe = self.K // self.O[0]

    def _boundary(self, q, k, t):
        self.bnd, self.nonvoid = [], False
        for a in range(self.nd):
            c = np.asarray(self.cos[a])
            Dex, Men = np.zeros((self.Nd, self.Nps)), np.zeros((self.Nd, self.Nps))
            src = np.full(self.Nd, -1)
            n2p = [k[f"n2p{2 * a + f}"] for f in (0, 1)]
            Ds = [k[f"Ds{2 * a + f}"].reshape((self.Nps, -1), order="F") for f in (0, 1)]
            Ms = [k[f"Ms{2 * a + f}"].reshape((-1, self.Nps), order="F") for f in (0, 1)]
            for n in range(self.Nd):
                f = 0 if n2p[0][n] else 1
                Dex[n], Men[n] = Ds[f][:, n2p[f][n] - 1], Ms[f][n2p[f][n] - 1]
                side = 0 if c[n] >= 0 else 1  # face it enters through
                code = k["bc"][2 * a + side]
                if code:
                    src[n] = side if code == 1 else 1 - side
                    self.nonvoid = True
            ex = [torch.as_tensor(np.nonzero((c >= 0) == (f == 1))[0], device=self.dev) for f in (0, 1)]
            self.bnd.append((t(Dex), t(Men), src, ex))

    def group(self, g):
        if self.g == g:
            return
        self.g, O, K = g, self.O, self.K
        dev, Nd, J = self.dev, self.Nd, self.cells
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev, dtype=torch.float64)
        self.sig = t(self.sigs[:, g, g, :])[:, [min(int(self.pl[i]), self.Ls) for i in self.act]]  # [mat, act]
        hi = torch.as_tensor([self.pl[i] > self.Ls for i in self.act], device=dev)
        self.sig[:, hi] = 0.0
        m = self.mat[self.cidx]                                                 # [Nd, J]
        C = [np.sqrt(2.0 * i + 1.0) for i in range(8)]
        hh = [t(np.abs(self.cos[a]))[:, None] / t(self.h[a])[self.ax[a]] if a < self.nd else None for a in range(3)]
        sg = [np.sign(np.asarray(self.cos[a])) for a in range(3)]
        A = torch.zeros(Nd, J, K, K, device=dev, dtype=torch.float64)
        St = t(self.sigt[g])[m]
        Sm = Sp = None
        if self.csd:
            Sm, Sp = t(self.Sb[g] / self.dE[g])[m], t(self.Sb[g + 1] / self.dE[g])[m]
            Sv = [(Sm + Sp) / 2, (Sm - Sp) / (2 * math.sqrt(3.0))]
        idx = [(e, a, b, c) for c in range(O[3]) for b in range(O[2]) for a in range(O[1]) for e in range(O[0])]
        self.fin = []  # (axis, face moment) -> coefficient of the inflow in each cell moment
        self.fout, self.face_of = [], []
        for ii, mi in enumerate(idx):
            A[:, :, ii, ii] += St
            for jj, mj in enumerate(idx):
                for ax in range(self.nd):
                    if any(mi[x] != mj[x] for x in range(4) if x != ax + 1):
                        continue
                    u, v, s = mi[ax + 1], mj[ax + 1], sg[ax]
                    cst = C[u] * C[v] * (s ** u * s ** v * self.w[ax + 1][v + 1] - (2 * s if u > v and (u - v) % 2 else 0))
                    A[:, :, ii, jj] += t(cst)[:, None] * hh[ax]
                if self.csd and mi[1:] == mj[1:]:
                    e, f = mi[0], mj[0]
                    if e == 1:
                        A[:, :, ii, jj] += 2 * C[1] * Sv[f]
                    A[:, :, ii, jj] += C[e] * (-1) ** e * C[f] * (-1) ** f * self.w[0][f + 1] * Sp
        axes = ([0] if self.csd else []) + [a + 1 for a in range(self.nd)]
        for ax in axes:
            rest = [x for x in range(4) if x != ax]
            size = K // O[ax]
            coef = torch.zeros(Nd, J, K, device=dev, dtype=torch.float64)
            out = torch.zeros(Nd, K, device=dev, dtype=torch.float64)
            of = []
            for ii, mi in enumerate(idx):
                r, st = 0, 1
                for x in rest:
                    r, st = r + mi[x] * st, st * O[x]
                of.append(r)
                v = mi[ax]
                if ax == 0:
                    coef[:, :, ii] = -C[v] * ((-1) ** v * self.w[0][0] * Sp - Sm)
                    out[:, ii] = C[v] * (-1) ** v * self.w[0][v + 1]
                else:
                    s = sg[ax - 1]
                    coef[:, :, ii] = -t(C[v] * (s ** v * self.w[ax][0] - (-s) ** v))[:, None] * hh[ax - 1]
                    out[:, ii] = t(C[v] * s ** v * self.w[ax][v + 1])
            self.fin.append(coef)
            self.fout.append(out)
            self.face_of.append((ax, torch.as_tensor(of, device=dev), size))
        if K == 1:
            self.inv = 1.0 / A
        else:
            flat = A.reshape(-1, K, K).cpu()
            self.inv = torch.linalg.inv(flat).reshape(Nd, J, K, K).to(dev)

    def sweep(self, src, bin_, Ein):
        """src [Nd, cells, K] -> (psi [Nd, cells, K], exit faces, energy outflow)."""
        Nd, K = self.Nd, self.K
        q = torch.gather(src, 1, self.cidx[:, :, None].expand(-1, -1, K))
        F = [torch.gather(b, 1, self.ppos[a][:, :, None].expand(-1, -1, self.fm[a])) for a, b in enumerate(bin_)]
        E = torch.gather(Ein, 1, self.cidx[:, :, None].expand(-1, -1, self.fe)) if Ein is not None else None
        Eo = torch.zeros(Nd, self.cells, self.fe, device=self.dev, dtype=torch.float64) if self.csd else None
        for a, b in self.planes:
            r, ins = q[:, a:b], []
            for (ax, of, size), coef in zip(self.face_of, self.fin):
                if ax == 0:
                    f = E[:, a:b] if E is not None else torch.zeros(Nd, b - a, size, device=self.dev, dtype=torch.float64)
                else:
                    f = F[ax - 1][:, self.pos[ax - 1][a:b]]
                ins.append(f)
                r = r + coef[:, a:b] * (f if K == 1 else f[:, :, of])
            x = self.inv[:, a:b, 0] * r if K == 1 else (self.inv[:, a:b] * r[:, :, None, :]).sum(-1)
            q[:, a:b] = x
            for (ax, of, size), out, f in zip(self.face_of, self.fout, ins):
                y = x * out[:, None]
                if K > 1:
                    y = torch.zeros_like(f).index_add_(2, of, y)
                y = y + self.w[ax][0] * f
                if ax == 0:
                    Eo[:, a:b] = y
                else:
                    F[ax - 1][:, self.pos[ax - 1][a:b]] = y
        psi = torch.empty_like(q).scatter_(1, self.cidx[:, :, None].expand(-1, -1, K), q)
        ex = [torch.empty_like(f).scatter_(1, self.ppos[a][:, :, None].expand(-1, -1, self.fm[a]), f) for a, f in enumerate(F)]
        if Eo is not None:
            Eo = torch.empty_like(Eo).scatter_(1, self.cidx[:, :, None].expand(-1, -1, self.fe), Eo)
        return psi, ex, Eo

    def angular(self, g, phi, bm, qlout, Ein):
        """One pass of group g on the active moments phi [act, col] and boundary moments bm."""
        self.group(g)
        s = torch.zeros(len(self.act), self.cells * self.K, device=self.dev, dtype=torch.float64) if qlout is None else qlout
        col = self.mat.repeat_interleave(self.K)
        if phi is not None:
            s = s + self.sig[col].t() * phi
            if self.T is not None:
                Tm = torch.as_tensor(self.T[g], device=self.dev)[col]
                s = s + Tm * (self.Mfp @ phi)
        src = (self.M @ s).view(self.Nd, self.cells, self.K)
        bin_ = []
        for a in range(self.nd):
            _, Men, fs, _ = self.bnd[a]
            b = torch.zeros(self.Nd, self.ppos[a].shape[1], self.fm[a], device=self.dev, dtype=torch.float64)
            if bm is not None:
                for f in (0, 1):  # bm[a]: [pos, 2, fm, Nps]
                    n = np.nonzero(fs == f)[0]
                    if len(n):
                        n = torch.as_tensor(n, device=self.dev)
                        x = bm[a][:, f]
                        b[n] = (Men[n] @ x.reshape(-1, self.Nps).t()).view(len(n), *x.shape[:2])
            bin_.append(b)
        return self.sweep(src, bin_, Ein)

    def moments_out(self, ex):
        out = []
        for a in range(self.nd):
            Dex, _, _, lists = self.bnd[a]
            o = torch.zeros(ex[a].shape[1], 2, self.fm[a], self.Nps, device=self.dev, dtype=torch.float64)
            for f in (0, 1):
                n = lists[f]
                o[:, f] = (ex[a][n].reshape(len(n), -1).t() @ Dex[n]).view(-1, self.fm[a], self.Nps)
            out.append(o)
        return out

    def split(self, v):
        """State vector [Phi_act | boundary moments] -> its parts."""
        n = len(self.act) * self.cells * self.K
        phi, b, o = v[:n].view(len(self.act), -1), [], n
        if not self.nonvoid:
            return phi, None
        for a in range(self.nd):
            s = (self.ppos[a].shape[1], 2, self.fm[a], self.Nps)
            b.append(v[o:o + math.prod(s)].view(s))
            o += math.prod(s)
        return phi, b

    def join(self, psi, ex):
        parts = [(self.Dact @ psi.view(self.Nd, -1)).reshape(-1)]
        if self.nonvoid:
            parts += [o.reshape(-1) for o in self.moments_out(ex)]
        return torch.cat(parts)

    def solve_group(self, g, qlout, Ein):
        psi, ex, _ = self.angular(g, None, None, qlout, Ein)
        c = self.join(psi, ex)
        z, cn = torch.zeros_like(c), float(c.norm())
        A = lambda v: v - self.join(*self.angular(g, *self.split(v), None, None)[:2])
        if cn > 0:
            for _ in range(6):  # restarted GMRES, each start from the true residual
                r = c - A(z) if float(z.norm()) > 0 else c
                beta = float(r.norm())
                if beta <= 1e-13 * cn:
                    break
                V, H = [r / beta], np.zeros((41, 40))
                for j in range(40):
                    w = A(V[j])
                    for _ in range(2):
                        for i in range(j + 1):
                            hij = float(w @ V[i])
                            H[i, j] += hij
                            w -= hij * V[i]
                    H[j + 1, j] = float(w.norm())
                    e = np.zeros(j + 2)
                    e[0] = beta
                    y, *_ = np.linalg.lstsq(H[:j + 2, :j + 1], e, rcond=None)
                    res = np.linalg.norm(H[:j + 2, :j + 1] @ y - e)
                    if res <= 2e-14 * cn or H[j + 1, j] <= 1e-15 * beta:
                        break
                    V.append(w / H[j + 1, j])
                for yi, v in zip(y, V):
                    z = z + float(yi) * v
        psi, _, Eo = self.angular(g, *self.split(z), qlout, Ein)
        return self.D @ psi.view(self.Nd, -1), Eo

    def solve(self):
        K, col = self.K, self.mat.repeat_interleave(self.K)
        phi = torch.zeros(self.G, self.Np, self.cells * K, device=self.dev, dtype=torch.float64)
        Ein = torch.zeros(self.Nd, self.cells, self.fe, device=self.dev, dtype=torch.float64) if self.csd else None
        for g in range(self.G):
            q = torch.zeros(len(self.act), self.cells * K, device=self.dev, dtype=torch.float64)
            for gi in range(g):
                for i, p in enumerate(self.act):
                    if self.pl[p] <= self.Ls:
                        s = torch.as_tensor(np.ascontiguousarray(self.sigs[:, gi, g, self.pl[p]]), device=self.dev)
                        q[i] += s[col] * phi[gi, p]
            q[0].view(self.cells, K)[:, 0] += self.qvol[g]
            phi[g], Eo = self.solve_group(g, q, Ein)
            if self.csd and g + 1 < self.G:
                Ein = Eo * (self.dE[g + 1] / self.dE[g])
        out = {"flux": phi.permute(2, 1, 0).reshape(-1)}
        if self.csd:
            cut = torch.zeros(self.cells, K, self.Np, device=self.dev, dtype=torch.float64)
            cut[:, :self.fe] = torch.einsum("pn,nci->cip", self.D, Eo)
            out["cutoff"] = cut.reshape(-1)
        return out


def exact(case, seed):
    c = case
    if c["kind"] in ("batch", "serve"):
        return None
    cells, K, N, _ = _sizes(c)
    if c["kind"] == "solve" and c.get("accel") == "bicgstab":
        return None
    p = _problem(c, seed)
    d = solver.Desc(p, **_handle_kw(c))
    t = _Transport(p, d, DEV if cells * N > 200000 else "cpu")
    if c["kind"] == "solve":
        return t.solve()
    nb = sum(2 * t.Nps * t.fm[a] * t.ppos[a].shape[1] for a in range(t.nd))
    z, q = _pass_inputs(c, seed, d, d.Nc * d.Np + nb)
    z, q = z.to(t.dev), q.to(t.dev)
    n = d.Nc * d.Np
    phi = z[:n].view(d.Nc, d.Np).t()[t.act].contiguous()
    bm, o = [], n
    for a in range(t.nd):
        s = (t.ppos[a].shape[1], 2, t.fm[a], t.Nps)
        bm.append(z[o:o + math.prod(s)].view(s))
        o += math.prod(s)
    ql = q.t()[t.act].contiguous() if c["mode"] == 0 else None
    psi, ex, _ = t.angular(1, phi, bm, ql, None)
    out = torch.cat([(t.D @ psi.view(t.Nd, -1)).t().reshape(-1)] + [b.reshape(-1) for b in t.moments_out(ex)])
    return {"state": z - out if c["mode"] == 2 else out}
