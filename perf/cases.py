"""Performance cases of the band solver: what a program does with it, through fame_amd.

A case is a dict of plain values:
  kind     what one pass runs
             "qbq" / "qr" / "qrs"   one operator apply for one wave vector (Solver.apply)
             "invar"                one shift-invert apply, the step of every Krylov solver on A_r^{-1}
             "fields"               E fields of every band from stored reduced eigenvectors (Solver.restore)
             "check"                relative residuals of given fields (Solver.residuals)
             "adjoint"              backward pass of the band eigenvalues: fields recomputed, then the
                                    gradient with respect to the permittivity (Solver.restore, eig_vjp)
             "eigs"                 the band solve of all wave vectors of one structure (Solver.eigs)
  lattice  lattice type of fame_amd.build_lattice; nx its nominal grid (the grid rule gives the other two)
  mixed    invar / eigs: FP32 CG inside FP64 refinement instead of FP64 throughout
  gamma    operators: the wave vector is Gamma (one mode fewer, the odd vector length) instead of a generic one
  tuned    operators: the program tuned the pass kernels for its grid (Solver.autotune) before its applies;
           otherwise it calls with the plans the context was created with
  nk, nwant, nstep   wave vectors, bands, Krylov dimension
The structures are those of the configurations, tests and benchmark: a sphere in a cubic, body-centred or
hexagonal cell, the diamond network in the FCC cell, and a smooth density for the adjoint.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PY = os.path.join(ROOT, "fame-isotropic-gpu_amd", "python")
if _PY not in sys.path:
    sys.path.insert(0, _PY)

import fame_amd as F  # noqa: E402

DEV = "cuda:0"
SC, FCC, BCC, HEX = "simple_cubic", "face_centered_cubic", "body_centered_cubic", "hexagonal"


def listed():
    return [
        # smallest apply: an operator check or a small supercell sweep, all latency
        dict(name="qbq sc16", kind="qbq", lattice=SC, nx=16, gamma=False, tuned=False),
        # an odd grid at Gamma, as the first point of a band path is
        dict(name="qbq bcc25 gamma", kind="qbq", lattice=BCC, nx=25, gamma=True, tuned=False),
        # field synthesis at the headline grid: plotting or post-processing an eigenvector
        dict(name="qr fcc96", kind="qr", lattice=FCC, nx=96, gamma=False, tuned=True),
        # projection of a given real-space field onto the reduced space, a ragged hexagonal grid
        dict(name="qrs hex50", kind="qrs", lattice=HEX, nx=50, gamma=False, tuned=False),
        # one Krylov step of the small FP64 configuration (SC 32, the parity configuration)
        dict(name="invar f64 sc32", kind="invar", lattice=SC, nx=32, mixed=False, tuned=True),
        # one Krylov step at the headline grid, the reference's arithmetic
        dict(name="invar f64 fcc96", kind="invar", lattice=FCC, nx=96, mixed=False, tuned=True),
        # the same step in the mixed precision that production runs use
        dict(name="invar mixed fcc96", kind="invar", lattice=FCC, nx=96, mixed=True, tuned=True),
        # the largest configured grid (128 x 121 x 105)
        dict(name="invar mixed bcc128", kind="invar", lattice=BCC, nx=128, mixed=True, tuned=True),
        # convergence check of every band of a band diagram's part
        dict(name="check fcc64", kind="check", lattice=FCC, nx=64, nk=4, nwant=12),
        # backward pass of an inverse-design step on the density configuration
        dict(name="adjoint sc64", kind="adjoint", lattice=SC, nx=64, nk=4, nwant=6),
        # whole solve of the parity configuration: one wave vector, FP64
        dict(name="eigs f64 sc32", kind="eigs", lattice=SC, nx=32, mixed=False, nk=1, nwant=10, nstep=30),
        # whole solve of four wave vectors of the headline workload, batched mixed precision
        dict(name="eigs mixed fcc96", kind="eigs", lattice=FCC, nx=96, mixed=True, nk=4, nwant=16, nstep=48),
    ]


def draw(rng):
    """One more case: grids of 12 to 160 points a side for the operators, batches for the rest."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["qbq", "qr", "qrs", "invar", "invar", "fields", "check", "adjoint", "eigs"])
    lat = rng.choice([SC, FCC, BCC, HEX])
    c = dict(kind=kind, lattice=lat)
    if kind in ("qbq", "qr", "qrs"):
        c.update(nx=log_int(12, 160), gamma=rng.random() < 0.25, tuned=rng.random() < 0.5)
    elif kind == "invar":
        c.update(nx=log_int(12, 128), mixed=rng.random() < 0.6, tuned=rng.random() < 0.7)
    elif kind == "eigs":
        nwant = rng.randint(4, 12)
        c.update(nx=log_int(12, 56), mixed=rng.random() < 0.6, nk=log_int(1, 8), nwant=nwant, nstep=3 * nwant)
    else:
        c.update(nx=log_int(16, 96), nk=rng.randint(1, 4), nwant=rng.randint(2, 12))
    return c


# ------------------------------------------------------------------ structures
DIAMOND = F.Material(sphere_centers=[[(0, 0, 0), (0.25, 0.25, 0.25)]], sphere_radius=[[0.15, 0.15]],
                     cylinder_top=[[(0.25, 0.25, 0.25)] * 4],
                     cylinder_bot=[[(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)]], cylinder_radius=[[0.10] * 4])
SPHERE = F.Material(sphere_centers=[[(0.5, 0.5, 0.5)]], sphere_radius=[[0.25]])


@functools.lru_cache(maxsize=32)
def _lattice(lat, nx):
    lo = F.build_lattice(lat, nx, **(dict(c=1.2) if lat == HEX else {}))
    return lo, F.to_fame_lattice(lo)


@functools.lru_cache(maxsize=8)
def _inside(lat, nx):
    lo, _ = _lattice(lat, nx)
    return F.material_index(lo, DIAMOND if lat == FCC else SPHERE)


def _eps(case, rng):
    """Permittivity on the 3N Yee edges (numpy): the lattice's structure with the contrast drawn from
    the configurations' range, or a smoothed random density for the adjoint."""
    lat, nx = case["lattice"], case["nx"]
    _, fl = _lattice(lat, nx)
    if case["kind"] == "adjoint":
        n = tuple(int(v) for v in fl.grid_nums)
        z = rng.standard_normal((n[2], n[1], n[0]))
        k2 = sum(np.fft.fftfreq(m).reshape([-1 if i == d else 1 for i in range(3)]) ** 2 for d, m in enumerate(z.shape))
        z = np.fft.ifftn(np.fft.fftn(z) * np.exp(-2.0 * (np.pi * 2.0) ** 2 * k2)).real
        z /= z.std()
        rho = torch.from_numpy(1.0 + 11.96 / (1.0 + np.exp(-4.0 * z)))
        return F.cell_to_yee(rho).numpy()
    inside = _inside(lat, nx)
    return np.where(inside >= 0, rng.uniform(12.0, 13.0), 1.0)


def _waves(nk, rng):
    """Generic wave vectors inside the first Brillouin zone, away from Gamma (units of 2 pi)."""
    k = rng.uniform(0.08, 0.42, (nk, 3)) * rng.choice([-1.0, 1.0], (nk, 3))
    return k


def _inputs(case, seed):
    """Everything a pass is given, from the seed alone: permittivity, wave vectors, vectors."""
    rng = np.random.default_rng([int(seed), 77])
    _, fl = _lattice(case["lattice"], case["nx"])
    kind, N = case["kind"], int(fl.grid_nums[0]) * int(fl.grid_nums[1]) * int(fl.grid_nums[2])
    d = dict(eps=_eps(case, rng), N=N, fl=fl)
    nk = case.get("nk", 1)
    d["k"] = np.zeros((1, 3)) if case.get("gamma") else _waves(nk, rng)
    gen = torch.Generator(device=DEV).manual_seed(int(seed))

    def normal(*shape):
        return torch.complex(torch.randn(*shape, generator=gen, device=DEV, dtype=torch.float64),
                             torch.randn(*shape, generator=gen, device=DEV, dtype=torch.float64))

    nd = N - 1 if case.get("gamma") else N
    if kind in ("qbq", "qr"):
        d["x"] = normal(2 * nd)
    elif kind == "qrs":
        d["x"] = normal(3 * N)
    elif kind == "invar":
        # a unit vector with a Krylov vector's spectrum: the long waves weigh most
        d["x"] = (normal(2, N) * _decay(fl)).reshape(-1)
        d["x"] /= torch.linalg.vector_norm(d["x"])
    elif kind in ("fields", "check", "adjoint"):
        nwant = case["nwant"]
        y = normal(nk, nwant, 2, N) * _decay(fl)
        d["y"] = (y / torch.linalg.vector_norm(y, dim=(2, 3), keepdim=True)).reshape(nk, nwant, 2 * N)
        d["freq"] = np.sort(rng.uniform(0.2, 0.9, (nk, nwant)), axis=1) * 2 * np.pi
        d["w"] = rng.standard_normal((nk, nwant))
    return d


def _decay(fl):
    """1 / (1 + m^2) per Fourier mode, m the mode's index length, in the reduced vectors' mode order."""
    n = [int(v) for v in fl.grid_nums]
    order = [n[0], n[1], n[2]] if fl.general else [n[2], n[1], n[0]]       # slowest first
    m = [torch.minimum(torch.arange(v, device=DEV), v - torch.arange(v, device=DEV)).double() ** 2 for v in order]
    return (1.0 / (1.0 + m[0][:, None, None] + m[1][None, :, None] + m[2][None, None, :])).reshape(-1)


# ---------------------------------------------------------------------- passes
def prepare(case, seed):
    """The solver of one structure with its wave vectors, and the vectors of the pass."""
    d = _inputs(case, seed)
    S = F.Solver(d["fl"], max_batch=len(d["k"]))
    S.set_eps(d["eps"])
    S.set_wave_vectors(d["k"])
    if case.get("tuned"):
        S.autotune(8)
        if case.get("mixed"):
            S.autotune(4)
    if case["kind"] == "check":
        d["E"] = S.restore(d["y"])
        # the fields as a program reads them back: normalised by its own rule
        d["E"] /= torch.linalg.vector_norm(d["E"], dim=2, keepdim=True)
    d.update(case=case, S=S)
    return d


def run(state):
    c, S, kind = state["case"], state["S"], state["case"]["kind"]
    if kind == "qbq":
        return S.apply(F.OP_QBQ, 0, state["x"])
    if kind == "qr":
        return S.apply(F.OP_QR, 0, state["x"])
    if kind == "qrs":
        return S.apply(F.OP_QRS, 0, state["x"])
    if kind == "invar":
        return S.apply(F.OP_INVAR_MIXED if c["mixed"] else F.OP_INVAR, 0, state["x"])
    if kind == "fields":
        return S.restore(state["y"])
    if kind == "check":
        return S.residuals(state["freq"], state["E"])
    if kind == "adjoint":
        E = S.restore(state["y"])
        return S.eig_vjp(state["freq"], E, state["w"])
    freq, _, _, _ = S.eigs(c["nwant"], c["nstep"], precision=F.PREC_F32_REFINE if c["mixed"] else F.PREC_F64)
    return freq


def work(case):
    """Operands read and results written once.  An iterative solve does that once per QBQ apply, in
    the precision of its iteration: about 30 applies per invAr (the tolerance and contrast fix it),
    and about 7 invAr per band of a whole solve, each with its orthogonalisation against the basis."""
    _, fl = _lattice(case["lattice"], case["nx"])
    N = float(fl.grid_nums[0]) * fl.grid_nums[1] * fl.grid_nums[2]
    fft = 5.0 * N * math.log2(N)                    # one complex 3-D transform of one component
    kind, nk = case["kind"], case.get("nk", 1)
    if kind == "qbq":
        return dict(bytes=(4 * 16 + 3 * 8) * N, flops=6 * fft + 100 * N)
    if kind in ("qr", "qrs"):
        return dict(bytes=5 * 16 * N, flops=3 * fft + 50 * N)
    if kind in ("invar", "eigs"):
        s = 8 if case["mixed"] else 16
        n = 30.0
        one = dict(bytes=n * (10 * s + 3 * s / 2) * N, flops=n * (6 * fft + 150 * N))
        if kind == "invar":
            return one
        m = 7.0 * case["nwant"] * nk
        return dict(bytes=m * (one["bytes"] + 2 * 16 * 2 * N * case["nstep"] / 2),
                    flops=m * (one["flops"] + 16 * 2 * N * case["nstep"] / 2))
    fields = nk * case["nwant"]
    if kind == "fields":
        return dict(bytes=fields * 5 * 16 * N, flops=fields * (3 * fft + 60 * N))
    if kind == "check":
        return dict(bytes=fields * 3 * 16 * N, flops=fields * (6 * fft + 100 * N))
    return dict(bytes=fields * 2 * 16 * N + 3 * 8 * N, flops=fields * (3 * fft + 70 * N))


# ----------------------------------------------------- the same in plain torch
class _Plain:
    """The operators for one wave vector in complex128, modes and grid as (slowest, middle, fastest)."""

    def __init__(self, fl, k):
        n = [int(v) for v in fl.grid_nums]
        h = [float(v) for v in fl.mesh_len]
        a = np.array(list(fl.lattice_vec_a)).reshape(3, 3)
        self.general, self.n = bool(fl.general), n
        if self.general:
            m1, m2, m3 = fl.m1, fl.m2, fl.m3
            c1 = (1.0 if a[1, 0] < 0 else 0.0) - m1 / n[0]
            c2, c3 = m3 / n[1], m2 / n[0]
            a2 = c1 * a[0] + a[1]
            a3 = a[2] - c2 * a2 - c3 * a[0] + np.array(list(fl.t1))
            t = (k @ a3, -m3 / n[1], m1 * m3 / (n[1] * n[0]) - m2 / n[0])
            s, r = (k @ a2, -m1 / n[0]), k @ a[0]
            nc, nb, na = n[0], n[1], n[2]
            hc, hb, ha = h[0], h[1], h[2]
        else:
            t, s, r = (k @ a[0], 0.0, 0.0), (k @ a[1], 0.0), k @ a[2]
            nc, nb, na = n[2], n[1], n[0]
            hc, hb, ha = h[2], h[1], h[0]
        self.shape, self.N = (nc, nb, na), nc * nb * na
        ar = lambda m: torch.arange(m, device=DEV, dtype=torch.float64)  # noqa: E731
        C, B, A = ar(nc)[:, None, None], ar(nb)[None, :, None], ar(na)[None, None, :]
        ex = lambda x: torch.polar(torch.ones_like(x), 2 * math.pi * (x - torch.round(x)))  # noqa: E731
        phi, psi = t[0] + t[1] * B + t[2] * C, s[0] + s[1] * C
        # symbols (e^{2 pi i x} - 1)/h as 2i sin(pi x) e^{i pi x}/h, without cancellation
        def lam(x, hh):
            p = math.pi * x
            return torch.complex(-2 * torch.sin(p) ** 2, 2 * torch.sin(p) * torch.cos(p)) / hh
        La, Lb, Lc = lam((A + phi) / na, ha), lam((B + psi) / nb, hb), lam((C + r) / nc, hc)
        La, Lb, Lc = (v.expand(self.shape) for v in (La, Lb, Lc))
        self.L = (Lc, Lb, La) if self.general else (La, Lb, Lc)
        self.ta, self.tb, self.tc = ex(phi * A / na), ex(psi * B / nb), ex(r * C / nc)
        lx, ly, lz = self.L
        self.q = sum(v.abs() ** 2 for v in self.L)
        self.gone = float(np.linalg.norm(k)) < (1e-3 if self.general else 1e-4)
        if self.general:
            S = lx + ly + lz
            d = 3 * self.q - S.abs() ** 2
            p1 = [(self.q - v * S.conj()) / torch.sqrt(self.q * d) for v in self.L]
            p2 = [v / torch.sqrt(d) for v in ((lz - ly).conj(), (lx - lz).conj(), (ly - lx).conj())]
        else:
            t1, t2, t3 = 5 * lz - ly, lx - 3 * lz, 3 * ly - 5 * lx
            d = torch.sqrt(t1.abs() ** 2 + t2.abs() ** 2 + t3.abs() ** 2)
            p2 = [v.conj() / d for v in (t1, t2, t3)]
            e = d * torch.sqrt(self.q)
            p1 = [(t3 * ly.conj() - t2 * lz.conj()) / e, (t1 * lz.conj() - t3 * lx.conj()) / e,
                  (t2 * lx.conj() - t1 * ly.conj()) / e]
        if self.gone:
            for v in p1 + p2:
                v.view(-1)[0] = 0
        self.p1, self.p2 = p1, p2

    def synth(self, u):
        return torch.fft.ifft(torch.fft.ifft(torch.fft.ifft(u, dim=2) * self.ta, dim=1) * self.tb, dim=0) * self.tc

    def analyse(self, v):
        v = torch.fft.fft(v * self.tc.conj(), dim=0) * self.tb.conj()
        return torch.fft.fft(torch.fft.fft(v, dim=1) * self.ta.conj(), dim=2)

    def pad(self, x):
        x = x.reshape(2, -1)
        if self.gone:
            x = torch.cat([torch.zeros(2, 1, dtype=x.dtype, device=x.device), x], 1)
        return x.reshape(2, *self.shape)

    def cut(self, y):
        y = y.reshape(2, -1)
        return (y[:, 1:] if self.gone else y).reshape(-1)

    def ref(self, v):          # own order -> x fastest
        return (v.permute(2, 1, 0) if self.general else v).reshape(-1)

    def own(self, v):          # x fastest -> own order
        nx, ny, nz = self.n
        v = v.reshape(nz, ny, nx)
        return v.permute(2, 1, 0).contiguous() if self.general else v

    def qr(self, x2):
        return [self.synth(self.p1[c] * x2[0] + self.p2[c] * x2[1]) for c in range(3)]

    def qrs(self, f):
        y = [self.analyse(v) for v in f]
        return torch.stack([sum(p[c].conj() * y[c] for c in range(3)) for p in (self.p1, self.p2)])

    def qbq(self, ib, x2):
        return self.qrs([b * v for b, v in zip(ib, self.qr(x2))])

    def curlcurl(self, f):
        l, e = self.L, [self.analyse(v) for v in f]
        cross = lambda p, q: [p[1] * q[2] - p[2] * q[1], p[2] * q[0] - p[0] * q[2], p[0] * q[1] - p[1] * q[0]]  # noqa: E731
        return [self.synth(v) for v in cross([-v.conj() for v in l], cross(l, e))]


def exact(case, seed):
    """What run returns, in plain torch and 64 bits; None for the eigensolves."""
    kind = case["kind"]
    if kind == "eigs":
        return None
    d = _inputs(case, seed)
    eps = torch.from_numpy(d["eps"]).to(DEV).reshape(3, -1)
    if kind in ("qbq", "qr", "qrs", "invar"):
        P = _Plain(d["fl"], d["k"][0])
        ib = [1.0 / P.own(e) for e in eps]
        if kind == "qbq":
            return P.cut(P.qbq(ib, P.pad(d["x"])))
        if kind == "qr":
            return torch.cat([P.ref(v) for v in P.qr(P.pad(d["x"]))])
        if kind == "qrs":
            return P.cut(P.qrs([P.own(v) for v in d["x"].reshape(3, -1)]))
        rs = torch.rsqrt(P.q)
        b = P.pad(d["x"]) * rs
        x, r = torch.zeros_like(b), b.clone()
        p, rr = r.clone(), torch.vdot(r.reshape(-1), r.reshape(-1)).real
        for _ in range(400):
            q = P.qbq(ib, p)
            al = rr / torch.vdot(p.reshape(-1), q.reshape(-1)).real
            x, r = x + al * p, r - al * q
            new = torch.vdot(r.reshape(-1), r.reshape(-1)).real
            if float(new) < 1e-28:
                break
            p, rr = r + (new / rr) * p, new
        return P.cut(x * rs)
    nk, nwant, N = case["nk"], case["nwant"], d["N"]
    E = torch.empty((nk, nwant, 3 * N), dtype=torch.complex128, device=DEV)
    res = torch.empty((nk, nwant), dtype=torch.float64, device=DEV)
    g = torch.zeros(3 * N, dtype=torch.float64, device=DEV)
    for i in range(nk):
        P = _Plain(d["fl"], d["k"][i])
        ib, e = [1.0 / P.own(v) for v in eps], [P.own(v) for v in eps]
        for j in range(nwant):
            lam = float(d["freq"][i, j]) ** 2
            f = [b * v for b, v in zip(ib, P.qr(P.pad(d["y"][i, j]) * torch.sqrt(P.q)))]
            nrm = torch.sqrt(sum((v.abs() ** 2).sum() for v in f))
            if kind == "check":
                f = [v / nrm for v in f]
                r = [c - lam * b * v for c, b, v in zip(P.curlcurl(f), e, f)]
                res[i, j] = torch.sqrt(sum((v.abs() ** 2).sum() for v in r))
                continue
            E[i, j] = torch.cat([P.ref(v * nrm) for v in f])
            if kind == "adjoint":
                w = E[i, j].abs() ** 2
                g -= d["w"][i, j] * lam * w / (eps.reshape(-1) * w).sum()
    return E if kind == "fields" else res if kind == "check" else g
