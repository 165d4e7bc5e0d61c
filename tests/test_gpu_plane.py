"""The plane path of the QBQ (the two outer axes in one pass over (b, c) planes in
LDS) against the FP64 oracle, at the sizes where its kernels can go wrong: odd and
even rows (linear or padded LDS rows), odd planes (padding of the plane pitch),
direct DFTs on the matrix cores along every axis (plane axes of 8 to 24 points and
prime ones; the radix passes of longer composite axes are in test_gpu_plane_passes),
line counts that leave the last block of the inner kernels ragged, Gamma, and every
lines-per-block and thread count its rule accepts.  Both precisions hold the bars of
the axis passes: 1e-11 of the oracle in FP64, 2e-6 in FP32, 1e-8 in lambda for an
FP32-refined solve, and the two paths agree within those bars."""
import numpy as np
import pytest

import fame_amd as F
import oracle as O
from cases import SPHERE

pytestmark = pytest.mark.gpu

O.set_threads(8)

# grid sides (a, b, c) reached: 9^3, 16^3, 17^3, 18^3 (direct DFTs along b and c), 26^3 (13 x 2 passes),
# 34^3 (2 x 17: direct), FCC 22x19x18, 41x36x33 (c = 41 direct, b = 36 passes), BCC 17x16x13,
# hexagonal 31x26x22 and 16x13x11
GRIDS = [("simple_cubic", 9), ("simple_cubic", 16), ("simple_cubic", 17), ("simple_cubic", 18), ("simple_cubic", 26),
         ("simple_cubic", 34), ("face_centered_cubic", 22), ("face_centered_cubic", 41), ("body_centered_cubic", 17),
         ("hexagonal", 31), ("hexagonal", 16)]


def _rand(n, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal(n) + 1j * rng.standard_normal(n)


def _rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


def _setup(lt, nx):
    lo = F.build_lattice(lt, nx, **({"c": 1.2} if lt == "hexagonal" else {}))
    fl = F.to_fame_lattice(lo)
    return fl, F.material_eps(lo, SPHERE, [13.0], 1.0)


def _accepted(S, prec, tiles):
    try:
        S.set_tiles(prec, tiles)
        return True
    except F.FameError:
        return False


@pytest.mark.parametrize("lt,nx", GRIDS, ids=lambda v: str(v))
@pytest.mark.parametrize("k", [(0.21, -0.13, 0.07), (0.0, 0.0, 0.0)], ids=["k", "gamma"])
def test_plane_qbq_vs_oracle(gpu, lt, nx, k):
    import torch
    fl, eps = _setup(lt, nx)
    T = O.Tables(O.lattice_from(fl), np.array(k))
    S = F.Solver(fl, max_batch=1)
    S.set_eps(eps)
    S.set_wave_vectors(np.array(k))
    x = _rand(2 * T.Nd, 3)
    ref = T.qbq(1.0 / eps, x)
    xd = torch.from_numpy(x).to("cuda")
    seen = 0
    for prec, op, bar in ((8, F.OP_QBQ, 1e-11), (4, F.OP_QBQ32, 2e-6)):
        for eng in (0, 1):
            for le, lc, nt in ((2, 4, 256), (4, 2, 512), (6, 8, 1024), (8, 12, 256), (16, 16, 512), (32, 24, 256)):
                t = {"inner": (eng, le), "mid": (2, lc), "outer": (2, nt)}
                if not _accepted(S, prec, t):
                    continue
                seen += 1
                y = S.apply(op, 0, xd).cpu().numpy()
                assert _rel(y, ref) < bar, (prec, t, _rel(y, ref))
                t["outer"] = (3, nt)        # FP64: 16 elements per thread, compound radices
                assert _accepted(S, prec, t) == (prec == 8 and nt <= 512)
                if prec == 8 and nt <= 512:
                    y = S.apply(op, 0, xd).cpu().numpy()
                    assert _rel(y, ref) < bar, (prec, t, _rel(y, ref))
        # the axis passes on the same grid
        if _accepted(S, prec, {"inner": (0, 4), "mid": (0, 8), "outer": (0, 8)}):
            assert _rel(S.apply(op, 0, xd).cpu().numpy(), ref) < bar
    assert seen >= 6
    S.close()


@pytest.mark.parametrize("lt,nx", [("simple_cubic", 17), ("face_centered_cubic", 22), ("body_centered_cubic", 16)])
def test_plane_eigs_vs_axis_passes(gpu, lt, nx):
    fl, eps = _setup(lt, nx)
    ks = np.array([[0.21, -0.13, 0.07], [0.05, 0.31, -0.22], [0.4, 0.1, 0.2]])
    S = F.Solver(fl, max_batch=3)
    S.set_eps(eps)
    S.set_wave_vectors(ks)
    lam = {}
    for plane in (False, True):
        for prec in (8, 4):
            t = {"inner": (1 if nx == 17 else 0, 4), "mid": (2, 8), "outer": (2, 256)} if plane else {"inner": (1, 4), "mid": (1, 16), "outer": (1, 16)}
            S.set_tiles(prec, t)
        for precision in (F.PREC_F64, F.PREC_F32_REFINE):
            f, _, _, prof = S.eigs(5, 18, precision=precision)
            assert all(p["converged"] for p in prof)
            lam[plane, precision] = f ** 2
    for key, v in lam.items():
        assert np.max(np.abs(v - lam[False, F.PREC_F64]) / lam[False, F.PREC_F64]) < 1e-8, key
    S.close()


def test_plane_tiles_are_refused_where_unavailable(gpu):
    fl, eps = _setup("simple_cubic", 18)
    S = F.Solver(fl, max_batch=1)
    S.set_eps(eps)
    for prec, t in ((4, {"inner": (0, 3), "mid": (2, 8), "outer": (2, 256)}),      # FP32 moves pairs of lines
                    (8, {"inner": (0, 64), "mid": (2, 8), "outer": (2, 256)}),
                    (8, {"inner": (0, 4), "mid": (2, 8), "outer": (2, 300)}),
                    (8, {"inner": (0, 4), "mid": (2, 8), "outer": (3, 1024)}),
                    (4, {"inner": (0, 4), "mid": (2, 8), "outer": (3, 256)}),
                    (8, {"inner": (2, 4), "mid": (2, 8), "outer": (2, 256)})):
        with pytest.raises(F.FameError):
            S.set_tiles(prec, t)
    S.close()


@pytest.mark.parametrize("lt,nx", GRIDS + [("face_centered_cubic", 96)], ids=lambda v: str(v))
def test_one_way_planes_vs_oracle(gpu, lt, nx):
    """Qr, Qrs, restored fields, residuals and the gradient, a generic wave vector and
    Gamma in one batch: per problem strides, the reference's layouts, and a
    permittivity that differs from cell to cell and component to component (its three
    layouts).  1e-11 of the oracle; residuals and gradients are sums of such terms."""
    import torch
    fl, _ = _setup(lt, nx)
    ks = np.array([[0.21, -0.13, 0.07], [0.0, 0.0, 0.0]])
    Ts = [O.Tables(O.lattice_from(fl), k) for k in ks]
    S = F.Solver(fl, max_batch=2)
    N, nw = S.N, 3
    rng = np.random.default_rng(5)
    eps = 1.0 + 12.0 * rng.random(3 * N)
    S.set_eps(eps)
    S.set_wave_vectors(ks)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda")
    v = _rand(3 * N, 11)
    evr = np.zeros((2, nw, 2 * N), complex)
    freq = np.array([[0.3, 0.7, 1.1], [0.4, 0.5, 0.9]])
    for i, T in enumerate(Ts):
        x = _rand(2 * T.Nd, 7 + i)
        assert _rel(S.apply(F.OP_QR, i, dev(x)).cpu().numpy(), T.qr(x)) < 1e-11
        assert _rel(S.apply(F.OP_QRS, i, dev(v)).cpu().numpy(), T.qrs(v)) < 1e-11
        if (lt, nx) in GRIDS:       # the largest element's error of any QBQ, axis passes too, is 1.7e-11 at FCC 96
            ref = T.qbq(1.0 / eps, x)
            for op, bar in ((F.OP_QBQ, 1e-11), (F.OP_QBQ32, 2e-6)):
                assert _rel(S.apply(op, i, dev(x)).cpu().numpy(), ref) < bar
        for j in range(nw):
            evr[i, j, :2 * T.Nd] = _rand(2 * T.Nd, 20 + 3 * i + j)
    E = S.restore(dev(evr))
    res = S.residuals(freq, E)
    Eh = E.cpu().numpy()
    g, w = np.zeros(3 * N), np.array([[1.0, 0.0, -0.5], [0.25, 2.0, 0.75]])
    for i, T in enumerate(Ts):
        sig = np.tile(T.get(3), 2)
        for j in range(nw):
            if i == 1 and j < 2:        # Gamma: two constant fields, then the bands
                e = np.full(3 * N, 1.0 / np.sqrt(3 * N))
            else:
                e = T.qr(sig * evr[i, j - 2 * i, :2 * T.Nd]) / eps
                e = e * np.linalg.norm(e)
            assert _rel(Eh[i, j], e) < 1e-11
            r = T.curlh(T.curl(Eh[i, j])) - freq[i, j] ** 2 * eps * Eh[i, j]
            r = np.linalg.norm(r) / np.linalg.norm(Eh[i, j])
            assert abs(res[i, j] - r) <= 1e-11 * r
            a = np.abs(Eh[i, j]) ** 2
            g -= w[i, j] * freq[i, j] ** 2 / (eps @ a) * a
    assert _rel(S.eig_vjp(freq, E, w).cpu().numpy(), g) < 1e-11
    S.close()


@pytest.mark.parametrize("prec", [8, 4])
def test_cg_scalars_in_the_inner_kernels(gpu, prec):
    """alpha and beta formed inside the inner kernels (up to 2048 blocks: 8 lines each
    here) against the separate reduction kernels (2304 blocks of 4 lines): the sums
    differ in order only, so the solutions of the 1e-12 solve agree to its accuracy."""
    import torch
    fl, eps = _setup("simple_cubic", 96)
    S = F.Solver(fl, max_batch=1)
    S.set_eps(eps)
    S.set_wave_vectors(np.array([[0.21, -0.13, 0.07]]))
    x = torch.from_numpy(_rand(2 * S.nd[0], 5)).to("cuda")
    y = []
    for lines in (4, 8):
        S.set_tiles(prec, {"inner": (0, lines), "mid": (2, lines), "outer": (2, 512)})
        y.append(S.apply(F.OP_INVAR if prec == 8 else F.OP_INVAR_MIXED, 0, x).cpu().numpy())
    assert np.linalg.norm(y[0] - y[1]) < 1e-10 * np.linalg.norm(y[1])
    S.close()
