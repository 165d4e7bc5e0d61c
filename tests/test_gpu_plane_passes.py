"""The Stockham passes of the plane kernels at operator level, which grids of axes up
to 24 points (direct DFTs) and prime axes do not reach: composite axes above 24 in
two and three passes with radices 2 to 16, every thread count, both FP64 variants,
one round of a pass and several (256 threads, or FCC 96, whose 83 columns take more
than one), the fused middle pass among them.  The error is measured in norm against
the FP64 oracle: a chain of some 40 roundings of random sign, amplified by the few
near-singular modes of the Pi basis, stays below 1e-12 in FP64 and 1e-6 in FP32."""
import os

import numpy as np
import pytest

import fame_amd as F
import oracle as O
from cases import SPHERE

pytestmark = pytest.mark.gpu

O.set_threads(8)


def _rand(n, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal(n) + 1j * rng.standard_normal(n)


def _norm_err(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


# 32 = 16 x 2 (8 x 4), 36 = 12 x 3 (4 x 3 x 3), 48 = 16 x 3 (8 x 3 x 2), 60 = 15 x 4 (5 x 4 x 3),
# 65 = 13 x 5, 77 = 11 x 7; FCC 55 is 55x48x45 (11 x 5, 16 x 3, 15 x 3), FCC 96 is 96x83x78
@pytest.mark.parametrize("lt,nx", [("simple_cubic", 32), ("simple_cubic", 36), ("simple_cubic", 48), ("simple_cubic", 60),
                                   ("simple_cubic", 65), ("simple_cubic", 77), ("face_centered_cubic", 55),
                                   ("face_centered_cubic", 96)], ids=lambda v: str(v))
def test_composite_axes_vs_oracle(gpu, lt, nx):
    import torch
    lo = F.build_lattice(lt, nx)
    fl = F.to_fame_lattice(lo)
    eps = F.material_eps(lo, SPHERE, [13.0], 1.0)
    ks = np.array([[0.21, -0.13, 0.07], [0.0, 0.0, 0.0]])
    S = F.Solver(fl, max_batch=2)
    S.set_eps(eps)
    S.set_wave_vectors(ks)
    for ik in range(2 if nx < 60 else 1):
        T = O.Tables(O.lattice_from(fl), ks[ik])
        x = _rand(2 * T.Nd, 3 + ik)
        ref = T.qbq(1.0 / eps, x)
        xd = torch.from_numpy(x).to("cuda")
        seen = set()
        for prec, op, bar in ((8, F.OP_QBQ, 1e-12), (4, F.OP_QBQ32, 1e-6)):
            for wide, nt in ((2, 256), (2, 512), (2, 1024), (3, 256), (3, 512)):
                try:
                    S.set_tiles(prec, {"inner": (0, 4), "mid": (2, 4), "outer": (wide, nt)})
                except F.FameError:
                    continue
                seen.add((prec, wide, nt))
                err = _norm_err(S.apply(op, ik, xd).cpu().numpy(), ref)
                assert err < bar, (ik, prec, wide, nt, err)
        assert len(seen) == 8, seen       # FP64: five, FP32: three
    S.close()


@pytest.mark.parametrize("lt,nx", [("simple_cubic", 36), ("simple_cubic", 64), ("simple_cubic", 75), ("face_centered_cubic", 55),
                                   ("body_centered_cubic", 64), ("hexagonal", 72)], ids=lambda v: str(v))
def test_one_way_passes_vs_oracle(gpu, lt, nx):
    """Qr, Qrs and the residuals through the one-way plane kernels, narrow and wide."""
    import torch
    fl = F.to_fame_lattice(F.build_lattice(lt, nx, **({"c": 1.2} if lt == "hexagonal" else {})))
    S = F.Solver(fl, max_batch=1)
    eps = 1.0 + 12.0 * np.random.default_rng(5).random(3 * S.N)
    S.set_eps(eps)
    S.set_wave_vectors(np.array([[0.21, -0.13, 0.07]]))
    T = O.Tables(O.lattice_from(fl), S.k[0])
    x, v = _rand(2 * S.N, 7), _rand(3 * S.N, 11)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda")
    assert _norm_err(S.apply(F.OP_QR, 0, dev(x)).cpu().numpy(), T.qr(x)) < 1e-12
    assert _norm_err(S.apply(F.OP_QRS, 0, dev(v)).cpu().numpy(), T.qrs(v)) < 1e-12
    res = S.residuals(np.array([[0.7]]), dev(v[None, None]))
    r = T.curlh(T.curl(v)) - 0.49 * eps * v
    assert abs(res[0, 0] - np.linalg.norm(r) / np.linalg.norm(v)) <= 1e-12 * res[0, 0]
    S.close()


@pytest.mark.parametrize("op", [F.OP_INVAR, F.OP_INVAR_MIXED])
def test_long_graphs_repeat_the_short_ones(gpu, op):
    """A solve that has come back often runs graphs of 16 iterations among those of 4:
    the same kernels, so every solve, with eager work and synchronisation in between,
    repeats the first one bit for bit, and that of a context without graphs."""
    import torch
    lo = F.build_lattice("simple_cubic", 26)
    fl = F.to_fame_lattice(lo)
    eps = F.material_eps(lo, SPHERE, [13.0], 1.0)
    y = {}
    for graphs in ("1", "0"):
        saved = os.environ.get("FAME_GRAPH")
        os.environ["FAME_GRAPH"] = graphs
        try:
            S = F.Solver(fl, max_batch=1)
        finally:
            if saved is None:
                del os.environ["FAME_GRAPH"]
            else:
                os.environ["FAME_GRAPH"] = saved
        S.set_eps(eps)
        S.set_wave_vectors(np.array([[0.21, -0.13, 0.07]]))
        xd = torch.from_numpy(_rand(2 * S.nd[0], 9)).to("cuda")
        y[graphs] = S.apply(op, 0, xd)
        for i in range(40 if graphs == "1" else 2):
            S.apply(F.OP_QBQ, 0, xd)
            assert torch.equal(S.apply(op, 0, xd), y[graphs]), i
        S.close()
    assert torch.equal(y["1"], y["0"])
