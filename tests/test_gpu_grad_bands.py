"""fame_eig_grad over its chunks of bands: more than the 16 bands of one launch, a
grid whose fields leave the cache fewer than 16 (SC 72: 11), few or no weighted
bands, zero frequencies, against the formula -sum w lambda |E|^2 / (E^H eps E) in
double precision.  Bar: the sums have at most 100 terms one after another and a
tree, the bands at most 33, so 1e-13 of the sum of the terms' magnitudes."""
import numpy as np
import pytest

import fame_amd as F

pytestmark = pytest.mark.gpu


def _fields(nk, nb, n3):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(nb)
    r = lambda: torch.randn((nk, nb, n3), dtype=torch.float64, device="cuda", generator=gen)
    return torch.complex(r(), r())


def _solver(nx, nk):
    rng = np.random.default_rng(nx)
    S = F.Solver(F.to_fame_lattice(F.build_lattice("simple_cubic", nx)), max_batch=nk)
    eps = 1.0 + 12.0 * rng.random(3 * S.N)
    S.set_eps(eps)
    S.set_wave_vectors(rng.uniform(0.1, 0.4, (nk, 3)))
    return S, eps, rng


@pytest.mark.parametrize("nx,nk,nb", [(10, 2, 16), (10, 2, 17), (12, 1, 33), (72, 1, 13)])
@pytest.mark.parametrize("kind", ["dense", "onehot", "sparse", "none", "last wave vector"])
def test_gradient_over_chunks_of_bands(gpu, nx, nk, nb, kind):
    import torch
    S, eps, rng = _solver(nx, nk)
    E = _fields(nk, nb, 3 * S.N)
    freq = np.tile(np.linspace(0.0, 1.5, nb), (nk, 1))      # the first band of frequency 0 has no share
    w = rng.standard_normal((nk, nb))
    if kind == "onehot":
        w *= np.arange(nb) == nb - 1
    elif kind == "sparse":
        w *= np.arange(nb) % 3 == 1
    elif kind == "none":
        w *= 0.0
    elif kind == "last wave vector":
        w[:-1] = 0.0
    got = S.eig_vjp(freq, E, w)
    e = torch.from_numpy(eps).to("cuda")
    ref, mag = torch.zeros_like(e), torch.zeros_like(e)
    for p in range(nk):
        for i in range(nb):
            a = E[p, i].real ** 2 + E[p, i].imag ** 2
            t = (w[p, i] * freq[p, i] ** 2 / (e * a).sum()) * a
            ref -= t
            mag += t.abs()
    assert bool((torch.abs(got - ref) <= 1e-13 * mag).all())
    S.close()


def test_bands_without_weight_are_not_read(gpu):
    """One weighted band of 16 costs well under the dense gradient: its two passes
    over one field against two over sixteen (0.12 of the time, and 0.75 where the
    norm of every band is taken)."""
    import time
    import torch
    S, _, _ = _solver(128, 1)
    E = _fields(1, 16, 3 * S.N)
    freq = np.linspace(0.3, 1.5, 16)[None]

    def best(w):
        t = []
        for _ in range(12):
            torch.cuda.synchronize()
            a = time.perf_counter()
            S.eig_vjp(freq, E, w)
            torch.cuda.synchronize()
            t.append(time.perf_counter() - a)
        return min(t)
    dense, one = best(np.ones((1, 16))), best(np.eye(16)[4][None])
    assert one < 0.4 * dense, (one, dense)
    S.close()
