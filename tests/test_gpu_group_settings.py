"""The concurrent groups of a batch.  They run with the settings their context was
created with: FAME_FFT at the time of a later solve changes neither their plans nor their
tables.  FCC 20 is 20x17x16, whose 17-point axis has no plane path under
FAME_FFT=stockham, so children built under another setting than the parent's lack
what the parent's tiles name.  And they repeat one batch bit for bit also where a
rule depends on how many problems there are."""
import os

import numpy as np
import pytest

import fame_amd as F
from cases import SPHERE

pytestmark = pytest.mark.gpu


class _Env:
    def __init__(self, fft):
        self.fft = fft

    def _set(self, v):
        if v is None:
            os.environ.pop("FAME_FFT", None)
        else:
            os.environ["FAME_FFT"] = v

    def __enter__(self):
        self.old = os.environ.get("FAME_FFT")
        self._set(self.fft)

    def __exit__(self, *exc):
        self._set(self.old)


@pytest.mark.parametrize("at_create,at_solve", [(None, "stockham"), ("stockham", None), ("mfma", "stockham")])
def test_groups_keep_their_contexts_settings(gpu, at_create, at_solve):
    import torch
    lo = F.build_lattice("face_centered_cubic", 20)
    fl = F.to_fame_lattice(lo)
    assert list(fl.grid_nums) == [20, 17, 16]
    ks = np.array([[0.21, -0.13, 0.07], [0.05, 0.31, -0.22], [0.0, 0.0, 0.0]])
    with _Env(at_create):
        S = F.Solver(fl, max_batch=3)
    S.set_eps(F.material_eps(lo, SPHERE, [13.0], 1.0))
    S.set_wave_vectors(ks)
    with _Env(at_solve):
        for prec in (F.PREC_F64, F.PREC_F32_REFINE):
            out = []
            for groups in (1, 2):
                S.set_groups(groups)
                f, _, E, prof = S.eigs(5, 16, precision=prec, want_fields=True)
                out.append((f, E.cpu(), [p["ls_iter"] for p in prof]))
            # a problem's arithmetic does not depend on the group it runs in
            assert np.array_equal(out[0][0], out[1][0])
            assert torch.equal(out[0][1], out[1][1])
            assert out[0][2] == out[1][2]
    S.close()


@pytest.mark.parametrize("n,nk", [((48, 48, 48), 6), ((400, 4, 4), 12)])
def test_groups_repeat_one_batch(gpu, n, nk):
    """48^3: six problems' one-way planes run in blocks of 256 threads, three alone would
    take 512, which sum |E|^2 in another order; 400 x 4 x 4: twelve problems restore
    their fields by axis passes, six alone would by planes."""
    import torch
    fl = F.to_fame_lattice(F.build_lattice("simple_cubic", 16))
    for i in range(3):
        fl.mesh_len[i] *= fl.grid_nums[i] / n[i]
        fl.grid_nums[i] = n[i]
    rng = np.random.default_rng(4)
    S = F.Solver(fl, max_batch=nk)
    S.set_eps(1.0 + 11.0 * rng.random(3 * S.N))
    S.set_wave_vectors(rng.uniform(0.08, 0.42, (nk, 3)))
    out = []
    for groups in (1, 2):
        S.set_groups(groups)
        f, _, E, _ = S.eigs(3, 9, maxit=2, want_fields=True)
        out.append((f, E))
    assert np.array_equal(out[0][0], out[1][0])
    assert torch.equal(out[0][1], out[1][1])
    S.close()
