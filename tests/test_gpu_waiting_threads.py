"""A solve that waits for the GPU gives its core to threads that have work: many
structures solved from one call take about as long on 2 CPUs as on all (2.1 times
as long if every waiting thread kept its core, 1.15 as it is)."""
import os
import time

import numpy as np
import pytest

import fame_amd as F

pytestmark = pytest.mark.gpu


def test_many_structures_on_two_cpus(gpu):
    cpus = os.sched_getaffinity(0)
    if len(cpus) < 8:
        pytest.skip("needs 8 CPUs to compare with")
    rng = np.random.default_rng(1)
    Ss = []
    for i in range(16):
        S = F.Solver(F.to_fame_lattice(F.build_lattice("simple_cubic", 16 + 2 * (i % 4))), max_batch=1)
        S.set_eps(1.0 + 11.0 * rng.random(3 * S.N))
        S.set_wave_vectors(rng.uniform(0.08, 0.42, (1, 3)))
        Ss.append(S)

    def best(n):
        t = []
        for _ in range(n):
            a = time.perf_counter()
            F.eigs_many(Ss, 6, 18)
            t.append(time.perf_counter() - a)
        return min(t)
    best(2)
    free = best(4)
    try:
        os.sched_setaffinity(0, set(sorted(cpus)[:2]))      # the solving threads inherit it
        two = best(4)
    finally:
        os.sched_setaffinity(0, cpus)
    for S in Ss:
        S.close()
    assert two < 1.6 * free, (two, free)
