"""Estimators, reweighting factors, sums, histograms and structure factors called
by several threads, each with systems of its own: every call has the memory
its results are written to for itself."""
import threading

import numpy as np
import pytest

import pyxmd
from orc import dptr
from test_gpu_recursion_paths import bridges

pytestmark = pytest.mark.gpu


def test_threads_with_systems_of_their_own():
    lib = pyxmd.Lib()
    jobs = []
    for i, (N, P, points) in enumerate([(5, 8, 2000), (70, 16, 40), (130, 8, 500), (33, 32, 5000)]):
        x = bridges(N, P, 1.0, 12, np.random.default_rng(i))
        s = pyxmd.System(lib, "trap", N, P, 1.0, 1.0, seed=1 + 2 * i, positions=x.reshape(N * P, 3))
        s.full_force()
        grid, fac, st = np.linspace(0.0, 1.0, 3 + 5 * i), np.zeros(3 + 5 * i), lib.md_alloc_stats_x(points)
        fx = np.ctypeslib.as_array(st.contents.fxs[0], shape=(points,))
        es = st.contents.es

        def job(s=s, grid=grid, fac=fac, st=st, fx=fx, es=es):
            out = []
            for call in (lib.md_pimd_calc_VBN_energy_x, lib.md_pimd_calc_virial_energy_x):
                es[0] = 0.0
                assert call(s.pimd, st) == 0
                out.append(es[0])
            es[0] = 0.0
            assert lib.md_calc_kinetic_x(s.sim, st) == 0
            out.append(es[0])
            assert lib.md_pimd_calc_vi_sign_grid_x(s.pimd, len(grid), dptr(grid), dptr(fac)) == 0
            fx[:] = 0.0
            assert lib.md_pimd_calc_density_distribution_x(s.pimd, st, 5.0, 0, dptr(np.zeros(3))) == 0
            out += [fac.copy(), fx.copy()]
            fx[:] = 0.0
            assert lib.md_pimd_calc_Sk_structure_x(s.pimd, st, 0.0, 0.1, 1) == 0
            return out + [fx.copy()]

        jobs.append(job)
    want = [job() for job in jobs]
    failed = []

    def run(i):
        for k in range(30):
            try:
                for a, b in zip(jobs[i](), want[i]):
                    np.testing.assert_array_equal(a, b)
            except AssertionError as e:
                failed.append((i, k, str(e)))
                return

    threads = [threading.Thread(target=run, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
