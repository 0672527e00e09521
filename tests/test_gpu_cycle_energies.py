"""Cycle energies at the edges of their kernels' blocks: particle blocks of
16, chunks of 80 springs, 32 x 32 tiles of the energy table in both layouts.

Every energy is a sum of non-negative springs, at most N P of them, so any
order of summation stays within (N P + 8) 2^-53 of the exact value, the oracle's
too; the bar is twice that.  The column layout is read by the backward
recursion, whose potentials are held to the bar of the other recursion tests.
"""
import ctypes as C

import numpy as np
import pytest

import pyxmd
from orc import Oracle, beads_from, dptr, ptr, tri_size
from test_gpu_recursion_paths import bridges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P", [(1, 2), (2, 79), (15, 78), (16, 80), (17, 81), (31, 159), (32, 160), (33, 161),
                                 (64, 5), (65, 24), (255, 3), (257, 4)])
def test_cycle_energies(N, P):
    lib = pyxmd.Lib()
    x = bridges(N, P, 1.0, 12, np.random.default_rng([7, N, P]))
    s = pyxmd.System(lib, "trap", N, P, 1.0, 1.0, seed=1, positions=x.reshape(N * P, 3))
    if N * P % 2:  # an odd number of draws leaves a spare, which the next seed does not clear
        lib.md_random_gaussian_x()
    hb = s.host_beads()
    o = Oracle()
    b = beads_from(hb["x"].reshape(-1), m=hb["m"])
    E, Ei, V, Vt = np.zeros(tri_size(N)), np.zeros(N), np.zeros(N + 1), np.zeros(N + 1)
    L = np.array([10.0] * 3)
    o.fast_fill_ENk(N, P, s.omegaP, 0, dptr(L), ptr(b), dptr(E), dptr(Ei))
    o.fill_VB(N, s.beta, 1.0, dptr(E), dptr(V))
    b["f"] = 0
    o.fast_force_VB(N, P, s.beta, 1.0, s.omegaP, 0, dptr(L), dptr(E), dptr(V), ptr(b), dptr(Vt), None)
    cfg = pyxmd.StepConfig(None, None, 0.01, 0, 0, 0)
    for fused in (False, True):
        print(f"N={N} P={P} fused={fused}", flush=True)
        if fused:
            assert lib.md_pimd_compute_forces_x(s.pimd, C.byref(cfg)) == 0
        else:
            assert lib.md_pimd_fast_fill_ENk_x(s.pimd, 0) == 0
            assert lib.md_pimd_fill_VB_x(s.pimd) == 0
            assert lib.md_pimd_fast_fill_force_VB_x(s.pimd, 0) == 0
        assert lib.md_hip_synchronize_x() == 0
        s.host_pimd()
        np.testing.assert_allclose(pyxmd.tri(s.pimd), E, rtol=2 * (N * P + 8) * 2.0 ** -53, atol=0)
        vt = np.zeros(N + 1)
        assert lib.md_pimd_get_backward_potentials_x(s.pimd, dptr(vt)) == 0
        np.testing.assert_allclose(pyxmd.vbn(s.pimd), V, rtol=1e-12, atol=1e-12)
        np.testing.assert_allclose(vt, Vt, rtol=1e-12, atol=1e-12)
