"""The exchange recursion on thermal states with permutation cycles.

Particles that are part of longer cycles lie far above the chain of
single-particle cycles, so the block solve's frame must follow the best
paths; a cycle that runs through whole blocks leaves even that frame's range
and takes the exact path.  Beads are Brownian bridges over cycles of
consecutive particles (geometric lengths, or one cycle of all particles), at
block sizes around the 64-row edges.  Bars as in the multi-block parity
test: V_B and the backward potentials 1e-12, exchange forces 1e-11 of the RMS
force or four times the reference fast path's own distance from the 80-bit
truth.
"""
import ctypes as C

import numpy as np
import pytest

import pyxmd
from orc import Oracle, beads_from, dptr, exchange_truth, ptr, rel_err, tri_size

pytestmark = pytest.mark.gpu

CASES = [(1, 4, 1.0, 3), (63, 32, 1.0, 12), (64, 32, 0.25, 12), (65, 64, 1.0, 12), (129, 32, 1.0, 40),
         (200, 16, 0.5, 200), (193, 72, 1.0, 193), (130, 8, 0.0, 1)]


def bridges(N, P, T, longest, rng):
    x = np.empty((N, P, 3))
    n = 0
    while n < N:
        k = min(N - n, longest if longest >= 40 else int(rng.geometric(0.5)), longest)
        w = rng.normal(size=(k * P, 3)) / np.sqrt(T * P)
        path = np.cumsum(w, 0) - np.arange(1, k * P + 1)[:, None] / (k * P) * w.sum(0)
        x[n:n + k] = (path + rng.normal(size=3) * 1.5).reshape(k, P, 3)
        n += k
    return x


@pytest.mark.parametrize("N,P,xi,longest", CASES)
def test_thermal_cycles(N, P, xi, longest):
    lib = pyxmd.Lib()
    T = 1.0
    x = bridges(N, P, T, longest, np.random.default_rng([N, P]))
    s = pyxmd.System(lib, "trap", N, P, T, xi, seed=1, positions=x.reshape(N * P, 3))
    L = np.array([10.0] * 3)
    hb = s.host_beads()
    o = Oracle()
    b = beads_from(hb["x"].reshape(-1), m=hb["m"])
    E, Ei, V, Vt = np.zeros(tri_size(N)), np.zeros(N), np.zeros(N + 1), np.zeros(N + 1)
    o.fast_fill_ENk(N, P, s.omegaP, 0, dptr(L), ptr(b), dptr(E), dptr(Ei))
    o.fill_VB(N, s.beta, xi, dptr(E), dptr(V))
    b["f"] = 0
    o.fast_force_VB(N, P, s.beta, xi, s.omegaP, 0, dptr(L), dptr(E), dptr(V), ptr(b), dptr(Vt), None)
    ft, _ = exchange_truth(o, hb["x"].reshape(-1), hb["m"], N, P, s.beta, xi, s.omegaP, 0, L[0])
    ref = rel_err(b["f"].reshape(-1), ft)
    # the per-stage calls and the fused step's recursion (coefficients from the tables / from positions)
    cfg = pyxmd.StepConfig(None, None, 0.01, 0, 0, 0)
    for fused in (False, True):
        print(f"N={N} P={P} xi={xi} cycles up to {longest} fused={fused}", flush=True)
        if fused:
            assert lib.md_pimd_compute_forces_x(s.pimd, C.byref(cfg)) == 0
        else:
            assert lib.md_reset_force_x(s.sim) == 0
            assert lib.md_pimd_fast_fill_ENk_x(s.pimd, 0) == 0
            assert lib.md_pimd_fill_VB_x(s.pimd) == 0
            assert lib.md_pimd_fast_fill_force_VB_x(s.pimd, 0) == 0
        assert lib.md_hip_synchronize_x() == 0
        s.host_pimd()
        vbn, vt = pyxmd.vbn(s.pimd), np.zeros(N + 1)
        assert lib.md_pimd_get_backward_potentials_x(s.pimd, dptr(vt)) == 0
        np.testing.assert_allclose(vbn, V, rtol=1e-12, atol=1e-12)
        np.testing.assert_allclose(vt, Vt, rtol=1e-12, atol=1e-12)
        err = rel_err(s.host_beads()["f"].reshape(-1), ft)
        print(f"  exchange force vs 80-bit truth: engine {err:.2e}, reference fast path {ref:.2e}", flush=True)
        assert err < max(1e-11, 4 * ref)
