"""The energy estimators' weighted recursion across its 64-row blocks and
64-column chunks against the recursion in extended precision on the same
cycle energies and potentials.  Bar: 1e-12, the estimators' bar in the parity
tests, of the estimator's own terms (the recursion's result and the kinetic
constant it is added to, which may nearly cancel)."""
import numpy as np
import pytest

import pyxmd
from test_gpu_recursion_paths import bridges

pytestmark = pytest.mark.gpu

CASES = [(1, 3, 1.0), (2, 8, 0.5), (63, 8, 1.0), (64, 4, 0.0), (65, 16, 1.0), (128, 8, 1.0), (257, 24, 0.25),
         (600, 16, 1.0)]


def recursion(E, B, V, beta, xi, N):
    ld = np.longdouble
    res = np.zeros(N + 1, ld)
    for n in range(1, N + 1):
        k = np.arange(1, n + 1) if xi != 0 else np.array([1])
        x = -ld(beta) * (E[n][k - 1].astype(ld) + V[n - k].astype(ld) - V[n])
        if xi != 0:
            x = x + (k - 1) * np.log(ld(xi))
        w = np.exp((x - x.max()).astype(float)).astype(ld)
        res[n] = (w * (res[n - k] - B[n][k - 1])).sum() / w.sum()
    return float(res[N])


@pytest.mark.parametrize("N,P,xi", CASES)
def test_estimator_blocks(N, P, xi):
    lib = pyxmd.Lib()
    rng = np.random.default_rng([3, N, P])
    s = pyxmd.System(lib, "trap", N, P, 1.0, xi, seed=1, positions=bridges(N, P, 1.0, 12, rng).reshape(N * P, 3))
    if N * P % 2:  # an odd number of draws leaves a spare, which the next seed does not clear
        lib.md_random_gaussian_x()
    s.full_force()
    assert lib.md_pimd_fast_fill_ENk2_x(s.pimd, 0) == 0
    got = s.stat(lib.md_pimd_calc_VBN_energy_x, s.pimd)
    s.host_pimd()
    rows = lambda t: [None] + [t[(n - 1) * n // 2:n * (n + 1) // 2] for n in range(1, N + 1)]
    E, V = rows(pyxmd.tri(s.pimd)), pyxmd.vbn(s.pimd)
    r = recursion(E, E, V, s.beta, xi, N)
    kin = 3 * N * P / (2 * s.beta)
    print(f"N={N} P={P} xi={xi}: V_B energy {got:.12e}, recursion {r + kin:.12e}", flush=True)
    assert abs(got - (r + kin)) <= 1e-12 * (abs(r) + kin)
    st = lib.md_alloc_stats_x(1)
    assert lib.md_pimd_calc_vi_virial_energy_x(s.pimd, st, 0) == 0
    b = s.host_beads()
    x, f = b["x"].reshape(N, P, 3), b["f"].reshape(N, P, 3)
    vir = -0.5 * ((x[:, 1:] - x[:, :1]) * f[:, 1:]).sum()
    r2 = recursion(E, rows(pyxmd.tri(s.pimd, "ENk2")), V, s.beta, xi, N)
    want = r2 + 3 * N / (2 * s.beta) + vir
    scale = abs(r2) + 3 * N / (2 * s.beta) + 0.5 * np.abs((x[:, 1:] - x[:, :1]) * f[:, 1:]).sum()
    assert abs(st.contents.es[0] - want) <= 1e-12 * scale
