"""The energy estimators' recursion with potentials V_B that are not the ones
of the current xi: filled at another xi, or supplied by the host.  A row's
weights are ratios, so it holds for any potential; every term of a row may
then lie far from exp(0) (64 beads: about 96 for each ring closed).

Tolerance: the first-order error bound carried through the reference recursion
itself.  A weight's exponent is computed with error 2^-53 (8 + 4 |its parts|),
which moves a row's average by at most that times the distance of the weighted
value from the average, and the sums of a row add 2^-53 * 128 of their
absolute terms."""
import numpy as np
import pytest

import pyxmd
from test_gpu_recursion_paths import bridges

pytestmark = pytest.mark.gpu


def recursion(E, V, beta, xi, N):
    """res(N) and its error bound; V_B enters row n through its differences."""
    ld, u = np.longdouble, 2.0 ** -53
    res, err = np.zeros(N + 1, ld), np.zeros(N + 1)
    for n in range(1, N + 1):
        k = np.arange(1, n + 1) if xi != 0 else np.array([1])
        c = -ld(beta) * E[n][k - 1].astype(ld) - np.log(ld(n))
        if xi != 0:
            c = c + (k - 1) * np.log(ld(xi))
        L = -ld(beta) * V[n - k].astype(ld)
        x = c + L
        p = np.exp((x - x.max()).astype(float))
        p /= p.sum()
        v = (res[n - k] - E[n][k - 1]).astype(float)
        res[n] = (p.astype(ld) * (res[n - k] - E[n][k - 1])).sum()
        scale = u * (8 + 4 * (np.abs(c) + np.abs(L) + abs(beta * V[n])).astype(float))
        err[n] = (p * (scale * np.abs(v - float(res[n])) + err[n - k] + 128 * u * np.abs(v))).sum()
    return float(res[N]), err[N]


def rows(t, N):
    return [None] + [t[(n - 1) * n // 2:n * (n + 1) // 2] for n in range(1, N + 1)]


@pytest.mark.parametrize("how", ["xi", 100.0, 500.0, 3000.0])
@pytest.mark.parametrize("N,P", [(1, 64), (5, 64), (64, 16), (65, 64), (150, 64)])
def test_potentials_of_another_state(N, P, how):
    lib = pyxmd.Lib()
    rng = np.random.default_rng([11, N, P])
    s = pyxmd.System(lib, "trap", N, P, 1.0, 1.0, seed=1, positions=bridges(N, P, 1.0, 12, rng).reshape(N * P, 3))
    if N * P % 2:  # an odd number of draws leaves a spare, which the next seed does not clear
        lib.md_random_gaussian_x()
    assert lib.md_pimd_fast_fill_ENk_x(s.pimd, 0) == 0
    assert lib.md_pimd_fill_VB_x(s.pimd) == 0
    xi = 1.0
    if how == "xi":
        xi = s.pimd.contents.vi = 0.0
    else:
        assert lib.md_pimd_sync_host_x(s.pimd, 0)  # the host's potentials count from here on
        V = np.ctypeslib.as_array(s.pimd.contents.VBN, shape=(N + 1,))
        V[1:] += rng.uniform(-how, how, N) / s.beta
    print(f"N={N} P={P} {how}", flush=True)
    got = s.stat(lib.md_pimd_calc_VBN_energy_x, s.pimd)
    s.host_pimd()
    r, err = recursion(rows(pyxmd.tri(s.pimd), N), pyxmd.vbn(s.pimd), s.beta, xi, N)
    kin = 3 * N * P / (2 * s.beta)
    print(f"  V_B energy {got:.12e}, recursion {r + kin:.12e}, bound {err:.1e}", flush=True)
    assert abs(got - (r + kin)) <= err + 2.0 ** -51 * (abs(r) + kin)
