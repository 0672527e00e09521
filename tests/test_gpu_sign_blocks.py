"""Sign-tracked recursion (md_pimd_calc_vi_sign_grid_x) across its 64-row
blocks, both signs of xi', against the same recursion in extended precision.

The alternating sums of xi' < 0 cancel, which amplifies rounding, so the
tolerance is the first-order error bound carried through the reference
recursion itself: every term exp(x) enters with relative error
2^-53 (8 + 4 max |x|'s parts), and a row's error is its terms' errors over its
(possibly cancelled) sum.  States whose bound exceeds 1e-3 are not compared.
"""
import numpy as np
import pytest

import pyxmd
from orc import dptr
from test_gpu_recursion_paths import bridges

pytestmark = pytest.mark.gpu

GRID = np.array([-1.0, -0.5, -0.1, 0.0, 0.3, 0.75, 1.0])


def reference(E, beta, xi, N):
    """(sign, L'(N), error bound of L'(N)): E[n][k-1] rows of the cycle-energy triangle."""
    ld = np.longdouble
    L, sg, err = np.zeros(N + 1, ld), np.ones(N + 1), np.zeros(N + 1)
    u = 2.0 ** -53
    for n in range(1, N + 1):
        k = np.arange(1, n + 1) if xi != 0 else np.array([1])
        c = -ld(beta) * E[n][k - 1].astype(ld) - np.log(ld(n))
        if xi != 0:
            c = c + (k - 1) * np.log(ld(abs(xi)))
        x = c + L[n - k]
        top = x.max()
        w = np.exp((x - top).astype(float)) * sg[n - k] * np.where((k - 1) % 2 == 1, np.sign(xi), 1.0)
        s = w.sum()
        scale = u * (8 + 4 * (np.abs(c) + np.abs(L[n - k])).astype(float))
        err[n] = (np.abs(w) * (scale + err[n - k])).sum() / abs(s)
        L[n] = top + np.log(ld(abs(s)))
        sg[n] = 1.0 if s >= 0 else -1.0
    return sg[N], L[N], err[N]


@pytest.mark.parametrize("N,P,xi", [(1, 4, 1.0), (5, 16, 1.0), (63, 4, 1.0), (64, 8, 0.5), (65, 16, 1.0),
                                    (130, 32, 1.0), (200, 12, 0.25), (257, 48, 0.0)])
def test_sign_grid_blocks(N, P, xi):
    lib = pyxmd.Lib()
    rng = np.random.default_rng([7, N, P])
    s = pyxmd.System(lib, "trap", N, P, 1.0, xi, seed=1, positions=bridges(N, P, 1.0, 12, rng).reshape(N * P, 3))
    assert lib.md_pimd_fast_fill_ENk_x(s.pimd, 0) == 0
    assert lib.md_pimd_fill_VB_x(s.pimd) == 0
    fac = np.zeros(len(GRID))
    assert lib.md_pimd_calc_vi_sign_grid_x(s.pimd, len(GRID), dptr(GRID), dptr(fac)) == 0
    s.host_pimd()
    tri, V = pyxmd.tri(s.pimd), pyxmd.vbn(s.pimd)
    E = [None] + [tri[(n - 1) * n // 2:n * (n + 1) // 2] for n in range(1, N + 1)]
    compared = 0
    for xi2, got in zip(GRID, fac):
        sg, Lr, err = reference(E, s.beta, xi2, N)
        err += 2.0 ** -53 * (8 + 4 * abs(s.beta * V[N]))
        if err > 1e-3:
            continue
        with np.errstate(over="ignore"):
            want = sg * np.exp(float(Lr + np.longdouble(s.beta) * np.longdouble(V[N])))
        print(f"N={N} P={P} xi'={xi2}: factor {got:.6e}, want {want:.6e}, bound {err:.1e}", flush=True)
        assert got == want or abs(got - want) <= err * abs(want) + 1e-300  # both may overflow to the same infinity
        compared += 1
    assert compared >= 4
