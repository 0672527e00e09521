"""Gaussian pair forces at both sides of the lines between the tile kernels'
two ways of dividing (ranges of 2^-30 and 2^30, strengths g / (pi s^2) of
2^800) and at short ranges, against the two-species kernel, which evaluates
the term plainly: bit for bit where the force is a normal number, and within
the rounding of its last division to a subnormal one below.  Layout as in
test_gpu_gauss_tiles: the other terms of a bead underflow to zero."""
import math

import numpy as np
import pytest

import pyxmd
from test_gpu_gauss_tiles import forces, system

pytestmark = pytest.mark.gpu

CASES = [(2.0 ** e * f, 3.0) for e in (-30, 30) for f in (0.999, 1.001)] + [(0.05, 3.0), (0.1, 3.0)] + \
        [(0.5, f * math.pi * 0.25 * 2.0 ** 800) for f in (0.999, 1.001)]


@pytest.mark.parametrize("kind", ["trap", "pgauss"])
@pytest.mark.parametrize("s,g", CASES)
@pytest.mark.parametrize("pairs", [3, 40])
def test_lines(kind, s, g, pairs):
    lib = pyxmd.Lib()
    P = 8
    rng = np.random.default_rng([pairs, int(1e3 * abs(math.log(s)))])
    L = 200.0 * s * pairs
    r = rng.normal(size=(P, pairs, 3))
    r *= (s * rng.uniform(0, 29, size=(P, pairs)) / np.linalg.norm(r, axis=2))[..., None]
    r[:, ::5, 1] = 0.0
    a = np.zeros((P, pairs, 3))
    a[..., 0] = 200.0 * s * np.arange(pairs)
    a += s * rng.uniform(0, 10, size=(P, pairs, 3)) + (L / 4 if kind == "pgauss" else 0.0)
    b = a + r
    m = 2.0 ** rng.integers(-2, 3, pairs)
    seat = rng.permutation(2 * pairs)
    x, mm = np.empty((P, 2 * pairs, 3)), np.empty(2 * pairs)
    x[:, seat[:pairs]], x[:, seat[pairs:]] = a, b
    mm[seat[:pairs]] = mm[seat[pairs:]] = m
    print(f"{kind} pairs={pairs} s={s} g={g}", flush=True)
    one, sa, sb = system(lib, kind, x, mm, L), system(lib, kind, a, m, L), system(lib, kind, b, m, L)
    lib.md_set_guassian_force_range_x(s)
    lib.md_set_gaussian_force_strength_x(g)
    try:
        assert lib.md_pimd_calc_pair_force_x(one.pimd, one.pair_cb()) == 0
        assert lib.md_pimd_calc_pair_force_2_x(sa.pimd, sb.pimd, one.pair_cb()) == 0
        assert lib.md_hip_synchronize_x() == 0
        f, fa, fb = forces(one), forces(sa), forces(sb)
    finally:
        lib.md_set_guassian_force_range_x(0.5)
        lib.md_set_gaussian_force_strength_x(3.0)
    for got, want in ((f[:, seat[:pairs]], fa), (f[:, seat[pairs:]], fb)):
        # one division, the product with 1/m (up to 4) and the division by P round to the smallest number, 5e-324
        big = np.abs(want) > 1e-290
        np.testing.assert_array_equal(got[big], want[big])
        assert np.all(np.abs(got[~big] - want[~big]) <= 1e-322)
    assert np.any(fa != 0)
