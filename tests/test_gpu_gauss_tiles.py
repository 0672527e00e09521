"""Gaussian pair forces of the tile kernels (divisions by a corrected
reciprocal, several rotations at a time) against the two-species kernel, which
evaluates the term plainly, bit for bit.

The beads come in pairs 200 ranges apart, where every other term underflows to
zero, so a bead's force is one term whatever the order of summation.  The
pairs join random beads, within tiles of 64 and across them; their distances
run to where the term underflows, and some share a coordinate or the place.
Masses and the slice count are powers of two (their products are exact; near
the smallest numbers one rounding each may differ)."""
import numpy as np
import pytest

import pyxmd

pytestmark = pytest.mark.gpu


def system(lib, kind, x, m, L):
    P, N = x.shape[:2]
    s = pyxmd.System(lib, kind, N, P, 1.0, 1.0, seed=1, L=L, positions=x.transpose(1, 0, 2).reshape(N * P, 3))
    hb = s.host_beads()
    hb["m"] = np.repeat(m, P)
    pyxmd.set_beads(s.sim, hb)
    assert lib.md_reset_force_x(s.sim) == 0
    return s


def forces(s):
    return s.host_beads()["f"].reshape(s.N, s.P, 3).transpose(1, 0, 2)


@pytest.mark.parametrize("kind", ["trap", "pgauss"])
@pytest.mark.parametrize("s", [0.5, 1e-3, 3e20])
@pytest.mark.parametrize("pairs", [1, 4, 16, 17, 32, 33, 65])
def test_tiles_match_plain_terms(kind, s, pairs):
    lib = pyxmd.Lib()
    P = 8
    rng = np.random.default_rng([pairs, int(1e4 * s) % 10 ** 9])
    L = 200.0 * s * pairs
    r = rng.normal(size=(P, pairs, 3))
    r *= (s * rng.uniform(0, 29, size=(P, pairs)) / np.linalg.norm(r, axis=2))[..., None]
    r[:, ::5, 1] = 0.0
    r[1, 0] = 0.0
    r[2, 0] = [1e-160 * s, 0.0, 0.0]
    a = np.zeros((P, pairs, 3))
    a[..., 0] = 200.0 * s * np.arange(pairs)
    a += s * rng.uniform(0, 10, size=(P, pairs, 3))
    a[2, 0] = 0.0
    if kind == "pgauss":
        a += L / 4
    b = a + r
    m = 2.0 ** rng.integers(-2, 3, pairs)
    seat = rng.permutation(2 * pairs)
    x, mm = np.empty((P, 2 * pairs, 3)), np.empty(2 * pairs)
    x[:, seat[:pairs]], x[:, seat[pairs:]] = a, b
    mm[seat[:pairs]] = mm[seat[pairs:]] = m
    print(f"{kind} pairs={pairs} s={s}", flush=True)
    one, sa, sb = system(lib, kind, x, mm, L), system(lib, kind, a, m, L), system(lib, kind, b, m, L)
    lib.md_set_guassian_force_range_x(s)
    try:
        assert lib.md_pimd_calc_pair_force_x(one.pimd, one.pair_cb()) == 0
        assert lib.md_pimd_calc_pair_force_2_x(sa.pimd, sb.pimd, one.pair_cb()) == 0
        assert lib.md_hip_synchronize_x() == 0
        f, fa, fb = forces(one), forces(sa), forces(sb)
    finally:
        lib.md_set_guassian_force_range_x(0.5)
    for got, want in ((f[:, seat[:pairs]], fa), (f[:, seat[pairs:]], fb)):
        big = np.abs(want) > 1e-290
        np.testing.assert_array_equal(got[big], want[big])
        assert np.all(np.abs(got[~big] - want[~big]) <= 1e-322)
    assert np.any(fa != 0)
