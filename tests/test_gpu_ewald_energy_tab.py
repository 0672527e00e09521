"""Tabulated real-space Ewald energies (k_ewald_real_energy) at the edges of
their 64-bead tiles and in each image enumeration, against the untabulated
tile kernel, which a cutoff beyond the table's range (x_cut = 6.6) selects.
Both sums are converged to the rounding floor; the energies are held to the
estimators' 1e-12."""
import pytest

import pyxmd

pytestmark = pytest.mark.gpu


def energy(lib, s):
    st = lib.md_alloc_stats_x(1)
    assert lib.md_pimd_calc_pair_energy_x(s.pimd, s.pair_energy_cb(), st) == 0
    return st.contents.es[0]


@pytest.mark.parametrize("N,P", [(2, 3), (33, 8), (63, 2), (64, 2), (65, 5), (130, 2), (257, 3)])
def test_energy_routes(N, P):
    lib = pyxmd.Lib()
    L = pyxmd.ueg_box(N, 2.0)
    s = pyxmd.System(lib, "ueg", N, P, pyxmd.ueg_temperature(N, L, 0.5), 1.0, seed=5 + N, L=L, nsum=8)
    if N * P % 2:  # an odd number of draws leaves a spare, which the next seed does not clear
        lib.md_random_gaussian_x()
    try:
        lib.md_set_ewald_real_cutoff_x(6.6)
        want = energy(lib, s)
        lib.md_set_ewald_real_cutoff_x(5.25)
        # alpha' L and the images it needs: face, near, corner
        for split in (-1.0, 9.0, 7.0, 5.0):
            lib.md_set_ewald_split_x(split)
            got = energy(lib, s)
            print(f"N={N} P={P} alpha'L={split}: {got:.15e} vs {want:.15e}", flush=True)
            assert abs(got - want) <= 1e-12 * max(abs(want), N / L)
    finally:
        lib.md_set_ewald_real_cutoff_x(5.25)
        lib.md_set_ewald_split_x(-1.0)
