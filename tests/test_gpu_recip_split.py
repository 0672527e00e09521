"""The reciprocal Ewald forces of 16 beads per workgroup against the general
kernel's 64, bit for bit: a slice's forces times P do not depend on how many
slices there are (P a power of two scales exactly), while the number of
workgroups, hence the kernel, does (fewer than 256 of 64 beads: split).  The
slices of the larger system repeat those of the smaller one."""
import numpy as np
import pytest

import pyxmd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("aL,nsum", [(4.0, 4), (5.0, 8)])
@pytest.mark.parametrize("N,P,many", [(1, 8, 256), (15, 8, 256), (16, 128, 256), (17, 8, 256), (33, 8, 256),
                                      (64, 8, 256), (65, 64, 128), (130, 64, 128), (200, 32, 64)])
def test_split_matches_general(N, P, many, aL, nsum):
    lib = pyxmd.Lib()
    L = 12.0
    lib.md_set_coulomb_truc_x(aL / L)
    lib.md_set_coulomb_n_sum_x(nsum)
    x = np.random.default_rng([N, P]).uniform(0, L, size=(N, P, 3))
    f = {}
    for p in (P, many):
        print(f"N={N} P={p} alpha L={aL}", flush=True)
        beads = np.tile(x, (1, p // P, 1)).reshape(N * p, 3)
        s = pyxmd.System(lib, "ueg", N, p, 0.4, 1.0, seed=1, L=L, nsum=nsum, positions=beads)
        assert lib.md_reset_force_x(s.sim) == 0
        assert lib.md_pimd_calc_pair_force_x(s.pimd, s.pair_cb()) == 0
        assert lib.md_hip_synchronize_x() == 0
        f[p] = s.host_beads()["f"].reshape(N, p, 3) * p
    for k in range(0, many, P):
        np.testing.assert_array_equal(f[many][:, k:k + P], f[P])
