"""A cycle energy that is NaN makes the reweighting factor of every xi' whose
sums hold it NaN: every row from its own on sums it or a row that does.  The
energies are the host's (nothing else of the state is used)."""
import numpy as np
import pytest

import pyxmd
from orc import dptr
from test_gpu_recursion_paths import bridges

pytestmark = pytest.mark.gpu

GRID = np.array([-1.0, -0.5, 0.0, 0.3, 1.0])


@pytest.mark.parametrize("N", [1, 5, 64, 65, 200])
def test_nan_energy(N):
    lib = pyxmd.Lib()
    P = 8
    s = pyxmd.System(lib, "trap", N, P, 1.0, 1.0, seed=1,
                     positions=bridges(N, P, 1.0, 12, np.random.default_rng(N)).reshape(N * P, 3))
    assert lib.md_pimd_fast_fill_ENk_x(s.pimd, 0) == 0
    assert lib.md_pimd_fill_VB_x(s.pimd) == 0
    s.host_pimd()
    E = pyxmd.tri(s.pimd)
    for n, k in sorted({(1, 1), (N, 1), (N, N), ((N + 1) // 2, 1), (N, (N + 1) // 2), (min(N, 64), min(N, 3))}):
        print(f"N={N} E_{n}^({k}) = NaN", flush=True)
        assert lib.md_pimd_sync_host_x(s.pimd, 0)  # the host's energies count from here on
        host = np.ctypeslib.as_array(s.pimd.contents.ENk[0], shape=(E.size,))
        host[:] = E
        host[(n - 1) * n // 2 + k - 1] = np.nan
        fac = np.zeros(len(GRID))
        assert lib.md_pimd_calc_vi_sign_grid_x(s.pimd, len(GRID), dptr(GRID), dptr(fac)) == 0
        for xi, f in zip(GRID, fac):
            assert np.isnan(f) == (xi != 0 or k == 1), (xi, f)
