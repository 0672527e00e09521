"""A row of the estimators' recursion that has no finite value makes the result
NaN, wherever the row stands: sums left unfinished behind it, or columns
passed over because their weight is zero, must not hide it.  The rows come
from host potentials that are NaN or infinite."""
import numpy as np
import pytest

import pyxmd
from test_gpu_recursion_paths import bridges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("N", [1, 5, 64, 65, 200])
def test_row_without_a_value(N, bad):
    lib = pyxmd.Lib()
    P = 8
    s = pyxmd.System(lib, "trap", N, P, 1.0, 1.0, seed=1,
                     positions=bridges(N, P, 1.0, 12, np.random.default_rng(N)).reshape(N * P, 3))
    assert lib.md_pimd_fast_fill_ENk_x(s.pimd, 0) == 0
    assert lib.md_pimd_fill_VB_x(s.pimd) == 0
    s.host_pimd()
    good = pyxmd.vbn(s.pimd)
    for m in sorted({0, 1, N // 2, N - 1, N}):
        print(f"N={N} V_B({m}) = {bad}", flush=True)
        assert lib.md_pimd_sync_host_x(s.pimd, 0)  # the host's potentials count from here on
        V = np.ctypeslib.as_array(s.pimd.contents.VBN, shape=(N + 1,))
        V[:] = good
        V[m] = bad
        assert np.isnan(s.stat(lib.md_pimd_calc_VBN_energy_x, s.pimd))
    assert lib.md_pimd_sync_host_x(s.pimd, 0)
    np.ctypeslib.as_array(s.pimd.contents.VBN, shape=(N + 1,))[:] = good
    assert np.isfinite(s.stat(lib.md_pimd_calc_VBN_energy_x, s.pimd))
