"""Reading the state on the host leaves the chains' group sizes as the host has
them (the device does not change them) and brings everything else, at the sizes
of both ways of the copy (below 3 MB at once, above in pieces)."""
import ctypes as C

import numpy as np
import pytest

import pyxmd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P,fgroup", [(3, 4, 1), (3, 4, 6), (200, 23, 1), (203, 24, 1), (700, 25, 1), (700, 25, 3)])
def test_group_sizes_stay_the_hosts(N, P, fgroup):
    lib = pyxmd.Lib()
    s = pyxmd.System(lib, "trap", N, P, 1.0, 1.0, seed=1, fgroup=fgroup)
    if N * P % 2:  # an odd number of draws leaves a spare, which the next seed does not clear
        lib.md_random_gaussian_x()
    before, Nf = pyxmd.nhcs(s.sim), s.sim.contents.Nf
    cfg = s.step_config(0.01)
    print(f"N={N} P={P} groups of {fgroup}", flush=True)
    assert lib.md_pimd_run_steps_x(s.pimd, C.byref(cfg), 3) == 0
    mark = np.arange(Nf) % 7 + 10
    for read_only in (1, 0):
        for i in range(Nf):
            s.sim.contents.nhcs[i].f = int(mark[i])
        assert lib.md_simulation_sync_host_x(s.sim, read_only)
        got = pyxmd.nhcs(s.sim)
        np.testing.assert_array_equal(got["f"], mark)
        np.testing.assert_array_equal(got["Q"], before["Q"])
        M = lib.md_get_nhc_length_x()
        assert np.all(got["theta"][:, :M] != before["theta"][:, :M])
        np.testing.assert_array_equal(got["theta"][:, M:], before["theta"][:, M:])
        assert np.all(got["vtheta"][:, :M] != before["vtheta"][:, :M])
