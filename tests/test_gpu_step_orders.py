"""Each order of the step's branches, at both sides of the lines between them
(w = N^2 P pair terms), against the serial single-stream order bit for bit:
eager, replayed and with stage events."""
import ctypes as C

import numpy as np
import pytest

import pyxmd
from test_gpu_graph_reuse import make, state, ueg_box

pytestmark = pytest.mark.gpu

# Ewald lines at 2.5e6, 1.2e7 and 5e7, other pair forces at 1.5e3 and 8e6
CASES = [("ueg", 16, 32), ("ueg", 176, 48), ("ueg", 177, 48), ("ueg", 611, 32), ("ueg", 613, 32), ("ueg", 1249, 32),
         ("ueg", 1251, 32), ("trap", 24, 16), ("trap", 353, 64), ("trap", 354, 64), ("ueg", 228, 48), ("ueg", 229, 48),
         ("trap", 8, 8), ("trap", 5, 59), ("trap", 5, 61)]


@pytest.mark.parametrize("kind,N,P", CASES)
def test_orders_match_serial(kind, N, P):
    lib = pyxmd.Lib()
    lib.md_set_nhc_length_x(4)
    lib.md_set_coulomb_truc_x(5.0 / ueg_box(N))
    lib.md_set_coulomb_n_sum_x(8)
    conc, prof, ser = (make(lib, kind, N, P, 5) for _ in range(3))
    stages = np.zeros(11)
    print(f"{kind} N={N} P={P}", flush=True)
    for n in (1, 5):
        cc, cp, cs = (s.step_config(0.01, use_graph=g) for s, g in ((conc, 1), (prof, 0), (ser, 0)))
        assert lib.md_pimd_run_steps_x(conc.pimd, C.byref(cc), n) == 0
        assert lib.md_pimd_profile_steps_x(prof.pimd, C.byref(cp), n, 0, pyxmd.dptr(stages)) == 0
        assert stages[8] > 0
        assert lib.md_pimd_profile_steps_x(ser.pimd, C.byref(cs), n, 1, pyxmd.dptr(stages)) == 0
        assert lib.md_hip_synchronize_x() == 0
        want = state(ser)
        for got in (state(conc), state(prof)):
            for a, b in zip(got, want):
                np.testing.assert_array_equal(a, b)
