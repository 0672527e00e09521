"""A kept step graph is not updated with one of another topology.

Steps of a trapped system with and without its pair force have as many kernels
and edges, but between others of them: with it the tile sums are left for NHC
half 2, without it the exchange forces are added by a kernel of their own.  A run
whose calls change between them must follow the eagerly launched trajectory bit
for bit."""
import ctypes as C

import numpy as np
import pytest

import pyxmd
from test_gpu_graph_reuse import state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P,steps", [(70, 64, 4), (70, 64, 36), (300, 64, 5)])
def test_pair_force_comes_and_goes(N, P, steps):
    lib = pyxmd.Lib()
    graph, eager = (pyxmd.System(lib, "trap", N, P, 1.0, 1.0, seed=7) for _ in range(2))
    trap = lib.cb["md_harmonic_trap_force_x"]
    for k, pair in enumerate([True, False, True, False, False, True]):
        print(f"N={N} P={P} call {k}, pair force {pair}", flush=True)
        for s, use_graph in ((graph, 1), (eager, 0)):
            cfg = pyxmd.StepConfig(trap, s.pair_cb() if pair else None, 0.005, 0, 0, use_graph)
            assert lib.md_pimd_run_steps_x(s.pimd, C.byref(cfg), steps) == 0
        assert lib.md_hip_synchronize_x() == 0
        for a, b in zip(state(graph), state(eager)):
            np.testing.assert_array_equal(a, b)
