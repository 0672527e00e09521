"""A replica's recursion error that is pending when a batch runs is reported by
the batch call, once, wherever the replica stands in the table.  The error is
forced from the host (md_pimd_inject_recursion_timeouts_x) in a force
evaluation of the replica alone, N = 200 being four row blocks."""
import ctypes as C

import pytest

import pyxmd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [0, 1])
@pytest.mark.parametrize("n,bad", [(1, 0), (3, 0), (3, 2), (300, 299)])
def test_batch_reports_a_pending_error_once(n, bad, use_graph):
    lib = pyxmd.Lib()
    lib.md_set_nhc_length_x(4)
    systems = [pyxmd.System(lib, "trap", 200 if i == bad else 6, 4, 1.0, 1.0, seed=i + 1) for i in range(n)]
    cfgs = (pyxmd.StepConfig * n)(*[s.step_config(0.01, use_graph=use_graph) for s in systems])
    ptrs = (pyxmd.PIMD_P * n)(*[s.pimd for s in systems])
    print(f"{n} replicas, error in {bad}, graph={use_graph}", flush=True)
    assert lib.md_pimd_run_batch_x(ptrs, cfgs, n, 2) == 0
    assert lib.md_pimd_inject_recursion_timeouts_x(systems[bad].pimd, 1) == 0
    assert lib.md_pimd_compute_forces_x(systems[bad].pimd, C.byref(cfgs[bad])) == 0  # queued only
    assert lib.md_pimd_run_batch_x(ptrs, cfgs, n, 2) == -1
    assert lib.md_pimd_run_batch_x(ptrs, cfgs, n, 2) == 0
    assert lib.md_hip_synchronize_x() == 0
    lib.md_set_nhc_length_x(8)
