"""Histogram counts start from zero whenever their buffer is made or grows.

The counts are cleared on the stream that fills them, so a call whose bins no
longer fit the buffer counts into cleared memory.  Each call here has more bins
than any before it; its counts are compared with numpy's."""
import numpy as np
import pytest

import pyxmd
from orc import dptr

pytestmark = pytest.mark.gpu


def test_counts_of_a_grown_buffer():
    lib = pyxmd.Lib()
    rng = np.random.default_rng(5)
    N, P, L = 40, 4, np.array([5.0, 5.0, 5.0])
    sim = lib.md_alloc_simulation_x(N * P, 1, 0, 0)
    lib.md_init_nd_rect_box_x(sim.contents.box, dptr(L))
    pimd = lib.md_alloc_pimd_x(sim, N, P, 1.0, 1.0)
    lib.md_init_particle_mass_x(sim, 1.0, 0, N * P)
    b = pyxmd.beads(sim)
    b["x"] = rng.uniform(0.0, 5.0, (N * P, 3))
    pyxmd.set_beads(sim, b)
    r = np.sqrt(((b["x"] - L / 2) ** 2).sum(1))
    for points in (30000, 60000, 120000, 240000, 480000, 960000):
        print(f"points={points}", flush=True)
        st = lib.md_alloc_stats_x(points)
        fx = np.ctypeslib.as_array(st.contents.fxs[0], shape=(points,))
        assert lib.md_pimd_calc_density_distribution_x(pimd, st, 5.0, 0, dptr(L / 2)) == 0
        want = np.bincount((r / (5.0 / points)).astype(np.int64), minlength=points)[:points] / P
        assert np.array_equal(fx, want)
