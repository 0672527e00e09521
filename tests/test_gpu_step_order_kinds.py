"""The step's branch orders for the states and interactions that
test_gpu_step_orders leaves out, against the serial single-stream order bit for
bit, eager and replayed: systems of the largest size without permutation cycles
(xi = 0, high temperature) and one whose xi changes between calls, grouped
chains, Ewald outside the tables, and tile sums left for NHC half 2 with one
and with several tiles, at both sides of the line below which the bead-local
forces ride with the springs (N^2 P = 2e5)."""
import ctypes as C

import numpy as np
import pytest

import pyxmd
from test_gpu_graph_reuse import state, ueg_box

pytestmark = pytest.mark.gpu

CB = {"trap": "md_gaussian_force_x", "pgauss": "md_periodic_gaussian_force_x", "ueg": "md_coulomb_3d_ewald_force_x",
      "ewr": "md_coulomb_3d_ewald_force_R_x", "lj": "md_LJ_periodic_force_x", "he": "md_periodic_helium_force_x"}


@pytest.fixture
def lib():
    """The library with chains of four links; its globals as they were afterwards."""
    lib = pyxmd.Lib()
    M = lib.md_get_nhc_length_x()
    lib.md_set_nhc_length_x(4)
    yield lib
    lib.md_set_nhc_length_x(M)
    lib.md_set_ewald_split_x(-1.0)


def system(lib, kind, N, P, xi=1.0, T=None, nsum=8, fgroup=1):
    s = build(lib, kind, N, P, xi, T, nsum, fgroup)
    if kind != "trap" and N * P % 2:  # an odd number of draws leaves a spare, which the next seed does not clear
        lib.md_random_gaussian_x()
    return s


def build(lib, kind, N, P, xi, T, nsum, fgroup):
    if kind in ("ueg", "ewr"):
        return pyxmd.System(lib, "ueg", N, P, T or 0.4, xi, seed=5, L=ueg_box(N), nsum=nsum, fgroup=fgroup)
    if kind == "trap":
        return pyxmd.System(lib, "trap", N, P, 1.0, xi, seed=5, fgroup=fgroup)
    # a jittered lattice of spacing 1.5 (the cores of LJ and helium kept apart)
    m = int(np.ceil(N ** (1 / 3)))
    site = np.arange(m ** 3)[:N]
    x = np.stack([site // (m * m), site // m % m, site % m], 1) + 0.5
    x = x[:, None] * 1.5 + np.random.default_rng(N).uniform(-0.1, 0.1, (N, P, 3))
    if kind == "he":
        lib.md_set_helium_parameters_x(10.8, 1.8443101e5, 10.43329537, 1.36745214, 0.42123807, 0.17473318, 1.4826, 1.0)
    return pyxmd.System(lib, "pgauss", N, P, 1.0, xi, seed=5, L=1.5 * m, positions=x.reshape(N * P, 3), fgroup=fgroup)


def check(lib, kind, systems, dt, split=-1.0):
    graph, eager, serial = systems
    trap = lib.cb["md_harmonic_trap_force_x"] if kind == "trap" else None
    cfg = [pyxmd.StepConfig(trap, lib.cb[CB[kind]], dt, s.image, s.image, int(s is graph)) for s in systems]
    stages = np.zeros(11)
    lib.md_set_ewald_split_x(split)
    for n in (1, 4):
        assert lib.md_pimd_run_steps_x(graph.pimd, C.byref(cfg[0]), n) == 0
        assert lib.md_pimd_run_steps_x(eager.pimd, C.byref(cfg[1]), n) == 0
        assert lib.md_pimd_profile_steps_x(serial.pimd, C.byref(cfg[2]), n, 1, pyxmd.dptr(stages)) == 0
        assert lib.md_hip_synchronize_x() == 0
        want = state(serial)
        assert np.all(np.isfinite(want[2]))
        for got in (state(graph), state(eager)):
            for a, b in zip(got, want):
                np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("xi,T", [(0.0, 0.4), (1.0, 60.0)])
@pytest.mark.parametrize("N", [1249, 1251])
def test_large_without_cycles(lib, N, xi, T):
    print(f"N={N} xi={xi} T={T}", flush=True)
    check(lib, "ueg", [system(lib, "ueg", N, 32, xi, T) for _ in range(3)], 0.001)


def test_xi_changes_between_calls(lib):
    s = [system(lib, "ueg", 1260, 32) for _ in range(3)]
    for xi in (1.0, 0.0, 0.5):
        print(f"xi={xi}", flush=True)
        for z in s:
            z.pimd.contents.vi = xi
        check(lib, "ueg", s, 0.001)


@pytest.mark.parametrize("kind,N,P", [("trap", 8, 8), ("trap", 70, 32), ("trap", 380, 56), ("ueg", 16, 32),
                                      ("ueg", 140, 48), ("ueg", 620, 32)])
def test_grouped_chains(lib, kind, N, P):
    print(f"{kind} N={N} P={P} groups of 3", flush=True)
    check(lib, kind, [system(lib, kind, N, P, fgroup=3) for _ in range(3)], 0.01)


@pytest.mark.parametrize("kind,N,P,split", [("ueg", 20, 8, 0.0), ("ueg", 150, 16, 0.0), ("ueg", 420, 48, 0.0),
                                            ("ewr", 20, 8, -1.0), ("ewr", 150, 16, -1.0), ("ewr", 420, 48, -1.0)])
def test_ewald_outside_the_tables(lib, kind, N, P, split):
    print(f"{kind} N={N} P={P}", flush=True)
    check(lib, kind, [system(lib, kind, N, P, nsum=2) for _ in range(3)], 0.01, split)


@pytest.mark.parametrize("kind", ["trap", "pgauss", "lj", "he"])
@pytest.mark.parametrize("N,P", [(40, 125), (40, 126), (64, 48), (64, 49), (65, 47), (65, 48), (150, 8), (150, 10),
                                 (200, 33)])
def test_tile_sums_left_for_the_thermostat(lib, kind, N, P):
    print(f"{kind} N={N} P={P} w={N * N * P}", flush=True)
    check(lib, kind, [system(lib, kind, N, P) for _ in range(3)], 1e-4)
