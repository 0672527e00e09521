"""Histogram observables at the edges of their work split (workgroups of 4096
samples, LDS or global counts, single rows, many counts per bin) against
numpy counts accumulated one increment at a time, bit for bit, on top of
values left by an earlier sample."""
import numpy as np
import pytest

import pyxmd
from orc import dptr

pytestmark = pytest.mark.gpu


def sequential(fx, counts, incr):
    out = fx.copy()
    for b, n in enumerate(counts):
        if n:
            out[b] = np.cumsum(np.concatenate([[fx[b]], np.full(int(n), incr)]))[-1]
    return out


@pytest.mark.parametrize("N,P,points", [(1, 2, 5), (2, 3, 64), (17, 4, 1), (64, 3, 200), (65, 5, 13000), (260, 2, 37),
                                        (701, 3, 200)])
def test_histograms(N, P, points):
    lib = pyxmd.Lib()
    rng = np.random.default_rng([N, P, points])
    L = np.array([5.0, 5.5, 6.0])
    sim = lib.md_alloc_simulation_x(N * P, 1, 0, 0)
    lib.md_init_nd_rect_box_x(sim.contents.box, dptr(L))
    pimd = lib.md_alloc_pimd_x(sim, N, P, 1.0, 1.0)
    lib.md_init_particle_mass_x(sim, 1.0, 0, N * P)
    b = pyxmd.beads(sim)
    x = rng.uniform(0.0, 5.0, (N, P, 3))
    b["x"] = x.reshape(N * P, 3)
    pyxmd.set_beads(sim, b)
    pi, norm, rmax = P, 7.0, 2.4
    off = ~np.eye(N, dtype=bool)

    def image(d):
        return d - L * np.round(d / L)

    def bins(r, width):
        k = (r / width).astype(np.int64)
        return np.bincount(k[(k >= 0) & (k < points)], minlength=points)

    n = int(np.sqrt(points))
    clamp = lambda i, j: np.bincount(np.clip(i * n + j, 0, points - 1).ravel(), minlength=points)
    d = image(x[:, 0][:, None] - x[:, pi - 1][None])
    w2 = rmax / n
    i1 = (x[:, 0, 0] / (5.0 / n)).astype(np.int64)
    i2 = (x[:, pi - 1, 0] / (5.0 / n)).astype(np.int64)
    c = x - L / 2
    plane = sum((bins(np.sqrt((dd ** 2).sum(-1))[off], rmax / points)
                 for dd in (x[:, j, None, :2] - x[None, :, j, :2] for j in range(P))), np.zeros(points, np.int64))
    box = np.array([-1.0, 6.0, -1.0, 6.0])
    cases = {
        "density": (lambda st: lib.md_pimd_calc_density_distribution_x(pimd, st, rmax, 0, dptr(L / 2)),
                    bins(np.sqrt((c * c).sum(-1)).ravel(), rmax / points), 1.0 / P),
        "radial": (lambda st: lib.md_pimd_calc_pair_correlation_x(pimd, st, rmax, norm, pi, 1),
                   bins(np.sqrt((d * d).sum(-1))[off], rmax / points), 1.0 / norm),
        "axes": (lambda st: lib.md_pimd_calc_2d_pair_correlation_x(pimd, st, rmax, norm, pi, 1),
                 clamp((np.abs(d[..., 0]) / w2).astype(np.int64)[off], (np.abs(d[..., 1]) / w2).astype(np.int64)[off]),
                 1.0 / norm),
        "itcf": (lambda st: lib.md_pimd_calc_ITCF_x(pimd, st, 0.0, 5.0, pi), clamp(i1[:, None], i2[None]), 1.0 / P),
        "plane": (lambda st: lib.md_pimd_calc_pair_correlation_2d_x(pimd, st, rmax, norm, dptr(box)), plane,
                  1.0 / norm),
    }
    for name, (call, counts, incr) in cases.items():
        st = lib.md_alloc_stats_x(points)
        fx = np.ctypeslib.as_array(st.contents.fxs[0], shape=(points,))
        fx[:] = rng.uniform(0, 3, points)
        want = fx.copy()
        for _ in range(2):
            print(f"N={N} P={P} points={points} {name}", flush=True)
            want = sequential(want, counts, incr)
            assert call(st) == 0
            assert np.array_equal(fx, want), name
