"""Workloads whose speed matters to a user of the PIMD engine, for timing one
build of it against another.

A user's program has the engine do five things, all through the C ABI:

  steps    md_pimd_run_steps_x: a block of MD steps of one system, replayed
           as a captured graph, after which the beads are read on the host
           (a block of a production run, ended by a checkpoint or analysis);
  driver   the reference's own driver loop, one call per stage
           (md_update_nhc_VV3_1_x ... md_update_nhc_VV3_2_x), as a ported C
           driver makes them;
  batch    md_pimd_run_batch_x: a table of independent replicas (a scan over
           N, P, r_s and the exchange parameter xi) advanced together;
  sample   the energy estimators of one sampled configuration, with the
           reweighting factors of a xi grid;
  observe  the histograms and structure factors of one sampled configuration.

Systems: harmonically trapped bosons with a Gaussian pair force (open
boundaries) and the spin-polarised uniform electron gas (UEG, periodic, 3-D
Ewald), both over the xi family used to extrapolate to fermions.  Sizes run
from the few-particle systems of the tests to twice the N=1024, P=32 electron
gas of the benchmark, odd ones among them.

Initial beads are those of an ideal thermal ensemble: cycles of consecutive
particles as Brownian bridges of the free ring polymer (so that exchange and
springs have the values they take in a run), placed on a jittered lattice
(UEG) or in the trap's thermal cloud.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "md-lab_amd"))

import pyxmd  # noqa: E402

TRAP_G, TRAP_S = 3.0, 0.5  # Gaussian pair force: strength, range (set by pyxmd.System)
SIGN_GRID = 16             # xi' values of a reweighting grid
BATCH_ALPHA, BATCH_NSUM = 2.0, 200  # one converged Ewald parameter set for the boxes of a batch


def listed():
    return [
        # The smallest system of the tests: nothing but launches and latency.
        dict(name="steps-trap-8", kind="steps", system="trap", N=8, P=8, xi=1.0, chain=8, steps=100),
        # A few-electron UEG, the size of published fermionic benchmarks; one point of a xi scan.
        dict(name="steps-ueg-16", kind="steps", system="ueg", N=16, P=32, xi=0.5, rs=2.0, chain=4, steps=100),
        # Trapped bosons at a production size (the xi extrapolation runs of the tests).
        dict(name="steps-trap-256", kind="steps", system="trap", N=256, P=64, xi=0.25, chain=8, steps=50),
        # A mid-size UEG with many beads (low temperature).
        dict(name="steps-ueg-128", kind="steps", system="ueg", N=128, P=64, xi=1.0, rs=2.0, chain=4, steps=50),
        # The benchmark's electron gas.
        dict(name="steps-ueg-1024", kind="steps", system="ueg", N=1024, P=32, xi=1.0, rs=2.0, chain=4, steps=20),
        # The largest: an odd particle number beyond the benchmark's size.
        dict(name="steps-ueg-2001", kind="steps", system="ueg", N=2001, P=24, xi=0.75, rs=4.0, chain=4, steps=16),
        # A ported driver on a small trapped system: one call per stage.
        dict(name="driver-trap-24", kind="driver", system="trap", N=24, P=16, xi=1.0, chain=8, steps=10),
        # A ported driver on a ragged UEG, bead count not a multiple of 8.
        dict(name="driver-ueg-333", kind="driver", system="ueg", N=333, P=27, xi=0.5, rs=1.0, chain=8, steps=5),
        # A scan over N, P, r_s and xi: trapped and UEG replicas advanced together.
        dict(name="batch-32", kind="batch", table=2024, n=32, nmax=512, chain=4, steps=20),
        # One sample of the energy estimators, trapped bosons.
        dict(name="sample-trap-150", kind="sample", system="trap", N=150, P=48, xi=0.75, chain=8),
        # One sample of the energy estimators on the benchmark's electron gas.
        dict(name="sample-ueg-1024", kind="sample", system="ueg", N=1024, P=32, xi=1.0, rs=2.0, chain=4),
        # One sample of the histograms and structure factors.
        dict(name="observe-ueg-700", kind="observe", system="ueg", N=700, P=40, xi=1.0, rs=2.0, chain=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "driver", "batch", "sample", "observe"])
    if kind == "batch":
        return dict(kind=kind, table=rng.randrange(1 << 20), n=rng.randint(6, 32), nmax=rng.choice([64, 128, 256, 512]),
                    chain=4, steps=rng.randint(10, 20))
    system = "ueg" if kind == "observe" else rng.choice(["trap", "ueg"])
    N = _log_int(rng, 5, 600) if system == "trap" else _log_int(rng, 8, 1500)
    c = dict(kind=kind, system=system, N=N, P=_log_int(rng, 6, 72), xi=rng.choice([0.0, 0.25, 0.5, 0.75, 1.0]),
             chain=rng.choice([4, 8]))
    while c["N"] * c["P"] > 48000:
        c["P"] = c["P"] // 2
    if system == "ueg":
        c["rs"] = rng.choice([1.0, 2.0, 4.0])
    if kind == "steps":
        c["steps"] = rng.randint(20, 100) if c["N"] * c["P"] < 16000 else rng.randint(10, 20)
    if kind == "driver":
        c["steps"] = rng.randint(4, 10)
    return c


# ------------------------------------------------------------- the systems


def _shape(c):
    """Box edge, temperature and time step of a single-system case; the time
    step is a tenth of the ring polymer's 1 / omega_P (0.05 for the
    benchmark's electron gas, as the benchmark has it)."""
    L, T = 10.0, 1.0
    if c["system"] == "ueg":
        L = pyxmd.ueg_box(c["N"], c["rs"])
        T = pyxmd.ueg_temperature(c["N"], L, 0.5)
    return L, T, 0.1 / (math.sqrt(c["P"]) * T)


def _beads(c, seed):
    """Positions and velocities [particle, bead, 3] of a thermal ensemble."""
    rng = np.random.default_rng([seed, c["N"], c["P"]])
    N, P = c["N"], c["P"]
    L, T, _ = _shape(c)
    tau = 1.0 / (T * P)  # hbar^2 beta / (m P)
    if c["system"] == "trap":
        centre = rng.normal(size=(N, 3)) * 1.5
    else:
        m = math.ceil(N ** (1 / 3) - 1e-9)
        site = rng.permutation(m ** 3)[:N]
        centre = (np.stack([site // (m * m), site // m % m, site % m], 1) + 0.5 + rng.uniform(-0.2, 0.2, (N, 3))) * L / m
    x = np.empty((N, P, 3))
    n = 0
    while n < N:
        k = 1 if c["xi"] == 0.0 else min(N - n, int(rng.geometric(0.5)), 12)
        w = rng.normal(size=(k * P, 3)) * math.sqrt(tau)
        path = np.cumsum(w, 0) - np.arange(1, k * P + 1)[:, None] / (k * P) * w.sum(0)
        x[n:n + k] = (path - path.mean(0) + centre[n]).reshape(k, P, 3)
        n += k
    if c["system"] == "ueg":
        x = x % L
    return x, rng.normal(size=(N, P, 3)) * math.sqrt(T)


def _system(lib, c, seed):
    L, T, _ = _shape(c)
    s = pyxmd.System(lib, c["system"], c["N"], c["P"], T, c["xi"], seed=1, L=L, nsum=8,
                     positions=np.zeros((c["N"] * c["P"], 3)))
    x, v = _beads(c, seed)
    pyxmd.load_state(s, x, v)
    return s


def _state_view(sim):
    """The beads' host mirror, without a copy: [bead, (m, x, v, f)]."""
    s = sim.contents
    buf = (C.c_double * (10 * s.N)).from_address(C.addressof(s.particles.contents))
    return np.frombuffer(buf, dtype=np.float64).reshape(s.N, 10)


def _replicas(c):
    """The replica table of a batch: N a power of two and P as in a scan, half
    trapped bosons, half UEG."""
    rng = np.random.default_rng(c["table"])
    top = int(math.log2(c["nmax"] / 8)) + 1
    out = []
    for _ in range(c["n"]):
        r = dict(system=str(rng.choice(["trap", "ueg"])), N=int(8 * 2 ** rng.integers(0, top)),
                 P=int(rng.choice([16, 32, 64])), xi=float(rng.choice([0.0, 0.25, 0.5, 0.75, 1.0])))
        if r["system"] == "ueg":
            r["rs"] = float(rng.choice([1.0, 2.0, 4.0]))
        out.append(r)
    return out


_LIB = []


def _lib():
    if not _LIB:
        _LIB.append(pyxmd.Lib())
    return _LIB[0]


def _checked(rc, what):
    if rc != 0:
        raise RuntimeError(what + " failed")


def _observe_grid(c):
    L = _shape(c)[0]
    return dict(L=L, dq=2 * math.pi / L, points=200, itcf=48 * 48, axes=32, shells=6, pi=c["P"] // 2)


# ------------------------------------------------------- prepare and run


def prepare(case, seed):
    lib = _lib()
    lib.md_set_nhc_length_x(case["chain"])
    kind = case["kind"]
    if kind == "batch":
        reps = _replicas(case)
        systems = [_system(lib, r, seed + 1000 * i) for i, r in enumerate(reps)]
        lib.md_set_coulomb_truc_x(BATCH_ALPHA)
        lib.md_set_coulomb_n_sum_x(BATCH_NSUM)
        cfgs = (pyxmd.StepConfig * len(systems))(*[s.step_config(_BATCH_DT) for s in systems])
        for s, cfg in zip(systems, cfgs):
            _checked(lib.md_pimd_compute_forces_x(s.pimd, C.byref(cfg)), "forces")
        _checked(lib.md_hip_synchronize_x(), "forces")
        return dict(case=case, systems=systems, cfgs=cfgs,
                    ptrs=(pyxmd.PIMD_P * len(systems))(*[s.pimd for s in systems]))
    s = _system(lib, case, seed)
    st = dict(case=case, s=s, dt=_shape(case)[2])
    s.full_force()
    if kind == "steps":
        st["cfg"] = s.step_config(st["dt"])
    if kind == "sample":
        st["stats"] = {k: lib.md_alloc_stats_x(1) for k in _SAMPLE}
        st["grid"], st["factor"] = np.linspace(0.0, 1.0, SIGN_GRID), np.zeros(SIGN_GRID)
    if kind == "observe":
        g = _observe_grid(case)
        sk = lib.md_alloc_sk_sphere_3d_x(0.0, g["dq"], (g["shells"] + 0.5) * g["dq"])
        npts = dict(density=g["points"], pairs=g["points"], itcf=g["itcf"], axes=g["axes"], sphere=sk.contents.N)
        st.update(g=g, sk=sk, centre=np.full(3, g["L"] / 2),
                  stats={k: lib.md_alloc_stats_x(n) for k, n in npts.items()},
                  out={})
        for k, n in npts.items():
            st["out"][k] = np.ctypeslib.as_array(st["stats"][k].contents.fxs[0], shape=(n,))
    _checked(lib.md_hip_synchronize_x(), "forces")
    return st


_BATCH_DT = 0.01
_SAMPLE = ("vbn", "trap", "pair", "virial", "vi_virial", "kinetic", "chains")


def run(state):
    lib, kind = _lib(), state["case"]["kind"]
    if kind == "batch":
        sys_ = state["systems"]
        _checked(lib.md_pimd_run_batch_x(state["ptrs"], state["cfgs"], len(sys_), state["case"]["steps"]), "batch")
        out = []
        for s in sys_:
            if not lib.md_simulation_sync_host_x(s.sim, 1):
                raise RuntimeError("sync failed")
            out.append(_state_view(s.sim)[:, 1:])
        return out
    s = state["s"]
    if kind in ("steps", "driver"):
        if kind == "steps":
            _checked(lib.md_pimd_run_steps_x(s.pimd, C.byref(state["cfg"]), state["case"]["steps"]), "steps")
        else:
            for _ in range(state["case"]["steps"]):
                s.step(state["dt"])
        if not lib.md_simulation_sync_host_x(s.sim, 1):
            raise RuntimeError("sync failed")
        b = _state_view(s.sim)
        return dict(x=b[:, 1:4], v=b[:, 4:7], f=b[:, 7:10])
    st = state["stats"]
    if kind == "sample":
        for v in st.values():
            v.contents.es[0] = 0.0
        rc = lib.md_pimd_calc_VBN_energy_x(s.pimd, st["vbn"])
        if s.kind == "trap":
            rc |= lib.md_pimd_calc_trap_energy_x(s.pimd, lib.cb["md_harmonic_trap_energy_x"], st["trap"])
        rc |= lib.md_pimd_calc_pair_energy_x(s.pimd, s.pair_energy_cb(), st["pair"])
        rc |= lib.md_pimd_calc_virial_energy_x(s.pimd, st["virial"])
        rc |= lib.md_pimd_fast_fill_ENk2_x(s.pimd, s.image)
        rc |= lib.md_pimd_calc_vi_virial_energy_x(s.pimd, st["vi_virial"], s.image)
        rc |= lib.md_calc_kinetic_x(s.sim, st["kinetic"])
        rc |= lib.md_calc_nhc_kinetic_x(s.sim, st["chains"])
        rc |= lib.md_pimd_calc_vi_sign_grid_x(s.pimd, SIGN_GRID, pyxmd.dptr(state["grid"]), pyxmd.dptr(state["factor"]))
        _checked(rc, "estimators")
        out = {k: np.array(v.contents.es[0]) for k, v in st.items()}
        out["factor"] = state["factor"]
        return out
    g = state["g"]
    for v in st.values():
        lib.md_reset_stats_f_x(v, 0.0)
    N, L, pi = s.N, g["L"], g["pi"]
    rc = lib.md_pimd_calc_density_distribution_x(s.pimd, st["density"], L / 2, 1, pyxmd.dptr(state["centre"]))
    rc |= lib.md_pimd_calc_pair_correlation_x(s.pimd, st["pairs"], L / 2, float(N), 1, 1)
    rc |= lib.md_pimd_calc_ITCF_x(s.pimd, st["itcf"], 0.0, L, pi)
    rc |= lib.md_pimd_calc_Sk_structure_x(s.pimd, st["axes"], g["dq"], g["dq"], 1)
    rc |= lib.md_pimd_calc_sphere_Sk_structure_x(s.pimd, st["sphere"], pi, state["sk"])
    _checked(rc, "observables")
    return state["out"]


# ------------------------------------------------------------------ work


def _step_work(c):
    """Bytes and FP64 operations of one MD step: the state (x, v, f, m and the
    chains) read and written once, the cycle-energy triangle written and read
    once; each pair (Gaussian 30, Ewald 90 with its share of the reciprocal
    sum), 60 per degree of freedom and chain link pair, the two recursions and
    the connection matrix (25 per entry)."""
    N, P, nb = c["N"], c["P"], c["N"] * c["P"]
    links = c.get("chain", 4)
    pair = 30 if c["system"] == "trap" else 90
    tri = N * (N + 1) / 2 if c["xi"] != 0 else N
    return dict(bytes=8.0 * (3 * nb * (6 + 5 * links) + nb + 2 * N * (N + 1) / 2),
                flops=P * N * (N - 1) / 2 * pair + 3 * nb * (30.0 * links + 15) + 4 * 25 * tri)


def work(case):
    if case["kind"] == "batch":
        w = [_step_work(dict(r, chain=case["chain"])) for r in _replicas(case)]
        return {k: case["steps"] * sum(x[k] for x in w) for k in ("bytes", "flops")}
    if case["kind"] in ("steps", "driver"):
        return {k: case["steps"] * v for k, v in _step_work(case).items()}
    N, nb = case["N"], case["N"] * case["P"]
    tri = N * (N + 1) / 2
    if case["kind"] == "sample":
        pair = 30 if case["system"] == "trap" else 90
        return dict(bytes=8.0 * (9 * nb + 2 * tri), flops=case["P"] * N * (N - 1) / 2 * pair + (4 + SIGN_GRID) * 25 * tri)
    g = _observe_grid(case)
    return dict(bytes=8.0 * (3 * nb + 2 * g["points"] + g["itcf"]),
                flops=10.0 * nb + 15.0 * N * (N - 1) + N * 40 * (3 * g["axes"] + 2 * 100))


# ----------------------------------------------------------------- exact
#
# The same quantities in plain numpy / torch FP64 from the definitions.  Bead
# arrays are [P, N, 3] (one bead slice a row).


def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _min_image(d, L):
    return d if L is None else d - L * torch.round(d / L)


def _pair_sums(c, x, want_energy, ewald):
    """Pair forces on every bead (raw, [P, N, 3]) and the pair energy summed over the slices."""
    P, N, _ = x.shape
    f, e = torch.zeros_like(x), 0.0
    L = None if c["system"] == "trap" else _shape(c)[0]
    chunk = max(1, int(3e7 // (N * N)))
    eye = torch.eye(N, dtype=torch.bool, device=x.device)
    for p0 in range(0, P, chunk):
        xs = x[p0:p0 + chunk]
        d = _min_image(xs[:, :, None, :] - xs[:, None, :, :], L)
        r2 = (d * d).sum(-1).masked_fill(eye, 1.0)
        if L is None:
            w = TRAP_G / (math.pi * TRAP_S ** 2) * torch.exp(-r2 / TRAP_S ** 2)
            g, u = w * 2 / TRAP_S ** 2, w
        else:  # alpha = 13.5 / L: the images beyond the nearest one are below erfc(6.7)
            r = torch.sqrt(r2)
            al = ewald["alpha"]
            u = torch.erfc(al * r) / r
            g = (u + 2 * al / math.sqrt(math.pi) * torch.exp(-(al * r) ** 2)) / r2
        g = g.masked_fill(eye, 0.0)
        f[p0:p0 + chunk] += (g[..., None] * d).sum(2)
        if want_energy:
            e += float(u.masked_fill(eye, 0.0).sum()) / 2
    if L is not None:
        for p in range(P):
            ph = [torch.exp(2j * math.pi / L * x[p, :, k, None] * ewald["m"][None, :]) for k in range(3)]
            a = ph[0][:, ewald["ix"]] * ph[1][:, ewald["iy"]]  # [N, columns]
            S = a.T @ ph[2]                                    # [columns, mz]
            W = ewald["coef"] * S.conj()
            U = ph[2] @ W.T                                    # [N, columns]
            V = ph[2] @ (W * ewald["m"]).T
            au = (a * U).imag
            q = 2 / L
            f[p, :, 0] += q * (au * ewald["mx"]).sum(1)
            f[p, :, 1] += q * (au * ewald["my"]).sum(1)
            f[p, :, 2] += q * (a * V).imag.sum(1)
            if want_energy:
                e += float((ewald["coef"] * (S.real ** 2 + S.imag ** 2 - N)).sum()) / (2 * math.pi)
        if want_energy:
            e -= math.pi / (ewald["alpha"] ** 2 * L ** 3) * N * (N - 1) / 2 * P
    return f, e


def _ewald_tables(c, dev):
    """k columns (half space) of the Ewald sum at alpha = 13.5 / L; coef = exp(-pi^2 G^2 / alpha^2) / (V G^2)."""
    L = _shape(c)[0]
    al = 13.5 / L
    M = int(6.5 * 13.5 / math.pi)
    m = torch.arange(-M, M + 1, device=dev, dtype=torch.float64)
    cols = [(i, j) for i in range(0, M + 1) for j in range(-M, M + 1) if (i > 0 or j >= 0) and i * i + j * j <= M * M]
    mx = torch.tensor([a for a, _ in cols], device=dev, dtype=torch.float64)
    my = torch.tensor([b for _, b in cols], device=dev, dtype=torch.float64)
    G2 = (mx[:, None] ** 2 + my[:, None] ** 2 + m[None] ** 2) / L ** 2
    keep = (G2 > 0) & ~((mx[:, None] == 0) & (my[:, None] == 0) & (m[None] < 0))
    G2 = torch.where(G2 > 0, G2, torch.ones_like(G2))
    coef = torch.where(keep, torch.exp(-math.pi ** 2 * G2 / al ** 2) / (G2 * L ** 3), torch.zeros_like(G2))
    return dict(alpha=al, m=m, ix=(mx + M).long(), iy=(my + M).long(), mx=mx, my=my, coef=2 * coef)


def _lse_rows(c):
    """L(n) = log sum_{m<n} exp(c[n, m] + L(m)), L(0) = 0, for a lower triangle c[1..N, 0..N-1]."""
    N = c.shape[0] - 1
    L = np.zeros(N + 1, dtype=c.dtype)
    for n in range(1, N + 1):
        t = c[n, :n] + L[:n]
        top = t.max()
        L[n] = top + math.log(np.exp((t - top).astype(np.float64)).sum())
    return L


class _Exchange:
    """Cycle energies, recursions and the connection matrix of one
    configuration.  beta V_B is large against the differences that matter, so
    the energies and exponents are summed in extended precision."""

    def __init__(self, c, x):
        self.P, self.N, _ = x.shape
        N, P = self.N, self.P
        self.L, self.T, _ = _shape(c)
        self.box = self.L if c["system"] == "ueg" else None
        self.beta = 1.0 / self.T
        self.om = math.sqrt(P) / self.beta
        self.x = x
        half = 0.5 * self.om ** 2
        inner = half * (_min_image(x[1:] - x[:-1], self.box) ** 2).sum((0, 2))
        self.d = _min_image(x[-1][:, None] - x[0][None], self.box)  # bead P of row, bead 1 of column
        self.close = (half * (self.d ** 2).sum(-1)).cpu().numpy()
        eint = inner.cpu().numpy()
        link = np.zeros(N, dtype=np.longdouble)
        link[1:] = np.cumsum((eint[:-1] + np.diagonal(self.close, 1)).astype(np.longdouble))
        # E[n, m]: the cycle of particles m+1 .. n (1-based), n > m
        self.E = np.zeros((N + 1, N + 1), dtype=np.longdouble)
        self.E[1:, :N] = link[:, None] - link[None, :] + eint[:, None] + self.close
        self.solve(c["xi"])

    def coef(self, xi):
        N = self.N
        n, m = np.arange(N + 1)[:, None], np.arange(N + 1)[None, :]
        with np.errstate(divide="ignore", invalid="ignore"):
            c = -self.beta * self.E - np.log(np.maximum(n, 1).astype(np.longdouble))
            c = c + (n - m - 1) * np.log(np.longdouble(xi)) if xi != 0 else np.where(n - m == 1, c, -np.inf)
        return np.where(n > m, c, -np.inf)

    def solve(self, xi):
        self.c = self.coef(xi)
        self.Lf = _lse_rows(self.c)
        self.Rb = _lse_rows(self.c[::-1, ::-1].T.copy())[::-1]

    def connection(self):
        """G[l, j]: probability that bead P of l links to bead 1 of j (0-based)."""
        N, LN = self.N, self.Lf[-1]
        G = np.exp((self.c[1:, :N] + self.Lf[None, :N] + self.Rb[1:, None] - LN).astype(np.float64))
        i = np.arange(N - 1)
        G[i, i + 1] = -np.expm1(np.minimum(0.0, (self.Lf[1:N] + self.Rb[1:N] - LN).astype(np.float64)))
        return torch.from_numpy(G).to(self.x)

    def force(self):
        x, k = self.x, self.om ** 2
        f = torch.zeros_like(x)
        step = _min_image(x[1:] - x[:-1], self.box)
        f[:-1] += k * step
        f[1:] -= k * step
        G = self.connection()
        f[-1] -= k * (G[..., None] * self.d).sum(1)
        f[0] += k * (G[..., None] * self.d).sum(0)
        return f

    def mean(self, B):
        """res(N) of res(n) = sum_m w(n, m) (res(m) - B(n, m)) / sum_m w(n, m)."""
        res = np.zeros(self.N + 1)
        for n in range(1, self.N + 1):
            w = np.exp((self.c[n, :n] + self.Lf[:n] - self.Lf[n]).astype(np.float64))
            res[n] = (w * (res[:n] - B[n, :n].astype(np.float64))).sum() / w.sum()
        return res[-1]

    def link_virial(self):
        """E2[n, m] of md_pimd_fast_fill_ENk2_x: 1/2 m w^2 (x_a - x_b).(x_a - x_c) over a cycle's links."""
        N, h = self.N, 0.5 * self.om ** 2
        x = self.x
        d1 = _min_image(x[0][:, None] - x[0][None], self.box)      # (a, c): beads 1
        e = (h * (-self.d.transpose(0, 1) * d1).sum(-1)).cpu().numpy()  # [a, c]: a's bead 1, c's beads P and 1
        link = np.zeros(N, dtype=np.longdouble)
        link[1:] = np.cumsum(np.diagonal(e, 1).astype(np.longdouble))
        E2 = np.zeros((N + 1, N + 1))
        E2[1:, :N] = (link[:, None] - link[None, :]).astype(np.float64) + e
        return E2


def _forces(c, x, ewald):
    f = _pair_sums(c, x, False, ewald)[0] / c["P"]
    if c["system"] == "trap":
        f = f - x / c["P"]
    return f + _Exchange(c, x).force()


class _Chains:
    """Massive Nose-Hoover chains of M links, the velocity-Verlet halves of md_update_nhc_VV3_1_x / _2_x (m = 1)."""

    def __init__(self, c, x, T, h):
        self.M, self.T, self.h = c["chain"], T, h
        om = math.sqrt(c["P"]) * T
        self.Q = T / om ** 2
        self.vt = [torch.ones_like(x) for _ in range(self.M)]

    def accel(self, v):
        a = [(v * v - self.T) / self.Q]
        return a + [(self.Q * u * u - self.T) / self.Q for u in self.vt[:-1]]

    def scale(self, u, a, up, h):
        return u * torch.exp(-h * up) + h * a * torch.exp(-0.5 * h * up)

    def odd(self, a):
        for k in range(1, self.M, 2):
            up = self.vt[k + 1] if k + 1 < self.M else torch.zeros_like(self.vt[k])
            self.vt[k] = self.scale(self.vt[k], a[k], up, 0.5 * self.h)

    def first(self, x, v, f):
        a = self.accel(v)
        v = self.scale(v, f, self.vt[0], 0.5 * self.h)
        self.odd(a)
        x = x + self.h * v
        a = self.accel(v)
        for k in range(0, self.M, 2):
            self.vt[k] = self.scale(self.vt[k], a[k], self.vt[k + 1], self.h)
        return x, v

    def second(self, v, f):
        v = self.scale(v, f, self.vt[0], 0.5 * self.h)
        self.odd(self.accel(v))
        return v


def _wrap(x, L):
    return torch.where(x < 0, x + L, torch.where(x > L, x - L, x))


def _trajectory(c, seed, steps, dt):
    x, v = (torch.from_numpy(a.transpose(1, 0, 2).copy()).to(_dev()) for a in _beads(c, seed))
    L, T, _ = _shape(c)
    ew = _ewald_tables(c, _dev()) if c["system"] == "ueg" else None
    chains = _Chains(c, x, T, dt)
    f = _forces(c, x, ew)
    for _ in range(steps):
        x, v = chains.first(x, v, f)
        if c["system"] == "ueg":
            x = _wrap(x, L)
        f = _forces(c, x, ew)
        v = chains.second(v, f)
    return {k: a.transpose(0, 1).reshape(-1, 3).cpu().numpy() for k, a in (("x", x), ("v", v), ("f", f))}


def _exact_sample(c, seed):
    x, v = (torch.from_numpy(a.transpose(1, 0, 2).copy()).to(_dev()) for a in _beads(c, seed))
    N, P = c["N"], c["P"]
    L, T, dt = _shape(c)
    ew = _ewald_tables(c, _dev()) if c["system"] == "ueg" else None
    pf, pe = _pair_sums(c, x, True, ew)
    ex = _Exchange(c, x)
    f = pf / P + ex.force()
    if c["system"] == "trap":
        f = f - x / P
    out = dict(vbn=ex.mean(ex.E) + 3 * N * P * T / 2, pair=pe / P,
               trap=float((x * x).sum()) / (2 * P) if c["system"] == "trap" else 0.0,
               virial=float((-(x - L / 2) * f).sum()) / 2,
               vi_virial=ex.mean(ex.link_virial()) + 3 * N * T / 2
               + float((-_min_image(x[1:] - x[0], ex.box) * f[1:]).sum()) / 2,
               kinetic=float((v * v).sum()) / 2)
    out["chains"] = 3 * N * P * c["chain"] * 0.5 * _Chains(c, x[:1, :1], T, dt).Q
    LN = ex.Lf[-1]
    fac = []
    for xi in np.linspace(0.0, 1.0, SIGN_GRID):
        fac.append(math.exp(float(_lse_rows(ex.coef(float(xi)))[-1] - LN)))
    out["factor"] = np.array(fac)
    return {k: np.array(u, dtype=np.float64) for k, u in out.items()}


def _sphere_q(g):
    """First q vector of each |q| shell of the cube 0, dq, 2 dq, ..., by |q|."""
    axis, q = [], 0.0
    while q <= (g["shells"] + 0.5) * g["dq"]:
        axis.append(q)
        q += g["dq"]
    qs, vec = [], []
    for a in axis:
        for b in axis:
            for d in axis:
                q = math.sqrt(a * a + b * b + d * d)
                if q < 1e-4 or any(abs(q - k) < 1e-4 for k in qs):
                    continue
                qs.append(q)
                vec.append((a, b, d))
    order = np.argsort(np.array(qs), kind="stable")
    return np.array(vec)[order]


def _exact_observe(c, seed):
    x = _beads(c, seed)[0].transpose(1, 0, 2)  # [P, N, 3]
    N, P = c["N"], c["P"]
    g = _observe_grid(c)
    L = g["L"]

    def image(d):
        return d - L * np.round(d / L)

    def counts(r, points, width):
        b = (r / width).astype(np.int64)
        return np.bincount(b[b < points], minlength=points).astype(np.float64)

    w = L / 2 / g["points"]
    r = np.sqrt((image(x - L / 2) ** 2).sum(-1)).ravel()
    out = dict(density=counts(r, g["points"], w) / P)
    d = image(x[0][:, None] - x[0][None])
    r = np.sqrt((d * d).sum(-1))[~np.eye(N, dtype=bool)]
    out["pairs"] = counts(r, g["points"], w) / N
    n = int(math.sqrt(g["itcf"]))
    i1, i2 = ((x[p, :, 0] / (L / n)).astype(np.int64) for p in (0, g["pi"] - 1))
    idx = np.clip(i1[:, None] * n + i2[None], 0, g["itcf"] - 1)
    out["itcf"] = np.bincount(idx.ravel(), minlength=g["itcf"]).astype(np.float64) / P
    q = g["dq"] * np.arange(1, g["axes"] + 1)
    ph = np.exp(1j * x[0][None] * q[:, None, None]).sum(1)  # [q, dimension]
    out["axes"] = (np.abs(ph) ** 2).sum(1) / 3 / N
    qv = _sphere_q(g)
    a, b = (np.exp(1j * (qv @ x[p].T)).sum(1) for p in (0, g["pi"] - 1))
    out["sphere"] = (a.real * b.real + a.imag * b.imag) / N
    return out


def exact(case, seed):
    if case["kind"] == "batch":
        out = []
        for i, r in enumerate(_replicas(case)):
            t = _trajectory(dict(r, chain=case["chain"]), seed + 1000 * i, case["steps"], _BATCH_DT)
            out.append(np.concatenate([t["x"], t["v"], t["f"]], 1))
        return out
    if case["kind"] == "sample":
        return _exact_sample(case, seed)
    if case["kind"] == "observe":
        return _exact_observe(case, seed)
    return _trajectory(case, seed, case["steps"], _shape(case)[2])
