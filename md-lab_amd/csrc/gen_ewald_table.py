"""Generates ewald_table.h: piecewise polynomials of the Ewald real-space
kernels on 0 <= x < 53/8, h(x) = erfc(x) + 2x/sqrt(pi) exp(-x^2) of the force
and erfc(x) of the energy.

Interval i covers [i/8, (i+1)/8); inside it h = sum_k c[i][k] y^k with
y = 16 x - (2 i + 1) in [-1, 1].  The coefficients interpolate h at the 10
Chebyshev nodes of the interval, computed at 40 digits (mpmath), and are
rounded once to FP64; the FP64 Horner evaluation then has max abs error
1.1e-16 on the whole range (h(0) = 1, so this is the rounding floor).

Run:  python md-lab_amd/csrc/gen_ewald_table.py > md-lab_amd/csrc/ewald_table.h
"""
import mpmath as mp

mp.mp.dps = 40
NINT, DEG, INV_W = 53, 9, 8


def h(x):
    return mp.erfc(x) + 2 * x / mp.sqrt(mp.pi) * mp.exp(-x * x)


def table(h):
    nodes = [mp.cos(mp.pi * (k + mp.mpf(1) / 2) / (DEG + 1)) for k in range(DEG + 1)]
    V = mp.matrix([[t ** j for j in range(DEG + 1)] for t in nodes])
    rows = []
    worst = 0.0
    for i in range(NINT):
        a = mp.mpf(i) / INV_W
        ys = [h(a + (t + 1) / (2 * INV_W)) for t in nodes]
        c = mp.lu_solve(V, mp.matrix(ys))
        cd = [float(c[j]) for j in range(DEG + 1)]
        for s in range(81):
            t = -1 + s / 40.0
            acc = 0.0
            for j in range(DEG, -1, -1):
                acc = acc * t + cd[j]
            worst = max(worst, abs(acc - float(h(a + (mp.mpf(t) + 1) / (2 * INV_W)))))
        rows.append(cd)
    return rows, worst


def main():
    force, ef = table(h)
    energy, ee = table(mp.erfc)
    print("// Generated by gen_ewald_table.py -- do not edit.")
    print(f"// h(x) = erfc(x) + 2x/sqrt(pi) exp(-x^2) (kEwTab) and erfc(x) (kEwTabE), {NINT} intervals of width 1/{INV_W}, degree {DEG};")
    print(f"// max abs errors of the FP64 Horner evaluation {ef:.2e} and {ee:.2e}.")
    print("#pragma once")
    print(f"constexpr int kEwTabIntervals = {NINT};")
    print(f"constexpr int kEwTabStride = {DEG + 1};")
    print(f"constexpr double kEwTabInvWidth = {INV_W}.0;")
    for name, rows in (("kEwTab", force), ("kEwTabE", energy)):
        print(f"__device__ __constant__ double {name}[{NINT * (DEG + 1)}] = {{")
        for cd in rows:
            print("    " + ", ".join(repr(v) for v in cd) + ",")
        print("};")


if __name__ == "__main__":
    main()
