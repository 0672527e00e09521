// Per-bead-slice pair forces and energies (md_pimd_x.c:1527-1824) for the
// Gaussian, periodic Gaussian and 3-D Ewald interactions
// (md_simulation_x.c:166-346, md_statistics_x.c:340-396).
//
// Kernel shapes (gfx950, wave64):
//  * k_pair_tiles / k_ewald_real: one wave per (slice, tile I <= tile J) of
//    64 x 64 beads; lane t meets partner (t + s) mod 64 at rotation step s,
//    so each pair is evaluated once and both reactions accumulate without
//    atomics (i in registers, j in LDS).  Result per bead:
//    f_i += sum_{j != i} F(x_i, x_j) / m_{max(i,j)} / P, i.e. the reference's
//    l > l' loop with Newton's third law (md_pimd_x.c:1669-1673).
//  * Ewald real space sums the images within r_c = x_cut/alpha (x_cut 5.25
//    by default, g_ewald_xcut; the reference sums its whole image cube
//    |n_d| <= n_sum, whose other terms are below erfc(x_cut) of the near
//    ones).  k_ewald_real evaluates the force kernel
//    from a piecewise-polynomial table in LDS; k_pair_tiles covers the R/NI
//    splits, energies and the general cube-clipped case.
//  * Ewald reciprocal space uses per-slice structure factors
//    S(k) = sum_l exp(i k.x_l) over half of the k set (k_phase, k_sk_mfma,
//    k_recip_force_mfma, k_recip_force_energy, k_recip_energy).
//  * When the reference's own Ewald parameters are converged, the same sum is
//    evaluated with the engine's split (plan_ewald).
#include <algorithm>
#include <climits>
#include <cmath>
#include <map>
#include <vector>

#include "ewald_table.h"
#include "xmd_device.h"
#include "xmd_internal.h"

namespace xmd {

__device__ __forceinline__ int pf_img_count(double x, double L) {
  int c = (int)(fabs(x) / L);
  if (x > L) return -c;
  if (x < 0) return c + 1;
  return 0;
}

__device__ __forceinline__ double pf_min_image(double a, double L) {
  double s = a + L / 2;
  s += L * pf_img_count(s, L);
  return s - L / 2;
}

struct PairParams {
  double L[3];
  double g, s2;        // Gaussian: strength, range^2
  double q, alpha;     // Ewald: charge product, splitting
  double rc2;          // real-space cutoff^2
  int nsum;            // Ewald cube half-width
  double P;            // beads (pair forces are divided by P)
  double he[8];        // helium: eps, A, alpha, C6, C8, C10, D, r_m
  double xcut;         // Ewald series cutoff in units of the split (real r_c = xcut / alpha)
};

// Real-space Ewald contribution of one raw separation (p1 - p2) to the
// force (accumulated into f) and/or the energy.  skip_min / only_min select
// the reference's R and NI splits (md_simulation_x.c:295-346).
template <bool FORCE, bool ENERGY>
__device__ __forceinline__ void ewald_real(double dx, double dy, double dz, const PairParams &pp, int skip_min,
                                           int only_min, double invm, double &fx, double &fy, double &fz,
                                           double &e) {
  const double al = pp.alpha, q = pp.q;
  const double c_gauss = q * 2 * al / sqrt(M_PI);
  if (only_min) {
    double rx = pf_min_image(dx, pp.L[0]), ry = pf_min_image(dy, pp.L[1]), rz = pf_min_image(dz, pp.L[2]);
    double R = sqrt(rx * rx + ry * ry + rz * rz);
    if (FORCE) {
      double w = c_gauss * exp(-al * al * R * R) / (R * R) + q * erfc(al * R) / (R * R * R);
      fx += rx * w * invm;
      fy += ry * w * invm;
      fz += rz * w * invm;
    }
    if (ENERGY) e += q * erfc(al * R) / R;
    return;
  }
  const double rc = sqrt(pp.rc2);
  double mx = 0, my = 0, mz = 0;
  if (skip_min) {
    mx = fabs(pf_min_image(-dx, pp.L[0]));
    my = fabs(pf_min_image(-dy, pp.L[1]));
    mz = fabs(pf_min_image(-dz, pp.L[2]));
  }
  const int n = pp.nsum;
  int ax = max(-n, (int)ceil((dx - rc) / pp.L[0])), bx = min(n, (int)floor((dx + rc) / pp.L[0]));
  int ay = max(-n, (int)ceil((dy - rc) / pp.L[1])), by = min(n, (int)floor((dy + rc) / pp.L[1]));
  int az = max(-n, (int)ceil((dz - rc) / pp.L[2])), bz = min(n, (int)floor((dz + rc) / pp.L[2]));
  for (int i = ax; i <= bx; ++i) {
    double rx = dx - i * pp.L[0];
    double rx2 = rx * rx;
    if (rx2 > pp.rc2) continue;
    for (int j = ay; j <= by; ++j) {
      double ry = dy - j * pp.L[1];
      double rxy2 = rx2 + ry * ry;
      if (rxy2 > pp.rc2) continue;
      for (int k = az; k <= bz; ++k) {
        double rz = dz - k * pp.L[2];
        double R2 = rxy2 + rz * rz;
        if (R2 > pp.rc2) continue;
        if (skip_min && fabs(fabs(rx) - mx) < 1e-4 && fabs(fabs(ry) - my) < 1e-4 && fabs(fabs(rz) - mz) < 1e-4)
          continue;
        double R = sqrt(R2);
        double ec = erfc(al * R);
        if (FORCE) {
          double w = c_gauss * exp(-al * al * R * R) / (R * R) + q * ec / (R * R * R);
          fx += rx * w * invm;
          fy += ry * w * invm;
          fz += rz * w * invm;
        }
        if (ENERGY) e += q * ec / R;
      }
    }
  }
}

// (1 + 2x) exp(x^2) erfc(x) on 0 <= x <= 6.5 as a degree-20 Chebyshev series
// in s(y), y = (x - 3)/(x + 3) (the transform of Shepherd & Laframboise,
// Math. Comp. 36 (1981) 249); coefficients fitted here at 40 digits,
// max relative error 4.4e-16 in FP64 evaluation.
__device__ __constant__ double kErfcxCheb[21] = {
    1.2007410605728304,     0.065198450961816964,   -0.092409466117412367,  0.034405477918768981,
    -0.0076296298533925291, 0.0010403531055794199,  -6.3272734583294028e-05, -4.6011890721509966e-06,
    1.0119739574626279e-06, 9.9431600651180912e-09, -1.3295432865350941e-08, -9.4590207011356631e-12,
    1.9114449190078913e-10, 3.6405902241118161e-12, -2.8882712550806537e-12, -1.780186683919635e-13,
    3.9543737314097065e-14, 5.4923737447575301e-15, -3.4794118944385234e-16, -1.0306316042149898e-16,
    -1.3876025693966222e-17};
constexpr double kErfcxY1 = 0.36842105263157893;  // y at x = 6.5

// erfc(x) given e = exp(-x^2), 0 <= x <= 6.5.  One reciprocal serves both
// the transform y = (x-3)/(x+3) and the final division by (1 + 2x).
__device__ __forceinline__ double erfc_cheb(double x, double e) {
  const double d1 = x + 3.0, d2 = 1.0 + 2.0 * x;
  const double a = d1 * d2;
  double r = __builtin_amdgcn_rcp(a);
  r = fma(fma(-a, r, 1.0), r, r);
  r = fma(fma(-a, r, 1.0), r, r);
  const double y = (x - 3.0) * (d2 * r);
  const double sc = 2.0 / (kErfcxY1 + 1.0), sh = (kErfcxY1 - 1.0) / (kErfcxY1 + 1.0);
  const double t = sc * y - sh, t2 = 2.0 * t;
  double b1 = 0.0, b2 = 0.0;
#pragma unroll
  for (int k = 20; k >= 1; --k) {
    const double b0 = fma(t2, b1, kErfcxCheb[k] - b2);
    b2 = b1;
    b1 = b0;
  }
  const double c = fma(t, b1, kErfcxCheb[0] - b2);
  return e * (c * (d1 * r));
}

__device__ __forceinline__ double erfc_from_exp(double x, double e) {
  if (x > 6.5) return erfc(x);
  return erfc_cheb(x, e);
}

// One real-space image r (= p1 - image of p2) at distance R: force factor
// (q 2 alpha exp(-alpha^2 R^2)/(sqrt(pi) R^2) + q erfc(alpha R)/R^3) as at
// md_simulation_x.c:288-289, energy q erfc(alpha R)/R (md_statistics_x.c:393).
// INRANGE: alpha R <= 6.5 is guaranteed by the caller (images inside the
// cutoff x_cut/alpha, x_cut <= 6.5).
template <bool FORCE, bool ENERGY, bool INRANGE = false>
__device__ __forceinline__ void ewald_image(double rx, double ry, double rz, double R2, const PairParams &pp,
                                            double &gx, double &gy, double &gz, double &e) {
  const double invR = rsqrt(R2);
  const double R = R2 * invR;
  const double x = pp.alpha * R;
  const double ex = exp(-x * x);
  const double ec = INRANGE ? erfc_cheb(x, ex) : erfc_from_exp(x, ex);
  if (FORCE) {
    const double i2 = invR * invR;
    const double w = i2 * ((pp.q * 2 * pp.alpha / sqrt(M_PI)) * ex + pp.q * ec * invR);
    gx += rx * w;
    gy += ry * w;
    gz += rz * w;
  }
  if (ENERGY) e += pp.q * ec * invR;
}

// Images of one pair within r_c when r_c < sqrt(2) L: every such image takes
// per dimension one of the three nearest periodic copies a (minimum image),
// b = a -+ L, c = a +- L, and at most one dimension takes c.  Candidates are
// numbered 0..19 (0-7: {a,b}^3, 8-11/12-15/16-19: c in x/y/z); each lane
// builds the bit mask of its candidates inside r_c and the wave walks the
// set bits, so a step costs the largest per-lane image count rather than
// all candidates any lane needs.  skip_min drops (a,a,a) (the R split),
// only_min keeps only it (the NI split).
template <bool FORCE, bool ENERGY>
__device__ __forceinline__ void ewald_real_near(double dx, double dy, double dz, const PairParams &pp, int skip_min,
                                                int only_min, double &gx, double &gy, double &gz, double &e) {
  const double ax = pf_min_image(dx, pp.L[0]), ay = pf_min_image(dy, pp.L[1]), az = pf_min_image(dz, pp.L[2]);
  if (only_min) {
    ewald_image<FORCE, ENERGY>(ax, ay, az, ax * ax + ay * ay + az * az, pp, gx, gy, gz, e);
    return;
  }
  const double bx = ax - copysign(pp.L[0], ax), by = ay - copysign(pp.L[1], ay), bz = az - copysign(pp.L[2], az);
  const double cx = ax + copysign(pp.L[0], ax), cy = ay + copysign(pp.L[1], ay), cz = az + copysign(pp.L[2], az);
  const double ax2 = ax * ax, ay2 = ay * ay, az2 = az * az;
  const double bx2 = bx * bx, by2 = by * by, bz2 = bz * bz;
  const double cx2 = cx * cx, cy2 = cy * cy, cz2 = cz * cz;
  const double rc2 = pp.rc2;
  unsigned mask = 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const double R2 = ((q & 1) ? bx2 : ax2) + ((q & 2) ? by2 : ay2) + ((q & 4) ? bz2 : az2);
    mask |= (R2 <= rc2 ? 1u : 0u) << q;
  }
  if (skip_min) mask &= ~1u;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const double yx = (u & 1) ? by2 : ay2, zx = (u & 2) ? bz2 : az2;  // c in x
    const double xy = (u & 1) ? bx2 : ax2, zy = (u & 2) ? bz2 : az2;  // c in y
    const double xz = (u & 1) ? bx2 : ax2, yz = (u & 2) ? by2 : ay2;  // c in z
    mask |= (cx2 + yx + zx <= rc2 ? 1u : 0u) << (8 + u);
    mask |= (xy + cy2 + zy <= rc2 ? 1u : 0u) << (12 + u);
    mask |= (xz + yz + cz2 <= rc2 ? 1u : 0u) << (16 + u);
  }
  while (mask) {
    const int q = __builtin_ctz(mask);
    mask &= mask - 1;
    const int cdim = q < 8 ? -1 : (q - 8) >> 2;
    const int u = q < 8 ? q : ((q - 8) & 3);
    const int xb = u & 1;
    const int yb = cdim == 0 ? (u & 1) : ((u >> 1) & 1);
    const int zb = cdim < 0 ? ((u >> 2) & 1) : ((u >> 1) & 1);
    const double rx = cdim == 0 ? cx : (xb ? bx : ax);
    const double ry = cdim == 1 ? cy : (yb ? by : ay);
    const double rz = cdim == 2 ? cz : (zb ? bz : az);
    ewald_image<FORCE, ENERGY, true>(rx, ry, rz, rx * rx + ry * ry + rz * rz, pp, gx, gy, gz, e);
  }
}

// Force (raw, not divided by mass) on bead i from bead j and/or pair energy.
template <int MODE, bool ENERGY, bool NEAR>
__device__ __forceinline__ void pair_term(double dx, double dy, double dz, const PairParams &pp, double &gx,
                                          double &gy, double &gz, double &e) {
  if (MODE == PK_GAUSS || MODE == PK_PGAUSS) {
    if (MODE == PK_PGAUSS) {
      dx = pf_min_image(dx, pp.L[0]);
      dy = pf_min_image(dy, pp.L[1]);
      dz = pf_min_image(dz, pp.L[2]);
    }
    const double d = sqrt(dx * dx + dy * dy + dz * dz);
    const double w = (pp.g / (M_PI * pp.s2)) * exp(-d * d / pp.s2);
    if (ENERGY) {
      e += w;
    } else {
      gx += w * (2 * dx) / pp.s2;
      gy += w * (2 * dy) / pp.s2;
      gz += w * (2 * dz) / pp.s2;
    }
  } else if (MODE == PK_LJ || MODE == PK_HE) {
    dx = pf_min_image(dx, pp.L[0]);
    dy = pf_min_image(dy, pp.L[1]);
    dz = pf_min_image(dz, pp.L[2]);
    const double r = sqrt(dx * dx + dy * dy + dz * dz);
    if (MODE == PK_LJ) {
      // 4 (r^-12 - r^-6); force factor 48 r^-14 - 24 r^-8 (md_simulation_x.c:116-122,
      // md_statistics_x.c:317-320)
      const double i2 = 1.0 / (r * r), i6 = i2 * i2 * i2;
      if (ENERGY) {
        e += 4 * (i6 * i6 - i6);
      } else {
        const double w = (48 * i6 - 24) * i6 * i2;
        gx += dx * w;
        gy += dy * w;
        gz += dz * w;
      }
    } else {
      // Aziz-type helium potential with damping F(x) below x = D, x = r / r_m
      // (md_simulation_x.c:385-399, md_statistics_x.c:496-506)
      const double eps = pp.he[0], A = pp.he[1], al = pp.he[2], C6 = pp.he[3], C8 = pp.he[4], C10 = pp.he[5],
                   D = pp.he[6], rm = pp.he[7];
      const double x = r / rm, ix = 1.0 / x, ix2 = ix * ix;
      const double ix6 = ix2 * ix2 * ix2, ix8 = ix6 * ix2, ix10 = ix8 * ix2;
      const bool damp = x < D;
      double F = 1.0;
      if (damp) {
        const double u = D * ix - 1;
        F = exp(-u * u);
      }
      const double disp = C6 * ix6 + C8 * ix8 + C10 * ix10;
      const double rep = A * exp(-al * x);
      if (ENERGY) {
        e += eps * (rep - disp * F);
      } else {
        double mult = al * rep - (6 * C6 * ix6 + 8 * C8 * ix8 + 10 * C10 * ix10) * ix * F;
        if (damp) mult += disp * F * 2 * D * (D * ix - 1) * ix2;
        const double w = eps * mult / (r * rm);
        gx += dx * w;
        gy += dy * w;
        gz += dz * w;
      }
    }
  } else if (MODE == PK_EWALD_R2) {
    if (ENERGY) {
      const double rx = pf_min_image(dx, pp.L[0]), ry = pf_min_image(dy, pp.L[1]), rz = pf_min_image(dz, pp.L[2]);
      const double R = sqrt(rx * rx + ry * ry + rz * rz);
      e += -pp.q * erf(pp.alpha * R) / R;
    }
  } else if (NEAR) {
    ewald_real_near<!ENERGY, ENERGY>(dx, dy, dz, pp, MODE == PK_EWALD_R, MODE == PK_EWALD_NI, gx, gy, gz, e);
  } else {
    ewald_real<!ENERGY, ENERGY>(dx, dy, dz, pp, MODE == PK_EWALD_R, MODE == PK_EWALD_NI, 1.0, gx, gy, gz, e);
  }
}

// a / b for many a by one divisor: y = RN(1/b), two residual corrections.
// After the first the quotient is within one ulp, and with a correctly rounded
// y the second then gives RN(a/b) (Markstein's theorem), provided no residual
// underflows or overflows: for 2^-960 <= |a| <= 2^960 (or a = 0) and a divisor
// within 2^+-60 of one.  A smaller |a| gives a quotient below 2^-900.
__device__ __forceinline__ double const_div(double a, double b, double y) {
  double q = a * y;
  q = fma(fma(-q, b, a), y, q);
  return fma(fma(-q, b, a), y, q);
}

// Force on a bead from GAUSS_U others: (dx, dy, dz)[u] -> the terms of
// pair_term<MODE, false>, to the last bit where they are normal numbers (below
// 2e-308 within one of their last places).  The chains (sqrt, exp, divisions)
// are free of branches so that they interleave, and the divisions by s^2 are
// const_div's for pairs at any distance: the exponent needs no lower bound
// (below 2^-900 its exp is 1), and the dividends of the force, which run down
// to the smallest subnormal at 27 ranges, are scaled by 2^120 and the quotients
// back.  Their upper bound follows from gauss_quick, so that only a wave with
// an infinite or undefined distance repeats its terms plainly.  Issue bound: a
// rotation was 160 FP64 instructions, 65 of them five divisions, which are 26
// now (2, 3 and 4 others at a time measure the same, 2 has the smallest code).
// Tiles and their reduction, us, plain divisions -> here: N=600 P=64 trap 91 ->
// 73, periodic 128 -> 108, N=512 P=32 52 -> 46, N=256 P=64 37 -> 34.6, N=24 P=16
// 18.2 -> 15, the same for ranges from 0.02 to 0.5.  (Unscaled dividends bounded by
// 2^-900, a wave with a smaller one repeating its terms plainly, took 74, 109, 47,
// 35 and 15 at a range of 0.5, but 125, 161, 73, 51 and 21 from 0.2 down, where
// most waves hold a pair 25 .. 27 ranges apart or more.)
constexpr int GAUSS_U = 2;

// Whether the quotients stay in range for every finite distance: |force| is at
// most pre 2 d e^(-d^2/s^2) / s^2, d e^(-d^2/s^2) < s.  Others (ranges beyond
// 2^+-30, strengths beyond 2^800) take the general loop with plain divisions.
__device__ __forceinline__ bool gauss_quick(double s2, double pre) {
  return s2 >= 0x1p-60 && s2 <= 0x1p60 && fabs(pre) <= 0x1p800;
}

template <int MODE>
__device__ __forceinline__ void gauss_terms(double *dx, double *dy, double *dz, const PairParams &pp, double pre,
                                            double y) {
  double a[GAUSS_U];
  bool in = true;
#pragma unroll
  for (int u = 0; u < GAUSS_U; ++u) {
    if (MODE == PK_PGAUSS) {
      dx[u] = pf_min_image(dx[u], pp.L[0]);
      dy[u] = pf_min_image(dy[u], pp.L[1]);
      dz[u] = pf_min_image(dz[u], pp.L[2]);
    }
    const double d = sqrt(dx[u] * dx[u] + dy[u] * dy[u] + dz[u] * dz[u]);
    a[u] = -d * d;
    in = in && a[u] >= -0x1p900;
  }
  double qx[GAUSS_U], qy[GAUSS_U], qz[GAUSS_U];
#pragma unroll
  for (int u = 0; u < GAUSS_U; ++u) {
    const double w = pre * exp(const_div(a[u], pp.s2, y));
    qx[u] = const_div(w * (2 * dx[u]) * 0x1p120, pp.s2, y) * 0x1p-120;
    qy[u] = const_div(w * (2 * dy[u]) * 0x1p120, pp.s2, y) * 0x1p-120;
    qz[u] = const_div(w * (2 * dz[u]) * 0x1p120, pp.s2, y) * 0x1p-120;
  }
  if (!__all(in)) {
#pragma unroll 1  // (unrolled, more waves fit a SIMD: no faster, and a batch's reciprocal kernels wait 10 us for room)
    for (int u = 0; u < GAUSS_U; ++u) {
      const double w = pre * exp(a[u] / pp.s2);
      qx[u] = w * (2 * dx[u]) / pp.s2;
      qy[u] = w * (2 * dy[u]) / pp.s2;
      qz[u] = w * (2 * dz[u]) / pp.s2;
    }
  }
#pragma unroll
  for (int u = 0; u < GAUSS_U; ++u) {
    dx[u] = qx[u];
    dy[u] = qy[u];
    dz[u] = qz[u];
  }
}

// A tile's partial sum into its slot, or (add = P > 0: one tile, whose slots
// lie as F does) into F as k_reduce_tiles would add it.
__device__ __forceinline__ void put_tile(double *slot, double v, double add) {
  if (add > 0.0)
    *slot += (0.0 + v) / add;
  else
    *slot = v;
}

// Symmetric tile-pair kernel.  One 64-lane workgroup per (slice, I, J),
// I <= J (64-bead tiles of one slice).  Lane t owns bead i = 64 I + t; the
// J tile sits in LDS together with its reaction accumulators.  At rotation
// step s lane t meets partner (t + s) mod 64, so within a step every lane
// updates a different reaction slot and no atomics are needed.  Each pair
// is evaluated once (Newton's third law), divided by the mass of the
// higher-index bead as in md_pimd_x.c:1669-1673.
//
// Output: per-bead partial sums in Fpart[(slot*3 + d)*nb + bead], where
// slot is the other tile of the pair, so every slot is written exactly once
// (a wave writes 64 consecutive doubles) and k_reduce_tiles sums them in a
// fixed order (deterministic forces).
template <int MODE, bool ENERGY, bool NEAR>
__device__ __forceinline__ void k_pair_tiles_body(int bx, const double *__restrict__ X, const double *__restrict__ M,
                                                   double *__restrict__ Fpart, double *__restrict__ Epart,
                                                   const int2 *__restrict__ tiles, int N, int nb, int T, int ntp,
                                                   PairParams pp, double add = 0.0) {
  __shared__ double jx[64], jy[64], jz[64], jm[64], rx[64], ry[64], rz[64];
  const int item = bx;
  const int slice = item / ntp;
  const int2 IJ = tiles[item - slice * ntp];
  const int I = IJ.x, J = IJ.y;
  const int t = threadIdx.x;
  const int base = slice * N;
  const int i = I * 64 + t, jl = J * 64 + t;
  const bool act = i < N;
  double xi = 0, yi = 0, zi = 0, mi = 1;
  if (act) {
    xi = X[base + i];
    yi = X[nb + base + i];
    zi = X[2 * nb + base + i];
    mi = M[base + i];
  }
  const bool jact = jl < N;
  jx[t] = jact ? X[base + jl] : 0.0;
  jy[t] = jact ? X[nb + base + jl] : 0.0;
  jz[t] = jact ? X[2 * nb + base + jl] : 0.0;
  constexpr bool GAUSS = !ENERGY && (MODE == PK_GAUSS || MODE == PK_PGAUSS);
  jm[t] = jact ? M[base + jl] : 1.0;
  const double pre = GAUSS ? pp.g / (M_PI * pp.s2) : 0.0;
  const bool quick = GAUSS && gauss_quick(pp.s2, pre);
  if (quick) jm[t] = 1.0 / jm[t];
  rx[t] = 0;
  ry[t] = 0;
  rz[t] = 0;
  __syncthreads();
  const bool diag = I == J;
  const int s_lo = diag ? 1 : 0, s_hi = diag ? 32 : 63;
  double fx = 0, fy = 0, fz = 0, e = 0;
  if (quick) {
    // GAUSS_U rotations at a time: their terms are independent chains (sqrt,
    // exp, divisions), added one rotation after the other
    const double y = 1.0 / pp.s2, im = 1.0 / mi;
    // a diagonal tile of n <= 32 beads has no pair past rotation n - 1
    const int nj = N - J * 64, s_end = diag && nj <= 32 ? nj - 1 : s_hi;
    for (int s = s_lo; s <= s_end; s += GAUSS_U) {
      double gx[GAUSS_U], gy[GAUSS_U], gz[GAUSS_U];
      bool ok[GAUSS_U];
#pragma unroll
      for (int u = 0; u < GAUSS_U; ++u) {
        const int j = (t + s + u) & 63;
        ok[u] = act && s + u <= s_end && J * 64 + j < N && !(diag && s + u == 32 && t >= 32);
        gx[u] = ok[u] ? xi - jx[j] : 1.0;
        gy[u] = ok[u] ? yi - jy[j] : 1.0;
        gz[u] = ok[u] ? zi - jz[j] : 1.0;
      }
      if constexpr (GAUSS) gauss_terms<MODE>(gx, gy, gz, pp, pre, y);
#pragma unroll
      for (int u = 0; u < GAUSS_U; ++u) {
        // a lane without a pair adds zeros (at a rotation no two lanes share j;
        // the next rotation's j is another lane's, so the rotations stay in order)
        const int j = (t + s + u) & 63;
        const double hx = ok[u] ? gx[u] : 0.0, hy = ok[u] ? gy[u] : 0.0, hz = ok[u] ? gz[u] : 0.0;
        const double invm = J * 64 + j > i ? jm[j] : im;
        fx += hx * invm;
        fy += hy * invm;
        fz += hz * invm;
        rx[j] -= hx * invm;
        ry[j] -= hy * invm;
        rz[j] -= hz * invm;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    }
  } else {
    for (int s = s_lo; s <= s_hi; ++s) {
      const int j = (t + s) & 63;
      const int jg = J * 64 + j;
      const bool ok = act && jg < N && !(diag && s == 32 && t >= 32);
      if (ok) {
        double gx = 0, gy = 0, gz = 0;
        pair_term<MODE, ENERGY, NEAR>(xi - jx[j], yi - jy[j], zi - jz[j], pp, gx, gy, gz, e);
        if (!ENERGY) {
          const double invm = 1.0 / (jg > i ? jm[j] : mi);
          fx += gx * invm;
          fy += gy * invm;
          fz += gz * invm;
          rx[j] -= gx * invm;
          ry[j] -= gy * invm;
          rz[j] -= gz * invm;
        }
      }
    }
  }
  __syncthreads();
  if (ENERGY) {
    e = wave_sum(e);
    if (t == 0) Epart[item] = e;
    return;
  }
  auto put = [&](int bead, int slot, double vx, double vy, double vz) {
    const size_t s0 = (size_t)slot * 3 * nb + base + bead;
    put_tile(Fpart + s0, vx, add);
    put_tile(Fpart + s0 + nb, vy, add);
    put_tile(Fpart + s0 + 2 * (size_t)nb, vz, add);
  };
  if (diag) {
    if (act) put(i, I, fx + rx[t], fy + ry[t], fz + rz[t]);
  } else {
    if (act) put(i, J, fx, fy, fz);
    if (jact) put(jl, I, rx[t], ry[t], rz[t]);
  }
}

template <int MODE, bool ENERGY, bool NEAR>
__global__ __launch_bounds__(64) void k_pair_tiles(const double *__restrict__ X, const double *__restrict__ M,
                                                   double *__restrict__ Fpart, double *__restrict__ Epart,
                                                   const int2 *__restrict__ tiles, int N, int nb, int T, int ntp,
                                                   PairParams pp, double add) {
  k_pair_tiles_body<MODE, ENERGY, NEAR>(blockIdx.x, X, M, Fpart, Epart, tiles, N, nb, T, ntp, pp, add);
}

// F[d*nb + s] += sum_slot Fpart / P, slots in a fixed order.
__device__ __forceinline__ void k_reduce_tiles_body(int bx, const double *__restrict__ Fpart, double *__restrict__ F, int n3, int T, double P) {
  const int k = bx * blockDim.x + threadIdx.x;
  if (k >= n3) return;
  double s = 0;
  for (int q = 0; q < T; ++q) s += Fpart[(size_t)q * n3 + k];
  F[k] += s / P;
}

__global__ void k_reduce_tiles(const double *__restrict__ Fpart, double *__restrict__ F, int n3, int T, double P) {
  k_reduce_tiles_body(blockIdx.x, Fpart, F, n3, T, P);
}

// ------------------------------------------------------ reciprocal space
//
// k set: columns (mx, my) of the half space (mx > 0, or mx == 0 and my >= 0)
// times m_z = slot_mz(z), z in [0, ZP), slots in order of |m_z| (0, 1, -1,
// 2, -2, ...); the other half follows from S(-k) = S(k)*.  coef = 4 pi A_k,
// A_k = q exp(-pi^2 G^2/alpha^2)/(pi V G^2), G_d = m_d / L_d, is zero on the
// slots outside the set in use:
//  * the reference's cube |m_d| <= n (md_simulation_x.c:266-281), or
//  * the ball |G| <= G_max of a converged split (all terms beyond G_max are
//    below exp(-x_cut^2)), stored as the columns of the disc |G_xy| <= G_max
//    with their m_z slots, columns ordered by |G_xy| so that a column tile's
//    largest |m_z| is small towards the rim of the disc.
// Column (0, 0) keeps m_z > 0 only; padding columns and the slot z = 2MZ+1
// (m_z = MZ + 1 by slot_mz) carry zero weight.  MZ is 7, 15, 23 or 31, so
// ZP = 2 MZ + 2 = 16 NZT and the MH = MZ + 1 = 8 NZT values m = 0..MZ fill
// whole 4-wide K steps.
//
// Both k kernels are GEMMs on the FP64 matrix cores (V_MFMA_F64_16X16X4:
// A[i][k] in lane i + 16k, B[k][j] in lane j + 16k, D[i][j] in lane
// j + 16 (i mod 4), register i div 4) that use the conjugate symmetry of the
// z phases, Z(-m) = Z(m)* with Z(m) = c_m + i s_m = e^{i m theta_z}, so they
// run over m = 0..MZ only and take the real c and s as operands:
//   structure factors  X_c[c][m] = sum_beads A[c][s] c_m[s],  X_s likewise
//                      with s_m (M = columns, N = m, K = beads; A =
//                      e^{i(mx tx + my ty)}, four real products), and
//                      S(+-m) = X_c +- i X_s;
//   forces             with W = coef conj(S), P_m = W(+m) + W(-m),
//                      Q_m = W(+m) - W(-m) (P_0 = W(0), Q_0 = 0):
//                      U[s][c] = sum_z Z W = sum_m (c_m P_m + i s_m Q_m),
//                      V[s][c] = sum_z m_z Z W = sum_m m (c_m Q_m + i s_m P_m)
//                      (M = beads, N = columns, K = m; eight real products),
// then f_s = sum_c (mx, my) Im(A U) / L + (0, 0, Im(A V)).  Against complex
// products over all 2 MZ + 1 values of m_z (three real products each in
// Gauss's form) this is a third fewer matrix-core operations per force
// K step and a quarter fewer per structure-factor K step.
//
// Phase tables (k_phase), table half-width MZ, all bead-major so that the 16
// columns of a tile (consecutive m_y, mostly one m_x) read one bead's
// contiguous run:
//   tx[s * (MZ + 1) + m]        e^{i 2 pi m x / L_x},  m = 0..MZ
//   ty[s * (MZ + 1) + m]        e^{i 2 pi m y / L_y},  m = 0..MZ (m_y < 0: the conjugate)
//   tz[s * (MZ + 1) + m]        e^{i 2 pi m z / L_z},  m = 0..MZ
constexpr int MAX_KM = 31;     // largest table half-width of the k kernels

// m_z of slot z: 0, 1, -1, 2, -2, ...
__host__ __device__ inline int slot_mz(int z) { return (z & 1) ? (z + 1) >> 1 : -(z >> 1); }

typedef double v4d __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4d mfma4(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

struct KSpace {
  double L[3] = {0, 0, 0}, alpha = 0, q = 0, gmax2 = 0;
  int n = -2;  // cube half-width, or -1 for the ball of radius^2 gmax2
  int MZ = 0, ZP = 0, ncol = 0, ncolp = 0, nk = 0;  // nk: k vectors with nonzero weight
  double e0 = 0;  // sum over the k set of coef / (4 pi): each bead's self term of the slice energy
  int2 *cols = nullptr;    // [ncolp] (mx, my), then [ncolp / 16] K-step range of each column tile
  double *coef = nullptr;  // [ncolp][ZP]
  double2 *tx = nullptr, *ty = nullptr, *tz = nullptr, *S = nullptr, *W = nullptr;
  size_t tx_cap = 0, ty_cap = 0, tz_cap = 0, s_cap = 0, w_cap = 0;
  int stamp = 0;
};

// Tile-pair schedule and partial-sum scratch (grown on demand, kept).
struct TileBufs {
  int N = -1, T = 0, ntp = 0;
  int2 *tiles = nullptr;
  int2 *tiles_r = nullptr;  // the same pairs, off-diagonal first (real-space Ewald order)
  double *Fpart = nullptr, *Epart = nullptr;
  double *Frec = nullptr;  // reciprocal forces kept apart for k_combine_forces (3 N P)
  size_t fcap = 0, ecap = 0, rcap = 0;
};

// Per-object buffers of the pair kernels, so that independent systems can
// run concurrently: the tile schedule and partial sums, and three k-space
// table sets (most recently used kept: the step's, the estimators', and the
// low shells of a surrogate).
constexpr int NKS = 3;
struct PairBufs {
  TileBufs tb;
  KSpace ks[NKS];
  int ks_clock = 0;
};

static PairBufs *pair_bufs(DevPimd *p) {
  if (!p->pair_bufs) p->pair_bufs = new PairBufs();
  return (PairBufs *)p->pair_bufs;
}

// Device allocations made by the pair buffers (pair_prepare reports them).
static unsigned g_pair_allocs = 0;
unsigned pair_alloc_epoch() { return g_pair_allocs; }

static int grow(double2 *&p, size_t &cap, size_t need) {
  if (need <= cap) return 0;
  ++g_pair_allocs;
  if (p) (void)hipFree(p);
  p = nullptr;
  XMD_CHECK(hipMalloc(&p, need * sizeof(double2)));
  cap = need;
  return 0;
}

// Table half-widths whose 2 MZ + 2 slots fill whole 16-wide tiles.
static int table_mz(int M) {
  for (int mz : {7, 15, 23, 31})
    if (M <= mz) return mz;
  return -1;
}

static KSpace *ensure_kspace(DevPimd *p, const double *L, double alpha, double q, int n, double gmax2, int nb,
                             int P) {
  PairBufs *pb = pair_bufs(p);
  KSpace *ks = pb->ks;
  KSpace *K = nullptr;
  for (int i = 0; i < NKS; ++i) {
    KSpace &k = ks[i];
    if (k.n == n && k.alpha == alpha && k.q == q && k.gmax2 == gmax2 && k.L[0] == L[0] && k.L[1] == L[1] &&
        k.L[2] == L[2])
      K = &k;
  }
  if (!K) {
    ++g_pair_allocs;
    K = &ks[0];
    for (int i = 1; i < NKS; ++i)
      if (ks[i].stamp < K->stamp) K = &ks[i];
    int M = n;
    if (n < 0) {
      M = 0;
      for (int d = 0; d < 3; ++d) M = std::max(M, (int)floor(sqrt(gmax2) * L[d]));
    }
    const int MZ = table_mz(M);
    if (MZ < 0) {
      fprintf(stderr, "xmd: Ewald k range %d exceeds the supported %d\n", M, MAX_KM);
      return nullptr;
    }
    const int ZP = 2 * MZ + 2;
    // Columns (mx, my) of the half space, each with its m_z slots: the cube
    // |m| <= n, or the ball |G|^2 <= gmax2.  Columns are ordered by |G_xy| so
    // that a tile of 16 has a narrow |m_z| range; beyond it the weights are
    // zero, and both k kernels skip the K steps (force) and m tiles
    // (structure factors) that are zero for the whole tile.
    struct Col {
      int mx, my, zlo, zhi;
      double gxy2;
      std::vector<double> c;
    };
    std::vector<Col> cl;
    const double V = L[0] * L[1] * L[2];
    int nk = 0;
    for (int mx = 0; mx <= M; ++mx)
      for (int my = -M; my <= M; ++my) {
        if (mx == 0 && my < 0) continue;
        const double gxy2 = (mx / L[0]) * (mx / L[0]) + (my / L[1]) * (my / L[1]);
        if (n < 0 && gxy2 > gmax2) continue;
        Col col{mx, my, MZ + 1, -1, gxy2, std::vector<double>(ZP, 0.0)};
        for (int z = 0; z < ZP; ++z) {
          const int mz = slot_mz(z);
          const double G2 = gxy2 + (mz / L[2]) * (mz / L[2]);
          bool in = mz <= MZ && (n < 0 ? G2 <= gmax2 : (mz >= -n && mz <= n));
          if (mx == 0 && my == 0 && mz <= 0) in = false;
          if (in) {
            col.c[z] = 4 * M_PI * q * exp(-M_PI * M_PI * G2 / (alpha * alpha)) / (G2 * V * M_PI);
            col.zlo = std::min(col.zlo, std::abs(mz));
            col.zhi = std::max(col.zhi, std::abs(mz));
            ++nk;
          }
        }
        cl.push_back(std::move(col));
      }
    std::stable_sort(cl.begin(), cl.end(), [](const Col &a, const Col &b) { return a.gxy2 < b.gxy2; });
    const int ncol = (int)cl.size(), ncolp = (ncol + 15) / 16 * 16;
    // cols: [ncolp] (mx, my), then per tile of 16 columns the first and last
    // 4-wide step of |m_z| holding a nonzero weight (first > last: none)
    std::vector<int2> cols;
    std::vector<double> coef;
    std::vector<int2> kr(ncolp / 16, make_int2(MZ + 1, -1));
    for (int c = 0; c < ncolp; ++c) {
      if (c < ncol) {
        cols.push_back(make_int2(cl[c].mx, cl[c].my));
        coef.insert(coef.end(), cl[c].c.begin(), cl[c].c.end());
        if (cl[c].zlo <= cl[c].zhi) {
          kr[c / 16].x = std::min(kr[c / 16].x, cl[c].zlo / 4);
          kr[c / 16].y = std::max(kr[c / 16].y, cl[c].zhi / 4);
        }
      } else {
        cols.push_back(make_int2(0, 0));
        coef.insert(coef.end(), ZP, 0.0);
      }
    }
    cols.insert(cols.end(), kr.begin(), kr.end());
    if (K->cols) {
      (void)hipFree(K->cols);
      (void)hipFree(K->coef);
    }
    XMD_CHECK_NULL(hipMalloc(&K->cols, cols.size() * sizeof(int2)));
    XMD_CHECK_NULL(hipMalloc(&K->coef, coef.size() * sizeof(double)));
    XMD_CHECK_NULL(hipMemcpy(K->cols, cols.data(), cols.size() * sizeof(int2), hipMemcpyHostToDevice));
    XMD_CHECK_NULL(hipMemcpy(K->coef, coef.data(), coef.size() * sizeof(double), hipMemcpyHostToDevice));
    K->n = n;
    K->gmax2 = gmax2;
    K->alpha = alpha;
    K->q = q;
    for (int d = 0; d < 3; ++d) K->L[d] = L[d];
    K->MZ = MZ;
    K->ZP = ZP;
    K->ncol = ncol;
    K->ncolp = ncolp;
    K->nk = nk;
    double csum = 0;
    for (double c : coef) csum += c;
    K->e0 = csum / (4 * M_PI);
  }
  K->stamp = ++pb->ks_clock;
  if ((long long)nb * 3 * (K->MZ + 1) > INT_MAX) {
    fprintf(stderr, "xmd: %d beads exceed the Ewald phase-table index range\n", nb);
    return nullptr;
  }
  const size_t slots = (size_t)K->ncolp * K->ZP;
  if (grow(K->tx, K->tx_cap, (size_t)(K->MZ + 1) * nb) || grow(K->ty, K->ty_cap, (size_t)(K->MZ + 1) * nb) ||
      grow(K->tz, K->tz_cap, (size_t)(K->MZ + 1) * nb) || grow(K->S, K->s_cap, (size_t)P * slots) ||
      grow(K->W, K->w_cap, (size_t)P * slots))
    return nullptr;
  return K;
}

// e^{i pi m u}, u = 2 x / L, m = 0..MZ, one thread per table entry: threads
// run over tx, then ty, then tz, each in storage order, so the stores of a
// wave are consecutive.
__host__ __device__ inline int phase_entries(int nb, int MZ) { return 3 * nb * (MZ + 1); }

__device__ __forceinline__ void k_phase_body(int bx, const double *__restrict__ X, int nb, int MZ, double L0, double L1,
                                             double L2, double2 *__restrict__ tx, double2 *__restrict__ ty,
                                             double2 *__restrict__ tz) {
  const int t = bx * blockDim.x + threadIdx.x;
  const int n1 = nb * (MZ + 1);
  if (t >= 3 * n1) return;
  const int d = t / n1, e = t - d * n1, s = e / (MZ + 1), m = e - s * (MZ + 1);
  double2 *out = (d == 0 ? tx : (d == 1 ? ty : tz)) + e;
  if (m == 0) {
    *out = make_double2(1.0, 0.0);
    return;
  }
  const double u = 2.0 * X[d * nb + s] / (d == 0 ? L0 : (d == 1 ? L1 : L2));
  double sn, cs;
  sincospi(m * u, &sn, &cs);
  *out = make_double2(cs, sn);
}

__global__ void k_phase(const double *__restrict__ X, int nb, int MZ, double L0, double L1, double L2,
                        double2 *__restrict__ tx, double2 *__restrict__ ty, double2 *__restrict__ tz) {
  k_phase_body(blockIdx.x, X, nb, MZ, L0, L1, L2, tx, ty, tz);
}

// Workgroups are numbered so that the tiles of one slice share an XCD
// (consecutive workgroup ids go to consecutive XCDs) when the slice count
// is a multiple of 8; otherwise the plain order.
__device__ __forceinline__ void xcd_tile(int w, int ntile, int P, int &slice, int &tile) {
  if ((P & 7) == 0) {
    const int x = w & 7, loc = w >> 3;
    slice = x + 8 * (loc / ntile);
    tile = loc % ntile;
  } else {
    slice = w / ntile;
    tile = w % ntile;
  }
}

// Structure factors of one 16-column tile of one slice: X_c[c][m] and
// X_s[c][m] over m = 0..MZ as four real products (ar c, ai c, ar s, ai s:
// A = ar + i ai, Z(m) = c + i s), then S(+-m) = X_c +- i X_s.  The four
// waves split the beads into quarters; their partial sums are added in a
// fixed order through `red` (4 x 4 x 256 doubles).  Writes S in the slot
// layout (slot 2m - 1: +m, slot 2m: -m) and the force kernel's operands
// PQ[c][2m] = P_m, PQ[c][2m + 1] = Q_m with W = coef conj(S),
// P_m = W(+m) + W(-m), Q_m = W(+m) - W(-m), P_0 = W(0), Q_0 = 0.
template <int NZT>
__device__ __forceinline__ void sk_tile(double *red, int slice, int c0, const double2 *__restrict__ tx,
                                        const double2 *__restrict__ ty, const double2 *__restrict__ tz, int2 cl,
                                        int2 kr, const double *__restrict__ coef, int ncolp, int MZ, int N,
                                        double2 *__restrict__ S, double2 *__restrict__ PQ) {
  constexpr int ZP = 16 * NZT, MH = 8 * NZT, NMT = (MH + 15) / 16;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int kb = lane >> 4;  // bead of this lane within a K step
  const int mb = lane & 15;  // B operand column: m within an m tile
  const int q0 = (N * wv) / 4, q1 = (N * (wv + 1)) / 4;
  const int nfull = (q1 - q0) >> 2;
  const int sx = 4 * (MZ + 1);
  const size_t s0 = (size_t)slice * N + q0 + kb;
  const double2 *px = tx + s0 * (MZ + 1) + cl.x;
  const bool yneg = cl.y < 0;  // e^{-i m y} = conj(e^{i m y})
  const double2 *py = ty + s0 * (MZ + 1) + (yneg ? -cl.y : cl.y);
  const double2 *pz = tz + s0 * MH + mb;
  // m tiles beyond the column tile's largest |m_z| (kr.y: its last 4-wide
  // step) hold zero weights: their sums are not formed (S and PQ stay zero)
  const int ntl = kr.x <= kr.y ? min(NMT, kr.y / 4 + 1) : 0;
  auto zok = [&](int t) { return t < ntl && (MH % 16 == 0 || 16 * t + mb < MH); };
  v4d xcr[NMT], xci[NMT], xsr[NMT], xsi[NMT];
#pragma unroll
  for (int t = 0; t < NMT; ++t) xcr[t] = xci[t] = xsr[t] = xsi[t] = v4d{0, 0, 0, 0};
  auto step = [&](double2 ex, double2 ey, const double2 *z, bool keep) {
    if (yneg) ey.y = -ey.y;
    double ar = ex.x * ey.x - ex.y * ey.y, ai = ex.x * ey.y + ex.y * ey.x;
    if (!keep) ar = ai = 0.0;
#pragma unroll
    for (int t = 0; t < NMT; ++t) {
      if (t >= ntl) continue;
      xcr[t] = mfma4(ar, z[t].x, xcr[t]);
      xci[t] = mfma4(ai, z[t].x, xci[t]);
      xsr[t] = mfma4(ar, z[t].y, xsr[t]);
      xsi[t] = mfma4(ai, z[t].y, xsi[t]);
    }
  };
  int k = 0;
  for (; k + 4 <= nfull; k += 4) {
    double2 ex[4], ey[4], z[4][NMT];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      ex[u] = px[u * sx];
      ey[u] = py[u * sx];
#pragma unroll
      for (int t = 0; t < NMT; ++t) z[u][t] = zok(t) ? pz[u * 4 * MH + 16 * t] : make_double2(0.0, 0.0);
    }
    px += 4 * sx;
    py += 4 * sx;
    pz += 16 * MH;
#pragma unroll
    for (int u = 0; u < 4; ++u) step(ex[u], ey[u], z[u], true);
  }
  for (; k < nfull; ++k) {
    double2 z[NMT];
#pragma unroll
    for (int t = 0; t < NMT; ++t) z[t] = zok(t) ? pz[16 * t] : make_double2(0.0, 0.0);
    step(px[0], py[0], z, true);
    px += sx;
    py += sx;
    pz += 4 * MH;
  }
  if ((q1 - q0) & 3) {
    // last partial K step: lanes whose bead is past the quarter read the
    // quarter's first bead and contribute zero
    const bool ok = q0 + 4 * nfull + kb < q1;
    const int back = ok ? 0 : 4 * nfull + kb;
    double2 z[NMT];
#pragma unroll
    for (int t = 0; t < NMT; ++t) z[t] = zok(t) ? pz[16 * t - back * MH] : make_double2(0.0, 0.0);
    step(px[-back * (MZ + 1)], py[-back * (MZ + 1)], z, ok);
  }
  // D[i = column][j = m]: lane j + 16 (i%4), register i/4
  const size_t base = (size_t)slice * ncolp * ZP;
#pragma unroll
  for (int t = 0; t < NMT; ++t) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int e = (4 * r + (lane >> 4)) * 16 + (lane & 15);
      red[(0 * 4 + wv) * 256 + e] = xcr[t][r];
      red[(1 * 4 + wv) * 256 + e] = xci[t][r];
      red[(2 * 4 + wv) * 256 + e] = xsr[t][r];
      red[(3 * 4 + wv) * 256 + e] = xsi[t][r];
    }
    __syncthreads();
    const int e = threadIdx.x, i = e >> 4, m = 16 * t + (e & 15);
    if (m < MH) {
      double x[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        x[q] = ((red[(q * 4 + 0) * 256 + e] + red[(q * 4 + 1) * 256 + e]) + red[(q * 4 + 2) * 256 + e]) +
               red[(q * 4 + 3) * 256 + e];
      const size_t row = base + (size_t)(c0 + i) * ZP;
      double2 P, Q;
      if (m == 0) {  // s_0 = 0: S = X_c
        const double2 S0 = make_double2(x[0], x[1]);
        const double c = coef[row - base];
        S[row] = S0;
        P = make_double2(c * S0.x, -c * S0.y);
        Q = make_double2(0.0, 0.0);
      } else {
        const double2 Sp = make_double2(x[0] - x[3], x[1] + x[2]), Sm = make_double2(x[0] + x[3], x[1] - x[2]);
        const double cp = coef[row - base + 2 * m - 1], cm = coef[row - base + 2 * m];
        S[row + 2 * m - 1] = Sp;
        S[row + 2 * m] = Sm;
        const double2 Wp = make_double2(cp * Sp.x, -cp * Sp.y), Wm = make_double2(cm * Sm.x, -cm * Sm.y);
        P = make_double2(Wp.x + Wm.x, Wp.y + Wm.y);
        Q = make_double2(Wp.x - Wm.x, Wp.y - Wm.y);
      }
      if (m == MH - 1) S[row + ZP - 1] = make_double2(0.0, 0.0);
      PQ[row + 2 * m] = P;
      PQ[row + 2 * m + 1] = Q;
    }
    __syncthreads();
  }
}

// Workgroup w covers (slice, column tile) for every slot; NZT = ZP / 16.
template <int NZT>
__device__ __forceinline__ void k_sk_mfma_body(int bx, const double2 *__restrict__ tx, const double2 *__restrict__ ty,
                                                 const double2 *__restrict__ tz, const int2 *__restrict__ cols,
                                                 const double *__restrict__ coef, int ncolp, int MZ, int N, int P,
                                                 double2 *__restrict__ S, double2 *__restrict__ W) {
  __shared__ double red[16 * 256];
  int slice, tile;
  xcd_tile(bx, ncolp / 16, P, slice, tile);
  const int c0 = tile * 16;
  const int2 cl = cols[c0 + (threadIdx.x & 15)];
  sk_tile<NZT>(red, slice, c0, tx, ty, tz, cl, cols[ncolp + tile], coef, ncolp, MZ, N, S, W);
}

template <int NZT>
__global__ __launch_bounds__(256) void k_sk_mfma(const double2 *__restrict__ tx, const double2 *__restrict__ ty,
                                                 const double2 *__restrict__ tz, const int2 *__restrict__ cols,
                                                 const double *__restrict__ coef, int ncolp, int MZ, int N, int P,
                                                 double2 *__restrict__ S, double2 *__restrict__ W) {
  k_sk_mfma_body<NZT>(blockIdx.x, tx, ty, tz, cols, coef, ncolp, MZ, N, P, S, W);
}

// Forces on the 64 beads [b0, b0 + 64) of one slice; wave w owns beads
// b0 + 16 w .. b0 + 16 w + 15 and walks every column tile in order.  Per tile,
// over m = 0..MZ (the conjugate pairs +-m_z folded into P and Q),
//   U[s][c] = sum_z Z[s][z] W[c][z] = sum_m (c_m P_m + i s_m Q_m),
//   V[s][c] = sum_z m_z Z[s][z] W[c][z] = sum_m m (c_m Q_m + i s_m P_m),
// and f_s += sum_c (mx Im(A U) / L_x, my Im(A U) / L_y, Im(A V) / L_z) / (m P).
// For bead i this is sum_k coef_k g_k Im(e^{i k.x_i} S_k*) / (m_i P), the
// reference's per-pair sum (md_simulation_x.c:266-281) since
// sum_{l != i} sin(k.(x_i - x_l)) = Im(e^{i k.x_i} S_k*).  The Z operands of
// a wave's 16 beads are the same for every column tile and stay in registers.
// The workgroup stages what its four waves share through LDS: the x and y
// phase rows of its 64 beads (read once per workgroup instead of gathered per
// bead and column) and the P, Q tile of the current column tile (double-
// buffered: the next tile is fetched into registers while the current one is
// multiplied, one barrier per tile), so each entry is fetched from L2 once
// per 64 beads.
// EN: also the bead's share of its slice's reciprocal energy,
//   e_i = sum_k A_k (Re(e^{i k.x_i} S_k*) - 1),  A_k = coef_k / (4 pi),
// (the slice energy sum_k A_k (|S_k|^2 - N) split over its beads), from the
// same U: Re(A U) = sum_{k of the column} coef_k Re(e^{i k.x_i} S_k*);
// e0 = sum_k A_k.
template <int NZT>
struct FrcLds {
  static constexpr int ZP = 16 * NZT, MZ = 8 * NZT - 1, RX = MZ + 1, WS = ZP + 1;
  // phase rows e^{i m theta_x}, e^{i m theta_y}, m = 0..MZ (negative m_y: the conjugate)
  double2 rx[64 * RX], ry[64 * RX];
  double2 wt[2][16 * WS];            // P, Q tile [column][2m + (0: P, 1: Q)], rows padded against bank conflicts
};

template <int NZT, bool EN = false>
__device__ __forceinline__ void recip_force_tile(FrcLds<NZT> &sh, int slice, int b0, const double2 *__restrict__ tx,
                                                 const double2 *__restrict__ ty, const double2 *__restrict__ tz,
                                                 const int2 *__restrict__ cols, int ncolp, int MZ,
                                                 const double2 *__restrict__ PQ, const double *__restrict__ Mass,
                                                 double *__restrict__ F, int N, int nb, double L0, double L1,
                                                 double L2, double Pd, double *__restrict__ Frec,
                                                 double *__restrict__ Erec = nullptr, double e0 = 0.0) {
  using S = FrcLds<NZT>;  // MZ = 8 NZT - 1 (table_mz)
  (void)MZ;
  constexpr int ZP = S::ZP, MH = S::RX, KS = MH / 4, RX = S::RX, WS = S::WS, TE = 16 * ZP;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int nloc = min(64, N - b0);  // beads of this workgroup
  // phase rows of the workgroup's beads (zero past the last bead)
  {
    const double2 *gx = tx + (size_t)(slice * N + b0) * RX;
    const double2 *gy = ty + (size_t)(slice * N + b0) * RX;
    for (int e = tid; e < 64 * RX; e += 256) {
      const bool ok = e < nloc * RX;
      sh.rx[e] = ok ? gx[e] : make_double2(0.0, 0.0);
      sh.ry[e] = ok ? gy[e] : make_double2(0.0, 0.0);
    }
  }
  const double2 *Ws = PQ + (size_t)slice * ncolp * ZP;
  // P, Q tile 0: 16 ZP entries, NZT per thread (entry e = tid + 256 i: column e / ZP, position e % ZP)
#pragma unroll
  for (int i = 0; i < NZT; ++i) {
    const int e = tid + 256 * i;
    sh.wt[0][(e / ZP) * WS + e % ZP] = Ws[e];
  }
  const int lb = 16 * wv + (lane & 15);  // A operand row (local bead) of this lane
  const bool aok = lb < nloc;
  // A operands c_m, s_m of bead lb, m = 4 k + lane / 16
  const double2 *pza = tz + (size_t)(slice * N + b0 + (aok ? lb : 0)) * MH + (lane >> 4);
  double zc[KS], zn[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    const double2 z = aok ? pza[4 * k] : make_double2(0.0, 0.0);
    zc[k] = z.x;
    zn[k] = z.y;
  }
  const int zl = lane >> 4;     // this lane's K row within a K step
  const int cq = lane & 15;     // this lane's column within a tile (B operand and D column)
  // D[i = bead][j = column]: lane j + 16 (i%4), register i/4; this lane's beads
  // are local 16 wv + 4 r + zl
  double fx[4] = {0, 0, 0, 0}, fy[4] = {0, 0, 0, 0}, fz[4] = {0, 0, 0, 0}, en[4] = {0, 0, 0, 0};
  const int nct = ncolp / 16;
  __syncthreads();
  for (int ct = 0; ct < nct; ++ct) {
    const int cur = ct & 1;
    const bool more = ct + 1 < nct;
    // next tile (the last tile re-reads itself, unused)
    double2 pre[NZT];
    const double2 *nxt = Ws + (size_t)(more ? ct + 1 : ct) * TE + tid;
#pragma unroll
    for (int i = 0; i < NZT; ++i) pre[i] = nxt[256 * i];
    // m steps outside [kr.x, kr.y] carry zero weights for every column of
    // the tile: skipping them leaves U and V unchanged
    const int2 kr = cols[ncolp + ct];
    const int2 cl = cols[ct * 16 + cq];
    const double2 *wrow = sh.wt[cur] + cq * WS + 2 * zl;
    v4d ur4 = {0, 0, 0, 0}, ui4 = ur4, vr4 = ur4, vi4 = ur4;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      if (k < kr.x || k > kr.y) continue;
      // B operands P_m, Q_m of column cq, m = 4 k + lane / 16
      const double2 Pm = wrow[8 * k], Qm = wrow[8 * k + 1];
      const double m = (double)(4 * k + zl);
      ur4 = mfma4(zc[k], Pm.x, ur4);
      ui4 = mfma4(zc[k], Pm.y, ui4);
      vr4 = mfma4(zc[k], m * Qm.x, vr4);
      vi4 = mfma4(zc[k], m * Qm.y, vi4);
      ur4 = mfma4(zn[k], -Qm.y, ur4);
      ui4 = mfma4(zn[k], Qm.x, ui4);
      vr4 = mfma4(zn[k], -m * Pm.y, vr4);
      vi4 = mfma4(zn[k], m * Pm.x, vi4);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int bl = 16 * wv + 4 * r + zl;
      const double2 ex = sh.rx[bl * RX + cl.x];
      double2 ey = sh.ry[bl * RX + (cl.y < 0 ? -cl.y : cl.y)];
      if (cl.y < 0) ey.y = -ey.y;
      const double ur = ur4[r], ui = ui4[r], vr = vr4[r], vi = vi4[r];
      const double ar = ex.x * ey.x - ex.y * ey.y, ai = ex.x * ey.y + ex.y * ey.x;
      const double g = fma(ar, ui, ai * ur);
      fx[r] = fma((double)cl.x, g, fx[r]);
      fy[r] = fma((double)cl.y, g, fy[r]);
      fz[r] = fma(ar, vi, fma(ai, vr, fz[r]));
      if (EN) en[r] = fma(ar, ur, fma(-ai, ui, en[r]));
    }
    if (more) {
#pragma unroll
      for (int i = 0; i < NZT; ++i) {
        const int e = tid + 256 * i;
        sh.wt[cur ^ 1][(e / ZP) * WS + e % ZP] = pre[i];
      }
    }
    __syncthreads();
  }
  // sum over the 16 columns held by the lanes of each 16-lane row
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      fx[r] += __shfl_xor(fx[r], o, 64);
      fy[r] += __shfl_xor(fy[r], o, 64);
      fz[r] += __shfl_xor(fz[r], o, 64);
      if (EN) en[r] += __shfl_xor(en[r], o, 64);
    }
  // lane 16 q + r of the wave writes bead 16 wv + 4 r + q
  if (cq < 4) {
    const int r = cq;
    const double gx = r == 0 ? fx[0] : r == 1 ? fx[1] : r == 2 ? fx[2] : fx[3];
    const double gy = r == 0 ? fy[0] : r == 1 ? fy[1] : r == 2 ? fy[2] : fy[3];
    const double gz = r == 0 ? fz[0] : r == 1 ? fz[1] : r == 2 ? fz[2] : fz[3];
    const int bl = 16 * wv + 4 * r + zl;
    if (bl < nloc) {
      const int s = slice * N + b0 + bl;
      const double m = Mass[s];
      if (Frec) {  // kept apart, added into F later in the same order
        Frec[s] = gx / L0 / m / Pd;
        Frec[nb + s] = gy / L1 / m / Pd;
        Frec[2 * nb + s] = gz / L2 / m / Pd;
      } else {
        F[s] += gx / L0 / m / Pd;
        F[nb + s] += gy / L1 / m / Pd;
        F[2 * nb + s] += gz / L2 / m / Pd;
      }
      if (EN) {
        const double e = r == 0 ? en[0] : r == 1 ? en[1] : r == 2 ? en[2] : en[3];
        Erec[s] = e / (4 * M_PI) - e0;
      }
    }
  }
}

// Workgroups per slice of the reciprocal force kernels (64 beads each).
__host__ __device__ inline int frc_tiles(int N) { return (N + 63) / 64; }

// Forces on the 16 beads [b0, b0 + 16) of one slice, the column tiles dealt
// to the four waves (tile 4 i + w to wave w): for grids too small to fill the
// device with 64 beads per workgroup, whose waves each walk every tile, and
// for slices of few beads, where most of those waves hold none.  A P, Q tile
// is used by one wave here, each entry by one lane, so it goes from memory
// straight to registers, a round ahead.  The products of a round's four tiles
// are exchanged through LDS and wave w adds them, tile after tile, for the
// beads 4 w .. 4 w + 3: every sum has the order, and the bits, of
// recip_force_tile.
template <int NZT>
struct FrcSplitLds {
  static constexpr int ZP = 16 * NZT, RX = 8 * NZT;
  double2 rx[16 * RX], ry[16 * RX];  // phase rows, as in FrcLds
  double u[4][5][4][64];             // [tile of the round][g, ar, ai, vr, vi][D register][lane]
  int2 cl[4][16];                    // (m_x, m_y) of the round's columns
};

template <int NZT>
__device__ __forceinline__ void recip_force_split(FrcSplitLds<NZT> &sh, int slice, int b0,
                                                  const double2 *__restrict__ tx, const double2 *__restrict__ ty,
                                                  const double2 *__restrict__ tz, const int2 *__restrict__ cols,
                                                  int ncolp, const double2 *__restrict__ PQ,
                                                  const double *__restrict__ Mass, double *__restrict__ F, int N,
                                                  int nb, double L0, double L1, double L2, double Pd,
                                                  double *__restrict__ Frec) {
  using S = FrcSplitLds<NZT>;
  constexpr int ZP = S::ZP, RX = S::RX, MH = RX, KS = MH / 4;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int nloc = min(16, N - b0);
  {
    const double2 *gx = tx + (size_t)(slice * N + b0) * RX;
    const double2 *gy = ty + (size_t)(slice * N + b0) * RX;
    for (int e = tid; e < 16 * RX; e += 256) {
      const bool ok = e < nloc * RX;
      sh.rx[e] = ok ? gx[e] : make_double2(0.0, 0.0);
      sh.ry[e] = ok ? gy[e] : make_double2(0.0, 0.0);
    }
  }
  const int zl = lane >> 4, cq = lane & 15;
  const bool aok = cq < nloc;
  const double2 *pza = tz + (size_t)(slice * N + b0 + (aok ? cq : 0)) * MH + zl;
  double zc[KS], zn[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    const double2 z = aok ? pza[4 * k] : make_double2(0.0, 0.0);
    zc[k] = z.x;
    zn[k] = z.y;
  }
  const int nct = ncolp / 16;
  // operands P_m, Q_m of column cq of tile ct, m = 4 k + zl
  const double2 *Ws = PQ + (size_t)slice * ncolp * ZP + cq * ZP + 2 * zl;
  double2 pq[2 * KS];
  int2 kr, cl;
  auto fetch = [&](int ct) {
    const int c = min(ct, nct - 1);  // past the last tile: unused
    const double2 *w = Ws + (size_t)c * 16 * ZP;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      pq[2 * k] = w[8 * k];
      pq[2 * k + 1] = w[8 * k + 1];
    }
    kr = cols[ncolp + c];
    cl = cols[c * 16 + cq];
  };
  fetch(wv);
  double fx = 0, fy = 0, fz = 0;
  for (int ct0 = 0; ct0 < nct; ct0 += 4) {
    __syncthreads();
    if (ct0 + wv < nct) {
      v4d ur4 = {0, 0, 0, 0}, ui4 = ur4, vr4 = ur4, vi4 = ur4;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        if (k < kr.x || k > kr.y) continue;
        const double2 Pm = pq[2 * k], Qm = pq[2 * k + 1];
        const double m = (double)(4 * k + zl);
        ur4 = mfma4(zc[k], Pm.x, ur4);
        ui4 = mfma4(zc[k], Pm.y, ui4);
        vr4 = mfma4(zc[k], m * Qm.x, vr4);
        vi4 = mfma4(zc[k], m * Qm.y, vi4);
        ur4 = mfma4(zn[k], -Qm.y, ur4);
        ui4 = mfma4(zn[k], Qm.x, ui4);
        vr4 = mfma4(zn[k], -m * Pm.y, vr4);
        vi4 = mfma4(zn[k], m * Pm.x, vi4);
      }
      const int2 c = cl;
      fetch(ct0 + 4 + wv);
      if (zl == 0) sh.cl[wv][cq] = c;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int bl = 4 * r + zl;
        const double2 ex = sh.rx[bl * RX + c.x];
        double2 ey = sh.ry[bl * RX + (c.y < 0 ? -c.y : c.y)];
        if (c.y < 0) ey.y = -ey.y;
        const double ur = ur4[r], ui = ui4[r];
        const double ar = ex.x * ey.x - ex.y * ey.y, ai = ex.x * ey.y + ex.y * ey.x;
        sh.u[wv][0][r][lane] = fma(ar, ui, ai * ur);
        sh.u[wv][1][r][lane] = ar;
        sh.u[wv][2][r][lane] = ai;
        sh.u[wv][3][r][lane] = vr4[r];
        sh.u[wv][4][r][lane] = vi4[r];
      }
    }
    __syncthreads();
    for (int t = 0; t < min(4, nct - ct0); ++t) {
      const int2 c = sh.cl[t][cq];
      const double g = sh.u[t][0][wv][lane], ar = sh.u[t][1][wv][lane], ai = sh.u[t][2][wv][lane];
      const double vr = sh.u[t][3][wv][lane], vi = sh.u[t][4][wv][lane];
      fx = fma((double)c.x, g, fx);
      fy = fma((double)c.y, g, fy);
      fz = fma(ar, vi, fma(ai, vr, fz));
    }
  }
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    fx += __shfl_xor(fx, o, 64);
    fy += __shfl_xor(fy, o, 64);
    fz += __shfl_xor(fz, o, 64);
  }
  const int bl = 4 * wv + zl;
  if (cq == 0 && bl < nloc) {
    const int s = slice * N + b0 + bl;
    const double m = Mass[s];
    if (Frec) {
      Frec[s] = fx / L0 / m / Pd;
      Frec[nb + s] = fy / L1 / m / Pd;
      Frec[2 * nb + s] = fz / L2 / m / Pd;
    } else {
      F[s] += fx / L0 / m / Pd;
      F[nb + s] += fy / L1 / m / Pd;
      F[2 * nb + s] += fz / L2 / m / Pd;
    }
  }
}

// Workgroups per slice with 16 beads each.
__host__ __device__ inline int frc_split_tiles(int N) { return (N + 15) / 16; }

template <int NZT>
__global__ __launch_bounds__(256) void k_recip_force_split(
    const double2 *__restrict__ tx, const double2 *__restrict__ ty, const double2 *__restrict__ tz,
    const int2 *__restrict__ cols, int ncolp, int MZ, const double2 *__restrict__ W,
    const double *__restrict__ Mass, double *__restrict__ F, int N, int nb, int P, double L0, double L1, double L2,
    double Pd, double *__restrict__ Frec) {
  __shared__ FrcSplitLds<NZT> sh;
  int slice, bt;
  xcd_tile(blockIdx.x, frc_split_tiles(N), P, slice, bt);
  recip_force_split<NZT>(sh, slice, bt * 16, tx, ty, tz, cols, ncolp, W, Mass, F, N, nb, L0, L1, L2, Pd, Frec);
}

template <int NZT, bool EN = false>
__device__ __forceinline__ void k_recip_force_mfma_body(int bx,
    const double2 *__restrict__ tx, const double2 *__restrict__ ty, const double2 *__restrict__ tz,
    const int2 *__restrict__ cols, int ncolp, int MZ, const double2 *__restrict__ W,
    const double *__restrict__ Mass, double *__restrict__ F, int N, int nb, int P, double L0, double L1, double L2,
    double Pd, double *__restrict__ Frec = nullptr, double *__restrict__ Erec = nullptr, double e0 = 0.0) {
  __shared__ FrcLds<NZT> sh;
  int slice, bt;
  xcd_tile(bx, frc_tiles(N), P, slice, bt);
  recip_force_tile<NZT, EN>(sh, slice, bt * 64, tx, ty, tz, cols, ncolp, MZ, W, Mass, F, N, nb, L0, L1, L2, Pd,
                            Frec, Erec, e0);
}

template <int NZT>
__global__ __launch_bounds__(256) void k_recip_force_mfma(
    const double2 *__restrict__ tx, const double2 *__restrict__ ty, const double2 *__restrict__ tz,
    const int2 *__restrict__ cols, int ncolp, int MZ, const double2 *__restrict__ W,
    const double *__restrict__ Mass, double *__restrict__ F, int N, int nb, int P, double L0, double L1, double L2,
    double Pd, double *__restrict__ Frec) {
  k_recip_force_mfma_body<NZT>(blockIdx.x, tx, ty, tz, cols, ncolp, MZ, W, Mass, F, N, nb, P, L0, L1, L2, Pd, Frec);
}

// Reciprocal forces (into Frec) and per-bead energies (into Erec) of every slice.
template <int NZT>
__global__ __launch_bounds__(256) void k_recip_force_energy(
    const double2 *__restrict__ tx, const double2 *__restrict__ ty, const double2 *__restrict__ tz,
    const int2 *__restrict__ cols, int ncolp, int MZ, const double2 *__restrict__ W,
    const double *__restrict__ Mass, int N, int nb, int P, double L0, double L1, double L2, double Pd,
    double *__restrict__ Frec, double *__restrict__ Erec, double e0) {
  k_recip_force_mfma_body<NZT, true>(blockIdx.x, tx, ty, tz, cols, ncolp, MZ, W, Mass, nullptr, N, nb, P, L0, L1, L2,
                                     Pd, Frec, Erec, e0);
}

// Reciprocal energy of every slice: sum_{k in half} A_k (|S_k|^2 - N), into partials.
__global__ __launch_bounds__(256) void k_recip_energy(const double2 *__restrict__ S, const double *__restrict__ coef,
                                                      int slots, int P, int N, double *__restrict__ part) {
  __shared__ double red[256];
  double s = 0;
  for (int t = blockIdx.x * 256 + threadIdx.x; t < slots * P; t += gridDim.x * 256) {
    const int kk = t % slots;
    const double2 v = S[t];
    s += coef[kk] / (4 * M_PI) * (v.x * v.x + v.y * v.y - N);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// ------------------------------------------ table-driven Ewald real space
//
// The force of one image at distance r is q h(alpha r) r_vec / r^3 with
// h(x) = erfc(x) + 2x/sqrt(pi) exp(-x^2) (md_simulation_x.c:288-289);
// h comes from the piecewise polynomial table of ewald_table.h (abs error
// 1.1e-16), staged in LDS once per workgroup.
//
// Images: with the minimum image a_d of the separation (|a_d| <= L_d/2),
// b_d = a_d - sign(a_d) L_d and c_d = a_d + sign(a_d) L_d, every image within
// r_c < sqrt(2) L takes per dimension a, b or c, and at most one dimension
// takes c (two would put it beyond sqrt(2) L).  Three enumerations, by r_c:
//   IMG_FACE   r_c^2 < min L_d^2 / 2: at most one image besides a, and it
//              takes b in one dimension only (two b's, or b in two
//              dimensions, are at least min L_d / sqrt(2) away), so each pair
//              evaluates exactly two candidates, a and the face image whose
//              distance is smallest, with no per-lane loop;
//   IMG_NEAR   r_c < min L_d: candidates a/b per dimension;
//   IMG_CORNER r_c < sqrt(2) min L_d: also the c candidates.
// IMG_NEAR and IMG_CORNER build the bit mask of the candidates inside r_c at
// bit kx | ky << 2 | kz << 4 with k = 0 (a), 1 (b), 3 (c), and walk it; the
// image is a_d - sext(k_d) s_d.  All three evaluate an image with the same
// arithmetic (ewald_image) and take the images in increasing bit order; the
// face enumeration's out-of-range candidate adds an exact zero.
enum { IMG_FACE, IMG_NEAR, IMG_CORNER };

struct EwReal {
  double L[3], iL[3];
  double q, al8, rc2;  // al8 = 8 alpha: table intervals of width 1/8 in x = alpha r
};

// 1/sqrt(x) for finite x > 0 (no zero, infinity or subnormal handling): the
// hardware estimate y refined by one second-order Newton-Raphson step,
// y (1 + e/2 + 3e^2/8) with e = 1 - x y^2.
__device__ __forceinline__ double rsqrt_pos(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(y * -x, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// Force of one image r of a pair, in three parts so that callers can keep
// the table loads of several images in flight together: ew_prep (distance,
// interval, local coordinate), ew_load (the interval's coefficients from the
// LDS table), ew_finish (Horner in y, force added to g when `in` holds).  r
// is never zero: distinct beads of a periodic system.
constexpr int kEwNC2 = kEwTabStride / 2;  // coefficient pairs per interval

struct EwImg {
  double rx, ry, rz, ir, y;
  int iv;
  bool in;
};

__device__ __forceinline__ EwImg ew_prep(double rx, double ry, double rz, bool in, const EwReal &ep) {
  EwImg m;
  m.rx = rx;
  m.ry = ry;
  m.rz = rz;
  m.in = in;
  const double R2 = fma(rx, rx, fma(ry, ry, rz * rz));
  m.ir = rsqrt_pos(R2);
  const double t8 = (R2 * m.ir) * ep.al8;
  m.iv = min((int)t8, kEwTabIntervals - 1);
  m.y = fma(2.0, t8, -(double)(2 * m.iv + 1));
  return m;
}

__device__ __forceinline__ void ew_load(const EwImg &m, const double2 *__restrict__ tab, double2 *cc) {
  const double2 *c = tab + m.iv * kEwNC2;
#pragma unroll
  for (int k = 0; k < kEwNC2; ++k) cc[k] = c[k];
}

__device__ __forceinline__ void ew_finish(const EwImg &m, const double2 *cc, const EwReal &ep, double &gx,
                                          double &gy, double &gz) {
  // coefficients c_0 .. c_DEG of the interval as (c_2k, c_2k+1) pairs
  double h = fma(cc[kEwNC2 - 1].y, m.y, cc[kEwNC2 - 1].x);
#pragma unroll
  for (int k = kEwNC2 - 2; k >= 0; --k) {
    h = fma(h, m.y, cc[k].y);
    h = fma(h, m.y, cc[k].x);
  }
  const double w = m.in ? ep.q * h * (m.ir * m.ir * m.ir) : 0.0;
  gx = fma(w, m.rx, gx);
  gy = fma(w, m.ry, gy);
  gz = fma(w, m.rz, gz);
}

// The loaded coefficients are pinned before use, so that the compiler issues
// every load of the group first (one wait) instead of waiting for each.
__device__ __forceinline__ void ew_pin(const double2 *cc, int n) {
  for (int k = 0; k < n; ++k) __asm__ volatile("" ::"v"(cc[k].x), "v"(cc[k].y));
}

__device__ __forceinline__ void ewald_image(double rx, double ry, double rz, bool in, const EwReal &ep,
                                            const double2 *__restrict__ tab, double &gx, double &gy, double &gz) {
  const EwImg m = ew_prep(rx, ry, rz, in, ep);
  double2 cc[kEwNC2];
  ew_load(m, tab, cc);
  ew_pin(cc, kEwNC2);
  ew_finish(m, cc, ep, gx, gy, gz);
}

// Energy of one image, q erfc(alpha r) / r, from the energy table.
__device__ __forceinline__ void ew_energy(const EwImg &m, const double2 *cc, const EwReal &ep, double &e) {
  double h = fma(cc[kEwNC2 - 1].y, m.y, cc[kEwNC2 - 1].x);
#pragma unroll
  for (int k = kEwNC2 - 2; k >= 0; --k) {
    h = fma(h, m.y, cc[k].y);
    h = fma(h, m.y, cc[k].x);
  }
  e += m.in ? ep.q * h * m.ir : 0.0;
}

// Force of a pair into g, or (ENERGY, tab the energy table) its energy into gx.
template <int IMG, bool ENERGY = false>
__device__ __forceinline__ void ewald_pair_tab(double dx, double dy, double dz, const EwReal &ep,
                                               const double2 *__restrict__ tab, double &gx, double &gy,
                                               double &gz) {
  const double ax = fma(-ep.L[0], rint(dx * ep.iL[0]), dx);
  const double ay = fma(-ep.L[1], rint(dy * ep.iL[1]), dy);
  const double az = fma(-ep.L[2], rint(dz * ep.iL[2]), dz);
  const double sx = copysign(ep.L[0], ax), sy = copysign(ep.L[1], ay), sz = copysign(ep.L[2], az);
  const double bx = ax - sx, by = ay - sy, bz = az - sz;
  const double ax2 = ax * ax, ay2 = ay * ay, az2 = az * az;
  const double bx2 = bx * bx, by2 = by * by, bz2 = bz * bz;
  const double rc2 = ep.rc2;
  const double xy[4] = {ax2 + ay2, bx2 + ay2, ax2 + by2, bx2 + by2};
  if (IMG == IMG_FACE) {
    const bool kx = xy[1] + az2 <= rc2, ky = xy[2] + az2 <= rc2, kz = xy[0] + bz2 <= rc2;
    const EwImg m0 = ew_prep(ax, ay, az, xy[0] + az2 <= rc2, ep);
    const EwImg m1 = ew_prep(kx ? bx : ax, ky ? by : ay, kz ? bz : az, kx || ky || kz, ep);
    double2 cc[2 * kEwNC2];
    ew_load(m0, tab, cc);
    ew_load(m1, tab, cc + kEwNC2);
    ew_pin(cc, 2 * kEwNC2);
    if (ENERGY) {
      ew_energy(m0, cc, ep, gx);
      ew_energy(m1, cc + kEwNC2, ep, gx);
    } else {
      ew_finish(m0, cc, ep, gx, gy, gz);
      ew_finish(m1, cc + kEwNC2, ep, gx, gy, gz);
    }
    return;
  }
  unsigned lo = 0, hi = 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const double R2 = xy[q & 3] + ((q & 4) ? bz2 : az2);
    const int pos = (q & 1) | ((q & 2) << 1) | ((q & 4) << 2);
    lo |= (R2 <= rc2) ? (1u << pos) : 0u;
  }
  if (IMG == IMG_CORNER) {
    const double cx = ax + sx, cy = ay + sy, cz = az + sz;
    const double cx2 = cx * cx, cy2 = cy * cy, cz2 = cz * cz;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k1 = u & 1, k2 = u >> 1;
      // c in x: (c, k1, k2); c in y: (k1, c, k2); c in z: (k1, k2, c)
      const double Rx = cx2 + (k1 ? by2 : ay2) + (k2 ? bz2 : az2);
      const double Ry = (k1 ? bx2 : ax2) + cy2 + (k2 ? bz2 : az2);
      const double Rz = xy[k1 | (k2 << 1)] + cz2;
      lo |= (Rx <= rc2) ? (1u << (3 | (k1 << 2) | (k2 << 4))) : 0u;
      lo |= (Ry <= rc2) ? (1u << (k1 | (3 << 2) | (k2 << 4))) : 0u;
      hi |= (Rz <= rc2) ? (1u << ((k1 | (k2 << 2) | (3 << 4)) - 32)) : 0u;
    }
  }
  unsigned long long m = ((unsigned long long)hi << 32) | lo;
  while (m) {
    const int pos = __builtin_ctzll(m);
    m &= m - 1;
    const double kx = (double)((pos << 30) >> 30), ky = (double)((pos << 28) >> 30), kz = (double)((pos << 26) >> 30);
    if (ENERGY) {
      const EwImg im = ew_prep(fma(-kx, sx, ax), fma(-ky, sy, ay), fma(-kz, sz, az), true, ep);
      double2 cc[kEwNC2];
      ew_load(im, tab, cc);
      ew_pin(cc, kEwNC2);
      ew_energy(im, cc, ep, gx);
    } else {
      ewald_image(fma(-kx, sx, ax), fma(-ky, sy, ay), fma(-kz, sz, az), true, ep, tab, gx, gy, gz);
    }
  }
}

// Rotates a double one lane down the wave (lane i takes lane i+1's value,
// lane 63 lane 0's); every lane of the wave must be active.
__device__ __forceinline__ double wave_rol1(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x134, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x134, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// WPB waves per workgroup, one tile pair per wave (the erfc table is staged
// once per workgroup); every choice computes the same partial sums.  Items
// run over the off-diagonal tile pairs of every slice first and the diagonal
// ones (half the rotation steps' work) last: tiles holds a slice's noff =
// ntp - T off-diagonal pairs followed by its T diagonal ones.  The grid's
// last workgroups, the fifth on some compute units when the grid holds 4.25
// waves per SIMD, then carry half a tile pair's work.  Lane t
// holds bead i = I*64 + t of tile I and, at step s, the record of bead
// j = J*64 + (t + s) mod 64 of tile J (its position and the reaction
// accumulated so far); the records move one lane down the wave after each
// step (DPP rotation, no LDS), so after 64 steps every record is home.  Each
// reaction thus gathers its terms in step order, lane t's own force likewise.
template <int IMG, int WPB = 4>
__device__ __forceinline__ void k_ewald_real_body(int bx, const double *__restrict__ X, const double *__restrict__ M,
                                                    double *__restrict__ Fpart, const int2 *__restrict__ tiles, int N,
                                                    int nb, int T, int ntp, int nitems, EwReal ep, double add = 0.0) {
  __shared__ double2 tab[kEwTabIntervals * kEwTabStride / 2];
  // the wave index and everything derived from it are wave-uniform: read
  // them as such, so the step loop below runs on scalar registers
  const int tid = threadIdx.x, t = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int k = tid; k < kEwTabIntervals * kEwTabStride / 2; k += 64 * WPB)
    tab[k] = make_double2(kEwTab[2 * k], kEwTab[2 * k + 1]);
  __syncthreads();
  const int item = bx * WPB + w;
  if (item >= nitems) return;
  const int noff = ntp - T, P = nitems / ntp;
  int slice, idx;
  if (item < P * noff) {
    slice = item / noff;
    idx = item - slice * noff;
  } else {
    slice = (item - P * noff) / T;
    idx = noff + (item - P * noff - slice * T);
  }
  const int2 IJ = tiles[idx];
  const int I = __builtin_amdgcn_readfirstlane(IJ.x), J = __builtin_amdgcn_readfirstlane(IJ.y);
  const int base = slice * N;
  const int i = I * 64 + t, jl = J * 64 + t;
  const bool act = i < N, jact = jl < N;
  double xi = 0, yi = 0, zi = 0, wi = 1;
  if (act) {
    xi = X[base + i];
    yi = X[nb + base + i];
    zi = X[2 * nb + base + i];
    wi = 1.0 / M[base + i];
  }
  double jx = jact ? X[base + jl] : 0.0, jy = jact ? X[nb + base + jl] : 0.0, jz = jact ? X[2 * nb + base + jl] : 0.0;
  double rx = 0, ry = 0, rz = 0;
  const bool diag = I == J, full = J * 64 + 64 <= N;
  double fx = 0, fy = 0, fz = 0;
  auto step = [&](bool on) {
    if (on) {
      double gx = 0, gy = 0, gz = 0;
      ewald_pair_tab<IMG>(xi - jx, yi - jy, zi - jz, ep, tab, gx, gy, gz);
      // the pair's force over the mass of its higher-index bead; the table
      // kernels run only for equal masses, so that is this lane's 1 / m_i
      const double iw = wi;
      fx = fma(gx, iw, fx);
      fy = fma(gy, iw, fy);
      fz = fma(gz, iw, fz);
      rx -= gx * iw;
      ry -= gy * iw;
      rz -= gz * iw;
    }
    jx = wave_rol1(jx);
    jy = wave_rol1(jy);
    jz = wave_rol1(jz);
    rx = wave_rol1(rx);
    ry = wave_rol1(ry);
    rz = wave_rol1(rz);
  };
  // an off-diagonal pair of full tiles meets a partner on every lane at
  // every step; a diagonal tile takes s = 1..31 and only lanes t < 32 at
  // s = 32 (each pair once), its remaining steps only rotate the records home
  const bool every = !diag && full && I * 64 + 64 <= N;  // wave-uniform
  for (int s = 0; s < 64; ++s) {
    bool on = true;
    if (!every) {
      const int j = (t + s) & 63;
      on = act && (full || J * 64 + j < N);
      if (diag) on = on && (s >= 1 && s <= 32) && (s < 32 || t < 32);
    }
    step(on);
  }
  auto put = [&](int bead, int slot, double vx, double vy, double vz) {
    const size_t s0 = (size_t)slot * 3 * nb + base + bead;
    put_tile(Fpart + s0, vx, add);
    put_tile(Fpart + s0 + nb, vy, add);
    put_tile(Fpart + s0 + 2 * (size_t)nb, vz, add);
  };
  if (diag) {
    if (act) put(i, I, fx + rx, fy + ry, fz + rz);
  } else {
    if (act) put(i, J, fx, fy, fz);
    if (jact) put(jl, I, rx, ry, rz);
  }
}

// Register budget for five waves per SIMD (every wave of the workload is
// resident at once; more registers keep the table loads of a step in
// flight together).
template <int IMG, int WPB>
__global__ __launch_bounds__(64 * WPB) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_ewald_real(const double *__restrict__ X, const double *__restrict__ M,
                                                         double *__restrict__ Fpart, const int2 *__restrict__ tiles,
                                                         int N, int nb, int T, int ntp, int nitems, EwReal ep, double add) {
  k_ewald_real_body<IMG, WPB>(blockIdx.x, X, M, Fpart, tiles, N, nb, T, ntp, nitems, ep, add);
}

// Real-space energy of every tile pair, items and rotation as in
// k_ewald_real (only the partner positions move), erfc from the energy table:
// UEG N=1024 P=32 (near images) 347 -> 110 us against k_pair_tiles, whose lanes walk their own
// image lists with an exp and a 20-term erfc series per image.
template <int IMG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_ewald_real_energy(
    const double *__restrict__ X, double *__restrict__ Epart, const int2 *__restrict__ tiles, int N, int nb, int T,
    int ntp, int nitems, EwReal ep) {
  __shared__ double2 tab[kEwTabIntervals * kEwTabStride / 2];
  const int tid = threadIdx.x, t = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int k = tid; k < kEwTabIntervals * kEwTabStride / 2; k += 256)
    tab[k] = make_double2(kEwTabE[2 * k], kEwTabE[2 * k + 1]);
  __syncthreads();
  const int item = blockIdx.x * 4 + w;
  if (item >= nitems) return;
  const int noff = ntp - T, P = nitems / ntp;
  int slice, idx;
  if (item < P * noff) {
    slice = item / noff;
    idx = item - slice * noff;
  } else {
    slice = (item - P * noff) / T;
    idx = noff + (item - P * noff - slice * T);
  }
  const int2 IJ = tiles[idx];
  const int I = __builtin_amdgcn_readfirstlane(IJ.x), J = __builtin_amdgcn_readfirstlane(IJ.y);
  const int base = slice * N;
  const int i = I * 64 + t, jl = J * 64 + t;
  const bool act = i < N, jact = jl < N;
  const double xi = act ? X[base + i] : 0.0, yi = act ? X[nb + base + i] : 0.0, zi = act ? X[2 * nb + base + i] : 0.0;
  double jx = jact ? X[base + jl] : 0.0, jy = jact ? X[nb + base + jl] : 0.0, jz = jact ? X[2 * nb + base + jl] : 0.0;
  const bool diag = I == J, full = J * 64 + 64 <= N;
  double e = 0, none = 0;
  auto step = [&](bool on) {
    if (on) ewald_pair_tab<IMG, true>(xi - jx, yi - jy, zi - jz, ep, tab, e, none, none);
    jx = wave_rol1(jx);
    jy = wave_rol1(jy);
    jz = wave_rol1(jz);
  };
  const bool every = !diag && full && I * 64 + 64 <= N;  // wave-uniform
  const int last = diag ? 32 : 63;
  for (int s = 0; s <= last; ++s) {
    bool on = true;
    if (!every) {
      const int j = (t + s) & 63;
      on = act && (full || J * 64 + j < N);
      if (diag) on = on && s >= 1 && (s < 32 || t < 32);
    }
    step(on);
  }
  e = wave_sum(e);
  if (t == 0) Epart[item] = e;
}

// ------------------------------------------------------------ launchers

int pair_kind_of(md_pair_force_t_x pf) {
  if (pf == md_gaussian_force_x) return PK_GAUSS;
  if (pf == md_periodic_gaussian_force_x) return PK_PGAUSS;
  if (pf == md_coulomb_3d_ewald_force_x) return PK_EWALD;
  if (pf == md_coulomb_3d_ewald_force_R_x) return PK_EWALD_R;
  if (pf == md_coulomb_3d_ewald_force_NI_x) return PK_EWALD_NI;
  if (pf == md_LJ_periodic_force_x) return PK_LJ;
  if (pf == md_periodic_helium_force_x) return PK_HE;
  return -1;
}

int pair_energy_kind_of(md_pair_energy_t_x pe) {
  if (pe == md_gaussian_energy_x) return PK_GAUSS;
  if (pe == md_periodic_gaussian_energy_x) return PK_PGAUSS;
  if (pe == md_coulomb_3d_ewald_energy_x) return PK_EWALD;
  if (pe == md_coulomb_3d_ewald_energy_R_x) return PK_EWALD_R;
  if (pe == md_coulomb_3d_ewald_energy_R2_x) return PK_EWALD_R2;
  if (pe == md_coulomb_3d_ewald_energy_NI_x) return PK_EWALD_NI;
  if (pe == md_LJ_periodic_energy_x) return PK_LJ;
  if (pe == md_periodic_helium_energy_x) return PK_HE;
  return -1;
}

// Cutoff of both Ewald series in units of the split: real space within
// x_cut / alpha, k space within pi |G| / alpha <= x_cut.  The omitted terms
// are below erfc(5.25) = 1.4e-13 and exp(-5.25^2) = 1.1e-12 of the leading
// ones; at N = 1024, P = 32 the forces differ from the reference's converged
// sum by 1.4e-13 of the RMS force (x_cut = 6: 4e-14, the rounding floor),
// for 20 % less work per step.
double g_ewald_xcut = 5.25;

// Energies are per-sample estimators, not per-step work: they sum both Ewald
// series to x_cut >= 6, where the omitted terms are at the rounding floor.
static double energy_xcut() { return std::max(g_ewald_xcut, 6.0); }

static PairParams make_params(DevPimd *p, double xcut = g_ewald_xcut) {
  PairParams pp;
  pp.xcut = xcut;
  md_simulation_t_x *sim = p->host->sim;
  for (int d = 0; d < 3; ++d) pp.L[d] = box_L(sim, d);
  pp.g = md_gaussian_strength_x;
  pp.s2 = md_gaussian_range_x * md_gaussian_range_x;
  pp.q = md_coulomb_strength_x;
  pp.alpha = md_coulomb_truc_x;
  double rc = xcut / md_coulomb_truc_x;
  pp.rc2 = rc * rc;
  pp.nsum = md_coulomb_n_sum_x;
  pp.P = (double)p->P;
  const double he[8] = {md_he_eps_x, md_he_A_x, md_he_alpha_x, md_he_C6_x,
                        md_he_C8_x,  md_he_C10_x, md_he_D_x,   md_he_rm_x};
  for (int k = 0; k < 8; ++k) pp.he[k] = he[k];
  return pp;
}

static int ensure_tiles(DevPimd *p) {
  const int N = p->N, P = p->P;
  TileBufs &B = pair_bufs(p)->tb;
  if (B.N != N) {
    ++g_pair_allocs;
    int T = (N + 63) / 64;
    std::vector<int2> tl;
    for (int I = 0; I < T; ++I)
      for (int J = I; J < T; ++J) tl.push_back(make_int2(I, J));
    std::vector<int2> tr;
    for (const int2 &ij : tl)
      if (ij.x != ij.y) tr.push_back(ij);
    for (const int2 &ij : tl)
      if (ij.x == ij.y) tr.push_back(ij);
    if (B.tiles) (void)hipFree(B.tiles);
    if (B.tiles_r) (void)hipFree(B.tiles_r);
    XMD_CHECK(hipMalloc(&B.tiles, tl.size() * sizeof(int2)));
    XMD_CHECK(hipMemcpy(B.tiles, tl.data(), tl.size() * sizeof(int2), hipMemcpyHostToDevice));
    XMD_CHECK(hipMalloc(&B.tiles_r, tr.size() * sizeof(int2)));
    XMD_CHECK(hipMemcpy(B.tiles_r, tr.data(), tr.size() * sizeof(int2), hipMemcpyHostToDevice));
    B.N = N;
    B.T = T;
    B.ntp = (int)tl.size();
  }
  size_t fneed = (size_t)3 * N * P * B.T, eneed = (size_t)P * B.ntp;
  if (fneed > B.fcap) {
    ++g_pair_allocs;
    if (B.Fpart) (void)hipFree(B.Fpart);
    XMD_CHECK(hipMalloc(&B.Fpart, fneed * sizeof(double)));
    B.fcap = fneed;
  }
  if (eneed > B.ecap) {
    ++g_pair_allocs;
    if (B.Epart) (void)hipFree(B.Epart);
    XMD_CHECK(hipMalloc(&B.Epart, eneed * sizeof(double)));
    B.ecap = eneed;
  }
  const size_t rneed = (size_t)3 * N * P;
  if (rneed > B.rcap) {
    ++g_pair_allocs;
    if (B.Frec) (void)hipFree(B.Frec);
    XMD_CHECK(hipMalloc(&B.Frec, rneed * sizeof(double)));
    B.rcap = rneed;
  }
  return 0;
}

// The near-image enumeration covers every image within r_c when
// r_c < sqrt(2) L and the reference's image cube (|n| <= n_sum around the raw
// separation) holds all of them, i.e. n_sum >= 3 for wrapped positions.
static int near_ok(const PairParams &pp) {
  double Lmin = fmin(pp.L[0], fmin(pp.L[1], pp.L[2]));
  // (the image kernel's erfc series also needs alpha r_c <= 6.5)
  return (pp.nsum >= 3 && pp.rc2 < 2.0 * Lmin * Lmin && pp.alpha * sqrt(pp.rc2) <= 6.5) ? 1 : 0;
}

template <int MODE, bool ENERGY>
static int launch_pair_mode(DevPimd *p, const PairParams &pp, hipStream_t st, double *esum, bool reduce = true) {
  DevSim *d = p->ds;
  if (ensure_tiles(p)) return -1;
  TileBufs &B = pair_bufs(p)->tb;
  const bool near = (MODE == PK_EWALD_NI) || (MODE == PK_EWALD_R2) || near_ok(pp);
  const int items = p->P * B.ntp;
  const bool direct = !ENERGY && reduce && B.T == 1;  // one tile: straight into F
  double *out = direct ? d->F : B.Fpart;
  const double add = direct ? pp.P : 0.0;
  if (near)
    hipLaunchKernelGGL((k_pair_tiles<MODE, ENERGY, true>), dim3(items), dim3(64), 0, st, d->X, d->M, out,
                       B.Epart, B.tiles, p->N, d->nb, B.T, B.ntp, pp, add);
  else
    hipLaunchKernelGGL((k_pair_tiles<MODE, ENERGY, false>), dim3(items), dim3(64), 0, st, d->X, d->M, out,
                       B.Epart, B.tiles, p->N, d->nb, B.T, B.ntp, pp, add);
  XMD_CHECK(hipGetLastError());
  if (ENERGY) return device_sum(B.Epart, items, esum);
  if (!reduce || direct) return 0;
  const int n3 = 3 * d->nb;
  hipLaunchKernelGGL(k_reduce_tiles, dim3((n3 + 255) / 256), dim3(256), 0, st, B.Fpart, d->F, n3, B.T, pp.P);
  XMD_CHECK(hipGetLastError());
  return 0;
}

// ------------------------------------------------------------ Ewald plan
//
// The Ewald sum does not depend on the split alpha once both of its series
// are converged.  When the reference's own parameters are converged -- its
// first omitted k shell has exp(-pi^2 (n+1)^2 / (alpha L_max)^2) <= 1e-13
// and its real-space image cube reaches erfc(alpha n L_min) < 1e-16 -- the
// engine evaluates the same sum with a split of its own: alpha', real space
// within x_cut / alpha' and k in the ball pi |G| / alpha' <= x_cut (dropped
// terms below exp(-x_cut^2) relative).  The result then differs from the
// reference's only by the reference's own truncation (<= 1e-13 relative) and
// rounding.  g_ewald_split_aL: 0 keeps the reference's alpha and k cube,
// > 0 fixes alpha' L_min, < 0 lets the cost model below choose.
double g_ewald_split_aL = -1.0;

static double lmin3(const double *L) { return fmin(L[0], fmin(L[1], L[2])); }
static double lmax3(const double *L) { return fmax(L[0], fmax(L[1], L[2])); }

static bool ref_converged(const PairParams &pp) {
  const int n = pp.nsum;
  if (n < 1 || !(pp.alpha > 0)) return false;
  const double a = M_PI * (n + 1) / (pp.alpha * lmax3(pp.L));
  return a * a >= 30.0 && pp.alpha * n * lmin3(pp.L) >= 6.0;
}

// Modelled device time (ps) of a split alpha L_min = aL, fitted to the
// kernels' measured times on MI355X (UEG, N = 256 .. 2048, P = 16 .. 32).
// Real space per pair: 6.5 ps with the face enumeration (two candidate images
// whatever r_c), else 1.0 + 5.2 ps per image inside r_c (11 + 2.1 when
// r_c >= L admits third copies); never below one wave's walk over its tile
// pair, about 5.9e6 pair costs (small systems do not fill the device).
// Reciprocal space 0.42 ps
// per (bead, padded k slot) plus 12 us per 32 slices.
static double split_cost(const PairParams &pp, int N, int P, double aL) {
  const double Lmin = lmin3(pp.L), V = pp.L[0] * pp.L[1] * pp.L[2];
  const double alpha = aL / Lmin, rc = pp.xcut / alpha;
  const double images = 4.0 / 3.0 * M_PI * rc * rc * rc / V;
  double per_pair;
  if (rc * rc < 0.5 * Lmin * Lmin * (1.0 - 1e-6))
    per_pair = 6.5;
  else if (rc >= Lmin)
    per_pair = 11.0 + 2.1 * images;
  else
    per_pair = 1.0 + 5.2 * images;
  const double real = std::max(P * 0.5 * N * (N - 1.0), 5.9e6) * per_pair;
  const double gmax = pp.xcut * alpha / M_PI;
  int M = 0;
  for (int d = 0; d < 3; ++d) M = std::max(M, (int)floor(gmax * pp.L[d]));
  const int MZ = table_mz(M);
  if (MZ < 0) return 1e300;
  long ncol = 0;
  for (int mx = 0; mx <= M; ++mx)
    for (int my = -M; my <= M; ++my)
      if ((mx > 0 || my >= 0) && (mx / pp.L[0]) * (mx / pp.L[0]) + (my / pp.L[1]) * (my / pp.L[1]) <= gmax * gmax)
        ++ncol;
  const double slots = (double)((ncol + 15) / 16 * 16) * (2 * MZ + 2);
  return real + 0.42 * N * P * slots + 12e6 * P / 32.0;
}

static bool split_ok(const PairParams &pp, double aL) {
  const double Lmin = lmin3(pp.L), alpha = aL / Lmin, rc = pp.xcut / alpha;
  const double gmax = pp.xcut * alpha / M_PI;
  return rc * rc < 2.0 * Lmin * Lmin && pp.xcut <= 6.5 && gmax * lmax3(pp.L) <= MAX_KM;
}

static EwaldPlan plan_ewald(const PairParams &pp, int N, int P) {
  EwaldPlan e;
  e.alpha = pp.alpha;
  e.rc2 = pp.rc2;
  e.cube_n = pp.nsum;
  if (g_ewald_split_aL == 0.0 || !ref_converged(pp)) return e;
  double aL = g_ewald_split_aL;
  if (aL < 0) {
    double best = 0;
    for (int h = 18; h <= 48; ++h) {  // alpha L_min = 4.5 .. 12 in steps of 1/4
      const double c = 0.25 * h;
      if (!split_ok(pp, c)) continue;
      const double w = split_cost(pp, N, P, c);
      if (aL < 0 || w < best) {
        best = w;
        aL = c;
      }
    }
    if (aL < 0) return e;
  } else if (!split_ok(pp, aL)) {
    return e;
  }
  const double alpha = aL / lmin3(pp.L), rc = pp.xcut / alpha, gmax = pp.xcut * alpha / M_PI;
  e.alpha = alpha;
  e.rc2 = rc * rc;
  e.gmax2 = gmax * gmax;
  e.cube_n = -1;
  e.own_split = true;
  return e;
}

// Parameters of the full Ewald interaction under its plan.
static PairParams planned(PairParams pp, const EwaldPlan &pl) {
  if (pl.own_split) {
    pp.alpha = pl.alpha;
    pp.rc2 = pl.rc2;
    pp.nsum = 1 << 20;  // coverage comes from r_c alone
  }
  return pp;
}

static PairParams ewald_params(DevPimd *p, EwaldPlan &pl, double xcut = g_ewald_xcut) {
  const PairParams pp = make_params(p, xcut);
  pl = plan_ewald(pp, p->N, p->P);
  return planned(pp, pl);
}

// Image enumeration of the real-space kernel for the cutoff of pp (the face
// bound keeps a relative margin of 1e-6 against rounding of the distances).
struct RealChoice {
  int img;   // IMG_FACE / IMG_NEAR / IMG_CORNER
  int wlog;  // log2 of the waves per workgroup (0..3)
};

static int image_mode(const PairParams &pp) {
  const double L2 = lmin3(pp.L) * lmin3(pp.L);
  if (pp.rc2 < 0.5 * L2 * (1.0 - 1e-6)) return IMG_FACE;
  return pp.rc2 >= L2 ? IMG_CORNER : IMG_NEAR;
}

// ---- launch choices of the real-space kernel and their autotuner ----
//
// Result-preserving choices: the image enumeration (every variant at least as
// general as the geometry needs takes the same images in the same order with
// the same arithmetic; an out-of-range candidate adds an exact zero) and the
// waves per workgroup (each wave owns whole tile pairs and their partial-sum
// slots).  Without tuning: the most specific enumeration, 4 waves.  The
// autotuner times every valid choice on an object's current positions and
// keeps the fastest per bucket (N rounded up to a power of two, P, and the
// most specific valid enumeration).
using RealKern = void (*)(const double *, const double *, double *, const int2 *, int, int, int, int, int, EwReal, double);
static const RealKern k_ewald_real_of[3][4] = {
    {k_ewald_real<IMG_FACE, 1>, k_ewald_real<IMG_FACE, 2>, k_ewald_real<IMG_FACE, 4>, k_ewald_real<IMG_FACE, 8>},
    {k_ewald_real<IMG_NEAR, 1>, k_ewald_real<IMG_NEAR, 2>, k_ewald_real<IMG_NEAR, 4>, k_ewald_real<IMG_NEAR, 8>},
    {k_ewald_real<IMG_CORNER, 1>, k_ewald_real<IMG_CORNER, 2>, k_ewald_real<IMG_CORNER, 4>,
     k_ewald_real<IMG_CORNER, 8>}};

int g_autotune = 0;                      // use tuned choices
static int g_real_force_img = -1, g_real_force_wlog = -1;  // fixed choice (diagnostics), -1: none
static std::map<long long, RealChoice> g_real_tuned;

static long long real_bucket(int N, int P, int img_min) {
  long long nb2 = 1;
  while (nb2 < N) nb2 <<= 1;
  return (nb2 << 24) | ((long long)P << 4) | img_min;
}

RealChoice real_choice(int N, int P, const PairParams &pp) {
  const int img_min = image_mode(pp);
  RealChoice c{img_min, 2};
  if (g_real_force_img >= img_min) c.img = g_real_force_img;
  if (g_real_force_wlog >= 0) c.wlog = g_real_force_wlog;
  if (g_real_force_img < 0 && g_real_force_wlog < 0 && g_autotune) {
    auto it = g_real_tuned.find(real_bucket(N, P, img_min));
    if (it != g_real_tuned.end()) c = it->second;
  }
  return c;
}

// Table-driven real space: per-tile partial forces (k_ewald_real), then
// their sum into F (k_reduce_tiles) unless `reduce` is false.
// Event recorded after the tabulated real-space kernel (before its partial-
// force reduction) while a serial stage profile runs; g_real_probe_hit tells
// the profile that it was.
static hipEvent_t g_real_probe = nullptr;
static bool g_real_probe_hit = false;

void set_real_space_probe(hipEvent_t e) {
  g_real_probe = e;
  g_real_probe_hit = false;
}

bool real_space_probe_hit() { return g_real_probe_hit; }

static EwReal real_args(const PairParams &pp) {
  EwReal ep;
  for (int k = 0; k < 3; ++k) {
    ep.L[k] = pp.L[k];
    ep.iL[k] = 1.0 / pp.L[k];
  }
  ep.q = pp.q;
  ep.al8 = kEwTabInvWidth * pp.alpha;
  ep.rc2 = pp.rc2;
  return ep;
}

static int launch_ewald_real_tab(DevPimd *p, const PairParams &pp, hipStream_t st, bool reduce = true) {
  DevSim *d = p->ds;
  if (ensure_tiles(p)) return -1;
  TileBufs &B = pair_bufs(p)->tb;
  const EwReal ep = real_args(pp);
  const int items = p->P * B.ntp;
  const RealChoice ch = real_choice(p->N, p->P, pp);
  const int wpb = 1 << ch.wlog;
  const bool direct = reduce && B.T == 1;  // one tile: straight into F
  hipLaunchKernelGGL(k_ewald_real_of[ch.img][ch.wlog], dim3((items + wpb - 1) / wpb), dim3(64 * wpb), 0, st, d->X, d->M,
                     direct ? d->F : B.Fpart, B.tiles_r, p->N, d->nb, B.T, B.ntp, items, ep, direct ? pp.P : 0.0);
  XMD_CHECK(hipGetLastError());
  if (g_real_probe) {
    XMD_CHECK(hipEventRecord(g_real_probe, st));
    g_real_probe_hit = true;
  }
  if (!reduce || direct) return 0;
  const int n3 = 3 * d->nb;
  hipLaunchKernelGGL(k_reduce_tiles, dim3((n3 + 255) / 256), dim3(256), 0, st, B.Fpart, d->F, n3, B.T, pp.P);
  XMD_CHECK(hipGetLastError());
  return 0;
}

static void (*const k_ewald_real_energy_of[3])(const double *, double *, const int2 *, int, int, int, int, int,
                                               EwReal) = {
    k_ewald_real_energy<IMG_FACE>, k_ewald_real_energy<IMG_NEAR>, k_ewald_real_energy<IMG_CORNER>};

// Tabulated real-space energies of every tile pair into Epart (P * ntp).
static int launch_ewald_real_energy(DevPimd *p, const PairParams &pp, hipStream_t st) {
  if (ensure_tiles(p)) return -1;
  TileBufs &B = pair_bufs(p)->tb;
  const int items = p->P * B.ntp;
  hipLaunchKernelGGL(k_ewald_real_energy_of[image_mode(pp)], dim3((items + 3) / 4), dim3(256), 0, st, p->ds->X, B.Epart,
                     B.tiles_r, p->N, p->ds->nb, B.T, B.ntp, items, real_args(pp));
  XMD_CHECK(hipGetLastError());
  return 0;
}

static void (*const k_sk_of[4])(const double2 *, const double2 *, const double2 *, const int2 *, const double *, int,
                                int, int, int, double2 *, double2 *) = {k_sk_mfma<1>, k_sk_mfma<2>, k_sk_mfma<3>,
                                                                         k_sk_mfma<4>};
static void (*const k_frc_of[4])(const double2 *, const double2 *, const double2 *, const int2 *, int, int,
                                 const double2 *, const double *, double *, int, int, int, double, double, double,
                                 double, double *) = {k_recip_force_mfma<1>, k_recip_force_mfma<2>, k_recip_force_mfma<3>,
                                            k_recip_force_mfma<4>};
static void (*const k_frs_of[4])(const double2 *, const double2 *, const double2 *, const int2 *, int, int,
                                 const double2 *, const double *, double *, int, int, int, double, double, double,
                                 double, double *) = {k_recip_force_split<1>, k_recip_force_split<2>, k_recip_force_split<3>,
                                            k_recip_force_split<4>};

// Phase tables of every slice (reads X only) for the k set of pp.
static int launch_recip_phase(DevPimd *p, const PairParams &pp, int cube_n, double gmax2, hipStream_t st,
                              KSpace **out) {
  DevSim *d = p->ds;
  KSpace *K = ensure_kspace(p, pp.L, pp.alpha, pp.q, cube_n, gmax2, d->nb, p->P);
  if (!K) return -1;
  *out = K;
  hipLaunchKernelGGL(k_phase, dim3((phase_entries(d->nb, K->MZ) + 255) / 256), dim3(256), 0, st, d->X, d->nb, K->MZ,
                     pp.L[0], pp.L[1], pp.L[2], K->tx, K->ty, K->tz);
  XMD_CHECK(hipGetLastError());
  return 0;
}

// Structure factors S and the force operands of every slice from the phase tables.
static int launch_sk(DevPimd *p, const KSpace *K, hipStream_t st) {
  hipLaunchKernelGGL(k_sk_of[K->ZP / 16 - 1], dim3((K->ncolp / 16) * p->P), dim3(256), 0, st, K->tx, K->ty, K->tz,
                     K->cols, K->coef, K->ncolp, K->MZ, p->N, p->P, K->S, K->W);
  XMD_CHECK(hipGetLastError());
  return 0;
}

// Phase tables, then structure factors S and the force operands (reads X only).
static int launch_recip_sk(DevPimd *p, const PairParams &pp, int cube_n, double gmax2, hipStream_t st,
                           KSpace **out) {
  if (launch_recip_phase(p, pp, cube_n, gmax2, st, out)) return -1;
  return launch_sk(p, *out, st);
}

// Reciprocal forces from the tables and W of launch_recip_sk, added into F
// (Frec null) or stored in Frec.
static int launch_recip_force(DevPimd *p, const PairParams &pp, const KSpace *K, hipStream_t st,
                              double *Frec = nullptr) {
  DevSim *d = p->ds;
  // fewer workgroups of 64 beads than compute units: 16 beads each, column
  // tiles dealt to the waves (stage of phases, structure factors and forces,
  // us, without -> with: N=16 P=32 34 -> 25, N=128 P=64 45 -> 36, N=333 P=27
  // 48 -> 45.5; N=512 P=32, one workgroup a unit, 51.5 -> 61.5)
  const bool split = frc_tiles(p->N) * p->P < 256;
  hipLaunchKernelGGL((split ? k_frs_of : k_frc_of)[K->ZP / 16 - 1],
                     dim3((split ? frc_split_tiles(p->N) : frc_tiles(p->N)) * p->P), dim3(256), 0, st, K->tx,
                     K->ty, K->tz, K->cols, K->ncolp, K->MZ, K->W, d->M, d->F, p->N, d->nb, p->P, pp.L[0], pp.L[1], pp.L[2], pp.P,
                     Frec);
  XMD_CHECK(hipGetLastError());
  return 0;
}

static int launch_recip(DevPimd *p, const PairParams &pp, int cube_n, double gmax2, hipStream_t st, bool force,
                        KSpace **out) {
  KSpace *K = nullptr;
  if (launch_recip_sk(p, pp, cube_n, gmax2, st, &K)) return -1;
  if (out) *out = K;
  return force ? launch_recip_force(p, pp, K, st) : 0;
}

int launch_pair_real(DevPimd *p, int kind, hipStream_t st, bool reduce) {
  PairParams pp = make_params(p);
  switch (kind) {
    case PK_GAUSS:
      return launch_pair_mode<PK_GAUSS, false>(p, pp, st, nullptr, reduce);
    case PK_PGAUSS:
      return launch_pair_mode<PK_PGAUSS, false>(p, pp, st, nullptr, reduce);
    case PK_LJ:
      return launch_pair_mode<PK_LJ, false>(p, pp, st, nullptr, reduce);
    case PK_HE:
      return launch_pair_mode<PK_HE, false>(p, pp, st, nullptr, reduce);
    case PK_EWALD:
    case PK_EWALD_R:
    case PK_EWALD_NI:
      if (!p->ds->uniform_mass) {
        fprintf(stderr, "xmd: the Ewald kernels need equal bead masses\n");
        return -1;
      }
      if (kind == PK_EWALD) {
        EwaldPlan pl;
        pp = ewald_params(p, pl);
        if (near_ok(pp)) return launch_ewald_real_tab(p, pp, st, reduce);
        return launch_pair_mode<PK_EWALD, false>(p, pp, st, nullptr, reduce);
      }
      if (kind == PK_EWALD_R) return launch_pair_mode<PK_EWALD_R, false>(p, pp, st, nullptr, reduce);
      return launch_pair_mode<PK_EWALD_NI, false>(p, pp, st, nullptr, reduce);
    default:
      return -1;
  }
}

bool pair_has_recip(int kind) { return kind == PK_EWALD || kind == PK_EWALD_R; }

// Times every valid real-space launch choice on the object's current
// positions (one warm-up, then `reps` launches each, HIP events on the main
// stream) and keeps the fastest for the object's bucket.  ms[4 img + wlog]:
// average milliseconds per launch, -1 for invalid choices.
int autotune_real(DevPimd *p, int reps, double *ms, int *choice) {
  DevSim *d = p->ds;
  if (!d->uniform_mass) return -1;
  EwaldPlan pl;
  PairParams pp = ewald_params(p, pl);
  if (!near_ok(pp) || ensure_tiles(p)) return -1;
  TileBufs &B = pair_bufs(p)->tb;
  const EwReal ep = real_args(pp);
  const int items = p->P * B.ntp, img_min = image_mode(pp);
  hipStream_t st = rt().s0;
  hipEvent_t e0, e1;
  XMD_CHECK(hipEventCreate(&e0));
  XMD_CHECK(hipEventCreate(&e1));
  RealChoice best{img_min, 2};
  double tbest = 1e300;
  for (int img = 0; img < 3; ++img)
    for (int wl = 0; wl < 4; ++wl) {
      if (ms) ms[4 * img + wl] = -1;
      if (img < img_min) continue;
      const int wpb = 1 << wl;
      auto launch = [&]() {
        hipLaunchKernelGGL(k_ewald_real_of[img][wl], dim3((items + wpb - 1) / wpb), dim3(64 * wpb), 0, st, d->X,
                           d->M, B.Fpart, B.tiles_r, p->N, d->nb, B.T, B.ntp, items, ep, 0.0);
      };
      launch();
      XMD_CHECK(hipEventRecord(e0, st));
      for (int r = 0; r < reps; ++r) launch();
      XMD_CHECK(hipEventRecord(e1, st));
      XMD_CHECK(hipEventSynchronize(e1));
      XMD_CHECK(hipGetLastError());
      float t = 0;
      XMD_CHECK(hipEventElapsedTime(&t, e0, e1));
      const double avg = (double)t / reps;
      if (ms) ms[4 * img + wl] = avg;
      if (avg < tbest) {
        tbest = avg;
        best = RealChoice{img, wl};
      }
    }
  XMD_CHECK(hipEventDestroy(e0));
  XMD_CHECK(hipEventDestroy(e1));
  g_real_tuned[real_bucket(p->N, p->P, img_min)] = best;
  if (choice) {
    choice[0] = best.img;
    choice[1] = best.wlog;
  }
  return 0;
}

// With autotuning on: tune the object's bucket unless it is tuned already.
int autotune_if_needed(DevPimd *p, int kind) {
  if (!g_autotune || kind != PK_EWALD || !p->ds->uniform_mass) return 0;
  EwaldPlan pl;
  PairParams pp = ewald_params(p, pl);
  if (!near_ok(pp) || g_real_tuned.count(real_bucket(p->N, p->P, image_mode(pp)))) return 0;
  return autotune_real(p, 5, nullptr, nullptr);
}

int launch_pair_recip(DevPimd *p, int kind, hipStream_t st) {
  if (kind == PK_EWALD) {
    EwaldPlan pl;
    PairParams pp = ewald_params(p, pl);
    return launch_recip(p, pp, pl.cube_n, pl.gmax2, st, true, nullptr);
  }
  PairParams pp = make_params(p);
  return launch_recip(p, pp, pp.nsum, 0.0, st, true, nullptr);
}

static void (*const k_frce_of[4])(const double2 *, const double2 *, const double2 *, const int2 *, int, int,
                                  const double2 *, const double *, int, int, int, double, double, double, double,
                                  double *, double *, double) = {k_recip_force_energy<1>, k_recip_force_energy<2>,
                                                                 k_recip_force_energy<3>, k_recip_force_energy<4>};

int launch_recip_labels(DevPimd *p, double *Frec, double *Erec, hipStream_t st, double *alpha_out) {
  DevSim *d = p->ds;
  if (!d->uniform_mass) {
    fprintf(stderr, "xmd: the Ewald kernels need equal bead masses\n");
    return -1;
  }
  EwaldPlan pl;
  PairParams pp = ewald_params(p, pl);
  if (alpha_out) *alpha_out = pp.alpha;
  KSpace *K = nullptr;
  if (launch_recip_sk(p, pp, pl.cube_n, pl.gmax2, st, &K)) return -1;
  hipLaunchKernelGGL(k_frce_of[K->ZP / 16 - 1], dim3(frc_tiles(p->N) * p->P), dim3(256), 0, st, K->tx, K->ty,
                     K->tz, K->cols, K->ncolp, K->MZ, K->W, d->M, p->N, d->nb, p->P, pp.L[0], pp.L[1], pp.L[2], pp.P,
                     Frec, Erec, K->e0);
  XMD_CHECK(hipGetLastError());
  return 0;
}

int launch_recip_shells(DevPimd *p, int nlow, double *Frec, double *Erec, hipStream_t st) {
  DevSim *d = p->ds;
  if (!d->uniform_mass || nlow < 1) return -1;
  EwaldPlan pl;
  PairParams pp = ewald_params(p, pl);
  const double Lmax = std::max(pp.L[0], std::max(pp.L[1], pp.L[2]));
  const double g = (nlow + 1e-6) / Lmax;  // |m| <= nlow along the longest side
  KSpace *K = nullptr;
  if (launch_recip_sk(p, pp, -1, g * g, st, &K)) return -1;
  hipLaunchKernelGGL(k_frce_of[K->ZP / 16 - 1], dim3(frc_tiles(p->N) * p->P), dim3(256), 0, st, K->tx, K->ty,
                     K->tz, K->cols, K->ncolp, K->MZ, K->W, d->M, p->N, d->nb, p->P, pp.L[0], pp.L[1], pp.L[2], pp.P,
                     Frec, Erec, K->e0);
  XMD_CHECK(hipGetLastError());
  return 0;
}

double ewald_split_alpha(DevPimd *p) {
  EwaldPlan pl;
  return ewald_params(p, pl).alpha;
}

bool pair_ewald_tab(DevPimd *p, int kind, EwaldPlan &pl) {
  return kind == PK_EWALD && p->ds->uniform_mass && near_ok(ewald_params(p, pl));
}

int launch_pair_ewald_real(DevPimd *p, const EwaldPlan &pl, hipStream_t st) {
  const PairParams pp = planned(make_params(p), pl);
  if (ensure_tiles(p) || launch_ewald_real_tab(p, pp, st, false)) return -1;
  // the learned stand-in (or the judge step: exact terms plus the
  // surrogate's for comparison) fills the reciprocal-force buffer here
  return p->sur_mode ? surrogate_kspace(p, pair_bufs(p)->tb.Frec, st) : 0;
}

int launch_pair_kspace(DevPimd *p, const EwaldPlan &pl, hipStream_t st) {
  if (p->sur_mode) return 0;
  const PairParams pp = planned(make_params(p), pl);
  KSpace *K = nullptr;
  if (ensure_tiles(p) || launch_recip_phase(p, pp, pl.cube_n, pl.gmax2, st, &K) || launch_sk(p, K, st) ||
      launch_recip_force(p, pp, K, st, pair_bufs(p)->tb.Frec))
    return -1;
  return 0;
}

// F += real-space tile sums / P, then the reciprocal forces, then (when Fx
// is given) the exchange forces of the end beads.
__global__ __launch_bounds__(256) void k_combine_forces(double *__restrict__ F, ForceSums c, int n3) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n3) return;
  F[k] = combined_force(F, c, n3, k);
}

int force_sums(DevPimd *p, const double *Fx, bool recip, ForceSums *out) {
  TileBufs &B = pair_bufs(p)->tb;
  ForceSums c;
  c.Fpart = B.Fpart;
  c.Frec = recip ? B.Frec : nullptr;
  c.Fx = Fx;
  c.T = B.T;
  c.N = p->N;
  c.P = p->P;
  *out = c;
  return 0;
}

int launch_combine_forces(DevPimd *p, const double *Fx, hipStream_t st) {
  ForceSums c;
  if (force_sums(p, Fx, true, &c)) return -1;
  const int n3 = 3 * p->ds->nb;
  hipLaunchKernelGGL(k_combine_forces, dim3((n3 + 255) / 256), dim3(256), 0, st, p->ds->F, c, n3);
  XMD_CHECK(hipGetLastError());
  return 0;
}

int pair_prepare(DevPimd *p, int kind) {
  const unsigned a0 = g_pair_allocs;
  if (kind < 0) return 0;
  if (ensure_tiles(p)) return -1;
  if (kind == PK_EWALD && p->ds->uniform_mass) {
    EwaldPlan pl;
    PairParams pp = ewald_params(p, pl);
    if (!ensure_kspace(p, pp.L, pp.alpha, pp.q, pl.cube_n, pl.gmax2, p->ds->nb, p->P)) return -1;
  } else if (kind == PK_EWALD_R) {
    PairParams pp = make_params(p);
    if (!ensure_kspace(p, pp.L, pp.alpha, pp.q, pp.nsum, 0.0, p->ds->nb, p->P)) return -1;
  }
  return g_pair_allocs != a0 ? 1 : 0;
}

int launch_pair_force(DevPimd *p, int kind, hipStream_t st) {
  if (launch_pair_real(p, kind, st)) return -1;
  if (pair_has_recip(kind)) return launch_pair_recip(p, kind, st);
  return 0;
}

int pair_energy(DevPimd *p, int kind, double *out) {
  PairParams pp = make_params(p, energy_xcut());
  DevSim *d = p->ds;
  hipStream_t st = rt().s0;
  double e = 0;  // every unordered pair once
  if (kind == PK_GAUSS) {
    if (launch_pair_mode<PK_GAUSS, true>(p, pp, st, &e)) return -1;
  } else if (kind == PK_PGAUSS) {
    if (launch_pair_mode<PK_PGAUSS, true>(p, pp, st, &e)) return -1;
  } else if (kind == PK_LJ) {
    if (launch_pair_mode<PK_LJ, true>(p, pp, st, &e)) return -1;
  } else if (kind == PK_HE) {
    if (launch_pair_mode<PK_HE, true>(p, pp, st, &e)) return -1;
  } else if (kind == PK_EWALD) {
    EwaldPlan pl;
    pp = ewald_params(p, pl, energy_xcut());
    // tabulated when the near images hold the whole real-space sum: then both
    // sums are queued before the one wait for their results
    const bool tab = near_ok(pp);
    if (tab ? launch_ewald_real_energy(p, pp, st) : launch_pair_mode<PK_EWALD, true>(p, pp, st, &e)) return -1;
    KSpace *K = nullptr;
    if (launch_recip(p, pp, pl.cube_n, pl.gmax2, st, false, &K)) return -1;
    const int nb2 = 256;
    hipLaunchKernelGGL(k_recip_energy, dim3(nb2), dim3(256), 0, st, K->S, K->coef, K->ncolp * K->ZP, p->P, p->N,
                       d->red);
    XMD_CHECK(hipGetLastError());
    const TileBufs &B = pair_bufs(p)->tb;
    const double *src[2] = {d->red, B.Epart};
    const int cnt[2] = {nb2, p->P * B.ntp};
    double er[2] = {0, 0};
    if (device_sums(src, cnt, tab ? 2 : 1, er)) return -1;
    if (tab) e = er[1];
    const double V = pp.L[0] * pp.L[1] * pp.L[2];
    const double bg = -pp.q * M_PI / (pp.alpha * pp.alpha * V) * 0.5 * p->N * (p->N - 1) * p->P;
    e += er[0] + bg;
  } else if (kind == PK_EWALD_NI) {
    if (launch_pair_mode<PK_EWALD_NI, true>(p, pp, st, &e)) return -1;
  } else if (kind == PK_EWALD_R || kind == PK_EWALD_R2) {
    // the reference's own alpha and k cube (as the R force split): real
    // space without the minimum image, reciprocal space, background; R2
    // adds -erf(alpha r)/r of the minimum image
    if (!d->uniform_mass) {
      fprintf(stderr, "xmd: the Ewald kernels need equal bead masses\n");
      return -1;
    }
    if (launch_pair_mode<PK_EWALD_R, true>(p, pp, st, &e)) return -1;
    if (kind == PK_EWALD_R2) {
      double e2 = 0;
      if (launch_pair_mode<PK_EWALD_R2, true>(p, pp, st, &e2)) return -1;
      e += e2;
    }
    KSpace *K = nullptr;
    if (launch_recip(p, pp, pp.nsum, 0.0, st, false, &K)) return -1;
    const int nb2 = 256;
    hipLaunchKernelGGL(k_recip_energy, dim3(nb2), dim3(256), 0, st, K->S, K->coef, K->ncolp * K->ZP, p->P, p->N,
                       d->red);
    XMD_CHECK(hipGetLastError());
    double er = 0;
    if (device_sum(d->red, nb2, &er)) return -1;
    const double V = pp.L[0] * pp.L[1] * pp.L[2];
    const double bg = -pp.q * M_PI / (pp.alpha * pp.alpha * V) * 0.5 * p->N * (p->N - 1) * p->P;
    e += er + bg;
  } else {
    return -1;
  }
  *out = e / p->P;
  return 0;
}

// ------------------------------------------------------- two species
//
// md_pimd_x.c:3282-3510 (nocl): every pair of bead (l, j) of species A and
// bead (l2, j) of species B in the same slice j,
//   f_A += F(x_A, x_B) / m_A / P,   f_B -= m_A (F / m_A) / P / m_B,
//   E   += e(x_A, x_B) / P,
// with F, e the pair callback's force and energy.  Two passes (lane = bead
// of A, then lane = bead of B), each summing its partners of the slice in a
// fixed order: deterministic without atomics.
template <int MODE, bool ON_B>
__global__ __launch_bounds__(256) void k_pair2_force(const double *__restrict__ XA, const double *__restrict__ MA,
                                                     double *__restrict__ FA, int NA, int nbA,
                                                     const double *__restrict__ XB, const double *__restrict__ MB,
                                                     double *__restrict__ FB, int NB, int nbB, PairParams pp) {
  const int slice = blockIdx.y;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int Nt = ON_B ? NB : NA, No = ON_B ? NA : NB;
  if (i >= Nt) return;
  const double *Xt = ON_B ? XB : XA, *Xo = ON_B ? XA : XB;
  const int nbt = ON_B ? nbB : nbA, nbo = ON_B ? nbA : nbB;
  const int st = slice * Nt + i;
  const double xt = Xt[st], yt = Xt[nbt + st], zt = Xt[2 * nbt + st];
  double gx = 0, gy = 0, gz = 0, e = 0;
  for (int j = 0; j < No; ++j) {
    const int so = slice * No + j;
    const double xo = Xo[so], yo = Xo[nbo + so], zo = Xo[2 * nbo + so];
    // force on the A bead of the pair, from the B bead
    if (ON_B)
      pair_term<MODE, false, true>(xo - xt, yo - yt, zo - zt, pp, gx, gy, gz, e);
    else
      pair_term<MODE, false, true>(xt - xo, yt - yo, zt - zo, pp, gx, gy, gz, e);
  }
  double *Ft = ON_B ? FB : FA;
  const double s = ON_B ? -1.0 / (pp.P * MB[st]) : 1.0 / (MA[st] * pp.P);
  Ft[st] += gx * s;
  Ft[nbt + st] += gy * s;
  Ft[2 * nbt + st] += gz * s;
}

template <int MODE>
__global__ __launch_bounds__(256) void k_pair2_energy(const double *__restrict__ XA, int NA, int nbA,
                                                      const double *__restrict__ XB, int NB, int nbB, PairParams pp,
                                                      double *__restrict__ part) {
  __shared__ double red[256];
  const int slice = blockIdx.y;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double e = 0;
  if (i < NA) {
    const int sa = slice * NA + i;
    const double xa = XA[sa], ya = XA[nbA + sa], za = XA[2 * nbA + sa];
    double gx, gy, gz;
    for (int j = 0; j < NB; ++j) {
      const int sb = slice * NB + j;
      pair_term<MODE, true, true>(xa - XB[sb], ya - XB[nbB + sb], za - XB[2 * nbB + sb], pp, gx, gy, gz, e);
    }
  }
  red[threadIdx.x] = e;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.y * gridDim.x + blockIdx.x] = red[0];
}

static bool pair2_kind_ok(int kind) { return kind == PK_GAUSS || kind == PK_PGAUSS || kind == PK_LJ || kind == PK_HE; }

static int pair2_check(md_pimd_t_x *a, md_pimd_t_x *b, int kind) {
  if (a->P != b->P) return -1;
  if (!pair2_kind_ok(kind)) {
    fprintf(stderr, "xmd: two-species pair kernels cover the Gaussian, Lennard-Jones and helium interactions\n");
    return -1;
  }
  if (ensure_pimd_device(a) || ensure_pimd_device(b)) return -1;
  return 0;
}

template <int MODE>
static void launch_pair2_force(DevPimd *a, DevPimd *b, const PairParams &pp, hipStream_t st) {
  DevSim *da = a->ds, *db = b->ds;
  const dim3 ga((a->N + 255) / 256, a->P), gb((b->N + 255) / 256, b->P);
  hipLaunchKernelGGL((k_pair2_force<MODE, false>), ga, dim3(256), 0, st, da->X, da->M, da->F, a->N, da->nb, db->X,
                     db->M, db->F, b->N, db->nb, pp);
  hipLaunchKernelGGL((k_pair2_force<MODE, true>), gb, dim3(256), 0, st, da->X, da->M, da->F, a->N, da->nb, db->X,
                     db->M, db->F, b->N, db->nb, pp);
}

template <int MODE>
static void launch_pair2_energy(DevPimd *a, DevPimd *b, const PairParams &pp, hipStream_t st, double *part) {
  DevSim *da = a->ds, *db = b->ds;
  const dim3 g((a->N + 255) / 256, a->P);
  hipLaunchKernelGGL(k_pair2_energy<MODE>, g, dim3(256), 0, st, da->X, a->N, da->nb, db->X, b->N, db->nb, pp, part);
}

// ------------------------------------------------- batched replicas
//
// One launch per kernel over every replica that uses it: the Gaussian tile
// kernels (per mode), the tabulated Ewald real space (per image variant),
// and the three reciprocal-space kernels (their parts are added into F by NHC
// half 2).  Each
// replica's blocks run the single-system body with its own arguments;
// replicas whose interaction has no batched kernel are launched one by one.
struct PairRep {
  const double *X, *M;
  double *F, *Fpart, *Frec;
  const int2 *tiles, *tiles_r;
  int N, nb, T, ntp, P, items;
  PairParams pp;
  EwReal ep;
  double2 *tx, *ty, *tz, *S, *W;
  const int2 *cols;
  const double *coef;
  int ncolp, MZ, ZP;
};

#define PAIR_REP const PairRep *__restrict__ reps, const int *__restrict__ start, int nrep
#define PAIR_R                                    \
  const int r = batch_rep(start, nrep, blockIdx.x); \
  const PairRep &R = reps[r];                     \
  const int bx = blockIdx.x - start[r];

template <int MODE>
__global__ __launch_bounds__(64) void kb_pair_tiles(PAIR_REP) {
  PAIR_R
  k_pair_tiles_body<MODE, false, true>(bx, R.X, R.M, R.Fpart, nullptr, R.tiles, R.N, R.nb, R.T, R.ntp, R.pp);
}

template <int IMG, int WPB>
__global__ __launch_bounds__(64 * WPB) void kb_ewald_real(PAIR_REP) {
  PAIR_R
  k_ewald_real_body<IMG, WPB>(bx, R.X, R.M, R.Fpart, R.tiles_r, R.N, R.nb, R.T, R.ntp, R.items, R.ep);
}

__global__ __launch_bounds__(256) void kb_phase(PAIR_REP) {
  PAIR_R
  k_phase_body(bx, R.X, R.nb, R.MZ, R.pp.L[0], R.pp.L[1], R.pp.L[2], R.tx, R.ty, R.tz);
}

template <int NZT>
__global__ __launch_bounds__(256) void kb_sk_mfma(PAIR_REP) {
  PAIR_R
  k_sk_mfma_body<NZT>(bx, R.tx, R.ty, R.tz, R.cols, R.coef, R.ncolp, R.MZ, R.N, R.P, R.S, R.W);
}

template <int NZT>
__global__ __launch_bounds__(256) void kb_recip_force_mfma(PAIR_REP) {
  PAIR_R
  k_recip_force_mfma_body<NZT>(bx, R.tx, R.ty, R.tz, R.cols, R.ncolp, R.MZ, R.W, R.M, R.F, R.N, R.nb, R.P,
                               R.pp.L[0], R.pp.L[1], R.pp.L[2], R.pp.P, R.Frec);
}

#undef PAIR_R
#undef PAIR_REP

// Batched kernel groups: G_GAUSS, G_PGAUSS (tiles), G_EW + image mode (Ewald
// real space: face, near, corner enumeration), G_PHASE / G_SK / G_FRC
// (reciprocal space; one group per slot-tile count ZP / 16 = 1..4).
enum { G_GAUSS, G_PGAUSS, G_EW, G_PHASE = G_EW + 12, G_SK, G_FRC = G_SK + 4, G_COUNT = G_FRC + 4 };

struct PairBatch {
  BatchTable g[G_COUNT];
  std::vector<std::pair<DevPimd *, int>> solo;  // (replica, pair kind) launched one by one
  std::vector<ForceSums> sums;                  // per item, what NHC half 2 adds into F
};

PairBatch *pair_batch_create(const std::vector<BatchItem> &items) {
  std::vector<PairRep> reps[G_COUNT];
  std::vector<int> blocks[G_COUNT];
  PairBatch *b = new PairBatch();
  auto fail = [&]() -> PairBatch * {
    pair_batch_free(b);
    return nullptr;
  };
  for (const BatchItem &it : items) {
    DevPimd *p = it.p;
    const int kind = it.pair_kind;
    b->sums.emplace_back();
    ForceSums &cs = b->sums.back();
    cs.Fx = p->Fx;
    cs.N = p->N;
    cs.P = p->P;
    if (kind < 0) continue;
    DevSim *d = p->ds;
    PairRep R{};
    R.X = d->X;
    R.M = d->M;
    R.F = d->F;
    R.N = p->N;
    R.nb = d->nb;
    R.P = p->P;
    PairParams pp = make_params(p);
    bool ew = false;
    if (kind == PK_EWALD && d->uniform_mass) {
      EwaldPlan pl;
      pp = ewald_params(p, pl);
      if (near_ok(pp)) {
        ew = true;
        KSpace *K = ensure_kspace(p, pp.L, pp.alpha, pp.q, pl.cube_n, pl.gmax2, d->nb, p->P);
        if (!K) return fail();
        R.tx = K->tx;
        R.ty = K->ty;
        R.tz = K->tz;
        R.S = K->S;
        R.W = K->W;
        R.cols = K->cols;
        R.coef = K->coef;
        R.ncolp = K->ncolp;
        R.MZ = K->MZ;
        R.ZP = K->ZP;
      }
    }
    if (!(ew || kind == PK_GAUSS || kind == PK_PGAUSS)) {
      b->solo.push_back({p, kind});
      continue;
    }
    if (ensure_tiles(p) || force_sums(p, p->Fx, ew, &cs)) return fail();
    TileBufs &B = pair_bufs(p)->tb;
    R.Fpart = B.Fpart;
    R.Frec = B.Frec;
    R.tiles = B.tiles;
    R.tiles_r = B.tiles_r;
    R.T = B.T;
    R.ntp = B.ntp;
    R.items = p->P * B.ntp;
    R.pp = pp;
    R.ep = real_args(pp);
    int grp;
    if (ew) {
      // Ewald real space grouped by launch choice (the autotuner's per bucket)
      const RealChoice ch = real_choice(p->N, p->P, pp);
      grp = G_EW + 4 * ch.img + ch.wlog;
      blocks[grp].push_back((R.items + (1 << ch.wlog) - 1) >> ch.wlog);
    } else {
      grp = kind == PK_GAUSS ? G_GAUSS : G_PGAUSS;
      blocks[grp].push_back(R.items);
    }
    reps[grp].push_back(R);
    if (ew) {
      reps[G_PHASE].push_back(R);
      blocks[G_PHASE].push_back((phase_entries(R.nb, R.MZ) + 255) / 256);
      const int nzt = R.ZP / 16;
      reps[G_SK + nzt - 1].push_back(R);
      blocks[G_SK + nzt - 1].push_back((R.ncolp / 16) * R.P);
      reps[G_FRC + nzt - 1].push_back(R);
      blocks[G_FRC + nzt - 1].push_back(frc_tiles(R.N) * R.P);
    }
  }
  for (int k = 0; k < G_COUNT; ++k)
    if (batch_table_make(b->g[k], reps[k].data(), sizeof(PairRep), blocks[k])) return fail();
  return b;
}

void pair_batch_free(PairBatch *b) {
  if (!b) return;
  for (auto &t : b->g) batch_table_free(t);
  delete b;
}

static void pair_batch_go(PairBatch *b, int k, void (*kern)(const PairRep *, const int *, int), int threads,
                          hipStream_t st) {
  const BatchTable &t = b->g[k];
  if (t.nrep == 0) return;
  hipLaunchKernelGGL(kern, dim3(t.total), dim3(threads), 0, st, (const PairRep *)t.reps, t.start, t.nrep);
}

const std::vector<ForceSums> &pair_batch_sums(PairBatch *b) { return b->sums; }

int pair_batch_real(PairBatch *b, hipStream_t st) {
  auto go = [&](int k, void (*kern)(const PairRep *, const int *, int), int threads) {
    pair_batch_go(b, k, kern, threads, st);
  };
  go(G_GAUSS, kb_pair_tiles<PK_GAUSS>, 64);
  go(G_PGAUSS, kb_pair_tiles<PK_PGAUSS>, 64);
  go(G_EW + 0, kb_ewald_real<IMG_FACE, 1>, 64);
  go(G_EW + 1, kb_ewald_real<IMG_FACE, 2>, 128);
  go(G_EW + 2, kb_ewald_real<IMG_FACE, 4>, 256);
  go(G_EW + 3, kb_ewald_real<IMG_FACE, 8>, 512);
  go(G_EW + 4, kb_ewald_real<IMG_NEAR, 1>, 64);
  go(G_EW + 5, kb_ewald_real<IMG_NEAR, 2>, 128);
  go(G_EW + 6, kb_ewald_real<IMG_NEAR, 4>, 256);
  go(G_EW + 7, kb_ewald_real<IMG_NEAR, 8>, 512);
  go(G_EW + 8, kb_ewald_real<IMG_CORNER, 1>, 64);
  go(G_EW + 9, kb_ewald_real<IMG_CORNER, 2>, 128);
  go(G_EW + 10, kb_ewald_real<IMG_CORNER, 4>, 256);
  go(G_EW + 11, kb_ewald_real<IMG_CORNER, 8>, 512);
  XMD_CHECK(hipGetLastError());
  return 0;
}

int pair_batch_kspace(PairBatch *b, hipStream_t st) {
  auto go = [&](int k, void (*kern)(const PairRep *, const int *, int), int threads) {
    pair_batch_go(b, k, kern, threads, st);
  };
  go(G_PHASE, kb_phase, 256);
  go(G_SK, kb_sk_mfma<1>, 256);
  go(G_SK + 1, kb_sk_mfma<2>, 256);
  go(G_SK + 2, kb_sk_mfma<3>, 256);
  go(G_SK + 3, kb_sk_mfma<4>, 256);
  go(G_FRC, kb_recip_force_mfma<1>, 256);
  go(G_FRC + 1, kb_recip_force_mfma<2>, 256);
  go(G_FRC + 2, kb_recip_force_mfma<3>, 256);
  go(G_FRC + 3, kb_recip_force_mfma<4>, 256);
  XMD_CHECK(hipGetLastError());
  return 0;
}

int pair_batch_solo(PairBatch *b, hipStream_t st) {
  for (auto &pk : b->solo)
    if (launch_pair_force(pk.first, pk.second, st)) return -1;
  return 0;
}

}  // namespace xmd


using namespace xmd;

extern "C" {

int md_pimd_calc_pair_force_x(md_pimd_t_x *pimd, md_pair_force_t_x pf) {
  int kind = pair_kind_of(pf);
  if (kind < 0) {
    fprintf(stderr, "xmd: pair-force callback has no device kernel\n");
    return -1;
  }
  if (ensure_pimd_device(pimd)) return -1;
  return launch_pair_force(pimd_state(pimd, false), kind, rt().s0);
}

int md_pimd_get_ewald_plan_x(md_pimd_t_x *pimd, md_num_t_x *alpha, md_num_t_x *r_cut, int *n_k) {
  if (ensure_pimd_device(pimd)) return -1;
  DevPimd *p = pimd_state(pimd, false);
  EwaldPlan pl;
  PairParams pp = ewald_params(p, pl);
  if (alpha) *alpha = pl.alpha;
  if (r_cut) *r_cut = sqrt(pl.rc2);
  if (n_k) {
    KSpace *K = ensure_kspace(p, pp.L, pp.alpha, pp.q, pl.cube_n, pl.gmax2, p->ds->nb, p->P);
    if (!K) return -1;
    *n_k = K->nk;
  }
  return 0;
}

int md_pimd_calc_pair_force_2_x(md_pimd_t_x *pimd, md_pimd_t_x *pimd2, md_pair_force_t_x pf) {
  const int kind = pair_kind_of(pf);
  if (pair2_check(pimd, pimd2, kind)) return -1;
  DevPimd *a = pimd_state(pimd, false), *b = pimd_state(pimd2, false);
  PairParams pp = make_params(a);
  hipStream_t st = rt().s0;
  switch (kind) {
    case PK_GAUSS: launch_pair2_force<PK_GAUSS>(a, b, pp, st); break;
    case PK_PGAUSS: launch_pair2_force<PK_PGAUSS>(a, b, pp, st); break;
    case PK_LJ: launch_pair2_force<PK_LJ>(a, b, pp, st); break;
    default: launch_pair2_force<PK_HE>(a, b, pp, st); break;
  }
  XMD_CHECK(hipGetLastError());
  return 0;
}

int md_pimd_calc_pair_energy_2_x(md_pimd_t_x *pimd, md_pimd_t_x *pimd2, md_pair_energy_t_x pe,
                                 md_stats_t_x *stats) {
  const int kind = pair_energy_kind_of(pe);
  if (pair2_check(pimd, pimd2, kind)) return -1;
  DevPimd *a = pimd_state(pimd, false), *b = pimd_state(pimd2, false);
  PairParams pp = make_params(a);
  hipStream_t st = rt().s0;
  const int nblk = ((a->N + 255) / 256) * a->P;
  double *part = nullptr;
  XMD_CHECK(hipMallocAsync((void **)&part, nblk * sizeof(double), st));
  switch (kind) {
    case PK_GAUSS: launch_pair2_energy<PK_GAUSS>(a, b, pp, st, part); break;
    case PK_PGAUSS: launch_pair2_energy<PK_PGAUSS>(a, b, pp, st, part); break;
    case PK_LJ: launch_pair2_energy<PK_LJ>(a, b, pp, st, part); break;
    default: launch_pair2_energy<PK_HE>(a, b, pp, st, part); break;
  }
  XMD_CHECK(hipGetLastError());
  double e = 0;
  const int rc = device_sum(part, nblk, &e);
  XMD_CHECK(hipFreeAsync(part, st));
  if (rc) return -1;
  stats->es[stats->N - 1] += e / a->P;
  return 0;
}

int md_pimd_calc_pair_energy_x(md_pimd_t_x *pimd, md_pair_energy_t_x pe, md_stats_t_x *stats) {
  int kind = pair_energy_kind_of(pe);
  if (kind < 0) {
    fprintf(stderr, "xmd: pair-energy callback has no device kernel\n");
    return -1;
  }
  if (ensure_pimd_device(pimd)) return -1;
  double e = 0;
  if (pair_energy(pimd_state(pimd, false), kind, &e)) return -1;
  stats->es[stats->N - 1] += e;
  return 0;
}

int md_set_autotune_x(int on) {
  g_autotune = on ? 1 : 0;
  return 0;
}

int md_set_ewald_real_variant_x(int img, int wlog) {
  if (img < -1 || img > 2 || wlog < -1 || wlog > 3) return -1;
  g_real_force_img = img;
  g_real_force_wlog = wlog;
  return 0;
}

int md_pimd_autotune_x(md_pimd_t_x *pimd, int reps, md_num_t_x *ms, int *choice) {
  if (reps < 1 || ensure_pimd_device(pimd)) return -1;
  return autotune_real(pimd_state(pimd, false), reps, ms, choice);
}

int md_autotune_save_x(const char *path) {
  FILE *f = fopen(path, "w");
  if (!f) return -1;
  fprintf(f, "# MI355X PIMD engine: Ewald real-space launch choices per (N bucket, P, enumeration) bucket\n");
  for (const auto &kv : g_real_tuned)
    fprintf(f, "%lld %lld %lld %d %d\n", kv.first >> 24, (kv.first >> 4) & 0xfffff, kv.first & 15, kv.second.img,
            kv.second.wlog);
  return fclose(f) == 0 ? 0 : -1;
}

int md_autotune_load_x(const char *path) {
  FILE *f = fopen(path, "r");
  if (!f) return -1;
  char line[256];
  int n = 0;
  while (fgets(line, sizeof line, f)) {
    if (line[0] == '#') continue;
    long long nb2, P, imin;
    int img, wl;
    if (sscanf(line, "%lld %lld %lld %d %d", &nb2, &P, &imin, &img, &wl) != 5 || img < imin || img > 2 || wl < 0 ||
        wl > 3) {
      fclose(f);
      return -1;
    }
    g_real_tuned[(nb2 << 24) | (P << 4) | imin] = RealChoice{img, wl};
    ++n;
  }
  fclose(f);
  return n;
}

}  // extern "C"
