// Per-sample observables on device-resident beads, nocl semantics:
// density distribution (md_pimd_x.c:1826-1967), imaginary-time correlation
// of x (ITCF, md_pimd_x.c:2723-2872), pair correlations (one and two systems,
// in-plane, and 2-D |dx|,|dy| histograms; md_pimd_x.c:2974-3280,4869-4956)
// and the structure factors S(q) on axes and on spherical shells
// (md_pimd_x.c:4958-5450, md_statistics_x.c:104-161).
//
// Histograms: the kernels count samples per bin with integer atomics (exact,
// order independent), each workgroup in LDS first (kLdsBins bins; 490,000
// pairs into 200 bins took 148 us as global atomics, whose bins are shared by
// all, 12 us this way), and k_hist_add adds the reference's increment (1/P or
// 1/norm) once per count to stats->fxs[stats->N-1][bin], which it reads and
// writes in pinned host memory.  Every bin only ever receives that one
// increment value, so the result equals the reference's sequential
// accumulation bit for bit.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>

#include "xmd_device.h"
#include "xmd_internal.h"

namespace xmd {

__device__ __forceinline__ double obs_dist(double dx, double dy, double dz, const double *L, int image) {
  if (image) {
    dx = dv_min_image(dx, L[0]);
    dy = dv_min_image(dy, L[1]);
    dz = dv_min_image(dz, L[2]);
  }
  return sqrt(dx * dx + dy * dy + dz * dz);
}

struct ObsGeo {
  double L[3];
  double c[3];
  double incre;
  int points, image;
};

// A workgroup's counts: in LDS (LDS true; points <= kLdsBins, dynamic shared
// memory of that many words), added to the global counts at the end, or
// straight into the global counts.
constexpr int kLdsBins = 12288;
constexpr int kHistWork = 4096;  // samples per workgroup of the pair histograms, about 20 per bin at 200 bins

template <bool LDS>
struct Hist {
  unsigned *lds;
  unsigned long long *cnt;
  int points;
  __device__ Hist(unsigned *l, unsigned long long *c, int n) : lds(l), cnt(c), points(n) {
    if (!LDS) return;
    for (int b = threadIdx.x; b < points; b += blockDim.x) lds[b] = 0;
    __syncthreads();
  }
  // bins below 0 or beyond the last are dropped
  __device__ void add(int b) {
    if ((unsigned)b >= (unsigned)points) return;
    if (LDS)
      atomicAdd(&lds[b], 1u);
    else
      atomicAdd(&cnt[b], 1ull);
  }
  __device__ void flush() {
    if (!LDS) return;
    __syncthreads();
    for (int b = threadIdx.x; b < points; b += blockDim.x)
      if (lds[b]) atomicAdd(&cnt[b], (unsigned long long)lds[b]);
  }
};

// Row and column of this workgroup's samples of a row-major (.. x n) matrix,
// thread tid taking samples tid, tid + 256, ... of [begin, begin + kHistWork).
struct RowCol {
  long row;
  int col, n, dr, dc;
  __device__ RowCol(long t, int n_) : row(t / n_), n(n_) {
    col = (int)(t - row * n);
    dr = 256 / n;
    dc = 256 - dr * n;
  }
  __device__ void next() {
    row += dr;
    col += dc;
    if (col >= n) {
      col -= n;
      ++row;
    }
  }
};

// md_pimd_x.c:1947-1962: every bead's distance to the center.
template <bool LDS>
__global__ __launch_bounds__(256) void k_density_hist(const double *__restrict__ X, int nb, ObsGeo g,
                                                      unsigned long long *__restrict__ cnt) {
  extern __shared__ unsigned bins[];
  Hist<LDS> h(bins, cnt, g.points);
  for (int s = blockIdx.x * 256 + threadIdx.x; s < nb; s += gridDim.x * 256) {
    const double r = obs_dist(X[s] - g.c[0], X[nb + s] - g.c[1], X[2 * nb + s] - g.c[2], g.L, g.image);
    h.add((int)(r / g.incre));
  }
  h.flush();
}

// Bead sets of a pair histogram: bead slots slot0 + l (l < N) of one
// system, in the slice-major layout X[d * nb + slot].
struct BeadSet {
  const double *X;
  int N, nb, slot0;
};

enum HistMode { HM_RADIAL = 0, HM_AXES2D = 1, HM_ITCF = 2 };

struct PairHist {
  BeadSet a, b;
  int mode;
  int same;   // a and b are one system: skip l == j
  int two;    // ITCF of two systems: count (i1, i2) and (i2, i1)
  int image;
  double L[3];
  double incre, rmin;
  int n, points;  // n = (int)sqrt(points) for the 2-D histograms
};

__device__ __forceinline__ int clamp_bin(int i1, int i2, int n, int points) {
  int idx = i1 * n + i2;
  if (idx < 0) idx = 0;
  if (idx >= points) idx = points - 1;
  return idx;
}

// Every (l of a, j of b):
//  HM_RADIAL (md_pimd_x.c:3019-3036, 3125-3136): bin (int)(r / incre), dropped beyond the last bin;
//  HM_AXES2D (md_pimd_x.c:4889-4909): bins (int)(|dx| / incre), (int)(|dy| / incre), clamped;
//  HM_ITCF   (md_pimd_x.c:2731-2746, 2851-2870): bins of (x - rmin) / incre along dimension 0, clamped.
template <bool LDS>
__global__ __launch_bounds__(256) void k_pair_hist(PairHist h, unsigned long long *__restrict__ cnt) {
  extern __shared__ unsigned bins[];
  Hist<LDS> H(bins, cnt, h.points);
  const long begin = (long)blockIdx.x * kHistWork, end = min(begin + kHistWork, (long)h.a.N * h.b.N);
  const double *XA = h.a.X, *XB = h.b.X;
  const int na = h.a.nb, nb = h.b.nb;
  RowCol at(begin + threadIdx.x, h.b.N);
  for (long t = begin + threadIdx.x; t < end; t += 256, at.next()) {
    const int l = (int)at.row, j = at.col;
    if (h.same && l == j) continue;
    const int sa = h.a.slot0 + l, sb = h.b.slot0 + j;
    if (h.mode == HM_RADIAL) {
      const double r =
          obs_dist(XA[sa] - XB[sb], XA[na + sa] - XB[nb + sb], XA[2 * na + sa] - XB[2 * nb + sb], h.L, h.image);
      H.add((int)(r / h.incre));
    } else if (h.mode == HM_AXES2D) {
      double dx = XA[sa] - XB[sb], dy = XA[na + sa] - XB[nb + sb];
      if (h.image) {
        dx = dv_min_image(dx, h.L[0]);
        dy = dv_min_image(dy, h.L[1]);
      }
      const int i1 = (int)(fabs(dx) / h.incre), i2 = (int)(fabs(dy) / h.incre);
      H.add(clamp_bin(i1, i2, h.n, h.points));
    } else {
      const int i1 = (int)((XA[sa] - h.rmin) / h.incre), i2 = (int)((XB[sb] - h.rmin) / h.incre);
      H.add(clamp_bin(i1, i2, h.n, h.points));
      if (h.two) H.add(clamp_bin(i2, i1, h.n, h.points));
    }
  }
  H.flush();
}

// md_pimd_x.c:3248-3278: in-plane distance of beads l != j of one slice,
// both inside the window box = {x0, x1, y0, y1}.
template <bool LDS>
__global__ __launch_bounds__(256) void k_paircorr_box2d(const double *__restrict__ X, int N, int nb, int P, double x0,
                                                        double x1, double y0, double y1, double incre, int points,
                                                        unsigned long long *__restrict__ cnt) {
  extern __shared__ unsigned bins[];
  Hist<LDS> H(bins, cnt, points);
  const long begin = (long)blockIdx.x * kHistWork, end = min(begin + kHistWork, (long)P * N * N);
  RowCol at(begin + threadIdx.x, N);
  for (long t = begin + threadIdx.x; t < end; t += 256, at.next()) {
    const int sa = (int)at.row, slice = sa / N, sb = slice * N + at.col;  // row: bead slot slice * N + l
    if (sa == sb) continue;
    const double ax = X[sa], ay = X[nb + sa], bx = X[sb], by = X[nb + sb];
    if (ax < x0 || ax > x1 || ay < y0 || ay > y1) continue;
    if (bx < x0 || bx > x1 || by < y0 || by > y1) continue;
    const double dx = ax - bx, dy = ay - by;
    const double r = sqrt(dx * dx + dy * dy);
    H.add((int)(r / incre));
  }
  H.flush();
}

// x + c, n times, each sum rounded (n repeated additions, bit for bit).
// While x stays in one binade every addition moves it by the same multiple of
// its last place (unless c lies midway between two, which rounds by parity),
// so all additions up to the binade's end are one product.
__host__ __device__ inline double add_repeated(double x, double c, unsigned long long n) {
  while (n) {
    const double y = x + c;
    if (!(c > 0.0) || !(x >= c) || !(y < 1e300) || n < 4) {  // the general case: one at a time
      if (y == x || y != y) return y;
      x = y;
      --n;
      continue;
    }
    const double d = y - x;  // exact, x <= y <= 2x
    if (d == 0.0) return x;
    int e;
    (void)frexp(x, &e);                                       // x in [2^(e-1), 2^e)
    const double top = ldexp(1.0, e), half = ldexp(1.0, e - 54);  // half of x's last place
    double k = floor((top - x) / d);
    if (k * d > top - x) k -= 1.0;
    if (k < 1.0 || fabs(c - d) == half) {
      x = y;
      --n;
      continue;
    }
    if (k > (double)n) k = (double)n;
    x += k * d;
    n -= (unsigned long long)k;
  }
  return x;
}

// fx[b] += incr, cnt[b] times; the counts are left zero for the next call.
__global__ __launch_bounds__(256) void k_hist_add(unsigned long long *__restrict__ cnt, double *__restrict__ fx,
                                                  int points, double incr) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b >= points) return;
  fx[b] = add_repeated(fx[b], incr, cnt[b]);
  cnt[b] = 0;
}

// S(q) of two bead sets (each the union of up to two BeadSets):
//   res(q) = sum [C1 C2 + S1 S2] / norm,  C = sum cos(q . x), S = sum sin(q . x),
// on axes (q along each dimension in turn, the three terms averaged;
// md_pimd_x.c:4967-4996, 5052-5083, 5152-5203) or for one q vector per point
// (md_pimd_x.c:5268-5340, 5344-5402, 5406-5450).  One workgroup per q point.
struct SkArgs {
  BeadSet s1[2], s2[2];
  int n1, n2;
  double norm;
  int sphere;
  double q0, qincre;
  const double *qis;  // sphere: 3 per point
};

__device__ __forceinline__ void sk_accum(const BeadSet &b, double qx, double qy, double qz, int axis, double &c,
                                         double &s) {
  for (int l = threadIdx.x; l < b.N; l += blockDim.x) {
    const int k = b.slot0 + l;
    const double t = axis >= 0 ? qx * b.X[axis * b.nb + k]
                               : qx * b.X[k] + qy * b.X[b.nb + k] + qz * b.X[2 * b.nb + k];
    double sn, cs;
    sincos(t, &sn, &cs);
    c += cs;
    s += sn;
  }
}

__global__ __launch_bounds__(256) void k_sk(SkArgs a, int j0, double *__restrict__ out) {
  __shared__ double red[4][256];
  const int j = j0 + blockIdx.x;
  double res = 0;
  const int nterm = a.sphere ? 1 : 3;
  for (int d = 0; d < nterm; ++d) {
    double qx, qy = 0, qz = 0;
    int axis;
    if (a.sphere) {
      qx = a.qis[3 * j];
      qy = a.qis[3 * j + 1];
      qz = a.qis[3 * j + 2];
      axis = -1;
    } else {
      qx = a.q0 + j * a.qincre;
      axis = d;
    }
    double c1 = 0, s1 = 0, c2 = 0, s2 = 0;
    for (int k = 0; k < a.n1; ++k) sk_accum(a.s1[k], qx, qy, qz, axis, c1, s1);
    for (int k = 0; k < a.n2; ++k) sk_accum(a.s2[k], qx, qy, qz, axis, c2, s2);
    red[0][threadIdx.x] = c1;
    red[1][threadIdx.x] = c2;
    red[2][threadIdx.x] = s1;
    red[3][threadIdx.x] = s2;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
      if ((int)threadIdx.x < w)
        for (int k = 0; k < 4; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + w];
      __syncthreads();
    }
    res += red[0][0] * red[1][0] / a.norm;
    res += red[2][0] * red[3][0] / a.norm;
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = a.sphere ? res : res / 3;
}

static int obs_geo(md_simulation_t_x *sim, ObsGeo &g) {
  for (int d = 0; d < 3; ++d) g.L[d] = box_L(sim, d);
  return 0;
}

// Device counts of at least `points` bins, all zero between calls (k_hist_add
// clears what it has read; a call that failed in between drops the buffer).
// g_counts_busy is held from obs_counts to the end of add_counts.
static std::mutex g_counts_busy;
static unsigned long long *g_counts = nullptr;
static int g_counts_cap = 0;

static void obs_counts_drop() {
  if (g_counts) (void)hipFree(g_counts);
  g_counts = nullptr;
  g_counts_cap = 0;
}

static unsigned long long *obs_counts(int points) {
  if (points > g_counts_cap) {
    obs_counts_drop();
    if (hipMalloc(&g_counts, points * sizeof(unsigned long long)) != hipSuccess) return nullptr;
    if (clear_device(g_counts, points * sizeof(unsigned long long))) {
      obs_counts_drop();
      return nullptr;
    }
    g_counts_cap = points;
  }
  return g_counts;
}

// counts -> stats->fxs[N-1][b] += incr, once per count
static int add_counts(md_stats_t_x *stats, int points, double incr) {
  HostScratch scratch(points);
  double *fx = stats->fxs[stats->N - 1], *h = scratch.p;
  const hipStream_t st = rt().s0;
  if (h) {
    memcpy(h, fx, points * sizeof(double));
    hipLaunchKernelGGL(k_hist_add, dim3((points + 255) / 256), dim3(256), 0, st, g_counts, h, points, incr);
  }
  if (!h || hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess) {
    fprintf(stderr, "xmd: histogram accumulation failed\n");
    obs_counts_drop();
    return -1;
  }
  memcpy(fx, h, points * sizeof(double));
  return 0;
}

// Bead slice `bead` (1-based) of every particle of a system.
static BeadSet bead_set(DevPimd *p, int bead) {
  BeadSet b;
  b.X = p->ds->X;
  b.N = p->N;
  b.nb = p->ds->nb;
  b.slot0 = (bead - 1) * p->N;
  return b;
}

static DevPimd *obs_pimd(md_pimd_t_x *pimd) {
  if (!pimd || ensure_pimd_device(pimd)) return nullptr;
  return pimd_state(pimd, false);
}

static int run_pair_hist(PairHist &h, md_stats_t_x *stats, double incr) {
  std::lock_guard<std::mutex> hold(g_counts_busy);
  unsigned long long *cnt = obs_counts(h.points);
  if (!cnt) return -1;
  const long work = (long)h.a.N * h.b.N;
  if (work > 0) {
    const dim3 grid((unsigned)((work + kHistWork - 1) / kHistWork));
    if (h.points <= kLdsBins)
      hipLaunchKernelGGL(k_pair_hist<true>, grid, dim3(256), h.points * sizeof(unsigned), rt().s0, h, cnt);
    else
      hipLaunchKernelGGL(k_pair_hist<false>, grid, dim3(256), 0, rt().s0, h, cnt);
  }
  return add_counts(stats, h.points, incr);
}

static PairHist pair_hist(DevPimd *a, int bead_a, DevPimd *b, int bead_b, md_simulation_t_x *box_sim, int mode,
                          int points) {
  PairHist h;
  h.a = bead_set(a, bead_a);
  h.b = bead_set(b, bead_b);
  h.mode = mode;
  h.same = 0;
  h.two = 0;
  h.image = 0;
  for (int d = 0; d < 3; ++d) h.L[d] = box_L(box_sim, d);
  h.incre = 0;
  h.rmin = 0;
  h.n = (int)sqrt((double)points);
  h.points = points;
  return h;
}

// S(q) for the points j < npts of stats, added into stats->fxs[N-1][j].
static int run_sk(SkArgs &a, md_stats_t_x *stats, int npts, const double *qis_host) {
  if (npts <= 0) return 0;
  hipStream_t st = rt().s0;
  HostScratch scratch(4 * (size_t)npts);
  double *out = scratch.p;  // results, then q vectors
  if (!out) return -1;
  a.qis = nullptr;
  if (a.sphere) {
    memcpy(out + npts, qis_host, 3 * npts * sizeof(double));
    a.qis = out + npts;
  }
  hipLaunchKernelGGL(k_sk, dim3(npts), dim3(256), 0, st, a, 0, out);
  XMD_CHECK(hipGetLastError());
  XMD_CHECK(hipStreamSynchronize(st));
  for (int j = 0; j < npts; ++j) stats->fxs[stats->N - 1][j] += out[j];
  return 0;
}

}  // namespace xmd

using namespace xmd;

extern "C" {

int md_pimd_calc_density_distribution_x(md_pimd_t_x *pimd, md_stats_t_x *stats, md_num_t_x rmax, int image,
                                        md_num_t_x *center) {
  if (!pimd || !stats || stats->points <= 0 || !center) return -1;
  if (ensure_pimd_device(pimd)) return -1;
  DevPimd *p = pimd_state(pimd, false);
  ObsGeo g;
  obs_geo(pimd->sim, g);
  for (int d = 0; d < 3; ++d) g.c[d] = center[d];
  g.incre = rmax / stats->points;
  g.points = stats->points;
  g.image = image;
  std::lock_guard<std::mutex> hold(g_counts_busy);
  unsigned long long *cnt = obs_counts(g.points);
  if (!cnt) return -1;
  const int nb = p->ds->nb;
  const dim3 grid(std::min((nb + 255) / 256, 128));
  if (g.points <= kLdsBins)
    hipLaunchKernelGGL(k_density_hist<true>, grid, dim3(256), g.points * sizeof(unsigned), rt().s0, p->ds->X, nb, g, cnt);
  else
    hipLaunchKernelGGL(k_density_hist<false>, grid, dim3(256), 0, rt().s0, p->ds->X, nb, g, cnt);
  return add_counts(stats, g.points, 1.0 / pimd->P);
}

int md_pimd_calc_pair_correlation_x(md_pimd_t_x *pimd, md_stats_t_x *stats, md_num_t_x rmax, md_num_t_x norm,
                                    int pi, int image) {
  DevPimd *p = obs_pimd(pimd);
  if (!p || !stats || stats->points <= 0 || pi < 1 || pi > pimd->P) return -1;
  PairHist h = pair_hist(p, 1, p, pi, pimd->sim, HM_RADIAL, stats->points);
  h.same = 1;
  h.image = image;
  h.incre = rmax / stats->points;
  return run_pair_hist(h, stats, 1.0 / norm);
}

int md_pimd_calc_pair_correlation_2_x(md_pimd_t_x *pimd, md_pimd_t_x *pimd2, md_stats_t_x *stats, md_num_t_x rmax,
                                      md_num_t_x norm, int pi, int image) {
  if (!pimd || !pimd2 || pimd->P != pimd2->P) return -1;
  DevPimd *a = obs_pimd(pimd), *b = obs_pimd(pimd2);
  if (!a || !b || !stats || stats->points <= 0 || pi < 1 || pi > pimd->P) return -1;
  PairHist h = pair_hist(a, 1, b, pi, pimd->sim, HM_RADIAL, stats->points);
  h.image = image;
  h.incre = rmax / stats->points;
  return run_pair_hist(h, stats, 1.0 / norm);
}

int md_pimd_calc_pair_correlation_2d_x(md_pimd_t_x *pimd, md_stats_t_x *stats, md_num_t_x rmax, md_num_t_x norm,
                                       md_num_t_x *box) {
  DevPimd *p = obs_pimd(pimd);
  if (!p || !stats || stats->points <= 0 || !box) return -1;
  const int points = stats->points;
  std::lock_guard<std::mutex> hold(g_counts_busy);
  unsigned long long *cnt = obs_counts(points);
  if (!cnt) return -1;
  const long work = (long)p->P * p->N * p->N;
  const dim3 grid((unsigned)((work + kHistWork - 1) / kHistWork));
  if (points <= kLdsBins)
    hipLaunchKernelGGL(k_paircorr_box2d<true>, grid, dim3(256), points * sizeof(unsigned), rt().s0, p->ds->X, p->N,
                       p->ds->nb, p->P, box[0], box[1], box[2], box[3], rmax / points, points, cnt);
  else
    hipLaunchKernelGGL(k_paircorr_box2d<false>, grid, dim3(256), 0, rt().s0, p->ds->X, p->N, p->ds->nb, p->P, box[0],
                       box[1], box[2], box[3], rmax / points, points, cnt);
  return add_counts(stats, points, 1.0 / norm);
}

int md_pimd_calc_2d_pair_correlation_x(md_pimd_t_x *pimd, md_stats_t_x *stats, md_num_t_x rmax, md_num_t_x norm,
                                       int pi, int image) {
  DevPimd *p = obs_pimd(pimd);
  if (!p || !stats || stats->points <= 0 || pi < 1 || pi > pimd->P) return -1;
  PairHist h = pair_hist(p, 1, p, pi, pimd->sim, HM_AXES2D, stats->points);
  h.same = 1;
  h.image = image;
  h.incre = rmax / h.n;
  return run_pair_hist(h, stats, 1.0 / norm);
}

int md_pimd_calc_2d_pair_correlation_2_x(md_pimd_t_x *pimd, md_pimd_t_x *pimd2, md_stats_t_x *stats,
                                         md_num_t_x rmax, md_num_t_x norm, int pi, int image) {
  if (!pimd || !pimd2 || pimd->P != pimd2->P) return -1;
  DevPimd *a = obs_pimd(pimd), *b = obs_pimd(pimd2);
  if (!a || !b || !stats || stats->points <= 0 || pi < 1 || pi > pimd->P) return -1;
  PairHist h = pair_hist(a, 1, b, pi, pimd->sim, HM_AXES2D, stats->points);
  h.image = image;
  h.incre = rmax / h.n;
  return run_pair_hist(h, stats, 1.0 / norm);
}

int md_pimd_calc_ITCF_x(md_pimd_t_x *pimd, md_stats_t_x *stats, md_num_t_x rmin, md_num_t_x rmax, int pi) {
  DevPimd *p = obs_pimd(pimd);
  if (!p || !stats || stats->points <= 0 || pi < 1 || pi > pimd->P) return -1;
  PairHist h = pair_hist(p, 1, p, pi, pimd->sim, HM_ITCF, stats->points);
  h.rmin = rmin;
  h.incre = (rmax - rmin) / h.n;
  return run_pair_hist(h, stats, 1.0 / pimd->P);
}

int md_pimd_calc_ITCF_2_x(md_pimd_t_x *pimd, md_pimd_t_x *pimd2, md_stats_t_x *stats, md_num_t_x rmin,
                          md_num_t_x rmax, int pi) {
  if (!pimd || !pimd2 || pimd->P != pimd2->P) return -1;
  DevPimd *a = obs_pimd(pimd), *b = obs_pimd(pimd2);
  if (!a || !b || !stats || stats->points <= 0 || pi < 1 || pi > pimd->P) return -1;
  PairHist h = pair_hist(a, 1, b, pi, pimd->sim, HM_ITCF, stats->points);
  h.two = 1;
  h.rmin = rmin;
  h.incre = (rmax - rmin) / h.n;
  return run_pair_hist(h, stats, 1.0 / pimd->P);
}

int md_pimd_calc_Sk_structure_x(md_pimd_t_x *pimd, md_stats_t_x *stats, md_num_t_x q0, md_num_t_x qincre, int pi) {
  DevPimd *p = obs_pimd(pimd);
  if (!p || !stats || stats->points <= 0 || pi < 1 || pi > pimd->P) return -1;
  SkArgs a{};
  a.s1[0] = bead_set(p, 1);
  a.s2[0] = bead_set(p, pi);
  a.n1 = a.n2 = 1;
  a.norm = p->N;
  a.q0 = q0;
  a.qincre = qincre;
  return run_sk(a, stats, stats->points, nullptr);
}

int md_pimd_calc_Sk_structure_2_x(md_pimd_t_x *pimd, md_pimd_t_x *pimd2, md_stats_t_x *stats, md_num_t_x q0,
                                  md_num_t_x qincre, int pi) {
  if (!pimd || !pimd2 || pimd->P != pimd2->P) return -1;
  DevPimd *p = obs_pimd(pimd), *p2 = obs_pimd(pimd2);
  if (!p || !p2 || !stats || stats->points <= 0 || pi < 1 || pi > pimd->P) return -1;
  SkArgs a{};
  a.s1[0] = bead_set(p, 1);
  a.s2[0] = bead_set(p2, pi);
  a.n1 = a.n2 = 1;
  a.norm = p->N;
  a.q0 = q0;
  a.qincre = qincre;
  return run_sk(a, stats, stats->points, nullptr);
}

int md_pimd_calc_Sk_structure_full_2_x(md_pimd_t_x *pimd, md_pimd_t_x *pimd2, md_stats_t_x *stats, md_num_t_x q0,
                                       md_num_t_x qincre, int pi) {
  if (!pimd || !pimd2 || pimd->P != pimd2->P) return -1;
  DevPimd *p = obs_pimd(pimd), *p2 = obs_pimd(pimd2);
  if (!p || !p2 || !stats || stats->points <= 0 || pi < 1 || pi > pimd->P) return -1;
  SkArgs a{};
  a.s1[0] = bead_set(p, 1);
  a.s1[1] = bead_set(p2, 1);
  a.s2[0] = bead_set(p, pi);
  a.s2[1] = bead_set(p2, pi);
  a.n1 = a.n2 = 2;
  a.norm = p->N + p2->N;
  a.q0 = q0;
  a.qincre = qincre;
  return run_sk(a, stats, stats->points, nullptr);
}

// Spherical variants: the second bead slice is (pi - 1) % P + 1 and the
// points are the first min(sk_sphere->N, stats->points) shells.
int md_pimd_calc_sphere_Sk_structure_x(md_pimd_t_x *pimd, md_stats_t_x *stats, int pi, md_sk_sphere_t_x *sk_sphere) {
  DevPimd *p = obs_pimd(pimd);
  if (!p || !stats || !sk_sphere || pi < 1) return -1;
  const int b2 = (pi - 1) % pimd->P + 1;
  SkArgs a{};
  a.s1[0] = bead_set(p, 1);
  a.s2[0] = bead_set(p, b2);
  a.n1 = a.n2 = 1;
  a.norm = p->N;
  a.sphere = 1;
  return run_sk(a, stats, std::min(sk_sphere->N, stats->points), sk_sphere->qis);
}

int md_pimd_calc_sphere_Sk_structure_full_2_x(md_pimd_t_x *pimd, md_pimd_t_x *pimd2, md_stats_t_x *stats, int pi,
                                              md_sk_sphere_t_x *sk_sphere) {
  if (!pimd || !pimd2 || pimd->P != pimd2->P) return -1;
  DevPimd *p = obs_pimd(pimd), *p2 = obs_pimd(pimd2);
  if (!p || !p2 || !stats || !sk_sphere || pi < 1) return -1;
  const int b2 = (pi - 1) % pimd->P + 1;
  SkArgs a{};
  a.s1[0] = bead_set(p, 1);
  a.s1[1] = bead_set(p2, 1);
  a.s2[0] = bead_set(p, b2);
  a.s2[1] = bead_set(p2, b2);
  a.n1 = a.n2 = 2;
  a.norm = p->N + p2->N;
  a.sphere = 1;
  return run_sk(a, stats, std::min(sk_sphere->N, stats->points), sk_sphere->qis);
}

int md_pimd_calc_sphere_Sk_structure_3_x(md_pimd_t_x *pimd, md_pimd_t_x *pimd2, md_pimd_t_x *pimd3,
                                         md_stats_t_x *stats, int pi, md_sk_sphere_t_x *sk_sphere) {
  if (!pimd || !pimd2 || !pimd3 || pimd->P != pimd2->P || pimd->P != pimd3->P) return -1;
  DevPimd *p = obs_pimd(pimd), *p2 = obs_pimd(pimd2), *p3 = obs_pimd(pimd3);
  if (!p || !p2 || !p3 || !stats || !sk_sphere || pi < 1) return -1;
  const int b2 = (pi - 1) % pimd->P + 1;
  SkArgs a{};
  a.s1[0] = bead_set(p, 1);
  a.s1[1] = bead_set(p2, 1);
  a.s2[0] = bead_set(p3, b2);
  a.n1 = 2;
  a.n2 = 1;
  a.norm = sqrt((double)((p->N + p2->N) * p3->N));
  a.sphere = 1;
  return run_sk(a, stats, std::min(sk_sphere->N, stats->points), sk_sphere->qis);
}

}  // extern "C"
