// The fused MD step and its hipGraph capture, plus run-time knobs.
//
// Stages of one step (the reference driver's): NHC half 1 (+ wrap), cycle
// energies and recursion set-up, recursions, end-bead exchange forces (into a
// side buffer), bead-local forces (reset, trap, springs), pair forces (for
// Ewald: real space; phase tables, structure factors, reciprocal forces, all
// into side buffers), sum of the parts, NHC half 2 (one kernel with massive
// thermostats, as are NHC half 1 with the wrap and the bead-local forces).
// Everything between the NHC halves reads positions only, so the exchange
// chain and the pair branch may run side by side; which parts go beside which
// depends on how much of the device the pair kernels fill (Order below).
// The serial profiling order runs every stage on s0.
//
// Batches of independent replicas (md_pimd_run_batch_x) run the same stages
// with one launch per stage over a packed table of all replicas, captured
// into one hipGraph per batch step.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "md_hip_x.h"
#include "xmd_internal.h"

namespace xmd {

struct StepPlan {
  DevPimd *p = nullptr;
  int trap = 0;
  int pair_kind = -1;
  double dt = 0;
  int pbc = 0, image = 0;
  double L[3] = {0, 0, 0};
};

static int plan_of(md_pimd_t_x *pimd, const md_pimd_step_config_x *cfg, StepPlan &sp) {
  if (ensure_pimd_device(pimd)) return -1;
  sp.p = pimd_state(pimd, false);
  if (cfg->trap && cfg->trap != md_harmonic_trap_force_x) {
    fprintf(stderr, "xmd: trap callback has no device kernel\n");
    return -1;
  }
  sp.trap = cfg->trap != nullptr;
  sp.pair_kind = -1;
  if (cfg->pair) {
    sp.pair_kind = pair_kind_of(cfg->pair);
    if (sp.pair_kind < 0) {
      fprintf(stderr, "xmd: pair-force callback has no device kernel\n");
      return -1;
    }
  }
  sp.dt = cfg->dt;
  sp.pbc = cfg->pbc;
  sp.image = cfg->image;
  for (int d = 0; d < 3; ++d) sp.L[d] = box_L(pimd->sim, d);
  return 0;
}

static BatchItem item_of(const StepPlan &sp) {
  BatchItem it;
  it.p = sp.p;
  it.dt = sp.dt;
  it.pbc = sp.pbc;
  it.image = sp.image;
  it.trap = sp.trap;
  it.pair_kind = sp.pair_kind;
  for (int d = 0; d < 3; ++d) it.L[d] = sp.L[d];
  return it;
}

// A stream pair for one system's step: s0 carries the step, s1 the
// recursion branch (fork / join events between them).
struct Lane {
  hipStream_t s0 = nullptr, s1 = nullptr, s2 = nullptr;
  hipEvent_t fork = nullptr, join = nullptr, fork2 = nullptr, join2 = nullptr;
};

static Lane main_lane() {
  Runtime &R = rt();
  Lane L;
  L.s0 = R.s0;
  L.s1 = R.s1;
  L.s2 = R.s2;
  L.fork = R.fork;
  L.join = R.join;
  L.fork2 = R.fork2;
  L.join2 = R.join2;
  return L;
}

// What runs beside the exchange chain (set-up, recursions, exchange forces).
// The chain is latency: short kernels, then two dependent solves on few
// workgroups that each want an empty compute unit.  Beside a pair grid that
// fills the device the short kernels wait for workgroup slots and the solves
// for room, and a fork costs its parent 5 us; so, with w = N^2 P pair terms
// (us per step, the order before -> the order chosen, on thermal states with
// exchange cycles t and uniform ones u):
//   Line    no Ewald, the smallest: everything on s0.  Such a graph costs the
//           host 10 us a step, one with branches 32, which at N=5 P=6 (36 ->
//           32) and N=8 P=8 (34 .. 38 -> 35) is what the device takes, so that
//           a busy host sets the pace; N=24 P=16 38 -> 45
//   Pairs   no Ewald: the pair branch on s2 and the chain on s0, both from NHC
//           on: no pair kernel fills the device (trap N=8 P=8 45 -> 34, N=256
//           P=64 t 92 -> 88, u 84 -> 65)
//   Wide    Ewald, smaller grids: likewise, the real space apart on s1, in
//           front of the kernels that follow one another (N=16 P=32 t 67 -> 46,
//           u 46 with a graph of four steps; 20-step calls, Wide and Beside: N=333
//           P=27 t 109 and 115, u 83 and 102; N=512 P=32 t 134 and 141, u 114 and
//           121; N=600 t 159 and 158, u 129 and 133; N=700 t 178 and 170, u 139 and
//           138; with real and reciprocal space on one stream N=333 t 108, u 109,
//           N=600 t 156, u 152)
//   Beside  Ewald, the real space on s2 from NHC on, bead-local and reciprocal
//           forces on s0 after the set-up, the solves on s1 (N=1024 P=32 t 235, u
//           191, and 226 and 211 with Late)
//   Late    as Beside, the real space after the set-up and behind the solves:
//           they are placed first (N=1350 P=32 t 348 -> 296, u 267 -> 287; N=1500 t
//           388 -> 337, u 310 -> 323; N=2001 P=24 t 519 -> 411, u 372 -> 384);
//           not where no cycles can be (cycles_expected), whose solves stay
//           short: xi = 0 N=1350 283 -> 263, N=1500 320 -> 305, N=1750 P=27
//           357 -> 346, N=2001 380 -> 368; Theta = 8 N=1500 323 -> 309
//   After   no Ewald: pair branch on s0 after the set-up, solves on s1 (trap
//           N=600 P=64 t 164, u 146; 214 and 161 with Pairs)
enum class Order { Serial, Line, Pairs, Wide, Beside, Late, After };

// Whether a system in a box may hold permutation cycles to speak of: at xi = 0
// there are none, and an ideal gas of degeneracy n lambda^3 has about xi n
// lambda^3 / 5 of its particles in cycles of two (repulsion makes it less), where
// a row block needs a dozen of its 64 in cycles to leave the solves' short way.
static bool cycles_expected(const DevPimd *p) {
  const md_pimd_t_x *h = p->host;
  const double lambda2 = 2 * M_PI * MD_hBar_X * MD_hBar_X * h->beta / h->sim->particles[0].m;
  const double n = p->N / (box_L(h->sim, 0) * box_L(h->sim, 1) * box_L(h->sim, 2));
  return fabs(h->vi) * n * lambda2 * sqrt(lambda2) >= 0.1;
}

static Order force_order(const StepPlan &sp, bool ewald) {
  const double w = (double)sp.p->N * sp.p->N * sp.p->P;
  if (ewald && sp.p->sur_mode) return Order::Beside;
  if (ewald) return w < 1.2e7 ? Order::Wide : w < 5e7 || !cycles_expected(sp.p) ? Order::Beside : Order::Late;
  return w < 1.5e3 ? Order::Line : w < 8e6 ? Order::Pairs : Order::After;
}

// ev: optional per-stage events (2 per stage: start, stop), may be null.
// serial: run every stage on s0 (true per-stage device times for profiling).
// fused (may be null: F complete on return): set (Fpart non-null) when the
// pair and exchange parts are left for NHC half 2 to add into F (massive
// thermostats), instead of a combine kernel.
static int enqueue_forces(StepPlan &sp, hipEvent_t *ev, bool serial, const Lane &R, ForceSums *fused) {
  DevPimd *p = sp.p;
  DevSim *d = p->ds;
  const int kind = sp.pair_kind;
  EwaldPlan plan;
  const bool ewald = !serial && kind >= 0 && pair_ewald_tab(p, kind, plan);
  const Order o = serial ? Order::Serial : force_order(sp, ewald);
  // pair forces without a reciprocal part: with massive thermostats their tile
  // sums and the exchange forces are left for NHC half 2 as well, two launches
  // and a pass over F fewer
  const bool parts = !serial && fused && d->massive && kind >= 0 && (ewald || !pair_has_recip(kind));
  // (then nothing but NHC half 2 reads F, and in small systems the bead-local
  // forces ride with the springs of the cycle energies: N=8 P=8 34.8 -> 33.2 us
  // per step, N=64 P=32 59.9 -> 59.5, but N=200 P=40 90 -> 93, their workgroups
  // in the way of the chain's)
  const bool ride = parts && (double)p->N * p->N * p->P < 2e5;
  const BeadRep ride_rep = bead_rep(item_of(sp));
  const bool pairs_s2 = o == Order::Pairs || o == Order::Wide;  // bead-local and pair forces on s2
  const bool fork_solve = o == Order::Beside || o == Order::Late || o == Order::After;
  const hipStream_t sx = fork_solve ? R.s1 : R.s0, sb = pairs_s2 ? R.s2 : R.s0;
  auto rec = [&](int k, hipStream_t st) -> int {
    if (ev) XMD_CHECK(hipEventRecord(ev[k], st));
    return 0;
  };
  auto fork = [&](hipEvent_t e, hipStream_t st) -> int {
    XMD_CHECK(hipEventRecord(e, R.s0));
    XMD_CHECK(hipStreamWaitEvent(st, e, 0));
    return 0;
  };
  auto real = [&](hipStream_t st) -> int {
    return rec(8, st) || launch_pair_ewald_real(p, plan, st) || rec(9, st) ? -1 : 0;
  };
  auto bead = [&](hipStream_t st) -> int {
    if (rec(6, st)) return -1;
    if (d->massive) {
      if (launch_step_bead_forces(item_of(sp), st)) return -1;
    } else {
      if (launch_reset_force(d, st)) return -1;
      if (sp.trap && launch_trap_force(d, md_trap_frequency_x, md_trap_center_x, (double)p->P, st)) return -1;
      if (launch_ring_springs(p, sp.image, sp.L, st)) return -1;
    }
    return rec(7, st);
  };
  auto kspace = [&](hipStream_t st) -> int {
    return rec(10, st) || launch_pair_kspace(p, plan, st) || rec(11, st) ? -1 : 0;
  };
  const bool s2 = pairs_s2 || o == Order::Beside || o == Order::Late;
  if (s2 && o != Order::Late && fork(R.fork2, R.s2)) return -1;
  if (o == Order::Wide) XMD_CHECK(hipStreamWaitEvent(R.s1, R.fork2, 0));
  // Wide: in a graph the real space is queued last (N=16 P=32 52 -> 46 us per
  // step); launched one by one it would then wait for the host to queue the
  // others first (N=600 P=32 u, one step 199 -> 186)
  bool real_first = o == Order::Beside;
  if (o == Order::Wide) {
    hipStreamCaptureStatus capture;
    XMD_CHECK(hipStreamIsCapturing(R.s0, &capture));
    real_first = capture == hipStreamCaptureStatusNone;
  }
  if (real_first && real(o == Order::Wide ? R.s1 : R.s2)) return -1;
  if (rec(2, R.s0) || (serial ? launch_enk(p, sp.image, R.s0)
                             : launch_enk_prep(p, sp.image, R.s0, ride ? &ride_rep : nullptr)) ||
      rec(3, R.s0))
    return -1;
  if (fork_solve && fork(R.fork, R.s1)) return -1;
  if (rec(4, sx) || (serial ? launch_recursion(p, true, true, sx, ev ? ev[16] : nullptr) : launch_recursion_solve(p, sx)) ||
      rec(5, sx))
    return -1;
  if (!serial && (rec(12, sx) || launch_exchange_force(p, sp.image, sx, true) || rec(13, sx))) return -1;
  if (fork_solve) XMD_CHECK(hipEventRecord(R.join, R.s1));
  if (o == Order::Late && (fork(R.fork2, R.s2) || real(R.s2))) return -1;
  // bead-local and pair forces
  if (ride ? rec(6, R.s0) || rec(7, R.s0) : bead(sb)) return -1;
  if (ewald) {
    if (kspace(sb)) return -1;
    if (o == Order::Wide) {
      if (!real_first && real(R.s1)) return -1;
      XMD_CHECK(hipEventRecord(R.join, R.s1));
    }
  } else {
    if (rec(8, sb) || (kind >= 0 && launch_pair_real(p, kind, sb, !parts)) || rec(9, sb)) return -1;
    if (rec(10, sb) || (kind >= 0 && pair_has_recip(kind) && launch_pair_recip(p, kind, sb)) || rec(11, sb)) return -1;
  }
  if (serial) return rec(12, R.s0) || launch_exchange_force(p, sp.image, R.s0, false) || rec(13, R.s0) ? -1 : 0;
  if (s2) {
    XMD_CHECK(hipEventRecord(R.join2, R.s2));
    XMD_CHECK(hipStreamWaitEvent(R.s0, R.join2, 0));
  }
  if (fork_solve || o == Order::Wide) XMD_CHECK(hipStreamWaitEvent(R.s0, R.join, 0));
  if (parts) return force_sums(p, p->Fx, ewald, fused);
  // one kernel adds the real-space, reciprocal and exchange forces
  return ewald ? launch_combine_forces(p, p->Fx, R.s0) : launch_add_exchange_force(p, R.s0);
}

// head: NHC half 1 starts the step (false: the previous step's chained tail
// did it).  chain (massive thermostats): NHC half 2 and the next step's half
// 1 run as one kernel at the end of this step.
static int enqueue_step(StepPlan &sp, hipEvent_t *ev, bool serial, const Lane &R, bool head = true,
                        bool chain = false) {
  DevSim *d = sp.p->ds;
  if (ev) XMD_CHECK(hipEventRecord(ev[0], R.s0));
  if (!head) {
  } else if (d->massive) {
    if (launch_step_nhc(item_of(sp), 1, R.s0)) return -1;
  } else {
    if (launch_nhc(d, 1, sp.dt, R.s0)) return -1;
    if (sp.pbc && launch_pbc(d, sp.L, R.s0)) return -1;
  }
  if (ev) XMD_CHECK(hipEventRecord(ev[1], R.s0));
  ForceSums fused;
  if (enqueue_forces(sp, ev, serial, R, &fused)) return -1;
  if (ev) XMD_CHECK(hipEventRecord(ev[14], R.s0));
  if (d->massive ? launch_step_nhc(item_of(sp), chain ? 3 : 2, R.s0, fused.Fpart ? &fused : nullptr)
                 : launch_nhc(d, 2, sp.dt, R.s0))
    return -1;
  if (ev) XMD_CHECK(hipEventRecord(ev[15], R.s0));
  return 0;
}

// Number of nodes and edges of a graph, the edges as pairs of node numbers.
static int graph_shape(hipGraph_t g, std::vector<int> &shape) {
  size_t nn = 0, ne = 0;
  XMD_CHECK(hipGraphGetNodes(g, nullptr, &nn));
  XMD_CHECK(hipGraphGetEdges(g, nullptr, nullptr, &ne));
  std::vector<hipGraphNode_t> node(nn), from(ne), to(ne);
  if (nn) XMD_CHECK(hipGraphGetNodes(g, node.data(), &nn));
  if (ne) XMD_CHECK(hipGraphGetEdges(g, from.data(), to.data(), &ne));
  auto number = [&](hipGraphNode_t n) { return (int)(std::find(node.begin(), node.end(), n) - node.begin()); };
  shape = {(int)nn};
  for (size_t k = 0; k < ne; ++k) {
    shape.push_back(number(from[k]));
    shape.push_back(number(to[k]));
  }
  return 0;
}

// One step of a whole batch, the single-system step's stages with one launch
// per stage over all replicas.
struct Batch {
  BeadBatch *bead = nullptr;
  ExchBatch *exch = nullptr;
  PairBatch *pair = nullptr;
  ~Batch() {
    bead_batch_free(bead);
    exch_batch_free(exch);
    pair_batch_free(pair);
  }
};

// A batch's tables and executable step graph are kept after a call and reused
// by the next call on the same objects with the same configs, interaction
// globals and object state (temperature, exchange parameter, box), as long
// as no pair-kernel buffer was reallocated in between; anything else
// rebuilds them.
struct BatchCache {
  std::vector<md_pimd_t_x *> pimds;
  std::vector<md_pimd_step_config_x> cfgs;
  std::vector<double> key;
  unsigned epoch = 0;
  Batch *B = nullptr;
  hipGraphExec_t exec = nullptr;
};
static BatchCache g_bcache;

static std::vector<double> batch_key(md_pimd_t_x *const *pimds, int n) {
  std::vector<double> k = {md_trap_frequency_x, md_trap_center_x[0], md_trap_center_x[1], md_trap_center_x[2],
                           md_gaussian_strength_x, md_gaussian_range_x, md_coulomb_strength_x, md_coulomb_truc_x,
                           (double)md_coulomb_n_sum_x, (double)g_nhc_len, g_ewald_xcut, g_ewald_split_aL,
                           md_he_eps_x, md_he_A_x, md_he_alpha_x, md_he_C6_x, md_he_C8_x, md_he_C10_x, md_he_D_x,
                           md_he_rm_x};
  for (int i = 0; i < n; ++i) {
    k.push_back(pimds[i]->beta);
    k.push_back(pimds[i]->omegaP);
    k.push_back(pimds[i]->vi);
    k.push_back(pimds[i]->sim->T);
    for (int d = 0; d < 3; ++d) k.push_back(box_L(pimds[i]->sim, d));
  }
  return k;
}

static void batch_cache_drop() {
  if (g_bcache.exec) (void)hipGraphExecDestroy(g_bcache.exec);
  delete g_bcache.B;
  g_bcache = BatchCache();
}

static int enqueue_batch(Batch &B, const Lane &L) {
  // set-up, recursions and exchange forces on s0; beside the recursions the
  // tile sums (Gaussian, Ewald real space) on s1 and the bead-local and
  // reciprocal forces on s2, every part in a buffer of its own that NHC half 2
  // adds: the recursions are few workgroups, the tile kernels vector and the
  // reciprocal ones matrix work.  (Pair forces one after another on s0 and
  // added into F: 32 replicas of N = 8 .. 512, 20 steps and the copy to the
  // host 14.6 ms, 13.4 so; forked from NHC half 1 on, before the set-up, 14.3.)
  if (bead_batch_nhc(B.bead, 1, L.s0) || exch_batch_enk(B.exch, L.s0)) return -1;
  XMD_CHECK(hipEventRecord(L.fork, L.s0));
  XMD_CHECK(hipStreamWaitEvent(L.s1, L.fork, 0));
  XMD_CHECK(hipStreamWaitEvent(L.s2, L.fork, 0));
  if (exch_batch_recursion(B.exch, L.s0) || exch_batch_force(B.exch, L.s0)) return -1;
  if (bead_batch_forces(B.bead, L.s2) || pair_batch_solo(B.pair, L.s2) || pair_batch_kspace(B.pair, L.s2)) return -1;
  if (pair_batch_real(B.pair, L.s1)) return -1;
  XMD_CHECK(hipEventRecord(L.join, L.s1));
  XMD_CHECK(hipEventRecord(L.join2, L.s2));
  XMD_CHECK(hipStreamWaitEvent(L.s0, L.join, 0));
  XMD_CHECK(hipStreamWaitEvent(L.s0, L.join2, 0));
  return bead_batch_nhc(B.bead, 2, L.s0);
}

}  // namespace xmd

using namespace xmd;

extern "C" {

int md_set_nhc_length_x(int M) {
  if (M < 2 || M > MD_NHC_LENGTH_X || M % 2) return -1;
  g_nhc_len = M;
  return 0;
}

int md_get_nhc_length_x(void) { return g_nhc_len; }

int md_set_ewald_real_cutoff_x(md_num_t_x x_cut) {
  if (!(x_cut > 0)) return -1;
  g_ewald_xcut = x_cut;
  return 0;
}

int md_set_ewald_split_x(md_num_t_x alpha_L) {
  if (!(alpha_L == alpha_L)) return -1;
  g_ewald_split_aL = alpha_L;
  return 0;
}

int md_hip_synchronize_x(void) {
  if (ensure_runtime()) return -1;
  XMD_CHECK(hipStreamSynchronize(rt().s1));
  XMD_CHECK(hipStreamSynchronize(rt().s0));
  return recursion_status_all();
}

int md_pimd_inject_recursion_timeouts_x(md_pimd_t_x *pimd, int count) {
  if (count < 0 || ensure_pimd_device(pimd)) return -1;
  return inject_recursion_timeouts(pimd_state(pimd, false), count);
}

int md_set_recursion_frame_limit_x(double limit) {
  set_recursion_frame_limit(limit);
  return 0;
}

int md_pimd_get_backward_potentials_x(md_pimd_t_x *pimd, md_num_t_x *Vt) {
  DevPimd *p = pimd_state(pimd, false);
  if (!p || !p->back_dev) return -1;
  XMD_CHECK(hipStreamSynchronize(rt().s0));
  return backward_potentials(p, Vt);
}

int md_pimd_get_connection_matrix_x(md_pimd_t_x *pimd, md_num_t_x *G) {
  DevPimd *p = pimd_state(pimd, false);
  if (!p || !p->back_dev || !p->vbn_dev) return -1;
  return connection_matrix(p, G);
}

int md_pimd_compute_forces_x(md_pimd_t_x *pimd, const md_pimd_step_config_x *cfg) {
  StepPlan sp;
  if (plan_of(pimd, cfg, sp)) return -1;
  return enqueue_forces(sp, nullptr, false, main_lane(), nullptr);
}

int md_pimd_run_steps_x(md_pimd_t_x *pimd, const md_pimd_step_config_x *cfg, int nsteps) {
  StepPlan sp;
  if (plan_of(pimd, cfg, sp)) return -1;
  if (nsteps <= 0) return 0;
  const Lane L = main_lane();
  if (!cfg->use_graph || nsteps == 1) {
    for (int s = 0; s < nsteps; ++s)
      if (enqueue_step(sp, nullptr, false, L)) return -1;
    return 0;
  }
  // Every call captures the step afresh, so the graph holds this call's
  // parameters and buffers.  The step's lazily created buffers are made
  // first, on the host; when that allocated anything, or on the first call
  // on an object, the first step runs eagerly (so allocation and the
  // capture's kernel-only graph cannot interfere) and the capture runs on the
  // host while the device works on that step.  A call of at least
  // kLongCall graph steps captures kStepsPerGraph consecutive steps into one
  // graph, which saves most of the boundaries between graph launches
  // (0.2486 -> 0.2479 ms per step for UEG N=1024 P=32); shorter calls
  // capture one (the capture's host time would not be amortised); steps left
  // over run eagerly after the launches.  With massive thermostats the
  // captured steps chain NHC half 2 of one step and half 1 of the next into
  // one kernel (one launch and one pass over the thermostat state fewer per
  // step boundary inside the graph).  An
  // executable graph kept from the previous call on the same object is
  // updated in place when the new graph has its topology, which saves the
  // instantiation.  The edges are compared here: hipGraphExecUpdate has
  // accepted a graph of as many kernels and edges between others of them, and
  // then run its kernels under the old edges.
  constexpr int kStepsPerGraph = 4, kLongCall = 32;
  Runtime &R = rt();
  DevPimd *p = sp.p;
  if (autotune_if_needed(p, sp.pair_kind)) return -1;
  const int fresh = pair_prepare(p, sp.pair_kind);
  if (fresh < 0) return -1;
  const int eager = (fresh || !p->step_exec) ? 1 : 0;
  if (eager && enqueue_step(sp, nullptr, false, L)) return -1;
  const int per = nsteps - eager >= kLongCall ? kStepsPerGraph : 1, launches = (nsteps - eager) / per;
  hipGraph_t graph = nullptr;
  XMD_CHECK(hipStreamBeginCapture(R.s0, hipStreamCaptureModeGlobal));
  int rc = 0;
  const bool chain = p->ds->massive;
  for (int k = 0; k < per && !rc; ++k) rc = enqueue_step(sp, nullptr, false, L, k == 0 || !chain, chain && k + 1 < per);
  const hipError_t ec = hipStreamEndCapture(R.s0, &graph);
  if (rc || ec != hipSuccess || !graph) {
    fprintf(stderr, "xmd: step capture failed\n");
    return -1;
  }
  hipGraphExec_t exec = (hipGraphExec_t)p->step_exec;
  bool updated = false;
  std::vector<int> shape;
  if (graph_shape(graph, shape)) return -1;
  if (exec) {
    hipGraphNode_t bad = nullptr;
    hipGraphExecUpdateResult res;
    updated = shape == p->step_shape && hipGraphExecUpdate(exec, graph, &bad, &res) == hipSuccess &&
              res == hipGraphExecUpdateSuccess;
    if (!updated) {
      (void)hipGetLastError();
      XMD_CHECK(hipGraphExecDestroy(exec));
      exec = nullptr;
    }
  }
  if (!updated) XMD_CHECK(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
  p->step_exec = exec;
  p->step_shape = shape;
  XMD_CHECK(hipGraphDestroy(graph));
  for (int s = 0; s < launches; ++s) XMD_CHECK(hipGraphLaunch(exec, R.s0));
  for (int s = eager + launches * per; s < nsteps; ++s)
    if (enqueue_step(sp, nullptr, false, L)) return -1;
  XMD_CHECK(hipStreamSynchronize(R.s0));
  return recursion_status(sp.p);
}

int md_pimd_profile_steps_x(md_pimd_t_x *pimd, const md_pimd_step_config_x *cfg, int nsteps, int serial,
                            double *stage_ms) {
  StepPlan sp;
  if (plan_of(pimd, cfg, sp)) return -1;
  const int NE = 18;
  hipEvent_t ev[NE];
  for (int k = 0; k < NE; ++k) XMD_CHECK(hipEventCreate(&ev[k]));
  for (int k = 0; k < MD_PIMD_NSTAGES_X; ++k) stage_ms[k] = 0;
  // stage k <- events (a, b)
  const int pairs[8][2] = {{0, 1}, {2, 3}, {4, 5}, {6, 7}, {8, 9}, {10, 11}, {12, 13}, {14, 15}};
  for (int s = 0; s < nsteps; ++s) {
    if (serial) set_real_space_probe(ev[17]);
    const int bad = enqueue_step(sp, ev, serial != 0, main_lane());
    const bool probe = serial && real_space_probe_hit();
    set_real_space_probe(nullptr);
    if (bad) return -1;
    XMD_CHECK(hipStreamSynchronize(rt().s0));
    if (recursion_status(sp.p)) return -1;
    for (int k = 0; k < 8; ++k) {
      float ms = 0;
      XMD_CHECK(hipEventElapsedTime(&ms, ev[pairs[k][0]], ev[pairs[k][1]]));
      stage_ms[k] += ms;
    }
    float ms = 0;
    XMD_CHECK(hipEventElapsedTime(&ms, ev[0], ev[15]));
    stage_ms[8] += ms;
    if (serial) {
      XMD_CHECK(hipEventElapsedTime(&ms, ev[16], ev[5]));
      stage_ms[9] += ms;
      if (probe) XMD_CHECK(hipEventElapsedTime(&ms, ev[8], ev[17]));
      stage_ms[10] += probe ? ms : 0.0f;
    }
  }
  for (int k = 0; k < MD_PIMD_NSTAGES_X; ++k) stage_ms[k] /= nsteps;
  for (int k = 0; k < NE; ++k) XMD_CHECK(hipEventDestroy(ev[k]));
  return 0;
}

int md_pimd_run_batch_x(md_pimd_t_x *const *pimds, const md_pimd_step_config_x *cfgs, int n, int nsteps) {
  if (!pimds || !cfgs || n <= 0) return -1;
  if (nsteps <= 0) return 0;
  std::vector<BatchItem> items(n);
  for (int i = 0; i < n; ++i) {
    for (int j = 0; j < i; ++j)
      if (pimds[j] == pimds[i] || pimds[j]->sim == pimds[i]->sim) {
        fprintf(stderr, "xmd: a batch lists one system twice\n");
        return -1;
      }
    StepPlan sp;
    if (plan_of(pimds[i], &cfgs[i], sp)) return -1;
    if (autotune_if_needed(sp.p, sp.pair_kind)) return -1;
    items[i] = item_of(sp);
  }
  const Lane L = main_lane();
  Runtime &R = rt();
  const bool graph = cfgs[0].use_graph != 0;
  if (graph) {
    // the kept graph of the previous call, when nothing it depends on changed
    const std::vector<double> key = batch_key(pimds, n);
    bool same = g_bcache.exec && g_bcache.pimds.size() == (size_t)n && g_bcache.key == key &&
                g_bcache.epoch == pair_alloc_epoch();
    for (int i = 0; same && i < n; ++i)
      same = g_bcache.pimds[i] == pimds[i] && !memcmp(&g_bcache.cfgs[i], &cfgs[i], sizeof(md_pimd_step_config_x));
    if (same) {
      for (int s = 0; s < nsteps; ++s) XMD_CHECK(hipGraphLaunch(g_bcache.exec, R.s0));
      return exch_batch_status(g_bcache.B->exch);
    }
    batch_cache_drop();
  }
  Batch *B = new Batch();
  B->exch = exch_batch_create(items);
  B->pair = pair_batch_create(items);
  if (B->pair) B->bead = bead_batch_create(items, pair_batch_sums(B->pair));
  if (!B->bead || !B->exch || !B->pair) {
    delete B;
    return -1;
  }
  // The first step runs eagerly; the rest replay one captured graph of a
  // whole batch step (or run eagerly when the configs ask for no graph).
  if (enqueue_batch(*B, L)) {
    delete B;
    return -1;
  }
  XMD_CHECK(hipStreamSynchronize(R.s0));
  if (!graph) {
    int rc = 0;
    for (int s = 1; s < nsteps && !rc; ++s) rc = enqueue_batch(*B, L);
    if (exch_batch_status(B->exch)) rc = -1;
    delete B;
    return rc;
  }
  hipGraph_t g;
  hipGraphExec_t exec;
  XMD_CHECK(hipStreamBeginCapture(R.s0, hipStreamCaptureModeGlobal));
  int rc = enqueue_batch(*B, L);
  hipError_t ec = hipStreamEndCapture(R.s0, &g);
  if (rc || ec != hipSuccess) {
    fprintf(stderr, "xmd: batch capture failed\n");
    delete B;
    return -1;
  }
  XMD_CHECK(hipGraphInstantiate(&exec, g, nullptr, nullptr, 0));
  XMD_CHECK(hipGraphDestroy(g));
  g_bcache.pimds.assign(pimds, pimds + n);
  g_bcache.cfgs.assign(cfgs, cfgs + n);
  g_bcache.key = batch_key(pimds, n);
  g_bcache.epoch = pair_alloc_epoch();
  g_bcache.B = B;
  g_bcache.exec = exec;
  for (int s = 1; s < nsteps; ++s) XMD_CHECK(hipGraphLaunch(exec, R.s0));
  return exch_batch_status(B->exch);
}

}  // extern "C"
