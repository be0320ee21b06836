// C ABI of liblulesh_hip (declared in include/lulesh_hip.h): context
// lifetime, Domain field access, the hot-path entry points, the device-side
// driver loop (graph replay), ragged batches and per-kernel event timing.
//
// A context holds a batch of one or more structured Sedov domains laid out
// back to back in flat SoA device buffers.  The single-domain entry points
// address instance 0 (their only instance); the lulesh_batch_* ones take an
// instance index.  Cycle-level entry points always advance every instance.
#include "lulesh_hip.h"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <exception>
#include <new>
#include <string>
#include <algorithm>
#include <vector>

#include "lulesh_adjoint.h"
#include "lulesh_hostcopy.h"
#include "lulesh_kernels.h"
#include "lulesh_regions.h"

using namespace lulesh;

// device buffers of the adjoint driver (allocated on first use)
struct AdjBuffers {
  bool ready = false;
  AdjArgs a{};
  double *dt = nullptr;        // recorded dt schedule
  int64_t dt_cap = 0;
  double *ckpt = nullptr;      // checkpoints, each 6N + 5E doubles
  int64_t ckpt_cap = 0;        // states
  double *seg = nullptr;       // states of the segment being reversed
  int64_t seg_cap = 0;
  double *final_state = nullptr;
  DevScalars *final_sc = nullptr;
  std::vector<void *> mem;
};

struct lulesh_ctx {
  int n = 0;  // instances
  int quirks = LULESH_QUIRKS_REFERENCE, device = 0;
  std::vector<InstDesc> inst;
  std::vector<int32_t> nr, balance, cost;
  int64_t E_total = 0, N_total = 0;
  hipStream_t stream = nullptr;
  Batch b{};                      // device pointers + launch geometry
  DevScalars *hsc = nullptr;      // pinned host mirror [n]
  HostCopy host;                  // field downloads
  // hsc holds what the device does: set by finish() when nothing has been
  // launched since pull_scalars, dropped by touch().  Reading a scalar then
  // takes no copy (13 us), nor does the node-set parity of a download.
  bool pulled = false, known = false;
  bool partials_valid = false;    // dtpart holds what the last lagrangeElements left
  int partials = 0;               // ... in so many pairs (one domain)
  int cus = 256, nodal_per_cu = 2;  // compute units; k_nodal workgroups resident per CU
  int keep_aux = 0;
  // timing
  bool timing = false;
  struct Pending {
    int id;
    hipEvent_t a, b;
  };
  std::vector<Pending> pending;
  std::vector<hipEvent_t> event_pool;
  double ktime[LULESH_K_COUNT] = {0};
  int64_t kcount[LULESH_K_COUNT] = {0};
  // driver-loop graph: kGraphCycles cycles of every instance
  hipGraphExec_t graph = nullptr;
  int graph_keep_aux = -1;
  std::string last_error;
  std::vector<void *> allocations;
  int tile_lo = 16, tile_hi = 32;  // k_nodal tile widths allowed (nodal_tile)
  int depth_req = 0;               // k_nodal z-depth asked for (0: the model's)
  bool nodal_ready = false;        // k_nodal's tables match c->inst (false after a failed plan)
  int *ginst = nullptr;            // device table of gblock_host (regrown by plan_nodal)
  int64_t ginst_cap = 0;
  std::vector<int> gblock_host;  // instance of each k_nodal block
  std::vector<int> gplanes_host; // element planes each k_nodal block marches
  int *gorder = nullptr;         // k_nodal dispatch table (regrown by plan_nodal)
  int64_t gorder_cap = 0;
  std::vector<int> gorder_host;
  std::vector<char> order_live;  // instances the table holds (empty: all)
  // k_kin / k_qeos work tables (kin_table, qeos_table), sized for every
  // instance at create; a live subset rewrites them in place
  std::vector<int> kin_base;       // band rotation per instance
  std::vector<int> eblock_host;    // instance of each element block
  KinWork *kin_work = nullptr;
  int *qeos_order = nullptr;
  AdjBuffers adj;
  // region index sets per instance, built on first use (they never change
  // and no default path reads them), and the cost mode's per-element reps
  std::vector<RegionSets> regions;
  int *elem_rep = nullptr;
  int graph_cost_mode = -1;
};

namespace {

const char *kErrText[] = {"",
                          "Early Volume Error",
                          "Mid Volume Error",
                          "Volume Error: Volume is negative",
                          "Volume Error: calcKinematicsForElems",
                          "Volume Error :2157",
                          "Error",
                          "QStopError",
                          "Volume Error :2887",
                          "Volume Error :2908"};

int fail(lulesh_ctx *c, int code, const std::string &msg) {
  if (c) c->last_error = msg;
  return code;
}

int hip_fail(lulesh_ctx *c, hipError_t e, const char *what) {
  std::string m = std::string(what) + ": " + hipGetErrorString(e);
  return fail(c, LULESH_ERR_HIP, m);
}

#define HIP_TRY(c, expr)                                   \
  do {                                                     \
    hipError_t _e = (expr);                                \
    if (_e != hipSuccess) return hip_fail((c), _e, #expr); \
  } while (0)

Batch make_args(lulesh_ctx *c, int gated, int loop_mode, int64_t num_iters = 0) {
  Batch a = c->b;
  a.gated = gated;
  a.loop_mode = loop_mode;
  a.keep_aux = c->keep_aux;
  a.num_iters = num_iters;
  a.flip = 1;
  // (timing reports k_kin and k_qeos each by itself)
  if (c->n == 1) {
    const int ebn = c->inst[0].ebn;
    const ElemsPlan p = elems_plan(c->inst[0].s, ebn, c->cus);
    const bool apart = c->timing || c->b.cost_mode;
    a.elems_form = apart ? ELEMS_APART : p.form;
    a.parts = apart ? ebn : p.parts;
  }
  return a;
}

hipEvent_t get_event(lulesh_ctx *c) {
  if (!c->event_pool.empty()) {
    hipEvent_t e = c->event_pool.back();
    c->event_pool.pop_back();
    return e;
  }
  hipEvent_t e = nullptr;
  if (hipEventCreate(&e) != hipSuccess) return nullptr;
  return e;
}

// before anything that may change the scalars on the device
void touch(lulesh_ctx *c) { c->pulled = c->known = false; }

// one launch on the context stream, bracketed by events when timing is on
int launch(lulesh_ctx *c, int id, const Batch &a) {
  touch(c);
  if (id == KID_NODAL && !c->nodal_ready)
    return fail(c, LULESH_ERR_HIP, "k_nodal tables unavailable (a device allocation failed)");
  hipEvent_t ea = nullptr, eb = nullptr;
  const bool timed = c->timing && id < LULESH_K_COUNT;
  if (timed) {
    ea = get_event(c);
    eb = get_event(c);
    if (!ea || !eb) return fail(c, LULESH_ERR_HIP, "hipEventCreate failed");
    HIP_TRY(c, hipEventRecord(ea, c->stream));
  }
  hipError_t e = launch_kernel(id, c->stream, a);
  if (e != hipSuccess) return hip_fail(c, e, "kernel launch");
  if (timed) {
    HIP_TRY(c, hipEventRecord(eb, c->stream));
    c->pending.push_back({id, ea, eb});
  }
  return 0;
}

int pull_scalars(lulesh_ctx *c) {
  HIP_TRY(c, hipMemcpyAsync(c->hsc, c->b.sc, sizeof(DevScalars) * c->n, hipMemcpyDeviceToHost,
                            c->stream));
  c->pulled = true;
  return 0;
}

// synchronise, fold pending event pairs into the timing totals, then report
// the lowest physics error raised on the device (if any, over all instances)
int finish(lulesh_ctx *c, bool check_err) {
  if (check_err && !c->pulled) {
    int rc = pull_scalars(c);
    if (rc) return rc;
  }
  HIP_TRY(c, hipStreamSynchronize(c->stream));
  c->known = c->known || c->pulled;
  for (auto &p : c->pending) {
    float ms = 0.f;
    HIP_TRY(c, hipEventElapsedTime(&ms, p.a, p.b));
    c->ktime[p.id] += ms;
    c->kcount[p.id] += 1;
    c->event_pool.push_back(p.a);
    c->event_pool.push_back(p.b);
  }
  c->pending.clear();
  if (!check_err) return 0;
  int err = ERR_NONE;
  for (int i = 0; i < c->n; ++i) err = c->hsc[i].err < err ? c->hsc[i].err : err;
  if (err != ERR_NONE) {
    if (err >= 1 && err <= 9) return fail(c, err, kErrText[err]);
    return fail(c, LULESH_ERR_HIP, "unknown device error code");
  }
  return 0;
}

// the scalars in hsc, fetched only if they are not there
int know_scalars(lulesh_ctx *c) {
  if (c->known) return 0;
  int rc = pull_scalars(c);
  return rc ? rc : finish(c, false);
}

int clear_err(lulesh_ctx *c) {
  bool clean = c->known;
  for (int i = 0; i < c->n && clean; ++i) clean = c->hsc[i].err == ERR_NONE;
  return clean ? 0 : launch(c, KID_CLEAR_ERR, make_args(c, 0, 0));
}

struct FieldRef {
  double *ptr;
  int64_t n;
};

// field of one instance; node positions/velocities live in the NodeSet the
// instance's parity selects
FieldRef find_field(lulesh_ctx *c, int inst, const char *name, int parity) {
  if (!name || inst < 0 || inst >= c->n) return {nullptr, 0};
  const std::string s(name);
  const DevFields &f = c->b.f;
  const InstDesc &I = c->inst[inst];
  const NodeSet &S = f.ns[parity & 1];
#define EF(nm) \
  if (s == #nm) return {f.nm + I.e0, I.E};
#define NF(nm) \
  if (s == #nm) return {f.nm + I.n0, I.N};
#define SF(nm) \
  if (s == #nm) return {S.nm + I.n0, I.N};
  EF(e) EF(p) EF(q) EF(ql) EF(qq) EF(v) EF(volo) EF(delv) EF(vdov) EF(arealg) EF(ss)
  EF(elemMass) EF(vnew) EF(delv_xi) EF(delv_eta) EF(delv_zeta) EF(delx_xi) EF(delx_eta)
  EF(delx_zeta) EF(dxx) EF(dyy) EF(dzz)
  SF(x) SF(y) SF(z) SF(xd) SF(yd) SF(zd)
  NF(xdd) NF(ydd) NF(zdd) NF(fx) NF(fy) NF(fz) NF(nodalMass)
#undef EF
#undef NF
#undef SF
  return {nullptr, 0};
}

double *scalar_slot(DevScalars *h, const std::string &s) {
#define SF(nm) \
  if (s == #nm) return &h->nm;
  SF(time) SF(deltatime) SF(dtcourant) SF(dthydro) SF(stoptime) SF(dtmax) SF(dtfixed)
  SF(deltatimemultlb) SF(deltatimemultub) SF(u_cut) SF(hgcoef) SF(qstop) SF(monoq_max_slope)
  SF(monoq_limiter_mult) SF(e_cut) SF(p_cut) SF(ss4o3) SF(q_cut) SF(v_cut) SF(qlc_monoq)
  SF(qqc_monoq) SF(qqc) SF(eosvmax) SF(eosvmin) SF(pmin) SF(emin) SF(dvovmax) SF(refdens)
#undef SF
  return nullptr;
}

template <typename T>
int dev_alloc(lulesh_ctx *c, T **p, int64_t n) {
  void *q = nullptr;
  c->allocations.reserve(c->allocations.size() + 1);  // the push below cannot throw
  hipError_t e = hipMalloc(&q, (size_t)(n > 0 ? n : 1) * sizeof(T));
  if (e != hipSuccess) return hip_fail(c, e, "hipMalloc");
  c->allocations.push_back(q);
  *p = (T *)q;
  return 0;
}

void drop_graph(lulesh_ctx *c) {
  if (c->graph) (void)hipGraphExecDestroy(c->graph);
  c->graph = nullptr;
}

void release(lulesh_ctx *c) {
  drop_graph(c);
  for (auto &p : c->pending) {
    (void)hipEventDestroy(p.a);
    (void)hipEventDestroy(p.b);
  }
  for (auto e : c->event_pool) (void)hipEventDestroy(e);
  for (void *p : c->allocations) (void)hipFree(p);
  for (void *p : c->adj.mem) (void)hipFree(p);
  if (c->gorder) (void)hipFree(c->gorder);
  if (c->ginst) (void)hipFree(c->ginst);
  if (c->hsc) (void)hipHostFree(c->hsc);
  if (c->stream) (void)hipStreamDestroy(c->stream);
}

// Whether the driver loop's cycles take their predecessor's end at their
// head (lulesh_kernels.hip, dt_fold_load) instead of in a k_dt launch: one
// domain of at most 4096 partial minima (s <= 101), sixteen reads for each of
// a workgroup's threads.  What it saves falls from 2.7 us a cycle at s=48 to
// 0.6-1 us at s=96, as every workgroup of the launch reads them all.
constexpr int kDeferBlocks = 4096;
bool defer_dt(const lulesh_ctx *c) {
  return c->n == 1 && c->inst[0].ebn <= kDeferBlocks && !c->b.nodal_wide;
}

// Cycles in the driver loop's graph.  A graph launch leaves the GPU idle for
// about 5 us before its first kernel; with eight cycles behind one a cycle at
// s=16 takes 17.2 us instead of 21.7, s=30 25.0 instead of 29.0, s=64 62.7
// instead of 67.5 (16 or 32 cycles: 0.1 us less again, and their capture is
// paid for by every context).
constexpr int kGraphCycles = 8;
// Launched kernel by kernel a cycle takes hardly longer where the host keeps
// ahead of the device (s=16 17.5 us), so only a call of this many cycles
// captures a graph, which takes about 100 us: a context's first 10 cycles at
// s=16 570 -> 190 us, and 20 cycles 438 -> 362.
constexpr int kGraphFrom = 64;

int build_graph(lulesh_ctx *c) {
  if (!c->nodal_ready)
    return fail(c, LULESH_ERR_HIP, "k_nodal tables unavailable (a device allocation failed)");
  if (c->graph_keep_aux != c->keep_aux || c->graph_cost_mode != c->b.cost_mode) {
    drop_graph(c);
    c->graph_keep_aux = c->keep_aux;
    c->graph_cost_mode = c->b.cost_mode;
  }
  if (c->graph) return 0;
  Batch a = make_args(c, 1, 1);
  a.defer_dt = defer_dt(c);
  hipGraph_t g = nullptr;
  HIP_TRY(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
  const int ids[] = {KID_NODAL, KID_KIN, KID_QEOS, KID_DT};
  for (int k = 0; k < kGraphCycles; ++k)
    for (int id : ids) {
      if (id == KID_DT && a.defer_dt) break;
      hipError_t e = launch_kernel(id, c->stream, a);
      if (e != hipSuccess) {
        (void)hipStreamEndCapture(c->stream, &g);
        if (g) (void)hipGraphDestroy(g);
        return hip_fail(c, e, "graph capture");
      }
    }
  HIP_TRY(c, hipStreamEndCapture(c->stream, &g));
  hipError_t e = hipGraphInstantiate(&c->graph, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (e != hipSuccess) {
    c->graph = nullptr;
    return hip_fail(c, e, "hipGraphInstantiate");
  }
  return 0;
}

// createRegionIndexSets! for every instance (lulesh_regions.h), once
int ensure_regions(lulesh_ctx *c) {
  if (!c->regions.empty()) return 0;
  std::vector<RegionSets> R((size_t)c->n);
  for (int i = 0; i < c->n; ++i)
    if (!build_regions(c->inst[i].E, c->nr[i], c->balance[i], c->cost[i], R[(size_t)i]))
      return fail(c, LULESH_ERR_INVALID_ARG, "region index sets: invalid nr/balance/cost");
  c->regions = std::move(R);
  return 0;
}

// z-chunk cut of the context's instances: balanced for a single domain;
// a batch keeps the plain cut (the balanced one measured slower there).
bool balanced_cut(const lulesh_ctx *c) { return c->n == 1; }

// Default z-march depth for the context's instances (auto_depth_one for a
// single domain; auto_depth, with a round of CUs x resident k_nodal
// workgroups per CU, for a batch).
int auto_depth(const lulesh_ctx *c) {
  std::vector<NodalPlanInst> pi;
  pi.reserve(c->inst.size());
  for (const InstDesc &I : c->inst) pi.push_back({I.s, NodalTile{I.etx, I.ety, I.tx, I.ty}});
  if (c->n == 1) return auto_depth_one(pi[0], c->cus, c->nodal_per_cu);
  return lulesh::auto_depth(pi.data(), pi.size(), (int64_t)c->cus * c->nodal_per_cu, false);
}

// k_nodal dispatch table (nodal_order) uploaded for the instances in
// `live` (null: all), so finished instances leave no hole in one XCD's
// share.  The first call for a plan (glaunch 0) sizes the launch.
// Synchronous.
int order_nodal(lulesh_ctx *c, const std::vector<char> *live) {
  c->gorder_host = nodal_order(c->gblock_host, c->gplanes_host, live, c->b.glaunch,
                               (int64_t)c->cus * c->nodal_per_cu);
  const std::vector<int> &order = c->gorder_host;
  c->nodal_ready = false;
  HIP_TRY(c, hipStreamSynchronize(c->stream));
  if ((int64_t)order.size() > c->gorder_cap) {
    // only a new plan grows the table (a live subset keeps glaunch), and a
    // new plan has already dropped the graph that holds the old pointer
    if (c->graph) return fail(c, LULESH_ERR_HIP, "k_nodal order table would move under the graph");
    c->b.gblock_order = nullptr;
    if (c->gorder) HIP_TRY(c, hipFree(c->gorder));
    c->gorder = nullptr;
    c->gorder_cap = 0;
    HIP_TRY(c, hipMalloc((void **)&c->gorder, order.size() * sizeof(int)));
    c->gorder_cap = (int64_t)order.size();
  }
  c->b.gblock_order = c->gorder;
  HIP_TRY(c, hipMemcpyAsync(c->gorder, order.data(), order.size() * sizeof(int),
                            hipMemcpyHostToDevice, c->stream));
  HIP_TRY(c, hipStreamSynchronize(c->stream));
  c->order_live = live ? *live : std::vector<char>();
  c->nodal_ready = true;
  return 0;
}

// the k_kin and k_qeos work tables for the instances in `live` (null: all),
// uploaded into the tables create sized for all of them
int order_elem(lulesh_ctx *c, const std::vector<char> *live) {
  std::vector<int> s(c->inst.size());
  for (size_t i = 0; i < s.size(); ++i) s[i] = c->inst[i].s;
  int launch = c->b.kin_launch;
  const std::vector<KinWork> kin = kin_table(s, live, c->kin_base, launch);
  if (launch != c->b.kin_launch) return fail(c, LULESH_ERR_HIP, "k_kin work table size changed");
  const std::vector<int> qeos = qeos_table(c->eblock_host, live);
  HIP_TRY(c, hipStreamSynchronize(c->stream));
  HIP_TRY(c, hipMemcpyAsync(c->kin_work, kin.data(), kin.size() * sizeof(KinWork),
                            hipMemcpyHostToDevice, c->stream));
  HIP_TRY(c, hipMemcpyAsync(c->qeos_order, qeos.data(), qeos.size() * sizeof(int),
                            hipMemcpyHostToDevice, c->stream));
  HIP_TRY(c, hipStreamSynchronize(c->stream));
  return 0;
}

int plan_nodal(lulesh_ctx *c, int cz) {
  // until the new tables are on the device, k_nodal must not run, and the
  // captured graph (which holds the old ones) is gone
  c->nodal_ready = false;
  drop_graph(c);
  c->b.nodal_wide = 0;
  for (InstDesc &I : c->inst) {
    const NodalTile t = nodal_tile(I.s, c->tile_lo, c->tile_hi);
    I.etx = t.etx;
    I.ety = t.ety;
    I.tx = t.tx;
    I.ty = t.ty;
    if (nodal_patch_wide(t)) c->b.nodal_wide = 1;
  }
  // default: auto_depth, balanced per instance; an explicit depth applies
  // unchanged to all instances
  const bool automatic = cz <= 0;
  if (automatic) cz = auto_depth(c);
  std::vector<int> gblock_inst, gplanes;
  int gb = 0;
  for (int i = 0; i < c->n; ++i) {
    InstDesc &I = c->inst[i];
    const NodalCut k = automatic ? depth_cut(I.s, cz, balanced_cut(c))
                                 : nodal_cut(I.s, cz, balanced_cut(c));
    I.cz = k.cz;
    I.cz0 = k.first;
    I.nch = k.chunks;
    I.gb0 = gb;
    I.gbn = nodal_blocks(NodalTile{I.etx, I.ety, I.tx, I.ty}, k);
    gb += I.gbn;
    gblock_inst.insert(gblock_inst.end(), I.gbn, i);
    for (int ch = 0; ch < k.chunks; ++ch)
      gplanes.insert(gplanes.end(), I.tx * I.ty, nodal_chunk_planes(k, ch, I.s));
  }
  // one small domain at the default geometry: a workgroup per node plane
  c->b.one = c->inst[0];
  c->b.ptile = plane_tile(c->inst[0].s);
  c->b.nodal_planes = c->n == 1 && automatic && c->tile_lo == 16 && c->tile_hi == 32 &&
                      nodal_planes_fit(c->inst[0].s, (int64_t)c->cus * c->nodal_per_cu);
  c->b.gblocks = gb;
  c->gblock_host = std::move(gblock_inst);
  c->gplanes_host = std::move(gplanes);
  c->b.glaunch = 0;
  HIP_TRY(c, hipStreamSynchronize(c->stream));
  if (gb > c->ginst_cap) {
    c->b.gblock_inst = nullptr;
    if (c->ginst) HIP_TRY(c, hipFree(c->ginst));
    c->ginst = nullptr;
    c->ginst_cap = 0;
    HIP_TRY(c, hipMalloc((void **)&c->ginst, sizeof(int) * gb));
    c->ginst_cap = gb;
  }
  c->b.gblock_inst = c->ginst;
  HIP_TRY(c, hipMemcpyAsync((void *)c->b.inst, c->inst.data(), sizeof(InstDesc) * c->n,
                            hipMemcpyHostToDevice, c->stream));
  HIP_TRY(c, hipMemcpyAsync(c->ginst, c->gblock_host.data(), sizeof(int) * gb,
                            hipMemcpyHostToDevice, c->stream));
  return order_nodal(c, nullptr);
}

int check_inst(lulesh_ctx *c, int32_t inst) {
  if (!c) return LULESH_ERR_INVALID_ARG;
  if (inst < 0 || inst >= c->n) return fail(c, LULESH_ERR_INVALID_ARG, "instance out of range");
  return 0;
}

int create(int32_t n, const int32_t *nx, const double *einit_scale, const double *hgcoef,
           const int32_t *nr, const int32_t *balance, const int32_t *cost, int32_t quirks,
           int32_t device, lulesh_ctx **out) {
  if (!out) return LULESH_ERR_INVALID_ARG;
  *out = nullptr;
  if (n < 1 || n > LULESH_MAX_INSTANCES || !nx || quirks < 0 || quirks > LULESH_QUIRKS_REFERENCE)
    return LULESH_ERR_INVALID_ARG;
  for (int i = 0; i < n; ++i) {
    // kernels address an instance's node and element arrays with 32-bit byte
    // offsets: (nx+1)^3 * 8 < 2^32 holds up to nx = 811 (s = 800 already
    // needs ~240 GB of HBM)
    if (nx[i] < 1 || nx[i] > 800) return LULESH_ERR_INVALID_ARG;
    if (einit_scale && !(einit_scale[i] > 0.0)) return LULESH_ERR_INVALID_ARG;
    // regions: nr in 1..LULESH_MAX_REGIONS, balance and cost >= 0, and the
    // cost denominator sum_r r^balance within Int64 (src/domain.jl:370-375)
    if (nr && (nr[i] < 1 || nr[i] > LULESH_MAX_REGIONS)) return LULESH_ERR_INVALID_ARG;
    if ((balance && balance[i] < 0) || (cost && cost[i] < 0)) return LULESH_ERR_INVALID_ARG;
    {
      const int64_t r = nr ? nr[i] : 1, b = balance ? balance[i] : 1;
      int64_t w = 0, tot = 0;
      for (int64_t k = 1; k <= r; ++k) {
        if (!ipow_checked(k, b, &w) || tot > INT64_MAX - w) return LULESH_ERR_INVALID_ARG;
        tot += w;
      }
    }
  }
  // all instances' nodes together below 2^31: block counts and the host's
  // block tables stay int-sized (far beyond what one GPU's memory holds)
  int64_t nodes = 0;
  for (int i = 0; i < n; ++i) nodes += (int64_t)(nx[i] + 1) * (nx[i] + 1) * (nx[i] + 1);
  if (nodes > INT32_MAX) return LULESH_ERR_INVALID_ARG;
  lulesh_ctx *c = new lulesh_ctx();
  // on every exit but success (an error code or an exception) the partly
  // built context is freed
  struct Owner {
    lulesh_ctx *c;
    ~Owner() {
      if (c) {
        release(c);
        delete c;
      }
    }
  } owner{c};
  c->n = n;
  c->quirks = quirks;
  c->device = device;
  {
    int cus = 0;
    if (hipSetDevice(device) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
        cus < 1)
      cus = 256;
    c->cus = cus;
    c->nodal_per_cu = nodal_blocks_per_cu();
  }
  c->inst.resize(n);
  int eb = 0, nb = 0;
  int64_t e0 = 0, n0 = 0;
  std::vector<int> eblock_inst, nblock_inst;
  for (int i = 0; i < n; ++i) {
    InstDesc &I = c->inst[i];
    const int s = nx[i];
    I.s = s;
    const NodalTile tile = nodal_tile(s);
    I.etx = tile.etx;
    I.ety = tile.ety;
    I.tx = tile.tx;
    I.ty = tile.ty;
    I.E = (int64_t)s * s * s;
    I.N = (int64_t)(s + 1) * (s + 1) * (s + 1);
    I.e0 = e0;
    I.n0 = n0;
    I.eb0 = eb;
    I.ebn = (int)((I.E + BLOCK - 1) / BLOCK);
    I.nb0 = nb;
    I.nbn = (int)((I.N + BLOCK - 1) / BLOCK);
    I.gb0 = 0;
    I.gbn = 0;
    I.cz = 0;
    I.einit_scale = einit_scale ? einit_scale[i] : 1.0;
    I.hgcoef = hgcoef ? hgcoef[i] : 3.0;
    e0 += I.E;
    n0 += I.N;
    eb += I.ebn;
    nb += I.nbn;
    eblock_inst.insert(eblock_inst.end(), I.ebn, i);
    nblock_inst.insert(nblock_inst.end(), I.nbn, i);
    c->nr.push_back(nr ? nr[i] : 1);
    c->balance.push_back(balance ? balance[i] : 1);
    c->cost.push_back(cost ? cost[i] : 1);
  }
  c->E_total = e0;
  c->N_total = n0;
  Batch &B = c->b;
  B.n = n;
  B.eblocks = eb;
  B.nblocks = nb;
  B.gblocks = 0;
  B.nodal_lead = c->cus / 8 > 1 ? c->cus / 8 : 1;
  B.quirks = quirks;
  int rc = 0;
  hipError_t he = hipSetDevice(device);
  if (he != hipSuccess) rc = hip_fail(c, he, "hipSetDevice");
  if (!rc) {
    he = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (he != hipSuccess) rc = hip_fail(c, he, "hipStreamCreate");
  }
  if (!rc) {
    // the scalars' mirror and the staging memory behind it
    size_t most = 0;
    for (const InstDesc &I : c->inst)
      for (const int64_t k : {I.N, I.E})
        if (HostCopy::small((size_t)k * sizeof(double))) most = std::max(most, (size_t)k * sizeof(double));
    const size_t mirror = (sizeof(DevScalars) * n + 255) / 256 * 256, stage = HostCopy::staging(most);
    he = hipHostMalloc((void **)&c->hsc, mirror + stage, hipHostMallocDefault);
    if (he != hipSuccess) rc = hip_fail(c, he, "hipHostMalloc");
    else c->host.use((char *)c->hsc + mirror, stage);
  }
  DevFields &f = B.f;
  double **ef[] = {&f.e, &f.p, &f.q, &f.ql, &f.qq, &f.v, &f.volo, &f.delv, &f.vdov, &f.arealg,
                   &f.ss, &f.elemMass, &f.vnew, &f.delv_xi, &f.delv_eta, &f.delv_zeta,
                   &f.delx_xi, &f.delx_eta, &f.delx_zeta, &f.dxx, &f.dyy, &f.dzz};
  double **nf[] = {&f.ns[0].x, &f.ns[0].y, &f.ns[0].z, &f.ns[0].xd, &f.ns[0].yd, &f.ns[0].zd,
                   &f.ns[1].x, &f.ns[1].y, &f.ns[1].z, &f.ns[1].xd, &f.ns[1].yd, &f.ns[1].zd,
                   &f.xdd, &f.ydd, &f.zdd, &f.fx, &f.fy, &f.fz, &f.nodalMass};
  for (double **p : ef)
    if (!rc) rc = dev_alloc(c, p, e0);
  for (double **p : nf)
    if (!rc) rc = dev_alloc(c, p, n0);
  if (!rc) rc = dev_alloc(c, &f.elemBC, e0);
  B.out = ElemState{f.e, f.p, f.q, f.v, f.ss};
  int64_t parts = eb;
  if (n == 1) parts = std::max<int64_t>(parts, elems_plan(c->inst[0].s, eb, c->cus).parts);
  if (!rc) rc = dev_alloc(c, &B.dtpart, 2 * parts);
  if (!rc) rc = dev_alloc(c, &B.sc, n);
  InstDesc *dinst = nullptr;
  int *deb = nullptr, *dnb = nullptr;
  if (!rc) rc = dev_alloc(c, &dinst, n);
  if (!rc) rc = dev_alloc(c, &deb, eb);
  if (!rc) rc = dev_alloc(c, &dnb, nb);
  if (!rc) {
    he = hipMemcpy(deb, eblock_inst.data(), sizeof(int) * eb, hipMemcpyHostToDevice);
    if (he == hipSuccess) he = hipMemcpy(dnb, nblock_inst.data(), sizeof(int) * nb, hipMemcpyHostToDevice);
    if (he != hipSuccess) rc = hip_fail(c, he, "hipMemcpy (batch tables)");
  }
  B.inst = dinst;
  B.eblock_inst = deb;
  B.nblock_inst = dnb;
  // k_kin / k_qeos work tables, sized for all instances
  c->eblock_host = std::move(eblock_inst);
  if (!rc) {
    std::vector<int> sz((size_t)n);
    for (int i = 0; i < n; ++i) sz[(size_t)i] = c->inst[(size_t)i].s;
    int launch = 0;
    (void)kin_table(sz, nullptr, c->kin_base, launch);
    B.kin_launch = launch;
    B.qeos_launch = qeos_launch(eb);
    rc = dev_alloc(c, &c->kin_work, launch);
    if (!rc) rc = dev_alloc(c, &c->qeos_order, B.qeos_launch);
    B.kin_work = c->kin_work;
    B.qeos_order = c->qeos_order;
    if (!rc) rc = order_elem(c, nullptr);
  }
  if (!rc) rc = plan_nodal(c, 0);
  if (!rc) rc = lulesh_reset(c);
  if (rc) return rc;
  owner.c = nullptr;
  *out = c;
  return 0;
}

// Fetch the instance's scalars (synchronous).
int get_inst_scalars(lulesh_ctx *c, int32_t inst, DevScalars *out) {
  HIP_TRY(c, hipSetDevice(c->device));
  if (!c->known) {
    HIP_TRY(c, hipMemcpyAsync(c->hsc + inst, c->b.sc + inst, sizeof(DevScalars),
                              hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    c->known = c->n == 1;
  }
  *out = c->hsc[inst];
  return 0;
}

// one cycle, launched kernel by kernel
int cycle_body(lulesh_ctx *c, bool constraints, const Batch &a) {
  const int ids[] = {KID_NODAL, KID_KIN, KID_QEOS, KID_DT};
  for (int id : ids) {
    if (id == KID_DT && !constraints) break;
    int rc = launch(c, id, a);
    if (rc) return rc;
  }
  return 0;
}

int run_cycles_body(lulesh_ctx *c, int64_t num_iters, int64_t *cycles_run) {
  HIP_TRY(c, hipSetDevice(c->device));
  int rc = know_scalars(c);
  if (rc) return rc;
  std::vector<long long> cycle0(c->n);
  long long min_cycle0 = 0;
  for (int i = 0; i < c->n; ++i) {
    cycle0[i] = c->hsc[i].cycle;
    min_cycle0 = (i == 0 || cycle0[i] < min_cycle0) ? cycle0[i] : min_cycle0;
  }
  // with timing on, kernels are launched one by one so each can carry its
  // events; otherwise captured cycles (all instances) are replayed while a
  // graph's worth of them is left
  const bool use_graph = !c->timing;
  Batch a = make_args(c, 1, 1, num_iters);
  a.defer_dt = use_graph && defer_dt(c);
  rc = launch(c, KID_RUN_BEGIN, a);
  if (rc) return rc;
  // replay exactly the cycles num_iters still allows the least advanced
  // active instance (its first cycle always runs); only stop-time exits,
  // errors and unequal instances leave gated no-op replays behind, one where
  // every instance has reached its stop time already.
  // The first batch is of 8 cycles: a no-op cycle still starts all its
  // workgroups, 6 us at s=48, 8 at s=96, 35 at s=192.  Where the element
  // kernels are one launch (s <= 40) it is 4 and a cycle 17 to 34, so that the
  // 10 us of each wait for the device between batches count for more: 32 (s=16,
  // 10 cycles 246 -> 207 us), unless the stop time is nearer than that many
  // of the last time step.
  bool go = false;
  for (int i = 0; i < c->n; ++i) go = go || c->hsc[i].time < c->hsc[i].stoptime;
  const DevScalars &S0 = c->hsc[0];
  const bool small = a.elems_form != ELEMS_APART && S0.stoptime - S0.time >= 32 * S0.deltatime;
  int64_t cap = small ? 32 : 8;
  long long next_cycle = min_cycle0 + 1;
  for (;;) {
    const long long left = (long long)num_iters - next_cycle + 1;
    const int64_t batch = !go || left < 1 ? 1 : (left < cap ? left : cap);
    for (int64_t i = 0; i < batch;) {
      if (use_graph && batch - i >= kGraphCycles && (c->graph || left >= kGraphFrom)) {
        rc = build_graph(c);
        if (rc) return rc;
        touch(c);
        HIP_TRY(c, hipGraphLaunch(c->graph, c->stream));
        i += kGraphCycles;
      } else {
        rc = cycle_body(c, !a.defer_dt, a);
        if (rc) return rc;
        ++i;
      }
    }
    if (a.defer_dt) {  // the last cycle's end
      rc = launch(c, KID_DT, a);
      if (rc) return rc;
    }
    rc = pull_scalars(c);
    if (!rc) rc = finish(c, false);
    if (rc) return rc;
    bool any = false;
    long long mn = 0;
    for (int i = 0; i < c->n; ++i)
      if (c->hsc[i].active) {
        if (!any || c->hsc[i].cycle < mn) mn = c->hsc[i].cycle;
        any = true;
      }
    if (!any) break;
    next_cycle = mn;
    if (cap < 256) cap *= 2;
    // instances that finished drop out of k_nodal's dispatch table
    std::vector<char> live(c->n);
    bool all = true;
    for (int i = 0; i < c->n; ++i) {
      live[i] = c->hsc[i].active != 0;
      all = all && live[i];
    }
    // (and out of k_kin's and k_qeos' work tables)
    if (all ? !c->order_live.empty() : live != c->order_live) {
      rc = order_nodal(c, all ? nullptr : &live);
      if (!rc) rc = order_elem(c, all ? nullptr : &live);
      if (rc) return rc;
    }
  }
  c->partials_valid = false;
  int err = ERR_NONE;
  for (int i = 0; i < c->n; ++i) {
    if (cycles_run) cycles_run[i] = (int64_t)(c->hsc[i].cycle - cycle0[i]);
    err = c->hsc[i].err < err ? c->hsc[i].err : err;
  }
  if (err != ERR_NONE) {
    if (err >= 1 && err <= 9) return fail(c, err, kErrText[err]);
    return fail(c, LULESH_ERR_HIP, "unknown device error code");
  }
  return 0;
}

// The driver loop; k_nodal's dispatch table is back to every instance on
// return, as the other entry points launch it for all of them.
int run_cycles(lulesh_ctx *c, int64_t num_iters, int64_t *cycles_run /* [n] or null */) {
  int rc = run_cycles_body(c, num_iters, cycles_run);
  if (!c->order_live.empty()) {
    int r2 = order_nodal(c, nullptr);
    if (!r2) r2 = order_elem(c, nullptr);
    if (!rc) rc = r2;
  }
  return rc;
}

// ---------------------------------------------------------------------------
// adjoint driver
// ---------------------------------------------------------------------------
int adj_alloc(lulesh_ctx *c, double **p, int64_t n) {
  void *q = nullptr;
  hipError_t e = hipMalloc(&q, (size_t)(n > 0 ? n : 1) * sizeof(double));
  if (e != hipSuccess) return hip_fail(c, e, "hipMalloc (adjoint)");
  c->adj.mem.push_back(q);
  *p = (double *)q;
  return 0;
}

// replaces a growable adjoint buffer (the old one is freed)
int adj_regrow(lulesh_ctx *c, double **p, int64_t n) {
  if (*p) {
    auto &m = c->adj.mem;
    for (size_t i = 0; i < m.size(); ++i)
      if (m[i] == *p) {
        (void)hipFree(m[i]);
        m.erase(m.begin() + (long)i);
        break;
      }
    *p = nullptr;
  }
  return adj_alloc(c, p, n);
}

// one cycle of a segment: its start state S_k (6N + 5E, the checkpoint
// layout) and its temporaries (9E); a segment of L cycles uses L + 1 slots,
// the last holding only the state after it
int64_t cycle_slot(const lulesh_ctx *c) {
  const int64_t E = c->inst[0].E, N = c->inst[0].N;
  return 6 * N + 14 * E;
}

// The adjoint fields, and room for `ncycles` recorded time steps, `nstates`
// saved states (6N + 5E doubles each) and, if `seg` > 0, a segment of so many
// cycle slots plus one.
int adj_setup(lulesh_ctx *c, int64_t ncycles, int64_t nstates, int64_t seg) {
  AdjBuffers &B = c->adj;
  const int64_t E = c->inst[0].E, N = c->inst[0].N;
  const int64_t state = 6 * N + 5 * E;
  int rc = 0;
  if (ncycles > B.dt_cap) {
    B.dt_cap = 0;  // no buffer until the regrow succeeds
    rc = adj_regrow(c, &B.dt, ncycles);
    if (rc) return rc;
    B.dt_cap = ncycles;
  }
  if (!B.ready) {
    // a_force addresses node and element values by 32-bit byte offsets
    if (8 * N > (int64_t)UINT32_MAX || 8 * E > (int64_t)UINT32_MAX)
      return fail(c, LULESH_ERR_UNSUPPORTED, "the adjoint supports at most 2^29 - 1 nodes");
    AdjArgs &a = B.a;
    a.sc = c->b.sc;
    a.f = c->b.f;
    a.s = c->inst[0].s;
    a.E = E;
    a.N = N;
    a.q1 = (c->quirks & LULESH_Q1_FACE5_NORMAL) != 0;
    a.q2 = (c->quirks & LULESH_Q2_DVDX_SWAP) != 0;
    a.q3 = (c->quirks & LULESH_Q3_XIP_SELF) != 0;
    double **nv[] = {&a.lx, &a.ly, &a.lz, &a.lxd, &a.lyd, &a.lzd};
    double **ev[] = {&a.le, &a.lp, &a.lq, &a.lv, &a.lss, &a.lvnew, &a.lvnew_delv};
    for (double **p : nv)
      if (!rc) rc = adj_alloc(c, p, N);
    for (double **p : ev)
      if (!rc) rc = adj_alloc(c, p, E);
    if (!rc) rc = adj_alloc(c, &a.lF, 3 * N);
    if (!rc) rc = adj_alloc(c, &a.nbr, 6 * E);
    if (!rc) rc = adj_alloc(c, &a.ldvs, 3 * E);
    if (!rc) rc = adj_alloc(c, &a.ldx, 3 * E);
    if (!rc) rc = adj_alloc(c, &a.corner, 48 * E);
    if (!rc) rc = adj_alloc(c, &a.corner_f, 48 * E);
    if (!rc) rc = adj_alloc(c, &a.pacc, 3 * E);
    if (!rc) rc = adj_alloc(c, &B.final_state, state);
    if (!rc) {
      hipError_t he = hipMalloc((void **)&B.final_sc, sizeof(DevScalars));
      if (he != hipSuccess) return hip_fail(c, he, "hipMalloc (adjoint)");
      B.mem.push_back(B.final_sc);
    }
    if (rc) return rc;
    // the shadow of lulesh_vjp_cycle starts at zero, on the stream that its
    // uploads and kernels follow on (a hipMemset goes to the null stream,
    // which this one does not wait for, and may return before it is done)
    double *zero[] = {a.lx, a.ly, a.lz, a.lxd, a.lyd, a.lzd};
    for (double *p : zero) HIP_TRY(c, hipMemsetAsync(p, 0, sizeof(double) * N, c->stream));
    double *zeroe[] = {a.le, a.lp, a.lq, a.lv, a.lss};
    for (double *p : zeroe) HIP_TRY(c, hipMemsetAsync(p, 0, sizeof(double) * E, c->stream));
    B.ready = true;
  }
  if (nstates > B.ckpt_cap) {
    B.ckpt_cap = 0;
    rc = adj_regrow(c, &B.ckpt, nstates * state);
    if (rc) return rc;
    B.ckpt_cap = nstates;
  }
  if (seg > B.seg_cap) {
    B.seg_cap = 0;
    rc = adj_regrow(c, &B.seg, (seg + 1) * cycle_slot(c));
    if (rc) return rc;
    B.seg_cap = seg;
  }
  return 0;
}

int state_copy(lulesh_ctx *c, double *buf, int to_buf) {
  touch(c);
  hipError_t e = launch_state_copy(c->stream, c->b.sc, c->b.f, c->inst[0].E, c->inst[0].N, buf,
                                   to_buf);
  return e == hipSuccess ? 0 : hip_fail(c, e, "state copy");
}

// slot j of the segment buffer; its temporaries follow the 6N + 5E state
double *seg_slot(lulesh_ctx *c, int64_t j) { return c->adj.seg + j * cycle_slot(c); }
double *slot_temps(lulesh_ctx *c, double *slot) {
  return slot + 6 * c->inst[0].N + 5 * c->inst[0].E;
}

// the state before or after a cycle, wherever it lies: in the context's own
// arrays (its current node set), or in a slot of the segment buffer
struct StateRef {
  NodeSet n;
  ElemState el;
};
StateRef slot_state(lulesh_ctx *c, double *slot) {
  const int64_t E = c->inst[0].E, N = c->inst[0].N;
  double *p = slot, *el = slot + 6 * N;
  return StateRef{NodeSet{p, p + N, p + 2 * N, p + 3 * N, p + 4 * N, p + 5 * N},
                  ElemState{el, el + E, el + 2 * E, el + 3 * E, el + 4 * E}};
}
StateRef own_state(lulesh_ctx *c, int parity) { return StateRef{c->b.f.ns[parity & 1], c->b.out}; }

// where the cycle leaves vnew delv vdov delx_* delv_* (null: where f says)
void set_temps(lulesh_ctx *c, DevFields &f, double *t) {
  if (!t) return;
  const int64_t E = c->inst[0].E;
  f.vnew = t; f.delv = t + E; f.vdov = t + 2 * E;
  f.delx_xi = t + 3 * E; f.delx_eta = t + 4 * E; f.delx_zeta = t + 5 * E;
  f.delv_xi = t + 6 * E; f.delv_eta = t + 7 * E; f.delv_zeta = t + 8 * E;
}

// The cycle `a` from the state at `from` to the one at `to`, its temporaries
// in `temps`: a cycle whose start state is to be kept writes the next state
// beside it, and nothing is copied (the copies were a launch of 7 us and a
// gap of 4 before each cycle of 44 at s=48).  parity: sc->parity at its start.
Batch between(lulesh_ctx *c, Batch a, const StateRef &from, const StateRef &to, double *temps, int parity) {
  a.f.ns[parity & 1] = from.n;
  a.f.ns[(parity & 1) ^ 1] = to.n;
  a.f.e = from.el.e; a.f.p = from.el.p; a.f.q = from.el.q; a.f.v = from.el.v; a.f.ss = from.el.ss;
  a.out = to.el;
  set_temps(c, a.f, temps);
  return a;
}
// ... from slot j of the segment to slot j + 1
Batch between_slots(lulesh_ctx *c, const Batch &a, int64_t j, int parity) {
  return between(c, a, slot_state(c, seg_slot(c, j)), slot_state(c, seg_slot(c, j + 1)),
                 slot_temps(c, seg_slot(c, j)), parity);
}
// ... with the recorded time step (timeIncrement! replaced)
Batch scheduled(Batch a, double dt) {
  a.scheduled = 1;
  a.dt = dt;
  return a;
}

// adjoint kernel arguments of the cycle that ran from `from` (start state and
// temporaries) to the node set `after`
AdjArgs stored_args(lulesh_ctx *c, const StateRef &from, double *temps, const NodeSet &after, double dt,
                    int force_pending) {
  AdjArgs a = c->adj.a;
  a.old = from.n;
  a.f.e = from.el.e; a.f.p = from.el.p; a.f.q = from.el.q; a.f.v = from.el.v; a.f.ss = from.el.ss;
  set_temps(c, a.f, temps);
  a.cur = after;
  a.dt = dt;
  a.force_pending = force_pending;
  return a;
}
AdjArgs stored_slots(lulesh_ctx *c, int64_t j, double dt, int force_pending) {
  return stored_args(c, slot_state(c, seg_slot(c, j)), slot_temps(c, seg_slot(c, j)),
                     slot_state(c, seg_slot(c, j + 1)).n, dt, force_pending);
}

// one cycle's adjoint kernels; a_node1 first folds in the force corners
// the later cycle's a_force left (force_pending), so the node-state gather
// of a_force runs as a separate a_node2 only after the last cycle
int adjoint_cycle(lulesh_ctx *c, const AdjArgs &aa, bool last) {
  const int ks[] = {AK_QEOS, AK_KIN, AK_NODE1, AK_FORCE, AK_NODE2};
  for (int kk : ks) {
    if (kk == AK_NODE2 && !last) break;
    hipError_t e = launch_adjoint(kk, c->stream, aa);
    if (e != hipSuccess) return hip_fail(c, e, "adjoint kernel");
  }
  return 0;
}

// sum_e e * elemMass, in element order (the products formed on the host too)
int energy_loss(lulesh_ctx *c, double *loss) {
  const int64_t E = c->inst[0].E;
  std::vector<double> e(E);
  HIP_TRY(c, c->host.fetch(c->stream, e.data(), c->b.f.e, sizeof(double) * E));
  double L = 0.0;
  const double *pe = e.data();
  HIP_TRY(c, c->host.stream(c->stream, c->b.f.elemMass, 1, E, [&](const double *v, int64_t, int64_t m) {
    for (int64_t i = 0; i < m; ++i) L += pe[i] * v[i];
    pe += m;
  }));
  if (loss) *loss = L;
  return 0;
}

// the parameter gradients: each the sum of its elements' shares in element order
int param_sums(lulesh_ctx *c, double (&sum)[3]) {
  double a0 = 0.0, a1 = 0.0, a2 = 0.0;
  HIP_TRY(c, c->host.stream(c->stream, c->adj.a.pacc, 3, c->inst[0].E,
                            [&](const double *v, int64_t stride, int64_t m) {
    for (int64_t i = 0; i < m; ++i) {
      a0 += v[i];
      a1 += v[i + stride];
      a2 += v[i + 2 * stride];
    }
  }));
  sum[0] = a0; sum[1] = a1; sum[2] = a2;
  return 0;
}

// The gradient run's forward pass: `ncycles` cycles of the driver loop from
// the current state with timeIncrement! recording each dt; the start state
// of cycle k is saved into save(k) when that is not null, and from cycle
// `slot_from` on each cycle's start state and temporaries go into the
// segment slots as the reverse sweep's replay would store them (so the
// last segment needs no replay).  Leaves the loss (sum_e e * elemMass,
// summed on the host in element order), the end state in
// final_state/final_sc and the dt schedule in B.dt (and dt_out).
template <typename Save>
int grad_forward(lulesh_ctx *c, int64_t ncycles, long long cycle0, Save save, int64_t slot_from,
                 double *loss, double *dt_out) {
  AdjBuffers &B = c->adj;
  const int parity0 = c->hsc[0].parity;
  const Batch a = make_args(c, 0, 0);
  Batch ta = a;  // timeIncrement! that also records the dt it takes
  ta.dt_record = B.dt;
  ta.dt_base = cycle0;
  Batch da = ta;  // k_dt that also takes the next cycle's timeIncrement!
  da.loop_mode = 2;
  int rc = clear_err(c);
  // the first cycle's timeIncrement! on its own, every later one at the end
  // of the previous cycle's k_dt (the copies between cycles read no scalar
  // it changes)
  if (!rc && ncycles > 0) rc = launch(c, KID_TIME_INCREMENT, ta);
  for (int64_t k = 0; k < ncycles && !rc; ++k) {
    double *buf = save(k);
    if (buf) rc = state_copy(c, buf, 1);
    const Batch &dk = k + 1 < ncycles ? da : a;
    Batch ak = a;
    if (!rc && k == slot_from) rc = state_copy(c, seg_slot(c, 0), 1);
    if (k >= slot_from) ak = between_slots(c, a, k - slot_from, parity0 + (int)(k & 1));
    const int ids[] = {KID_NODAL, KID_KIN, KID_QEOS};
    for (int id : ids)
      if (!rc) rc = launch(c, id, ak);
    if (!rc) rc = launch(c, KID_DT, dk);
  }
  if (!rc && slot_from < ncycles) rc = state_copy(c, seg_slot(c, ncycles - slot_from), 0);
  if (!rc) rc = finish(c, true);
  if (rc) return rc;
  if (dt_out) HIP_TRY(c, c->host.fetch(c->stream, dt_out, B.dt, sizeof(double) * ncycles));
  rc = energy_loss(c, loss);
  if (rc) return rc;
  rc = state_copy(c, B.final_state, 1);
  if (rc) return rc;
  HIP_TRY(c, hipMemcpyAsync(B.final_sc, c->b.sc, sizeof(DevScalars), hipMemcpyDeviceToDevice, c->stream));
  hipError_t e = launch_adjoint(AK_SEED, c->stream, B.a);
  if (e != hipSuccess) return hip_fail(c, e, "adjoint seed");
  return 0;
}

// gradients out, then the state the forward pass ended in
int grad_results(lulesh_ctx *c, double *grad_e, double grad_params[3]) {
  AdjBuffers &B = c->adj;
  const int64_t E = c->inst[0].E;
  if (grad_e) HIP_TRY(c, c->host.fetch(c->stream, grad_e, B.a.le, sizeof(double) * E));
  if (grad_params) {
    double sum[3];
    int r = param_sums(c, sum);
    if (r) return r;
    for (int k = 0; k < 3; ++k) grad_params[k] = sum[k];
  }
  touch(c);
  HIP_TRY(c, hipMemcpyAsync(c->b.sc, B.final_sc, sizeof(DevScalars), hipMemcpyDeviceToDevice, c->stream));
  int rc = state_copy(c, B.final_state, 0);
  if (!rc) rc = finish(c, false);
  c->partials_valid = false;
  return rc;
}

int grad_run(lulesh_ctx *c, int64_t ncycles, int64_t every, double *grad_e, double grad_params[3],
             double *loss, double *dt_out) {
  if (c->n != 1) return fail(c, LULESH_ERR_UNSUPPORTED, "the adjoint needs a one-domain context");
  if (ncycles < 1 || every < 1) return fail(c, LULESH_ERR_INVALID_ARG, "ncycles and checkpoint interval must be >= 1");
  HIP_TRY(c, hipSetDevice(c->device));
  // a checkpoint for each segment of `every` cycles but the last, whose
  // cycles the forward pass leaves in the slots
  every = std::min(every, ncycles);
  const int64_t nseg = (ncycles + every - 1) / every, slot_from = (nseg - 1) * every;
  int rc = adj_setup(c, ncycles, nseg - 1, every);
  if (rc) return rc;
  AdjBuffers &B = c->adj;
  const int64_t state = 6 * c->inst[0].N + 5 * c->inst[0].E;
  rc = know_scalars(c);
  if (rc) return rc;
  const long long cycle0 = c->hsc[0].cycle;
  int parity = c->hsc[0].parity + (int)(ncycles & 1);  // after the forward pass
  // 1. forward pass: dt schedule recorded, checkpoints and slots filled
  rc = grad_forward(
      c, ncycles, cycle0,
      [&](int64_t k) -> double * {
        return k < slot_from && k % every == 0 ? B.ckpt + (k / every) * state : nullptr;
      },
      slot_from, loss, dt_out);
  if (rc) return rc;
  // 2. reverse sweep, segment by segment: every one but the last is replayed
  // from its checkpoint, from slot to slot; then the adjoint kernels of its
  // cycles run backwards against the slots
  std::vector<double> hdt(ncycles);
  HIP_TRY(c, c->host.fetch(c->stream, hdt.data(), B.dt, sizeof(double) * ncycles));
  for (int64_t sg = nseg - 1; sg >= 0 && !rc; --sg) {
    const int64_t k0 = sg * every, k1 = (k0 + every < ncycles) ? k0 + every : ncycles;
    const int64_t L = k1 - k0;
    if (sg < nseg - 1) {
      HIP_TRY(c, hipMemcpyAsync(seg_slot(c, 0), B.ckpt + sg * state, sizeof(double) * state,
                                hipMemcpyDeviceToDevice, c->stream));
      const Batch a = make_args(c, 0, 0);
      for (int64_t j = 0; j < L && !rc; ++j, ++parity)
        rc = cycle_body(c, false, scheduled(between_slots(c, a, j, parity), hdt[k0 + j]));
    }
    for (int64_t j = L - 1; j >= 0 && !rc; --j) {
      const int64_t k = k0 + j;
      rc = adjoint_cycle(c, stored_slots(c, j, hdt[k], k == ncycles - 1 ? 0 : 1), k == 0);
    }
  }
  if (rc) return rc;
  // 3. results, then the state the forward pass ended in
  return grad_results(c, grad_e, grad_params);
}

// ---------------------------------------------------------------------------
// binomial checkpointing (revolve_cost, revolve_split and the recursion
// revolve_reverse live in lulesh_plan.h): Revolve carries the schedule out
// on the device
// ---------------------------------------------------------------------------
struct Revolve {
  lulesh_ctx *c;
  int64_t n;
  Batch a, ta, da;           // the cycle; timeIncrement! recording its dt; k_dt with it
  std::vector<int64_t> pos;  // cycle whose start state each buffer holds (-1: free)
  std::vector<double> hdt;
  int64_t frontier = 0;      // first cycle not run yet (its dt not recorded)
  int64_t cur = -1;          // cycle whose start state the context holds (-1: other)
  int64_t forward = 0;       // cycles run
  int parity = 0;            // sc->parity, which every cycle flips
  double *loss = nullptr;
  double *buf(int i) {
    const int64_t E = c->inst[0].E, N = c->inst[0].N;
    return c->adj.ckpt + (int64_t)i * (6 * N + 5 * E);
  }
  int find(int64_t k) const {
    for (size_t i = 0; i < pos.size(); ++i)
      if (pos[i] == k) return (int)i;
    return -1;
  }
  // where the start state of cycle k is: the context's own arrays, or the
  // buffer it was saved in
  int start_of(int64_t k, StateRef &from) {
    if (cur == k) {
      from = own_state(c, parity);
      return 0;
    }
    const int i = find(k);
    if (i < 0) return fail(c, LULESH_ERR_HIP, "revolve: missing saved state");
    from = slot_state(c, buf(i));
    return 0;
  }
  // cycle k as `b` places it: the first time with timeIncrement! recording
  // its dt and the time constraints, after that at the recorded dt
  int step(int64_t k, const Batch &b) {
    int rc = 0;
    if (k == frontier) {
      // (the first pass runs the cycles in order, and a k_dt takes the next
      // one's timeIncrement! along, as in grad_forward)
      if (k == 0) rc = launch(c, KID_TIME_INCREMENT, ta);
      if (!rc) rc = cycle_body(c, false, b);
      if (!rc) rc = launch(c, KID_DT, k + 1 < n ? da : a);
      ++frontier;
    } else {
      rc = cycle_body(c, false, scheduled(b, hdt[k]));
    }
    ++forward;
    ++parity;
    return rc;
  }
  int advance(int64_t from, int64_t to) {
    for (int64_t k = from; k < to; ++k) {
      StateRef start;
      int rc = start_of(k, start);
      if (!rc) rc = step(k, between(c, a, start, own_state(c, parity ^ 1), nullptr, parity));
      if (rc) return rc;
      cur = k + 1;
    }
    return 0;
  }
  int save(int64_t k) {
    const int i = find(-1);
    if (i < 0) return fail(c, LULESH_ERR_HIP, "revolve: no free state buffer");
    pos[i] = k;
    return state_copy(c, buf(i), 1);
  }
  // the forward pass has reached the end: errors, dt record, and with the
  // context's own arrays holding the end state its loss and a copy of it
  int end_of_forward() {
    AdjBuffers &B = c->adj;
    int rc = state_copy(c, seg_slot(c, 1), 0);
    if (!rc) rc = finish(c, true);
    if (!rc) rc = energy_loss(c, loss);
    if (rc) return rc;
    const size_t state = (size_t)(6 * c->inst[0].N + 5 * c->inst[0].E);
    HIP_TRY(c, hipMemcpyAsync(B.final_state, seg_slot(c, 1), sizeof(double) * state, hipMemcpyDeviceToDevice,
                              c->stream));
    HIP_TRY(c, hipMemcpyAsync(B.final_sc, c->b.sc, sizeof(DevScalars), hipMemcpyDeviceToDevice,
                              c->stream));
    HIP_TRY(c, c->host.fetch(c->stream, hdt.data(), B.dt, sizeof(double) * n));
    return 0;
  }
  // cycle k forward into slot 1, with its temporaries in slot 0, then its
  // adjoint kernels.  Its start state is read where it is, but the forward
  // pass's last cycle ends in the context's own arrays and starts from a copy.
  int youturn(int64_t k) {
    StateRef from;
    int rc = start_of(k, from);
    const bool last = k == frontier;
    double *s0 = seg_slot(c, 0), *s1 = seg_slot(c, 1);
    if (!rc && last) {
      rc = state_copy(c, s0, 1);
      from = slot_state(c, s0);
    }
    const StateRef to = slot_state(c, s1);
    if (!rc) rc = step(k, between(c, a, from, to, slot_temps(c, s0), parity));
    if (!rc && last) rc = end_of_forward();
    if (!rc) rc = adjoint_cycle(c, stored_args(c, from, slot_temps(c, s0), to.n, hdt[k], k == n - 1 ? 0 : 1), k == 0);
    cur = -1;
    return rc;
  }
  int drop(int64_t k) {
    const int i = find(k);
    if (i < 0) return fail(c, LULESH_ERR_HIP, "revolve: missing saved state");
    pos[i] = -1;
    return 0;
  }
};

int grad_run_revolve(lulesh_ctx *c, int64_t ncycles, int64_t snapshots, double *grad_e,
                     double grad_params[3], double *loss, double *dt_out, int64_t *forward_cycles) {
  if (c->n != 1) return fail(c, LULESH_ERR_UNSUPPORTED, "the adjoint needs a one-domain context");
  if (ncycles < 1 || snapshots < 1)
    return fail(c, LULESH_ERR_INVALID_ARG, "ncycles and snapshots must be >= 1");
  if (snapshots > ncycles) snapshots = ncycles;
  HIP_TRY(c, hipSetDevice(c->device));
  int rc = adj_setup(c, ncycles, snapshots, 1);
  if (rc) return rc;
  rc = know_scalars(c);
  if (rc) return rc;
  Revolve R;
  R.c = c;
  R.n = ncycles;
  R.parity = c->hsc[0].parity;
  R.a = make_args(c, 0, 0);
  R.ta = R.a;
  R.ta.dt_record = c->adj.dt;
  R.ta.dt_base = c->hsc[0].cycle;
  R.da = R.ta;
  R.da.loop_mode = 2;
  R.pos.assign((size_t)snapshots, -1);
  R.hdt.resize(ncycles);
  R.loss = loss;
  rc = clear_err(c);
  if (!rc) {
    hipError_t e = launch_adjoint(AK_SEED, c->stream, c->adj.a);
    if (e != hipSuccess) rc = hip_fail(c, e, "adjoint seed");
  }
  if (!rc) rc = R.save(0);
  R.cur = 0;
  if (!rc) rc = revolve_reverse(R, 0, ncycles, snapshots - 1);
  if (rc) return rc;
  if (dt_out) std::memcpy(dt_out, R.hdt.data(), sizeof(double) * ncycles);
  if (forward_cycles) *forward_cycles = R.forward;
  return grad_results(c, grad_e, grad_params);
}

// one lagrangeLeapFrog with the shadow mapped from the adjoint of the state
// after it to that of the state before it (Enzyme's Duplicated semantics)
int vjp_cycle(lulesh_ctx *c, double grad_params[3]) {
  if (c->n != 1) return fail(c, LULESH_ERR_UNSUPPORTED, "the adjoint needs a one-domain context");
  HIP_TRY(c, hipSetDevice(c->device));
  int rc = adj_setup(c, 0, 0, 0);
  if (rc) return rc;
  const int64_t E = c->inst[0].E;
  rc = know_scalars(c);
  if (rc) return rc;
  const int parity = c->hsc[0].parity;
  // the forward cycle exactly as lulesh_lagrange_leapfrog runs it, reading its
  // start state's element fields from a copy in the gradients' end state (the
  // node set it started from and its temporaries are there afterwards anyway)
  StateRef from = own_state(c, parity);
  const StateRef to = own_state(c, parity ^ 1);
  from.el = slot_state(c, c->adj.final_state).el;
  rc = clear_err(c);
  if (!rc) {
    hipError_t e = launch_state_copy(c->stream, c->b.sc, c->b.f, E, 0, from.el.e, 1);
    if (e != hipSuccess) rc = hip_fail(c, e, "state copy");
  }
  if (!rc) rc = cycle_body(c, true, between(c, make_args(c, 0, 0), from, to, nullptr, parity));
  // the adjoint follows without a wait for the cycle's error code: its kernels
  // look at it themselves, and leave the shadow alone if there is one
  AdjArgs aa = stored_args(c, from, nullptr, to.n, c->hsc[0].deltatime, 0);
  aa.pacc_set = aa.gated = 1;
  if (!rc) rc = adjoint_cycle(c, aa, true);
  if (!rc) rc = pull_scalars(c);
  double sum[3] = {0.0, 0.0, 0.0};
  if (!rc && grad_params) rc = param_sums(c, sum);
  if (!rc) rc = finish(c, true);
  if (rc) return rc;
  c->partials_valid = false;
  for (int k = 0; k < 3 && grad_params; ++k) grad_params[k] += sum[k];
  return 0;
}

// shadow buffer of one state field, or nullptr
double *shadow_field(lulesh_ctx *c, const char *name, int64_t *n) {
  if (!name) return nullptr;
  AdjArgs &a = c->adj.a;
  struct Entry {
    const char *name;
    double *p;
    bool node;
  };
  const Entry tab[] = {{"x", a.lx, true},   {"y", a.ly, true},   {"z", a.lz, true},
                       {"xd", a.lxd, true}, {"yd", a.lyd, true}, {"zd", a.lzd, true},
                       {"e", a.le, false},  {"p", a.lp, false},  {"q", a.lq, false},
                       {"v", a.lv, false},  {"ss", a.lss, false}};
  for (const Entry &t : tab)
    if (std::strcmp(t.name, name) == 0) {
      *n = t.node ? c->inst[0].N : c->inst[0].E;
      return t.p;
    }
  return nullptr;
}

int shadow_move(lulesh_ctx *c, const char *field, double *host, int64_t n, bool up) {
  if (c->n != 1) return fail(c, LULESH_ERR_UNSUPPORTED, "the adjoint needs a one-domain context");
  if (!host) return fail(c, LULESH_ERR_INVALID_ARG, "null buffer");
  HIP_TRY(c, hipSetDevice(c->device));
  int rc = adj_setup(c, 0, 0, 0);
  if (rc) return rc;
  int64_t len = 0;
  double *p = shadow_field(c, field, &len);
  if (!p) return fail(c, LULESH_ERR_INVALID_ARG, std::string("no shadow for field ") + (field ? field : "(null)"));
  if (n != len) return fail(c, LULESH_ERR_INVALID_ARG, "shadow field length mismatch");
  if (up) HIP_TRY(c, c->host.send(c->stream, p, host, sizeof(double) * n));
  else HIP_TRY(c, c->host.fetch(c->stream, host, p, sizeof(double) * n));
  return 0;
}

// A C++ exception must not cross the C ABI (it would terminate the host
// process): every entry point that can allocate on the host turns one into
// a status code and the context's last_error text.
int exception_status(lulesh_ctx *c) noexcept {
  int code = LULESH_ERR_HIP;
  try {
    throw;
  } catch (const std::bad_alloc &) {
    code = LULESH_ERR_HOST_MEMORY;
    if (c) try { c->last_error = "host memory allocation failed"; } catch (...) {}
  } catch (const std::exception &e) {
    if (c) try { c->last_error = std::string("C++ exception: ") + e.what(); } catch (...) {}
  } catch (...) {
    if (c) try { c->last_error = "unknown C++ exception"; } catch (...) {}
  }
  return code;
}

}  // namespace

extern "C" {

int lulesh_vjp_cycle(lulesh_ctx *c, double *grad_params) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    return vjp_cycle(c, grad_params);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_shadow_upload(lulesh_ctx *c, const char *field, const double *src, int64_t n) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    return shadow_move(c, field, const_cast<double *>(src), n, true);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_shadow_download(lulesh_ctx *c, const char *field, double *dst, int64_t n) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    return shadow_move(c, field, dst, n, false);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_grad_run(lulesh_ctx *c, int64_t ncycles, int64_t checkpoint_every, double *grad_e,
                    double *grad_params, double *loss, double *dt_schedule) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    return grad_run(c, ncycles, checkpoint_every, grad_e, grad_params, loss, dt_schedule);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_grad_run_revolve(lulesh_ctx *c, int64_t ncycles, int64_t snapshots, double *grad_e,
                            double *grad_params, double *loss, double *dt_schedule,
                            int64_t *forward_cycles) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    return grad_run_revolve(c, ncycles, snapshots, grad_e, grad_params, loss, dt_schedule,
                            forward_cycles);
  } catch (...) {
    return exception_status(c);
  }
}

int64_t lulesh_revolve_cycles(int64_t ncycles, int64_t snapshots) {
  if (ncycles < 1 || snapshots < 1) return -1;
  if (snapshots > ncycles) snapshots = ncycles;
  return ncycles + revolve_cost(ncycles, snapshots - 1);
}

int lulesh_replay(lulesh_ctx *c, const double *dt, int64_t ncycles) {
  try {
    if (!c || !dt || ncycles < 0) return LULESH_ERR_INVALID_ARG;
    if (c->n != 1) return fail(c, LULESH_ERR_UNSUPPORTED, "replay needs a one-domain context");
    HIP_TRY(c, hipSetDevice(c->device));
    const Batch a = make_args(c, 0, 0);
    int rc = clear_err(c);
    for (int64_t k = 0; k < ncycles && !rc; ++k) rc = cycle_body(c, true, scheduled(a, dt[k]));
    if (rc) return rc;
    c->partials_valid = false;
    return finish(c, true);
  } catch (...) {
    return exception_status(c);
  }
}

const char *lulesh_error_string(int code) {
  if (code == LULESH_OK) return "ok";
  if (code >= 1 && code <= 9) return kErrText[code];
  if (code == LULESH_ERR_INVALID_ARG) return "invalid argument";
  if (code == LULESH_ERR_HIP) return "HIP runtime error";
  if (code == LULESH_ERR_UNSUPPORTED) return "unsupported";
  if (code == LULESH_ERR_HOST_MEMORY) return "host memory allocation failed";
  if (code == LULESH_ERR_SCRATCH)
    return "domain too large for the fixed scratch array (nx > LULESH_NOALLOC_MAX_NX)";
  return "unknown error";
}

int lulesh_create(int32_t nx, int32_t nr, int32_t balance, int32_t cost, int32_t quirks,
                  int32_t device, lulesh_ctx **out) {
  try {
    return create(1, &nx, nullptr, nullptr, &nr, &balance, &cost, quirks, device, out);
  } catch (...) {
    return exception_status(nullptr);
  }
}

int lulesh_batch_create(int32_t n, const int32_t *nx, const double *einit_scale,
                        const double *hgcoef, const int32_t *nr, int32_t quirks, int32_t device,
                        lulesh_ctx **out) {
  try {
    return create(n, nx, einit_scale, hgcoef, nr, nullptr, nullptr, quirks, device, out);
  } catch (...) {
    return exception_status(nullptr);
  }
}

int32_t lulesh_batch_size(const lulesh_ctx *c) { return c ? c->n : -1; }

int lulesh_destroy(lulesh_ctx *c) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    release(c);
    delete c;
    return 0;
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_reset(lulesh_ctx *c) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    HIP_TRY(c, hipSetDevice(c->device));
    touch(c);
    hipError_t e = launch_init(c->stream, c->b);
    if (e != hipSuccess) return hip_fail(c, e, "init kernels");
    c->partials_valid = false;
    int rc = pull_scalars(c);
    return rc ? rc : finish(c, false);
  } catch (...) {
    return exception_status(c);
  }
}

int64_t lulesh_num_elem(const lulesh_ctx *c) { return c ? c->inst[0].E : -1; }
int64_t lulesh_num_node(const lulesh_ctx *c) { return c ? c->inst[0].N : -1; }
int64_t lulesh_batch_num_elem(const lulesh_ctx *c, int32_t inst) {
  return (c && inst >= 0 && inst < c->n) ? c->inst[inst].E : -1;
}
int64_t lulesh_batch_num_node(const lulesh_ctx *c, int32_t inst) {
  return (c && inst >= 0 && inst < c->n) ? c->inst[inst].N : -1;
}
const char *lulesh_last_error(const lulesh_ctx *c) { return c ? c->last_error.c_str() : "null context"; }

int lulesh_batch_download(lulesh_ctx *c, int32_t inst, const char *field, double *dst, int64_t n) {
  try {
    int rc = check_inst(c, inst);
    if (rc) return rc;
    if (!dst) return LULESH_ERR_INVALID_ARG;
    DevScalars s;
    rc = get_inst_scalars(c, inst, &s);
    if (rc) return rc;
    FieldRef r = find_field(c, inst, field, s.parity);
    if (!r.ptr) return fail(c, LULESH_ERR_INVALID_ARG, std::string("unknown field ") + (field ? field : "(null)"));
    if (n != r.n) return fail(c, LULESH_ERR_INVALID_ARG, "field length mismatch");
    HIP_TRY(c, c->host.fetch(c->stream, dst, r.ptr, (size_t)n * sizeof(double)));
    return finish(c, false);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_batch_upload(lulesh_ctx *c, int32_t inst, const char *field, const double *src, int64_t n) {
  try {
    int rc = check_inst(c, inst);
    if (rc) return rc;
    if (!src) return LULESH_ERR_INVALID_ARG;
    DevScalars s;
    rc = get_inst_scalars(c, inst, &s);
    if (rc) return rc;
    FieldRef r = find_field(c, inst, field, s.parity);
    if (!r.ptr) return fail(c, LULESH_ERR_INVALID_ARG, std::string("unknown field ") + (field ? field : "(null)"));
    if (n != r.n) return fail(c, LULESH_ERR_INVALID_ARG, "field length mismatch");
    HIP_TRY(c, c->host.send(c->stream, r.ptr, src, (size_t)n * sizeof(double)));
    c->partials_valid = false;
    return finish(c, false);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_download(lulesh_ctx *c, const char *field, double *dst, int64_t n) {
  try {
    return lulesh_batch_download(c, 0, field, dst, n);
  } catch (...) {
    return exception_status(c);
  }
}
int lulesh_upload(lulesh_ctx *c, const char *field, const double *src, int64_t n) {
  try {
    return lulesh_batch_upload(c, 0, field, src, n);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_batch_download_elem_bc(lulesh_ctx *c, int32_t inst, uint32_t *dst, int64_t n) {
  try {
    int rc = check_inst(c, inst);
    if (rc) return rc;
    if (!dst || n != c->inst[inst].E) return fail(c, LULESH_ERR_INVALID_ARG, "elemBC length mismatch");
    HIP_TRY(c, hipSetDevice(c->device));
    HIP_TRY(c, c->host.fetch(c->stream, dst, c->b.f.elemBC + c->inst[inst].e0, (size_t)n * 4));
    return finish(c, false);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_batch_upload_elem_bc(lulesh_ctx *c, int32_t inst, const uint32_t *src, int64_t n) {
  try {
    int rc = check_inst(c, inst);
    if (rc) return rc;
    if (!src || n != c->inst[inst].E) return fail(c, LULESH_ERR_INVALID_ARG, "elemBC length mismatch");
    HIP_TRY(c, hipSetDevice(c->device));
    HIP_TRY(c, c->host.send(c->stream, c->b.f.elemBC + c->inst[inst].e0, src, (size_t)n * 4));
    return finish(c, false);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_download_elem_bc(lulesh_ctx *c, uint32_t *dst, int64_t n) {
  try {
    return lulesh_batch_download_elem_bc(c, 0, dst, n);
  } catch (...) {
    return exception_status(c);
  }
}
int lulesh_upload_elem_bc(lulesh_ctx *c, const uint32_t *src, int64_t n) {
  try {
    return lulesh_batch_upload_elem_bc(c, 0, src, n);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_batch_get_scalar(lulesh_ctx *c, int32_t inst, const char *name, double *value) {
  try {
    int rc = check_inst(c, inst);
    if (rc) return rc;
    if (!name || !value) return LULESH_ERR_INVALID_ARG;
    DevScalars s;
    rc = get_inst_scalars(c, inst, &s);
    if (rc) return rc;
    const std::string nm(name);
    if (nm == "cycle") {
      *value = (double)s.cycle;
      return 0;
    }
    double *slot = scalar_slot(&s, nm);
    if (!slot) return fail(c, LULESH_ERR_INVALID_ARG, "unknown scalar " + nm);
    *value = *slot;
    return 0;
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_batch_set_scalar(lulesh_ctx *c, int32_t inst, const char *name, double value) {
  try {
    int rc = check_inst(c, inst);
    if (rc) return rc;
    if (!name) return LULESH_ERR_INVALID_ARG;
    DevScalars s;
    rc = get_inst_scalars(c, inst, &s);
    if (rc) return rc;
    const std::string nm(name);
    if (nm == "cycle") {
      if (!(value >= 0.0) || value != std::floor(value))
        return fail(c, LULESH_ERR_INVALID_ARG, "cycle must be a non-negative integer");
      s.cycle = (long long)value;
    } else {
      double *slot = scalar_slot(&s, nm);
      if (!slot) return fail(c, LULESH_ERR_INVALID_ARG, "unknown scalar " + nm);
      *slot = value;
    }
    const bool known = c->known;
    touch(c);
    c->hsc[inst] = s;
    HIP_TRY(c, hipMemcpyAsync(c->b.sc + inst, c->hsc + inst, sizeof(DevScalars),
                              hipMemcpyHostToDevice, c->stream));
    c->partials_valid = false;
    rc = finish(c, false);
    c->known = known && !rc;
    return rc;
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_get_scalar(lulesh_ctx *c, const char *name, double *value) {
  try {
    return lulesh_batch_get_scalar(c, 0, name, value);
  } catch (...) {
    return exception_status(c);
  }
}
int lulesh_set_scalar(lulesh_ctx *c, const char *name, double value) {
  try {
    return lulesh_batch_set_scalar(c, 0, name, value);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_region_download(lulesh_ctx *c, int32_t inst, const char *name, int64_t *dst,
                           int64_t n) {
  try {
    int rc = check_inst(c, inst);
    if (rc) return rc;
    if (!name || !dst) return fail(c, LULESH_ERR_INVALID_ARG, "null name or buffer");
    rc = ensure_regions(c);
    if (rc) return rc;
    const RegionSets &R = c->regions[(size_t)inst];
    const std::string s(name);
    if (s == "regNumList" || s == "regElemlist") {
      const std::vector<int32_t> &v = s == "regNumList" ? R.numList : R.elemList;
      if (n != (int64_t)v.size()) return fail(c, LULESH_ERR_INVALID_ARG, "region field length mismatch");
      for (int64_t i = 0; i < n; ++i) dst[i] = v[(size_t)i];
      return 0;
    }
    const std::vector<int64_t> *v = s == "regCSR" ? &R.csr
                                    : s == "regReps" ? &R.reps
                                    : s == "regSorted" ? &R.sorted : nullptr;
    if (!v) return fail(c, LULESH_ERR_INVALID_ARG, "unknown region field " + s);
    if (n != (int64_t)v->size()) return fail(c, LULESH_ERR_INVALID_ARG, "region field length mismatch");
    std::copy(v->begin(), v->end(), dst);
    return 0;
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_set_cost_mode(lulesh_ctx *c, int32_t on) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    if (!on) {
      c->b.cost_mode = 0;
      return 0;
    }
    if (!c->elem_rep) {
      int rc = ensure_regions(c);
      if (rc) return rc;
      // an element's rep is its region's: regReps[regSorted[regNumList[e]]]
      std::vector<int> rep((size_t)c->E_total);
      for (int i = 0; i < c->n; ++i) {
        const RegionSets &R = c->regions[(size_t)i];
        const int64_t e0 = c->inst[i].e0;
        for (int64_t e = 0; e < c->inst[i].E; ++e) {
          const int64_t r = R.sorted[(size_t)R.numList[(size_t)e] - 1];
          const int64_t k = R.reps[(size_t)r - 1];
          rep[(size_t)(e0 + e)] = (int)(k < 1 ? 1 : (k > INT32_MAX ? INT32_MAX : k));
        }
      }
      HIP_TRY(c, hipSetDevice(c->device));
      int *d = nullptr;
      rc = dev_alloc(c, &d, c->E_total);
      if (rc) return rc;
      HIP_TRY(c, hipMemcpy(d, rep.data(), sizeof(int) * rep.size(), hipMemcpyHostToDevice));
      c->elem_rep = d;
    }
    c->b.elem_rep = c->elem_rep;
    c->b.cost_mode = 1;
    return 0;
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_set_keep_aux(lulesh_ctx *c, int32_t on) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    c->keep_aux = on ? 1 : 0;
    return 0;
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_time_increment(lulesh_ctx *c) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    HIP_TRY(c, hipSetDevice(c->device));
    int rc = launch(c, KID_TIME_INCREMENT, make_args(c, 0, 0));
    if (!rc) rc = pull_scalars(c);  // the caller's loop test reads them
    if (rc) return rc;
    return finish(c, false);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_lagrange_nodal(lulesh_ctx *c) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    HIP_TRY(c, hipSetDevice(c->device));
    const Batch a = make_args(c, 0, 0);
    int rc = clear_err(c);
    if (!rc) rc = launch(c, KID_NODAL, a);
    if (rc) return rc;
    c->partials_valid = false;
    return finish(c, true);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_lagrange_elements(lulesh_ctx *c) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    HIP_TRY(c, hipSetDevice(c->device));
    const Batch a = make_args(c, 0, 0);
    int rc = clear_err(c);
    if (!rc) rc = launch(c, KID_KIN, a);
    if (!rc) rc = launch(c, KID_QEOS, a);
    if (rc) return rc;
    rc = finish(c, true);
    c->partials_valid = (rc == 0);
    c->partials = a.parts;
    return rc;
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_calc_time_constraints(lulesh_ctx *c) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    HIP_TRY(c, hipSetDevice(c->device));
    Batch a = make_args(c, 0, 0);
    a.parts = c->partials_valid ? c->partials : c->inst[0].ebn;
    int rc = 0;
    if (!c->partials_valid) rc = launch(c, KID_DTPART, a);
    if (!rc) rc = launch(c, KID_DT, a);
    if (rc) return rc;
    c->partials_valid = false;
    return finish(c, false);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_lagrange_leapfrog(lulesh_ctx *c) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    HIP_TRY(c, hipSetDevice(c->device));
    const Batch a = make_args(c, 0, 0);
    int rc = clear_err(c);
    const int ids[] = {KID_NODAL, KID_KIN, KID_QEOS, KID_DT};
    for (int id : ids)
      if (!rc) rc = launch(c, id, a);
    if (rc) return rc;
    c->partials_valid = false;
    return finish(c, true);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_run(lulesh_ctx *c, int64_t num_iters, int64_t *cycles_run) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    std::vector<int64_t> cyc(c->n, 0);
    int rc = run_cycles(c, num_iters, cyc.data());
    if (cycles_run) *cycles_run = cyc[0];
    return rc;
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_batch_run(lulesh_ctx *c, int64_t num_iters, int64_t *cycles_run) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    return run_cycles(c, num_iters, cycles_run);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_batch_error(const lulesh_ctx *c, int32_t inst) {
  if (!c || inst < 0 || inst >= c->n) return LULESH_ERR_INVALID_ARG;
  const int err = c->hsc[inst].err;
  return (err >= 1 && err <= 9) ? err : 0;
}

int lulesh_batch_verify(lulesh_ctx *c, int32_t inst, double out[4]) {
  try {
    int rc = check_inst(c, inst);
    if (rc) return rc;
    if (!out) return LULESH_ERR_INVALID_ARG;
    const int64_t nx = c->inst[inst].s;
    std::vector<double> e(nx * nx);
    HIP_TRY(c, hipSetDevice(c->device));
    HIP_TRY(c, c->host.fetch(c->stream, e.data(), c->b.f.e + c->inst[inst].e0, e.size() * sizeof(double)));
    rc = finish(c, false);
    if (rc) return rc;
    // src/utils.jl:134-152
    double MaxAbsDiff = 0.0, MaxRelDiff = 0.0, TotalAbsDiff = 0.0;
    for (int64_t j = 1; j <= nx; ++j)
      for (int64_t k = j + 1; k <= nx; ++k) {
        const double a = e[(j - 1) * nx + k - 1], b = e[(k - 1) * nx + j - 1];
        const double AbsDiff = std::fabs(a - b);
        TotalAbsDiff = TotalAbsDiff + AbsDiff;
        if (MaxAbsDiff < AbsDiff) MaxAbsDiff = AbsDiff;
        const double RelDiff = AbsDiff / b;
        if (MaxRelDiff < RelDiff) MaxRelDiff = RelDiff;
      }
    out[0] = e[0];
    out[1] = MaxAbsDiff;
    out[2] = TotalAbsDiff;
    out[3] = MaxRelDiff;
    return 0;
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_verify(lulesh_ctx *c, double out[4]) { return lulesh_batch_verify(c, 0, out); }

int lulesh_set_timing(lulesh_ctx *c, int32_t on) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    c->timing = on != 0;
    for (int i = 0; i < LULESH_K_COUNT; ++i) {
      c->ktime[i] = 0.0;
      c->kcount[i] = 0;
    }
    return 0;
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_kernel_time(lulesh_ctx *c, int32_t id, double *total_ms, int64_t *launches) {
  try {
    if (!c || id < 0 || id >= LULESH_K_COUNT) return LULESH_ERR_INVALID_ARG;
    if (total_ms) *total_ms = c->ktime[id];
    if (launches) *launches = c->kcount[id];
    return 0;
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_math_check(int32_t op, const double *a, const double *b, double *out, int64_t n,
                      int32_t device) {
  try {
    if (op < 0 || op > 2 || !a || !out || n < 0 || (op == 2 && !b)) return LULESH_ERR_INVALID_ARG;
    if (n == 0) return 0;
    if (hipSetDevice(device) != hipSuccess) return LULESH_ERR_HIP;
    double *d = nullptr;
    const size_t bytes = (size_t)n * sizeof(double);
    if (hipMalloc(&d, 3 * bytes) != hipSuccess) return LULESH_ERR_HIP;
    int rc = 0;
    if (hipMemcpy(d, a, bytes, hipMemcpyHostToDevice) != hipSuccess) rc = LULESH_ERR_HIP;
    if (!rc && op == 2 && hipMemcpy(d + n, b, bytes, hipMemcpyHostToDevice) != hipSuccess)
      rc = LULESH_ERR_HIP;
    if (!rc && launch_math(nullptr, op, d, d + n, d + 2 * n, n) != hipSuccess) rc = LULESH_ERR_HIP;
    if (!rc && hipDeviceSynchronize() != hipSuccess) rc = LULESH_ERR_HIP;
    if (!rc && hipMemcpy(out, d + 2 * n, bytes, hipMemcpyDeviceToHost) != hipSuccess)
      rc = LULESH_ERR_HIP;
    (void)hipFree(d);
    return rc;
  } catch (...) {
    return exception_status(nullptr);
  }
}

int lulesh_set_nodal_depth(lulesh_ctx *c, int32_t cz) {
  try {
    if (!c || cz < 0 || cz > 1024) return LULESH_ERR_INVALID_ARG;
    HIP_TRY(c, hipSetDevice(c->device));
    c->depth_req = cz;
    return plan_nodal(c, cz);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_set_nodal_tiles(lulesh_ctx *c, int32_t lo, int32_t hi) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    if (lo == 0 && hi == 0) {
      lo = 16;
      hi = 32;
    }
    if (lo < 2 || hi < lo || hi > BLOCK / 2)
      return fail(c, LULESH_ERR_INVALID_ARG, "tile widths must satisfy 2 <= lo <= hi <= 128");
    HIP_TRY(c, hipSetDevice(c->device));
    c->tile_lo = lo;
    c->tile_hi = hi;
    return plan_nodal(c, c->depth_req);
  } catch (...) {
    return exception_status(c);
  }
}

int lulesh_nodal_tile(const lulesh_ctx *c, int32_t inst, int32_t *shape) {
  if (!c || !shape || inst < 0 || inst >= c->n) return LULESH_ERR_INVALID_ARG;
  const InstDesc &I = c->inst[inst];
  shape[0] = I.etx;
  shape[1] = I.ety;
  shape[2] = I.tx;
  shape[3] = I.ty;
  return 0;
}

int32_t lulesh_nodal_depth(const lulesh_ctx *c) { return c ? c->inst[0].cz : -1; }

int lulesh_autotune(lulesh_ctx *c, int32_t *chosen, double *best_ms) {
  try {
    if (!c) return LULESH_ERR_INVALID_ARG;
    HIP_TRY(c, hipSetDevice(c->device));
    // k_nodal with its parity flip switched off reads the current node set
    // and writes only the other one, so it can be timed on the live state
    // without changing it.  Candidates: tile-width ranges (the default first)
    // x z-depths (the model's first).
    const int fam[][2] = {{16, 32}, {16, 16}, {12, 21}, {8, 32}, {24, 32}};
    const int cand[] = {0, 2, 4, 8, 16, 32};
    int maxs = 0;
    for (const InstDesc &I : c->inst) maxs = I.s > maxs ? I.s : maxs;
    // the tuning launches may raise an error code the live state would
    // raise on its next cycle; the scalars are put back as they were, so
    // an error already on the device survives and a new one does not appear
    int rc = know_scalars(c);
    if (rc) return rc;
    const std::vector<DevScalars> saved(c->hsc, c->hsc + c->n);
    touch(c);
    int best_f = -1, best_cz = -1;
    float best_t = 0.f;
    hipEvent_t ea = get_event(c), eb = get_event(c);
    if (!ea || !eb) return fail(c, LULESH_ERR_HIP, "hipEventCreate failed");
    for (int fi = 0; fi < (int)(sizeof(fam) / sizeof(fam[0])) && !rc; ++fi) {
      c->tile_lo = fam[fi][0];
      c->tile_hi = fam[fi][1];
      for (int cz : cand) {
        if (cz > 2 && cz / 2 > maxs + 1) break;
        rc = plan_nodal(c, cz);
        if (rc) break;
        Batch a = make_args(c, 0, 0);
        a.flip = 0;      // the current node set stays current
        a.keep_aux = 0;  // fx.. and xdd.. keep the last real cycle's values
        hipError_t e = hipSuccess;
        for (int w = 0; w < 2 && e == hipSuccess; ++w) e = launch_kernel(KID_NODAL, c->stream, a);
        if (e == hipSuccess) e = hipEventRecord(ea, c->stream);
        for (int r = 0; r < 5 && e == hipSuccess; ++r) e = launch_kernel(KID_NODAL, c->stream, a);
        if (e == hipSuccess) e = hipEventRecord(eb, c->stream);
        if (e == hipSuccess) e = hipEventSynchronize(eb);
        float ms = 0.f;
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, ea, eb);
        if (e != hipSuccess) {
          rc = hip_fail(c, e, "autotune");
          break;
        }
        if (best_f < 0 || ms < best_t) {
          best_f = fi;
          best_cz = cz;
          best_t = ms;
        }
      }
    }
    c->event_pool.push_back(ea);
    c->event_pool.push_back(eb);
    if (rc) return rc;
    c->tile_lo = fam[best_f][0];
    c->tile_hi = fam[best_f][1];
    c->depth_req = best_cz;
    rc = plan_nodal(c, best_cz);
    if (rc) return rc;
    std::copy(saved.begin(), saved.end(), c->hsc);
    HIP_TRY(c, hipMemcpyAsync(c->b.sc, c->hsc, sizeof(DevScalars) * c->n, hipMemcpyHostToDevice,
                              c->stream));
    rc = finish(c, false);
    if (rc) return rc;
    if (chosen) *chosen = c->inst[0].cz;
    if (best_ms) *best_ms = best_t / 5.0;
    return 0;
  } catch (...) {
    return exception_status(c);
  }
}

const char *lulesh_kernel_name(int32_t id) {
  static const char *names[] = {"k_nodal", "k_kin", "k_qeos", "k_dt"};
  if (id < 0 || id >= LULESH_K_COUNT) return "";
  return names[id];
}

}  // extern "C"
