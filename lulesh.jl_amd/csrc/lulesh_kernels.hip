// MI355X (gfx950) kernels of one LULESH Lagrange leap-frog cycle, FP64.
//
// One cycle = four launches on the context stream (a small domain's has
// other forms of the first three, k_nodal_planes and k_elems, below):
//   k_nodal  stress corner forces (integrateStressForElems), Flanagan-
//            Belytschko hourglass corner forces (calcHourglassControlForElems
//            + calcFBHourglassForceForElems), their fixed-order sums at the
//            nodes (stress, then hourglass, as the reference sums them),
//            acceleration, symmetry-plane BCs, velocity, position
//   k_kin    element-parallel: calcKinematicsForElems + the deviatoric loop
//            + calcMonotonicQGradientsForElems
//   k_qeos   element-parallel: calcMonotonicQRegionForElems, the QStop check,
//            applyMaterialPropertiesForElems/evalEOSForElems,
//            updateVolumesForElems and the per-element Courant/hydro terms,
//            reduced to one minimum per block
//   k_dt     one block: the final minima (calcTimeConstraintsForElems) and,
//            in driver-loop mode, the loop test and the next timeIncrement!
//            (one domain of few minima: the next nodal launch does that)
// No atomics touch field data: a node sums its corners in the reference's
// order, so the FP64 result is deterministic run to run.
#include "lulesh_elem.h"
#include "lulesh_kernels.h"

namespace lulesh {

// ---------------------------------------------------------------------------
// structured-mesh indexing (buildMesh!, src/domain.jl:117-174)
// ---------------------------------------------------------------------------
LDEV void elem_nodes(int64_t e, int s, int64_t (&nid)[8]) {
  const int64_t s1 = s + 1, P = s1 * s1;
  const int64_t col = e % s, rest = e / s;
  const int64_t row = rest % s, plane = rest / s;
  const int64_t n0 = plane * P + row * s1 + col;
  nid[0] = n0;
  nid[1] = n0 + 1;
  nid[2] = n0 + s1 + 1;
  nid[3] = n0 + s1;
  nid[4] = n0 + P;
  nid[5] = n0 + P + 1;
  nid[6] = n0 + P + s1 + 1;
  nid[7] = n0 + P + s1;
}

template <typename T>
LDEV void gather8(const T *__restrict__ src, const int64_t (&nid)[8], T (&out)[8]) {
#pragma unroll
  for (int n = 0; n < 8; ++n) out[n] = src[nid[n]];
}

LDEV void raise(int *err, int code) { atomicMin(err, code); }
LDEV void raise(DevScalars *sc, int code) { raise(&sc->err, code); }

// Stores of k_kin's and k_qeos' outputs that do not keep their lines in the
// caches: the next kernel reads them back from memory anyway, and with the
// lines not left behind the following kernel's reads run faster (k_qeos
// 229 -> 214 us at s=192 with k_kin's outputs so written, and k_kin 289 ->
// 285 us with k_qeos' outputs; k_nodal's node stores so written make
// k_nodal slower, 670 -> 685 us, and stay ordinary).  k_qeos reads its own
// element's values the same way (they are used once): k_qeos 213 -> 205 us,
// and k_dt, whose partial minima then stay in cache, 13 -> 10 us.
template <typename T>
LDEV T ld_nt(const T *p) {
  return __builtin_nontemporal_load(p);
}
template <typename T>
LDEV void st_nt(T *base, uint32_t boff, T v) {
  __builtin_nontemporal_store(v, (T *)((char *)base + boff));
}
template <typename T>
LDEV void st_nt(T *p, T v) {
  __builtin_nontemporal_store(v, p);
}

// instance i's view of the flat field arrays
LDEV DevFields slice(const DevFields &f, const InstDesc &I) {
  DevFields g;
  const int64_t a = I.e0, b = I.n0;
  g.e = f.e + a; g.p = f.p + a; g.q = f.q + a; g.ql = f.ql + a; g.qq = f.qq + a;
  g.v = f.v + a; g.volo = f.volo + a; g.delv = f.delv + a; g.vdov = f.vdov + a;
  g.arealg = f.arealg + a; g.ss = f.ss + a; g.elemMass = f.elemMass + a; g.vnew = f.vnew + a;
  g.delv_xi = f.delv_xi + a; g.delv_eta = f.delv_eta + a; g.delv_zeta = f.delv_zeta + a;
  g.delx_xi = f.delx_xi + a; g.delx_eta = f.delx_eta + a; g.delx_zeta = f.delx_zeta + a;
  g.dxx = f.dxx + a; g.dyy = f.dyy + a; g.dzz = f.dzz + a; g.elemBC = f.elemBC + a;
  for (int k = 0; k < 2; ++k) {
    g.ns[k].x = f.ns[k].x + b; g.ns[k].y = f.ns[k].y + b; g.ns[k].z = f.ns[k].z + b;
    g.ns[k].xd = f.ns[k].xd + b; g.ns[k].yd = f.ns[k].yd + b; g.ns[k].zd = f.ns[k].zd + b;
  }
  g.xdd = f.xdd + b; g.ydd = f.ydd + b; g.zdd = f.zdd + b;
  g.fx = f.fx + b; g.fy = f.fy + b; g.fz = f.fz + b; g.nodalMass = f.nodalMass + b;
  return g;
}

LDEV ElemState slice(const ElemState &s, const InstDesc &I) {
  return ElemState{s.e + I.e0, s.p + I.e0, s.q + I.e0, s.v + I.e0, s.ss + I.e0};
}

// NodeSet k of a sliced field view, chosen without indexing a local array
// by a run-time value (that would put the struct in scratch memory)
LDEV NodeSet pick(const DevFields &f, int k) {
  NodeSet r;
  r.x = k ? f.ns[1].x : f.ns[0].x;
  r.y = k ? f.ns[1].y : f.ns[0].y;
  r.z = k ? f.ns[1].z : f.ns[0].z;
  r.xd = k ? f.ns[1].xd : f.ns[0].xd;
  r.yd = k ? f.ns[1].yd : f.ns[0].yd;
  r.zd = k ? f.ns[1].zd : f.ns[0].zd;
  return r;
}

// Per-block instance lookup for the element-, node- and k_nodal-shaped
// grids: every block belongs to exactly one instance (instances start on a
// block boundary), so the lookup is uniform over the block.  k_kin and
// k_qeos take their blocks from host-built tables (kin_table, qeos_table:
// XCD-aware orders that leave finished instances out).
// k_kin (no barriers, no LDS, three waves per SIMD by its registers) runs
// one-wave workgroups of KIN_CHUNK elements: a finished wave's slot is
// refilled without waiting for a whole 4-wave workgroup to fit (at s=192:
// 0.292 against 0.304 ms per launch)
static_assert(KIN_CHUNK == 64, "k_kin workgroups are one wave");

#define LULESH_ELEM_PREAMBLE(B)                                                  \
  const int inst_ = (B).eblock_inst[blockIdx.x];                               \
  const InstDesc I = (B).inst[inst_];                                          \
  DevScalars *sc = (B).sc + inst_;                                             \
  const int s = I.s;                                                           \
  const int64_t E = I.E;                                                       \
  const int64_t e = (int64_t)(blockIdx.x - I.eb0) * BLOCK + threadIdx.x;       \
  const DevFields f = slice((B).f, I);
#define LULESH_ELEM_PREAMBLE_T(B, TABLE)                                         \
  const int vb_ = (B).TABLE[blockIdx.x];                                       \
  if (vb_ < 0) return;                                                         \
  const int inst_ = (B).eblock_inst[vb_];                                      \
  const InstDesc I = (B).inst[inst_];                                          \
  DevScalars *sc = (B).sc + inst_;                                             \
  const int s = I.s;                                                           \
  const int64_t E = I.E;                                                       \
  const int64_t e = (int64_t)(vb_ - I.eb0) * BLOCK + threadIdx.x;              \
  const DevFields f = slice((B).f, I);
#define LULESH_NODE_PREAMBLE(B)                                                  \
  const int inst_ = (B).nblock_inst[blockIdx.x];                               \
  const InstDesc I = (B).inst[inst_];                                          \
  DevScalars *sc = (B).sc + inst_;                                             \
  const int s = I.s;                                                           \
  const int64_t N = I.N;                                                       \
  const int64_t n = (int64_t)(blockIdx.x - I.nb0) * BLOCK + threadIdx.x;       \
  const DevFields f = slice((B).f, I);

// timeIncrement!, src/domain.jl:920-961, from given time constraints
struct TimeStep {
  double time, deltatime;
  long long cycle;
};
LDEV TimeStep next_time_step(const DevScalars &S, double dtcourant, double dthydro) {
  TimeStep r{S.time, S.deltatime, S.cycle};
  double targetdt = S.stoptime - r.time;
  if (S.dtfixed <= 0.0 && r.cycle != 0) {
    const double olddt = r.deltatime;
    double gnewdt = __builtin_huge_val();
    if (dtcourant < gnewdt) gnewdt = dtcourant / 2.0;
    if (dthydro < gnewdt) gnewdt = (dthydro * 2.0) / 3.0;
    double newdt = gnewdt;
    const double ratio = newdt / olddt;
    if (ratio >= 1.0) {
      if (ratio < S.deltatimemultlb) newdt = olddt;
      else if (ratio > S.deltatimemultub) newdt = olddt * S.deltatimemultub;
    }
    newdt = jmin(newdt, S.dtmax);
    r.deltatime = newdt;
  }
  if (r.deltatime < targetdt && targetdt < (4.0 * r.deltatime) / 3.0)
    targetdt = (2.0 * r.deltatime) / 3.0;
  if (targetdt < r.deltatime) r.deltatime = targetdt;
  r.time = r.time + r.deltatime;
  r.cycle = r.cycle + 1;
  return r;
}
LDEV void store(DevScalars *sc, const TimeStep &ts) {
  sc->time = ts.time;
  sc->deltatime = ts.deltatime;
  sc->cycle = ts.cycle;
}
LDEV void time_increment(DevScalars *sc) {
  store(sc, next_time_step(*sc, sc->dtcourant, sc->dthydro));
}
// the driver loop's test (examples/benchmark.jl:82,95)
LDEV bool loop_goes_on(const DevScalars *sc, int err) {
  return err == ERR_NONE && sc->cycle < sc->num_iters && sc->time < sc->stoptime;
}
// The error code the loop test sees when a nodal launch makes it: what that
// launch itself raises goes to err_nodal[parity] (a workgroup that starts
// late must not take it for the previous cycle's), what the previous one
// raised is in err_nodal[parity ^ 1].
LDEV int previous_err(const DevScalars *sc, int par) {
  const int e = par ? sc->err_nodal[0] : sc->err_nodal[1];
  return e < sc->err ? e : sc->err;
}
LDEV void gather_errs(DevScalars *sc) {
  int e = sc->err;
  e = sc->err_nodal[0] < e ? sc->err_nodal[0] : e;
  e = sc->err_nodal[1] < e ? sc->err_nodal[1] : e;
  sc->err = e;
  sc->err_nodal[0] = sc->err_nodal[1] = ERR_NONE;
}

// The end of the previous cycle of the driver loop, taken at the head of the
// next one (B.defer_dt: one domain whose partial minima are few).  k_dt on
// its own is a launch of one workgroup, 4-5 us of a small domain's cycle of
// 29 with the gap before it; here every workgroup of the nodal launch folds the partial minima for
// itself, beside its own first loads, and the last one to finish stores the
// scalars (all the others have read the old ones by then).  A cycle of the
// device loop at s=16 takes 28.6 -> 26.2 us, s=48 54.1 -> 51.3, s=64 70.4 ->
// 67.9, s=96 142.3 -> 141.7.  Each wave's minimum goes through LDS and a
// barrier the kernel has anyway (dt_fold_wave, then dt_fold_take).
struct DtFold {
  double courant, hydro;
};
LDEV DtFold dt_fold_load(const Batch &B) {
  const double2 *__restrict__ p = (const double2 *)B.dtpart;
  double a = 1.0e+20, b = 1.0e+20;
  for (int i = threadIdx.x; i < B.parts; i += BLOCK) {
    const double2 v = p[i];
    a = v.x < a ? v.x : a;
    b = v.y < b ? v.y : b;
  }
  return DtFold{a, b};
}
LDEV void dt_fold_wave(DtFold d, double (*m)[2]) {
  double a = d.courant, b = d.hydro;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double oa = __shfl_xor(a, off, 64), ob = __shfl_xor(b, off, 64);
    a = oa < a ? oa : a;
    b = ob < b ? ob : b;
  }
  if ((threadIdx.x & 63) == 0) {
    m[threadIdx.x >> 6][0] = a;
    m[threadIdx.x >> 6][1] = b;
  }
}
LDEV DtFold dt_fold_take(const DevScalars &S, const double (*m)[2]) {
  double a = m[0][0], b = m[0][1];
#pragma unroll
  for (int w = 1; w < BLOCK / 64; ++w) {
    a = m[w][0] < a ? m[w][0] : a;
    b = m[w][1] < b ? m[w][1] : b;
  }
  return DtFold{a < 1.0e+20 ? a : S.dtcourant, b < 1.0e+20 ? b : S.dthydro};
}
// what the last workgroup to finish stores
struct DtNow {
  DtFold d;
  TimeStep ts;
};
// what a nodal workgroup that defers keeps of it in LDS
struct DtShared {
  double m[BLOCK / 64][2];
  DtNow now;
};
LDEV DtShared &dt_shared() {
  __shared__ DtShared d;
  return d;
}
LDEV DtNow dt_now_of(const DevScalars &S, bool fold, const double (*m)[2]) {
  if (!fold) return DtNow{DtFold{S.dtcourant, S.dthydro}, TimeStep{S.time, S.deltatime, S.cycle}};
  const DtFold d = dt_fold_take(S, m);
  return DtNow{d, next_time_step(S, d.courant, d.hydro)};
}
// A nodal workgroup of a loop that has ended: the constraints are folded all
// the same, and the last workgroup stores them.
LDEV void dt_fold_end(DevScalars *sc, int last, double (*m)[2], const Batch &B) {
  dt_fold_wave(dt_fold_load(B), m);
  __syncthreads();
  if (threadIdx.x == 0 && atomicAdd(&sc->nodal_done, 1) == last) {
    const DtFold d = dt_fold_take(*sc, m);
    sc->nodal_done = 0;
    sc->dtcourant = d.courant;
    sc->dthydro = d.hydro;
    gather_errs(sc);
    sc->active = 0;
    sc->dt_pending = 0;
  }
}

// ---------------------------------------------------------------------------
// Domain(prob) on the device (src/domain.jl:117-174, 615-771, 822-916)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(BLOCK) void k_init_nodes(Batch B) {
  LULESH_NODE_PREAMBLE(B)
  (void)sc;
  if (n >= N) return;
  const int64_t s1 = s + 1;
  const int64_t col = n % s1, rest = n / s1;
  const int64_t row = rest % s1, plane = rest / s1;
  // tx = 1.125*(colLoc*nx + col)/meshEdgeElems with colLoc = 0, tp = 1
  const NodeSet &S = f.ns[0];
  S.x[n] = (1.125 * (double)col) / (double)s;
  S.y[n] = (1.125 * (double)row) / (double)s;
  S.z[n] = (1.125 * (double)plane) / (double)s;
  S.xd[n] = 0.0; S.yd[n] = 0.0; S.zd[n] = 0.0;
  f.xdd[n] = 0.0; f.ydd[n] = 0.0; f.zdd[n] = 0.0;
  f.fx[n] = 0.0; f.fy[n] = 0.0; f.fz[n] = 0.0;
}

__global__ __launch_bounds__(BLOCK) void k_init_elems(Batch B) {
  LULESH_ELEM_PREAMBLE(B)
  (void)sc;
  if (e >= E) return;
  int64_t nid[8];
  elem_nodes(e, s, nid);
  double X[8], Y[8], Z[8];
  gather8(f.ns[0].x, nid, X); gather8(f.ns[0].y, nid, Y); gather8(f.ns[0].z, nid, Z);
  const double vol = elem_volume(X, Y, Z);
  f.volo[e] = vol;
  f.elemMass[e] = vol;
  f.v[e] = 1.0;
  f.e[e] = 0.0; f.p[e] = 0.0; f.q[e] = 0.0; f.ss[e] = 0.0;
  f.ql[e] = 0.0; f.qq[e] = 0.0; f.delv[e] = 0.0; f.vdov[e] = 0.0; f.arealg[e] = 0.0;
  f.vnew[e] = 0.0; f.dxx[e] = 0.0; f.dyy[e] = 0.0; f.dzz[e] = 0.0;
  f.delv_xi[e] = 0.0; f.delv_eta[e] = 0.0; f.delv_zeta[e] = 0.0;
  f.delx_xi[e] = 0.0; f.delx_eta[e] = 0.0; f.delx_zeta[e] = 0.0;
  // setupBoundaryConditions for the single rank: SYMM on min faces, FREE on max
  const int64_t col = e % s, rest = e / s;
  const int64_t row = rest % s, plane = rest / s;
  uint32_t bc = 0;
  if (plane == 0) bc |= ZETA_M_SYMM;
  if (plane == s - 1) bc |= ZETA_P_FREE;
  if (row == 0) bc |= ETA_M_SYMM;
  if (row == s - 1) bc |= ETA_P_FREE;
  if (col == 0) bc |= XI_M_SYMM;
  if (col == s - 1) bc |= XI_P_FREE;
  f.elemBC[e] = bc;
}

// nodal mass: volume/8 of each adjacent element added in ascending element
// order, the order of the element loop at src/domain.jl:709-727
__global__ __launch_bounds__(BLOCK) void k_init_mass(Batch B) {
  LULESH_NODE_PREAMBLE(B)
  (void)sc;
  if (n >= N) return;
  const int64_t s1 = s + 1;
  const int i = (int)(n % s1), j = (int)((n / s1) % s1), k = (int)(n / (s1 * s1));
  double m = 0.0;
  for (int dk = -1; dk <= 0; ++dk) {
    const int ek = k + dk;
    if (ek < 0 || ek >= s) continue;
    for (int dj = -1; dj <= 0; ++dj) {
      const int ej = j + dj;
      if (ej < 0 || ej >= s) continue;
      for (int di = -1; di <= 0; ++di) {
        const int ei = i + di;
        if (ei < 0 || ei >= s) continue;
        const int64_t e = ((int64_t)ek * s + ej) * s + ei;
        m = m + f.volo[e] / 8.0;
      }
    }
  }
  f.nodalMass[n] = m;
}

// scalars of src/domain.jl:663-701, energy deposit and dt0 (738-749)
// one thread per instance; the deposit is einit_scale * einit (1 for the
// reference problem) and dt0 is computed from it
__global__ void k_init_scalars(Batch B) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= B.n) return;
  const InstDesc I = B.inst[i];
  DevScalars *sc = B.sc + i;
  const int s = I.s;
  double *e0 = B.f.e + I.e0;
  const double *volo = B.f.volo + I.e0;
  sc->dthydro = 1e20;
  sc->dtcourant = 1e20;
  sc->time = 0.;
  sc->dtfixed = -1.0e-6;
  sc->deltatimemultlb = 1.1;
  sc->deltatimemultub = 1.2;
  sc->stoptime = 1.0e-2;
  sc->dtmax = 1.0e-2;
  sc->cycle = 0;
  sc->e_cut = 1.0e-7;
  sc->p_cut = 1.0e-7;
  sc->q_cut = 1.0e-7;
  sc->u_cut = 1.0e-7;
  sc->v_cut = 1.0e-10;
  sc->hgcoef = I.hgcoef;
  sc->ss4o3 = 4.0 / 3.0;
  sc->qstop = 1.0e+12;
  sc->monoq_max_slope = 1.0;
  sc->monoq_limiter_mult = 2.0;
  sc->qlc_monoq = 0.5;
  sc->qqc_monoq = 2.0 / 3.0;
  sc->qqc = 2.0;
  sc->pmin = 0.;
  sc->emin = -1.0e+15;
  sc->dvovmax = 0.1;
  sc->eosvmax = 1.0e+9;
  sc->eosvmin = 1.0e-9;
  sc->refdens = 1.0;
  const double ebase = 3.948746e+7;
  const double scale = (double)s / 45.0;
  const double einit = (((ebase * scale) * scale) * scale) * I.einit_scale;
  e0[0] = einit;
  sc->deltatime = (.5 * cbrt_cr(volo[0])) / sqrt(2.0 * einit);
  sc->err = ERR_NONE;
  sc->active = 0;
  sc->num_iters = 0;
  sc->parity = 0;
  sc->nodal_done = 0;
  sc->dt_pending = 0;
  sc->err_nodal[0] = sc->err_nodal[1] = ERR_NONE;
}

// ---------------------------------------------------------------------------
// the cycle
// ---------------------------------------------------------------------------
__global__ void k_time_increment(Batch B) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= B.n) return;
  DevScalars *sc = B.sc + i;
  time_increment(sc);
  if (i == 0 && B.dt_record) B.dt_record[sc->cycle - 1 - B.dt_base] = sc->deltatime;
}

// driver loop head (examples/benchmark.jl:82-84): the first iteration is
// entered whenever time < stoptime
__global__ void k_run_begin(Batch B) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= B.n) return;
  DevScalars *sc = B.sc + i;
  sc->num_iters = B.num_iters;
  sc->err = ERR_NONE;
  sc->err_nodal[0] = sc->err_nodal[1] = ERR_NONE;
  sc->dt_pending = 0;
  const int go = sc->time < sc->stoptime;
  sc->active = go;
  if (go) time_increment(sc);
}

// ---------------------------------------------------------------------------
// lagrangeNodal (src/domain.jl:1840-1872) as one kernel.
//
// A workgroup owns a column of nodes (up to etx x ety; 16 x 14 for inner
// tiles at s=192, see nodal_tile) and a z-chunk of its node planes (the
// instance's NodalCut: cz0 planes for the first chunk, cz for the others,
// the last one up to node plane s).  It marches
// up the chunk one element plane at a time: its threads compute the corner
// forces of the etx x ety elements around the node tile
// (integrateStressForElems + calcFBHourglassForceForElems arithmetic), stage
// them in LDS, and the node threads fold them into per-node running sums.
// A node's sum takes its elements in ascending element id -- the plane below
// first, then its own plane, each in (row, col) order -- which is exactly
// the nodeElemCornerList order of the reference's gathers
// (src/domain.jl:1112-1127, 1678-1693); stress and hourglass corners are
// summed separately and added at the end, as the reference does.  Finished
// node planes are updated at once (acceleration, symmetry BCs, velocity,
// position; src/domain.jl:1781-1838) into the other NodeSet, so tiles that
// still read the old positions of shared halo nodes never see new values.
// Elements on tile edges are computed by every tile that needs them
// (17x15x(cz+1) per 16x14xcz nodes for an inner 17 x 15 tile): no corner
// force ever goes to HBM.
//
// What bounds it: FP64 issue.  A wave needs about 1,500 vector instructions
// per element plane (6,000 cycles of a SIMD, whose two waves belong to two
// workgroups), and a wave alone waits for as long again unless its memory
// and LDS accesses are few and early.  Hence the node ring (a plane is
// fetched once per tile, one plane ahead, instead of 24 16-byte gathers per
// element, which kept the address path busy for 700 cycles per wave and
// plane), the element values and nodal mass asked for a phase ahead, and
// LDS reads without branches.  Timestamps inside the kernel at s=192: 19,000
// cycles per plane for the workgroup issued first before, 12,500 now.  At
// s=192 a launch takes 487 us against 615 (26 TFLOP/s with the 1,430
// additions and products per element and plane, halo included), the batch of
// 64 domains 396 against 500, s=63 36 against 39.  252 VGPRs and 78 KB of
// LDS: two workgroups per CU by either.
// ---------------------------------------------------------------------------
// Corner forces in LDS: [corner q of the bottom face][element slot][x y z of
// corner q, x y z of corner q + 4 above it], so that a node takes what one
// element gives it in three 16-byte reads (the 48-byte stride spreads
// sixteen lanes over all 64 banks).  Slot BLOCK holds zeros.
constexpr int LDS_PAIR = (BLOCK + 1) * 6;  // doubles per corner q
LDEV int lds_at(int q, int slot) { return q * LDS_PAIR + slot * 6; }
LDEV void lds_put(double *lds, int slot, const double (&F)[8][3]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    double2 *p = (double2 *)(lds + lds_at(q, slot));
    p[0] = make_double2(F[q][0], F[q][1]);
    p[1] = make_double2(F[q][2], F[q + 4][0]);
    p[2] = make_double2(F[q + 4][1], F[q + 4][2]);
  }
}
// one phase of a node's sums: the bottom corners of its four elements end
// the sum c of its own plane, their top corners start the sum n of the next
LDEV void lds_fold(const double *lds, int p00, int p10, int p01, int p11, double &c0, double &c1,
                   double &c2, double &n0, double &n1, double &n2) {
  const int at4[4] = {p00, p10, p01, p11};
  double2 v[4][3];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const double2 *p = (const double2 *)(lds + at4[k]);
    v[k][0] = p[0]; v[k][1] = p[1]; v[k][2] = p[2];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    c0 = c0 + v[k][0].x; c1 = c1 + v[k][0].y; c2 = c2 + v[k][1].x;
    n0 = n0 + v[k][1].y; n1 = n1 + v[k][2].x; n2 = n2 + v[k][2].y;
  }
}

// The node planes the element and node lanes of a tile read, kept in LDS:
// the (etx + 1) x (ety + 1) nodes around its elements, six arrays of
// `NPATCH` doubles per plane (NODAL_PATCH, or NODAL_PATCH_WIDE for tiles
// whose patch is larger: one workgroup per CU instead of two).
// an LDS read the compiler neither moves past pinned values nor merges
LDEV double lds_read(const double *p) {
  typedef __attribute__((address_space(3))) const volatile double lds_double;
  return *(lds_double *)p;
}
// the values of one node array at an element's eight corners: the bottom
// nodes from plane b, the top ones from plane t of the ring (rows of w)
LDEV void hex_patch(const double *b, const double *t, int p, int w, double (&out)[8]) {
  out[0] = b[p]; out[1] = b[p + 1]; out[3] = b[p + w]; out[2] = b[p + w + 1];
  out[4] = t[p]; out[5] = t[p + 1]; out[7] = t[p + w]; out[6] = t[p + w + 1];
}

// The hourglass columns g[n][m] = Gamma[n][m] - (dV/dx_n . projection m) / V
// and their velocity projections h[m] = sum_n g[n][m] v_n of an element,
// node by node (src/domain.jl:1516-1600): node n's volume derivative and
// velocity are used and dropped before the next node's, every sum in the
// reference's order.
template <int NPATCH>
LDEV void hourglass_gh(double (&X)[8], double (&Y)[8], double (&Z)[8], const double (*rb)[NPATCH],
                       const double (*rt)[NPATCH], int pe, int pw, int quirks, double volinv,
                       double (&g)[8][4], double (&h)[4][3]) {
  // the 36 edge sums the face normals and the volume derivatives have in
  // common are formed twice: kept over both, they alone hold 72 registers
  // and k_nodal needs 294
#pragma unroll
  for (int n = 0; n < 8; ++n) pin3(X[n], Y[n], Z[n]);
  double hmx[4], hmy[4], hmz[4];
  hourglass_modes(X, hmx);
  hourglass_modes(Y, hmy);
  hourglass_modes(Z, hmz);
  // node n + 1's velocity is asked for before node n's arithmetic (a
  // volatile read stays on its side of the statements that pin values), and
  // one wait per node leaves the run of FP64 instructions aligned: k_nodal
  // at s=192 501 -> 487 us
  double v[2][3];
  auto velocity = [&](int n) {
    const bool right = n == 1 || n == 2 || n == 5 || n == 6, back = n == 2 || n == 3 || n == 6 || n == 7;
    const double(*rv)[NPATCH] = n < 4 ? rb : rt;
    const int vo = pe + (right ? 1 : 0) + (back ? pw : 0);
#pragma unroll
    for (int c = 0; c < 3; ++c) v[n & 1][c] = lds_read(&rv[3 + c][vo]);
  };
  velocity(0);
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    double &vx = v[n & 1][0], &vy = v[n & 1][1], &vz = v[n & 1][2];
    pin3(vx, vy, vz);
    if (n < 7) velocity(n + 1);
    double dx, dy, dz;
    volume_derivative_node(X, Y, Z, quirks, n, dx, dy, dz);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      g[n][m] = gam(n, m) - volinv * (((dx * hmx[m]) + (dy * hmy[m])) + (dz * hmz[m]));
      if (n == 0) {
        h[m][0] = g[n][m] * vx; h[m][1] = g[n][m] * vy; h[m][2] = g[n][m] * vz;
      } else {
        h[m][0] = h[m][0] + g[n][m] * vx;
        h[m][1] = h[m][1] + g[n][m] * vy;
        h[m][2] = h[m][2] + g[n][m] * vz;
      }
    }
    pin3(h[0][0], h[1][0], h[2][0]);
  }
}
LDEV double hourglass_force(const double (&g)[4], const double (&h)[4][3], int c, double coefficient) {
  return coefficient * (((g[0] * h[0][c] + g[1] * h[1][c]) + g[2] * h[2][c]) + g[3] * h[3][c]);
}
// acceleration, symmetry planes, velocity and position of one node
// (src/domain.jl:1781-1838), written to the other node set
struct NodeOld {
  double mass, x, y, z, xd, yd, zd;
};
LDEV void node_update(const NodeSet &out, const DevFields &f, uint32_t no, int ni, int nj, int k,
                      double fx, double fy, double fz, const NodeOld &o, double dt, double u_cut,
                      int keep_aux) {
  double xdd = fx / o.mass, ydd = fy / o.mass, zdd = fz / o.mass;
  // symmetry planes: the col 0, row 0 and plane 0 node sets
  // (src/domain.jl:773-791, 1787-1806)
  if (ni == 0) xdd = 0.0;
  if (nj == 0) ydd = 0.0;
  if (k == 0) zdd = 0.0;
  double xd = o.xd + xdd * dt;
  if (fabs(xd) < u_cut) xd = 0.0;
  double yd = o.yd + ydd * dt;
  if (fabs(yd) < u_cut) yd = 0.0;
  double zd = o.zd + zdd * dt;
  if (fabs(zd) < u_cut) zd = 0.0;
  at(out.xd, no) = xd;
  at(out.yd, no) = yd;
  at(out.zd, no) = zd;
  at(out.x, no) = o.x + xd * dt;
  at(out.y, no) = o.y + yd * dt;
  at(out.z, no) = o.z + zd * dt;
  if (keep_aux) {
    at(f.fx, no) = fx; at(f.fy, no) = fy; at(f.fz, no) = fz;
    at(f.xdd, no) = xdd; at(f.ydd, no) = ydd; at(f.zdd, no) = zdd;
  }
}

// The instance's last workgroup to finish makes the node set just written
// current: every workgroup of the instance has then started (and read the
// old parity and scalars), and the next kernel sees the new ones (a kernel
// boundary orders the stores; no fence is needed inside a launch).
LDEV void nodal_finish(const Batch &B, DevScalars *sc, int par, const DtNow *now) {
  if (now) {
    sc->dtcourant = now->d.courant;
    sc->dthydro = now->d.hydro;
    store(sc, now->ts);
    sc->dt_pending = 1;
  }
  if (B.scheduled) {
    sc->deltatime = B.dt;
    sc->time = sc->time + B.dt;
    sc->cycle = sc->cycle + 1;
  }
  sc->nodal_done = 0;
  sc->parity = par ^ 1;
}

// QK: the quirk bits Q1 | Q2 known at compile time, -1: taken from the batch
// DEFER: one domain whose previous cycle's end is taken here (B.defer_dt)
template <int QK, int NPATCH, bool DEFER>
__global__ __launch_bounds__(BLOCK) void k_nodal(Batch B) {
  // values a thread fetches of the patch nodes past BLOCK
  constexpr int XV = (6 * (NPATCH - 1 - BLOCK) + BLOCK - 1) / BLOCK;
  // XCD-aware order: the dispatcher deals workgroups round-robin over the 8
  // XCDs, and the host's table gives each XCD a contiguous run of blocks
  // (neighbouring tiles, whose halos then share its L2; -8 % at s=192)
  const int vb = B.gblock_order[blockIdx.x];
  if (vb < 0) return;
  const int inst_ = DEFER ? 0 : B.gblock_inst[vb];
  const InstDesc I = DEFER ? B.one : B.inst[inst_];
  DevScalars *sc = B.sc + inst_;
  if (B.gated && !sc->active) return;
  const int s = I.s, quirks = QK < 0 ? B.quirks : QK, keep_aux = B.keep_aux;
  const int etx = I.etx, ety = I.ety;
  const DevFields f = slice(B.f, I);
  const int lb = vb - I.gb0;
  const int tx = lb % I.tx, ty = (lb / I.tx) % I.ty, chunk = lb / (I.tx * I.ty);
  // the tile's first node column (the first tile owns etx columns, inner
  // ones etx-1) and how far its first element lane sits before it (none
  // before node 0)
  const int i0 = tx == 0 ? 0 : etx + (tx - 1) * (etx - 1);
  const int j0 = ty == 0 ? 0 : ety + (ty - 1) * (ety - 1);
  const int oi = tx != 0, oj = ty != 0;
  const int iend = tx == I.tx - 1 ? s + 1 : i0 + etx - oi;
  const int jend = ty == I.ty - 1 ? s + 1 : j0 + ety - oj;
  const NodalCut cut{I.cz0, I.cz, I.nch};
  const int k0 = nodal_chunk_begin(cut, chunk);
  const int k1 = nodal_chunk_end(cut, chunk, s);
  const int t = threadIdx.x, ti = t % etx, tj = t / etx;
  const int s1 = s + 1;
  // this thread's element in each plane, and its node column (threads past
  // the etx x ety tile take part in the barriers only)
  const int ei = i0 - oi + ti, ej = j0 - oj + tj;
  const bool elem_col = tj < ety && ei < s && ej < s;
  const int ni = i0 + ti, nj = j0 + tj;
  const bool node_col = tj < ety && ni < iend && nj < jend;
  // the four elements around the node column, in ascending id order:
  // (ni-1,nj-1) (ni,nj-1) (ni-1,nj) (ni,nj) at lanes (ti+oi-1, tj+oj-1) ..
  // (ti+oi, tj+oj); where one does not exist, the slot that holds zeros
  // stands in for it (a node column the tile owns has its elements among
  // the tile's lanes).  Adding that zero changes no bit, and every lane's
  // reads are unconditional: all of a phase's are in flight together
  // instead of one exec-masked group after the other.
  const bool h00 = ni >= 1 && nj >= 1, h10 = ni < s && nj >= 1;
  const bool h01 = ni >= 1 && nj < s, h11 = ni < s && nj < s;
  const int l00 = (tj + oj - 1) * etx + (ti + oi - 1);
  const int p00 = lds_at(2, node_col && h00 ? l00 : BLOCK);
  const int p10 = lds_at(3, node_col && h10 ? l00 + 1 : BLOCK);
  const int p01 = lds_at(1, node_col && h01 ? l00 + etx : BLOCK);
  const int p11 = lds_at(0, node_col && h11 ? l00 + etx + 1 : BLOCK);
  // corner of the node in element (ox,oy) = node offset inside it:
  // (1,1)->2, (0,1)->3, (1,0)->1, (0,0)->0 at the bottom; +4 at the top

  const int par = sc->parity;
  const NodeSet in = pick(f, par), out = pick(f, par ^ 1);
  const double hourg = sc->hgcoef;
  const bool hg_on = hourg > 0.0;
  const double u_cut = sc->u_cut;
  const double dt = B.scheduled ? B.dt : sc->deltatime;
  int *const err = DEFER ? &sc->err_nodal[par] : &sc->err;
  [[maybe_unused]] DevScalars S;
  [[maybe_unused]] bool fold = false;
  if constexpr (DEFER) {
    S = *sc;
    fold = S.dt_pending;
    if (fold) {
      if (!loop_goes_on(sc, previous_err(sc, par))) {
        dt_fold_end(sc, I.gbn - 1, dt_shared().m, B);
        return;
      }
      dt_fold_wave(dt_fold_load(B), dt_shared().m);
    }
  }

  // [corner of the bottom face][element slot, slot BLOCK zero][bottom xyz, top xyz]
  __shared__ __align__(16) double lds[LDS_PAIR * 4];
  if (t < 24) lds[lds_at(t / 6, BLOCK) + t % 6] = 0.0;
  // Two node planes of the tile, [plane & 1][x y z xd yd zd][node]: the
  // (etx + 1) x (ety + 1) nodes around its elements.  An element takes its
  // eight nodes from here, so a plane is fetched once per tile (six 8-byte
  // loads per thread) instead of 24 paired 16-byte gathers per element.
  __shared__ double ring[2][6][NPATCH];
  const int pw = etx + 1, np = pw * (ety + 1);
  const uint32_t us1 = (uint32_t)s1, node_plane = us1 * us1;
  // What this thread fetches of a plane: the six values of patch node t,
  // and the values t, t + BLOCK .. of the patch nodes past BLOCK (array by
  // array), all clamped into the domain
  const int pa = t < np ? t : np - 1;
  auto node_of = [&](int p) {
    const int i = i0 - oi + p % pw, j = j0 - oj + p / pw;
    return (uint32_t)(j < s ? j : s) * us1 + (uint32_t)(i < s ? i : s);
  };
  const uint32_t na = node_of(pa);
  uint32_t nx[XV];
  int px[XV];  // where it goes in a plane of the ring, -1: nothing
  const double *xsrc[XV];
#pragma unroll
  for (int k = 0; k < XV; ++k) {
    const int xn = np - BLOCK, xi = t + k * BLOCK, xc = xn > 0 ? xi / xn : 6;
    nx[k] = 0;
    px[k] = -1;
    xsrc[k] = in.x;
    if (xc < 6) {
      const int p = BLOCK + xi % xn;
      nx[k] = node_of(p);
      px[k] = xc * NPATCH + p;
      xsrc[k] = xc == 0 ? in.x : xc == 1 ? in.y : xc == 2 ? in.z : xc == 3 ? in.xd : xc == 4 ? in.yd : in.zd;
    }
  }
  const int pe = tj < ety ? tj * pw + ti : 0;               // the element's first node
  const int po = tj < ety ? (tj + oj) * pw + ti + oi : 0;   // the own node column

  double cs0 = 0.0, cs1 = 0.0, cs2 = 0.0, ch0 = 0.0, ch1 = 0.0, ch2 = 0.0;  // node plane ek

  // Issue order.  A CU holds two k_nodal workgroups, one wave of each per
  // SIMD, and a SIMD issues the older wave first when both are ready, so a
  // workgroup that starts beside a running one falls behind it and marches
  // its last planes alone, at the issue rate of one wave.  Such a workgroup
  // (any after the first nodal_lead dealt to its XCD, one per CU) is issued
  // first for the first 55 % of its planes (50 % leaves it ~20 us behind
  // at s=192).
  const int lead_end = k0 - 1 + (11 * (k1 - k0 + 1)) / 20;
  if ((int)(blockIdx.x >> 3) >= B.nodal_lead) __builtin_amdgcn_s_setprio(1);

  // Element and node addresses are clamped into the domain, so that every
  // lane loads without a branch; lanes without an element or node column of
  // their own use none of it.
  const uint32_t ce = (uint32_t)(ej < s ? ej : s - 1) * (uint32_t)s + (uint32_t)(ei < s ? ei : s - 1);
  const uint32_t cn = (uint32_t)(nj < s1 ? nj : s) * us1 + (uint32_t)(ni < s1 ? ni : s);
  const uint32_t elem_plane = (uint32_t)s * (uint32_t)s;
  // the first element plane; node planes ek0 and ek0 + 1 and the first
  // plane's element values
  const int ek0 = k0 > 0 ? k0 - 1 : 0;
  for (int k = 0; k < 2; ++k) {
    const uint32_t o = ((uint32_t)(ek0 + k) * node_plane + na) * 8u;
    double(*r)[NPATCH] = ring[(ek0 + k) & 1];
    const double a0 = at(in.x, o), a1 = at(in.y, o), a2 = at(in.z, o);
    const double a3 = at(in.xd, o), a4 = at(in.yd, o), a5 = at(in.zd, o);
    r[0][pa] = a0; r[1][pa] = a1; r[2][pa] = a2; r[3][pa] = a3; r[4][pa] = a4; r[5][pa] = a5;
#pragma unroll
    for (int j = 0; j < XV; ++j)
      if (px[j] >= 0) (&r[0][0])[px[j]] = xsrc[j][(uint32_t)(ek0 + k) * node_plane + nx[j]];
  }
  double vp, vq, vv, vvolo, vss, vem;
  {
    const uint32_t eo = ((uint32_t)ek0 * elem_plane + ce) * 8u;
    vp = at(f.p, eo); vq = at(f.q, eo); vv = at(f.v, eo);
    vvolo = at(f.volo, eo); vss = at(f.ss, eo); vem = at(f.elemMass, eo);
  }
  __syncthreads();
  // (read in the first plane's node update, several barriers from here)
  if constexpr (DEFER) {
    const DtNow w = dt_now_of(S, fold, dt_shared().m);
    if (t == 0) dt_shared().now = w;
  }

  for (int ek = ek0; ek < k1; ++ek) {
    const bool plane = ek < s;
    if (ek == lead_end) __builtin_amdgcn_s_setprio(0);
    // asked for now, used after this plane's arithmetic: node plane ek + 2
    // (for the next element plane) and the nodal mass of plane ek
    const bool more = ek + 1 < k1 && ek + 1 < s;
    double a0, a1, a2, a3, a4, a5, ax[XV];
    if (more) {
      const uint32_t o = ((uint32_t)(ek + 2) * node_plane + na) * 8u;
      a0 = at(in.x, o); a1 = at(in.y, o); a2 = at(in.z, o);
      a3 = at(in.xd, o); a4 = at(in.yd, o); a5 = at(in.zd, o);
#pragma unroll
      for (int j = 0; j < XV; ++j)
        if (px[j] >= 0) ax[j] = xsrc[j][(uint32_t)(ek + 2) * node_plane + nx[j]];
    }
    const uint32_t no = ((uint32_t)ek * node_plane + cn) * 8u;
    const double mass = at(f.nodalMass, no);
    double hgf[8][3];
    if (plane && elem_col) {
      const double(*rb)[NPATCH] = ring[ek & 1], (*rt)[NPATCH] = ring[(ek + 1) & 1];
      double X[8], Y[8], Z[8];
      hex_patch(rb[0], rt[0], pe, pw, X);
      hex_patch(rb[1], rt[1], pe, pw, Y);
      hex_patch(rb[2], rt[2], pe, pw, Z);
      // stress corners, src/domain.jl:1097-1108 (sig from 963-969)
      if (jacobian_volume64(X, Y, Z) <= 0.0) raise(err, ERR_EARLY_VOLUME);
      {
        double B[8][3];
        node_normals16(X, Y, Z, quirks, B);
        const double ms = (-((-vp) - vq)) * 0.0625;
#pragma unroll
        for (int n = 0; n < 8; ++n)
#pragma unroll
          for (int c = 0; c < 3; ++c) B[n][c] = ms * B[n][c];
        lds_put(lds, t, B);
      }
      // hourglass corners, src/domain.jl:1707-1729 and 1505-1639
      const double determ = vvolo * vv;
      if (vv <= 0.0) raise(err, ERR_HG_VOLUME);
      if (hg_on) {
        const double volume13 = cbrt_cr(determ);
        const double coefficient = ((((-hourg) * 0.01) * vss) * vem) / volume13;
        double g[8][4], h[4][3];
        hourglass_gh(X, Y, Z, rb, rt, pe, pw, quirks, 1.0 / determ, g, h);
#pragma unroll
        for (int n = 0; n < 8; ++n)
#pragma unroll
          for (int c = 0; c < 3; ++c)
            hgf[n][c] = hourglass_force(g[n], h, c, coefficient);
      }
    }
    __syncthreads();
    // stress: finish node plane ek with the bottom corners of plane ek, start
    // node plane ek+1 with its top corners (plane ek precedes plane ek+1)
    double ns0 = 0.0, ns1 = 0.0, ns2 = 0.0, nh0 = 0.0, nh1 = 0.0, nh2 = 0.0;
    if (plane) lds_fold(lds, p00, p10, p01, p11, cs0, cs1, cs2, ns0, ns1, ns2);
    const double(*ro)[NPATCH] = ring[ek & 1];
    const double ox = ro[0][po], oy = ro[1][po], oz = ro[2][po];
    const double oxd = ro[3][po], oyd = ro[4][po], ozd = ro[5][po];
    __syncthreads();
    if (hg_on && plane && elem_col) lds_put(lds, t, hgf);
    // every wave is past its reads of node plane ek: plane ek + 2 takes its
    // place, and the next plane's element values are asked for
    if (more) {
      double(*r)[NPATCH] = ring[ek & 1];
      r[0][pa] = a0; r[1][pa] = a1; r[2][pa] = a2; r[3][pa] = a3; r[4][pa] = a4; r[5][pa] = a5;
#pragma unroll
      for (int j = 0; j < XV; ++j)
        if (px[j] >= 0) (&r[0][0])[px[j]] = ax[j];
      const uint32_t eo = ((uint32_t)(ek + 1) * elem_plane + ce) * 8u;
      vp = at(f.p, eo); vq = at(f.q, eo); vv = at(f.v, eo);
      vvolo = at(f.volo, eo); vss = at(f.ss, eo); vem = at(f.elemMass, eo);
    }
    __syncthreads();
    if (hg_on && plane) lds_fold(lds, p00, p10, p01, p11, ch0, ch1, ch2, nh0, nh1, nh2);
    __syncthreads();
    // node plane ek is complete: calcAccelerationForNodes ..
    // calcPositionForNodes for it
    if (node_col && ek >= k0) {
      double fx = cs0, fy = cs1, fz = cs2;
      if (hg_on) {
        fx = fx + ch0;
        fy = fy + ch1;
        fz = fz + ch2;
      }
      double step = dt;
      if constexpr (DEFER) step = dt_shared().now.ts.deltatime;
      node_update(out, f, no, ni, nj, ek, fx, fy, fz, NodeOld{mass, ox, oy, oz, oxd, oyd, ozd}, step,
                  u_cut, keep_aux);
    }
    cs0 = ns0; cs1 = ns1; cs2 = ns2;
    ch0 = nh0; ch1 = nh1; ch2 = nh2;
  }
  if (B.flip) {
    __syncthreads();
    if (t == 0) {
      if (atomicAdd(&sc->nodal_done, 1) == I.gbn - 1) {
        const DtNow *now = nullptr;
        if constexpr (DEFER) now = &dt_shared().now;
        nodal_finish(B, sc, par, now);
      }
    }
  }
}

// lagrangeNodal of a single small domain: one node plane per workgroup, the
// element planes below and above it computed side by side.
//
// On a domain that leaves the chip mostly idle a launch of k_nodal lasts as
// long as one wave's march, at least two element planes one after the other
// (4.5 us each).  Here a workgroup's first two waves take the plane below
// the node plane and the other two the plane above, so both take one plane's
// time; each keeps only the corners that touch the node plane, which leaves
// room to stage stress and hourglass corners together: one barrier instead
// of four per plane.  The arithmetic and every sum's order are k_nodal's.
// It does twice k_nodal's element work per node plane, so it is used only
// while its workgroups all run at once (nodal_planes_fit).  Event-timed
// launches: s=8 10.1 us against the march's 17.6, s=16 10.8 against 17.8,
// s=30 15.3 against 17.9.  Bound by one wave's latency: launch, the loads of
// the patch, 7,500 cycles of arithmetic, one fold.
constexpr int PLANE_LANES = BLOCK / 2;  // element lanes per element plane
template <int QK>
__global__ __launch_bounds__(BLOCK) void k_nodal_planes(Batch B) {
  DevScalars *sc = B.sc;
  if (B.gated && !sc->active) return;
  const InstDesc &I = B.one;
  const DevFields &f = B.f;
  const int s = I.s, s1 = s + 1, etx = B.ptile.etx, ety = B.ptile.ety;
  const int tx = blockIdx.x, ty = blockIdx.y, k = blockIdx.z;
  const int i0 = tx == 0 ? 0 : etx + (tx - 1) * (etx - 1);
  const int j0 = ty == 0 ? 0 : ety + (ty - 1) * (ety - 1);
  const int oi = tx != 0, oj = ty != 0;
  const int iend = tx == B.ptile.tx - 1 ? s + 1 : i0 + etx - oi;
  const int jend = ty == B.ptile.ty - 1 ? s + 1 : j0 + ety - oj;
  const int t = threadIdx.x, l = t % PLANE_LANES;
  const int upper = __builtin_amdgcn_readfirstlane(t / PLANE_LANES);
  const int ti = l % etx, tj = l / etx;
  const int ei = i0 - oi + ti, ej = j0 - oj + tj, ek = k - 1 + upper;
  const bool elem = tj < ety && ei < s && ej < s && ek >= 0 && ek < s;
  const int ni = i0 + ti, nj = j0 + tj;
  const bool node = upper && tj < ety && ni < iend && nj < jend;

  const int par = sc->parity;
  const NodeSet in = pick(f, par), out = pick(f, par ^ 1);
  const double hourg = sc->hgcoef;
  const bool hg_on = hourg > 0.0;
  const double u_cut = sc->u_cut;
  const int last = (int)(gridDim.x * gridDim.y * gridDim.z) - 1;
  DtShared &dts = dt_shared();
  const bool fold = B.defer_dt && sc->dt_pending;
  int *const err = B.defer_dt ? &sc->err_nodal[par] : &sc->err;
  const DevScalars S = *sc;
  DtFold mine{1.0e+20, 1.0e+20};
  if (fold) {
    if (!loop_goes_on(sc, previous_err(sc, par))) {
      dt_fold_end(sc, last, dts.m, B);
      return;
    }
    mine = dt_fold_load(B);
  }

  // three node planes around k (those outside the domain repeat the edge)
  __shared__ double patch[3][6][PLANE_PATCH];
  // [corner mod 4][lane, slot BLOCK zero][stress xyz, hourglass xyz]
  __shared__ __align__(16) double lds[LDS_PAIR * 4];
  const int pw = etx + 1, np = pw * (ety + 1);
  const uint32_t us1 = (uint32_t)s1, node_plane = us1 * us1;
  double nv[2][6];
  int at_[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int m = t + j * BLOCK, pl = m / np, p = m % np;
    at_[j] = pl < 3 ? pl * 6 * PLANE_PATCH + p : -1;
    const int i = i0 - oi + p % pw, jj = j0 - oj + p / pw;
    const int kk = k - 1 + pl;
    const uint32_t o = ((uint32_t)(kk < 0 ? 0 : kk < s ? kk : s) * node_plane +
                        (uint32_t)(jj < s ? jj : s) * us1 + (uint32_t)(i < s ? i : s)) * 8u;
    nv[j][0] = at(in.x, o); nv[j][1] = at(in.y, o); nv[j][2] = at(in.z, o);
    nv[j][3] = at(in.xd, o); nv[j][4] = at(in.yd, o); nv[j][5] = at(in.zd, o);
  }
  const uint32_t eo = ((uint32_t)(ek < 0 ? 0 : ek < s ? ek : s - 1) * ((uint32_t)s * (uint32_t)s) +
                       (uint32_t)(ej < s ? ej : s - 1) * (uint32_t)s + (uint32_t)(ei < s ? ei : s - 1)) * 8u;
  const double vp = at(f.p, eo), vq = at(f.q, eo), vv = at(f.v, eo);
  const double vvolo = at(f.volo, eo), vss = at(f.ss, eo), vem = at(f.elemMass, eo);
  const uint32_t no = ((uint32_t)k * node_plane + (uint32_t)(nj < s1 ? nj : s) * us1 +
                       (uint32_t)(ni < s1 ? ni : s)) * 8u;
  const double mass = at(f.nodalMass, no);
  if (t < 24) lds[lds_at(t / 6, BLOCK) + t % 6] = 0.0;
  if (fold) dt_fold_wave(mine, dts.m);
#pragma unroll
  for (int j = 0; j < 2; ++j)
    if (at_[j] >= 0) {
      double *r = &patch[0][0][0] + at_[j];
#pragma unroll
      for (int c = 0; c < 6; ++c) r[c * PLANE_PATCH] = nv[j][c];
    }
  __syncthreads();
  if (B.defer_dt) {
    const DtNow w = dt_now_of(S, fold, dts.m);
    if (t == 0) dts.now = w;
  }

  if (elem) {
    const double(*rb)[PLANE_PATCH] = patch[upper], (*rt)[PLANE_PATCH] = patch[upper + 1];
    const int pe = tj * pw + ti;
    const int quirks = QK;
    double X[8], Y[8], Z[8];
    hex_patch(rb[0], rt[0], pe, pw, X);
    hex_patch(rb[1], rt[1], pe, pw, Y);
    hex_patch(rb[2], rt[2], pe, pw, Z);
    if (jacobian_volume64(X, Y, Z) <= 0.0) raise(err, ERR_EARLY_VOLUME);
    double2 *p[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) p[q] = (double2 *)(lds + lds_at(q, t));
    double z[4];
    {
      double N[8][3];
      node_normals16(X, Y, Z, quirks, N);
      const double ms = (-((-vp) - vq)) * 0.0625;
      // the corners on the node plane: the top ones of the element below,
      // the bottom ones of the element above
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double a = upper ? N[q][0] : N[q + 4][0], b = upper ? N[q][1] : N[q + 4][1];
        z[q] = ms * (upper ? N[q][2] : N[q + 4][2]);
        p[q][0] = make_double2(ms * a, ms * b);
      }
    }
    const double determ = vvolo * vv;
    if (vv <= 0.0) raise(err, ERR_HG_VOLUME);
    if (hg_on) {
      const double volume13 = cbrt_cr(determ);
      const double coefficient = ((((-hourg) * 0.01) * vss) * vem) / volume13;
      double g[8][4], h[4][3];
      hourglass_gh(X, Y, Z, rb, rt, pe, pw, quirks, 1.0 / determ, g, h);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        double gq[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) gq[m] = upper ? g[q][m] : g[q + 4][m];
        p[q][1] = make_double2(z[q], hourglass_force(gq, h, 0, coefficient));
        p[q][2] = make_double2(hourglass_force(gq, h, 1, coefficient),
                               hourglass_force(gq, h, 2, coefficient));
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        p[q][1] = make_double2(z[q], 0.0);
        p[q][2] = make_double2(0.0, 0.0);
      }
    }
  }
  __syncthreads();
  if (node) {
    // the element plane below, then the one above, each in (row, col) order
    const int l00 = (tj + oj - 1) * etx + (ti + oi - 1);
    double cs0 = 0.0, cs1 = 0.0, cs2 = 0.0, ch0 = 0.0, ch1 = 0.0, ch2 = 0.0;
    double2 v[8][3];
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      const int dj = (w >> 1) & 1, di = w & 1, up = w >> 2;
      const int x = ni - 1 + di, y = nj - 1 + dj, zk = k - 1 + up;
      const bool there = x >= 0 && x < s && y >= 0 && y < s && zk >= 0 && zk < s;
      const int q = dj ? (di ? 0 : 1) : (di ? 3 : 2);
      const double2 *r = (const double2 *)(lds + lds_at(q, there ? up * PLANE_LANES + l00 + dj * etx + di : BLOCK));
      v[w][0] = r[0]; v[w][1] = r[1]; v[w][2] = r[2];
    }
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      cs0 = cs0 + v[w][0].x; cs1 = cs1 + v[w][0].y; cs2 = cs2 + v[w][1].x;
      ch0 = ch0 + v[w][1].y; ch1 = ch1 + v[w][2].x; ch2 = ch2 + v[w][2].y;
    }
    if (hg_on) {
      cs0 = cs0 + ch0;
      cs1 = cs1 + ch1;
      cs2 = cs2 + ch2;
    }
    const int po = (tj + oj) * pw + ti + oi;
    node_update(out, f, no, ni, nj, k, cs0, cs1, cs2,
                NodeOld{mass, patch[1][0][po], patch[1][1][po], patch[1][2][po], patch[1][3][po],
                        patch[1][4][po], patch[1][5][po]},
                B.defer_dt ? dts.now.ts.deltatime : B.scheduled ? B.dt : S.deltatime, u_cut, B.keep_aux);
  }
  // as in k_nodal: the last workgroup to finish makes the set just written
  // current
  if (B.flip) {
    __syncthreads();
    if (t == 0) {
      if (atomicAdd(&sc->nodal_done, 1) == last) nodal_finish(B, sc, par, B.defer_dt ? &dts.now : nullptr);
    }
  }
}

// the node values of the element at (col, row, plane) of a domain of s
// elements per edge
struct ElemNodes {
  double X[8], Y[8], Z[8], XV[8], YV[8], ZV[8];
};
LDEV void load_nodes(const NodeSet &S, uint32_t col, uint32_t row, uint32_t plane, uint32_t s1, ElemNodes &n) {
  uint32_t nid[4];
  hex_pairs((plane * s1 + row) * s1 + col, s1, nid);
  gather8p(S.x, nid, n.X); gather8p(S.y, nid, n.Y); gather8p(S.z, nid, n.Z);
  gather8p(S.xd, nid, n.XV); gather8p(S.yd, nid, n.YV); gather8p(S.zd, nid, n.ZV);
}

// calcMonotonicQGradientsForElems (src/domain.jl:2175-2320) of one element
// along one axis (0 xi, 1 eta, 2 zeta): the side's length delx and the
// velocity gradient delv.
//
// Four times the reference's side differences d' = 4 d: powers of two
// factor out exactly, so an area vector is a' = 16 a, sqrt(a.a + ptiny) =
// sqrt(a'.a' + 256 ptiny) / 16, and a.dv norm = a'.dv' (norm / 64).
#define LULESH_SIDE(v, a, b, c, d, e, f, g, h) (sum4(v[a], v[b], v[c], v[d]) - sum4(v[e], v[f], v[g], v[h]))
#define LULESH_ETA(v) (-LULESH_SIDE(v, 0, 1, 5, 4, 3, 2, 6, 7))
#define LULESH_XI(v) LULESH_SIDE(v, 1, 2, 6, 5, 0, 3, 7, 4)
#define LULESH_ZETA(v) LULESH_SIDE(v, 4, 5, 6, 7, 0, 1, 2, 3)
template <int AXIS>
LDEV void monoq_gradient(const ElemNodes &n, double vol, double &delx, double &delv) {
  const double norm = 1.0 / (vol + 1.e-36);
  const double ptiny256 = 256.0 * 1.e-36, norm64 = norm * 0.015625, vol16 = vol * 16.0;
  // zeta: i cross j, xi: j cross k, eta: k cross i
  double u[3], w[3], dv[3];
  if constexpr (AXIS == 0) {
    u[0] = LULESH_ETA(n.X); u[1] = LULESH_ETA(n.Y); u[2] = LULESH_ETA(n.Z);
    w[0] = LULESH_ZETA(n.X); w[1] = LULESH_ZETA(n.Y); w[2] = LULESH_ZETA(n.Z);
    dv[0] = LULESH_XI(n.XV); dv[1] = LULESH_XI(n.YV); dv[2] = LULESH_XI(n.ZV);
  } else if constexpr (AXIS == 1) {
    u[0] = LULESH_ZETA(n.X); u[1] = LULESH_ZETA(n.Y); u[2] = LULESH_ZETA(n.Z);
    w[0] = LULESH_XI(n.X); w[1] = LULESH_XI(n.Y); w[2] = LULESH_XI(n.Z);
    dv[0] = LULESH_ETA(n.XV); dv[1] = LULESH_ETA(n.YV); dv[2] = LULESH_ETA(n.ZV);
  } else {
    u[0] = LULESH_XI(n.X); u[1] = LULESH_XI(n.Y); u[2] = LULESH_XI(n.Z);
    w[0] = LULESH_ETA(n.X); w[1] = LULESH_ETA(n.Y); w[2] = LULESH_ETA(n.Z);
    dv[0] = LULESH_ZETA(n.XV); dv[1] = LULESH_ZETA(n.YV); dv[2] = LULESH_ZETA(n.ZV);
  }
  const double ax = (u[1] * w[2]) - (u[2] * w[1]);
  const double ay = (u[2] * w[0]) - (u[0] * w[2]);
  const double az = (u[0] * w[1]) - (u[1] * w[0]);
  delx = vol16 / sqrt((((ax * ax) + (ay * ay)) + (az * az)) + ptiny256);
  delv = (((ax * norm64) * dv[0]) + ((ay * norm64) * dv[1])) + ((az * norm64) * dv[2]);
}
#undef LULESH_SIDE
#undef LULESH_ETA
#undef LULESH_XI
#undef LULESH_ZETA

// What calcKinematicsForElems (src/domain.jl:2099-2147) and the deviatoric
// loop (2156-2171) leave of one element, each value handed to
// put(field, value, index) where it is known; v_old() is the element's
// relative volume before the cycle.  Returns the one after it.
enum KinValue { KV_VDOV, KV_VNEW, KV_AREALG, KV_OTHER };
template <class Put, class VOld>
LDEV double kin_strain(const ElemNodes &n, const DevFields &f, DevScalars *sc, double volo, VOld v_old,
                       int keep_aux, Put put) {
  const double volume = elem_volume(n.X, n.Y, n.Z);
  const double vnew = volume / volo;
  if (vnew <= 0.0) raise(sc, ERR_KIN_VOLUME);
  put(f.vnew, vnew, KV_VNEW);
  put(f.delv, vnew - v_old(), KV_OTHER);
  put(f.arealg, char_length(n.X, n.Y, n.Z, volume), KV_AREALG);
  {
    const double dt2 = 0.5 * sc->deltatime;
    double XS[8], YS[8], ZS[8], b[4][3];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      XS[k] = n.X[k] - dt2 * n.XV[k];
      YS[k] = n.Y[k] - dt2 * n.YV[k];
      ZS[k] = n.Z[k] - dt2 * n.ZV[k];
    }
    // (64 x detJ and 64 x b: the factors cancel exactly)
    const double detJ = shape_derivatives4_64(XS, YS, ZS, b);
    const double inv_detJ = 1.0 / detJ;
    const double d1 = inv_detJ * vgrad_term(b, 0, n.XV);
    const double d2 = inv_detJ * vgrad_term(b, 1, n.YV);
    const double d3 = inv_detJ * vgrad_term(b, 2, n.ZV);
    const double vdov = (d1 + d2) + d3;
    put(f.vdov, vdov, KV_VDOV);
    if (keep_aux) {
      const double vdovthird = vdov / 3.0;
      put(f.dxx, d1 - vdovthird, KV_OTHER);
      put(f.dyy, d2 - vdovthird, KV_OTHER);
      put(f.dzz, d3 - vdovthird, KV_OTHER);
    }
    if (vnew <= 0.0) raise(sc, ERR_LAG_VOLUME);
  }
  return vnew;
}
// its side lengths and velocity gradients along all three axes, vol its volume
template <class Put>
LDEV void kin_gradients(const ElemNodes &n, const DevFields &f, double vol, Put put) {
  double delx, delv;
  monoq_gradient<2>(n, vol, delx, delv);
  put(f.delx_zeta, f.delv_zeta, delx, delv, 2);
  monoq_gradient<0>(n, vol, delx, delv);
  put(f.delx_xi, f.delv_xi, delx, delv, 0);
  monoq_gradient<1>(n, vol, delx, delv);
  put(f.delx_eta, f.delv_eta, delx, delv, 1);
}

// kin_strain and kin_gradients of every element.
//
// Bound by its memory pattern (the same 24 gathers, 2 reads and 10 writes
// alone take 240 us at s=192) and the vector instructions beside it.  Without
// the power-of-two scalings and the select chains of Julia's max: s=192 281
// -> 270 us, batch 209 -> 202, s=96 34.0 -> 32.0.  Fetching a 256-element
// chunk's node rows once into LDS instead (10 loads per thread and plane, one
// barrier) takes 320 us: the loads no longer run under other waves' work.
__global__ __launch_bounds__(KIN_CHUNK) void k_kin(Batch B) {
  // the chunk of one element plane this workgroup runs: kin_table bands
  // the planes so that an XCD's consecutive chunks climb one band of the
  // domain plane by plane and share node rows in its L2
  const KinWork w = B.kin_work[blockIdx.x];
  if (w.inst < 0) return;
  const InstDesc I = B.inst[w.inst];
  DevScalars *sc = B.sc + w.inst;
  if (B.gated && !sc->active) return;
  const int s = I.s;
  const uint32_t plane = (uint32_t)s * (uint32_t)s;
  const uint32_t plane_end = ((uint32_t)w.start / plane + 1u) * plane;
  const int64_t e = (int64_t)w.start + threadIdx.x;
  const DevFields f = slice(B.f, I);
  if (e >= (int64_t)plane_end) return;
  const int keep_aux = B.keep_aux;
  const uint32_t eo = (uint32_t)e * 8u;
  ElemNodes n;
  {
    const uint32_t ue = (uint32_t)e, us = (uint32_t)s, rest = ue / us;
    load_nodes(pick(f, sc->parity), ue % us, rest % us, rest / us, us + 1u, n);
  }
  const double volo = at(f.volo, eo);
  const double vnew = kin_strain(n, f, sc, volo, [&] { return at(f.v, eo); }, keep_aux,
                                 [&](double *p, double v, int) { st_nt(p, eo, v); });
  kin_gradients(n, f, volo * vnew, [&](double *px, double *pv, double delx, double delv, int) {
    st_nt(px, eo, delx);
    st_nt(pv, eo, delv);
  });
}

// Neighbour ids as setupElementConnectivities stores them
// (src/domain.jl:793-820), 0-based, its odd entries included; a read the
// reference would make out of bounds (only reachable with an uploaded elemBC
// that marks a boundary face interior, or s = 1) is clamped.
LDEV uint32_t nb_xim(uint32_t e, uint32_t E) { return e ? e - 1u : (E > 1u ? 1u : 0u); }
LDEV uint32_t nb_xip(uint32_t e, uint32_t E, bool q3) {
  const uint32_t nb = e < E - 1u ? e + 1u : E - 1u;
  return q3 ? (nb ? nb - 1u : 0u) : nb;
}
LDEV uint32_t nb_minus(uint32_t e, uint32_t step) { return e < step ? e : e - step; }  // eta, zeta
LDEV uint32_t nb_etap(uint32_t e, uint32_t s, uint32_t E) { return e < E - s ? e + s : e - (E - s); }
LDEV uint32_t nb_zetap(uint32_t e, uint32_t s2, uint32_t E) { return e < E - s2 ? e + s2 : e; }

// minimum of two values over a workgroup's first THREADS threads (64-wide
// wavefronts), in thread 0; every thread calls it
template <int THREADS = BLOCK>
LDEV void block_min2(double &a, double &b) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double oa = __shfl_xor(a, off, 64);
    const double ob = __shfl_xor(b, off, 64);
    a = oa < a ? oa : a;
    b = ob < b ? ob : b;
  }
  if constexpr (THREADS == 64) return;
  __shared__ double sa[THREADS / 64], sb[THREADS / 64];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (l == 0 && w < THREADS / 64) { sa[w] = a; sb[w] = b; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < THREADS / 64; ++i) {
      a = sa[i] < a ? sa[i] : a;
      b = sb[i] < b ? sb[i] : b;
    }
  }
}

// calcMonotonicQRegionForElems (src/domain.jl:2322-2513, quirk Q3), the
// QStop check (2567-2582), applyMaterialPropertiesForElems + evalEOSForElems
// + calcEnergyForElems + calcSoundSpeedForElems (2585-2910, one element at a
// time; the reference's element-wise temporaries never mix elements),
// updateVolumesForElems (2912-2930) and the per-element terms of
// calcCourantConstraintForElems / calcHydroConstraintForElems (2964-3054)
//
// own(field, index): the element's own value of a field; nb: the values of
// delv_xi, delv_eta and delv_zeta at its six neighbours (xi -, +, eta -, +,
// zeta -, +), whatever its boundary mask makes of them.
enum QeosValue { QV_VDOV, QV_VOLO, QV_VNEW, QV_DELX, QV_MASS = QV_DELX + 3, QV_V, QV_AREALG, QV_E, QV_P, QV_Q, QV_COUNT };
template <bool COST, class Own>
LDEV void qeos_element(const DevFields &f, const ElemState &out, DevScalars *sc, uint32_t eo, uint32_t bc, double dvxi, double dveta,
                       double dvzeta, const double (&nb)[6], Own own, int keep_aux, const int *elem_rep,
                       double &cand_c, double &cand_h) {
  const double ptiny = 1e-36;
  const double mult = sc->monoq_limiter_mult, maxslope = sc->monoq_max_slope;
  bool bad = false;
  // what a face's bits select: the neighbour (interior or COMM), the
  // element itself (SYMM), zero (FREE); anything else is the reference's
  // "Error" path
  auto side = [&](uint32_t mask, uint32_t symm, uint32_t free, uint32_t comm, double there, double self) {
    const uint32_t c = bc & mask;
    const bool read = c == 0 || c == comm;
    bad = bad || !(read || c == symm || c == free);
    return read ? there : c == symm ? self : 0.0;
  };
  const double phixi = limit_phi(side(XI_M, XI_M_SYMM, XI_M_FREE, XI_M_COMM, nb[0], dvxi),
                                 side(XI_P, XI_P_SYMM, XI_P_FREE, XI_P_COMM, nb[1], dvxi),
                                 1.0 / (dvxi + ptiny), mult, maxslope);
  const double phieta = limit_phi(side(ETA_M, ETA_M_SYMM, ETA_M_FREE, ETA_M_COMM, nb[2], dveta),
                                  side(ETA_P, ETA_P_SYMM, ETA_P_FREE, ETA_P_COMM, nb[3], dveta),
                                  1.0 / (dveta + ptiny), mult, maxslope);
  const double phizeta = limit_phi(side(ZETA_M, ZETA_M_SYMM, ZETA_M_FREE, ZETA_M_COMM, nb[4], dvzeta),
                                   side(ZETA_P, ZETA_P_SYMM, ZETA_P_FREE, ZETA_P_COMM, nb[5], dvzeta),
                                   1.0 / (dvzeta + ptiny), mult, maxslope);
  if (bad) raise(sc, ERR_BC);

  const double vdov = own(f.vdov, QV_VDOV), volo = own(f.volo, QV_VOLO), vnew = own(f.vnew, QV_VNEW);
  double qlin, qquad;
  if (vdov > 0.0) {
    qlin = 0.0;
    qquad = 0.0;
  } else {
    double delvxxi = dvxi * own(f.delx_xi, QV_DELX);
    double delvxeta = dveta * own(f.delx_eta, QV_DELX + 1);
    double delvxzeta = dvzeta * own(f.delx_zeta, QV_DELX + 2);
    if (delvxxi > 0.0) delvxxi = 0.0;
    if (delvxeta > 0.0) delvxeta = 0.0;
    if (delvxzeta > 0.0) delvxzeta = 0.0;
    const double rho = own(f.elemMass, QV_MASS) / (volo * vnew);
    qlin = ((-sc->qlc_monoq) * rho) *
           (((delvxxi * (1.0 - phixi)) + (delvxeta * (1.0 - phieta))) + (delvxzeta * (1.0 - phizeta)));
    qquad = (sc->qqc_monoq * rho) *
            ((((delvxxi * delvxxi) * (1.0 - (phixi * phixi))) +
              ((delvxeta * delvxeta) * (1.0 - (phieta * phieta)))) +
             ((delvxzeta * delvxzeta) * (1.0 - (phizeta * phizeta))));
  }
  if (keep_aux) {
    st_nt(f.qq, eo, qquad);
    st_nt(f.ql, eo, qlin);
  }

  // QStop on the q of the previous cycle
  double q_old = own(f.q, QV_Q);
  if (q_old > sc->qstop) raise(sc, ERR_QSTOP);

  // material properties
  const double eosvmin = sc->eosvmin, eosvmax = sc->eosvmax;
  const double v_old = own(f.v, QV_V);
  double vc = v_old;
  if (eosvmin != 0.0 && vc < eosvmin) vc = eosvmin;
  if (eosvmax != 0.0 && vc > eosvmax) vc = eosvmax;
  if (vc <= 0.0) raise(sc, ERR_EOS_VOLUME);
  double vnewc = vnew;
  if (eosvmin != 0.0 && vnewc < eosvmin) vnewc = eosvmin;
  if (eosvmax != 0.0 && vnewc > eosvmax) vnewc = eosvmax;

  // delv as k_kin formed it from the same two values: 8 of 172 bytes per
  // element less to read (s=192 200 -> 190 us, batch 162 -> 151)
  const double delvc_in = vnew - v_old, e_old_in = own(f.e, QV_E), p_old_in = own(f.p, QV_P);
  const double TINY1 = 0.111111e-36, TINY3 = 0.333333e-18, SIXTH = 1.0 / 6.0;
  const double pmin = sc->pmin, p_cut = sc->p_cut, e_cut = sc->e_cut, q_cut = sc->q_cut;
  const double emin = sc->emin, rho0 = sc->refdens;
  // LULESH-2.0 cost mode: the energy update of an element is evaluated as
  // many times as its region's regReps says (the same inputs each time, so
  // the same result); the empty asm statements make every evaluation real
  int rep = 1;
  if constexpr (COST) rep = *elem_rep;
  double p_new = 0.0, e_new = 0.0, q_new = 0.0, bvc = 0.0, pbvc = 0.0;
  for (int rr = 0; rr < rep; ++rr) {
  double delvc = delvc_in, e_old = e_old_in, p_old = p_old_in, q_o = q_old, vn = vnewc,
         ql_r = qlin, qq_r = qquad;
  if constexpr (COST) {
    __asm__ volatile("" : "+v"(delvc), "+v"(e_old), "+v"(p_old), "+v"(q_o));
    __asm__ volatile("" : "+v"(vn), "+v"(ql_r), "+v"(qq_r));
  }
  {
  const double q_old = q_o, vnewc = vn, qlin = ql_r, qquad = qq_r;
  double compression = 1.0 / vnewc - 1.0;
  const double vchalf = vnewc - delvc * 0.5;
  double compHalfStep = (1.0 / vchalf) - 1.0;
  if (eosvmin != 0.0 && vnewc <= eosvmin) compHalfStep = compression;
  if (eosvmax != 0.0 && vnewc >= eosvmax) {
    p_old = 0.0;
    compression = 0.0;
    compHalfStep = 0.0;
  }
  const double work = 0.0;
  e_new = (e_old - ((0.5 * delvc) * (p_old + q_old))) + (0.5 * work);
  if (e_new < emin) e_new = emin;
  const double pHalfStep = pressure(bvc, pbvc, e_new, compHalfStep, vnewc, pmin, p_cut, eosvmax);
  const double vhalf = 1.0 / (1.0 + compHalfStep);
  if (delvc > 0.0) {
    q_new = 0.0;
  } else {
    double ssc = ((pbvc * e_new) + (((vhalf * vhalf) * bvc) * pHalfStep)) / rho0;
    ssc = (ssc <= TINY1) ? TINY3 : sqrt(ssc);
    q_new = (ssc * qlin) + qquad;
  }
  e_new = e_new + ((0.5 * delvc) * ((3.0 * (p_old + q_old)) - (4.0 * (pHalfStep + q_new))));
  e_new = e_new + 0.5 * work;
  if (fabs(e_new) < e_cut) e_new = 0.0;
  if (e_new < emin) e_new = emin;
  p_new = pressure(bvc, pbvc, e_new, compression, vnewc, pmin, p_cut, eosvmax);
  double q_tilde;
  if (delvc > 0.0) {
    q_tilde = 0.0;
  } else {
    double ssc = ((pbvc * e_new) + (((vnewc * vnewc) * bvc) * p_new)) / rho0;
    ssc = (ssc <= TINY1) ? TINY3 : sqrt(ssc);
    q_tilde = (ssc * qlin) + qquad;
  }
  e_new = e_new - (((((7.0 * (p_old + q_old)) - (8.0 * (pHalfStep + q_new))) + (p_new + q_tilde)) *
                    delvc) *
                   SIXTH);
  if (fabs(e_new) < e_cut) e_new = 0.0;
  if (e_new < emin) e_new = emin;
  p_new = pressure(bvc, pbvc, e_new, compression, vnewc, pmin, p_cut, eosvmax);
  if (delvc <= 0.0) {
    double ssc = ((pbvc * e_new) + (((vnewc * vnewc) * bvc) * p_new)) / rho0;
    ssc = (ssc <= TINY1) ? TINY3 : sqrt(ssc);
    q_new = (ssc * qlin) + qquad;
    if (fabs(q_new) < q_cut) q_new = 0.0;
  }
  }
  if constexpr (COST) {
    __asm__ volatile("" ::"v"(p_new), "v"(e_new), "v"(q_new));
    __asm__ volatile("" ::"v"(bvc), "v"(pbvc));
  }
  }
  double ss = ((pbvc * e_new) + (((vnewc * vnewc) * bvc) * p_new)) / rho0;
  ss = (ss <= TINY1) ? TINY3 : sqrt(ss);
  st_nt(out.p, eo, p_new);
  st_nt(out.e, eo, e_new);
  st_nt(out.q, eo, q_new);
  st_nt(out.ss, eo, ss);

  // updateVolumesForElems
  double tmpV = vnew;
  if (fabs(tmpV - 1.0) < sc->v_cut) tmpV = 1.0;
  st_nt(out.v, eo, tmpV);
  if (tmpV <= 0.0) raise(sc, ERR_UPDATE_VOLUME);

  // time-constraint terms; an element only counts where vdov != 0 and its
  // value beats the 1e20 start value (strict <, as in the reference)
  if (vdov != 0.0) {
    const double qqc = sc->qqc;
    const double qqc2 = (64.0 * qqc) * qqc;
    const double arealg = own(f.arealg, QV_AREALG);
    double dtf = ss * ss;
    if (vdov < 0.0) dtf = dtf + ((((qqc2 * arealg) * arealg) * vdov) * vdov);
    dtf = sqrt(dtf);
    dtf = arealg / dtf;
    if (dtf < cand_c) cand_c = dtf;
    const double dtdvov = sc->dvovmax / (fabs(vdov) + 1.e-20);
    if (dtdvov < cand_h) cand_h = dtdvov;
  }
}

// EARLY: every value the element may need is read up front.  A small launch
// lasts as long as its chain of waits and is shorter that way (s=16 9.1 ->
// 8.7 us, s=48 10.8 -> 10.3); a large one streams, and the values held over
// the limiter cost it resident waves (s=96 30.9 -> 31.6, s=192 198 -> 203).
// The line lies at 1024 blocks: s=64 (1024) 14.3 -> 13.85, s=72 (1458) alike.
constexpr int QEOS_EARLY = 1024;
template <bool COST, bool EARLY>
__global__ __launch_bounds__(BLOCK) void k_qeos(Batch B) {
  LULESH_ELEM_PREAMBLE_T(B, qeos_order)
  if (B.gated && !sc->active) return;  // uniform over the block
  const int quirks = B.quirks;
  double *__restrict__ dtpart = B.dtpart;
  double cand_c = 1.0e+20, cand_h = 1.0e+20;
  if (e < E) {
    const uint32_t bc = ld_nt(&f.elemBC[e]);
    // The six neighbours' values are read before the boundary mask is known
    // (their ids are valid whatever it says), so nothing waits for it first:
    // s=16 9.6 -> 8.9 us a launch, s=48 11.3 -> 10.8, large domains alike.
    const uint32_t ue = (uint32_t)e, uE = (uint32_t)E, us = (uint32_t)s, s2 = us * us;
    const uint32_t eo = ue * 8u;
    const double dvxi = at(f.delv_xi, eo), dveta = at(f.delv_eta, eo), dvzeta = at(f.delv_zeta, eo);
    const double nb[6] = {
        at(f.delv_xi, nb_xim(ue, uE) * 8u),         at(f.delv_xi, nb_xip(ue, uE, quirks & Q3) * 8u),
        at(f.delv_eta, nb_minus(ue, us) * 8u),      at(f.delv_eta, nb_etap(ue, us, uE) * 8u),
        at(f.delv_zeta, nb_minus(ue, s2) * 8u),     at(f.delv_zeta, nb_zetap(ue, s2, uE) * 8u)};
    double early[QV_COUNT];
    if constexpr (EARLY) {
      const double *src[QV_COUNT] = {f.vdov, f.volo, f.vnew, f.delx_xi, f.delx_eta, f.delx_zeta,
                                     f.elemMass, f.v, f.arealg, f.e, f.p, f.q};
#pragma unroll
      for (int k = 0; k < QV_COUNT; ++k) early[k] = ld_nt(&src[k][e]);
    }
    auto own = [&](const double *p, int k) { return EARLY ? early[k] : ld_nt(&p[e]); };
    const int *rep = COST ? B.elem_rep + I.e0 + e : nullptr;
    qeos_element<COST>(f, slice(B.out, I), sc, eo, bc, dvxi, dveta, dvzeta, nb, own, B.keep_aux, rep, cand_c, cand_h);
  }
  block_min2(cand_c, cand_h);
  if (threadIdx.x == 0) {
    dtpart[2 * vb_] = cand_c;
    dtpart[2 * vb_ + 1] = cand_h;
  }
}

// k_kin and k_qeos of one small domain in one launch (elems_form): a
// workgroup runs its BX x BY x BZ block of elements and beside them the
// velocity gradient of the elements behind each face along that face's axis;
// after one barrier qeos_element finds its six neighbours in LDS.  Both
// kernels last there as long as their launches and waits, so the elements
// behind the faces, computed again by their own workgroups, cost nothing.
// SPLIT: an element's kin_strain and kin_gradients run on two threads, a
// third of the arithmetic off the longest chain; for launches that leave
// SIMDs idle.  A cycle of the device loop loses 2.9 us of 24 at s=16 (2.3
// unsplit), 3.1 of 27 at s=24, 1.4 of 30 at s=30; unsplit in blocks of 256
// 3.3 of 35 at s=34, 0.9 of 39 at s=40.
template <int BX, int BY, int BZ, bool SPLIT>
struct ElemBlock {
  static constexpr int CORE = BX * BY * BZ, FX = 2 * BY * BZ, FY = 2 * BX * BZ, FZ = 2 * BX * BY;
  static constexpr int OWN = (SPLIT ? 2 : 1) * CORE;  // threads on the block's own elements
  static constexpr int THREADS = (OWN + FX + FY + FZ + 63) / 64 * 64;
  static_assert(CORE % 64 == 0, "the block's own elements fill whole waves");
};
template <int BX, int BY, int BZ, bool SPLIT>
__global__ __launch_bounds__((ElemBlock<BX, BY, BZ, SPLIT>::THREADS)) void k_elems(Batch B) {
  using EB = ElemBlock<BX, BY, BZ, SPLIT>;
  __shared__ double lx[BZ][BY][BX + 2], ly[BZ][BY + 2][BX], lz[BZ + 2][BY][BX], ldelx[3][EB::CORE];
  DevScalars *sc = B.sc;
  if (B.gated && !sc->active) return;
  const DevFields &f = B.f;
  const int s = B.one.s, t = threadIdx.x;
  // which element this thread runs, and what of it
  enum { XI, ETA, ZETA, GRADIENTS, STRAIN, NONE };
  int i, j, k, what;
  if (t < EB::OWN) {
    const int h = t % EB::CORE;
    what = t < EB::CORE ? STRAIN : GRADIENTS;
    i = h % BX; j = h / BX % BY; k = h / (BX * BY);
  } else if (t < EB::OWN + EB::FZ) {
    const int h = t - EB::OWN;
    what = ZETA;
    i = h % BX; j = h / BX % BY; k = h < EB::FZ / 2 ? -1 : BZ;
  } else if (t < EB::OWN + EB::FZ + EB::FY) {
    const int h = t - (EB::OWN + EB::FZ);
    what = ETA;
    i = h % BX; k = h / BX % BZ; j = h < EB::FY / 2 ? -1 : BY;
  } else {
    const int h = t - (EB::OWN + EB::FZ + EB::FY);
    what = h < EB::FX ? XI : NONE;
    j = h % BY; k = h / BY % BZ; i = h < EB::FX / 2 ? -1 : BX;
  }
  const int col = (int)blockIdx.x * BX + i, row = (int)blockIdx.y * BY + j, plane = (int)blockIdx.z * BZ + k;
  const bool there = what != NONE && col >= 0 && col < s && row >= 0 && row < s && plane >= 0 && plane < s;
  const uint32_t us = (uint32_t)s, ue = ((uint32_t)plane * us + (uint32_t)row) * us + (uint32_t)col, eo = ue * 8u;
  const NodeSet S = pick(f, sc->parity);
  double own[QV_COUNT];
  uint32_t bc = 0;
  if (there) {
    ElemNodes n;
    load_nodes(S, (uint32_t)col, (uint32_t)row, (uint32_t)plane, us + 1u, n);
    const double volo = at(f.volo, eo);
    double vnew;
    if (what == STRAIN) {
      own[QV_V] = at(f.v, eo); own[QV_MASS] = at(f.elemMass, eo);
      own[QV_E] = at(f.e, eo); own[QV_P] = at(f.p, eo); own[QV_Q] = at(f.q, eo);
      bc = f.elemBC[ue];
      own[QV_VOLO] = volo;
      vnew = kin_strain(n, f, sc, volo, [&] { return own[QV_V]; }, B.keep_aux, [&](double *p, double v, int kv) {
        at(p, eo) = v;
        if (kv == KV_VDOV) own[QV_VDOV] = v;
        if (kv == KV_AREALG) own[QV_AREALG] = v;
      });
      own[QV_VNEW] = vnew;
    } else {
      vnew = elem_volume(n.X, n.Y, n.Z) / volo;
    }
    const double vol = volo * vnew;
    double delx, delv;
    if (what == GRADIENTS || (!SPLIT && what == STRAIN)) {
      kin_gradients(n, f, vol, [&](double *px, double *pv, double dx, double dv, int axis) {
        at(px, eo) = dx;
        at(pv, eo) = dv;
        ldelx[axis][t % EB::CORE] = dx;
        if (axis == 0) lx[k][j][i + 1] = dv;
        if (axis == 1) ly[k][j + 1][i] = dv;
        if (axis == 2) lz[k + 1][j][i] = dv;
      });
    } else if (what == ZETA) {
      monoq_gradient<2>(n, vol, delx, delv);
      lz[k + 1][j][i] = delv;
    } else if (what == ETA) {
      monoq_gradient<1>(n, vol, delx, delv);
      ly[k][j + 1][i] = delv;
    } else if (what == XI) {
      monoq_gradient<0>(n, vol, delx, delv);
      lx[k][j][i + 1] = delv;
    }
  }
  __syncthreads();
  double cand_c = 1.0e+20, cand_h = 1.0e+20;
  if (there && what == STRAIN) {
    const double dv[3] = {lx[k][j][i + 1], ly[k][j + 1][i], lz[k + 1][j][i]};
#pragma unroll
    for (int a = 0; a < 3; ++a) own[QV_DELX + a] = ldelx[a][t];
    // The neighbours the reference's lists name are those beside the element
    // except at the domain's faces and, with quirk Q3, along +xi; there it is
    // the element itself or one elsewhere (an uploaded mask that marks a
    // boundary face interior), whose gradient is then formed here.
    const uint32_t uE = us * us * us, s2 = us * us;
    const uint32_t id[6] = {nb_xim(ue, uE), nb_xip(ue, uE, B.quirks & Q3), nb_minus(ue, us),
                            nb_etap(ue, us, uE), nb_minus(ue, s2), nb_zetap(ue, s2, uE)};
    const bool beside[6] = {col > 0, col < s - 1 && !(B.quirks & Q3), row > 0, row < s - 1, plane > 0, plane < s - 1};
    constexpr uint32_t mask[6] = {XI_M, XI_P, ETA_M, ETA_P, ZETA_M, ZETA_P};
    constexpr uint32_t comm[6] = {XI_M_COMM, XI_P_COMM, ETA_M_COMM, ETA_P_COMM, ZETA_M_COMM, ZETA_P_COMM};
    double nb[6] = {lx[k][j][i], lx[k][j][i + 2], ly[k][j][i], ly[k][j + 2][i], lz[k][j][i], lz[k + 2][j][i]};
    uint32_t far = 0;
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      const uint32_t c = bc & mask[q];
      if (!beside[q]) {
        nb[q] = dv[q >> 1];
        if ((c == 0 || c == comm[q]) && id[q] != ue) far |= 1u << q;
      }
    }
    if (far) {
#pragma unroll 1
      for (int q = 0; q < 6; ++q) {
        if (!((far >> q) & 1u)) continue;
        uint32_t g = id[0];
#pragma unroll
        for (int r = 1; r < 6; ++r) g = q == r ? id[r] : g;
        ElemNodes n;
        load_nodes(S, g % us, g / us % us, g / s2, us + 1u, n);
        const double volo = at(f.volo, g * 8u), vol = volo * (elem_volume(n.X, n.Y, n.Z) / volo);
        double delx, d;
        if (q < 2) monoq_gradient<0>(n, vol, delx, d);
        else if (q < 4) monoq_gradient<1>(n, vol, delx, d);
        else monoq_gradient<2>(n, vol, delx, d);
#pragma unroll
        for (int r = 0; r < 6; ++r) nb[r] = q == r ? d : nb[r];
      }
    }
    qeos_element<false>(f, B.out, sc, eo, bc, dv[0], dv[1], dv[2], nb, [&](const double *, int v) { return own[v]; },
                        B.keep_aux, nullptr, cand_c, cand_h);
  }
  block_min2<EB::CORE>(cand_c, cand_h);
  if (t == 0) {
    const int g = ((int)blockIdx.z * gridDim.y + (int)blockIdx.y) * gridDim.x + (int)blockIdx.x;
    B.dtpart[2 * g] = cand_c;
    B.dtpart[2 * g + 1] = cand_h;
  }
}

// per-element time-constraint terms from the fields alone, for a
// calcTimeConstraintsForElems call that does not follow k_qeos
__global__ __launch_bounds__(BLOCK) void k_dtpart(Batch B) {
  LULESH_ELEM_PREAMBLE(B)
  (void)s;
  double *__restrict__ dtpart = B.dtpart;
  double cand_c = 1.0e+20, cand_h = 1.0e+20;
  if (e < E) {
    const double vdov = f.vdov[e];
    if (vdov != 0.0) {
      const double qqc2 = (64.0 * sc->qqc) * sc->qqc;
      const double arealg = f.arealg[e], ss = f.ss[e];
      double dtf = ss * ss;
      if (vdov < 0.0) dtf = dtf + ((((qqc2 * arealg) * arealg) * vdov) * vdov);
      dtf = sqrt(dtf);
      dtf = arealg / dtf;
      if (dtf < cand_c) cand_c = dtf;
      const double dtdvov = sc->dvovmax / (fabs(vdov) + 1.e-20);
      if (dtdvov < cand_h) cand_h = dtdvov;
    }
  }
  block_min2(cand_c, cand_h);
  if (threadIdx.x == 0) {
    dtpart[2 * blockIdx.x] = cand_c;
    dtpart[2 * blockIdx.x + 1] = cand_h;
  }
}

// final minima; in driver-loop mode (loop_mode 1) also the loop test of
// examples/benchmark.jl:82,95 and the timeIncrement! of the next cycle;
// with loop_mode 2 the next cycle's timeIncrement! unconditionally, its dt
// recorded as k_time_increment records it (a fixed number of cycles)
__global__ __launch_bounds__(1024) void k_dt(Batch B) {
  const InstDesc I = B.inst[blockIdx.x];
  DevScalars *sc = B.sc + blockIdx.x;
  if (B.gated && !sc->active) return;
  if (B.defer_dt && !sc->dt_pending) return;
  const int loop_mode = B.loop_mode;
  // (courant, hydro) pairs, 16-byte aligned; four independent loads in
  // flight per thread (a minimum does not depend on the order it is taken in)
  const double2 *__restrict__ dtpart = (const double2 *)(B.dtpart + 2 * (int64_t)I.eb0);
  const int64_t nb = B.n == 1 ? B.parts : I.ebn, bd = blockDim.x;
  double a = 1.0e+20, b = 1.0e+20, a1 = 1.0e+20, b1 = 1.0e+20;
  int64_t i = threadIdx.x;
  for (; i + 3 * bd < nb; i += 4 * bd) {
    const double2 p0 = dtpart[i], p1 = dtpart[i + bd], p2 = dtpart[i + 2 * bd],
                  p3 = dtpart[i + 3 * bd];
    a = p0.x < a ? p0.x : a;
    b = p0.y < b ? p0.y : b;
    a1 = p1.x < a1 ? p1.x : a1;
    b1 = p1.y < b1 ? p1.y : b1;
    a = p2.x < a ? p2.x : a;
    b = p2.y < b ? p2.y : b;
    a1 = p3.x < a1 ? p3.x : a1;
    b1 = p3.y < b1 ? p3.y : b1;
  }
  for (; i < nb; i += bd) {
    const double2 p0 = dtpart[i];
    a = p0.x < a ? p0.x : a;
    b = p0.y < b ? p0.y : b;
  }
  a = a1 < a ? a1 : a;
  b = b1 < b ? b1 : b;
  __shared__ double sa[16], sb[16];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double oa = __shfl_xor(a, off, 64);
    const double ob = __shfl_xor(b, off, 64);
    a = oa < a ? oa : a;
    b = ob < b ? ob : b;
  }
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (l == 0) { sa[w] = a; sb[w] = b; }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i) {
    a = sa[i] < a ? sa[i] : a;
    b = sb[i] < b ? sb[i] : b;
  }
  if (a < 1.0e+20) sc->dtcourant = a;
  if (b < 1.0e+20) sc->dthydro = b;
  if (loop_mode == 1) {
    if (B.defer_dt) gather_errs(sc);
    const bool go = loop_goes_on(sc, sc->err);
    sc->active = go;
    sc->dt_pending = 0;
    if (go) time_increment(sc);
  } else if (loop_mode == 2) {
    time_increment(sc);
    if (blockIdx.x == 0 && B.dt_record) B.dt_record[sc->cycle - 1 - B.dt_base] = sc->deltatime;
  }
}

__global__ void k_math(int op, const double *__restrict__ a, const double *__restrict__ b,
                       double *__restrict__ out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double x = a[i];
  out[i] = op == 0 ? cbrt_cr(x) : (op == 1 ? sqrt(x) : x / b[i]);
}

__global__ void k_clear_err(Batch B) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < B.n) B.sc[i].err = ERR_NONE;
}

}  // namespace lulesh

// ---------------------------------------------------------------------------
// launchers (called from the C ABI)
// ---------------------------------------------------------------------------
namespace lulesh {

static inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }
static inline unsigned per_inst_grid(int n) { return (unsigned)((n + 63) / 64); }

int nodal_blocks_per_cu() {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_nodal<3, NODAL_PATCH, false>, BLOCK, 0) != hipSuccess || n < 1)
    n = 1;
  return n;
}

hipError_t launch_init(hipStream_t st, const Batch &b) {
  hipLaunchKernelGGL(k_init_nodes, dim3(b.nblocks), dim3(BLOCK), 0, st, b);
  hipLaunchKernelGGL(k_init_elems, dim3(b.eblocks), dim3(BLOCK), 0, st, b);
  hipLaunchKernelGGL(k_init_mass, dim3(b.nblocks), dim3(BLOCK), 0, st, b);
  hipLaunchKernelGGL(k_init_scalars, dim3(per_inst_grid(b.n)), dim3(64), 0, st, b);
  return hipGetLastError();
}

hipError_t launch_math(hipStream_t st, int op, const double *a, const double *b, double *out,
                       int64_t n) {
  hipLaunchKernelGGL(k_math, dim3(nblk(n, BLOCK)), dim3(BLOCK), 0, st, op, a, b, out, n);
  return hipGetLastError();
}

template <bool DEFER>
static void launch_nodal(hipStream_t st, const Batch &b) {
  const dim3 g(b.glaunch), w(BLOCK);
  switch (b.quirks & (Q1 | Q2)) {
    case 0: hipLaunchKernelGGL((k_nodal<0, NODAL_PATCH, DEFER>), g, w, 0, st, b); break;
    case Q1: hipLaunchKernelGGL((k_nodal<Q1, NODAL_PATCH, DEFER>), g, w, 0, st, b); break;
    case Q2: hipLaunchKernelGGL((k_nodal<Q2, NODAL_PATCH, DEFER>), g, w, 0, st, b); break;
    default: hipLaunchKernelGGL((k_nodal<Q1 | Q2, NODAL_PATCH, DEFER>), g, w, 0, st, b); break;
  }
}

template <bool SPLIT, int BX, int BY, int BZ>
static void launch_elems(hipStream_t st, const Batch &b) {
  const int s = b.one.s;
  hipLaunchKernelGGL((k_elems<BX, BY, BZ, SPLIT>), dim3((s + BX - 1) / BX, (s + BY - 1) / BY, (s + BZ - 1) / BZ),
                     dim3(ElemBlock<BX, BY, BZ, SPLIT>::THREADS), 0, st, b);
}

hipError_t launch_kernel(int id, hipStream_t st, const Batch &b) {
  switch (id) {
    case KID_NODAL:
      // glaunch workgroups, dealt to blocks by the XCD-aware order table
      if (b.nodal_planes) {
        const dim3 g(b.ptile.tx, b.ptile.ty, b.one.s + 1);
        switch (b.quirks & (Q1 | Q2)) {
          case 0: hipLaunchKernelGGL(k_nodal_planes<0>, g, dim3(BLOCK), 0, st, b); break;
          case Q1: hipLaunchKernelGGL(k_nodal_planes<Q1>, g, dim3(BLOCK), 0, st, b); break;
          case Q2: hipLaunchKernelGGL(k_nodal_planes<Q2>, g, dim3(BLOCK), 0, st, b); break;
          default: hipLaunchKernelGGL((k_nodal_planes<Q1 | Q2>), g, dim3(BLOCK), 0, st, b); break;
        }
      } else if (b.nodal_wide) {
        hipLaunchKernelGGL((k_nodal<-1, NODAL_PATCH_WIDE, false>), dim3(b.glaunch), dim3(BLOCK), 0, st, b);
      } else if (b.defer_dt) {
        launch_nodal<true>(st, b);
      } else {
        launch_nodal<false>(st, b);
      }
      break;
    case KID_KIN:
      if (b.elems_form) break;  // part of KID_QEOS' launch
      hipLaunchKernelGGL(k_kin, dim3(b.kin_launch), dim3(KIN_CHUNK), 0, st, b);
      break;
    case KID_QEOS:
      if (b.elems_form == ELEMS_SMALL)
        launch_elems<true, ELEMS_SMALL_BLOCK>(st, b);
      else if (b.elems_form == ELEMS_MID)
        launch_elems<false, ELEMS_MID_BLOCK>(st, b);
      else if (b.cost_mode)
        hipLaunchKernelGGL((k_qeos<true, false>), dim3(b.qeos_launch), dim3(BLOCK), 0, st, b);
      else if (b.eblocks <= QEOS_EARLY)
        hipLaunchKernelGGL((k_qeos<false, true>), dim3(b.qeos_launch), dim3(BLOCK), 0, st, b);
      else
        hipLaunchKernelGGL((k_qeos<false, false>), dim3(b.qeos_launch), dim3(BLOCK), 0, st, b);
      break;
    case KID_DT:
      hipLaunchKernelGGL(k_dt, dim3(b.n), dim3(1024), 0, st, b);
      break;
    case KID_DTPART:
      hipLaunchKernelGGL(k_dtpart, dim3(b.eblocks), dim3(BLOCK), 0, st, b);
      break;
    case KID_TIME_INCREMENT:
      hipLaunchKernelGGL(k_time_increment, dim3(per_inst_grid(b.n)), dim3(64), 0, st, b);
      break;
    case KID_RUN_BEGIN:
      hipLaunchKernelGGL(k_run_begin, dim3(per_inst_grid(b.n)), dim3(64), 0, st, b);
      break;
    case KID_CLEAR_ERR:
      hipLaunchKernelGGL(k_clear_err, dim3(per_inst_grid(b.n)), dim3(64), 0, st, b);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace lulesh
