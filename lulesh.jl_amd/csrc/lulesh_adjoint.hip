// Adjoint kernels of one LULESH cycle on gfx950 (reverse of k_nodal ->
// k_kin -> k_qeos with the cycle's dt held fixed).
//
// The kernels read cycle c from where it ran (AdjArgs): its start state
// S_c = (x y z xd yd zd, e p q v ss), the node set after it (x', xd') and its
// temporaries (vnew delv vdov delx_* delv_*), all kept when the forward
// cycle ran.  On entry the adjoint buffers hold the adjoint of S_{c+1}; on
// exit that of S_c:
//   a_qeos  EOS + volume update + MonoQ region (limiter) adjoints
//   a_kin   MonoQ gradients + relative volume adjoints -> corners (x', xd')
//   a_node1 corner gather + node-update adjoint -> force adjoint per node
//   a_force stress + hourglass corner-force adjoints -> corners (x, xd)
//   a_node2 corner gather -> adjoint of the node state
// Gathers run over fixed lists, so the gradient is deterministic.
#include "lulesh_adj.h"
#include "lulesh_elem.h"
#include "lulesh_adjoint.h"

namespace lulesh {

using lulesh_adj::EosParams;
using lulesh_adj::EosOut;
using lulesh_adj::QIn;
using lulesh_adj::QOut;

namespace {

LDEV void elem_nodes_a(int64_t e, int s, int64_t (&nid)[8]) {
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

LDEV int64_t clampi(int64_t i, int64_t E) { return i < 0 ? 0 : (i >= E ? E - 1 : i); }

// element whose delv a (direction d, side sd) read of element i addresses,
// as k_qeos computes it (setupElementConnectivities ids, quirk Q3)
LDEV int64_t read_target(int d, int sd, int64_t i, int64_t s, int64_t E, bool q3) {
  const int64_t s2 = s * s;
  if (d == 0) {
    if (sd == 0) return clampi(i == 0 ? 1 : i - 1, E);
    const int64_t nb = i < E - 1 ? i + 1 : E - 1;
    return q3 ? clampi(nb - 1, E) : clampi(nb, E);
  }
  if (d == 1) {
    if (sd == 0) return clampi(i < s ? i : i - s, E);
    return clampi(i < E - s ? i + s : i - (E - s), E);
  }
  if (sd == 0) return clampi(i < s2 ? i : i - s2, E);
  return clampi(i < E - s2 ? i + s2 : i, E);
}

constexpr uint32_t MASK_M[3] = {XI_M, ETA_M, ZETA_M};
constexpr uint32_t MASK_P[3] = {XI_P, ETA_P, ZETA_P};
constexpr uint32_t SYMM_M[3] = {XI_M_SYMM, ETA_M_SYMM, ZETA_M_SYMM};
constexpr uint32_t SYMM_P[3] = {XI_P_SYMM, ETA_P_SYMM, ZETA_P_SYMM};
constexpr uint32_t COMM_M[3] = {XI_M_COMM, ETA_M_COMM, ZETA_M_COMM};
constexpr uint32_t COMM_P[3] = {XI_P_COMM, ETA_P_COMM, ZETA_P_COMM};

// 0 = neighbour read, 1 = self, 2 = zero (FREE or invalid)
LDEV int bc_source(uint32_t bc, int d, int sd) {
  const uint32_t c = bc & (sd == 0 ? MASK_M[d] : MASK_P[d]);
  if (c == 0 || c == (sd == 0 ? COMM_M[d] : COMM_P[d])) return 0;
  if (c == (sd == 0 ? SYMM_M[d] : SYMM_P[d])) return 1;
  return 2;
}

}  // namespace

// ---- reverse of k_qeos ------------------------------------------------------
__global__ __launch_bounds__(BLOCK) void a_qeos(AdjArgs A) {
  const int64_t e = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (e >= A.E) return;
  if (A.gated && A.sc->err != ERR_NONE) return;
  const DevScalars *sc = A.sc;
  const DevFields &f = A.f;
  const double *dvs[3] = {f.delv_xi, f.delv_eta, f.delv_zeta};
  const double *dxs[3] = {f.delx_xi, f.delx_eta, f.delx_zeta};
  const uint32_t bc = f.elemBC[e];
  QIn qi;
  int src[3][2];
  int64_t tgt[3][2];
  for (int d = 0; d < 3; ++d) {
    qi.dv[d] = dvs[d][e];
    qi.dx[d] = dxs[d][e];
    for (int sd = 0; sd < 2; ++sd) {
      src[d][sd] = bc_source(bc, d, sd);
      tgt[d][sd] = read_target(d, sd, e, A.s, A.E, A.q3);
      const double there = dvs[d][tgt[d][sd]];  // (read before the mask is known)
      const double val = src[d][sd] == 0 ? there : (src[d][sd] == 1 ? qi.dv[d] : 0.0);
      if (sd == 0) qi.dm[d] = val;
      else qi.dp[d] = val;
    }
  }
  qi.vdov = f.vdov[e];
  qi.elemMass = f.elemMass[e];
  qi.volo = f.volo[e];
  qi.vnew = f.vnew[e];
  qi.qlc = sc->qlc_monoq;
  qi.qqc = sc->qqc_monoq;
  qi.mult = sc->monoq_limiter_mult;
  qi.maxslope = sc->monoq_max_slope;
  // forward q terms (a zero adjoint gives just the forward values)
  double z3[3] = {0, 0, 0}, z3b[3] = {0, 0, 0}, z3c[3] = {0, 0, 0}, z3d[3] = {0, 0, 0};
  double zv = 0.0, zl = 0.0, zq = 0.0;
  const QOut q = lulesh_adj::monoq_region_rev(qi, 0.0, 0.0, z3, z3b, z3c, z3d, &zv, &zl, &zq);

  // EOS adjoint
  EosParams P;
  P.e_cut = sc->e_cut; P.p_cut = sc->p_cut; P.q_cut = sc->q_cut; P.eosvmax = sc->eosvmax;
  P.eosvmin = sc->eosvmin; P.pmin = sc->pmin; P.emin = sc->emin; P.rho0 = sc->refdens;
  const double vnew = qi.vnew;
  double vnewc = vnew, dclamp = 1.0;
  if (P.eosvmin != 0.0 && vnewc < P.eosvmin) { vnewc = P.eosvmin; dclamp = 0.0; }
  if (P.eosvmax != 0.0 && vnewc > P.eosvmax) { vnewc = P.eosvmax; dclamp = 0.0; }
  const double lo[4] = {A.lp[e], A.le[e], A.lq[e], A.lss[e]};
  double li[7] = {0, 0, 0, 0, 0, 0, 0};
  lulesh_adj::eos_rev(vnewc, f.delv[e], f.e[e], f.p[e], f.q[e], q.qlin, q.qquad, P, lo, li);
  double lvnew = li[0] * dclamp;
  // v' = vnew unless snapped to 1
  if (!(fabs(vnew - 1.0) < sc->v_cut)) lvnew += A.lv[e];

  // MonoQ region adjoint with the EOS's (lql, lqq)
  double ldv[3] = {0, 0, 0}, ldm[3] = {0, 0, 0}, ldp[3] = {0, 0, 0}, ldx[3] = {0, 0, 0};
  double lqlc = 0.0, lqqc = 0.0;
  lulesh_adj::monoq_region_rev(qi, li[5], li[6], ldv, ldm, ldp, ldx, &lvnew, &lqlc, &lqqc);
  for (int d = 0; d < 3; ++d) {
    double own = ldv[d];
    const double side[2] = {ldm[d], ldp[d]};
    for (int sd = 0; sd < 2; ++sd) {
      double out = 0.0;
      if (src[d][sd] == 0) {
        if (tgt[d][sd] == e) own += side[sd];
        else out = side[sd];
      } else if (src[d][sd] == 1) {
        own += side[sd];
      }
      A.nbr[(int64_t)(d * 2 + sd) * A.E + e] = out;
    }
    A.ldvs[(int64_t)d * A.E + e] = own;
    A.ldx[(int64_t)d * A.E + e] = ldx[d];
  }
  A.lvnew[e] = lvnew;
  // adjoint of S_c so far: e final; p, q from the EOS (stress adds later);
  // v through delv = vnew - v (hourglass adds later); ss only via hourglass
  A.le[e] = li[2];
  A.lp[e] = li[3];
  A.lq[e] = li[4];
  A.lv[e] = -li[1];
  A.lss[e] = 0.0;
  A.lvnew_delv[e] = li[1];
  if (!A.pacc_set) {
    lqlc = A.pacc[(int64_t)1 * A.E + e] + lqlc;
    lqqc = A.pacc[(int64_t)2 * A.E + e] + lqqc;
  }
  A.pacc[(int64_t)1 * A.E + e] = lqlc;
  A.pacc[(int64_t)2 * A.E + e] = lqqc;
}

// ---- reverse of k_kin (MonoQ gradients + relative volume) -------------------
__global__ __launch_bounds__(BLOCK) void a_kin(AdjArgs A) {
  const int64_t e = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (e >= A.E) return;
  if (A.gated && A.sc->err != ERR_NONE) return;
  const DevFields &f = A.f;
  const NodeSet S = A.cur;
  // Own delv adjoint plus what the elements that read this delv sent back:
  // by read_target, the next element's minus read (and element 0's, which
  // reads element 1), the last element's plus read under quirk Q3 or the
  // previous element's without it, and along eta and zeta the neighbour's
  // minus and plus reads (the last eta row's plus reads wrap to the first).
  // With a branch per candidate and 48 eight-byte node loads a launch took
  // 10.2 us at s=24 and 13.7 at s=48, now 7.1 and 12.4.
  const uint32_t ue = (uint32_t)e, us = (uint32_t)A.s, s2 = us * us, uE = (uint32_t)A.E;
  const uint32_t eo = ue * 8u;
  double l6[6];
  {
    auto sent = [&](int q, bool there, uint32_t i) {
      const double x = at(A.nbr + (int64_t)q * A.E, there ? i * 8u : 0u);
      return there ? x : 0.0;
    };
    const double own[3] = {at(A.ldvs, eo), at(A.ldvs + A.E, eo), at(A.ldvs + 2 * A.E, eo)};
    const double x0 = sent(0, ue == 1u, 0u), x1 = sent(0, ue + 1u < uE, ue + 1u);
    const double x2 = A.q3 ? sent(1, ue + 2u == uE, uE - 1u) : sent(1, ue >= 1u, ue - 1u);
    const double y0 = sent(2, ue + us < uE, ue + us);
    const bool wraps = ue < us && uE > us;
    const double y1 = sent(3, ue >= us || wraps, ue >= us ? ue - us : ue + (uE - us));
    const double z0 = sent(4, ue + s2 < uE, ue + s2), z1 = sent(5, ue >= s2, ue - s2);
    l6[0] = at(A.ldx, eo); l6[1] = at(A.ldx + A.E, eo); l6[2] = at(A.ldx + 2 * A.E, eo);
    l6[3] = ((own[0] + x0) + x1) + x2;
    l6[4] = (own[1] + y0) + y1;
    l6[5] = (own[2] + z0) + z1;
  }
  double X[8], Y[8], Z[8], VX[8], VY[8], VZ[8];
  {
    const uint32_t s1 = us + 1u, col = ue % us, rest = ue / us;
    uint32_t nid[4];
    hex_pairs(((rest / us) * s1 + rest % us) * s1 + col, s1, nid);
    gather8p(S.x, nid, X); gather8p(S.y, nid, Y); gather8p(S.z, nid, Z);
    gather8p(S.xd, nid, VX); gather8p(S.yd, nid, VY); gather8p(S.zd, nid, VZ);
  }
  double lX[8] = {0}, lY[8] = {0}, lZ[8] = {0}, lVX[8] = {0}, lVY[8] = {0}, lVZ[8] = {0};
  const double volo = at(f.volo, eo);
  double lvnew = at(A.lvnew, eo) + at(A.lvnew_delv, eo);  // delv = vnew - v
  lvnew += lulesh_adj::monoq_grad_rev(X, Y, Z, VX, VY, VZ, volo, at(f.vnew, eo), l6, lX, lY, lZ, lVX,
                                      lVY, lVZ);
  lulesh_adj::volume_grad_rev(X, Y, Z, lvnew / volo, lX, lY, lZ);
  double *cr = A.corner;
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    at(cr + (int64_t)(0 * 8 + n) * A.E, eo) = lX[n];
    at(cr + (int64_t)(1 * 8 + n) * A.E, eo) = lY[n];
    at(cr + (int64_t)(2 * 8 + n) * A.E, eo) = lZ[n];
    at(cr + (int64_t)(3 * 8 + n) * A.E, eo) = lVX[n];
    at(cr + (int64_t)(4 * 8 + n) * A.E, eo) = lVY[n];
    at(cr + (int64_t)(5 * 8 + n) * A.E, eo) = lVZ[n];
  }
}

// corner of element (ei,ej,ek) that node (i,j,k) occupies
LDEV int corner_of_a(int ox, int oy, int oz) { return 4 * oz + (oy ? (ox ? 2 : 3) : (ox ? 1 : 0)); }

// The eight elements around node (i, j, k), in ascending order: byte offset
// of each in an element array and whether it exists (a missing one reads
// element 0 and adds zero).
struct NodeElems {
  uint32_t off[8];
  bool has[8];
  LDEV NodeElems(int i, int j, int k, int s) {
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      const int ei = i - 1 + (w & 1), ej = j - 1 + ((w >> 1) & 1), ek = k - 1 + (w >> 2);
      has[w] = ei >= 0 && ei < s && ej >= 0 && ej < s && ek >= 0 && ek < s;
      off[w] = has[w] ? (((uint32_t)ek * (uint32_t)s + (uint32_t)ej) * (uint32_t)s + (uint32_t)ei) * 8u : 0u;
    }
  }
};
// Sum over a node's corners of comp c (0..5) of a corner buffer.  The reads
// are unconditional, sixteen in flight together: with a branch per element
// a_node1 waited for sixteen groups of six one after the other, 8.0 us a
// launch at s=24 against 5.9 now.  From s=48 on (18.7 us) what bounds it is
// the 96 values per element it reads back, at 5 TB/s.
LDEV void gather_corners(const AdjArgs &A, const double *corner, const NodeElems &ne, double out[6]) {
#pragma unroll 2
  for (int c = 0; c < 6; ++c) {
    const double *p = corner + (int64_t)(c * 8) * A.E;
    double v[8];
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      const int cn = corner_of_a(1 - (w & 1), 1 - ((w >> 1) & 1), 1 - (w >> 2));
      v[w] = at(p + (int64_t)cn * A.E, ne.off[w]);
    }
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < 8; ++w) sum += ne.has[w] ? v[w] : 0.0;
    out[c] = sum;
  }
}

// ---- reverse of the node update (calcAcceleration .. calcPosition) ----------
__global__ __launch_bounds__(BLOCK) void a_node1(AdjArgs A) {
  const int64_t n = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (n >= A.N) return;
  if (A.gated && A.sc->err != ERR_NONE) return;
  const int s1 = A.s + 1, un = (int)n;
  const int i = un % s1, j = (un / s1) % s1, k = un / (s1 * s1);
  const NodeElems ne(i, j, k, A.s);
  double g[6];
  if (A.force_pending) {
    // what a_node2 of the later cycle would add: corner_f into the node state
    gather_corners(A, A.corner_f, ne, g);
    A.lx[n] += g[0]; A.ly[n] += g[1]; A.lz[n] += g[2];
    A.lxd[n] += g[3]; A.lyd[n] += g[4]; A.lzd[n] += g[5];
  }
  gather_corners(A, A.corner, ne, g);
  const double dt = A.dt;
  const double mass = A.f.nodalMass[n];
  double *lxs[3] = {A.lx, A.ly, A.lz};
  double *lvs[3] = {A.lxd, A.lyd, A.lzd};
  const double *vnew[3] = {A.cur.xd, A.cur.yd, A.cur.zd};
  const bool bcz[3] = {i == 0, j == 0, k == 0};
  for (int c = 0; c < 3; ++c) {
    const double lxn = lxs[c][n] + g[c];        // adjoint of x'
    double lvn = lvs[c][n] + g[3 + c];          // adjoint of xd'
    lvn += lxn * dt;                             // x' = x + xd' dt
    double lv_old = 0.0, lF = 0.0;
    if (vnew[c][n] != 0.0) {                     // not cut by u_cut
      lv_old = lvn;
      if (!bcz[c]) lF = lvn * dt / mass;          // xd' = xd + (F/m) dt
    }
    lxs[c][n] = lxn;
    lvs[c][n] = lv_old;
    A.lF[(int64_t)c * A.N + n] = lF;
  }
}

// ---- reverse of the corner forces (stress + FB hourglass) -------------------
// velocities of S_c and force adjoints read from memory node by node, so
// they do not occupy registers across the whole element
// The element's node values are addressed by 32-bit byte offsets from
// uniform array bases (the host keeps 8 N and 8 E below 2^32), so each
// node costs one offset register shared by every array read there instead
// of a 64-bit address per array.
LDEV const double &at_off(const double *base, uint32_t off) {
  return *(const double *)((const char *)base + off);
}
struct NodeSrc {
  const double *vx, *vy, *vz, *lF;
  int64_t N;
  uint32_t off[8];  // byte offsets of the element's nodes
  LDEV double v(int c, int n) const { return at_off(c == 0 ? vx : (c == 1 ? vy : vz), off[n]); }
  LDEV double lf(int n, int c) const { return at_off(lF + (int64_t)c * N, off[n]); }
};
// per-corner adjoints straight to the corner buffer ([6][8][E])
struct CornerSink {
  double *cr;
  int64_t E;
  uint32_t off;  // byte offset of the element
  LDEV void put(int k, int n, double x) {
    *(double *)((char *)(cr + (int64_t)(k * 8 + n) * E) + off) = x;
  }
  LDEV void lv(int c, int n, double x) { put(3 + c, n, x); }
};
// One coordinate axis of the element's eight nodes, parked in LDS (stride
// BLOCK, so a wave's reads are conflict-free) and re-read at every use: a
// volatile LDS read cannot be merged with an earlier one, so the 24
// coordinates hold no registers between uses.  That, with the 32-bit node
// offsets, keeps a_force within 256 VGPRs: two waves per SIMD instead of one.
struct LdsAxis {
  const double *p;
  __device__ double operator[](int n) const {
    typedef __attribute__((address_space(3))) const volatile double lds_double;
    return *(lds_double *)(p + n * BLOCK);
  }
};

template <bool Q1, bool Q2>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(2))) void a_force(AdjArgs A) {
  const int64_t e = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (e >= A.E) return;
  if (A.gated && A.sc->err != ERR_NONE) return;
  const DevFields &f = A.f;
  const NodeSet S = A.old;
  int64_t nid[8];
  elem_nodes_a(e, A.s, nid);
  NodeSrc src{S.xd, S.yd, S.zd, A.lF, A.N, {}};
  for (int n = 0; n < 8; ++n) src.off[n] = (uint32_t)nid[n] * 8u;
  __shared__ double pos[3][8][BLOCK];
  for (int n = 0; n < 8; ++n) {
    pos[0][n][threadIdx.x] = S.x[nid[n]];
    pos[1][n][threadIdx.x] = S.y[nid[n]];
    pos[2][n][threadIdx.x] = S.z[nid[n]];
  }
  const LdsAxis X{&pos[0][0][threadIdx.x]}, Y{&pos[1][0][threadIdx.x]}, Z{&pos[2][0][threadIdx.x]};
  CornerSink sink{A.corner_f, A.E, (uint32_t)e * 8u};
  double lX[8] = {0}, lY[8] = {0}, lZ[8] = {0};
  const double hourg = A.sc->hgcoef;
  if (hourg > 0.0) {
    const double volo = f.volo[e];
    const double determ = volo * f.v[e];
    const double ss = f.ss[e], mass = f.elemMass[e], c13 = cbrt_cr(determ);
    const lulesh_adj::HgRev r = lulesh_adj::hourglass_rev_s<Q2>(X, Y, Z, src, sink, determ, ss,
                                                                mass, hourg, c13, lX, lY, lZ);
    A.lv[e] += r.ldeterm * volo;
    A.lss[e] += r.lss;
    A.pacc[e] = A.pacc_set ? r.lhgcoef : A.pacc[e] + r.lhgcoef;
  } else {
    if (A.pacc_set) A.pacc[e] = 0.0;
    for (int c = 0; c < 3; ++c)
      for (int n = 0; n < 8; ++n) sink.lv(c, n, 0.0);
  }
  const double ms = f.p[e] + f.q[e];
  const double lms = lulesh_adj::stress_rev_s(X, Y, Z, Q1, ms, src, lX, lY, lZ);
  A.lp[e] += lms;
  A.lq[e] += lms;
  for (int n = 0; n < 8; ++n) {
    sink.put(0, n, lX[n]);
    sink.put(1, n, lY[n]);
    sink.put(2, n, lZ[n]);
  }
}

__global__ __launch_bounds__(BLOCK) void a_node2(AdjArgs A) {
  const int64_t n = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (n >= A.N) return;
  if (A.gated && A.sc->err != ERR_NONE) return;
  const int s1 = A.s + 1, un = (int)n;
  const NodeElems ne(un % s1, (un / s1) % s1, un / (s1 * s1), A.s);
  double g[6];
  gather_corners(A, A.corner_f, ne, g);
  A.lx[n] += g[0];
  A.ly[n] += g[1];
  A.lz[n] += g[2];
  A.lxd[n] += g[3];
  A.lyd[n] += g[4];
  A.lzd[n] += g[5];
}

// loss seed: dL/de = elemMass (L = sum e * elemMass), everything else 0
__global__ __launch_bounds__(BLOCK) void a_seed(AdjArgs A) {
  const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (i < A.E) {
    A.le[i] = A.f.elemMass[i];
    A.lp[i] = 0.0; A.lq[i] = 0.0; A.lv[i] = 0.0; A.lss[i] = 0.0;
    A.pacc[i] = 0.0; A.pacc[A.E + i] = 0.0; A.pacc[2 * A.E + i] = 0.0;
  }
  if (i < A.N) {
    A.lx[i] = 0.0; A.ly[i] = 0.0; A.lz[i] = 0.0;
    A.lxd[i] = 0.0; A.lyd[i] = 0.0; A.lzd[i] = 0.0;
  }
}

// copy the cycle state (current node set + e p q v ss) to/from a buffer
// laid out as [x y z xd yd zd][N] then [e p q v ss][E]
__global__ __launch_bounds__(BLOCK) void a_state_copy(DevScalars *sc, DevFields f, int64_t E,
                                                      int64_t N, double *buf, int to_buf) {
  const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
  const int par = sc->parity;
  double *nd[6] = {par ? f.ns[1].x : f.ns[0].x, par ? f.ns[1].y : f.ns[0].y,
                   par ? f.ns[1].z : f.ns[0].z, par ? f.ns[1].xd : f.ns[0].xd,
                   par ? f.ns[1].yd : f.ns[0].yd, par ? f.ns[1].zd : f.ns[0].zd};
  double *el[5] = {f.e, f.p, f.q, f.v, f.ss};
  if (i < N)
    for (int k = 0; k < 6; ++k) {
      if (to_buf) buf[k * N + i] = nd[k][i];
      else nd[k][i] = buf[k * N + i];
    }
  if (i < E)
    for (int k = 0; k < 5; ++k) {
      if (to_buf) buf[6 * N + k * E + i] = el[k][i];
      else el[k][i] = buf[6 * N + k * E + i];
    }
}

static inline unsigned nblk_a(int64_t n) { return (unsigned)((n + BLOCK - 1) / BLOCK); }

hipError_t launch_adjoint(int which, hipStream_t st, const AdjArgs &a) {
  switch (which) {
    case AK_QEOS:
      hipLaunchKernelGGL(a_qeos, dim3(nblk_a(a.E)), dim3(BLOCK), 0, st, a);
      break;
    case AK_KIN:
      hipLaunchKernelGGL(a_kin, dim3(nblk_a(a.E)), dim3(BLOCK), 0, st, a);
      break;
    case AK_NODE1:
      hipLaunchKernelGGL(a_node1, dim3(nblk_a(a.N)), dim3(BLOCK), 0, st, a);
      break;
    case AK_FORCE:
      if (a.q1 && a.q2)
        hipLaunchKernelGGL((a_force<true, true>), dim3(nblk_a(a.E)), dim3(BLOCK), 0, st, a);
      else if (a.q1)
        hipLaunchKernelGGL((a_force<true, false>), dim3(nblk_a(a.E)), dim3(BLOCK), 0, st, a);
      else if (a.q2)
        hipLaunchKernelGGL((a_force<false, true>), dim3(nblk_a(a.E)), dim3(BLOCK), 0, st, a);
      else
        hipLaunchKernelGGL((a_force<false, false>), dim3(nblk_a(a.E)), dim3(BLOCK), 0, st, a);
      break;
    case AK_NODE2:
      hipLaunchKernelGGL(a_node2, dim3(nblk_a(a.N)), dim3(BLOCK), 0, st, a);
      break;
    case AK_SEED:
      hipLaunchKernelGGL(a_seed, dim3(nblk_a(a.N > a.E ? a.N : a.E)), dim3(BLOCK), 0, st, a);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_state_copy(hipStream_t st, DevScalars *sc, const DevFields &f, int64_t E,
                             int64_t N, double *buf, int to_buf) {
  hipLaunchKernelGGL(a_state_copy, dim3(nblk_a(N > E ? N : E)), dim3(BLOCK), 0, st, sc, f, E, N,
                     buf, to_buf);
  return hipGetLastError();
}

}  // namespace lulesh
