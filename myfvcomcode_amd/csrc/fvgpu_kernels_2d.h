// fvgpu_kernels_2d.h -- the barotropic (external) mode on the device.
//
// One Runge-Kutta stage of EXTERNAL_STEP (FVCOM_source/external_step.F:159-438)
// is one kernel over compact element tiles, k_ext_stage: EXTEL_EDGE
// (extel_edge.F:32-229) as a gather of each node's control-volume sub-edge
// terms (formed per sub-edge by the previous stage, or by k_ext_begin), the
// open-boundary conditions and RK blend (BCOND_GCN(1,K), bcond_gcn.F:116;
// mod_obcs.F:509-737), FLUX_OBN (mod_obcs.F:1181-1215), D = H + EL,
// DEPTH_CHECK, N2E2D, the ADVAVE_EDGE_GCN edge terms
// (advave_edge_gcn.F:546-884), EXTUV_EDGE (extuv_edge.F:33-196), the wall
// projection BCOND_GCN(2,K) (bcond_gcn.F:325-420), D1 = H1 + EL1, the
// stage-3 EGF / UARD / VARD and stage-4 UARD_OBCN accumulations, and the
// EXTEL terms of the next stage.
// The per-node and per-element gather lists are sorted by sub-edge / edge
// index, so every sum is formed in the order of the reference's scatter loop.
#pragma once
#include "fvgpu_common.h"
#include "../../include/fv_detmath.h"

struct Ext2DState {      // one buffer set of the 2-D state
  double *el, *d;        // nodes
  double *ua, *va, *el1, *d1;  // elements
};

// RAMP and ExtTime of one external step (k_int_clock).
struct ExtClock { double ramp, time; };

struct ExtArgs {
  Ext2DState cur;        // stage input
  Ext2DState base;       // RK base (UARK, VARK, ELRK1)
  Ext2DState nxt;        // stage output (may alias base: pointwise use only)
  int K;                 // RK stage 1..4
  double alpha;          // ALPHA_RK(K)
  const double* elrk;    // RK base elevation: the base's own array in stage 1, its copy afterwards
  double* elrk_copy;     // stage 1 fills the copy, else null
  double *uard_obcn, *egf, *fluxobn, *uard, *vard;
  double *adx2d, *ady2d; // written by the INT form only
  const double *drx2d, *dry2d, *wubot, *wvbot;
  // the six constants of the external steps in block order: ADX2D, ADY2D,
  // DRX2D, DRY2D, WUBOT, WVBOT of element t at (6*b + q)*FV_CVB + t
  // (written by the INT form)
  double* own2d;
  const double *qdis;    // QDIS (internal-mode river discharge)
  const double* phi;     // per sub-edge EXTEL terms of the stage input
  double* phi_next;      // those of the stage output
  const double *ws2x, *ws2y;   // wind stress of the external step (before RAMP*0.001)
  double *elm1, *elm2;         // the elevation one and two RK stages back (Orlanski OBC)
  const ExtClock* ec;    // of this external step
  DevClock* clk;
  StageTab st;
};

// PSIMPLE_DRAG (mod_bulk.F:58-90): wind stress of a wind speed (Large and
// Pond drag coefficient, 1.2 kg/m^3 air), on the host and the device.
__host__ __device__ __forceinline__ void psimple_drag(double tx, double ty, double& sx, double& sy) {
  const double wds = sqrt(tx * tx + ty * ty);
  double cd = (double)1.2E-3f;
  if (wds >= 11.0) cd = (0.49 + 0.065 * wds) * 1.E-3;
  if (wds >= 25.0) cd = (0.49 + 0.065 * 25.0) * 1.E-3;
  sx = 1.2 * cd * tx * wds;
  sy = 1.2 * cd * ty * wds;
}

// BCOND_GCN(9) wind of EXTERNAL_STEP iext (bcond_gcn.F:878-895): the speed
// interpolated linearly in time between the internal step's start (u0, v0)
// and end (u1, v1) to ExtTime, fraction iext/ISPLIT, then its stress.
__global__ void k_ext_wind(DevGrid g, const double* u0, const double* v0, const double* u1, const double* v1,
                           int iext, double* sx, double* sy) {
  const int i = (int)xcd_thread() + 1;
  if (i > g.N) return;
  const double frac = (double)iext / (double)g.isplit;
  const double uu = u0[i] + frac * (u1[i] - u0[i]);
  const double vv = v0[i] + frac * (v1[i] - v0[i]);
  psimple_drag(uu, vv, sx[i], sy[i]);
}

// New end-of-step wind speeds (nu, nv) at elements 0..n1-1: the previous ones
// become the start of the step; the stress of the new ones at elements 1...
__global__ void k_wind_shift(long n1, double* u0, double* v0, double* u1, double* v1, const double* nu,
                             const double* nv, double* sx, double* sy) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n1) return;
  u0[i] = u1[i];
  v0[i] = v1[i];
  u1[i] = nu[i];
  v1[i] = nv[i];
  sx[i] = 0.0;
  sy[i] = 0.0;
  if (i >= 1) psimple_drag(nu[i], nv[i], sx[i], sy[i]);
}

// Wall projection of a velocity pair (BCOND_GCN cases 2/3/5): the element's
// case, found once (wall_prep), then applied to any number of pairs of its
// column (wall_apply).  Case 3 zeroes the pair; on a solid wall (ISBCE 1)
// an element that is the first or last of a river node's NBVE ring keeps
// only the inflowing part along the river, any other the component along
// the wall.
struct WallOp {
  int kind;   // 0: unchanged, 1: river (p, q = COS, SIN of its angle), 2: wall (p, q = SIN, COS of ALPHA), 3: zero
  double p, q;
};

__device__ __forceinline__ WallOp wall_prep(const DevGrid& g, int i) {
  const int b = g.isbce[i];
  if (b == 3) return {3, 0.0, 0.0};
  if (b != 1) return {0, 0.0, 0.0};
  // the first river (in river order) whose mouth is this cell: the first
  // and last cells around a node river's node, an edge river's own cell
  if (g.re_off[i] < g.re_off[i + 1]) {
    const int j = g.re_riv[g.re_off[i]];
    return {1, g.cos_angleq[j], g.sin_angleq[j]};
  }
  return {2, g.sin_alpha[i], g.cos_alpha[i]};
}

__device__ __forceinline__ void wall_apply(const WallOp& w, double& u, double& v) {
  if (w.kind == 3) {
    u = 0.0;
    v = 0.0;
  } else if (w.kind == 1) {
    const double ca = w.p, sa = w.q;
    double untmp = u * ca + v * sa;
    const double vntmp = -u * sa + v * ca;
    untmp = fmax(untmp, 0.0);
    u = untmp * ca - vntmp * sa;
    v = untmp * sa + vntmp * ca;
  } else if (w.kind == 2) {
    const double s = w.p, c = w.q;
    const double ui = u * (s * s) - v * s * c;
    const double vi = -u * s * c + v * (c * c);
    u = ui;
    v = vi;
  }
}

__device__ __forceinline__ void wall_project(const DevGrid& g, int i, double& u, double& v) {
  wall_apply(wall_prep(g, i), u, v);
}

// Spectral tide at OBC node index `obc` (BCOND_ASL, mod_obcs.F:552-582).
__device__ __forceinline__ double tide_force(const DevGrid& g, int obc, double rk_time, double ramp) {
  const double PI2 = 6.283185307179586;
  double force = 0.0;
  for (int j = 0; j < g.NTIDE; ++j) {
    const double phai_ij = g.phai[(long)j * g.IOBCN + obc] * PI2 / 360.0;
    const double time_flt = rk_time * PI2 / g.period[j];
    force = g.apt[(long)j * g.IOBCN + obc] * fv_cos(time_flt - phai_ij) + force;
  }
  force = force + g.emean[obc];
  return force * ramp;
}

// The new elevation of node i before its open-boundary condition:
// EXTEL_EDGE's sum over the node's sub-edges in sub-edge order, its rivers
// (rv: the first, or -1) and the RK update; at an OBC node `xobc` is the sum
// itself (extel_edge.F:155-160).  The term of sub-edge c, D1*(-UA*DLTYE +
// VA*DLTXE) of its element for side IB, is exactly the negative for side IA
// (DLTXE/DLTYE negated; round to nearest is symmetric), so the stored term
// is added or subtracted.  ce: the node's list entries; the slots past them
// hold the unused entry 0, whose term is zero and leaves the sum as it is
// (x - 0 is x), so all term loads are unconditional and issue together.
template <int SMAX>
__device__ __forceinline__ double ext_node_update(const DevGrid& g, const ExtArgs& a, int i, const int (&ce)[SMAX],
                                                  int rv, bool obc, double art1, double elrk, double& xobc) {
  double t[SMAX];
  static_for<SMAX>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    t[j] = at(a.phi, ce[j] >> 1);
  });
  double xflux = 0.0;
  static_for<SMAX>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    xflux = xflux + flip_sign(t[j], ~ce[j]);
  });
  xobc = 0.0;
  if (obc) { xobc = xflux; xflux = 0.0; }
  if (rv >= 0) {
    for (int j = rv; j < g.NUMQBC; ++j) {
      double w;
      if (river_share(g, j, i, w)) xflux = xflux - a.qdis[j] * w;
    }
  }
  const double dtk = a.alpha * g.dte;
  return elrk - dtk * xflux / art1;
}

// The elevation of OBC node `obc` of TYPE_OBC 1..4 from the unconstrained
// one.  1/2: BCOND_ASL (mod_obcs.F:552-582), then the RK blend
// (external_step.F:262-266); 3/4: BCOND_ASL_CLP (mod_obcs.F:599-617).
__device__ __forceinline__ double ext_obc_given(const DevGrid& g, const ExtArgs& a, int obc, int ty, double elrk,
                                                double elf) {
  if (ty > 2) return 0.0;
  if (g.obc_elev) {
    const double rk_time = a.ec->time + g.dte * (a.alpha - 1.0);
    elf = tide_force(g, obc, rk_time, a.ec->ramp);
  }
  return elrk + a.alpha * (elf - elrk);
}

// The open-boundary condition of OBC node i (index obc) of TYPE_OBC 5..10.
// 5/6: BCOND_GWI (mod_obcs.F:624-658) and 7/8: BCOND_BKI (mod_obcs.F:665-699)
// from the new elevation el2 of the neighbour NEXT_OBC; 9/10: BCOND_ORE
// (mod_obcs.F:706-737) from the stage input EL and the elevations ELM1/ELM2
// one and two stages back.
__device__ __forceinline__ double ext_obc_radiated(const DevGrid& g, const ExtArgs& a, int i, int obc, int ty,
                                                   double elrk, double el2) {
  if (ty >= 9) {
    const int i2 = g.next_obc[obc], i3 = g.next_obc2[obc];
    const double cl = (a.elm2[i2] - a.cur.el[i2]) / (a.cur.el[i2] + a.elm2[i2] - 2.0 * a.elm1[i3]);
    double mu;                            // a NaN CL (0/0 at rest) gives MU = 0, as in the reference
    if (cl >= 1.0) mu = 1.0;
    else if (cl > 0.0 && cl < 1.0) mu = cl;
    else mu = 0.0;
    return (a.elm1[i] * (1.0 - mu) + 2.0 * mu * a.cur.el[i2]) / (1.0 + mu);
  }
  const double cc = sqrt(g.grav_n[i] * g.h[i]) * g.dte / g.dltn_obc[obc] * a.alpha;
  const double cp = cc + 1.0;
  return ty <= 6 ? (cc * el2 + elrk) / cp : (cc * el2 + elrk * (1.0 - g.dte / 10800.0)) / cp;
}

// FLUX_OBN's flux defect (mod_obcs.F:1196) of every OBC node, as k_ext_stage
// forms it, for a mesh on which an element that it goes to does not have the
// node, so that the node's tile cannot hand it over (the grid's ADJC_OBC are
// cells around the node; a host may set others).  One thread per OBC node,
// before the stage.
__global__ void k_ext_fobn(const DevGrid* __restrict__ gp, ExtArgs a) {
  const DevGrid& g = *gp;
  const int obc = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (obc >= g.IOBCN) return;
  auto update = [&](int i, int ob, double& xobc) {
    int ce[FV_MAX_CV];
    static_for<FV_MAX_CV>([&](auto jc) {
      constexpr int q = decltype(jc)::value;
      ce[q] = q < g.cv_max ? g.cvl_ent[(long)q * g.m1 + i] : 0;
    });
    const double e = ext_node_update<FV_MAX_CV>(g, a, i, ce, g.node_riv[i], ob >= 0, g.art1[i], a.elrk[i], xobc);
    const int ty = ob >= 0 ? g.type_obc[ob] : 5;
    return ty < 5 ? ext_obc_given(g, a, ob, ty, a.elrk[i], e) : e;
  };
  const int j = g.i_obc_n[obc], ty = g.type_obc[obc];
  const double elrk = a.elrk[j];
  double xobc, x2, el2 = 0.0;
  double elf = update(j, obc, xobc);
  if (ty >= 5 && ty <= 8) el2 = update(g.next_obc[obc], g.node_obc[g.next_obc[obc]], x2);
  if (ty >= 5) elf = ext_obc_radiated(g, a, j, obc, ty, elrk, el2);
  g.fobn[obc] = -(elf - elrk) * g.art1[j] / (a.alpha * g.dte) - xobc;
}

// ASSIGN_ELM1_TO_ELM2 (mod_obcs.F:178-199) at the end of a stage
// (external_step.F:333): ELM2 = ELM1, ELM1 = the stage input EL.  Run
// after k_ext_stage, the only reader; launched only when Orlanski nodes exist.
__global__ void k_elm_shift(DevGrid g, ExtArgs a) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i > g.M) return;
  a.elm2[i] = a.elm1[i];
  a.elm1[i] = a.cur.el[i];
}

// What the INT form of k_ext_stage leaves for the external steps, from the
// current state: the EXTEL terms and the block-order constants.  For a
// direct EXTERNAL_STEP call; one workgroup per element tile.
__global__ __launch_bounds__(FV_CVB) void k_ext_begin(DevGrid g, ExtArgs a) {
  const int b = (int)blockIdx.x, t = threadIdx.x;
  if (t >= g.cvb_ne[b]) return;
  const int i = g.cvb_elems[(long)FV_CVB * b + t];
  const double v[6] = {a.adx2d[i], a.ady2d[i], a.drx2d[i], a.dry2d[i], a.wubot[i], a.wvbot[i]};
#pragma unroll
  for (int q = 0; q < 6; ++q) a.own2d[(6L * b + q) * FV_CVB + t] = v[q];
  const double ua = a.cur.ua[i], va = a.cur.va[i], d1 = a.cur.d1[i];
  const long p0 = 3L * (i - 1) + 1;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const long q = (long)j * g.n1 + i;
    a.phi_next[p0 + j] = d1 * (-ua * g.ecv_dy[q] + va * g.ecv_dx[q]);
  }
}

// Fills the 2-D stage's tables (StageTab) from the grid, one workgroup per
// element tile; stn[FV_CVB*b + t]: 2*node + 1 in the first tile that has it.
__global__ __launch_bounds__(256) void k_stage_tables(DevGrid g, StageTab st, const int* stn) {
  const long b = blockIdx.x;
  const int t = threadIdx.x;
  const UvBlocks& B = g.ub_tile;
  const int nown = B.nown[b];
  int4 rec = make_int4(INT_MIN, 0, 0, 0);
  if (t < B.ns[b]) {
    const int x = B.elems[256 * b + t];
    rec = make_int4(t < nown ? x : ~x, NBE_(x, 1), NBE_(x, 2), NBE_(x, 3));
  }
  st.rec[256 * b + t] = rec;
  unsigned pl = ~0u;
  double v[6] = {};
  if (t < B.ne[b]) {
    const int c = B.edges[256 * b + t], ia = IEC_(c, 1), ib = IEC_(c, 2);
    const int isbc = g.isbc[c];
    pl = (unsigned)B.eloc[256 * b + t] | (unsigned)(isbc >= 0 && isbc <= 2 ? isbc : 3) << 30;
    // the edge's nodes are nodes of whichever of its elements the tile owns
    const int sa = pl & 255, sb = (pl >> 8) & 255;
    const int e = B.elems[256 * b + (sa < nown ? sa : sb)], loc = g.cvb_loc[e];
    for (int q = 0; q < 2; ++q) {
      const int j = IENODE_(c, q + 1);
      const int l = j == NV_(e, 1) ? loc & 255 : j == NV_(e, 2) ? (loc >> 8) & 255 : (loc >> 16) & 255;
      pl |= (unsigned)l << (16 + 7 * q);
    }
    v[0] = g.xijc[c] - g.xc[ia]; v[1] = g.yijc[c] - g.yc[ia];
    v[2] = g.xijc[c] - g.xc[ib]; v[3] = g.yijc[c] - g.yc[ib];
    v[4] = g.dltxc[c]; v[5] = g.dltyc[c];
  }
  st.edge[256 * b + t] = pl;
  for (int q = 0; q < 6; ++q) st.egeo[(6 * b + q) * 256 + t] = v[q];
  if (t >= FV_CVB) return;
  const bool nact = t < g.cvb_nn[b];
  const int i = nact ? g.cvb_nodes[FV_CVB * b + t] : 0;
  st.node[FV_CVB * b + t] = nact ? make_int4(stn[FV_CVB * b + t], 0, g.node_obc[i], g.node_riv[i])
                                 : make_int4(-1, 0, -1, -1);
  for (int j = 0; j < st.nslot; ++j)
    st.list[(st.nslot * b + j) * FV_CVB + t] = nact && j < g.cv_max ? g.cvl_ent[(long)j * g.m1 + i] : 0;
  st.nd[2 * b * FV_CVB + t] = nact ? g.art1[i] : 1.0;
  st.nd[(2 * b + 1) * FV_CVB + t] = nact ? g.h[i] : 0.0;
  const bool oact = t < nown;
  const int e = oact ? B.elems[256 * b + t] : 0;
  const int isbce = g.isbce[e] >= 0 && g.isbce[e] <= 3 ? g.isbce[e] : 0;
  st.elem[FV_CVB * b + t] = oact ? make_int4(B.epos[e], g.cvb_loc[e],
                                             isbce | (g.re_off[e] < g.re_off[e + 1] ? 4 : 0), g.iucp[e])
                                 : make_int4(0, 0, 0, 0);
  double w[12] = {};
  if (oact) {
    w[0] = g.epor[e]; w[1] = g.grav_e[e]; w[2] = g.art[e]; w[3] = g.cor[e]; w[4] = g.h1[e]; w[5] = g.cc_sponge[e];
    for (int j = 0; j < 3; ++j) {
      w[6 + j] = g.ecv_dx[(long)j * g.n1 + e];
      w[9 + j] = g.ecv_dy[(long)j * g.n1 + e];
    }
  }
  for (int q = 0; q < 12; ++q) st.ed[(12 * b + q) * FV_CVB + t] = w[q];
}

// One 2-D stage by element tile.  A workgroup of 256 lanes takes a compact
// tile of at most 128 elements (DevGrid::ub_tile, cvb_*) and
// does the whole stage for it, so that neither the edge terms nor the new
// elevation cross HBM between launches:
//   1. lanes 0, 1, ..: the least-squares velocity gradients of the tile's
//      elements and of the other elements of their edges (at most 256), one
//      element a lane, into LDS; lanes 255, 254, ..: the new elevation of
//      the tile's nodes, one node a lane;
//   2. one edge a lane: the ADVAVE_EDGE_GCN edge terms from the two
//      elements' gradients (at most 256 edges), into LDS;
//   3. one own element a lane: its three edges' terms summed in edge order,
//      EXTUV_EDGE, the wall projection and the sub-edge terms of the next
//      stage.
// A node on a tile's border is formed by every tile that has it, with the
// same operations on the same operands, and stored by the first of them.
// So that no lane can read what another workgroup has already replaced, the
// sub-edge terms go from one buffer to another, and stages 2-4 read the RK
// base elevation from a copy (stage 4 writes over the base).
//
// Bound: on a large mesh HBM (1,000,000 elements in FP64: 622 MB a stage,
// 147 us, 4.2 TB/s; as separate elevation, edge and momentum kernels 196 us,
// 180 with the first two side by side), on a small one the launches and the
// dependent loads of one tile (3,200 elements: 21 -> 9 us a stage).  The
// constants come in block order because gathering them by index had every
// tile wait for one more load and fetch rows of partly used lines (206 ->
// 164 us); the own elements' data is loaded after the node part, so that
// their registers do not add up (159 -> 112 VGPRs, 153 us).
//
// INT: the same edge terms for ADVAVE_EDGE_GCN of INTERNAL_STEP
// (internal_step.F:387-392) instead of a stage: ADX2D/ADY2D -= the sums, the
// accumulators of the coming external steps set to zero
// (internal_step.F:395-397) and the first stage's sub-edge terms formed.
//
// ODD: for tables that a host has set otherwise than the grid builder does
// (fvgpu_handle::stage_odd) -- ISBC outside 0..2, a radiating node whose
// NEXT_OBC is an OBC node, an ADJC_OBC without its node.  A kernel of its own:
// in the others' code the three cost 1 % of a 3,200-element step (515.4 us,
// 510.6 without).
template <typename FT>
struct ExtRecsLds {   // one array per quantity: a wave's reads of one spread over the banks
  FT u[256], v[256], c1[256], c2[256], c5[256], c6[256], p[256], cc[256];
};
template <typename FT>
struct ExtFluxLds {
  FT xadv[256], yadv[256], fx[256], fy[256];
  double elij[256], dlx[256], dly[256];
  int isbc[256];
};

template <int SMAX, typename FT, bool INT, bool ODD>
__global__ __launch_bounds__(256) void k_ext_stage(const DevGrid* __restrict__ gp, ExtArgs a) {
  const DevGrid& g = *gp;   // in device memory, for the boundary parts: by value its pointers
                            // overflow the scalar registers
  __shared__ ExtRecsLds<FT> sr;
  __shared__ ExtFluxLds<FT> sf;
  __shared__ double s_elf[FV_CVB], s_el[FV_CVB], s_d[FV_CVB], s_fobn[FV_CVB];
  const FT half = (FT)0.5, one = (FT)1.0;
  const int b = xcd_block(), t = threadIdx.x;
  const StageTab& st = a.st;
  // the block-order constants of the first two parts, so that their
  // latencies overlap
  int4 xs = make_int4(INT_MIN, 0, 0, 0), nd = make_int4(-1, 0, -1, -1);
  if (t < st.n_rec) xs = st.rec[256L * b + t];
  const int tn = 255 - t;   // lane 255 - tn: the tile's node tn
  if (tn < st.n_node) nd = st.node[(long)FV_CVB * b + tn];
  int ce[SMAX];
  if constexpr (!INT) {
    const int* lst = st.list + (long)st.nslot * b * FV_CVB + min(tn, FV_CVB - 1);
    if (tn < st.n_node)
      static_for<SMAX>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        ce[j] = j < st.nslot ? lst[j * FV_CVB] : 0;   // 0: the zero term
      });
  }
  unsigned pl = ~0u;
  double eg[6];   // XIJC-XC, YIJC-YC of IA, the same of IB, DLTXC, DLTYC
  if (t < st.n_edge) {
    pl = st.edge[256L * b + t];
#pragma unroll
    for (int q = 0; q < 6; ++q) eg[q] = st.egeo[(6L * b + q) * 256 + t];
  }
  const bool ract = xs.x != INT_MIN, oact = xs.x > 0, eact = pl != ~0u, nact = nd.x >= 0;
  const bool n0 = b == 0 && tn == FV_CVB;   // node 0 by block 0
  if (n0) nd.x = 1;
  const int i = xs.x >= 0 ? xs.x : ~xs.x;
  double ua = 0.0, va = 0.0;
  // 1. gradients
  if (ract) {
    FT ra1[4], ra2[4];
    lsq_coef<FT>(st.a12, i, ra1, ra2);
    const FT rart = (FT)at(st.art, i), rcc = (FT)at(st.cc_hvc, i);
    ua = at(a.cur.ua, i);
    va = at(a.cur.va, i);
    const FT us = (FT)ua, u1 = (FT)at(a.cur.ua, xs.y), u2 = (FT)at(a.cur.ua, xs.z), u3 = (FT)at(a.cur.ua, xs.w);
    const FT vs = (FT)va, v1 = (FT)at(a.cur.va, xs.y), v2 = (FT)at(a.cur.va, xs.z), v3 = (FT)at(a.cur.va, xs.w);
    const FT c1 = ra1[0] * us + ra1[1] * u1 + ra1[2] * u2 + ra1[3] * u3;
    const FT c2 = ra2[0] * us + ra2[1] * u1 + ra2[2] * u2 + ra2[3] * u3;
    const FT c5 = ra1[0] * vs + ra1[1] * v1 + ra1[2] * v2 + ra1[3] * v3;
    const FT c6 = ra2[0] * vs + ra2[1] * v1 + ra2[2] * v2 + ra2[3] * v3;
    const FT vis = rart * sqrt(sq(c1) + sq(c6) + half * sq(c2 + c5));
    sr.u[t] = us; sr.v[t] = vs;
    sr.c1[t] = c1; sr.c2[t] = c2; sr.c5[t] = c5; sr.c6[t] = c6;
    sr.p[t] = vis * rcc;
    sr.cc[t] = rcc;
  }
  // 1. nodes
  if (nact || n0) {
    const int j = nd.x >> 1, obc = nd.z;
    const bool keep = (nd.x & 1) != 0;   // this tile stores the node
    if (nact) {
      s_el[tn] = at(a.cur.el, j);
      s_d[tn] = at(a.cur.d, j);
    }
    if constexpr (INT) {
      if (keep) {
        a.egf[j] = 0.0;
        if (obc >= 0) a.uard_obcn[obc] = 0.0;
      }
      if (n0) { a.uard[0] = 0.0; a.vard[0] = 0.0; }
    } else {
      double art1, hn;
      if (nact) {
        art1 = st.nd[2L * b * FV_CVB + tn];
        hn = st.nd[(2L * b + 1) * FV_CVB + tn];
      } else {
        art1 = g.art1[0];
        hn = g.h[0];
      }
      const double elrk = at(a.elrk, j);
      if (keep && a.elrk_copy) a.elrk_copy[j] = elrk;
      const int ty = obc >= 0 ? g.type_obc[obc] : 0;
      // GWI / BKI need their neighbour's new elevation: a second pass forms
      // it, as the tile that has that node does (ODD: an OBC node of TYPE_OBC
      // 1..4 with its given elevation)
      double elf = 0.0, el2 = 0.0, xobc = 0.0;
      int id = j, rv = nd.w;
      double ar = art1, er = elrk;
      if (n0)
        static_for<SMAX>([&](auto jc) { ce[decltype(jc)::value] = 0; });
      for (bool next = false;;) {
        double xo;
        const int ob = ODD && next ? g.node_obc[id] : next ? -1 : obc;
        const double e = ext_node_update<SMAX>(g, a, id, ce, rv, ob >= 0, ar, er, xo);
        if (next) {
          el2 = ODD && ob >= 0 && g.type_obc[ob] < 5 ? ext_obc_given(g, a, ob, g.type_obc[ob], er, e) : e;
          break;
        }
        elf = e;
        xobc = xo;
        if (ty < 5 || ty > 8) break;
        id = g.next_obc[obc];
        static_for<SMAX>([&](auto jc) {
          constexpr int q = decltype(jc)::value;
          ce[q] = q < st.nslot ? g.cvl_ent[(long)q * g.m1 + id] : 0;
        });
        rv = g.node_riv[id];
        ar = g.art1[id]; er = a.elrk[id];
        next = true;
      }
      if (obc >= 0) {
        elf = ty < 5 ? ext_obc_given(g, a, obc, ty, elrk, elf) : ext_obc_radiated(g, a, j, obc, ty, elrk, el2);
        // FLUX_OBN's flux defect (mod_obcs.F:1196) and, in the last stage,
        // the node's UARD_OBCN share (external_step.F:423-430)
        if (nact) s_fobn[tn] = -(elf - elrk) * art1 / (a.alpha * g.dte) - xobc;
        if (a.K == 4 && keep) {
          const double tmp = -(elf - elrk) * art1 / g.dte - xobc;
          a.uard_obcn[obc] = a.uard_obcn[obc] + tmp / (double)g.isplit;
        }
      }
      if (nact) s_elf[tn] = elf;
      if (keep) {
        const double dnew = hn + elf;
        a.nxt.el[j] = elf;
        a.nxt.d[j] = dnew;
        if (a.K == 3) a.egf[j] = a.egf[j] + elf / (double)g.isplit;
        if (j >= 1 && dnew < g.min_depth) a.clk->depth_fail = 1;
      }
    }
  }
  // the element part's constants and state (the block's own elements are its
  // first records): issued before the barrier, after the node part, whose
  // registers are free again
  int4 oe = make_int4(0, 0, 0, 0);
  double ed[12], own[6], d1 = 0.0, el1b = 0.0, uab = 0.0, vab = 0.0, wsx = 0.0, wsy = 0.0;
  if (oact) {
    oe = st.elem[(long)FV_CVB * b + t];
#pragma unroll
    for (int q = 0; q < 12; ++q) ed[q] = st.ed[(12L * b + q) * FV_CVB + t];
    d1 = at(a.cur.d1, i);
    if constexpr (INT) {
      own[0] = a.adx2d[i]; own[1] = a.ady2d[i]; own[2] = a.drx2d[i]; own[3] = a.dry2d[i];
      own[4] = a.wubot[i]; own[5] = a.wvbot[i];
    } else {
#pragma unroll
      for (int q = 0; q < 6; ++q) own[q] = a.own2d[(6L * b + q) * FV_CVB + t];
      el1b = at(a.base.el1, i); uab = at(a.base.ua, i); vab = at(a.base.va, i);
      if (g.wind_on) { wsx = at(a.ws2x, i); wsy = at(a.ws2y, i); }
    }
  }
  __syncthreads();
  // 2. edge terms
  if (eact) {
    const int sa = pl & 255, sb = (pl >> 8) & 255, n1 = (pl >> 16) & 127, n2 = (pl >> 23) & 127;
    const FT dij = half * ((FT)s_d[n1] + (FT)s_d[n2]);
    const FT xija = (FT)eg[0], yija = (FT)eg[1], xijb = (FT)eg[2], yijb = (FT)eg[3], dlx = (FT)eg[4],
             dly = (FT)eg[5];
    const FT cofa1 = sr.c1[sa], cofa2 = sr.c2[sa], cofa5 = sr.c5[sa], cofa6 = sr.c6[sa];
    const FT cofa3 = sr.c1[sb], cofa4 = sr.c2[sb], cofa7 = sr.c5[sb], cofa8 = sr.c6[sb];
    const FT uij1 = sr.u[sa] + cofa1 * xija + cofa2 * yija;
    const FT vij1 = sr.v[sa] + cofa5 * xija + cofa6 * yija;
    const FT uij2 = sr.u[sb] + cofa3 * xijb + cofa4 * yijb;
    const FT vij2 = sr.v[sb] + cofa7 * xijb + cofa8 * yijb;
    const FT uij = half * (uij1 + uij2), vij = half * (vij1 + vij2);
    const FT un_tmp = -uij * dly + vij * dlx;
    FT viscof = (FT)g.fact * half * (sr.p[sa] + sr.p[sb]) + (FT)g.fm1 * half * (sr.cc[sa] + sr.cc[sb]);
    if ((FT)g.hprnu != one) viscof = viscof / (FT)g.hprnu;   // x / 1 is x
    const FT txxij = (cofa1 + cofa3) * viscof;
    const FT tyyij = (cofa6 + cofa8) * viscof;
    const FT txyij = half * (cofa2 + cofa4 + cofa5 + cofa7) * viscof;
    sf.fx[t] = dij * (txxij * dly - txyij * dlx);
    sf.fy[t] = dij * (txyij * dly - tyyij * dlx);
    const FT sgn = fsign1(un_tmp);
    sf.xadv[t] = dij * un_tmp * ((one - sgn) * uij2 + (one + sgn) * uij1) * half;
    sf.yadv[t] = dij * un_tmp * ((one - sgn) * vij2 + (one + sgn) * vij1) * half;
    sf.elij[t] = 0.5 * (s_el[n1] + s_el[n2]);
    sf.dlx[t] = eg[4];
    sf.dly[t] = eg[5];
    sf.isbc[t] = ODD ? g.isbc[g.ub_tile.edges[256L * b + t]] : (int)(pl >> 30);
  }
  __syncthreads();
  if (!oact) return;
  // 3. FLUX_OBN: contributions to this open-boundary element, in OBC order
  const int ep3 = oe.x, nl = oe.y, isb = oe.z & 3;
  const double ep = ed[0], ge = ed[1], art = ed[2], cor = ed[3], h1 = ed[4], spg = ed[5], iu = (double)oe.w;
  double fl = 0.0;
  if (isb == 2) {
    if constexpr (INT) {
      fl = a.fluxobn[i];
    } else {
      for (int p = g.fo_off[i]; p < g.fo_off[i + 1]; ++p) {
        const int ent = g.fo_obc[p], ob = ent >> 1, slot = ent & 1;
        const int j = g.i_obc_n[ob];   // one of the element's nodes (ODD: or g.fobn has it)
        const int ln = j == NV_(i, 1) ? nl & 255 : j == NV_(i, 2) ? (nl >> 8) & 255 : (nl >> 16) & 255;
        fl = fl + g.fluxf_obc[(long)slot * g.IOBCN + ob] * (ODD && g.fobn ? g.fobn[ob] : s_fobn[ln]);
      }
      a.fluxobn[i] = fl;
    }
  }
  // ADVAVE_EDGE_GCN's sums (advave_edge_gcn.F:746-992) in edge order
  double xf = 0.0, yf = 0.0, px = 0.0, py = 0.0;
  const double gdi = ge * d1;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int s = (ep3 >> (8 * q)) & 255;
    const bool ib = (ep3 >> (24 + q)) & 1;   // the element is IB of the edge
    const double xadv = (double)sf.xadv[s], yadv = (double)sf.yadv[s], fx = (double)sf.fx[s], fy = (double)sf.fy[s];
    const double isbc_tmp = (double)sf.isbc[s];
    const double gd = gdi * sf.elij[s];
    const double tx = (xadv + fx * ep) * (1.0 - isbc_tmp) * iu;
    const double ty = (yadv + fy * ep) * (1.0 - isbc_tmp) * iu;
    const double gy = gd * sf.dly[s], gx = gd * sf.dlx[s];
    xf = ib ? xf - tx : xf + tx;
    yf = ib ? yf - ty : yf + ty;
    px = ib ? px + gy : px - gy;
    py = ib ? py - gx : py + gx;
  }
  if (isb == 2) {
    xf = (xf + fl * ua) * iu;
    yf = (yf + fl * va) * iu;
  }
  if (oe.z & 4) {
    for (int p = g.re_off[i]; p < g.re_off[i + 1]; ++p) {
      // a node river's momentum is split between two cells, an edge river's
      // enters its cell whole (advave_edge_gcn.F:971-992)
      const int k = g.re_riv[p];
      const double fq = g.icellq[k] > 0 ? 1.0 : 0.5;
      const double vlctyq = a.qdis[k] / g.qarea[k];
      xf = xf - fq * a.qdis[k] * vlctyq * g.cos_angleq[k];
      yf = yf - fq * a.qdis[k] * vlctyq * g.sin_angleq[k];
    }
  }
  double un = ua, vn = va, dn = d1;
  if constexpr (INT) {
    own[0] = own[0] - xf;
    own[1] = own[1] - yf;
    a.adx2d[i] = own[0];
    a.ady2d[i] = own[1];
    a.uard[i] = 0.0;
    a.vard[i] = 0.0;
#pragma unroll
    for (int q = 0; q < 6; ++q) a.own2d[(6L * b + q) * FV_CVB + t] = own[q];
  } else {
    // EXTUV_EDGE
    const double one_third = 1.0 / 3.0, ramp = a.ec->ramp;
    const double elf1 = one_third * (s_elf[nl & 255] + s_elf[(nl >> 8) & 255] + s_elf[(nl >> 16) & 255]);
    const double wus2 = g.wind_on ? wsx * ramp * 0.001 : 0.0;
    const double wvs2 = g.wind_on ? wsy * ramp * 0.001 : 0.0;
    const double resx = own[0] + xf + own[2] + px - cor * va * d1 * art - (wus2 + own[4]) * art;
    const double resy = own[1] + yf + own[3] + py + cor * ua * d1 * art - (wvs2 + own[5]) * art;
    un = (uab * (h1 + el1b) - a.alpha * g.dte * resx / art) / (h1 + elf1);
    vn = (vab * (h1 + el1b) - a.alpha * g.dte * resy / art) / (h1 + elf1);
    un = un / (1.0 + spg * un * un);
    vn = vn / (1.0 + spg * vn * vn);
    if (isb != 0) wall_project(g, i, un, vn);
    dn = h1 + elf1;
    a.nxt.ua[i] = un;
    a.nxt.va[i] = vn;
    a.nxt.el1[i] = elf1;
    a.nxt.d1[i] = dn;
    if (a.K == 3) {
      a.uard[i] = a.uard[i] + un * dn;
      a.vard[i] = a.vard[i] + vn * dn;
    }
  }
  // the next stage's EXTEL terms of the element's sub-edges (side IB)
  const long p0 = 3L * (i - 1) + 1;
#pragma unroll
  for (int j = 0; j < 3; ++j) a.phi_next[p0 + j] = dn * (-un * ed[9 + j] + vn * ed[6 + j]);
}
