// fvgpu_kernels_tracer.h -- node-centred kernels of the MY2.5 turbulence
// quantities (FCT_Q2/Q2L, VDIF_Q) and the tracers (FCT_T/FCT_S, VDIF_TS,
// BCOND_TS), plus DENS2.  Their horizontal advection is in
// fvgpu_kernels_cv.h.
#pragma once
#include "fvgpu_kernels_3d.h"

// ADJUST_TS (adjust_ts.F:150-172), run when RIVER_TS_SETTING is
// 'calculated' (internal_step.F:1374-1376), in one workgroup: T1/S1 of
// every river node raised to its river's TDIS/SDIS on layers 1..KBM1, one
// thread per layer walking the rivers in order (two rivers at one node see
// each other's result, as in the reference's loop); then N2E3D of T1 and S1
// for the elements around the river nodes, the only elements whose three
// nodes changed (the others' T/S already hold the same values).
__global__ void k_adjust_ts(DevGrid g, IntArgs a) {
  // a river's nodes: its node, or the two nodes of its solid edge
  auto river_nodes = [&](int r, int (&nd)[2]) {
    if (g.icellq[r] > 0) { nd[0] = g.n_icellq[r]; nd[1] = g.n_icellq[g.NUMQBC + r]; return 2; }
    nd[0] = g.inodeq[r];
    return 1;
  };
  for (int k = threadIdx.x + 1; k <= g.KBM1; k += blockDim.x)
    for (int r = 0; r < g.NUMQBC; ++r) {
      int nd[2];
      const int c = river_nodes(r, nd);
      for (int q = 0; q < c; ++q) {
        const long p = NI(g, nd[q], k);
        a.t1[p] = fmax(a.t1[p], g.tdis[r]);
        a.s1[p] = fmax(a.s1[p], g.sdis[r]);
      }
    }
  __syncthreads();
  const double one_third = 1.0 / 3.0;
  for (int r = 0; r < g.NUMQBC; ++r) {
    int nd[2];
    const int c = river_nodes(r, nd);
    for (int q0 = 0; q0 < c; ++q0) {
      const int j = nd[q0], off = g.nbve_off[j], nt = g.ntve[j];
      for (int q = threadIdx.x; q < nt * g.KB; q += blockDim.x) {
        const int i = g.nbve[off + q % nt], k = q / nt + 1;
        const int j1 = NV_(i, 1), j2 = NV_(i, 2), j3 = NV_(i, 3);
        a.t[EI(g, i, k)] = one_third * (a.t1[NI(g, j1, k)] + a.t1[NI(g, j2, k)] + a.t1[NI(g, j3, k)]);
        a.s[EI(g, i, k)] = one_third * (a.s1[NI(g, j1, k)] + a.s1[NI(g, j2, k)] + a.s1[NI(g, j3, k)]);
      }
    }
  }
}

// BCOND_TS(NCON) (bcond_ts.F:28-268) at the open boundary, one wave per OBC
// node and pass (blockIdx.y): the column sums of the node (T2D), the interior
// neighbour (T2D_NEXT) and the OBC advective flux (XFLUX2D) -- the products of
// all layers formed by the lanes at once, then one lane per sum adds them from
// LDS in layer order -- and the radiated value (TYPE_TSOBC 1-4) of each layer,
// one lane per layer, limited to the ring and vertical-neighbour bounds, or
// F1 itself when the node has no inflow.  NEXT_OBC is an interior node, so no
// wave reads what another writes.  (The rivers' specified values: VDIF_TS.)
// Bound: the latency of its loads; 62,000 elements x 40 layers, T and S: 2 x
// (sums with one thread a node 31 us, layers 9 us) -> 10.4 us.
__global__ __launch_bounds__(64) void k_bcond_ts(DevGrid g, IntArgs a, Passes P) {
  __shared__ double prod[5][65], sums[5];
  const Pass ps = blockIdx.y == 0 ? P.p[0] : P.p[1];
  const int t = (int)blockIdx.x, lane = (int)threadIdx.x, KBM1 = g.KBM1;
  double* ff = ps.ff;
  const double* f1 = ps.f;
  const int j = g.i_obc_n[t], j1 = g.next_obc[t];
  // the Orlanski form's column sums of F1 at NEXT_OBC and NEXT_OBC2 (its
  // F1M1 is F1 here: see below)
  const bool orl = g.type_tsobc == 4;
  const int j2 = orl ? g.next_obc2[t] : j1;
  double acc = 0.0;
  for (int c = 0; c < KBM1; c += 64) {
    const int k = c + lane + 1;
    if (k <= KBM1) {
      prod[0][lane] = f1[NI(g, j, k)] * DZ(j, k);
      prod[1][lane] = ff[NI(g, j1, k)] * DZ(j1, k);
      prod[2][lane] = ps.xflux_obc[(long)(k - 1) * g.IOBCN + t];
      if (orl) {
        prod[3][lane] = f1[NI(g, j1, k)] * DZ(j1, k);
        prod[4][lane] = f1[NI(g, j2, k)] * DZ(j2, k);
      }
    }
    __syncthreads();
    if (lane < (orl ? 5 : 3))
      for (int q = 0; q < min(64, KBM1 - c); ++q) acc = acc + prod[lane][q];
    __syncthreads();
  }
  if (lane < 5) sums[lane] = acc;
  __syncthreads();
  const double t2d = sums[0], t2d_next = sums[1], xflux2d = sums[2];
  const bool inflow = a.uard_obcn[t] > 0.0;
  for (int k = lane + 1; k <= KBM1; k += 64) {
    if (!inflow) {
      ff[NI(g, j, k)] = f1[NI(g, j, k)];
      continue;
    }
    const double tmp = xflux2d + t2d * a.uard_obcn[t];
    const double t2d_obc = (t2d * a.dt[j] - tmp * g.dti / g.art1[j]) / a.d[j];
    const double cc = sqrt(g.grav_n[j] * g.h[j]) * g.dti / g.dltn_obc[t], cp = cc + 1.0;
    const double pert_next = ff[NI(g, j1, k)] - t2d_next, pert = f1[NI(g, j, k)] - t2d;
    double ttmp;
    if (g.type_tsobc == 1) ttmp = ff[NI(g, j1, k)] - t2d_next;
    else if (g.type_tsobc == 2) ttmp = (cc * pert_next + pert) / cp;
    else if (g.type_tsobc == 3) ttmp = (cc * pert_next + pert * (1.0 - g.dti / 10800.0)) / cp;
    else {
      // Orlanski (mod_obcs.F:1258-1285, 1336-1363).  Its F1M1/F1M2 are F1
      // one and two external RK stages back (ASSIGN_ELM1_TO_ELM2, called at
      // every stage, mod_obcs.F:190-196); F1 does not change during the
      // external steps, which run before BCOND_TS, so both equal F1 here, and
      // their column sums are the same sums of F1 (T2D at the OBC node,
      // T2D_NEXT1 at NEXT_OBC) formed in the same order.
      const double t2d_next1 = sums[3], tm12d_next2 = sums[4];
      const double tm12d_next1 = t2d, tm22d_next1 = t2d_next1;
      const double f1j1 = f1[NI(g, j1, k)], m2j1 = f1j1, m1j2 = f1[NI(g, j2, k)], m1j = f1[NI(g, j, k)];
      const double cl = ((m2j1 - tm22d_next1) - (f1j1 - t2d_next1)) /
                        ((f1j1 - t2d_next1) + (m2j1 - tm22d_next1) - 2.0 * (m1j2 - tm12d_next2));
      double mu;
      if (cl >= 1.0) mu = 1.0;
      else if (cl > 0.0 && cl < 1.0) mu = cl;
      else mu = 0.0;
      ttmp = ((m1j - tm12d_next1) * (1.0 - mu) + 2.0 * mu * (f1j1 - t2d_next1)) / (1.0 + mu);
    }
    double x = t2d_obc + ttmp;
    const long ko = (long)(k - 1) * g.m1;
    const int o = g.nbsn_off[j], nt = g.ntsn[j];
    double tmax = f1[ko + g.nbsn[o]], tmin = tmax;
    for (int jj = 1; jj < nt; ++jj) { const double y = f1[ko + g.nbsn[o + jj]]; tmax = fmax(tmax, y); tmin = fmin(tmin, y); }
    const double fk = f1[ko + j];
    if (k == 1) {
      const double v = (fk * DZ(j, k + 1) + f1[ko + g.m1 + j] * DZ(j, k)) / (DZ(j, k) + DZ(j, k + 1));
      tmax = fmax(tmax, v); tmin = fmin(tmin, v);
    } else if (k == KBM1) {
      const double v = (fk * DZ(j, k - 1) + f1[ko - g.m1 + j] * DZ(j, k)) / (DZ(j, k) + DZ(j, k - 1));
      tmax = fmax(tmax, v); tmin = fmin(tmin, v);
    } else {
      const double v1 = (fk * DZ(j, k - 1) + f1[ko - g.m1 + j] * DZ(j, k)) / (DZ(j, k) + DZ(j, k - 1));
      const double v2 = (fk * DZ(j, k + 1) + f1[ko + g.m1 + j] * DZ(j, k)) / (DZ(j, k) + DZ(j, k + 1));
      tmax = fmax(tmax, fmax(v1, v2)); tmin = fmin(tmin, fmin(v1, v2));
    }
    if (tmin - x > 0.0) x = tmin;
    if (x - tmax > 0.0) x = tmax;
    ff[ko + j] = x;
  }
}

// DENS2 (eqs_of_state.F:254-403): RHO1 of node-layer t from its S and T;
// zero at the bottom level and node 0.
__device__ __forceinline__ double dens2(const DevGrid& g, long t, double s, double tt) {
  const int i = (int)(t % g.m1), k = (int)(t / g.m1) + 1;
  if (k == g.KB || i == 0) return 0.0;
  double r = s * s * s * 6.76786136E-6 - s * s * 4.8249614E-4 + s * 8.14876577E-1 - 0.22584586E0;
  r = r * (tt * tt * tt * 1.667E-8 - tt * tt * 8.164E-7 + tt * 1.803E-5);
  r = r + 1.0 - tt * tt * tt * 1.0843E-6 + tt * tt * 9.8185E-5 - tt * 4.786E-3;
  r = r * (s * s * s * 6.76786136E-6 - s * s * 4.8249614E-4 + s * 8.14876577E-1 + 3.895414E-2);
  r = r - (tt - 3.98) * (tt - 3.98) * (tt + 283.0) / (503.57 * (tt + 67.26));
  return r * 1.e-3;
}

__global__ void k_dens2(DevGrid g, IntArgs a) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < g.m1 * g.KB) a.rho1[t] = dens2(g, t, a.s1[t], a.t1[t]);
}

// End of INTERNAL_STEP (internal_step.F:1355-1590), one thread per position:
// T1 = TF1 and S1 = SF1 (t_on, s_on), then DENS2 of them where nothing comes
// between (dens); U = UF, V = VF; ET = EL, DT = D, ET1 = EL1, DT1 = D1.
// Bound: memory (1,000,000 elements x 40 layers, six launches 473 us -> 363).
__global__ __launch_bounds__(256) void k_step_end(DevGrid g, IntArgs a, int t_on, int s_on, int dens) {
  const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < g.n1 * g.KB) {
    a.u[q] = a.uf[q];
    a.v[q] = a.vf[q];
  }
  if (q < g.m1 * g.KB) {
    const double t = t_on ? a.tf1[q] : a.t1[q], s = s_on ? a.sf1[q] : a.s1[q];
    if (t_on) a.t1[q] = t;
    if (s_on) a.s1[q] = s;
    if (dens) a.rho1[q] = dens2(g, q, s, t);
  }
  if (q <= g.M) { a.et[q] = a.el[q]; a.dt[q] = a.d[q]; }
  if (q <= g.N) { a.et1[q] = a.el1[q]; a.dt1[q] = a.d1[q]; }
}
