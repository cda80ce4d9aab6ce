// fvgpu_kernels_column.h -- the implicit vertical solves with their Thomas
// coefficients in registers.
//
// One thread owns one column.  The recursion coefficients VH/VHP of the
// forward sweep are the only per-level state the back substitution needs;
// they live in register arrays of a compile-time bound KMAX >= KB (the loops
// are fully unrolled, so every index is a constant), and everything else
// (A, C, BOY, L, GH, STF, DTEF) is recomputed where it is used with the same
// operations, so the results are bit-identical to the straightforward form.
// The "last level" values are carried in scalars because KBM1/KBM2 are
// runtime values.
#pragma once
#include "fvgpu_kernels_tracer.h"

// x of the wave's lower 32 lanes and of its upper 32 lanes, in every lane
// (lane l gets those of lanes l%32 and 32 + l%32).
__device__ __forceinline__ void wave_halves(double x, double& lower, double& upper) {
  const unsigned lo = (unsigned)__double2loint(x), hi = (unsigned)__double2hiint(x);
  const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  lower = __hiloint2double((int)b[0], (int)a[0]);
  upper = __hiloint2double((int)b[1], (int)a[1]);
}

// VDIF_UV (vdif_uv.F:34-189), its sponge (vdif_uv.F:155-161) and the wall
// projection BCOND_GCN(3,0) (bcond_gcn.F:424-530).  A wave takes 32 element
// columns: its lower lanes solve U, its upper lanes V of the same elements,
// so that the coefficient VHU = VHV, evaluated by both with the same
// operations, is loaded once, and each level's pair meets in registers for
// the projection on the way up instead of in a pass of its own over both
// arrays.  Columns with D1 <= 0 are not solved but still projected.
// The loads of a level are issued FV_AHEAD levels before its elimination: the
// recursion is one dependent chain, each level in a branch of its own that no
// load crosses by itself, and two waves a SIMD are all that its registers
// leave; the sigma values are scalar loads (UNI), as a vector load in the
// middle of a level would wait for the levels ahead of it too.
// 1,000,000 elements x 40 layers: 907 us as a solve per component and a
// finishing pass, 832 fused without the loads ahead, 645 now (62,500: 59, 50,
// 41 us).
#define FV_AHEAD 4
template <int KMAX, bool UNI>
__global__ __launch_bounds__(256) void k_vdif_uv_r(DevGrid g, IntArgs a) {
  const int l = threadIdx.x & 63;
  const int f = l >> 5;                    // 0: U, 1: V
  const int col = (int)blockIdx.x * 128 + (int)(threadIdx.x >> 6) * 32 + (l & 31) + 1;
  const bool act = col <= g.N;
  const int i = min(col, g.N);
  const int KBM1 = g.KBM1, KBM2 = g.KBM2;
  const double dti = g.dti, umol = g.umol, d1 = a.d1[i];
  const bool solve = d1 > 0.0;
  const long n1 = g.n1;
  double* X = f ? a.vf : a.uf;
  auto dz1 = [&](int k) { return DZ1(i, k); };
  auto dzz1 = [&](int k) { return DZZ1(i, k); };
  // KM1 of level k+1 and X of layer k (past the column: its last)
  double kmp[KMAX + FV_AHEAD + 1], xk[KMAX + FV_AHEAD + 1];
  auto ahead = [&](auto kc) {
    constexpr int k = decltype(kc)::value;
    kmp[k] = at(a.km1 + (long)min(k, KBM1 - 1) * n1, i);
    xk[k] = at(X + (long)(min(k, KBM1) - 1) * n1, i);
  };
  static_for<FV_AHEAD>([&](auto jc) { ahead(std::integral_constant<int, decltype(jc)::value + 1>{}); });
  const double kmb = at(a.km1 + (long)(KBM1 - 1) * n1, i), xb = at(X + (long)(KBM1 - 1) * n1, i);
  const WallOp wop = wall_prep(g, i);
  const double sp = g.cc_sponge[i];
  const int it1 = g.isonb[NV_(i, 1)], it2 = g.isonb[NV_(i, 2)], it3 = g.isonb[NV_(i, 3)];
  const double tmp = (it1 == 2 || it2 == 2 || it3 == 2) ? 0.0 : 1.0;
  const double ramp = a.clk->ramp_int;
  const double ub = a.u[EI(g, i, KBM1)], vb = a.v[EI(g, i, KBM1)];
  const double tps = a.cbc[i] * sqrt(ub * ub + vb * vb);
  if (f == 0 && act && solve) {
    a.tps[i] = tps;
    a.wubot[i] = -tps * ub;
    a.wvbot[i] = -tps * vb;
  }
  const double ws = g.wind_on ? -(f ? g.wsy[i] : g.wsx[i]) * ramp * 0.001 : 0.0;
  double VH[KMAX + 1], VHP[KMAX + 1];
  const double a1 = -dti * (kmp[1] + umol) / (dz1(1) * dzz1(1) * d1 * d1);
  VH[1] = a1 / (a1 - 1.);
  VHP[1] = (-dti * ws * tmp / (-dz1(1) * d1) - xk[1]) / (a1 - 1.);
  double lastvh = VH[1], lastvhp = VHP[1];
  static_for<KMAX - 1>([&](auto kc) {
    constexpr int k = decltype(kc)::value + 2;
    if (k <= KBM2) {
      ahead(std::integral_constant<int, k + FV_AHEAD - 1>{});
      const double ak = -dti * (kmp[k] + umol) / (dz1(k) * dzz1(k) * d1 * d1);
      const double ck = -dti * (kmp[k - 1] + umol) / (dz1(k) * dzz1(k - 1) * d1 * d1);
      const double t = 1.0 / (ak + ck * (1. - VH[k - 1]) - 1.);
      VH[k] = ak * t;
      VHP[k] = (ck * VHP[k - 1] - xk[k]) * t;
      lastvh = VH[k];
      lastvhp = VHP[k];
    }
  });
  const double cb = -dti * (kmb + umol) / (dz1(KBM1) * dzz1(KBM1 - 1) * d1 * d1);
  double x = (cb * lastvhp - xb) / (tps * dti / (-dz1(KBM1) * d1) - 1. - (lastvh - 1.) * cb);
  // the finished value of layer k from the solved one, this lane's component
  auto finish = [&](int k, double v) {
    if (!solve) v = at(X + (long)(k - 1) * n1, i);
    const double own = v / (1.0 + sp * v * v);
    double uu, vv;
    wave_halves(own, uu, vv);
    wall_apply(wop, uu, vv);
    if (act) X[(long)(k - 1) * n1 + i] = f ? vv : uu;
  };
  finish(KBM1, x);
  static_for<KMAX>([&](auto kc) {
    constexpr int k = KMAX - decltype(kc)::value;
    if (k <= KBM2) {
      x = (VH[k] * x + VHP[k]);
      finish(k, x);
    }
  });
}

// VDIF_TS(NCON,F) (vdif_ts.F:42-385), FP64, no surface flux; loads ahead and
// sigma values as in VDIF_UV (1,000,000 elements x 40 layers: 157 -> 114 us; the
// loads ahead alone changed nothing).
template <int KMAX, bool UNI>
__global__ __launch_bounds__(256) void k_vdif_ts_r(DevGrid g, IntArgs a, Passes P) {
  Pass ps;
  int b;
  if (!pass_block(P, (int)(g.M / blockDim.x) + 1, ps, b)) return;
  const int i = b * (int)blockDim.x + (int)threadIdx.x;
  if (i < 1 || i > g.M) return;
  double* f = ps.ff;
  const int ncon = ps.which;
  const int KBM1 = g.KBM1, KBM2 = g.KBM2;
  if (g.river_ts_specified) {
    // BCOND_TS at the river nodes: the last river at the node sets it (the
    // reference sets TF1 and SF1 in both calls; each pass here sets its own,
    // which leaves T1 and S1 unchanged, F1 = FF following in both)
    const int rv = g.node_riv[i];
    if (rv >= 0) {
      double w;
      int last = -1;
      for (int j = rv; j < g.NUMQBC; ++j)
        if (river_share(g, j, i, w)) last = j;
      if (last >= 0) {
        for (int k = 1; k <= KBM1; ++k) f[NI(g, i, k)] = ps.fdis[last];
        return;
      }
    }
  }
  if (g.isonb[i] == 2) return;   // OBC columns keep F (vdif_ts.F:259,313)
  const double dti = g.dti, umolpr = g.umol * 1.E0, d = a.d[i];
  const long m1 = g.m1;
  auto dz = [&](int k) { return DZ(i, k); };
  auto dzz = [&](int k) { return DZZ(i, k); };
  double VHF[KMAX + 1], VHPF[KMAX + 1];
  // KH of level k+1 and F of layer k (past the column: its last)
  double khp[KMAX + FV_AHEAD + 1], fk[KMAX + FV_AHEAD + 1];
  auto ahead = [&](auto kc) {
    constexpr int k = decltype(kc)::value;
    khp[k] = at(a.kh + (long)min(k, KBM1 - 1) * m1, i);
    fk[k] = at(f + (long)(min(k, KBM1) - 1) * m1, i);
  };
  static_for<FV_AHEAD>([&](auto jc) { ahead(std::integral_constant<int, decltype(jc)::value + 1>{}); });
  const double khbottom = at(a.kh + (long)(KBM1 - 1) * m1, i), fbottom = at(f + (long)(KBM1 - 1) * m1, i);
  const double af1 = -dti * (khp[1] + umolpr) / (dz(1) * dzz(1) * d * d);
  VHF[1] = af1 / (af1 - 1.);
  VHPF[1] = -dti * (0.0 + 0.0 - 0.0 + 0.0 - 0.0) / (-dz(1) * d) - fk[1];
  VHPF[1] = VHPF[1] / (af1 - 1.);
  double lastvh = VHF[1], lastvhp = VHPF[1];
  static_for<KMAX - 1>([&](auto kc) {
    constexpr int k = decltype(kc)::value + 2;
    if (k <= KBM2) {
      ahead(std::integral_constant<int, k + FV_AHEAD - 1>{});
      const double afk = -dti * (khp[k] + umolpr) / (dz(k) * dzz(k) * d * d);
      const double cfk = -dti * (khp[k - 1] + umolpr) / (dz(k) * dzz(k - 1) * d * d);
      const double t = 1. / (afk + cfk * (1. - VHF[k - 1]) - 1.);
      VHF[k] = afk * t;
      VHPF[k] = (cfk * VHPF[k - 1] - fk[k] + dti * (0.0 - 0.0) / (d * dz(k))) * t;
      lastvh = VHF[k];
      lastvhp = VHPF[k];
    }
  });
  const double cfb = -dti * (khbottom + umolpr) / (dz(KBM1) * dzz(KBM1 - 1) * d * d);
  const double tmp1 = ps.pfpxb[i] * g.cos_sita[i] + ps.pfpyb[i] * g.sin_sita[i];
  const double tmp2 = ps.ah_bottom[i] * g.phpn[i];
  const double tmp3 = khbottom + umolpr + ps.ah_bottom[i] * g.phpn[i] * g.phpn[i];
  double tmp = tmp1 * tmp2 / tmp3 * (khbottom + umolpr);
  if (g.noflux_bot) {
    if (ncon == 1) { if (tmp1 > 0.0) tmp = 0.0; }
    else { if (tmp1 < 0.0) tmp = 0.0; tmp = -tmp; }
  } else {
    tmp = 0.0;
  }
  double x = (cfb * lastvhp - fbottom - 0.0 + dti * (0.0 - 0.0 - tmp) / (d * dz(KBM1))) /
             (cfb * (1. - lastvh) - 1.);
  f[NI(g, i, KBM1)] = x;
  static_for<KMAX>([&](auto kc) {
    constexpr int k = KMAX - decltype(kc)::value;
    if (k <= KBM2) {
      x = (VHF[k] * x + VHPF[k]);
      f[(long)(k - 1) * m1 + i] = x;
    }
  });
}

// Per-level quantities of VDIF_Q (vdif_q.F:255-368): from Q2, Q2L and RHO1
// at levels k-1 and k of node i, DZZ(k-1) and Z(k) (the values passed in).
struct Q25Level { double q2, boy, ll, gh, stf, dtef; };

__device__ __forceinline__ Q25Level q25_eval(const DevGrid& g, int i, int k, double d, double l0, double q2raw,
                                             double q2l, double rho_km1, double rho_k, double dzz, double z) {
  const double SMALL = 1.E-8, KAPPA = 0.40, GH_MAX = .0233, GHC = -6.0, GH_MIN = -.281, B1 = 16.6;
  const double p9 = (double)0.9f, p1 = (double)0.1f;
  Q25Level r;
  r.q2 = fabs(q2raw + SMALL);
  r.boy = 0.0;
  if (k >= 2 && k <= g.KBM1) r.boy = g.grav_n[i] * (rho_km1 - rho_k) / (dzz * d);
  if (k == 1) r.ll = KAPPA * l0;
  else if (k == g.KB) r.ll = 0.0;
  else {
    double ll = fabs(q2l) / r.q2;
    if (z > -0.5) ll = fmax(ll, KAPPA * l0);
    if (r.boy < 0.0) {
      const double lmax = sqrt(fabs(GH_MIN) * r.q2 / (-r.boy + SMALL));
      ll = fmin(ll, lmax);
    }
    r.ll = ll;
  }
  r.gh = 0.0;
  if (k >= 2 && k <= g.KBM1) r.gh = fmin((sq(r.ll) / r.q2) * r.boy, GH_MAX);
  r.stf = 1.0;
  if (r.gh < 0.0) r.stf = 1.0 - p9 * fv_pow15(r.gh / GHC);
  if (r.gh < GHC) r.stf = p1;
  r.dtef = sqrt(r.q2) / (B1 * r.ll + SMALL) * r.stf;
  return r;
}

// What VDIF_Q's downward sweep reads at one level: RHO1, KQ of the level
// below, Q2, Q2L, KM, KH, Q2F, Q2LF of the node, DZZ(k-1), DZ(k), Z(k) and
// U, V of its element ring.  (The sigma values too: a load issued inside the
// level's arithmetic is waited for after every load before it.)
template <int RMAX>
struct Q25Loads {
  double rho, kq, q2, q2l, km, kh, q2f, q2lf, dzz, dz, z, ur[RMAX], vr[RMAX];
};

// Columns a block of k_vdif_q_blk takes, and its arrays in LDS per level.
#define FV_VQN 16
#define FV_VQARR 11

// VDIF_Q, MY2.5 (vdif_q.F:34-551), one thread per node column in two
// sweeps.  The downward sweep k = 1..KB reads every node-layer value once
// (sliding windows over RHO1 and KQ, the ring averages of U/V): it forms the
// level quantities (vdif_q.F:255-368) and PROD (vdif_q.F:259-302), runs the
// forward elimination of both the Q2 solve (vdif_q.F:372-378) and the Q2L
// solve (vdif_q.F:398-417), and updates KQ/KM/KH and L, which depend on the
// old Q2/Q2L only (vdif_q.F:466-487; L(1)=KAPPA*L0, L(KB)=0).  The
// elimination coefficients VH of both solves go to the node-layer pair
// scratch `vhs`; VHP(k) is parked in Q2F(k)/Q2LF(k), which the elimination
// has just consumed.  The upward
// sweep does both back-substitutions (vdif_q.F:380-391, 420-431) and the
// threshold (vdif_q.F:440-448), and stores each final value both to
// Q2F/Q2LF and to Q2/Q2L, the copy that follows VDIF_Q in INTERNAL_STEP
// (internal_step.F:1034-1035); column 0 is copied by its thread.  Every value is formed by the reference's
// operations in its order; only the loops are fused.
//
// Bound: the latency of a level's loads where the mesh has few columns, HBM
// where it has many.  So the downward sweep issues the loads of level k+1
// before it works on level k, and the upward sweep takes UP levels' loads at
// once; both loops stay rolled (unrolled to 40 levels the code outgrew the
// instruction cache, and no load could cross a level's branch).  62,500
// elements x 40 layers: 257 -> 173 us; 1,000,000 x 40: 1277 -> 1082 us (4.9 GB,
// 4.5 TB/s; 2 waves a SIMD instead of 3).
template <int RMAX, bool UNI>
__global__ __launch_bounds__(256) void k_vdif_q(DevGrid g, IntArgs a, double2* vhs, const int* only) {
  constexpr int UP = 4;
  const int i = (int)xcd_thread();
  if (i > g.M) return;
  if (only && !only[i]) return;   // column subset (the learned closure's fallback)
  const int KB = g.KB, KBM1 = g.KBM1;
  const double A1 = 0.92, B1 = 16.6, A2 = 0.74, B2 = 10.1, C1 = 0.08, E1 = 1.80, E2 = 1.33, SEF = 1.00;
  const double KAPPA = 0.40, SMALL = 1.E-8, SURFL = 2.E+5;
  double* Q2F = a.q2f; double* Q2LF = a.q2lf; double* L = a.l; double* KM = a.km; double* KH = a.kh; double* KQ = a.kq;
  const long m1 = g.m1;
  if (i == 0) {
    L[NI(g, 0, 1)] = 0.0;
    L[NI(g, 0, KB)] = 0.0;
    for (int k = 1; k <= KB; ++k) {
      const double kn0 = L[NI(g, 0, k)] * sqrt(fabs(a.q2[NI(g, 0, k)] + SMALL));
      KQ[NI(g, 0, k)] = 0.5 * (kn0 * KAPPA * 0.0 + KQ[NI(g, 0, k)]);
      KM[NI(g, 0, k)] = 0.5 * (kn0 * 0.0 + KM[NI(g, 0, k)]);
      KH[NI(g, 0, k)] = 0.5 * (kn0 * 0.0 * g.vprnu + KH[NI(g, 0, k)]);
    }
    for (int k = 1; k <= KB; ++k) {
      a.q2[NI(g, 0, k)] = Q2F[NI(g, 0, k)];
      a.q2l[NI(g, 0, k)] = Q2LF[NI(g, 0, k)];
    }
    return;
  }
  const double dti = g.dti, umol = g.umol, d = a.d[i];
  const int o = g.nbve_off[i], nt = g.ntve[i];
  const double ramp = a.clk->ramp_int;
  double wus = 0.0, wvs = 0.0, wub = 0.0, wvb = 0.0;
  for (int j = 0; j < nt; ++j) {
    const int e = g.nbve[o + j];
    wus = wus + (g.wind_on ? -g.wsx[e] * ramp * 0.001 : 0.0);
    wvs = wvs + (g.wind_on ? -g.wsy[e] * ramp * 0.001 : 0.0);
  }
  const double ntd = (double)nt;
  wus = wus / ntd; wvs = wvs / ntd;
  const double utau2 = sqrt(sq(wus) + sq(wvs));
  const double l0 = SURFL * utau2 / g.grav_n[i];
  for (int j = 0; j < nt; ++j) {
    const int e = g.nbve[o + j];
    wub = wub + a.wubot[e];
    wvb = wvb + a.wvbot[e];
  }
  wub = wub / ntd; wvb = wvb / ntd;
  const double q2f_kb = sqrt(sq(wub) + sq(wvb)) * g.const1;
  Q2F[NI(g, i, KB)] = q2f_kb;
  int re[RMAX];
  static_for<RMAX>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    re[j] = j < nt ? g.nbve[o + j] : 0;
  });
  // ring values loaded unconditionally (slots past the ring read element
  // 0) so that the loads issue together; the sum takes the ring in order
  auto load_ring_uv = [&](int k, double (&ur)[RMAX], double (&vr)[RMAX]) {
    const long eo = (long)(k - 1) * g.n1;
    static_for<RMAX>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      ur[j] = at(a.u + eo, re[j]);
      vr[j] = at(a.v + eo, re[j]);
    });
  };
  auto ring_avg = [&](const double (&fv)[RMAX]) {
    double x = 0.0;
    static_for<RMAX>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if (j < nt) x = x + fv[j];
    });
    return x / ntd;
  };
  auto load_level = [&](int k) {
    Q25Loads<RMAX> r;
    const long ko = (long)(k - 1) * m1;
    r.rho = at(a.rho1 + ko, i);
    r.kq = at(KQ + (ko + m1), i);
    r.q2 = at(a.q2 + ko, i);
    r.q2l = at(a.q2l + ko, i);
    r.km = at(KM + ko, i);
    r.kh = at(KH + ko, i);
    r.q2f = at(Q2F + ko, i);
    r.q2lf = at(Q2LF + ko, i);
    r.dzz = DZZ(i, k - 1);
    r.dz = DZ(i, k);
    r.z = ZN(i, k);
    load_ring_uv(k, r.ur, r.vr);
    return r;
  };
  const double coef4 = 18.0 * A1 * A1 + 9.0 * A1 * A2, coef5 = 9.0 * A1 * A2;
  // stability functions and the under-relaxed mixing coefficients at level k
  auto mix = [&](long q, const Q25Level& lv, double kq_old, double km_old, double kh_old) {
    const double coef1 = A2 * (1.0 - 6.0 * A1 / B1 * lv.stf);
    const double coef2 = 3.0 * A2 * B2 / lv.stf + 18.0 * A1 * A2;
    const double coef3 = A1 * (1.0 - 3.0 * C1 - 6.0 * A1 / B1 * lv.stf);
    const double sh = coef1 / (1.0 - coef2 * lv.gh);
    const double sm = (coef3 + sh * coef4 * lv.gh) / (1. - coef5 * lv.gh);
    const double kn = lv.ll * sqrt(lv.q2);
    KQ[q] = 0.5 * (kn * KAPPA * sm + kq_old);
    KM[q] = 0.5 * (kn * sm + km_old);
    KH[q] = 0.5 * (kn * sh * g.vprnu + kh_old);
    L[q] = lv.ll;
  };
  const double z1 = ZN(i, 1), zkb = ZN(i, KB);
  double vh1p = 0.0, vh2p = 0.0;             // VH(k-1) of the two solves
  const double vhp1_1 = g.cvhp1 * utau2;
  double vhp1 = vhp1_1, vhp2 = 0.0;          // VHP(k-1) of the two solves
  // level 1, and the loads of level 2
  double rho_km1 = a.rho1[NI(g, i, 1)];
  double kq_km1 = KQ[NI(g, i, 1)];           // old KQ(k-1)
  double kq_k = KQ[NI(g, i, 2)];             // old KQ(k)
  double dz_km1 = DZ(i, 1);
  double ukm1 = 0.0, vkm1 = 0.0;
  Q25Loads<RMAX> nx;
  {
    const long q = NI(g, i, 1);
    const double q21 = a.q2[q], q2l1 = a.q2l[q], km1 = KM[q], kh1 = KH[q];
    double ur[RMAX], vr[RMAX];
    load_ring_uv(1, ur, vr);
    nx = load_level(min(2, KBM1));
    __builtin_amdgcn_sched_barrier(0);
    const Q25Level lv = q25_eval(g, i, 1, d, l0, q21, q2l1, 0.0, 0.0, 0.0, 0.0);
    mix(q, lv, kq_km1, km1, kh1);
    if (d > 0.0) { ukm1 = ring_avg(ur); vkm1 = ring_avg(vr); }
  }
  for (int k = 2; k <= KBM1; ++k) {
    const Q25Loads<RMAX> c = nx;
    nx = load_level(min(k + 1, KBM1));   // past the last level: reloads it, unused
    __builtin_amdgcn_sched_barrier(0);
    const long q = (long)(k - 1) * m1 + i;
    const Q25Level lv = q25_eval(g, i, k, d, l0, c.q2, c.q2l, rho_km1, c.rho, c.dzz, c.z);
    // PROD (vdif_q.F:259-302)
    const double boy = lv.boy;
    // the reference's KM*0*x**1.5, x >= 0: zero (or NaN) whatever the power
    double pr = c.km * 0.0 * (.5 * (-boy + fabs(boy)));
    if (d > 0.0) {
      const double uk = ring_avg(c.ur), vk = ring_avg(c.vr);
      pr = pr + c.km * SEF * (sq(uk - ukm1) + sq(vk - vkm1)) / sq(c.dzz * d);
      pr = pr + c.kh * boy;
      ukm1 = uk;
      vkm1 = vk;
    }
    // the threshold before the solves (vdif_q.F:136-145): both to SMALL
    // if either is at or below it
    double q2f = c.q2f, q2lf = c.q2lf;
    if (q2f <= SMALL || q2lf <= SMALL) { q2f = SMALL; q2lf = SMALL; }
    const double ak = -0.5 * dti * (c.kq + kq_k + 2.0 * umol) / (c.dzz * c.dz * d * d);
    const double ck = -0.5 * dti * (kq_km1 + kq_k + 2.0 * umol) / (c.dzz * dz_km1 * d * d);
    const double t1 = 1. / (ak + ck * (1. - vh1p) - (2. * dti * lv.dtef + 1.));
    const double vh1 = ak * t1;
    const double p1 = (-2. * dti * pr + ck * vhp1 - q2f) * t1;
    double vh2, p2;
    if (d > 0.0) {
      const double zk = c.z;
      const double dtef = lv.dtef * (1. + E2 * sq((1. / fabs(zk - z1) + 1. / fabs(zk - zkb)) * lv.ll / (d * KAPPA)));
      const double t2 = 1. / (ak + ck * (1. - vh2p) - (dti * dtef + 1.));
      vh2 = ak * t2;
      p2 = (dti * (-pr * lv.ll * E1) + ck * vhp2 - q2lf) * t2;
    } else {              // D <= 0: VH/VHP keep the first solve's values
      vh2 = vh1;
      p2 = p1;
    }
    vhs[q] = make_double2(vh1, vh2);
    Q2F[q] = p1;
    Q2LF[q] = p2;
    vh1p = vh1;
    vh2p = vh2;
    vhp1 = p1;
    vhp2 = p2;
    mix(q, lv, kq_k, c.km, c.kh);
    rho_km1 = c.rho;
    kq_km1 = kq_k;
    kq_k = c.kq;
    dz_km1 = c.dz;
  }
  {
    // level KB (kq_k is the old KQ(KB) here)
    const long q = NI(g, i, KB);
    const Q25Level lv = q25_eval(g, i, KB, d, l0, a.q2[q], a.q2l[q], 0.0, 0.0, 0.0, 0.0);
    mix(q, lv, kq_k, KM[q], KH[q]);
  }
  // upward sweep: both back-substitutions, then the threshold on each level
  double x1 = q2f_kb, x2 = Q2LF[NI(g, i, KB)];
  a.q2[NI(g, i, KB)] = x1;
  a.q2l[NI(g, i, KB)] = x2;
  for (int kt = KBM1; kt >= 1; kt -= UP) {
    double2 w[UP];
    double p1[UP], p2[UP];
#pragma unroll
    for (int j = 0; j < UP; ++j) {
      const long q = (long)(max(kt - j, 1) - 1) * m1 + i;
      w[j] = vhs[q];
      p1[j] = Q2F[q];
      p2[j] = Q2LF[q];
    }
#pragma unroll
    for (int j = 0; j < UP; ++j) {
      const int k = kt - j;
      if (k < 1) break;
      const long q = (long)(k - 1) * m1 + i;
      if (k == 1) {   // VH(1) = 0, VHP(1) of the two solves
        x1 = 0.0 * x1 + vhp1_1;
        x2 = 0.0 * x2 + 0.0;
      } else {
        x1 = w[j].x * x1 + p1[j];
        x2 = w[j].y * x2 + p2[j];
      }
      double y1 = x1, y2 = x2;
      if (k >= 2 && (x1 <= SMALL || x2 <= SMALL)) { y1 = SMALL; y2 = SMALL; }
      Q2F[q] = y1;
      Q2LF[q] = y2;
      a.q2[q] = y1;
      a.q2l[q] = y2;
    }
  }
}

// VDIF_Q by block of FV_VQN = 16 node columns, for meshes with too few
// columns to fill the chip (vdif_q_blocks of the host side).  Only the two
// eliminations are serial in the level: first all 256 lanes form the ring
// averages of U/V, then the level quantities, PROD and the new KQ/KM/KH and
// L, a lane for a node and every 16th level, into LDS; then one lane for each
// node and solve runs the elimination and back-substitution on LDS; then all
// lanes store the result.  The same operations as k_vdif_q in the same order;
// `vhs` is not needed and VHP is not parked in Q2F/Q2LF.
//
// Bound: latency -- of two rounds of loads, the dependent divisions of the
// elimination (KBM1 of them instead of about 20 KBM1) -- and with many columns
// the instructions, which one lane per column packs better.  Channel of 3,200
// elements x 10 layers: 44 -> 12 us; 17,000 x 20: 80 -> 23; 62,500 x 40: 174 ->
// 113.  512 lanes a block: 109 at 62,500 x 40, but 29 at 17,000 x 20.
template <int RMAX>
__global__ __launch_bounds__(256) void k_vdif_q_blk(DevGrid g, IntArgs a, const int* only) {
  constexpr int NB = FV_VQN, KL = 256 / NB;
  enum { sKQ, sU, sV, sAK, sCK, sC1, sC2, sR1, sR2, sF1, sF2 };
  extern __shared__ double lds[];   // FV_VQARR x KB x NB
  __shared__ double snode[3][NB];   // L0, Q2F(KB), VHP(1) of Q2
  const int t = (int)threadIdx.x, n = t % NB, kl = t / NB;
  const int i0 = xcd_block() * NB + n;
  const bool col = i0 <= g.M && (!only || only[i0]);   // column subset (the learned closure's fallback)
  if (!__syncthreads_or(col)) return;
  const int KB = g.KB, KBM1 = g.KBM1;
  const double A1 = 0.92, B1 = 16.6, A2 = 0.74, B2 = 10.1, C1 = 0.08, E1 = 1.80, E2 = 1.33, SEF = 1.00;
  const double KAPPA = 0.40, SMALL = 1.E-8, SURFL = 2.E+5;
  double* Q2F = a.q2f; double* Q2LF = a.q2lf; double* L = a.l; double* KM = a.km; double* KH = a.kh; double* KQ = a.kq;
  const long m1 = g.m1;
  if (i0 == 0 && col) {
    for (int k = kl + 1; k <= KB; k += KL) {
      const long q = NI(g, 0, k);
      if (k == 1 || k == KB) L[q] = 0.0;
      const double kn0 = (k == 1 || k == KB ? 0.0 : L[q]) * sqrt(fabs(a.q2[q] + SMALL));
      KQ[q] = 0.5 * (kn0 * KAPPA * 0.0 + KQ[q]);
      KM[q] = 0.5 * (kn0 * 0.0 + KM[q]);
      KH[q] = 0.5 * (kn0 * 0.0 * g.vprnu + KH[q]);
      a.q2[q] = Q2F[q];
      a.q2l[q] = Q2LF[q];
    }
  }
  const bool act = col && i0 >= 1;
  const int i = act ? i0 : 1;
  auto S = [&](int v, int k) -> double& { return lds[(v * KB + (k - 1)) * NB + n]; };
  const double dti = g.dti, umol = g.umol, d = a.d[i];
  const int o = g.nbve_off[i], nt = g.ntve[i];
  int re[RMAX];
  static_for<RMAX>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    re[j] = j < nt ? g.nbve[o + j] : 0;
  });
  const double ntd = (double)nt;
  auto ring_sum = [&](const double* p) {   // the ring in order, slots past it read element 0
    double v[RMAX], x = 0.0;
    static_for<RMAX>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      v[j] = at(p, re[j]);
    });
    static_for<RMAX>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if (j < nt) x = x + v[j];
    });
    return x;
  };
  if (act)
    for (int k = kl + 1; k <= KB; k += KL) {
      S(sKQ, k) = at(KQ + (long)(k - 1) * m1, i);
      if (k <= KBM1) {
        S(sU, k) = ring_sum(a.u + (long)(k - 1) * g.n1) / ntd;
        S(sV, k) = ring_sum(a.v + (long)(k - 1) * g.n1) / ntd;
      }
    }
  if (kl == KL - 1) {   // the node's own values
    const double ramp = a.clk->ramp_int;
    double wus = 0.0, wvs = 0.0;
    static_for<RMAX>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      const double wx = at(g.wsx, re[j]), wy = at(g.wsy, re[j]);
      if (j < nt) {
        wus = wus + (g.wind_on ? -wx * ramp * 0.001 : 0.0);
        wvs = wvs + (g.wind_on ? -wy * ramp * 0.001 : 0.0);
      }
    });
    wus = wus / ntd; wvs = wvs / ntd;
    const double utau2 = sqrt(sq(wus) + sq(wvs));
    snode[0][n] = SURFL * utau2 / g.grav_n[i];
    const double wub = ring_sum(a.wubot) / ntd, wvb = ring_sum(a.wvbot) / ntd;
    snode[1][n] = sqrt(sq(wub) + sq(wvb)) * g.const1;
    snode[2][n] = g.cvhp1 * utau2;
  }
  const double coef4 = 18.0 * A1 * A1 + 9.0 * A1 * A2, coef5 = 9.0 * A1 * A2;
  const double z1 = ZN(i, 1), zkb = ZN(i, KB);
  __syncthreads();
  const double l0 = snode[0][n], q2f_kb = snode[1][n], vhp1_1 = snode[2][n];
  if (act)
    for (int k = kl + 1; k <= KB; k += KL) {
      const bool inner = k >= 2 && k <= KBM1;
      const long ko = (long)(k - 1) * m1, kup = inner ? ko - m1 : ko;
      const double rho_km1 = at(a.rho1 + kup, i), rho = at(a.rho1 + ko, i);
      const double q2 = at(a.q2 + ko, i), q2l = at(a.q2l + ko, i), km = at(KM + ko, i), kh = at(KH + ko, i);
      double q2f = at(Q2F + ko, i), q2lf = at(Q2LF + ko, i);
      const double dzz = DZZ(i, inner ? k - 1 : 1), dz = DZ(i, inner ? k : 1), dz_km1 = DZ(i, inner ? k - 1 : 1);
      const double zk = ZN(i, k);
      const double kq_k = S(sKQ, k);
      const Q25Level lv = q25_eval(g, i, k, d, l0, q2, q2l, rho_km1, rho, dzz, zk);
      {
        // stability functions and the under-relaxed mixing coefficients
        const double coef1 = A2 * (1.0 - 6.0 * A1 / B1 * lv.stf);
        const double coef2 = 3.0 * A2 * B2 / lv.stf + 18.0 * A1 * A2;
        const double coef3 = A1 * (1.0 - 3.0 * C1 - 6.0 * A1 / B1 * lv.stf);
        const double sh = coef1 / (1.0 - coef2 * lv.gh);
        const double sm = (coef3 + sh * coef4 * lv.gh) / (1. - coef5 * lv.gh);
        const double kn = lv.ll * sqrt(lv.q2);
        const long q = ko + i;
        KQ[q] = 0.5 * (kn * KAPPA * sm + kq_k);
        KM[q] = 0.5 * (kn * sm + km);
        KH[q] = 0.5 * (kn * sh * g.vprnu + kh);
        L[q] = lv.ll;
      }
      if (!inner) continue;
      // PROD (vdif_q.F:259-302)
      const double boy = lv.boy;
      // the reference's KM*0*x**1.5, x >= 0: zero (or NaN) whatever the power
      double pr = km * 0.0 * (.5 * (-boy + fabs(boy)));
      if (d > 0.0) {
        pr = pr + km * SEF * (sq(S(sU, k) - S(sU, k - 1)) + sq(S(sV, k) - S(sV, k - 1))) / sq(dzz * d);
        pr = pr + kh * boy;
      }
      // the threshold before the solves (vdif_q.F:136-145): both to SMALL
      // if either is at or below it
      if (q2f <= SMALL || q2lf <= SMALL) { q2f = SMALL; q2lf = SMALL; }
      S(sAK, k) = -0.5 * dti * (S(sKQ, k + 1) + kq_k + 2.0 * umol) / (dzz * dz * d * d);
      S(sCK, k) = -0.5 * dti * (S(sKQ, k - 1) + kq_k + 2.0 * umol) / (dzz * dz_km1 * d * d);
      const double c1 = 2. * dti * lv.dtef + 1., r1 = -2. * dti * pr;
      S(sC1, k) = c1;
      S(sR1, k) = r1;
      S(sF1, k) = q2f;
      if (d > 0.0) {
        const double dtef = lv.dtef * (1. + E2 * sq((1. / fabs(zk - z1) + 1. / fabs(zk - zkb)) * lv.ll / (d * KAPPA)));
        S(sC2, k) = dti * dtef + 1.;
        S(sR2, k) = dti * (-pr * lv.ll * E1);
        S(sF2, k) = q2lf;
      } else {              // D <= 0: VH/VHP keep the first solve's values
        S(sC2, k) = c1;
        S(sR2, k) = r1;
        S(sF2, k) = q2f;
      }
    }
  __syncthreads();
  if (act && t < 2 * NB) {
    const int s = t / NB;   // 0: Q2, 1: Q2L
    double vh = 0.0, vhp = s == 0 || !(d > 0.0) ? vhp1_1 : 0.0;
#pragma unroll 4
    for (int k = 2; k <= KBM1; ++k) {
      const double ak = S(sAK, k), ck = S(sCK, k);
      const double t1 = 1. / (ak + ck * (1. - vh) - S(sC1 + s, k));
      vhp = (S(sR1 + s, k) + ck * vhp - S(sF1 + s, k)) * t1;
      vh = ak * t1;
      S(sC1 + s, k) = vh;
      S(sR1 + s, k) = vhp;
    }
    double x = s == 0 ? q2f_kb : Q2LF[NI(g, i, KB)];
#pragma unroll 4
    for (int k = KBM1; k >= 2; --k) {
      x = S(sC1 + s, k) * x + S(sR1 + s, k);
      S(sF1 + s, k) = x;
    }
    S(sF1 + s, 1) = 0.0 * x + (s == 0 ? vhp1_1 : 0.0);   // VH(1) = 0, VHP(1) of the two solves
  }
  __syncthreads();
  if (act)
    for (int k = kl + 1; k <= KB; k += KL) {
      const long q = (long)(k - 1) * m1 + i;
      double y1, y2;
      if (k == KB) {
        y1 = q2f_kb;
        y2 = Q2LF[q];
      } else {
        y1 = S(sF1, k);
        y2 = S(sF2, k);
        if (k >= 2 && (y1 <= SMALL || y2 <= SMALL)) { y1 = SMALL; y2 = SMALL; }
      }
      Q2F[q] = y1;
      Q2LF[q] = y2;
      a.q2[q] = y1;
      a.q2l[q] = y2;
    }
}
