// fvgpu_common.h -- device-side layout shared by the HIP kernels.
//
// All arrays keep the reference's dummy entry 0 and its column-major 3-D
// layout A(0:MT,1:KB): entity index fastest, so a wavefront of consecutive
// nodes/elements at one layer reads consecutive addresses.
#pragma once
#include <hip/hip_runtime.h>
#include <limits.h>
#include <stdint.h>

#include <utility>

#define FV_MAXKB 64
#define FV_MAX_CV 32   // control-volume sub-edges per node (twice the node degree)
#define FV_MAX_RING 16 // NTSN / NTVE bound of the node rings held in registers
#define FV_CVB 128     // elements and nodes per block of the fused CV kernels
#define FV_CVH 256     // a block's nodes with the nodes of their rings
#define FV_NTN 64      // owned nodes per node tile
#define FV_NTE 192     // elements per node tile

// Element blocks of the blocked ADVECTION / ADV_UV kernels: block b owns
// nown[b] (<= 128) elements, its records 0 .. nown[b]-1, followed by the
// other elements of their edges: ns[b] (<= 256) records, element
// elems[256*b + t]; its ne[b] (<= 256) edges edges[256*b + t], with the
// record slots of IA and IB in bits 0-7 and 8-15 of eloc[256*b + t];
// epos[e] packs the edge slots of element e's three edges (in ed_ent
// order) in bits 0-7, 8-15, 16-23, and in bits 24-26 whether e is their IB.
struct UvBlocks {
  int nblk;
  const int *nown, *ns, *elems, *ne, *edges, *eloc, *epos;
};

// The 2-D stage's tables of the element tiles (DevGrid::ub_tile, the same
// blocks as cvb_*), in block order so that a stage reads them directly and
// contiguously: no list length or index has to arrive before the first
// loads go out.  Lanes past a block's entries read a marked pad; n_* are the
// most entries of any block.
//   rec[256*b + t]   the gradient record's element x and its neighbours
//                    NBE; x = e for the block's own element t, ~e for
//                    another element, INT_MIN for a pad
//   edge[256*b + t]  the record slots of IA and IB in bits 0-7 and 8-15, the
//                    node slots of IENODE in bits 16-22 and 23-29, ISBC in
//                    bits 30-31 (3: not 0..2); all ones for a pad
//   egeo[(6*b + q)*256 + t]  XIJC-XC and YIJC-YC of IA, the same of IB,
//                    DLTXC, DLTYC
//   node[FV_CVB*b + t]  {2*node + 1 in the first block that has it, 0, OBC
//                    index or -1, river index or -1}, x = -1 for a pad
//   list[(nslot*b + j)*FV_CVB + t]  the node's cvl_ent list
//   nd[(2*b + q)*FV_CVB + t]  ART1, H
//   elem[FV_CVB*b + t]  {epos, cvb_loc, ISBCE (0 where it is not 0..3) + 4
//                    if it has rivers, IUCP}
//   ed[(12*b + q)*FV_CVB + t]  EPOR, GRAV_E, ART, COR, H1, CC_SPONGE, DLTXE
//                    and DLTYE of the three sub-edges
// a12, art and cc_hvc are DevGrid's.
struct StageTab {
  int n_rec, n_edge, n_node, nslot;
  int4* rec;
  unsigned* edge;
  double* egeo;
  int4* node;
  int* list;
  double* nd;
  int4* elem;
  double* ed;
  const double *a12, *art, *cc_hvc;
};

struct DevGrid {
  int M, N, NE, NCV, KB, KBM1, KBM2, IOBCN, NUMQBC, NTIDE;
  long m1, n1;
  // sigma value of layer k at entity i: a[(k-1)*sk + i*si], one column for
  // all (sk = 1, si = 0) when all node and all element columns are identical
  long nsk, nsi, esk, esi;
  double dte, dti, umol, vprnu, hprnu, cbcmin, min_depth;
  double fact, fm1;         // horizontal mixing closure / constant switches
  double const1, cvhp1;     // 16.6**.6666667*SEF and (15.8*CBCNST)**0.6666667
  int isplit, iramp, noflux_bot, river_ts_specified, type_tsobc, obc_on, obc_elev, wind_on;
  // nodes
  const double *vx, *vy, *h, *art1, *art2, *grav_n, *nn_hvc, *cos_sita, *sin_sita, *phpn;
  const int *isonb, *ntsn, *nbsn_off, *nbsn, *ntve, *nbve_off, *nbve;
  const double *dltxtrie, *dltytrie, *dltxecec, *dltyecec, *dltxnec, *dltynec;
  // elements
  const double *xc, *yc, *art, *h1, *cor, *cc_hvc, *cc_sponge, *cc_z0b, *grav_e, *epor;
  const double *sin_alpha, *cos_alpha, *wsx, *wsy;
  const int *isbce, *iucp, *nv, *nbe;
  const double *awx, *awy;
  const double* a12;               // A1U(e,1..4), A2U(e,1..4) of element e at 8e..8e+7 (64-byte aligned)
  // edges and CV sub-edges
  const int *iec, *ienode, *isbc, *niec;
  const double *xijc, *yijc, *dltxc, *dltyc, *dltxe, *dltye, *dltxncve, *dltyncve;
  // sigma (per column, or one column for all: nsk ..)
  const double *z, *zz, *dz, *dzz, *z1, *zz1, *dz1, *dzz1;
  // gather lists
  // node -> control-volume sub-edges in increasing order, slot-major (entry j
  // of node i at j*m1+i, j < cv_cnt[i]): consecutive nodes read consecutive
  // addresses for each slot.  cvl_ent holds (p<<1 | side), p the
  // element-major position of the sub-edge's flux in the per-layer flux
  // buffers (below).
  int cv_max;
  int ring_max, ve_max;            // max NTSN, max NTVE
  const int *cv_cnt, *cvl_ent;
  // element -> its 3 sub-edges, slot-major (slot j of element e at
  // j*n1+e), slot j being the sub-edge on the element edge from NV(e,j+1)
  // to NV(e,(j+1)%3+1): the sub-edge index, and 1 if its IA is the second
  // of those nodes.  The flux of slot j of element e is stored at position
  // 3*(e-1)+j+1.
  const int *ecv_c, *ecv_swap;
  const double *ecv_dx, *ecv_dy;   // DLTXE/DLTYE of slot j's sub-edge, same layout
  const int *ed_ent;               // element -> 3 x (edge<<1 | side), sorted by edge
  const int *fo_off, *fo_obc;      // element -> FLUXOBN contributions (obc<<1 | slot)
  const int *node_obc;             // node -> OBC index or -1
  const int *node_riv;             // node -> river index or -1
  const int *re_off, *re_riv;      // element -> rivers whose NBVE(1) / NBVE(NTVE) it is
  const int *fct_skip;             // node skipped by FCT (OBC or river node)
  // Element blocks of the fused record + face-flux kernels: block b holds
  // the cvb_ne[b] (<= FV_CVB) elements cvb_elems[FV_CVB*b + t] and the
  // cvb_nn[b] (<= FV_CVB) distinct nodes they use, cvb_nodes[FV_CVB*b + t];
  // cvb_loc[e] packs the local indices of NV(e,1..3) in bits 0-7, 8-15,
  // 16-23.  The nodes whose records other kernels read at every layer (the
  // OBC nodes and the other ends of their sub-edges) are numbered 0 .. nkeep-1
  // in rec_keep[i], -1 at the others.  A pass's records (Pass::rec): node i's
  // of the bottom layer at i, that of number q at layer k at
  // m1 + (k-1)*nkeep + q.  obc_sub[cv_max*n + j]: sub-edge j of OBC node n
  // (2*sub-edge + side, its NTRG, the numbers of its nodes IA and IB), or -1.
  int cvb_nblk, nkeep;
  const int *cvb_nn, *cvb_nodes, *cvb_ne, *cvb_elems, *cvb_loc, *rec_keep;
  const int4* obc_sub;
  // The block's nodes and the nodes of their rings: cvr_nn[b] (<= FV_CVH)
  // distinct, cvr_nodes[FV_CVH*b + q], the block's own first and in the order
  // of cvb_nodes.  Byte j%4 of cvr_loc[(cvr_w*b + j/4)*FV_CVB + t] is the
  // position q of ring slot j of local node t.
  int cvr_w;
  const int *cvr_nn, *cvr_nodes, *cvr_loc;
  StageTab st;
  // Node tiles (VERTVL): tile b owns the nt_nown[b] (<= FV_NTN) nodes
  // nt_nodes[FV_NTN*b + t]; nt_elems[FV_NTE*b + t] are the nt_nel[b]
  // (<= FV_NTE) elements that have one of them as a vertex.  Slot j of
  // owned node i: nt_lpos[j*m1 + i] = (3*local element + element slot) << 1
  // | side, in the order of cvl_ent.
  int nt_nblk;
  const int *nt_nown, *nt_nodes, *nt_nel, *nt_elems, *nt_lpos;
  // Element blocks of the blocked momentum kernels (UvBlocks): the blocks of
  // cvb_* (compact tiles) for the 2-D stage and ADVECTION, runs of
  // consecutive elements for ADV_UV.
  UvBlocks ub_tile, ub_run;
  // OBC / tide / rivers
  const int *i_obc_n, *next_obc, *type_obc, *next_obc2;
  int obc_ore;                     // some OBC node has TYPE_OBC 9/10 (Orlanski)
  double* fobn;                    // the OBC nodes' flux defects where k_ext_fobn forms them, else null
  const double *fluxf_obc, *dltn_obc, *emean, *apt, *phai, *period;
  const int *inodeq;               // node river: its node, else 0
  const int *icellq, *n_icellq;    // edge river: its cell and the two nodes of its solid edge, else 0
  const double *rdisq;             // edge river: the two nodes' shares of its discharge
  const double *qarea, *cos_angleq, *sin_angleq, *qdis0, *tdis, *sdis, *vqdist;
};

// Workgroup index in XCD-contiguous order.  The dispatcher deals consecutive
// workgroups round-robin to the 8 XCDs, each with its own L2; this remap gives
// XCD x one contiguous range of indices, so workgroups over neighbouring mesh
// entities (which gather the same node/element data) share an L2.  It is a
// bijection on [0, gridDim.x).
__device__ __forceinline__ int xcd_block() {
  const int nb = (int)gridDim.x, b = (int)blockIdx.x;
  const int per = nb >> 3, rem = nb & 7, x = b & 7;
  return x * per + (x < rem ? x : rem) + (b >> 3);
}
__device__ __forceinline__ long xcd_thread() { return (long)xcd_block() * blockDim.x + threadIdx.x; }

// The layers of this workgroup's share of [first, last] where a kernel's
// layers are split over gridDim.y (layer_chunks of the host side); k0 > k1:
// none.
__device__ __forceinline__ void layer_share(int first, int last, int& k0, int& k1) {
  const int c = (last - first + (int)gridDim.y) / (int)gridDim.y;
  k0 = first + (int)blockIdx.y * c;
  k1 = min(k0 + c - 1, last);
}

// p[i] where p is the same for every lane and i an entity or flux position:
// the address is the scalar base plus a 32-bit byte offset (no 64-bit lane
// arithmetic).  fvgpu_create refuses meshes whose offsets would not fit.
template <typename T>
__device__ __forceinline__ T at(const T* p, int i) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + (unsigned)i * (unsigned)sizeof(T));
}

// 1-based layer accessors
__device__ __forceinline__ long NI(const DevGrid& g, int i, int k) { return (long)(k - 1) * g.m1 + i; }
__device__ __forceinline__ long EI(const DevGrid& g, int i, int k) { return (long)(k - 1) * g.n1 + i; }
// (by strides, not by a branch, which no other load could cross)
__device__ __forceinline__ double SIGN_(const DevGrid& g, const double* a, int i, int k) {
  return a[(long)(k - 1) * g.nsk + (long)i * g.nsi];
}
__device__ __forceinline__ double SIGE_(const DevGrid& g, const double* a, int i, int k) {
  return a[(long)(k - 1) * g.esk + (long)i * g.esi];
}
// The same in kernels instantiated for identical columns (template parameter
// UNI; the others see this one): a scalar load, which waits for no vector
// load and holds no vector register (1,000,000 elements x 40 layers: ADVECTION
// 819 -> 715 us, ADV_UV 1687 -> 1565, adv_q 616 -> 532, vertvl 390 -> 332).
constexpr bool UNI = false;
template <bool U>
__device__ __forceinline__ double sign_u(const DevGrid& g, const double* a, int i, int k) {
  if constexpr (U) return ((const __attribute__((address_space(4))) double*)a)[k - 1];
  else return SIGN_(g, a, i, k);
}
template <bool U>
__device__ __forceinline__ double sige_u(const DevGrid& g, const double* a, int i, int k) {
  if constexpr (U) return ((const __attribute__((address_space(4))) double*)a)[k - 1];
  else return SIGE_(g, a, i, k);
}
#define DZ(i, k) sign_u<UNI>(g, g.dz, i, k)
#define DZZ(i, k) sign_u<UNI>(g, g.dzz, i, k)
#define ZN(i, k) sign_u<UNI>(g, g.z, i, k)
#define ZZN(i, k) sign_u<UNI>(g, g.zz, i, k)
#define DZ1(i, k) sige_u<UNI>(g, g.dz1, i, k)
#define DZZ1(i, k) sige_u<UNI>(g, g.dzz1, i, k)
#define Z1(i, k) sige_u<UNI>(g, g.z1, i, k)
#define ZZ1(i, k) sige_u<UNI>(g, g.zz1, i, k)
#define NV_(i, j) g.nv[(long)((j)-1) * g.n1 + (i)]
#define NBE_(i, j) g.nbe[(long)((j)-1) * g.n1 + (i)]
#define AWX_(i, j) g.awx[(long)((j)-1) * g.n1 + (i)]
#define AWY_(i, j) g.awy[(long)((j)-1) * g.n1 + (i)]
#define IEC_(e, j) g.iec[(long)((j)-1) * (g.NE + 1) + (e)]
#define IENODE_(e, j) g.ienode[(long)((j)-1) * (g.NE + 1) + (e)]
#define NIEC_(c, j) g.niec[(long)((j)-1) * (g.NCV + 1) + (c)]
#define DLTXNCVE_(c, j) g.dltxncve[(long)((j)-1) * (g.NCV + 1) + (c)]
#define DLTYNCVE_(c, j) g.dltyncve[(long)((j)-1) * (g.NCV + 1) + (c)]

// The least-squares coefficients A1U(e,1..4) and A2U(e,1..4) of element
// e, in the flux type, from the interleaved copy (two 32-byte loads each).
template <typename FT>
__device__ __forceinline__ void lsq_coef(const double* a12, int e, FT (&a1)[4], FT (&a2)[4]) {
  const double4* p = reinterpret_cast<const double4*>(a12) + 2L * e;
  const double4 u = p[0], w = p[1];
  a1[0] = (FT)u.x; a1[1] = (FT)u.y; a1[2] = (FT)u.z; a1[3] = (FT)u.w;
  a2[0] = (FT)w.x; a2[1] = (FT)w.y; a2[2] = (FT)w.z; a2[3] = (FT)w.w;
}

__device__ __forceinline__ double fsign1(double b) { return b >= 0.0 ? 1.0 : -1.0; }
__device__ __forceinline__ float fsign1(float b) { return b >= 0.0f ? 1.0f : -1.0f; }
// x, negated where bit 0 of m is set
__device__ __forceinline__ double flip_sign(double x, int m) {
  return __hiloint2double(__double2hiint(x) ^ (m << 31), __double2loint(x));
}
__device__ __forceinline__ double sq(double x) { return x * x; }
__device__ __forceinline__ float sq(float x) { return x * x; }

// Whether river j's discharge enters node i, and its share there: all of
// it at a node river's node (INODEQ), RDISQ(J,1) / RDISQ(J,2) at the two
// nodes of an edge river's solid edge (N_ICELLQ).  A node river's share is
// exactly 1, so QDIS*share is QDIS bit for bit.
__device__ __forceinline__ bool river_share(const DevGrid& g, int j, int i, double& w) {
  if (g.inodeq[j] == i) { w = 1.0; return true; }
  if (g.icellq[j] > 0) {
    if (g.n_icellq[j] == i) { w = g.rdisq[j]; return true; }
    if (g.n_icellq[g.NUMQBC + j] == i) { w = g.rdisq[g.NUMQBC + j]; return true; }
  }
  return false;
}

// Device clock: the time-dependent scalars of the current step, written by
// tiny kernels so that a captured graph replays correctly.
struct DevClock {
  long long iint;
  double ramp_int;      // RAMP of INTERNAL_STEP
  double time0, dti, dte;
  int isplit, iramp;
  int depth_fail;
  int pad;
};

// Compile-time loop: f(std::integral_constant<int, K>) for K = 0..N-1, fully
// expanded so that register arrays are indexed by constants.
template <typename F, int... Ks>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, Ks...>) {
  (f(std::integral_constant<int, Ks>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Host-side choice of the register-array bound KMAX >= KBM1 for the
// column kernels templated on it.
#define FV_KMAX_DISPATCH(KBM1, CALL)                 \
  do {                                               \
    if ((KBM1) <= 8) { CALL(8); }                    \
    else if ((KBM1) <= 16) { CALL(16); }             \
    else if ((KBM1) <= 24) { CALL(24); }             \
    else if ((KBM1) <= 32) { CALL(32); }             \
    else if ((KBM1) <= 40) { CALL(40); }             \
    else if ((KBM1) <= 48) { CALL(48); }             \
    else { CALL(64); }                               \
  } while (0)

// Host-side choice of the per-node sub-edge bound SMAX >= cv_max.
#define FV_SMAX_DISPATCH(SMAX_, CALL)                \
  do {                                               \
    if ((SMAX_) <= 16) { CALL(16); }                 \
    else if ((SMAX_) <= 24) { CALL(24); }            \
    else { CALL(32); }                               \
  } while (0)

// Host-side choice of the node-ring bound RMAX >= ring_max (NTSN or NTVE).
#define FV_RMAX_DISPATCH(RM_, CALL)                  \
  do {                                               \
    if ((RM_) <= 10) { CALL(10); }                   \
    else { CALL(16); }                               \
  } while (0)
