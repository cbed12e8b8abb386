// fdm_kernels.hpp -- device kernels of the time-stepping path.
//
//   edge_kernel  : one lane per boundary node or interface node.  Boundary
//                  hats (set_bc_mode2), locked interface hats, and for
//                  frictional interfaces the fault-rate scaling, the
//                  rate-and-state solve, hats, state rates and the fault RK
//                  update, all in FP64.
//   bulk_kernel  : one lane per grid point.  DF <- A*DF, SAT penalties,
//                  SBP2/4/6 stencils with curvilinear metrics, szz overwrite,
//                  sources, F <- F + B*dt*DF and (last stage) the
//                  Drucker-Prager return map.  Templated on the storage
//                  type T of fields/rates/metrics (double, or float for the
//                  FP32-bulk mode).
#pragma once

#include "fdm_physics.hpp"

namespace fdm {

struct BlockDev {
  int mx, px, my, py;
  int plastic, mms, id, pad;
  double rho, G, M, gamma, nu;
  double cI[5][3];  // interior coefficients DI(s)/rho, DI(s)*M, DI(s)*G, s = 1..3 (rates.f90:400-405)
  double mu, beta, b, h, eta, K;
  double s0[6];
  int side_off[4], side_n[4], side_bc[4];
  // FP32-bulk stores each field as its deviation from this per-block
  // constant (zero in FP64); totals are formed in FP64 where needed
  double Fb[6];
  // artificial dissipation (rates.f90:1397-2021): Cdiss as the rates use it
  // (0: none) and the interior weights d(0) = 2 AI(0) Cdiss, d(s) =
  // AI(s) Cdiss (rates.f90:1416-1421)
  double Cdiss;
  double dA[3];
  // perfectly matched layer (rates.f90:2024-2619): pmlx/pmly are zero unless
  // the layer is in effect (mode 2, no dissipation in the block); pml = n,
  // sigma, kappa, mx, px, my, py; phx/phy: Ji*yr and Ji*xq at the first
  // point of each of the block's nine regions, index 3*ry + rx with rx, ry
  // 0 (minus-side closure), 1 (interior), 2 (plus-side closure)
  int pmlx, pmly;
  double pml[7];
  double phx[9], phy[9];
  // FP32-delta metrics (FP64 contexts): xq, xr, yq, yr of a point of this
  // block are mbase[q] + (double)d with d the stored FP32 delta, exactly; a
  // NaN delta sends the reader to the FP64 plane
  double mbase[4];
};

struct IfaceDev {
  int direction, bm, bp, m, p, coupling, law, reg, rup_field, node_off, n, pad;
  double rup_threshold, skempton, flock, ld_T;
  // kinematic forcing: c0, fd, dfdx, vL, vR, xL, xR, tmax
  int force, pad2;
  double kn[8];
};

struct SourcePlaceDev {
  int block, i0, j0, pad;
  double dx[5], dy[5];
};

// concatenated per-node arrays of all block sides; component-major, stride NS
struct SidesDev {
  const double* M;       // [5][NS]
  const double* normal;  // [2][NS]
  const double* F0;      // [6][NS]
  const double* x;       // [NS] (may be null)
  const double* y;
  double* Fhat;          // [6][NS]
  int NS;
};

// concatenated per-node arrays of all interfaces; component-major, stride NI
struct IfacesDev {
  const IfaceDev* tab;
  const double* nhat;    // [2][NI]
  const double* rs;      // [7][NI]
  const double* sw;      // [4][NI]
  const double* S0b;     // [NI]
  const double* N0b;
  const double* ldS;
  const double* ldN;
  const int* outside;
  const double* knx;     // [NI] distance along the fault (kinematic forcing)
  double* st;            // [18][NI] fault state (FDM_IF_* order)
  double* st1;           // [18][NI] stage-1 snapshot
  int NI;
};

// One edge node, resolved at fdm_create: a boundary node of a block side
// (iface = -1; ccm, som, bm: its point, side node and block; bc, id the
// side's condition and the block's number) or an interface node (both
// sides' points, side nodes and blocks; q its index in the interface
// arrays).  A lane's loads depend on this record alone, not on a chain of
// task, block and side tables.
struct EdgeNode {
  int iface, q;       // boundary: -1, -1
  unsigned ccm, ccp;  // boundary: point, unused
  int som, sop;       // boundary: side node, bc
  int bm, bp;         // boundary: block, block number
};

// Rim groups (see the band section of fdm_bulk.hpp): the most edge nodes of a
// group, one wave of boundary nodes, fewer where some are interface nodes
// (their staged values take the same LDS), and the stride of its points
constexpr int kRimNodes = 64, kRimIface = 24, kRimPts = 64;

// On whole lines of the scalar cache in a stage kernel's argument segment: 8
// bytes off them, a stage of 401^2 points took 13.9 us against 13.7.
template <typename T>
struct alignas(64) EdgeArgs {
  const T* F;
  int ld;
  long long ps;
  const EdgeNode* nodes;
  int ntasks;
  // rim groups of the stage launch: (nodes, points, has an interface node,
  // 0); nodes and points of group g at kRimNodes g and kRimPts g
  const int4* rim;
  const EdgeNode* rimnodes;
  const struct RimPt* rimpts;
  const BlockDev* blocks;
  SidesDev sd;
  IfacesDev fi;
  double t, Bdt, A, Bload;
  int do_scale, do_update, snapshot;
  int* fail;
  // graph replays: when set, the stage time is formed on the device from the
  // step index *nstep as (t_init + (nstep - 1) dt) + rkc dt, the expression
  // the host uses, instead of t
  const long long* nstep;
  double t_init, dt, rkc;
  // when set, [3][NI]: slip velocity, state variable at the start of the
  // stage and normal stress of every frictional node (adjoint trajectories)
  double* trace;
};

template <typename T>
__device__ __forceinline__ double stage_time(const EdgeArgs<T>& a) {
  if (!a.nstep) return a.t;
  const double t0 = a.t_init + (double)(*a.nstep - 1) * a.dt;
  return t0 + a.rkc * a.dt;
}

// The values of one edge node, read at their point of use from a source SRC:
// rows of kNodeRow* by node.  A boundary node uses the first rows alone.
enum {
  kRowFm = 0, kRowF0m = 6, kRowN = 12, kRowMm = 14,  // F, F0, normal, Zs Zp gamma: boundary node or minus side
  kNodeRowsBnd = 17,
  kRowFp = 17, kRowF0p = 23, kRowMp = 29,  // plus side
  kRowS0 = 32, kRowN0 = 33, kRowOut = 34,  // loaded prestress, outside flag
  kRowSt = 35,                             // fault arrays, in the order of kNodeSt
  kRowRs = 50,
  kNodeRows = 57
};
constexpr int kNodeStRows = 15;
__device__ constexpr int kNodeSt[kNodeStRows] = {
    FDM_IF_PSI, FDM_IF_V, FDM_IF_S, FDM_IF_N, FDM_IF_NREG, FDM_IF_D, FDM_IF_DDS, FDM_IF_DDN, FDM_IF_DPSI,
    FDM_IF_DW, FDM_IF_DNREG, FDM_IF_TRUP, FDM_IF_DS, FDM_IF_DN, FDM_IF_W};
enum { kStPsi = 0, kStV, kStS, kStN, kStNreg, kStD, kStDDS, kStDDN, kStDPsi, kStDW, kStDNreg, kStTrup, kStDS, kStDN, kStW };

// row r of a node from the arrays themselves; the fields come as totals (the
// FP32-bulk background added).  r is a constant at every call.
template <typename T>
__device__ __forceinline__ double node_row(const EdgeArgs<T>& a, const EdgeNode& nd, const int r) {
  const int NS = a.sd.NS, NI = a.fi.NI, q = nd.q;
  if (r < kRowF0m) {
    const double v = (double)a.F[r * a.ps + nd.ccm];
    if constexpr (sizeof(T) == 4) return v + a.blocks[nd.bm].Fb[r];
    return v;
  }
  if (r < kRowN) return a.sd.F0[(r - kRowF0m) * NS + nd.som];
  if (r < kRowMm) {
    const int k = r - kRowN;
    return nd.iface < 0 ? a.sd.normal[k * NS + nd.som] : a.fi.nhat[(long long)k * NI + q];
  }
  if (r < kRowFp) return a.sd.M[(r - kRowMm) * NS + nd.som];
  if (r < kRowF0p) {
    const double v = (double)a.F[(r - kRowFp) * a.ps + nd.ccp];
    if constexpr (sizeof(T) == 4) return v + a.blocks[nd.bp].Fb[r - kRowFp];
    return v;
  }
  if (r < kRowMp) return a.sd.F0[(r - kRowF0p) * NS + nd.sop];
  if (r < kRowS0) return a.sd.M[(r - kRowMp) * NS + nd.sop];
  // load_stress (friction.f90:1335-1374) with the ramp B(t) precomputed
  if (r == kRowS0) return a.fi.S0b[q] + a.fi.ldS[q] * a.Bload;
  if (r == kRowN0) return a.fi.N0b[q] + a.fi.ldN[q] * a.Bload;
  if (r == kRowOut) return (double)a.fi.outside[q];
  if (r < kRowRs) return a.fi.st[(long long)kNodeSt[r - kRowSt] * NI + q];
  return a.fi.rs[(long long)(r - kRowRs) * NI + q];
}

// sources: the arrays (edge kernels of their own), or rows staged in LDS
// with the given stride (rim groups)
// fence(): a source in LDS is read at its uses and not ahead of the fault
// solve, whose registers are the kernel's most; put() keeps a value in a
// row that is not read again (the arrays have no such place: values stay in
// registers)
template <typename T>
struct NodeArrays {
  static constexpr bool kPut = false;
  const EdgeArgs<T>& a;
  const EdgeNode& nd;
  __device__ __forceinline__ double operator()(int r) const { return node_row<T>(a, nd, r); }
  __device__ __forceinline__ void put(int, double) const {}
  __device__ __forceinline__ void fence() const {}
};
struct NodeRows {
  static constexpr bool kPut = true;
  double* s;
  int stride;
  __device__ __forceinline__ double operator()(int r) const { return s[r * stride]; }
  __device__ __forceinline__ void put(int r, double v) const { s[r * stride] = v; }
  __device__ __forceinline__ void fence() const { asm volatile("" ::: "memory"); }
};

// what the friction solve leaves for the rest of the node's stage
struct FaultSolved {
  double V, S, O, N, Nreg, E, fS0, fN0;
};

// The fault node after load_stress: the friction solve under the hat
// tractions phis, phip and the total prestress fS0, fN0 (solve_friction,
// friction.f90:655-826), for both modes.
template <typename T, bool FORCE, typename SRC>
__device__ __forceinline__ void fault_solve(const EdgeArgs<T>& a, const IfaceDev& I, const int q, const SRC& src,
                                            const double phip, const double phis, const double etas,
                                            const double tst, FaultSolved& f) {
  const int NI = a.fi.NI;
  const int law = I.law;
  double rs[7], sw[4];
  rs[0] = law >= FDM_LAW_SL ? src(kRowRs) : 1.0;
  rs[2] = law >= FDM_LAW_SL ? src(kRowRs + 2) : 1.0;
#pragma unroll
  for (int c = 0; c < 4; c++) sw[c] = law == FDM_LAW_SW ? a.fi.sw[(long long)c * NI + q] : 1.0;
  const double Psi = src(kRowSt + kStPsi), D = src(kRowSt + kStD);
  f.V = src(kRowSt + kStV);
  f.Nreg = src(kRowSt + kStNreg);
  f.S = src(kRowSt + kStS);
  f.N = src(kRowSt + kStN);
  // exp(Psi/a) of the regularised laws, shared by every strength
  // evaluation of the Newton solve and by the state rate
  f.E = law >= FDM_LAW_RSL ? exp(Psi / rs[0]) : 0.0;
  const int force = FORCE ? I.force : 0;
  const double kf = force ? kinematic_friction(I.kn, a.fi.knx[q], tst) : 0.0;
  const bool fail = solve_friction_core(law, rs, sw, I.reg, src(kRowOut) != 0.0, I.flock, f.fS0, f.fN0, phip, phis,
                                        etas, D, Psi, f.E, I.skempton, a.Bdt, f.V, f.S, f.O, f.N, f.Nreg, force,
                                        force ? I.kn[0] : 0.0, kf);
  if (fail) *a.fail = 1;
}

// The rest of a fault node's stage, off the chain from its fields to its
// hats: the fault rates (set_rates_friction, friction.f90:1101-1124), their
// RK update (scale_rates_friction, update_fields_friction, friction.f90:
// 555-590), the stage-1 snapshot and the trace.
template <typename T, typename SRC>
__device__ __forceinline__ void fault_update(const EdgeArgs<T>& a, const IfaceDev& I, const int q, const SRC& src,
                                             const FaultSolved& f, const double tst) {
  const int NI = a.fi.NI;
  double* __restrict__ st = a.fi.st;
  double* __restrict__ s1 = a.fi.st1;
  const int law = I.law;
  const double V = f.V, S = f.S, N = f.N, Nreg = f.Nreg;
  const double Psi = src(kRowSt + kStPsi), D = src(kRowSt + kStD);
  if (a.trace) {
    a.trace[q] = V;
    a.trace[NI + q] = Psi;
    a.trace[2 * NI + q] = N;
  }
  const double Bdt = a.Bdt;
#define PUT(k, v) st[(long long)(k) * NI + q] = (v)
#define SNAP(k, v) if (a.snapshot) s1[(long long)(k) * NI + q] = (v)
#define SCALED(r) (a.do_scale ? a.A * src(kRowSt + (r)) : src(kRowSt + (r)))
  PUT(FDM_IF_S0, f.fS0);
  PUT(FDM_IF_N0, f.fN0);
  PUT(FDM_IF_V, V);
  PUT(FDM_IF_S, S);
  PUT(FDM_IF_O, f.O);
  PUT(FDM_IF_N, N);
  SNAP(FDM_IF_S0, f.fS0);
  SNAP(FDM_IF_N0, f.fN0);
  SNAP(FDM_IF_V, V);
  SNAP(FDM_IF_S, S);
  SNAP(FDM_IF_O, f.O);
  SNAP(FDM_IF_N, N);
  SNAP(FDM_IF_NREG, Nreg);
  SNAP(FDM_IF_PSI, Psi);
  SNAP(FDM_IF_D, D);
  const double dDS = SCALED(kStDDS) + V;
  const double dDN = SCALED(kStDDN) + f.O;
  PUT(FDM_IF_DDS, dDS);
  PUT(FDM_IF_DDN, dDN);
  SNAP(FDM_IF_DDS, dDS);
  SNAP(FDM_IF_DDN, dDN);
  const double dW = SCALED(kStDW) + S * V;
  PUT(FDM_IF_DW, dW);
  SNAP(FDM_IF_DW, dW);
  const bool ruptured = I.rup_field == 1 ? (D > I.rup_threshold) : (fabs(V) > I.rup_threshold);
  double trup = src(kRowSt + kStTrup);
  if (ruptured) {
    trup = fmin(trup, tst);
    PUT(FDM_IF_TRUP, trup);
  }
  SNAP(FDM_IF_TRUP, trup);
  const double DS = src(kRowSt + kStDS), DN = src(kRowSt + kStDN), W = src(kRowSt + kStW);
  SNAP(FDM_IF_DS, DS);
  SNAP(FDM_IF_DN, DN);
  SNAP(FDM_IF_W, W);
  if (a.do_update) {
    PUT(FDM_IF_DS, DS + Bdt * dDS);
    PUT(FDM_IF_DN, DN + Bdt * dDN);
    PUT(FDM_IF_D, D + Bdt * fabs(dDS));
    PUT(FDM_IF_W, W + Bdt * dW);
  }
  src.fence();
  double rs[7];
#pragma unroll
  for (int c = 0; c < 7; c++) rs[c] = law >= FDM_LAW_SL ? src(kRowRs + c) : 1.0;
  const double dPsi = SCALED(kStDPsi) + state_rate(law, rs, V, Psi, f.E);
  PUT(FDM_IF_DPSI, dPsi);
  SNAP(FDM_IF_DPSI, dPsi);
  double dNreg = SCALED(kStDNreg);
  if (I.reg) {
    const double absV = fabs(V);
    const double Nr = -(absV / rs[4]) * (Nreg - fmax(N, 0.0));
    dNreg = dNreg + Nr;
  }
  PUT(FDM_IF_DNREG, dNreg);
  SNAP(FDM_IF_DNREG, dNreg);
  if (a.do_update) {
    PUT(FDM_IF_PSI, Psi + Bdt * dPsi);
    PUT(FDM_IF_NREG, Nreg + Bdt * dNreg);
  } else {
    PUT(FDM_IF_NREG, Nreg);
  }
#undef PUT
#undef SNAP
#undef SCALED
}

// interface node in antiplane shear: locked_interface_mode3
// (interfaces.f90:676-712), or frictional_interface_mode3 (interfaces.f90:
// 806-897).  The normal stress is the plus block's in-plane prestress
// resolved on the fault (rotate_xy2nt_mat, geometry.f90:311-322), the stress
// transfer phip is zero, and the initial fields arrive in their own order
// (interfaces.f90:798).
template <typename T, bool FORCE, typename SRC>
__device__ __forceinline__ void iface_node3(const EdgeArgs<T>& a, const EdgeNode& nd, const IfaceDev& I,
                                            const SRC& src, const double tst, double (&Fhm)[6], double (&Fhp)[6],
                                            FaultSolved& f) {
  double Fm[3], Fp[3], F0m[3], F0p[3];
#pragma unroll
  for (int l = 0; l < 3; l++) {
    Fm[l] = src(kRowFm + l);
    Fp[l] = src(kRowFp + l);
  }
  const double n1 = src(kRowN), n2 = src(kRowN + 1), Zsm = src(kRowMm), Zsp = src(kRowMp);
  if (I.coupling == FDM_COUPLING_LOCKED) {
    locked_interface_mode3(Fhm, Fhp, Fm, Fp, n1, n2, Zsm, Zsp);
    return;
  }
  const BlockDev& Bp = a.blocks[nd.bp];
#pragma unroll
  for (int l = 0; l < 3; l++) {
    F0m[l] = src(kRowF0m + l);
    F0p[l] = src(kRowF0p + l);
  }
  double vz0p, stz0p, snz0p;
  xy2nt3(F0p, n1, n2, vz0p, stz0p, snz0p);
  double dp[3], dm[3];
#pragma unroll
  for (int l = 0; l < 3; l++) {
    dp[l] = Fp[l] - F0p[l];
    dm[l] = Fm[l] - F0m[l];
  }
  double vzFDp, stzFDp, snzFDp, vzFDm, stzFDm, snzFDm;
  xy2nt3(dp, n1, n2, vzFDp, stzFDp, snzFDp);
  xy2nt3(dm, n1, n2, vzFDm, stzFDm, snzFDm);
  const double Zsip = 1.0 / Zsp, Zsim = 1.0 / Zsm;
  const double etas = 1.0 / (Zsip + Zsim);
  const double phis = etas * (snzFDp * Zsip + snzFDm * Zsim + vzFDp - vzFDm);
  const double S0 = snz0p;
  const double snn = 2.0 * n1 * n2 * Bp.s0[1] + n1 * n1 * Bp.s0[0] + n2 * n2 * Bp.s0[3];
  const double N0 = -snn - 0.0;
  f.fS0 = src(kRowS0) + S0;
  f.fN0 = src(kRowN0) + N0;
  src.fence();
  fault_solve<T, FORCE>(a, I, nd.q, src, 0.0, phis, etas, tst, f);
  src.fence();
  const double snzp = f.S - f.fS0, snzm = f.S - f.fS0;
  const double vzp = vzFDp + Zsip * (snzFDp - snzp);
  const double vzm = vzFDm - Zsim * (snzFDm - snzm);
  nt2xy3(Fhp, n1, n2, vzp, stzFDp, snzp);
  nt2xy3(Fhm, n1, n2, vzm, stzFDm, snzm);
#pragma unroll
  for (int l = 0; l < 3; l++) {
    Fhp[l] = Fhp[l] + src(kRowF0p + l);
    Fhm[l] = Fhm[l] + src(kRowF0m + l);
  }
}

// interface node in plane strain (interfaces.f90:520-1012)
template <typename T, bool FORCE, typename SRC>
__device__ __forceinline__ void iface_node2(const EdgeArgs<T>& a, const EdgeNode& nd, const IfaceDev& I,
                                            const SRC& src, const double tst, double (&Fhm)[6], double (&Fhp)[6],
                                            FaultSolved& f) {
  double n1 = src(kRowN), n2 = src(kRowN + 1);
  if (I.coupling == FDM_COUPLING_LOCKED) {
    double Fm[6], Fp[6];
#pragma unroll
    for (int l = 0; l < 6; l++) {
      Fm[l] = src(kRowFm + l);
      Fp[l] = src(kRowFp + l);
    }
    locked_interface_mode2(Fhm, Fhp, Fm, Fp, n1, n2, src(kRowMm), src(kRowMp), src(kRowMm + 1), src(kRowMp + 1),
                           src(kRowMm + 2), src(kRowMp + 2));
    return;
  }
  // frictional_interface_mode2 (interfaces.f90:900-1012).  The reference
  // passes the minus-side initial fields to its dummy "F0p" and the
  // plus-side ones to "F0m" (interfaces.f90:795 vs :900); kept as is.
  NT p0, p, m;
  {
    double dF0p[6], d[6];
#pragma unroll
    for (int l = 0; l < 6; l++) dF0p[l] = src(kRowF0m + l);
    p0 = xy2nt(dF0p, n1, n2);
#pragma unroll
    for (int l = 0; l < 6; l++) d[l] = src(kRowFp + l) - dF0p[l];
    p = xy2nt(d, n1, n2);
#pragma unroll
    for (int l = 0; l < 6; l++) d[l] = src(kRowFm + l) - src(kRowF0p + l);
    m = xy2nt(d, n1, n2);
  }
  double Zsip = 1.0 / src(kRowMp), Zsim = 1.0 / src(kRowMm);
  double Zpip = 1.0 / src(kRowMp + 1), Zpim = 1.0 / src(kRowMm + 1);
  const double etas = 1.0 / (Zsip + Zsim);
  const double phis = etas * (p.snt * Zsip + m.snt * Zsim + p.vt - m.vt);
  const double etap = 1.0 / (Zpip + Zpim);
  const double phip = etap * (p.snn * Zpip + m.snn * Zpim + p.vn - m.vn);
  const double S0 = p0.snt;
  const double N0 = -p0.snn - 0.0;
  f.fS0 = src(kRowS0) + S0;
  f.fN0 = src(kRowN0) + N0;
  if constexpr (SRC::kPut) {
    // the rotated fields wait in the rows of the fields themselves
    const double w[12] = {p.vt, p.vn, p.stt, p.snt, p.snn, p.szz, m.vt, m.vn, m.stt, m.snt, m.snn, m.szz};
#pragma unroll
    for (int k = 0; k < 6; k++) {
      src.put(kRowFm + k, w[k]);
      src.put(kRowFp + k, w[6 + k]);
    }
    src.put(kRowMm, Zsim);
    src.put(kRowMm + 1, Zpim);
    src.put(kRowMp, Zsip);
    src.put(kRowMp + 1, Zpip);
  }
  src.fence();
  fault_solve<T, FORCE>(a, I, nd.q, src, phip, phis, etas, tst, f);
  src.fence();
  if constexpr (SRC::kPut) {
    p = NT{src(kRowFm), src(kRowFm + 1), src(kRowFm + 2), src(kRowFm + 3), src(kRowFm + 4), src(kRowFm + 5)};
    m = NT{src(kRowFp), src(kRowFp + 1), src(kRowFp + 2), src(kRowFp + 3), src(kRowFp + 4), src(kRowFp + 5)};
    Zsim = src(kRowMm);
    Zpim = src(kRowMm + 1);
    Zsip = src(kRowMp);
    Zpip = src(kRowMp + 1);
    n1 = src(kRowN);
    n2 = src(kRowN + 1);
  }
  const double gm = src(kRowMm + 2), gp = src(kRowMp + 2);
  const double skm = 1.0 - I.skempton;
  const double snnp = -(f.N - f.fN0) / skm;
  const double snnm = -(f.N - f.fN0) / skm;
  const double vnp = p.vn + Zpip * (p.snn - snnp);
  const double vnm = m.vn - Zpim * (m.snn - snnm);
  const double sttp = p.stt - gp * (p.snn - snnp);
  const double sttm = m.stt - gm * (m.snn - snnm);
  const double szzp = p.szz - gp * (p.snn - snnp);
  const double szzm = m.szz - gm * (m.snn - snnm);
  const double sntp = f.S - f.fS0;
  const double sntm = f.S - f.fS0;
  const double vtp = p.vt + Zsip * (p.snt - sntp);
  const double vtm = m.vt - Zsim * (m.snt - sntm);
  nt2xy(Fhp, n1, n2, vtp, vnp, sttp, sntp, snnp, szzp);
  nt2xy(Fhm, n1, n2, vtm, vnm, sttm, sntm, snnm, szzm);
#pragma unroll
  for (int l = 0; l < 6; l++) {
    Fhp[l] = Fhp[l] + src(kRowF0m + l);
    Fhm[l] = Fhm[l] + src(kRowF0p + l);
  }
}

// The hats of one edge node, as stored (FP32-bulk: less the block's
// background): Fhm of its minus side (a boundary node's only one), Fhp of
// its plus side.  MODE 2 or 3: each kernel carries the code of one mode
// only; FORCE = false leaves out kinematic forcing, MMS = false the
// manufactured solution's boundary data (whose registers would set the
// kernel's).
template <typename T, int MODE, bool FORCE, bool MMS, typename SRC>
__device__ __forceinline__ void edge_node(const EdgeArgs<T>& a, const EdgeNode& nd, const SRC& src,
                                          double (&Fhm)[6], double (&Fhp)[6], FaultSolved& f) {
  constexpr int NF = MODE == 3 ? 3 : 6;
  const double tst = stage_time(a);
  if (nd.iface < 0) {
    // boundary node (boundaries.f90:106-129)
    double F[NF], F0[NF];
#pragma unroll
    for (int l = 0; l < NF; l++) {
      F[l] = src(kRowFm + l);
      F0[l] = src(kRowF0m + l);
    }
    const double n1 = src(kRowN), n2 = src(kRowN + 1), Zs = src(kRowMm);
    if constexpr (MODE == 3) {
      // set_bc_mode3 (boundaries.f90:148-149, 155-213)
      set_bc_mode3(Fhm, F, F0, n1, n2, nd.sop, Zs);
    } else {
      const bool xy = MMS && nd.sop == FDM_BC_MMS_SIN_W;
      const double x = xy ? a.sd.x[nd.som] : 0.0, y = xy ? a.sd.y[nd.som] : 0.0;
      set_bc_mode2<MMS>(Fhm, F, F0, n1, n2, nd.sop, Zs, src(kRowMm + 1), src(kRowMm + 2), x, y, tst, nd.bp);
    }
  } else {
    const IfaceDev& I = a.fi.tab[nd.iface];
    if constexpr (MODE == 3) iface_node3<T, FORCE>(a, nd, I, src, tst, Fhm, Fhp, f);
    else iface_node2<T, FORCE>(a, nd, I, src, tst, Fhm, Fhp, f);
    if constexpr (sizeof(T) == 4) {
      const BlockDev& Bp = a.blocks[nd.bp];
#pragma unroll
      for (int l = 0; l < NF; l++) Fhp[l] = Fhp[l] - Bp.Fb[l];
    }
  }
  if constexpr (sizeof(T) == 4) {
    const BlockDev& Bm = a.blocks[nd.bm];
#pragma unroll
    for (int l = 0; l < NF; l++) Fhm[l] = Fhm[l] - Bm.Fb[l];
  }
}

// what edge_node leaves of a frictional node's stage
template <typename T, typename SRC>
__device__ __forceinline__ void edge_finish(const EdgeArgs<T>& a, const EdgeNode& nd, const SRC& src,
                                            const FaultSolved& f) {
  if (nd.iface < 0) return;
  const IfaceDev& I = a.fi.tab[nd.iface];
  if (I.coupling != FDM_COUPLING_LOCKED) fault_update<T>(a, I, nd.q, src, f, stage_time(a));
}

// the hats to the side arrays, where the per-point kernels read them
template <typename T, int MODE, bool FORCE>
__device__ __forceinline__ void edge_store(const EdgeArgs<T>& a, const EdgeNode& nd) {
  constexpr int NF = MODE == 3 ? 3 : 6;
  const int NS = a.sd.NS;
  double Fhm[6], Fhp[6];
  FaultSolved f;
  edge_node<T, MODE, FORCE, true>(a, nd, NodeArrays<T>{a, nd}, Fhm, Fhp, f);
  edge_finish<T>(a, nd, NodeArrays<T>{a, nd}, f);
#pragma unroll
  for (int l = 0; l < NF; l++) a.sd.Fhat[l * NS + nd.som] = Fhm[l];
  if (nd.iface >= 0) {
#pragma unroll
    for (int l = 0; l < NF; l++) a.sd.Fhat[l * NS + nd.sop] = Fhp[l];
  }
}

template <typename T, int MODE, bool FORCE>
__global__ void __launch_bounds__(64) edge_kernel(EdgeArgs<T> a) {
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= a.ntasks) return;
  edge_store<T, MODE, FORCE>(a, a.nodes[tid]);
}

}  // namespace fdm
