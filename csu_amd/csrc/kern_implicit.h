// kern_implicit.h -- implicit time stepping: LU-SGS by level scheduling and
// DPLUR by damped Jacobi (reference implicit.c).
//
// LU-SGS: the reference sweeps cells in index order, a cell using the final
// increments of its lower-index (forward) or higher-index (backward)
// neighbours.  The host groups cells into levels of that dependency DAG; each
// level is one launch, cells of a level are independent.  Every cell does the
// reference's arithmetic on the same inputs, so the result equals the serial
// sweep for any cell order; a colour-sorted numbering makes the number of
// levels equal to the number of colours.
#pragma once
#include "kern_common.h"

namespace csu {

__device__ __forceinline__ double gamma_of(const GasD& g, double T) { return gas_T2gamma<double>(g, T); }

// Four lanes of a wavefront work on one cell, a lane per face slot, where a
// thread per cell would walk its neighbours one memory round trip after the
// other.  slot_val: lane q's value in all four lanes of its cell (a quad
// permutation, no LDS), from which every lane takes the sums in slot order.
#define SLOT_CELLS (CSU_BLOCK / 4)  // cells of a workgroup
template <int Q>
__device__ __forceinline__ double slot_val(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_mov_dpp(hi, Q * 0x55, 0xF, 0xF, true),
                          __builtin_amdgcn_mov_dpp(lo, Q * 0x55, 0xF, 0xF, true));
}

// implicitCalcD (implicit.c:19-181), everything but the global-time-step
// term: writes Dp = 0.5 w Lc (+ Lv/Omega) and the minimum of Omega/Lc per
// SLOT_CELLS cells.
// A lane per face slot (slot_val): SA, 250k cells 22.7 -> 21.8 us, bound by
// its gathers' bytes; the smaller meshes' latency gains more.
template <int NV, bool VISC>
__global__ __launch_bounds__(CSU_BLOCK) void k_impD(KP kp, Geo g, St s, double wimp, double* __restrict__ Dp,
                                                    double* __restrict__ red_min, double* __restrict__ caux) {
  __shared__ double sw[1][CSU_BLOCK / 64];
  const int t = threadIdx.x, c0 = blockIdx.x * SLOT_CELLS, i = c0 + (t >> 2), j = t & 3;
  const int nc = kp.nc;
  if (g.sol) kp.cend = g.sol[solve_of(g.csolk, c0)].c1;
  double val = INFINITY;
  if (i < kp.cend) {
    const double* P = s.P;
    // The face's two states are the cell's and the neighbour's (cfn) in
    // either order: the face means add them, and a sum of two doubles does
    // not depend on their order.
    const int cf = g.cface[j * nc + i], nbr = g.cnbr[j * nc + i], nb = cf == 0 ? i : g.cfn[j * nc + i];
    const int np = g.cnp[i], fi = cf > 0 ? cf - 1 : (cf < 0 ? -cf - 1 : 0);
    double Pa[4], Pb[4];
#pragma unroll
    for (int q = 0; q < 4; q++) Pa[q] = P[(q == 3 ? 4 : q) * nc + i];  // r u v T
#pragma unroll
    for (int q = 0; q < 4; q++) Pb[q] = P[(q == 3 ? 4 : q) * nc + nb];
    const double om = g.omega[i];
    double lc = 0.0, lv = 0.0, lcb = 0.0, lvb = 0.0;
    if (cf != 0) {
      const double dSx = g.fdsx[fi], dSy = g.fdsy[fi], dS = g.fds[fi];
      double r = (Pa[0] + Pb[0]) * 0.5;
      double u = (Pa[1] + Pb[1]) * 0.5;
      double v = (Pa[2] + Pb[2]) * 0.5;
      double T = (Pa[3] + Pb[3]) * 0.5;
      double c = gas_T2c<double>(kp.gas, T);
      const Den<double> dl(dS);
      double nx = dl(dSx), ny = dl(dSy);
      lc = (fabs(nx * u + ny * v) + c) * dS;
      if (VISC) {
        double mi = sutherland(T);
        const double mp = Den<double>(kp.pr, kp.rpr)(mi);
        double mt = NV == 4 ? mp : mp + Den<double>(kp.pr_t, kp.rpr_t)(s.miT[fi]);
        lv = fmax(4 / (3 * r), gamma_of(kp.gas, T) / r) * mt * dS * dS;
      }
    }
    if (j < np && nbr < 0) {
      const int q = -1 - nbr;
      const double dSx = g.bdsx[q], dSy = g.bdsy[q], dS = g.bds[q];
      const double r = Pa[0], u = Pa[1], v = Pa[2], T = Pa[3];
      const double c = gas_T2c<double>(kp.gas, T);
      double nx, ny;
      if (dS > 0) { nx = dSx / dS; ny = dSy / dS; } else { nx = 0.0; ny = 1.0; }
      lcb = (fabs(nx * u + ny * v) + c) * dS;
      if (VISC) {
        double mi = sutherland(T);
        lvb = fmax(4 / (3 * r), gamma_of(kp.gas, T) / r) * (mi / kp.pr) * dS * dS;
      }
    }
    if (caux && j == 3) {
      // LU-SGS: the cell-state factors of its neighbour terms, evaluated
      // once per cell instead of once per face and sweep (same expressions
      // of the same values: implicit.c:307-313, 555-595); by the lane that
      // has no face on a triangle
      caux[i] = gas_T2c<double>(kp.gas, Pa[3]);
      if (VISC) {
        caux[nc + i] = fmax(4 / (3 * Pa[0]), gamma_of(kp.gas, Pa[3]) / Pa[0]);
        caux[2 * nc + i] = sutherland(Pa[3]) / kp.pr;
      }
    }
    // sums in slot order: interior faces, then boundary faces (slots
    // without one hold 0, which changes no sum of non-negative terms)
    const double Lc = ((slot_val<0>(lc) + slot_val<1>(lc)) + slot_val<2>(lc)) + slot_val<3>(lc);
    const double Lv = ((slot_val<0>(lv) + slot_val<1>(lv)) + slot_val<2>(lv)) + slot_val<3>(lv);
    double dtl = Lc;
    double D = 0.5 * wimp * Lc;
    if (VISC) D += Lv / om;
    const double bc[4] = {slot_val<0>(lcb), slot_val<1>(lcb), slot_val<2>(lcb), slot_val<3>(lcb)};
    const double bv[4] = {slot_val<0>(lvb), slot_val<1>(lvb), slot_val<2>(lvb), slot_val<3>(lvb)};
#pragma unroll
    for (int q = 0; q < 4; q++) {
      dtl += bc[q];
      D += 0.5 * wimp * bc[q];
      if (VISC) D += bv[q] / om;
    }
    if (j == 0) {
      Dp[i] = D;
      val = om / dtl;
    }
  }
  double m[1] = {val};
  block_reduce<CSU_BLOCK, 1>(m, sw, RedMin());
  if (t == 0) red_min[blockIdx.x] = m[0];
}

// diagonal with the global-time-step term (implicit.c:176-180); dtg holds
// one step per solve
__device__ __forceinline__ double diag(const double* Dp, const double* omega, const double* dtg, int i, int sid) {
  return Dp[i] + omega[i] / dtg[sid];
}

// x / Cv(T): the ideal gas's Cv inverted once on the host
__device__ __forceinline__ double over_cv(const GasD& g, double x, double T) {
  if (!g.tp) return Den<double>(g.Cv, g.rCv)(x);
  return x / gas_T2Cv<double>(g, T);
}

// implicitCalcDeltaFlux_sa (implicit.c:495-553): with the positivity clamps
__device__ __forceinline__ void delta_flux_sa(const KP& kp, const double* Pj, const double* d, double nx, double ny,
                                              double* dF) {
  double rho = Pj[0], u = Pj[1], v = Pj[2], p = Pj[3], n = Pj[5];
  double T = p / (kp.gas.R * rho);
  double e0 = gas_T2e<double>(kp.gas, T);
  double E = e0 + (u * u + v * v) / 2;
  double U[5] = {rho, rho * u, rho * v, rho * E, rho * n};
  double V = (nx * U[1] + ny * U[2]) / U[0];
  double F0[5] = {U[0] * V, U[1] * V + nx * p, U[2] * V + ny * p, (U[3] + p) * V, U[4] * V};
#pragma unroll
  for (int k = 0; k < 5; k++) U[k] = U[k] + d[k];
  rho = U[0];
  rho = fmax(rho, kp.rlim);
  U[0] = rho;
  const Den<double> dr(rho);
  u = dr(U[1]); v = dr(U[2]); E = dr(U[3]);
  double e1 = E - (u * u + v * v) * 0.5;
  e1 = fmax(e1, 7.176325e+02);
  T = T + over_cv(kp.gas, e1 - e0, T);
  if (T < 1) {
    T = 1;
    e1 = gas_T2e<double>(kp.gas, T);
    E = e1 + (u * u + v * v) * 0.5;
    U[3] = rho * E;
  }
  p = kp.gas.R * T * rho;
  n = dr(U[4]);
  n = fmax(n, 0.0);
  U[4] = rho * n;
  V = dr(nx * U[1] + ny * U[2]);
  dF[0] = U[0] * V - F0[0];
  dF[1] = (U[1] * V + nx * p) - F0[1];
  dF[2] = (U[2] * V + ny * p) - F0[2];
  dF[3] = (U[3] + p) * V - F0[3];
  dF[4] = U[4] * V - F0[4];
}

// implicitCalcDeltaFlux_sst (implicit.c:1048-1117): k and omega clamps
__device__ __forceinline__ void delta_flux_sst(const KP& kp, const double* Pj, const double* d, double nx, double ny,
                                               double* dF) {
  double rho = Pj[0], u = Pj[1], v = Pj[2], p = Pj[3], k = Pj[5], om = Pj[6];
  double T = p / (kp.gas.R * rho);
  double e0 = gas_T2e<double>(kp.gas, T);
  double E = e0 + (u * u + v * v) * 0.5 + k;
  double U[6] = {rho, rho * u, rho * v, rho * E, rho * k, rho * om};
  double V = (nx * U[1] + ny * U[2]) / U[0];
  double F0[6] = {U[0] * V, U[1] * V + nx * p, U[2] * V + ny * p, (U[3] + p) * V, U[4] * V, U[5] * V};
#pragma unroll
  for (int q = 0; q < 6; q++) U[q] = U[q] + d[q];
  rho = fmax(U[0], kp.rlim);
  U[0] = rho;
  const Den<double> dr(rho);
  u = dr(U[1]); v = dr(U[2]);
  k = dr(U[4]);
  if (k < 1e-14) { k = 1e-14; U[4] = rho * k; }
  om = dr(U[5]);
  if (om < 0.0) { om = 0.0; U[5] = rho * om; }
  E = dr(U[3]);
  double e1 = E - (u * u + v * v) * 0.5 - k;
  e1 = fmax(e1, 7.176325e+02);
  T = T + over_cv(kp.gas, e1 - e0, T);
  if (T < 1) {
    T = 1;
    e1 = gas_T2e<double>(kp.gas, T);
    E = e1 + (u * u + v * v) * 0.5 + k;
    U[3] = rho * E;
  }
  p = kp.gas.R * T * rho;
  V = dr(nx * U[1] + ny * U[2]);
  dF[0] = U[0] * V - F0[0];
  dF[1] = (U[1] * V + nx * p) - F0[1];
  dF[2] = (U[2] * V + ny * p) - F0[2];
  dF[3] = (U[3] + p) * V - F0[3];
  dF[4] = U[4] * V - F0[4];
  dF[5] = U[5] * V - F0[5];
}

// implicitCalcDeltaFlux (implicit.c:194-231) at state Pj with increment d
template <int NV>
__device__ __forceinline__ void delta_flux(const KP& kp, const double* Pj, const double* d, double nx, double ny,
                                           double* dF) {
  if (NV == 6) {
    delta_flux_sst(kp, Pj, d, nx, ny, dF);
    return;
  }
  if (NV == 5) {
    delta_flux_sa(kp, Pj, d, nx, ny, dF);
    return;
  }
  double rho = Pj[0], u = Pj[1], v = Pj[2], p = Pj[3];
  double T = p / (kp.gas.R * rho);
  double e0 = gas_T2e<double>(kp.gas, T);
  double E = e0 + (u * u + v * v) / 2;
  double U[4] = {rho, rho * u, rho * v, rho * E};
  double V = (nx * U[1] + ny * U[2]) / U[0];
  double F0[4] = {U[0] * V, U[1] * V + nx * p, U[2] * V + ny * p, (U[3] + p) * V};
#pragma unroll
  for (int k = 0; k < 4; k++) U[k] = U[k] + d[k];
  rho = U[0];
  const Den<double> dr(rho);
  u = dr(U[1]); v = dr(U[2]); E = dr(U[3]);
  double e1 = E - 0.5 * (u * u + v * v);
  T = T + over_cv(kp.gas, e1 - e0, T);
  p = kp.gas.R * T * rho;
  V = dr(nx * U[1] + ny * U[2]);
  dF[0] = U[0] * V - F0[0];
  dF[1] = (U[1] * V + nx * p) - F0[1];
  dF[2] = (U[2] * V + ny * p) - F0[2];
  dF[3] = (U[3] + p) * V - F0[3];
}

// Face slot j of cell i seen from i: neighbour id and outward face vector
// (the reference flips p0/p1 when i is the face's e1, implicit.c:288-305;
// the flipped vector is the exact negation).
__device__ __forceinline__ int face_from(const Geo& g, int nc, int i, int j, double& dSx, double& dSy, double& dS,
                                         int& fi) {
  const int f = g.cface[j * nc + i], nb = g.cfn[j * nc + i];
  if (f == 0) return -1;
  fi = f > 0 ? f - 1 : -f - 1;
  dS = g.fds[fi];
  if (f > 0) { dSx = g.fdsx[fi]; dSy = g.fdsy[fi]; return nb; }
  dSx = -g.fdsx[fi]; dSy = -g.fdsy[fi];
  return nb;
}

// One LU-SGS level.  DIR 0: forward sweep (implicitLUSGS_L, implicit.c:274-363),
// dW = -R then lower neighbours.  DIR 1: backward sweep (implicitLUSGS_U,
// implicit.c:365-482) from the forward result dW0: the cell's start value
// D*dW0 (implicit.c:369-399), then upper neighbours; a cell's dW is final
// once its level has run, so the level also applies it to the state
// (solverUpdateUImplicit, solver.c:1945-1955; a held solve of a batch keeps
// its state).
// A level is a fraction of the cells, and what bounds it is the chain of
// round trips of one wavefront; a lane per face slot (slot_val) loads and
// evaluates a cell's neighbours side by side.  Passes of 25 iterations, a
// thread per cell -> a lane per slot (with k_impD's): SST, 110k cells 4.57 ->
// 4.28 ms, SA, 250k cells 5.65 -> 5.52 ms; no change for Euler ramps.
template <int NV, bool VISC, int DIR>
__global__ __launch_bounds__(CSU_BLOCK) void k_lusgs(KP kp, Geo g, St s, const int* __restrict__ cells, int ncell_lvl,
                                                     const double* __restrict__ Dp, const double* __restrict__ dtg,
                                                     const double* __restrict__ R, double* dW,
                                                     const double* __restrict__ dW0, double* __restrict__ U,
                                                     const double* __restrict__ caux) {
  const int t = (blockIdx.x * blockDim.x + threadIdx.x) >> 2, j = threadIdx.x & 3;
  if (t >= ncell_lvl) return;
  const int nc = kp.nc;
  const int i = cells[t];
  const int sid = g.sol ? g.csol[i] : 0;
  const double D = diag(Dp, g.omega, dtg, i, sid);
  double acc[NV];
  if (DIR == 0) {
#pragma unroll
    for (int k = 0; k < NV; k++) acc[k] = -R[k * nc + i];
  } else {
#pragma unroll
    for (int k = 0; k < NV; k++) acc[k] = D * dW0[k * nc + i];
    if (NV == 6) {  // implicit.c:372-392: the k-omega block times dW0
      const double a = D - s.dq[nc + i], b = -s.dq[2 * nc + i], c = -s.dq[4 * nc + i], dd = D - s.dq[5 * nc + i];
      const double det = a * dd - b * c;
      if (!(fabs(det) < 1e-14)) {
        acc[NV > 4 ? 4 : 0] = a * dW0[4 * nc + i] + b * dW0[5 * nc + i] - s.dq[i] * dW0[i];
        acc[NV > 5 ? 5 : 0] = c * dW0[4 * nc + i] + dd * dW0[5 * nc + i] - s.dq[3 * nc + i] * dW0[i];
      }
    }
  }
  // this lane's slot: its face and neighbour, then the neighbour term (0
  // where the sweep does not use the slot: subtracting 0 changes nothing)
  const int cf = g.cface[j * nc + i], e = g.cfn[j * nc + i], fi = cf > 0 ? cf - 1 : (cf < 0 ? -cf - 1 : 0);
  const double dS = g.fds[fi], fx = g.fnx[fi], fy = g.fny[fi], fd = VISC ? g.fdd[fi] : 1.0;
  const int nb = cf == 0 ? i : e;
  double term[NV];
#pragma unroll
  for (int k = 0; k < NV; k++) term[k] = 0.0;
  if (cf != 0 && (DIR == 0 ? nb < i : nb > i)) {
    // outward unit normal (face_from: negated when i is the face's e1,
    // implicit.c:288-305; dS/|dS| with the sign of dS, stored per face)
    const double nx = cf > 0 ? fx : -fx, ny = cf > 0 ? fy : -fy;
    double Pj[NV + 1], d[NV], dF[NV];
#pragma unroll
    for (int m = 0; m < NV + 1; m++) Pj[m] = s.P[m * nc + nb];
#pragma unroll
    for (int k = 0; k < NV; k++) d[k] = dW[k * nc + nb];
    delta_flux<NV>(kp, Pj, d, nx, ny, dF);
    // the neighbour's sound speed and viscous factors max(4/(3r), gamma/r)
    // and mu/Pr (k_impD, per cell)
    const double c = caux[nb];
    double ra = kp.wimp * (fabs(nx * Pj[1] + ny * Pj[2]) + c) * dS;
    if (NV >= 5) {
      // implicitFunc_sa / _sst (implicit.c:555-595, 1120-1161)
      ra += caux[nc + nb] * (caux[2 * nc + nb] + Den<double>(kp.pr_t, kp.rpr_t)(s.miT[fi])) * dS / fd;
    } else if (VISC && kp.laminar) {
      ra += caux[nc + nb] * caux[2 * nc + nb] * dS / fd;
    }
#pragma unroll
    for (int k = 0; k < NV; k++) term[k] = 0.5 * (dF[k] * dS - ra * d[k]);
  }
#pragma unroll
  for (int k = 0; k < NV; k++) {
    acc[k] -= slot_val<0>(term[k]);
    acc[k] -= slot_val<1>(term[k]);
    acc[k] -= slot_val<2>(term[k]);
    acc[k] -= slot_val<3>(term[k]);
  }
  double out[NV];
  const Den<double> dD(D);
#pragma unroll
  for (int k = 0; k < NV; k++) out[k] = dD(acc[k]);
  if (NV == 6) {
    // SST: k-omega block with the source Jacobians, Cramer's rule
    // (implicit.c:326-351, 447-472).  The reference divides by a long double
    // determinant that holds a double value; the quotient here is the
    // correctly rounded double one.
    constexpr int K = NV > 4 ? 4 : 0, O = NV > 5 ? 5 : 0;
    const double x0 = out[0];
    const double A = acc[K] + s.dq[i] * x0;
    const double B = acc[O] + s.dq[3 * nc + i] * x0;
    const double a = D - s.dq[nc + i], b = -s.dq[2 * nc + i], c = -s.dq[4 * nc + i], dd = D - s.dq[5 * nc + i];
    const double det = a * dd - b * c;
    if (!(fabs(det) < 1e-14)) {
      out[K] = (A * dd - B * b) / det;
      out[O] = (-A * c + B * a) / det;
    }
  }
  // every lane of the cell has all of out: each stores its share
  const bool upd = DIR == 1 && (!g.sol || g.sol[sid].active);
#pragma unroll
  for (int k = 0; k < NV; k++)
    if ((k & 3) == j) {
      dW[k * nc + i] = out[k];
      if (upd) U[k * nc + i] += out[k];
    }
}

// Place of slot j's block of cell i among the DPLUR blocks; entry e (row NV +
// column) is at block_entry(e) from there.  The blocks of 64 cells are one
// run, entries in pairs: a wavefront reads a pair with one 16-byte load per
// lane, and a sweep's wavefront touches one stretch of memory where planes
// [4][NV*NV][nc] spread it over every page of the array (56k cells: 7.9 ->
// 6.4 us per sweep; the blocks are re-read every sweep, 28.7 MB).
// The runs are 1 KB longer than their entries: at a multiple of 32 KB every
// wavefront would be on the same memory channels at the same time.  Passes of
// 25 iterations, 56k cells: planes 6.06 ms, runs of 32 KB 5.76, of 33 KB 5.15.
constexpr int block_len(int nv) { return (nv * nv + 1) / 2 * 2; }
constexpr size_t block_run(int nv) { return (size_t)4 * block_len(nv) * 64 + 128; }
constexpr size_t block_total(int nv, size_t nc) { return (nc + 63) / 64 * block_run(nv); }
template <int NV>
__device__ __forceinline__ size_t block_at(int i, int j) {
  return (size_t)(i >> 6) * block_run(NV) + (size_t)j * block_len(NV) * 64 + 2 * (i & 63);
}
__device__ __forceinline__ constexpr int block_entry(int e) { return (e >> 1) * 128 + (e & 1); }

// DPLUR finite-difference blocks of every interior neighbour
// (implicitUpdateA, implicit.c:689-813; implicitUpdateA_sa :815-936),
// h = 1e-6.  SST (NV 6) has no DPLUR in the
// reference (implicitCalcDPLUR builds 4x4 blocks for it); its 6x6 blocks
// here take implicitUpdateA_sa's form with two convected scalars (the
// fluxes of implicitAuxCalcFlux_sst2, implicit.c:1036-1046) and k taken out
// of the internal energy, as implicitCalcDeltaFlux_sst does (:1048-1117).
template <int NV, bool VISC>
__global__ __launch_bounds__(CSU_BLOCK) void k_blocks(KP kp, Geo g, St s, const double* __restrict__ U,
                                                      double* __restrict__ A) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int nc = kp.nc;
  if (g.sol) kp.cend = g.sol[solve_of(g.csolk, blockIdx.x * blockDim.x)].c1;
  if (i >= kp.cend) return;
  const double h = 1.0e-6;
  // Every slot's face data and neighbour state first (one memory round trip
  // for all slots instead of one chain per slot); slots without a face
  // read the cell itself and are skipped.
  int nbs[4], fis[4];
  double sxs[4], sys_[4], sds[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    fis[j] = 0;
    sxs[j] = sys_[j] = 0.0;
    sds[j] = 1.0;
    nbs[j] = face_from(g, nc, i, j, sxs[j], sys_[j], sds[j], fis[j]);
  }
  double Ujs[4][NV], P1s[4], P2s[4], P3s[4], P4s[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int nb = nbs[j] >= 0 ? nbs[j] : i;
#pragma unroll
    for (int k = 0; k < NV; k++) Ujs[j][k] = U[k * nc + nb];
    P1s[j] = s.P[nc + nb]; P2s[j] = s.P[2 * nc + nb]; P3s[j] = s.P[3 * nc + nb]; P4s[j] = s.P[4 * nc + nb];
  }
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int nb = nbs[j], fi = fis[j];
    if (nb < 0) continue;
    const double dSx = sxs[j], dSy = sys_[j], dS = sds[j];
    const double nx = dSx / dS, ny = dSy / dS;
    const double P3 = P3s[j], P4 = P4s[j];
    double Uj[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) Uj[k] = Ujs[j][k];
    double rho = Uj[0], u = Uj[1] / rho, v = Uj[2] / rho, E = Uj[3] / rho;
    double V = (nx * Uj[1] + ny * Uj[2]) / Uj[0];
    double F0[NV];
    F0[0] = Uj[0] * V; F0[1] = Uj[1] * V + nx * P3; F0[2] = Uj[2] * V + ny * P3; F0[3] = (Uj[3] + P3) * V;
    if (NV >= 5) F0[4] = Uj[4] * V;
    if (NV == 6) F0[5] = Uj[5] * V;
    const double ee0 = NV == 6 ? E - 0.5 * (u * u + v * v) - Uj[4] / rho : E - 0.5 * (u * u + v * v);
    const double cv = gas_T2Cv<double>(kp.gas, P4);
    // the diagonal's spectral-radius term, subtracted from each diagonal
    // entry as it is stored (the reference subtracts it from the stored
    // block, implicit.c:792-809: the same two roundings)
    double c = gas_T2c<double>(kp.gas, P4);
    double ra = kp.wimp * (fabs(nx * P1s[j] + ny * P2s[j]) + c) * dS;
    if (NV >= 5) {
      // implicitUpdateA_sa (implicit.c:815-936); SST the same with its
      // face eddy viscosity
      double r = (s.P[i] + s.P[nb]) * 0.5;
      double T = (s.P[4 * nc + i] + P4) * 0.5;
      double mi = sutherland(T);
      double ddx = g.xc[nb] - g.xc[i], ddy = g.yc[nb] - g.yc[i];
      double dd_ = sqrt(ddx * ddx + ddy * ddy);
      ra += fmax(4 / (3 * r), gamma_of(kp.gas, T) / r) * (mi / kp.pr + s.miT[fi] / kp.pr_t) * dS / dd_;
    } else if (VISC && kp.laminar) {
      double r = (s.P[i] + s.P[nb]) * 0.5;
      double T = (s.P[4 * nc + i] + P4) * 0.5;
      double mi = sutherland(T);
      double ddx = g.xc[nb] - g.xc[i], ddy = g.yc[nb] - g.yc[i];
      double dd_ = sqrt(ddx * ddx + ddy * ddy);
      ra += fmax(4 / (3 * r), gamma_of(kp.gas, T) / r) * (mi / kp.pr) * dS / dd_;
    }
    double* Aj = A + block_at<NV>(i, j);
#pragma unroll
    for (int mm = 0; mm < NV; mm++) {
      double Up[NV];
#pragma unroll
      for (int n = 0; n < NV; n++) Up[n] = mm == n ? Uj[n] + h : Uj[n];
      rho = Up[0]; u = Up[1] / rho; v = Up[2] / rho; E = Up[3] / rho;
      double ee1 = NV == 6 ? E - 0.5 * (u * u + v * v) - Up[4] / rho : E - 0.5 * (u * u + v * v);
      double T = P4 + (ee1 - ee0) / cv;
      double p = kp.gas.R * rho * T;
      double Vp = (nx * Up[1] + ny * Up[2]) / Up[0];
      double F[NV];
      F[0] = Up[0] * Vp; F[1] = Up[1] * Vp + nx * p; F[2] = Up[2] * Vp + ny * p; F[3] = (Up[3] + p) * Vp;
      if (NV >= 5) F[4] = Up[4] * Vp;
      if (NV == 6) F[5] = Up[5] * Vp;
#pragma unroll
      for (int n = 0; n < NV; n++) {
        const double a = 0.5 * (F[n] - F0[n]) * dS / h;
        Aj[block_entry(n * NV + mm)] = n == mm ? a - 0.5 * ra : a;
      }
    }
  }
}

// An increment of the DPLUR sweeps: [nc][4] for four variables (a neighbour's
// is one 32-byte run), else [NV][nc].
template <int NV>
__device__ __forceinline__ void jac_load(const double* x, int nc, int i, double* v) {
  if (NV == 4) {
    const double2* p = (const double2*)x + 2 * (size_t)i;
    const double2 a = p[0], b = p[1];
    v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
  } else {
#pragma unroll
    for (int k = 0; k < NV; k++) v[k] = x[k * nc + i];
  }
}

// Largest of every thread's v in the workgroup (fmax: NaN is the identity,
// the maximum is exact in any order), in every thread.
__device__ __forceinline__ double block_fmax(double v, double (*sw)[CSU_BLOCK / 64]) {
  double r[1] = {v};
  block_reduce<CSU_BLOCK, 1>(r, sw, RedMax());
  return r[0];
}

// One damped Jacobi sweep m (implicitMultA + update, implicit.c:938-1022):
// y = D x + sum_j A_j x_j;  x_new = w (-R - y)/D + x, from buf[(state[1] +
// m) & 1] into the other buffer; state[1] is the buffer holding the last
// implicit step's result.  The block maxima of |dx_rho| go to red_sw[m][.];
// each sweep first reduces the previous sweep's (the reference's test
// after every sweep, implicit.c:1026-1031), and once that is below 1e-14
// (or marked -1: the sweeps had already stopped) it writes -1 and does
// nothing: the reference breaks out of its loop.
// SST: the diagonal is LU-SGS's block (implicit.c:326-351), D with the
// k-omega source Jacobians dq; y takes its product and x_new solves with it
// by Cramer's rule (D alone where its determinant is below 1e-14).
template <int NV>
__global__ __launch_bounds__(CSU_BLOCK) void k_jacobi(KP kp, Geo g, const double* __restrict__ A,
                                                      const double* __restrict__ Dp, const double* __restrict__ dtg,
                                                      const double* __restrict__ R, double* buf0, double* buf1,
                                                      const int* __restrict__ state, double* __restrict__ red_sw,
                                                      int m, const double* __restrict__ dq) {
  __shared__ double sw0[1][CSU_BLOCK / 64], sw1[1][CSU_BLOCK / 64];
  const int t = threadIdx.x, i = blockIdx.x * blockDim.x + t;
  const int nc = kp.nc, stride = gridDim.x;
  // batch: the solve's own blocks and buffer state
  int sid = 0, b0 = 0, nblocks = gridDim.x;
  if (g.sol) {
    sid = solve_of(g.csolk, blockIdx.x * blockDim.x);
    const SolveP& q = g.sol[sid];
    kp.cend = q.c1;
    b0 = q.c0 / CSU_BLOCK;
    nblocks = (q.c1 - q.c0 + CSU_BLOCK - 1) / CSU_BLOCK;
  }
  const int par = (state[2 * sid + 1] + m) & 1;
  const double* x = par ? buf1 : buf0;
  double* y = par ? buf0 : buf1;
  const bool act = i < kp.cend;
  // Every load that does not depend on the stop test is issued before it:
  // the cell's x, R, diagonal and neighbour ids (per face slot, cfn), then
  // the neighbours' x.  Slots without a face read the cell itself and are
  // skipped; lanes past the last cell read cell 0 and store nothing.
  const int ii = act ? i : 0;
  double xi[NV], Ri[NV];
#pragma unroll
  for (int k = 0; k < NV; k++) xi[k] = 0.0;
  jac_load<NV>(x, nc, ii, xi);
  int nbj[4];
  bool has[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int c = act ? g.cfn[j * nc + ii] : -1;
    has[j] = c >= 0;
    nbj[j] = c >= 0 ? c : ii;
  }
#pragma unroll
  for (int k = 0; k < NV; k++) Ri[k] = R[k * nc + ii];
  const double D = diag(Dp, g.omega, dtg, ii, sid);
  double dqi[6];
#pragma unroll
  for (int q = 0; q < 6; q++) dqi[q] = NV == 6 ? dq[q * nc + ii] : 0.0;
  double xj[4][NV];
#pragma unroll
  for (int j = 0; j < 4; j++)
    jac_load<NV>(x, nc, nbj[j], xj[j]);
  if (m > 0) {
    // The maximum over the solve's blocks is at least this block's own
    // (a number >= 1e-14 rules the stop out, so the reduction is skipped:
    // the common case while the sweeps run).  Otherwise reduce every
    // block's.  NaN is fmax's identity: the maximum is NaN only when every
    // cell's change is, which the reference's loop (implicit.c:1023-1031)
    // does not take as converged.  The branch is uniform in the block.
    const double* prev = red_sw + (size_t)(m - 1) * stride + b0;
    const double own = red_sw[(size_t)(m - 1) * stride + blockIdx.x];
    if (!(own >= 1e-14)) {
      double pm = __builtin_nan("");
      for (int b = t; b < nblocks; b += CSU_BLOCK) pm = fmax(pm, prev[b]);
      if (block_fmax(pm, sw0) < 1e-14) {
        if (t == 0) red_sw[(size_t)m * stride + blockIdx.x] = -1.0;
        return;
      }
    }
  }
  double diff = __builtin_nan("");  // lanes past the last cell: fmax's identity
  if (act) {
    double acc[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) acc[k] = D * xi[k];
    double qa = D, qb = 0.0, qc = 0.0, qd = D, q0 = 0.0, q3 = 0.0, det = 0.0;
    bool blk = false;
    if (NV == 6) {
      q0 = dqi[0]; q3 = dqi[3];
      qa = D - dqi[1]; qb = -dqi[2]; qc = -dqi[4]; qd = D - dqi[5];
      det = qa * qd - qb * qc;
      blk = !(fabs(det) < 1e-14);
      if (blk) {
        acc[4] = qa * xi[4] + qb * xi[5] - q0 * xi[0];
        acc[5] = qc * xi[4] + qd * xi[5] - q3 * xi[0];
      }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (!has[j]) continue;
      const double2* Aj = (const double2*)(A + block_at<NV>(i, j));
      double2 Ae[block_len(NV) / 2];
#pragma unroll
      for (int e = 0; e < block_len(NV) / 2; e++) Ae[e] = Aj[e * 64];
#pragma unroll
      for (int k = 0; k < NV; k++)
#pragma unroll
        for (int n = 0; n < NV; n++)
          acc[k] += ((k * NV + n) & 1 ? Ae[(k * NV + n) >> 1].y : Ae[(k * NV + n) >> 1].x) * xj[j][n];
    }
    const double w = 2. / 3.;
    if (NV == 6 && blk) {
      double z[NV];
#pragma unroll
      for (int k = 0; k < 4; k++) z[k] = (-Ri[k] - acc[k]) / D;
      const double Ak = -Ri[4] - acc[4] + q0 * z[0];
      const double Bo = -Ri[5] - acc[5] + q3 * z[0];
      z[4] = (Ak * qd - Bo * qb) / det;
      z[5] = (-Ak * qc + Bo * qa) / det;
#pragma unroll
      for (int k = 0; k < NV; k++) {
        const double yk = w * z[k] + xi[k];
        y[k * nc + i] = yk;
        if (k == 0) diff = fabs(yk - xi[0]);
      }
    } else {
      const Den<double> dD(D);
      double yk[NV];
#pragma unroll
      for (int k = 0; k < NV; k++) yk[k] = dD(w * (-Ri[k] - acc[k])) + xi[k];
      diff = fabs(yk[0] - xi[0]);
      if (NV == 4) {
        double2* o = (double2*)y + 2 * (size_t)i;
        o[0] = make_double2(yk[0], yk[1]);
        o[1] = make_double2(yk[2], yk[3]);
      } else {
#pragma unroll
        for (int k = 0; k < NV; k++) y[k * nc + i] = yk[k];
      }
    }
  }
  const double bm = block_fmax(diff, sw1);
  if (t == 0) red_sw[(size_t)m * stride + blockIdx.x] = bm;
}

// After the sweeps: the buffer holding each solve's result becomes its base
// (the update's increment, and the next step's start).  Sweeps 0..k-1 ran
// (k = the first sweep marked -1 in red_sw, rows of length stride, or nlin),
// so the last one wrote buf[(state[2 sid + 1] + k) & 1].  A wavefront per
// solve, a lane per mark.
__global__ __launch_bounds__(64) void k_jac_base(int* state, const double* __restrict__ red_sw, int nlin, int stride,
                                                 const SolveP* __restrict__ sol) {
  const int sid = blockIdx.x, b0 = sol ? sol[sid].c0 / CSU_BLOCK : 0;
  int k = nlin;
  for (int k0 = 0; k0 < nlin && k == nlin; k0 += 64) {
    const int q = k0 + (int)threadIdx.x;
    const unsigned long long hit = __ballot(q < nlin && red_sw[(size_t)(q < nlin ? q : 0) * stride + b0] < 0.0);
    if (hit) k = k0 + __ffsll(hit) - 1;
  }
  if (threadIdx.x == 0) state[2 * sid + 1] = (state[2 * sid + 1] + k) & 1;
}

// solverUpdateUImplicit (solver.c:1945-1955) for DPLUR: U += dW, the sweeps'
// result (k_jac_base).  Batch: a solve that is not active keeps its state.
template <int NV>
__global__ __launch_bounds__(CSU_BLOCK) void k_upd_imp(int nc, double* __restrict__ U, const double* buf0,
                                                       const double* buf1, const int* __restrict__ state,
                                                       const SolveP* __restrict__ sol, const int* __restrict__ csolk) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  int sid = 0, cend = nc;
  if (sol) {
    sid = solve_of(csolk, blockIdx.x * blockDim.x);
    const SolveP& q = sol[sid];
    if (!q.active) return;
    cend = q.c1;
  }
  if (i >= cend) return;
  double d[NV];
  jac_load<NV>(state[2 * sid + 1] ? buf1 : buf0, nc, i, d);
#pragma unroll
  for (int k = 0; k < NV; k++) U[k * nc + i] += d[k];
}

}  // namespace csu
