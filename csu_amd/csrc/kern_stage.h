// kern_stage.h -- one explicit stage of the inviscid path (reference
// solverCalcR + solverRK, solver.c:685-766) as one kernel: second order, and
// first order without phase 1.
//
// A workgroup owns a tile of CSU_CHUNK consecutive cells and keeps what the
// three split kernels (k_grad, k_flux, k_update) pass to each other through
// memory in LDS:
//   0  boundary faces of the tile's cells and of its halo (the cells across
//      its outer faces): ghost states, and the tile's own boundary fluxes
//   1  the tile's cells and its halo: gradients, limiter, and the
//      reconstructed state at every edge of a tile face, into the face's left
//      or right half
//   2  the tile's faces: Riemann flux of the two halves, in place
//   3  the tile's cells: sums in the cell's slot order, RK update
// The values and their order are those of the split kernels, so results are
// the same bit for bit.  A halo cell's gradient and a face between two tiles
// are evaluated by every tile that needs them.
//
// What bounds it: memory traffic and FP64 issue about alike.  4.0M cells in
// Morton order: 315 us a stage, 1,560 MB counted (277 B per cell that it
// cannot do without; the split kernels' stage 540: edge states and face
// fluxes written and read back), 4.95 TB/s or 0.74 of the streaming rate,
// with FP64 instructions issuing in 62 % of its cycles; the halo's gradients
// are a third of phase 1.  Contiguous copies of the halo cells' geometry
// changed nothing.  Below about 100k cells: the latency of its four phases.
// RK5 iterations, split kernels with the face fluxes in the update -> this
// kernel: 2.0M cells 1,247 -> 890 us (4.0M 2,380 -> 1,607 us); 406k cells in
// mixed precision 250 -> 190 us; 40k cells 114 -> 71 us (launches: 22 -> 7).
#pragma once
#include "kernels.h"

namespace csu {

// Lists of the tile form (device pointers): tile t has the interior faces
// [toff[t], toff[t+1]) of the entry arrays, the boundary faces [boff[t],
// boff[t+1]) of tbq (the first bown[t] of its own cells, then those of halo
// cells) and the halo cells [hoff[t], hoff[t+1]).
struct Tile {
  const int *toff, *boff, *bown, *hoff;
  const int *tbq, *tbc;             // boundary face, its cell
  const int* hcell;                 // halo cell
  const double *fx, *fy, *fs;       // entry: face vector and length (copies in entry order: coalesced)
  const float *fx32, *fy32, *fs32;  // mixed precision
  const short *csl, *hsl;           // [4][nc], [4][nh]: slot j's entry, +(1 + place) where the cell is the face's
                                    // e0, -(1 + place) where e1; boundary slots 1 + place in the boundary list
  const short *cel, *hel;           // [4][nc], [4][nh]: edge j's entry, + left half, - right half, 0 none
  const int *fa, *fb;               // first-order runs: entry's cells
  int nh;                           // stride of hsl, hel
  int capf;                         // interior entries the LDS array holds
};

// Primitives r u v p of cell i: [nc][4], one 32-byte run per gathered
// neighbour instead of one line in each of four planes.
__device__ __forceinline__ void load4(const dbl2* P, int i, double* v) {
  const dbl2 a = P[2 * (size_t)i], b = P[2 * (size_t)i + 1];
  v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
}
__device__ __forceinline__ void store4(dbl2* P, int i, const double* v) {
  P[2 * (size_t)i] = dbl2{v[0], v[1]};
  P[2 * (size_t)i + 1] = dbl2{v[2], v[3]};
}
// That layout from the planes k_prim writes (after the state was set from the
// host).
__global__ __launch_bounds__(CSU_BLOCK) void k_pack4(int nc, const double* __restrict__ P, dbl2* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nc) return;
  const double v[4] = {P[i], P[nc + i], P[2 * nc + i], P[3 * nc + i]};
  store4(out, i, v);
}

// Phase 1 of one cell: its reconstructed edge states into the halves of the
// tile's faces (sf: [8][cap], left then right state).  sl, el: the cell's
// slot and edge places; sb: the boundary entries ([place][8]: flux, ghost
// state).
template <int NE, bool MIX, bool LD, typename TF>
__device__ __forceinline__ void stage_cell(const KP& kp, const Geo& g, const St& s, const Tile& tl,
                                           const dbl2* __restrict__ Pin, const SolveP* sv, const double* __restrict__ pref, int i, const short* sl,
                                           const short* el, int lst, TF* sf, const double* sb) {
  const int nc = kp.nc, cap = tl.capf;
  // NE 3: a mesh of triangles only; 4: slot 3 exists for quads
  const int np = NE == 3 ? 3 : g.cnp[i];
  int nbr[4];
#pragma unroll
  for (int j = 0; j < NE; j++) nbr[j] = j == 3 && np < 4 ? i : g.cnbr[j * nc + i];
  double Pi[4], un[4][4];
  load4(Pin, i, Pi);
#pragma unroll
  for (int j = 0; j < NE; j++) {
    if (j == 3 && np < 4) break;
    load4(Pin, nbr[j] >= 0 ? nbr[j] : i, un[j]);
  }
  TF ex[4], ey[4], wx[4], wy[4];
#pragma unroll
  for (int j = 0; j < NE; j++) {
    ex[j] = ey[j] = wx[j] = wy[j] = 0;
    if (j == 3 && np < 4) break;
    const size_t w = 4 * ((size_t)j * nc + i);
    if (MIX) {
      const flt4 v = *(const flt4*)(g.wg32 + w);
      wx[j] = v.x; wy[j] = v.y; ex[j] = v.z; ey[j] = v.w;
    } else {
      const dbl2 v = *(const dbl2*)(g.wg + w), e = *((const dbl2*)(g.wg + w) + 1);
      wx[j] = v.x; wy[j] = v.y; ex[j] = e.x; ey[j] = e.y;
    }
  }
  int pl[4];
#pragma unroll
  for (int j = 0; j < NE; j++) pl[j] = el[j * lst];
  double lim_aux = 0.0;
  if (kp.limiter == 0) {
    lim_aux = kp.limK * sqrt(g.omega[i] / (sv ? sv->volmax : kp.volmax));
    lim_aux = lim_aux * lim_aux * lim_aux;
  }
  double dx[4], dy[4];
  if (LD) {
#pragma unroll
    for (int j = 0; j < NE; j++) {
      dx[j] = dy[j] = 0.0;
      if (j >= np) break;
      const int n = nbr[j];
      dx[j] = (n >= 0 ? g.xc[n] : g.bxm[-1 - n]) - g.xc[i];
      dy[j] = (n >= 0 ? g.yc[n] : g.bym[-1 - n]) - g.yc[i];
    }
  }
  dd a = {0, 0}, b = {0, 0}, c = {0, 0}, det = {0, 0}, nb_ = {0, 0};
  if (LD) {
#pragma unroll
    for (int j = 0; j < NE; j++) {
      if (j >= np) break;
      a = dd_add_d(a, dx[j] * dx[j]);
      b = dd_add_d(b, dx[j] * dy[j]);
      c = dd_add_d(c, dy[j] * dy[j]);
    }
    det = dd_sub(dd_mul(a, c), dd_mul(b, b));
    nb_ = dd_neg(b);
  }
#pragma unroll
  for (int j = 0; j < NE; j++) {
    if (j == 3 && np < 4) break;
    if (nbr[j] < 0) {
      const double* o = sb + 8 * (sl[j * lst] - 1) + 4;
#pragma unroll
      for (int k = 0; k < 4; k++) un[j][k] = o[k];
    }
  }
#pragma unroll
  for (int kk = 0; kk < 4; kk++) {
    const double v0 = Pi[kk];
    double du[4];
    double Pmin = v0, Pmax = v0;
#pragma unroll
    for (int j = 0; j < NE; j++) {
      if (j == 3 && np < 4) break;
      du[j] = un[j][kk] - v0;
      Pmax = fmax(Pmax, un[j][kk]);
      Pmin = fmin(Pmin, un[j][kk]);
    }
    TF tgx, tgy;
    if (LD) {
      double gx, gy;
      lsq_grad<NE>(np, dx, dy, du, a, b, nb_, c, det, gx, gy);
      tgx = (TF)gx;
      tgy = (TF)gy;
    } else {
      tgx = wx[0] * (TF)du[0];
      tgy = wy[0] * (TF)du[0];
#pragma unroll
      for (int j = 1; j < NE; j++) {
        if (j == 3 && np < 4) break;
        tgx += wx[j] * (TF)du[j];
        tgy += wy[j] * (TF)du[j];
      }
    }
    const double pref2 = kp.limiter == 0 ? pref[kk] * lim_aux : pref[kk];
    const TF d1max = (TF)(Pmax - v0), d1min = (TF)(Pmin - v0);
    TF ph = 0, d2[4];
#pragma unroll
    for (int j = 0; j < NE; j++) {
      if (j == 3 && np < 4) break;
      d2[j] = tgx * ex[j] + tgy * ey[j];
    }
    if (kp.limiter == 2) {
#pragma unroll
      for (int j = 0; j < NE; j++) {
        if (j == 3 && np < 4) break;
        const TF p0 = limiter_bj<TF>(d1max, d1min, d2[j]);
        ph = (j == 0) ? p0 : fmin(ph, p0);
      }
    } else {
#pragma unroll
      for (int j = 0; j < NE; j++) {
        if (j == 3 && np < 4) break;
        const TF p0 = limiter_v2d<TF, LD>(d1max, d1min, d2[j], (TF)pref2);
        ph = (j == 0) ? p0 : fmin(ph, p0);
      }
    }
#pragma unroll
    for (int j = 0; j < NE; j++) {
      if (j == 3 && np < 4) break;
      const int p = pl[j];
      if (p == 0) continue;
      const TF r = MIX ? (TF)(v0 + (double)(d2[j] * ph)) : (TF)(v0 + d2[j] * ph);
      sf[(p > 0 ? kk * cap + p - 1 : (4 + kk) * cap - p - 1)] = r;
    }
  }
}

// Phase 0 of one boundary face: its ghost state (boundaryCalcPrimitive) and,
// for one of the tile's own cells, its convective flux (bc_flux,
// kern_common.h, with the two states at hand).
template <int FLX>
__device__ __forceinline__ void stage_bface(const KP& kp, const Geo& g, const St& s, const dbl2* Pin, int q, int i,
                                            bool own, bool lastst, double* o) {
  const int nb = kp.nb, type = g.btype[q];
  const double dSx = g.bdsx[q], dSy = g.bdsy[q], dS = g.bds[q];
  double PL[4], PR[5], fl[4];
  load4(Pin, i, PL);
  ghost_state<4>(kp, type, dSx, dSy, dS, PL, 0.0, PR);
#pragma unroll
  for (int k = 0; k < 4; k++) o[4 + k] = PR[k];
  if (!own) return;
  if (lastst)  // the forces read them
#pragma unroll
    for (int m = 0; m < 5; m++) s.Pb[m * nb + q] = PR[m];
  rotate<double>(PL[1], PL[2], dSx, dSy, dS);
  if (type == CSU_BC_SYMMETRY) {
    PR[0] = PL[0]; PR[1] = -PL[1]; PR[2] = PL[2]; PR[3] = PL[3];
  } else {
    rotate<double>(PR[1], PR[2], dSx, dSy, dS);
  }
  if (type == CSU_BC_WALL || type == CSU_BC_WALLT) flux_free<double>(kp.gas, PR[0], PR[1], PR[2], PR[3], fl);
  else
    flux_dispatch<double, 0>(kp.gas, FLX >= 0 ? FLX : kp.flux, kp.efix, kp.minf, PL[0], PL[1], PL[2], PL[3], PL, PR[0], PR[1], PR[2],
                             PR[3], PR, 0.0, 0.0, fl);
  rotate<double>(fl[1], fl[2], dSx, -dSy, dS);
#pragma unroll
  for (int k = 0; k < 4; k++) o[k] = dS > 0 ? 0.0 + fl[k] * dS : 0.0;
}

// One RK stage: the primitives r u v p of the stage's state (Pin, read with
// the neighbours' and the halo's) -> those of the next stage's state (Pout,
// another buffer); the last stage also writes the state (Uout).  Un, the
// iteration's start state, is clamped where it is used (F_CLAMP_UN:
// solverCalcPrimitive writes the clamps back into U^n on the first residual;
// they are a function of U^n alone, so every stage can repeat them).
// FLX: the flux function, -1: kp.flux (one function inlined instead of five
// keeps the code in the instruction cache: 64 KB with all of them); NE: the
// most edges of a cell; O1: a first-order run, whose faces take the states of
// their cells from memory (phase 2 alone beside the boundary faces: launch and
// one gather chain bound it).
template <int NT, int NE, int FLX, bool MIX, bool LD, bool O1 = false>
__global__ __launch_bounds__(NT, 4) void k_stage(KP kp, Geo g, St s, Tile tl, int flags, double sigma, double rk_a,
                                              double cfl, double* dtl, const double* dtg,
                                              const double* __restrict__ Un, double* __restrict__ Uout,
                                              const dbl2* __restrict__ Pin, dbl2* __restrict__ Pout,
                                              double* __restrict__ red_res, double* __restrict__ red_dt) {
  using TF = typename std::conditional<MIX, float, double>::type;
  kp.gas.tp = 0;  // the tile form exists for the ideal gas only
  extern __shared__ double smem[];
  __shared__ double sw[5][CSU_CHUNK / 64];
  const int tile = kp.xcd ? xcd_tile(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  const int t = threadIdx.x, c0 = tile * CSU_CHUNK;
  const int nc = kp.nc;
  const bool lastst = (flags & F_LAST) != 0;
  // batch: what differs between solves is read from the table where it is
  // used (patching kp up front, as the split kernels do, kept ~30 scalars
  // alive through all phases and spilled them)
  const int sid = g.sol ? solve_of(g.csolk, c0) : 0;
  const SolveP* sv = g.sol ? g.sol + sid : nullptr;
  const double minf = sv ? sv->minf : kp.minf;
  TF* sf = (TF*)smem;
  double* sb = smem + (MIX ? 4 : 8) / (O1 ? 2 : 1) * tl.capf;  // O1: sf holds the fluxes only
  const int f0 = tl.toff[tile], nft = tl.toff[tile + 1] - f0;
  const int b0 = tl.boff[tile], h0 = tl.hoff[tile], nh = tl.hoff[tile + 1] - h0;
  const int nown = min(CSU_CHUNK, (sv ? sv->c1 : nc) - c0), nbt = tl.boff[tile + 1] - b0;
  if (nbt > 0) {
    KP kb = kp;
    kb.pout = sv ? sv->pout : kp.pout;
    kb.twall = sv ? sv->twall : kp.twall;
    kb.minf = minf;
#pragma unroll
    for (int k = 0; k < 7; k++) kb.pin[k] = sv ? sv->pin[k] : kp.pin[k];
    for (int k = t; k < nbt; k += NT)
      stage_bface<FLX>(kb, g, s, Pin, tl.tbq[b0 + k], tl.tbc[b0 + k], k < tl.bown[tile], lastst, sb + 8 * k);
    if (!O1) __syncthreads();
  }
  for (int k = t; !O1 && k < CSU_CHUNK + nh; k += NT) {
    const bool own = k < CSU_CHUNK;
    if (own && k >= nown) continue;
    const int h = h0 + k - CSU_CHUNK, i = own ? c0 + k : tl.hcell[h];
    stage_cell<NE, MIX, LD, TF>(kp, g, s, tl, Pin, sv, s.pref2 + 6 * sid, i, own ? tl.csl + i : tl.hsl + h,
                                own ? tl.cel + i : tl.hel + h, own ? nc : tl.nh, sf, sb);
  }
  if (!O1) __syncthreads();
  for (int k = t; k < nft; k += NT) {
    TF dSx, dSy, dS;
    if (MIX) {
      dSx = tl.fx32[f0 + k]; dSy = tl.fy32[f0 + k]; dS = tl.fs32[f0 + k];
    } else {
      dSx = tl.fx[f0 + k]; dSy = tl.fy[f0 + k]; dS = tl.fs[f0 + k];
    }
    TF PL[4], PR[4], fl[4];
    if (O1) {
      double a[4], b[4];
      load4(Pin, tl.fa[f0 + k], a);
      load4(Pin, tl.fb[f0 + k], b);
#pragma unroll
      for (int kk = 0; kk < 4; kk++) { PL[kk] = (TF)a[kk]; PR[kk] = (TF)b[kk]; }
    } else {
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {
        PL[kk] = sf[kk * tl.capf + k];
        PR[kk] = sf[(4 + kk) * tl.capf + k];
      }
    }
    const Den<TF> dl(dS);
    rotate<TF>(PL[1], PL[2], dSx, dSy, dl);
    rotate<TF>(PR[1], PR[2], dSx, dSy, dl);
    flux_dispatch<TF, 0>(kp.gas, FLX >= 0 ? FLX : kp.flux, (TF)kp.efix, (TF)minf, PL[0], PL[1], PL[2], PL[3], PL, PR[0], PR[1],
                         PR[2], PR[3], PR, (TF)0, (TF)0, fl);
    rotate<TF>(fl[1], fl[2], dSx, -dSy, dl);
#pragma unroll
    for (int kk = 0; kk < 4; kk++) sf[kk * tl.capf + k] = fl[kk] * dS;
  }
  __syncthreads();
  const int i = c0 + t;
  double R[4] = {0.0, 0.0, 0.0, 0.0}, dt_next = INFINITY;
  if (t < nown) {
    int cs[4];
    const int bm = g.bmask[i];
#pragma unroll
    for (int j = 0; j < NE; j++) cs[j] = tl.csl[j * nc + i];
    double un0[4], un[4], p[5];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) un0[kk] = un[kk] = Un[kk * nc + i];
    const double dt = (flags & F_CUR_LOCAL) ? dtl[i] : dtg[sid];
    const double om = g.omega[i];
#pragma unroll
    for (int j = 0; j < NE; j++) {
      const int f = ((bm >> j) & 1) ? 0 : cs[j], q = f > 0 ? f - 1 : (f < 0 ? -f - 1 : 0);
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {
        const double v = (double)sf[kk * tl.capf + q];
        R[kk] = f > 0 ? R[kk] + v : (f < 0 ? R[kk] - v : R[kk]);
      }
    }
    if (bm)
#pragma unroll
      for (int j = 0; j < NE; j++)
        if ((bm >> j) & 1)
#pragma unroll
          for (int kk = 0; kk < 4; kk++) R[kk] += sb[8 * (cs[j] - 1) + kk];
    const bool hold = (s.tube && s.tube[2] > 1.5) || (sv && !sv->active);
    if ((flags & F_CLAMP_UN) && !hold) {
      // the clamps act below rlim or T = e/Cv = 1; a state far from both
      // (twice the energy, no division needed to see it) is left as it is
      const double k2 = un[3] * un[0] - 0.5 * (un[1] * un[1] + un[2] * un[2]);
      if (!(un[0] > kp.rlim && k2 > 2.0 * fmax(kp.gas.Cv, 7.176325e+02) * un[0] * un[0])) prim_point<4>(kp, un, p);
    }
    double unew[4];
    const Den<double> dom(om);
#pragma unroll
    for (int kk = 0; kk < 4; kk++) unew[kk] = hold ? un0[kk] : un[kk] - dom(dt * sigma * rk_a * R[kk]);
    if (lastst) {
      dt_next = cell_dt<4>(kp, unew, om, g.dsxm[i], g.dsym[i]);
      if (flags & F_NEXT_LOCAL) dtl[i] = (sv ? sv->cfl : cfl) * dt_next;
#pragma unroll
      for (int kk = 0; kk < 4; kk++) Uout[kk * nc + i] = unew[kk];
    }
    prim_point<4>(kp, unew, p);
    store4(Pout, i, p);
  }
  if (!lastst) return;
  // residual-norm partials and time-step minimum, as k_update's
  if (t < CSU_CHUNK) {
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
      const double v = wave_reduce(R[kk] * R[kk], RedSum());
      if ((t & 63) == 0) sw[kk][t >> 6] = v;
    }
    const double v = wave_reduce(dt_next, RedMin());
    if ((t & 63) == 0) sw[4][t >> 6] = v;
  }
  __syncthreads();
  if (t == 0) {
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
      double v = sw[kk][0];
#pragma unroll
      for (int w = 1; w < CSU_CHUNK / 64; w++) v += sw[kk][w];
      red_res[kk * gridDim.x + tile] = v;
    }
    red_dt[tile] = fmin(fmin(fmin(sw[4][0], sw[4][1]), sw[4][2]), sw[4][3]);
  }
}

}  // namespace csu
