// kern_setup.h -- set-up kernels run once per mesh.
#pragma once
#include "kern_stage.h"

namespace csu {

// HBM streaming reference: y = s x over n doubles, two per lane (16-byte
// accesses), one pair per lane over a grid that covers the arrays, with
// non-temporal loads and stores.  Of the forms measured on MI355X (grid-
// stride loops of 8-64 workgroups per CU: 4.4-4.9 TB/s read + write; one
// pair per lane: 6.2 TB/s; four pairs per lane: 5.8 TB/s; a device-to-device
// hipMemcpy: 5.3 TB/s) this one is the fastest, 6.7 TB/s: the practical
// read + write ceiling the stage kernels' bytes are compared with.
__global__ __launch_bounds__(CSU_BLOCK) void k_stream(const double2* __restrict__ x, double2* __restrict__ y,
                                                      size_t n2, double s) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n2) {
    const double a = __builtin_nontemporal_load(&x[i].x), b = __builtin_nontemporal_load(&x[i].y);
    __builtin_nontemporal_store(a * s, &y[i].x);
    __builtin_nontemporal_store(b * s, &y[i].y);
  }
}

// FP32 copy of an FP64 array (round to nearest, as a host conversion does).
__global__ __launch_bounds__(CSU_BLOCK) void k_to_f32(const double* __restrict__ src, float* __restrict__ dst,
                                                      size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = (float)src[i];
}

// The tile form's lists (struct Tile), a workgroup per tile, from the faces
// (ent, ascending), halo cells and boundary entries that the host found for
// it: the faces' vectors in entry order, and the places of every own and halo
// cell's slots and edges in the tile's lists (O1: the faces' cells, and the
// own cells' slots only).
// csl, cel, hsl, hel are zero before.  Each own face slot's face is in ent
// (HostMesh::linked), each cell across an outer face in the halo list.
// Bound by its gathers: 33 us at 400k cells in Morton order, where the host's
// loops took 30 ms.
template <bool O1>
__global__ __launch_bounds__(CSU_CHUNK) void k_tile_lists(int nc, Geo g, Tile tl, const int* __restrict__ ent,
                                                          const int* __restrict__ btgt, double* __restrict__ fx,
                                                          double* __restrict__ fy, double* __restrict__ fs,
                                                          int* __restrict__ fa, int* __restrict__ fb, short* csl,
                                                          short* cel, short* hsl, short* hel) {
  const int tile = blockIdx.x, t = threadIdx.x;
  const int e0 = tl.toff[tile], n = tl.toff[tile + 1] - e0, h0 = tl.hoff[tile], h1 = tl.hoff[tile + 1];
  // place of v in the ascending a[0 .. n)
  auto find = [](const int* a, int n, int v) {
    int lo = 0;
    while (n > 0) {
      const int half = n >> 1;
      if (a[lo + half] < v) { lo += half + 1; n -= half + 1; } else n = half;
    }
    return lo;
  };
  auto edge = [&](int cell, int j, int v) {
    if (cell / CSU_CHUNK == tile) cel[(size_t)j * nc + cell] = (short)v;
    else {
      const int h = find(tl.hcell + h0, h1 - h0, cell);
      if (h < h1 - h0) hel[(size_t)j * tl.nh + h0 + h] = (short)v;
    }
  };
  for (int k = t; k < n; k += CSU_CHUNK) {
    const int f = ent[e0 + k], a = g.fe0[f], b = g.fe1[f], sl = g.fsl[f];
    fx[e0 + k] = g.fdsx[f]; fy[e0 + k] = g.fdsy[f]; fs[e0 + k] = g.fds[f];
    if (O1) {
      fa[e0 + k] = a; fb[e0 + k] = b;
    } else {
      edge(a, sl & 3, k + 1);
      edge(b, sl >> 2, -(k + 1));
    }
  }
  const int i = tile * CSU_CHUNK + t;
  for (int j = 0; j < 4 && i < nc; j++) {
    const int cf = g.cface[(size_t)j * nc + i];
    if (cf == 0) continue;
    const int k = find(ent + e0, n, (cf > 0 ? cf : -cf) - 1) + 1;
    if (k <= n) csl[(size_t)j * nc + i] = (short)(cf > 0 ? k : -k);
  }
  for (int b = tl.boff[tile] + t; b < tl.boff[tile + 1]; b += CSU_CHUNK) {
    const int q = btgt[b], x = q >= 0 ? q : -1 - q;
    (q >= 0 ? csl[(size_t)(x & 3) * nc + (x >> 2)] : hsl[(size_t)(x & 3) * tl.nh + (x >> 2)]) =
        (short)(b - tl.boff[tile] + 1);
  }
}

// saCalcD (sa.c:703-763): distance from each cell's vertex-average centre to
// the nearest wall / wallT segment (point-to-segment, parameter clamped to
// [0, 1]), the minimum taken with the reference's strict comparison, so that
// a degenerate segment (NaN distance) is skipped as it is there.
//
// Bound by FP64 issue.  Against a division and a square root for every cell
// and segment: the segments' reciprocal lengths come from the host (Den: the
// same quotient), the minimum is taken of the squares (sqrt is monotonic, so
// the root of the least square is the least root), and a group of WD_GROUP
// consecutive segments is only evaluated where its bounding box can hold the
// nearest one: its least possible distance, less a margin above the rounding
// of the distances, does not exceed the least over all groups of the largest
// possible, nor the least found so far.  250k cells, 1,000 segments: 597 -> 162 us; the whole call, with the centres on the device, 1.32 -> 0.56 ms.
#define WD_GROUP 16
// seg: [6][nw] p0x, p0y, p1x - p0x, p1y - p0y, their squared length, 1/it;
// box: [4][ng] xlo, xhi, ylo, yhi of each group's segments of non-zero length
// (a group without one: infinities), then the largest coordinate's size.
// Cells by their centres (xc, yc), or with VERT by their vertices (cv, -1 pads
// triangles; a vertex id out of range gives a NaN centre, as far from every
// wall): the averages that the host's loop over the cells formed, which took
// longer than this kernel.
template <bool VERT>
__global__ __launch_bounds__(CSU_BLOCK) void k_wall_dist(int nc, const double* __restrict__ xc,
                                                         const double* __restrict__ yc, const int4* __restrict__ cv,
                                                         const double2* __restrict__ node, int nnode, int nw,
                                                         const double* __restrict__ seg, int ng,
                                                         const double* __restrict__ box, double* __restrict__ dist) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, ii = min(i, nc - 1);
  double x, y;
  if (VERT) {
    const int4 c = cv[ii];
    const int v[4] = {c.x, c.y, c.z, c.w >= 0 ? c.w : c.x}, np = c.w >= 0 ? 4 : 3;
    double2 p[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const bool ok = (unsigned)v[k] < (unsigned)nnode;
      p[k] = node[ok ? v[k] : 0];
      if (!ok) p[k].x = __builtin_nan("");
    }
    x = 0.0; y = 0.0;
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (k < np) { x += p[k].x; y += p[k].y; }
    x /= np; y /= np;
  } else {
    x = xc[ii]; y = yc[ii];
  }
  // a distance's coordinates carry a few roundings of their own size
  const double tx = 4e-15 * (fabs(x) + box[4 * ng]), ty = 4e-15 * (fabs(y) + box[4 * ng]);
  // group indexes are the same in every lane: scalar loads
  double ub = INFINITY;
  for (int k = 0; k < ng; k++) {
    const double dx = fmax(x - box[k], box[ng + k] - x), dy = fmax(y - box[2 * ng + k], box[3 * ng + k] - y);
    ub = fmin(ub, dx * dx + dy * dy);
  }
  ub *= 1.0 + 1e-12;
  double best = INFINITY;
  for (int k = 0; k < ng; k++) {
    const double dx = fmax(fmax(box[k] - x, x - box[ng + k]) - tx, 0.0);
    const double dy = fmax(fmax(box[2 * ng + k] - y, y - box[3 * ng + k]) - ty, 0.0);
    if (!__any(!((dx * dx + dy * dy) * (1.0 - 1e-12) > ub))) continue;
    const int j1 = min(nw, (k + 1) * WD_GROUP);
    for (int j = k * WD_GROUP; j < j1; j++) {
      const double p0x = seg[j], p0y = seg[nw + j], ex = seg[2 * nw + j], ey = seg[3 * nw + j];
      const double num = ex * (x - p0x) + ey * (y - p0y);
      double tt = Den<double>(seg[4 * nw + j], seg[5 * nw + j])(num);
      if (tt > 1.) tt = 1.;
      else if (tt < 0.) tt = 0.;
      const double rx = ex * tt + p0x - x, ry = ey * tt + p0y - y;
      const double d2 = rx * rx + ry * ry;
      if (best > d2) best = d2;
    }
    ub = fmin(ub, best);
  }
  if (i >= nc) return;
  const double d = sqrt(best);
  dist[i] = d < 1e6 ? d : 1e6;
}

}  // namespace csu
