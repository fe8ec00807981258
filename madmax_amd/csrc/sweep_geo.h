// sweep_geo.h -- what a workgroup of a resident sweep (engine_sweep.hip) owns,
// publishes and reads, as functions of the split alone: the kernel runs them on
// the device and mm_sweep_check on the host.
#pragma once

#include <hip/hip_runtime.h>

#include "mm_internal.h"

namespace mm {

// The tile of one workgroup: rank rk = rz sty + ry of the RVE's scw owns the
// interior planes zs .. ze-1 and of each the nr interior rows from ys (counted
// from 0).  LDS plane s holds plane zs - 1 + s; inside a plane, node (ix, iy) of
// the tile (both counted from 0) sits at pos = 1 + (iy + 1) (nix + 1) + ix, so
// that a zero column lies between the rows, and a row before and after them
// holds the neighbouring tiles' or is zero.  Zeros stand for the boundary nodes,
// whose z is zero in every correction solve.
struct SweepGeo {
  int nix, rsx, pw;  // interior columns per row; row and plane strides
  int npos, nstrip;  // positions of a plane's rows with their zero column; strips of them
  int zs, ze, np, ys, nr, rk, cw;
  bool zlo, zhi, ylo, yhi;  // neighbouring ranks
  int lp, nch;              // planes per item; items per column
  int nx, nxy, nixy, ni;
};

__host__ __device__ __forceinline__ SweepGeo sweep_geo(int nx, int ny, int nz, int cw, int ty, int lp, int nch,
                                                       int rk)
{
  SweepGeo g;
  const int niz = nz - 2;
  g.nx = nx;
  g.nix = nx - 2;
  g.rsx = g.nix + 1;
  g.rk = rk;
  g.cw = cw;
  const int cz = cw / ty, rz = rk / ty, ry = rk - rz * ty;
  g.zs = 1 + rz * niz / cz;
  g.ze = 1 + (rz + 1) * niz / cz;
  g.np = g.ze - g.zs;
  g.ys = ry * (ny - 2) / ty;
  g.nr = (ry + 1) * (ny - 2) / ty - g.ys;
  g.zlo = rz > 0;
  g.zhi = rz + 1 < cz;
  g.ylo = ry > 0;
  g.yhi = ry + 1 < ty;
  g.pw = sweep_plane(nx, g.nr + 2);
  g.npos = g.rsx * g.nr;
  g.nstrip = sweep_strips(nx, g.nr + 2);
  g.nixy = g.nix * (ny - 2);
  g.ni = g.nixy * niz;
  g.lp = lp;
  g.nch = nch;
  g.nxy = nx * ny;
  return g;
}

// Strip st of the tile, lane ln of its wave: the LDS position of the lane's column
// in the plane below its first node, that node, the planes of the strip's run (0:
// none), and whether the lane has a node there (if not it only supplies z to its
// neighbours).  The tile has nstrip strips per run of planes; lanes 1 .. 62 work.
struct SweepItem {
  int lds, node, cnt, word;  // word: the first node's among the interior nodes
  bool on, edge;             // edge: in a row that a neighbouring rank reads
  bool first, last;          // the run holds the tile's first, last plane
};
__host__ __device__ __forceinline__ SweepItem sweep_item(const SweepGeo &g, int st, int ln)
{
  const int h = st / g.nstrip, pos = (st - h * g.nstrip) * kSweepStrip + ln - 1;
  const int iy = pos < 0 ? 0 : pos / g.rsx, ix = pos < 0 ? g.nix : pos - iy * g.rsx;
  const int zf = g.zs + h * g.lp, left = g.ze - zf, cut = left < g.lp ? left : g.lp;
  SweepItem it;
  it.cnt = h < g.nch && cut > 0 ? cut : 0;
  it.on = it.cnt > 0 && ix < g.nix && pos < g.npos && ln >= 1 && ln <= kSweepStrip;
  it.lds = (h < g.nch ? h * g.lp : 0) * g.pw + (pos < g.npos ? pos : g.npos - 1) + g.rsx + 1;
  it.node = it.on ? (ix + 1) + (g.ys + iy + 1) * g.nx + zf * g.nxy : 1 + g.nx + g.nxy;  // any interior one if off
  it.word = ix + g.nix * (g.ys + iy) + g.nixy * (zf - 1);
  it.edge = (g.ylo && iy == 0) || (g.yhi && iy == g.nr - 1);
  it.first = h == 0;
  // by position: the runs are cut for the largest share, so that a smaller one may
  // end in a run before the last and leave that empty
  it.last = zf + it.cnt == g.ze;
  return it;
}

// What the lane publishes after an update: bit l: its node l; bit 31: it has nodes.
__host__ __device__ __forceinline__ unsigned sweep_put(const SweepGeo &g, const SweepItem &it)
{
  if (!it.on) return 0u;
  const unsigned own = (1u << it.cnt) - 1u;
  unsigned put = it.edge ? own : 0u;
  if (g.zlo && it.first) put |= 1u;
  if (g.zhi && it.last) put |= own & ~(own >> 1);  // the last plane
  return put | 1u << 31;
}

// The nodes beside the tile: the planes below and above with the rows beside the
// tile (the first n1 of n), then of the tile's own planes the rows before and after
// it.  Place c of the lower side (lo: there is one) is the words of interior node at
// and the LDS position dst, of the upper side (hi) dat and ddst further on.
// (Scalars by reference: with a struct the kernel spills eight more registers.)
struct SweepHalo {
  int r0, n1, n;
};
__host__ __device__ __forceinline__ SweepHalo sweep_halo(const SweepGeo &g)
{
  SweepHalo h;
  h.r0 = g.ylo ? 0 : 1;
  h.n1 = (g.zlo || g.zhi) ? (g.nr + (g.ylo ? 1 : 0) + (g.yhi ? 1 : 0)) * g.nix : 0;
  h.n = h.n1 + ((g.ylo || g.yhi) ? g.np * g.nix : 0);
  return h;
}
__host__ __device__ __forceinline__ void sweep_place(const SweepGeo &g, int r0, int n1, int n, int c, int &at, int &dst,
                                                     int &dat, int &ddst, bool &lo, bool &hi)
{
  const bool in = c < n, plane = c < n1;
  if (!plane) c -= n1;
  const int r = c / g.nix, ix = c - r * g.nix;
  if (plane) {  // row r0 + r of planes 0 and np + 1
    at = ix + g.nix * (g.ys + r0 + r - 1) + g.nixy * (g.zs - 2);
    dst = 1 + (r0 + r) * g.rsx + ix;
    dat = (g.np + 1) * g.nixy;
    ddst = (g.np + 1) * g.pw;
  } else {  // rows 0 and nr + 1 of plane r + 1
    at = ix + g.nix * (g.ys - 1) + g.nixy * (g.zs - 1 + r);
    dst = 1 + ix + (r + 1) * g.pw;
    dat = (g.nr + 1) * g.nix;
    ddst = (g.nr + 1) * g.rsx;
  }
  lo = in && (plane ? g.zlo : g.ylo);
  hi = in && (plane ? g.zhi : g.yhi);
}

}  // namespace mm
