// fe.hip -- per-element FE assembly on the GPU: element stiffness matrices
// and residuals from a tangent / stress per gauss point, summed into the
// reference's ELL (and residual vector) by one lane per node in ascending
// element order.  Serves the micro's request path with re-assembly per
// Newton iteration (micro/src/homogenize.c:175-225), the periodic boundary
// condition (micro/src/assembly.c:175-220, 272-354) and the macro mesh
// (macro/src/assembly.c:5-222).  Every kernel is FP64 with multiply-add
// contraction off, in the reference's operation order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "fe.h"
#include "mm_device.h"

namespace mm {

namespace {

constexpr int kNnz = 81;  // ELL width of the 3D hex8 Jacobian (micro/src/alloc.c:6)
constexpr int kEB = 8;    // elements per wavefront in the residual kernel
constexpr double kGauss = 0.577350269189626;  // src/fem.c:324

// Device view of the mesh.
struct FeDev {
  int nex, ney, nez, nx, ny, nz;
  int nelm, nunk, nrow, periodic, iso, flush;
  double hx, hy, hz, vol;
  const double *coords;      // [structured node][3] (iso)
  const uint8_t *elem_mat;   // [elem]
  const double *cmat;        // [mat][36]
  const double *c_gp;        // [elem][8][36] or null
  const uint8_t *dir;        // [dof] Dirichlet flag
  int zero_cols;
};

// hex8 master derivative ds[a][i] at gauss point g (src/fem.c:364-405 order:
// node a and gauss point g at signs (-,-,-) (+,-,-) (+,+,-) (-,+,-), then z +)
__device__ __forceinline__ double hex_sign(int a, int d)
{
  if (d == 0) return (a == 1 || a == 2 || a == 5 || a == 6) ? 1.0 : -1.0;
  if (d == 1) return (a == 2 || a == 3 || a == 6 || a == 7) ? 1.0 : -1.0;
  return (a >= 4) ? 1.0 : -1.0;
}
__device__ __forceinline__ void master_ds(int a, int g, double (&ds)[3])
{
#pragma clang fp contract(off)
  double f[3];
  for (int d = 0; d < 3; d++) f[d] = 1.0 + hex_sign(a, d) * (hex_sign(g, d) * kGauss);
  ds[0] = hex_sign(a, 0) * f[1] * f[2] * 0.125;
  ds[1] = hex_sign(a, 1) * f[0] * f[2] * 0.125;
  ds[2] = hex_sign(a, 2) * f[0] * f[1] * 0.125;
}

// Structured node of local node a of element e.
__device__ __forceinline__ void elem_node(const FeDev &F, int e, int a, int &ix, int &iy, int &iz)
{
  int lx, ly, lz;
  local_coords(a, &lx, &ly, &lz);
  ix = e % F.nex + lx;
  iy = (e / F.nex) % F.ney + ly;
  iz = e / (F.nex * F.ney) + lz;
}
__device__ __forceinline__ int unknown_of(const FeDev &F, int ix, int iy, int iz)
{
  if (F.periodic) return (ix % F.nex) + (iy % F.ney) * F.nex + (iz % F.nez) * F.nex * F.ney;
  return ix + iy * F.nx + iz * F.nx * F.ny;
}
__device__ __forceinline__ void node_coord(const FeDev &F, int ix, int iy, int iz, double (&X)[3])
{
  if (F.iso) {
    const double *c = F.coords + 3 * ((long long)ix + (long long)iy * F.nx + (long long)iz * F.nx * F.ny);
    X[0] = c[0];
    X[1] = c[1];
    X[2] = c[2];
  } else {
    X[0] = ix * F.hx;
    X[1] = iy * F.hy;
    X[2] = iz * F.hz;
  }
}

// Gauss point g of element e: what its nodes' physical derivatives are formed
// from, and the weight.  Structured: ds * 2 / h, w = vol_e / 8
// (src/fem.c:42-54 extended to 3D).  Isoparametric: J = sum_n ds X, its cofactor
// inverse, dsh = J^-1 ds, w = |det J| times the unit hex8 weight
// (src/fem.c:411-471, macro/src/assembly.c:115).
struct GpGeo {
  double iJ[3][3], w;
};
__device__ void gp_geo(const FeDev &F, int e, int g, GpGeo &G)
{
#pragma clang fp contract(off)
  if (!F.iso) {
    const double vol = F.hx * F.hy * F.hz;
    G.w = vol / 8;
    return;
  }
  double J[3][3];
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++) J[i][j] = 0.0;
#pragma unroll
  for (int n = 0; n < 8; n++) {
    int ix, iy, iz;
    double X[3], ds[3];
    elem_node(F, e, n, ix, iy, iz);
    node_coord(F, ix, iy, iz, X);
    master_ds(n, g, ds);
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = 0; j < 3; j++) J[i][j] += ds[i] * X[j];
  }
  const double c00 = +J[1][1] * J[2][2] - J[2][1] * J[1][2], c01 = -J[1][0] * J[2][2] + J[2][0] * J[1][2],
               c02 = +J[1][0] * J[2][1] - J[2][0] * J[1][1];
  const double c10 = -J[0][1] * J[2][2] + J[2][1] * J[0][2], c11 = +J[0][0] * J[2][2] - J[2][0] * J[0][2],
               c12 = -J[0][0] * J[2][1] + J[2][0] * J[0][1];
  const double c20 = +J[0][1] * J[1][2] - J[1][1] * J[0][2], c21 = -J[0][0] * J[1][2] + J[1][0] * J[0][2],
               c22 = +J[0][0] * J[1][1] - J[1][0] * J[0][1];
  const double det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
  const double iJ[3][3] = {{c00 / det, c10 / det, c20 / det}, {c01 / det, c11 / det, c21 / det},
                           {c02 / det, c12 / det, c22 / det}};
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++) G.iJ[i][j] = iJ[i][j];
  G.w = fabs(det) * 1.0;
}
__device__ __forceinline__ void gp_node_dsh(const FeDev &F, const GpGeo &G, int a, int g, double (&dsh)[3])
{
#pragma clang fp contract(off)
  double ds[3];
  master_ds(a, g, ds);
  if (!F.iso) {
    dsh[0] = ds[0] * 2 / F.hx;
    dsh[1] = ds[1] * 2 / F.hy;
    dsh[2] = ds[2] * 2 / F.hz;
    return;
  }
#pragma unroll
  for (int i = 0; i < 3; i++) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < 3; j++) s += G.iJ[i][j] * ds[j];
    dsh[i] = s;
  }
}

// Reads an address that is the same in every lane through the scalar unit.
__device__ __forceinline__ double wave_load(const double *p)
{
  return *(const __attribute__((address_space(4))) double *)p;
}

// B[v][3a + d] from dsh[a][.] (Voigt xx, yy, zz, xy, yz, xz; engineering
// shears; micro/src/init.c:40-50 extended to 3D)
__device__ __forceinline__ double bval(const double (&dsh)[3], int v, int d)
{
  switch (v) {
    case 0: return d == 0 ? dsh[0] : 0.0;
    case 1: return d == 1 ? dsh[1] : 0.0;
    case 2: return d == 2 ? dsh[2] : 0.0;
    case 3: return d == 0 ? dsh[1] : (d == 1 ? dsh[0] : 0.0);
    case 4: return d == 1 ? dsh[2] : (d == 2 ? dsh[1] : 0.0);
    default: return d == 0 ? dsh[2] : (d == 2 ? dsh[0] : 0.0);
  }
}

// Rows of B with a value in column d of a node, ascending, and which of the
// node's derivatives stands there (bval).
__device__ constexpr int kBRow[3][3] = {{0, 3, 5}, {1, 3, 4}, {2, 4, 5}};
__device__ constexpr int kBDer[3][3] = {{0, 1, 2}, {1, 0, 2}, {2, 1, 0}};

// Element stiffness k[i][j] = sum_gp sum_k sum_h B[h][i] C[h][k] B[k][j] w
// (micro/src/assembly.c:97-107, macro/src/assembly.c:173-181), one wavefront
// per element: lane 8 g + a forms the derivatives of node a at gauss point g,
// then lane 8 a + b sums the 3 x 3 block of nodes a and b.  Terms with a zero
// factor are skipped (adding an exact zero leaves every sum unchanged): B's
// structural zeros by construction, a zero of C for the whole wavefront.
// Bound by FP64 issue (3 multiplies and an add per term, no contraction).  With
// one entry per lane and all 36 (k, h) pairs tested in turn it took 1.44 ms for
// 4,096 elements with full tangents and 1.37 for 720 with isotropic ones (a
// chain of branches per lane); this 0.075 and 0.025.
__global__ __launch_bounds__(256) void k_fe_ke(FeDev F, double *__restrict__ ke_out)
{
#pragma clang fp contract(off)
  __shared__ double s_dsh[4][8][8][3];
  __shared__ double s_w[4][8];
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int e = __builtin_amdgcn_readfirstlane((int)blockIdx.x * 4 + wv);
  const bool on = e < F.nelm;
  if (on) {
    GpGeo G;
    gp_geo(F, e, l >> 3, G);
    double dsh[3];
    gp_node_dsh(F, G, l & 7, l >> 3, dsh);
#pragma unroll
    for (int d = 0; d < 3; d++) s_dsh[wv][l >> 3][l & 7][d] = dsh[d];
    if ((l & 7) == 0) s_w[wv][l >> 3] = G.w;
  }
  __syncthreads();
  if (!on) return;
  const int a = l >> 3, b = l & 7;
  const double *cg = F.c_gp ? F.c_gp + (long long)e * 8 * 36
                            : F.cmat + (size_t)__builtin_amdgcn_readfirstlane((int)F.elem_mat[e]) * 36;
  const int cstep = F.c_gp ? 36 : 0;
  double acc[3][3];
#pragma unroll
  for (int d = 0; d < 3; d++)
#pragma unroll
    for (int dd = 0; dd < 3; dd++) acc[d][dd] = 0.0;
#pragma unroll 1
  for (int g = 0; g < 8; g++) {
    const double w = s_w[wv][g];
    double ba[3], bb[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
      ba[d] = s_dsh[wv][g][a][d];
      bb[d] = s_dsh[wv][g][b][d];
    }
    const double *C = cg + g * cstep;
#pragma unroll
    for (int dd = 0; dd < 3; dd++)
#pragma unroll
      for (int d = 0; d < 3; d++)
#pragma unroll
        for (int ik = 0; ik < 3; ik++)
#pragma unroll
          for (int ih = 0; ih < 3; ih++) {
            const double c = wave_load(C + kBRow[d][ih] * 6 + kBRow[dd][ik]);
            if (c == 0.0) continue;
            const double bh = ba[kBDer[d][ih]], bk = bb[kBDer[dd][ik]];
            const double t = acc[d][dd] + bh * c * bk * w;
            acc[d][dd] = (bh == 0.0 || bk == 0.0) ? acc[d][dd] : t;
          }
  }
  double *out = ke_out + (long long)e * 576 + 72 * a + 3 * b;
#pragma unroll
  for (int d = 0; d < 3; d++)
#pragma unroll
    for (int dd = 0; dd < 3; dd++) out[24 * d + dd] = acc[d][dd];
}

// Affine displacement u = E X of Voigt strain s (micro/src/homogenize.c:335-342).
__device__ __forceinline__ double affine(const double *s, const double (&X)[3], int d)
{
#pragma clang fp contract(off)
  if (d == 0) return s[0] * X[0] + s[3] / 2 * X[1] + s[5] / 2 * X[2];
  if (d == 1) return s[3] / 2 * X[0] + s[1] * X[1] + s[4] / 2 * X[2];
  return s[5] / 2 * X[0] + s[4] / 2 * X[1] + s[2] * X[2];
}

// Element residual res_e[i] = sum_gp sum_j B[j][i] sigma_j w
// (micro/src/assembly.c:45-56, macro/src/assembly.c:29-41), kEB elements per
// wavefront: lane 8 el + n loads the displacement of the element's node n (x at
// its unknown, plus E X at its true coordinates for the periodic fluctuation),
// lane 8 el + g forms the strain (all 24 terms, src order) and the stress (C
// strain, or given) of gauss point g, and the lanes then share the elements'
// rows and averages, each summed over the gauss points in order.  Optional
// outputs: the residual, the strains, and the averages' sums and weight.
// Latency-bound at the sizes in use (a handful of wavefronts); one lane per
// element took 37 us for 4,096 elements, this 13.
__global__ __launch_bounds__(64) void k_fe_res(FeDev F, const double *__restrict__ x, const double *strain,
                                              const double *__restrict__ stress_gp, double *__restrict__ res_out,
                                              double *__restrict__ eps_out, double *__restrict__ avg_out)
{
#pragma clang fp contract(off)
  __shared__ double s_u[kEB][24];
  __shared__ double s_dsh[kEB][8][24];
  __shared__ double s_es[kEB][8][12];  // strain, stress
  __shared__ double s_w[kEB][8];
  const int l = threadIdx.x, el = l >> 3, g = l & 7, e0 = blockIdx.x * kEB, e = e0 + el;
  const bool on = e < F.nelm;
  if (on) {
    int ix, iy, iz;
    elem_node(F, e, g, ix, iy, iz);
    const long long u = unknown_of(F, ix, iy, iz);
    double X[3];
    if (F.periodic) node_coord(F, ix, iy, iz, X);
    for (int d = 0; d < 3; d++)
      s_u[el][3 * g + d] = F.periodic ? x[3 * u + d] + affine(strain, X, d) : x[3 * u + d];
  }
  __syncthreads();
  if (on) {
    GpGeo G;
    gp_geo(F, e, g, G);
    double eps[6];
#pragma unroll
    for (int v = 0; v < 6; v++) eps[v] = 0.0;
#pragma unroll
    for (int a = 0; a < 8; a++) {
      double dsh[3];
      gp_node_dsh(F, G, a, g, dsh);
#pragma unroll
      for (int d = 0; d < 3; d++) s_dsh[el][g][3 * a + d] = dsh[d];
#pragma unroll
      for (int v = 0; v < 6; v++)
#pragma unroll
        for (int d = 0; d < 3; d++) eps[v] += bval(dsh, v, d) * s_u[el][3 * a + d];
    }
#pragma unroll
    for (int v = 0; v < 6; v++) {
      if (F.flush && fabs(eps[v]) < 1.0e-6) eps[v] = 0.0;
      s_es[el][g][v] = eps[v];
    }
    if (eps_out)
      for (int v = 0; v < 6; v++) eps_out[((long long)e * 8 + g) * 6 + v] = eps[v];
    const double *c = F.c_gp ? F.c_gp + ((long long)e * 8 + g) * 36 : F.cmat + (size_t)F.elem_mat[e] * 36;
#pragma unroll
    for (int i = 0; i < 6; i++) {
      double s = 0.0;
      if (stress_gp) {
        s = stress_gp[((long long)e * 8 + g) * 6 + i];
      } else {
#pragma unroll
        for (int j = 0; j < 6; j++) s += c[i * 6 + j] * eps[j];
      }
      s_es[el][g][6 + i] = s;
    }
    s_w[el][g] = G.w;
  }
  __syncthreads();
  const int ne = min(kEB, F.nelm - e0);
  if (res_out)
    for (int i = l; i < ne * 24; i += 64) {
      const int q = i / 24, r = i - q * 24, a = r / 3, d = r - a * 3;
      double s = 0.0;
      for (int k = 0; k < 8; k++) {
        const double w = s_w[q][k];
        const double dsh[3] = {s_dsh[q][k][3 * a], s_dsh[q][k][3 * a + 1], s_dsh[q][k][3 * a + 2]};
#pragma unroll
        for (int j = 0; j < 6; j++) s = s + bval(dsh, j, d) * s_es[q][k][6 + j] * w;
      }
      res_out[(long long)e0 * 24 + i] = s;
    }
  if (avg_out)  // element sums (for the volume average) and the element's weight (micro/src/homogenize.c:344-368)
    for (int i = l; i < ne * 13; i += 64) {
      const int q = i / 13, v = i - q * 13;
      double s = 0.0;
      for (int k = 0; k < 8; k++) s += (v == 12) ? s_w[q][k] : s_es[q][k][v] * s_w[q][k];
      avg_out[(long long)e0 * 13 + i] = s;
    }
}

// Unknown node u's place on the grid (or the torus).
__device__ __forceinline__ void unknown_place(const FeDev &F, int u, int &ux, int &uy, int &uz)
{
  const int sx = F.periodic ? F.nex : F.nx, sy = F.periodic ? F.ney : F.ny;
  ux = u % sx;
  uy = (u / sx) % sy;
  uz = u / (sx * sy);
}
// The c-th of the up to 8 elements around an unknown node in ascending element
// id, the order in which the reference's element loop reaches the node, and the
// node's corner a there; false if there is none (c counts absent ones too).
// Along each axis the element before the node comes first, on the torus the
// element after it at place 0 (the one before is the last).
__device__ __forceinline__ bool node_elem(const FeDev &F, int ux, int uy, int uz, int c, int &e, int &a)
{
  int lx = 1 - (c & 1), ly = 1 - ((c >> 1) & 1), lz = 1 - (c >> 2);
  if (F.periodic) {
    if (ux == 0) lx = 1 - lx;
    if (uy == 0) ly = 1 - ly;
    if (uz == 0) lz = 1 - lz;
  }
  int ex = ux - lx, ey = uy - ly, ez = uz - lz;
  if (F.periodic) {
    if (ex < 0) ex += F.nex;
    if (ey < 0) ey += F.ney;
    if (ez < 0) ez += F.nez;
  } else if (ex < 0 || ey < 0 || ez < 0 || ex >= F.nex || ey >= F.ney || ez >= F.nez) {
    return false;
  }
  e = ex + ey * F.nex + ez * F.nex * F.ney;
  a = local_node(lx, ly, lz);
  return true;
}

// Residual of unknown node u: res[3u+d] = sum over its (element, a) pairs in
// order of res_e[3a+d] (micro/src/assembly.c:57); Dirichlet dofs 0.
// Partial ||res||^2 per workgroup.
__global__ __launch_bounds__(256) void k_fe_node_res(FeDev F, const double *__restrict__ res_e,
                                                    double *__restrict__ res, double *__restrict__ part)
{
#pragma clang fp contract(off)
  __shared__ double lds[16];
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  double v[1] = {0.0};
  if (u < F.nunk) {
    int ux, uy, uz;
    unknown_place(F, u, ux, uy, uz);
    double r[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < 8; c++) {
      int e, a;
      if (!node_elem(F, ux, uy, uz, c, e, a)) continue;
#pragma unroll
      for (int d = 0; d < 3; d++) r[d] = r[d] + res_e[(long long)e * 24 + 3 * a + d];
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
      if (F.dir[3 * (long long)u + d]) r[d] = 0.0;
      res[3 * (long long)u + d] = r[d];
      v[0] += r[d] * r[d];
    }
  }
  block_sum<1>(v, lds);
  if (threadIdx.x == 0) part[blockIdx.x] = v[0];
}

// Workgroup i sums the n partial values i of width w (value i of item k at
// p[k * w + i]) in item order; out[i] receives the total.
__global__ __launch_bounds__(256) void k_fe_sum(const double *__restrict__ p, int n, int w, double *__restrict__ out)
{
  __shared__ double lds[16];
  double s[1] = {0.0};
  for (int k = threadIdx.x; k < n; k += blockDim.x) s[0] += p[(long long)k * w + blockIdx.x];
  block_sum<1>(s, lds);
  if (threadIdx.x == 0) out[blockIdx.x] = s[0];
}

// ELL rows of the unknown nodes in the reference's layout: a node's neighbours
// in first-touch order (elements ascending, then their local nodes), each
// slot the sum of the contributing element entries in ascending element
// order (src/ell.c:46-84 over micro/src/assembly.c:93-110).  Dirichlet rows
// become identity rows with their columns kept (src/ell.c:86-101); with
// zero_cols, Dirichlet columns are zeroed in the other rows.  Output in the
// slab layout of the device ELL (S rows per slab, column-major slots), and
// dinv = 1 / diagonal.
//
// 32 lanes per node, lane k for the neighbour at offset key k = (dx + 1) + 3 (dy
// + 1) + 9 (dz + 1): of the node's elements in order, those with a corner there
// contribute (at most one corner each, also on the torus, whose sides have three
// or more elements), and the slot is the number of neighbours touched before the
// key's first (element, corner).  The rows are collected in LDS and written as
// runs of kNodes * 3 rows per slot.  Bound by the write (974 bytes a row) from
// some 10^5 nodes on, by latency below.  One lane per node searching all
// (element, corner) pairs for every entry took 1.62 ms for the 4,913 nodes of a
// 16^3 block and 1.59 for the 990 of 9 x 8 x 10; this 0.024 and 0.017.
constexpr int kNodes = 16;
__global__ __launch_bounds__(32 * kNodes) void k_fe_node_ell(FeDev F, const double *__restrict__ ke, int S,
                                                            int *__restrict__ cols, double *__restrict__ vals,
                                                            double *__restrict__ dinv)
{
#pragma clang fp contract(off)
  __shared__ double s_val[kNnz][3 * kNodes];
  __shared__ int s_col[kNnz][3 * kNodes];
  const int u0 = blockIdx.x * kNodes, nd = threadIdx.x >> 5, key = threadIdx.x & 31, u = u0 + nd;
  const int nrows = 3 * min(kNodes, F.nunk - u0);
  for (int i = threadIdx.x; i < kNnz * 3 * kNodes; i += blockDim.x) {
    (&s_val[0][0])[i] = 0.0;
    (&s_col[0][0])[i] = -1;
  }
  __syncthreads();
  const bool on = u < F.nunk && key < 27;
  int pos = 64, ux, uy, uz;
  unknown_place(F, u, ux, uy, uz);
  double v[3][3];
  if (on) {
    const int dx = key % 3 - 1, dy = (key / 3) % 3 - 1, dz = key / 9 - 1;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      int e, a, lx, ly, lz;
      if (!node_elem(F, ux, uy, uz, c, e, a)) continue;
      local_coords(a, &lx, &ly, &lz);
      lx += dx;
      ly += dy;
      lz += dz;
      if (((lx | ly | lz) & ~1) != 0) continue;  // not a corner of this element
      const int b = local_node(lx, ly, lz);
      const double *k = ke + (long long)e * 576 + 72 * a + 3 * b;
#pragma unroll
      for (int d = 0; d < 3; d++)
#pragma unroll
        for (int dd = 0; dd < 3; dd++) v[d][dd] = (pos == 64) ? k[24 * d + dd] : v[d][dd] + k[24 * d + dd];
      if (pos == 64) pos = 8 * c + b;
    }
  }
  // the neighbours touched before this one
  unsigned long long touched = (pos < 64) ? 1ull << pos : 0ull;
#pragma unroll
  for (int off = 16; off > 0; off >>= 1) touched |= __shfl_xor(touched, off, 32);
  if (pos < 64) {
    const int slot = __popcll(touched & ((1ull << pos) - 1ull));
    int nb;
    if (F.periodic) {
      const int mx = ux + key % 3 - 1 + F.nex, my = uy + (key / 3) % 3 - 1 + F.ney, mz = uz + key / 9 - 1 + F.nez;
      nb = mx % F.nex + (my % F.ney) * F.nex + (mz % F.nez) * F.nex * F.ney;
    } else {
      nb = u + key % 3 - 1 + ((key / 3) % 3 - 1) * F.nx + (key / 9 - 1) * F.nx * F.ny;
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const long long row = 3LL * u + d;
      const bool drow = F.dir[row];
#pragma unroll
      for (int dd = 0; dd < 3; dd++) {
        const int col = 3 * nb + dd;
        double t = v[d][dd];
        if (drow) t = (col == row) ? 1.0 : 0.0;
        else if (F.zero_cols && F.dir[col]) t = 0.0;
        if (col == row) dinv[row] = 1 / t;
        s_val[3 * slot + dd][3 * nd + d] = t;
        s_col[3 * slot + dd][3 * nd + d] = col;
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kNnz * 3 * kNodes; i += blockDim.x) {
    const int j = i / (3 * kNodes), r = i - j * (3 * kNodes);
    if (r >= nrows) continue;
    const long long row = 3LL * u0 + r;
    const long long at = (row / S) * (long long)S * kNnz + (long long)j * S + row % S;
    cols[at] = s_col[j][r];
    vals[at] = s_val[j][r];
  }
}

// x[dof] = E X on the Dirichlet dofs (set_disp_0).
__global__ void k_fe_disp0(FeDev F, const double *strain, double *__restrict__ x)
{
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= F.nunk || F.periodic) return;
  const int ix = u % F.nx, iy = (u / F.nx) % F.ny, iz = u / (F.nx * F.ny);
  double X[3];
  node_coord(F, ix, iy, iz, X);
  for (int d = 0; d < 3; d++)
    if (F.dir[3LL * u + d]) x[3LL * u + d] = affine(strain, X, d);
}

// b = -r
__global__ void k_fe_neg(const double *__restrict__ r, double *__restrict__ b, int n)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = -r[i];
}

// x += dx
__global__ void k_fe_add(double *__restrict__ x, const double *__restrict__ dx, int n)
{
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = x[i] + dx[i];
}

__global__ void k_fe_zero(double *__restrict__ x, int n)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = 0.0;
}

}  // namespace

struct Fe {
  FeDev F;
  int device = 0;
  hipStream_t s = nullptr;
  ell_device *A = nullptr;
  int *ell_cols = nullptr;
  double *ell_vals = nullptr, *ell_dinv = nullptr;
  int S = 256;
  double *coords = nullptr, *cmat = nullptr, *c_gp = nullptr;
  uint8_t *elem_mat = nullptr, *dir = nullptr;
  double *x = nullptr, *res = nullptr, *b = nullptr, *dx = nullptr;
  double *ke = nullptr, *res_e = nullptr, *part = nullptr, *tot = nullptr, *strain = nullptr;
  double *stress_gp = nullptr, *gp_buf = nullptr, *avg = nullptr;
  std::vector<uint8_t> phase;
};

static int grid_of(long long n, int bs) { return (int)((n + bs - 1) / bs); }

int fe_create(const FeMeshDesc &d, Fe **out)
{
  if (!out || d.nex < 1 || d.ney < 1 || d.nez < 1 || !(d.lx > 0) || !(d.ly > 0) || !(d.lz > 0)) return MM_ERR_ARG;
  if (d.nmat < 1 || !d.cmat) return MM_ERR_ARG;
  if (d.periodic && (d.nex < 3 || d.ney < 3 || d.nez < 3 || d.coords)) return MM_ERR_ARG;
  const long long nn = (long long)(d.nex + 1) * (d.ney + 1) * (d.nez + 1);
  const long long nunk = d.periodic ? (long long)d.nex * d.ney * d.nez : nn;
  const long long nelm = (long long)d.nex * d.ney * d.nez;
  if (3 * nunk > 2000000000LL || nelm * 576 > (1LL << 40)) return MM_ERR_ARG;
  MM_HIP(hipSetDevice(d.device));
  Fe *f = new Fe();
  f->device = d.device;
  FeDev &F = f->F;
  memset(&F, 0, sizeof(F));
  F.nex = d.nex;
  F.ney = d.ney;
  F.nez = d.nez;
  F.nx = d.nex + 1;
  F.ny = d.ney + 1;
  F.nz = d.nez + 1;
  F.nelm = (int)nelm;
  F.nunk = (int)nunk;
  F.nrow = (int)(3 * nunk);
  F.periodic = d.periodic;
  F.iso = d.coords ? 1 : 0;
  F.flush = d.flush_strain;
  F.hx = d.lx / d.nex;
  F.hy = d.ly / d.ney;
  F.hz = d.lz / d.nez;
  F.vol = d.lx * d.ly * d.lz;
  f->phase.assign((size_t)nelm, 0);
  for (long long e = 0; e < nelm; e++) {
    const int m = d.elem_mat ? d.elem_mat[e] : 0;
    if (m < 0 || m >= d.nmat) {
      delete f;
      return MM_ERR_ARG;
    }
    f->phase[e] = (uint8_t)m;
  }
  int rc = 0;
#define FALLOC(ptr, bytes)                                          \
  do {                                                              \
    if (hipMalloc((void **)&(ptr), (bytes) ? (bytes) : 8) != hipSuccess) { \
      rc = MM_ERR_ALLOC;                                            \
      goto fail;                                                    \
    }                                                               \
  } while (0)
  if (hipStreamCreateWithFlags(&f->s, hipStreamNonBlocking) != hipSuccess) {
    delete f;
    return MM_ERR_HIP;
  }
  FALLOC(f->elem_mat, (size_t)nelm);
  FALLOC(f->cmat, (size_t)d.nmat * 36 * 8);
  FALLOC(f->dir, (size_t)F.nrow);
  FALLOC(f->x, (size_t)F.nrow * 8);
  FALLOC(f->res, (size_t)F.nrow * 8);
  FALLOC(f->b, (size_t)F.nrow * 8);
  FALLOC(f->dx, (size_t)F.nrow * 8);
  FALLOC(f->ke, (size_t)nelm * 576 * 8);
  FALLOC(f->res_e, (size_t)nelm * 24 * 8);
  FALLOC(f->avg, (size_t)nelm * 13 * 8);
  FALLOC(f->part, (size_t)(grid_of(nunk, 256) + 1) * 8);
  FALLOC(f->tot, 16 * 8);
  FALLOC(f->strain, 8 * 8);
  if (d.coords) {
    FALLOC(f->coords, (size_t)nn * 3 * 8);
    MM_HIP(hipMemcpyAsync(f->coords, d.coords, (size_t)nn * 3 * 8, hipMemcpyHostToDevice, f->s));
  }
#undef FALLOC
  if (hipMemcpyAsync(f->elem_mat, f->phase.data(), (size_t)nelm, hipMemcpyHostToDevice, f->s) != hipSuccess ||
      hipMemcpyAsync(f->cmat, d.cmat, (size_t)d.nmat * 36 * 8, hipMemcpyHostToDevice, f->s) != hipSuccess ||
      hipMemsetAsync(f->dir, 0, (size_t)F.nrow, f->s) != hipSuccess ||
      hipMemsetAsync(f->x, 0, (size_t)F.nrow * 8, f->s) != hipSuccess) {
    rc = MM_ERR_HIP;
    goto fail;
  }
  if ((rc = ell_device_alloc(F.nrow, kNnz, 256, &f->A))) goto fail;
  {
    hipStream_t as;
    ell_device_arrays(f->A, &f->ell_cols, &f->ell_vals, &f->ell_dinv, &f->S, &as);
    // the nodes of a slab's 256 rows (at most 87), and one node and its corner
    // neighbours to either side; on the torus any column
    if (!F.periodic) ell_device_set_band(f->A, 3LL * (87 + 2LL * (1 + F.nx + (long long)F.nx * F.ny)));
  }
  F.coords = f->coords;
  F.elem_mat = f->elem_mat;
  F.cmat = f->cmat;
  F.c_gp = nullptr;
  F.dir = f->dir;
  if (F.periodic) {  // the fluctuation of node (0,0,0) is pinned (all corners get u = E X)
    const uint8_t one[3] = {1, 1, 1};
    if (hipMemcpyAsync(f->dir, one, 3, hipMemcpyHostToDevice, f->s) != hipSuccess) {
      rc = MM_ERR_HIP;
      goto fail;
    }
    F.zero_cols = 1;
  }
  if (hipStreamSynchronize(f->s) != hipSuccess) {
    rc = MM_ERR_HIP;
    goto fail;
  }
  *out = f;
  return 0;
fail:
  fe_destroy(f);
  return rc ? rc : MM_ERR_HIP;
}

void fe_destroy(Fe *f)
{
  if (!f) return;
  if (f->s) (void)hipStreamSynchronize(f->s);
  void *p[] = {f->coords, f->cmat, f->c_gp, f->elem_mat, f->dir, f->x, f->res, f->b, f->dx, f->ke,
               f->res_e, f->part, f->tot, f->strain, f->stress_gp, f->gp_buf, f->avg};
  for (void *q : p)
    if (q) (void)hipFree(q);
  if (f->A) ell_device_destroy(f->A);
  if (f->s) (void)hipStreamDestroy(f->s);
  delete f;
}

int fe_sizes(const Fe *f, int *nrow, int *nelm, int *nnode)
{
  if (!f) return MM_ERR_ARG;
  if (nrow) *nrow = f->F.nrow;
  if (nelm) *nelm = f->F.nelm;
  if (nnode) *nnode = f->F.nunk;
  return 0;
}

int fe_set_dirichlet(Fe *f, int ndof, const int *dofs, int zero_cols)
{
  if (!f || ndof < 0 || (ndof && !dofs)) return MM_ERR_ARG;
  std::vector<uint8_t> h((size_t)f->F.nrow, 0);
  for (int i = 0; i < ndof; i++) {
    if (dofs[i] < 0 || dofs[i] >= f->F.nrow) return MM_ERR_ARG;
    h[dofs[i]] = 1;
  }
  if (f->F.periodic) h[0] = h[1] = h[2] = 1;
  MM_HIP(hipMemcpyAsync(f->dir, h.data(), h.size(), hipMemcpyHostToDevice, f->s));
  MM_HIP(hipStreamSynchronize(f->s));
  f->F.zero_cols = (zero_cols || f->F.periodic) ? 1 : 0;
  return 0;
}

int fe_set_dirichlet_boundary(Fe *f)
{
  if (!f || f->F.periodic) return MM_ERR_ARG;
  std::vector<int> dofs;
  const FeDev &F = f->F;
  for (int u = 0; u < F.nunk; u++) {
    const int ix = u % F.nx, iy = (u / F.nx) % F.ny, iz = u / (F.nx * F.ny);
    if (ix == 0 || iy == 0 || iz == 0 || ix == F.nx - 1 || iy == F.ny - 1 || iz == F.nz - 1)
      for (int d = 0; d < 3; d++) dofs.push_back(3 * u + d);
  }
  return fe_set_dirichlet(f, (int)dofs.size(), dofs.data(), 0);
}

int fe_set_x(Fe *f, const double *x)
{
  if (!f || !x) return MM_ERR_ARG;
  MM_HIP(hipMemcpyAsync(f->x, x, (size_t)f->F.nrow * 8, hipMemcpyHostToDevice, f->s));
  MM_HIP(hipStreamSynchronize(f->s));
  return 0;
}

int fe_get_x(Fe *f, double *x)
{
  if (!f || !x) return MM_ERR_ARG;
  MM_HIP(hipMemcpyAsync(x, f->x, (size_t)f->F.nrow * 8, hipMemcpyDeviceToHost, f->s));
  MM_HIP(hipStreamSynchronize(f->s));
  return 0;
}

static int upload_strain(Fe *f, const double *strain)
{
  double s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (strain)
    for (int i = 0; i < 6; i++) s[i] = strain[i];
  MM_HIP(hipMemcpyAsync(f->strain, s, sizeof(s), hipMemcpyHostToDevice, f->s));
  return 0;
}

int fe_set_disp_0(Fe *f, const double *strain)
{
  if (!f || !strain) return MM_ERR_ARG;
  int rc = upload_strain(f, strain);
  if (rc) return rc;
  k_fe_disp0<<<grid_of(f->F.nunk, 256), 256, 0, f->s>>>(f->F, f->strain, f->x);
  MM_HIP(hipGetLastError());
  MM_HIP(hipStreamSynchronize(f->s));
  return 0;
}

int fe_set_c_gp(Fe *f, const double *c_gp)
{
  if (!f) return MM_ERR_ARG;
  if (!c_gp) {
    f->F.c_gp = nullptr;
    return 0;
  }
  if (!f->c_gp && hipMalloc((void **)&f->c_gp, (size_t)f->F.nelm * 8 * 36 * 8) != hipSuccess) return MM_ERR_ALLOC;
  MM_HIP(hipMemcpyAsync(f->c_gp, c_gp, (size_t)f->F.nelm * 8 * 36 * 8, hipMemcpyHostToDevice, f->s));
  MM_HIP(hipStreamSynchronize(f->s));
  f->F.c_gp = f->c_gp;
  return 0;
}

static int upload_stress(Fe *f, const double *stress_gp, const double **dev)
{
  *dev = nullptr;
  if (!stress_gp) return 0;
  if (!f->stress_gp && hipMalloc((void **)&f->stress_gp, (size_t)f->F.nelm * 8 * 6 * 8) != hipSuccess)
    return MM_ERR_ALLOC;
  MM_HIP(hipMemcpyAsync(f->stress_gp, stress_gp, (size_t)f->F.nelm * 8 * 6 * 8, hipMemcpyHostToDevice, f->s));
  *dev = f->stress_gp;
  return 0;
}

int fe_residual(Fe *f, const double *strain, const double *stress_gp, double *norm)
{
  if (!f) return MM_ERR_ARG;
  int rc = upload_strain(f, strain);
  if (rc) return rc;
  const double *sg = nullptr;
  if ((rc = upload_stress(f, stress_gp, &sg))) return rc;
  const FeDev &F = f->F;
  k_fe_res<<<grid_of(F.nelm, kEB), 64, 0, f->s>>>(F, f->x, f->strain, sg, f->res_e, nullptr, nullptr);
  const int g = grid_of(F.nunk, 256);
  k_fe_node_res<<<g, 256, 0, f->s>>>(F, f->res_e, f->res, f->part);
  k_fe_sum<<<1, 256, 0, f->s>>>(f->part, g, 1, f->tot);
  MM_HIP(hipGetLastError());
  double t = 0.0;
  MM_HIP(hipMemcpyAsync(&t, f->tot, 8, hipMemcpyDeviceToHost, f->s));
  MM_HIP(hipStreamSynchronize(f->s));
  if (norm) *norm = std::sqrt(t);
  return 0;
}

int fe_get_residual(Fe *f, double *r)
{
  if (!f || !r) return MM_ERR_ARG;
  MM_HIP(hipMemcpyAsync(r, f->res, (size_t)f->F.nrow * 8, hipMemcpyDeviceToHost, f->s));
  MM_HIP(hipStreamSynchronize(f->s));
  return 0;
}

int fe_gp_strain(Fe *f, const double *strain, double *out)
{
  if (!f || !out) return MM_ERR_ARG;
  int rc = upload_strain(f, strain);
  if (rc) return rc;
  if (!f->gp_buf && hipMalloc((void **)&f->gp_buf, (size_t)f->F.nelm * 8 * 6 * 8) != hipSuccess)
    return MM_ERR_ALLOC;
  // the stress of the gauss points is computed and discarded: with a
  // stress input absent the tangent supplies it
  k_fe_res<<<grid_of(f->F.nelm, kEB), 64, 0, f->s>>>(f->F, f->x, f->strain, nullptr, nullptr, f->gp_buf, nullptr);
  MM_HIP(hipGetLastError());
  MM_HIP(hipMemcpyAsync(out, f->gp_buf, (size_t)f->F.nelm * 8 * 6 * 8, hipMemcpyDeviceToHost, f->s));
  MM_HIP(hipStreamSynchronize(f->s));
  return 0;
}

int fe_assemble(Fe *f)
{
  if (!f) return MM_ERR_ARG;
  const FeDev &F = f->F;
  k_fe_ke<<<grid_of(F.nelm, 4), 256, 0, f->s>>>(F, f->ke);
  k_fe_node_ell<<<grid_of(F.nunk, kNodes), 32 * kNodes, 0, f->s>>>(F, f->ke, f->S, f->ell_cols, f->ell_vals, f->ell_dinv);
  MM_HIP(hipGetLastError());
  MM_HIP(hipStreamSynchronize(f->s));
  return 0;
}

int fe_get_ell(Fe *f, int *cols, double *vals)
{
  if (!f || !cols || !vals) return MM_ERR_ARG;
  return ell_device_download(f->A, cols, vals);
}

int fe_solve_update(Fe *f, double rtol, int max_its, int *its)
{
  if (!f) return MM_ERR_ARG;
  const int n = f->F.nrow;
  k_fe_neg<<<grid_of(n, 256), 256, 0, f->s>>>(f->res, f->b, n);
  k_fe_zero<<<grid_of(n, 256), 256, 0, f->s>>>(f->dx, n);
  MM_HIP(hipGetLastError());
  MM_HIP(hipStreamSynchronize(f->s));
  ell_solver sv = {max_its, 0, rtol, 0.0};
  const int rc = ell_device_pcg_device(f->A, &sv, f->b, f->dx);
  if (its) *its = sv.its;
  if (rc && rc != MM_NOT_CONVERGED) return rc;
  k_fe_add<<<grid_of(n, 256), 256, 0, f->s>>>(f->x, f->dx, n);
  MM_HIP(hipGetLastError());
  MM_HIP(hipStreamSynchronize(f->s));
  return rc;
}

int fe_solve(Fe *f, const double *b, double *du, double rtol, int max_its, int *its)
{
  if (!f || !b || !du) return MM_ERR_ARG;
  const int n = f->F.nrow;
  MM_HIP(hipMemcpyAsync(f->b, b, (size_t)n * 8, hipMemcpyHostToDevice, f->s));
  k_fe_zero<<<grid_of(n, 256), 256, 0, f->s>>>(f->dx, n);
  MM_HIP(hipGetLastError());
  MM_HIP(hipStreamSynchronize(f->s));
  ell_solver sv = {max_its, 0, rtol, 0.0};
  const int rc = ell_device_pcg_device(f->A, &sv, f->b, f->dx);
  if (its) *its = sv.its;
  if (rc && rc != MM_NOT_CONVERGED) return rc;
  MM_HIP(hipMemcpyAsync(du, f->dx, (size_t)n * 8, hipMemcpyDeviceToHost, f->s));
  MM_HIP(hipStreamSynchronize(f->s));
  return rc;
}

int fe_averages(Fe *f, const double *strain, double *strain_ave, double *stress_ave, double *elem_strain,
                double *elem_stress)
{
  if (!f) return MM_ERR_ARG;
  int rc = upload_strain(f, strain);
  if (rc) return rc;
  const FeDev &F = f->F;
  k_fe_res<<<grid_of(F.nelm, kEB), 64, 0, f->s>>>(F, f->x, f->strain, nullptr, nullptr, nullptr, f->avg);
  k_fe_sum<<<13, 256, 0, f->s>>>(f->avg, F.nelm, 13, f->tot);
  MM_HIP(hipGetLastError());
  double t[16];
  MM_HIP(hipMemcpyAsync(t, f->tot, 13 * 8, hipMemcpyDeviceToHost, f->s));
  MM_HIP(hipStreamSynchronize(f->s));
  for (int v = 0; v < 6; v++) {
    if (strain_ave) strain_ave[v] = t[v] / F.vol;
    if (stress_ave) stress_ave[v] = t[6 + v] / F.vol;
  }
  if (elem_strain || elem_stress) {
    std::vector<double> h((size_t)F.nelm * 13);
    MM_HIP(hipMemcpyAsync(h.data(), f->avg, h.size() * 8, hipMemcpyDeviceToHost, f->s));
    MM_HIP(hipStreamSynchronize(f->s));
    for (int e = 0; e < F.nelm; e++)
      for (int v = 0; v < 6; v++) {
        const double *o = &h[(size_t)e * 13];
        if (elem_strain) elem_strain[(size_t)e * 6 + v] = o[v] / o[12];
        if (elem_stress) elem_stress[(size_t)e * 6 + v] = o[6 + v] / o[12];
      }
  }
  return 0;
}

int fe_get_phase(Fe *f, int *elem_type)
{
  if (!f || !elem_type) return MM_ERR_ARG;
  for (int e = 0; e < f->F.nelm; e++) elem_type[e] = f->phase[e];
  return 0;
}

}  // namespace mm
