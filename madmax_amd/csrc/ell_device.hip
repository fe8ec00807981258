// ell_device.hip -- device mirror of the reference ELL matrix and the GPU
// compute entry points of include/ell.h (ell_mvp, ell_solve_jacobi,
// ell_solve_pcg).
//
// HBM layout: rows are grouped into slabs of S rows (S a multiple of 64);
// inside a slab the slots are column-major, element (row, j) at
// slab*S*nnz + j*S + row%S, so a wavefront reading slot j of 64 consecutive
// rows issues one coalesced 256-byte (int32) / 512-byte (FP64) access.
// Padding rows of the last slab hold cols = -1, vals = 0.
//
// Bit-exactness: the SpMV accumulates each row in ascending slot order,
// stops at the first -1 and keeps multiply and add separate, which is the
// arithmetic of src/ell.c:127-141 (the reference is built without FMA).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <pthread.h>

#include "ell.h"
#include "fair_share.h"
#include "fe.h"
#include "mm_device.h"
#include "mm_internal.h"

using namespace mm;

namespace {

struct IterState {
  double bnorm, rnorm, rz, alpha, beta, err;
  int its, done, max_its, pbuf;
  double rtol, min_err;
  int pad0, pad1, pad2;  // k_pcg_fused: fault flag, and the counts a failed barrier wait saw
  int fresh;             // PCG: 1 from the start until the first update's partials exist
};

// Dot products: every workgroup of a big kernel writes its partial sums
// (part[slab * 4 + i]).  Jacobi and the PCG start sum them in a one-workgroup
// kernel (k_reduce) in slab order; in the PCG iteration every workgroup of
// the consuming kernel sums them itself, in the same order, so all hold the
// same scalars.  Kernel boundaries order producer and consumer, so no
// workgroup fences for another.
enum RedMode : int { RED_JAC = 0, RED_INIT = 1, RED_PQ = 2, RED_RR = 3 };

// The scalar steps of Jacobi-PCG, shared by every kernel that takes them so
// that they round alike.  After q = A p: alpha from p.q.  After the update:
// count the iteration, test ||r|| <= rtol ||b|| or the cap, else beta and
// the new r.z.
__device__ inline double pcg_alpha(double rz, double pq) { return rz / pq; }
__device__ inline void pcg_after_update(double rr, double rzn, double rtol, double bnorm, int max_its, int &its,
                                        double &rnorm, double &rz, double &beta, int &done)
{
  its += 1;
  rnorm = sqrt(rr);
  if (rnorm <= rtol * bnorm || its >= max_its) {
    done = 1;
  } else {
    beta = rzn / rz;
    rz = rzn;
  }
}

// Row `lane` of the slab times x: ascending slots, stop at the first -1,
// separate multiply and add.  Slots are fetched kU at a time (column ids and
// values in one round trip, the x entries in a second) and then accumulated
// in slot order, so the loads of a batch overlap instead of waiting on each
// other.  Column ids are -1 or in [0, ncol) (checked on upload), so the
// entries fetched past a row's first -1 are in bounds and are never added.
constexpr int kU = 8;
// Matrices of at most this many slabs sum the PCG partials in every
// workgroup (two launches per iteration); larger ones reduce them in
// k_reduce launches (four).  On one MI355X: 350 slabs (30^3 RVE) 0.042 ms
// against 0.045 ms per iteration; 12,070 slabs (100^3) 0.89 against 0.73.
constexpr int kSelfSumSlabs = 1024;
// Slots that k_pcg_spmv fetches ahead on matrices of up to kAheadSlabs slabs,
// where a row's chain of memory round trips is what the kernel waits for, and
// where the chip is full of waves (kU) beyond.  us per iteration with kU, 14, 21
// and 27: 46,875 rows 27.7, 25.0, 25.2, 27.4; 89,373 rows (350 slabs) 36.2, 32.5,
// 33.7, 46.
constexpr int kAhead = 14;
constexpr int kAheadSlabs = 1024;
__device__ inline double row_dot_exact(const int *__restrict__ cols, const double *__restrict__ vals,
                                       long long slab_base, int S, int nnz, int lane,
                                       const double *__restrict__ x)
{
#pragma clang fp contract(off)
  double acc = 0.0;
  for (int j0 = 0; j0 < nnz; j0 += kU) {
    int c[kU];
    double v[kU], xv[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const bool in = j0 + u < nnz;
      const long long e = slab_base + (long long)(j0 + u) * S + lane;
      c[u] = in ? __builtin_nontemporal_load(&cols[e]) : -1;
      v[u] = in ? __builtin_nontemporal_load(&vals[e]) : 0.0;
    }
#pragma unroll
    for (int u = 0; u < kU; u++) xv[u] = (c[u] >= 0) ? x[c[u]] : 0.0;
    bool stop = false;
#pragma unroll
    for (int u = 0; u < kU; u++) {
      if (c[u] == -1) {
        stop = true;
        break;
      }
      acc = acc + v[u] * xv[u];
    }
    if (stop) break;
  }
  return acc;
}

// y = A x, one lane per row (src/ell.c:127-141)
__global__ void k_spmv64_exact(const int *__restrict__ cols, const double *__restrict__ vals,
                               int nrow, int nnz, int S, const double *__restrict__ x,
                               double *__restrict__ y)
{
  const int lane = threadIdx.x;
  const long long row = (long long)blockIdx.x * S + lane;
  if (row >= nrow) return;
  const long long base = (long long)blockIdx.x * S * nnz;
  y[row] = row_dot_exact(cols, vals, base, S, nnz, lane, x);
}

// The one-workgroup reduction and the scalar steps of both solvers.
__global__ __launch_bounds__(256) void k_reduce(const double *__restrict__ part, int nslab, int mode,
                                                IterState *st)
{
  __shared__ double lds[48];
  if (st->done) return;
  if (mode == RED_JAC && st->its >= st->max_its) {  // loop condition of the reference
    if (threadIdx.x == 0) st->done = 1;
    return;
  }
  double s[3];
  group_sum_rows<3>(part, nslab, 4, s, lds);
  if (threadIdx.x != 0) return;
  switch (mode) {
    case RED_JAC:  // src/ell.c:160-180: err = ||A x - b||; stop, or update and count
      st->err = sqrt(s[0]);
      if (st->err < st->min_err) st->done = 1;
      else st->its += 1;
      break;
    case RED_INIT:
      st->bnorm = sqrt(s[0]);
      st->rnorm = sqrt(s[1]);
      st->rz = s[2];
      st->beta = 0.0;
      st->its = 0;
      st->pbuf = 0;
      st->fresh = 1;
      st->done = (st->bnorm == 0.0 || st->rnorm <= st->rtol * st->bnorm) ? 1 : 0;
      break;
    case RED_PQ:
      st->alpha = pcg_alpha(st->rz, s[0]);
      st->pbuf ^= 1;
      break;
    default:  // RED_RR: r.r and r.z are k_pcg_update's part[.][1..2]
      pcg_after_update(s[1], s[2], st->rtol, st->bnorm, st->max_its, st->its, st->rnorm, st->rz, st->beta, st->done);
  }
}

// ---- stationary Jacobi (src/ell.c:143-184) --------------------------------
// k_jac_res: r = A x - b and the partial ||r||^2 (part[.][0]).
__global__ void k_jac_res(const int *__restrict__ cols, const double *__restrict__ vals, int nrow,
                          int nnz, int S, const double *__restrict__ x, const double *__restrict__ b,
                          double *__restrict__ r, double *__restrict__ part, const IterState *st)
{
#pragma clang fp contract(off)
  __shared__ double lds[16];
  if (st->done || st->its >= st->max_its) return;
  const int lane = threadIdx.x;
  const long long row = (long long)blockIdx.x * S + lane;
  double v[1] = {0.0};
  if (row < nrow) {
    const long long base = (long long)blockIdx.x * S * nnz;
    double ri = row_dot_exact(cols, vals, base, S, nnz, lane, x);
    ri = ri - b[row];
    r[row] = ri;
    v[0] = ri * ri;
  }
  block_sum<1>(v, lds);
  if (threadIdx.x == 0) {
    part[blockIdx.x * 4] = v[0];
    part[blockIdx.x * 4 + 1] = 0.0;
    part[blockIdx.x * 4 + 2] = 0.0;
  }
}

// k_jac_upd: x -= dinv * r
__global__ void k_jac_upd(int nrow, int S, const double *__restrict__ dinv,
                          const double *__restrict__ r, double *__restrict__ x, const IterState *st)
{
#pragma clang fp contract(off)
  if (st->done) return;
  const long long row = (long long)blockIdx.x * S + threadIdx.x;
  if (row >= nrow) return;
  const double e = dinv[row] * r[row];
  x[row] = x[row] - e;
}

// ---- Jacobi-preconditioned CG in FP64 ---------------------------------------
// init: r = b - A x, z = dinv r; partials ||b||^2, ||r||^2, r.z
__global__ void k_pcg_init(const int *__restrict__ cols, const double *__restrict__ vals, int nrow,
                           int nnz, int S, const double *__restrict__ x, const double *__restrict__ b,
                           const double *__restrict__ dinv, double *__restrict__ r,
                           double2 *__restrict__ zp0, double2 *__restrict__ zp1, double *__restrict__ part)
{
  __shared__ double lds[48];
  const int lane = threadIdx.x;
  const long long row = (long long)blockIdx.x * S + lane;
  double v[3] = {0.0, 0.0, 0.0};
  if (row < nrow) {
    const long long base = (long long)blockIdx.x * S * nnz;
    const double ax = row_dot_exact(cols, vals, base, S, nnz, lane, x);
    const double bi = b[row];
    const double ri = bi - ax;
    const double zi = dinv[row] * ri;
    r[row] = ri;
    zp0[row] = make_double2(zi, 0.0);
    zp1[row] = make_double2(0.0, 0.0);
    v[0] = bi * bi;
    v[1] = ri * ri;
    v[2] = ri * zi;
  }
  block_sum<3>(v, lds);
  if (threadIdx.x == 0)
    for (int i = 0; i < 3; i++) part[blockIdx.x * 4 + i] = v[i];
}

// z and p are stored as pairs {z, p} per row, in two buffers that the
// iterations alternate between (the state's pbuf): q = A p reads the current
// buffer's pairs (one 16-byte gather per column) and writes the new p into
// the other buffer, whose z the update then writes.

// Slots j0 .. j0 + U - 1 of one row: column ids and values, fetched together.
template <int U>
struct PcgSlots {
  int c[U];
  double v[U];
};
template <int U>
__device__ __forceinline__ void pcg_fetch(const int *__restrict__ cols, const double *__restrict__ vals, int nnz, int S,
                                          long long base, int lane, int j0, PcgSlots<U> &s)
{
#pragma unroll
  for (int u = 0; u < U; u++) {
    const bool in = j0 + u < nnz;
    const long long e = base + (long long)(j0 + u) * S + lane;
    s.c[u] = in ? __builtin_nontemporal_load(&cols[e]) : -1;
    s.v[u] = in ? __builtin_nontemporal_load(&vals[e]) : 0.0;
  }
}

// Row `row` (lane `lane` of slab `slab`) of q = A p with p = z + beta p_old
// formed on the fly from the current pairs zc, both for the own row, whose p
// is stored in zn, and for every gathered column; returns q_row * p_row.
// `cur` holds the row's first U slots; accumulated in slot order whatever U is.
// Shared by the per-step kernels and the fused kernel, so all do the same
// arithmetic.  With AHEAD the next U slots are fetched before the pairs of the
// current ones are used, so a trip costs one memory round trip, not two.
template <int U, bool AHEAD>
__device__ __forceinline__ double pcg_q_row(const int *__restrict__ cols, const double *__restrict__ vals, int nnz,
                                            int S, int slab, int lane, long long row,
                                            const double2 *__restrict__ zc, double beta, double2 *__restrict__ zn,
                                            double *__restrict__ q, PcgSlots<U> cur)
{
  const long long base = (long long)slab * S * nnz;
  const double2 own = zc[row];
  double acc = 0.0;
  for (int j0 = 0; j0 < nnz; j0 += U) {
    double2 w[U];
#pragma unroll
    for (int u = 0; u < U; u++) w[u] = (cur.c[u] >= 0) ? zc[cur.c[u]] : make_double2(0.0, 0.0);
    PcgSlots<U> next;
    if (AHEAD && j0 + U < nnz) pcg_fetch<U>(cols, vals, nnz, S, base, lane, j0 + U, next);
    bool stop = false;
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (cur.c[u] == -1) {
        stop = true;
        break;
      }
      acc += cur.v[u] * (w[u].x + beta * w[u].y);
    }
    if (stop) break;
    if (!AHEAD && j0 + U < nnz) pcg_fetch<U>(cols, vals, nnz, S, base, lane, j0 + U, next);
    cur = next;
  }
  const double pi = own.x + beta * own.y;
  zn[row].y = pi;
  q[row] = acc;
  return pi * acc;
}

// Row `row` of x += alpha p, r -= alpha q, z = dinv r, the new z into the pairs
// zp; v = {r.r, r.z} terms.
struct PcgRow {
  double dinv, q, x, r, p;
};
__device__ __forceinline__ void pcg_row_load(long long row, const double *__restrict__ dinv,
                                             const double *__restrict__ q, const double *__restrict__ x,
                                             const double *__restrict__ r, PcgRow &w)
{
  w.dinv = dinv[row];
  w.q = q[row];
  w.x = x[row];
  w.r = r[row];
}
__device__ __forceinline__ void pcg_update_row(long long row, double alpha, const PcgRow &w,
                                               double2 *__restrict__ zp, double *__restrict__ x,
                                               double *__restrict__ r, double (&v)[2])
{
  const double xi = w.x + alpha * w.p;
  const double ri = w.r - alpha * w.q;
  const double zi = w.dinv * ri;
  x[row] = xi;
  r[row] = ri;
  zp[row].x = zi;
  v[0] = ri * ri;
  v[1] = ri * zi;
}

// Jacobi-PCG as two launches per iteration (one lane per row: S lanes, up to
// 1024, per workgroup).  The state is kept in two
// copies: k_pcg_spmv reads st_in (written by the PCG start or the last
// update) and writes st_out, k_pcg_update the reverse, so that no launch
// reads a copy it writes.  Workgroup 0 writes the copy.  With self_sum every
// workgroup forms the scalars from the other kernel's slab partials itself
// (the same values in every workgroup); without it (matrices of many slabs,
// where nslab workgroups reading nslab partials each would cost more than a
// launch) a k_reduce launch before each kernel has already applied them to
// st_in.

// First the update's r.r / r.z (part[.][1..2]) give the iteration count, the
// convergence test and beta (nothing to sum right after the start); then
// q = A p (pcg_q_row) with partial p.q (part[.][0]).  The row's first slots are
// asked for before the scalars are formed.  Without AHEAD four waves per SIMD, though
// the registers would allow six: 3,090,903 rows 618 us with six and 607 with four.
template <int U, bool AHEAD>
__global__ __launch_bounds__(AHEAD ? 256 : 1024)
__attribute__((amdgpu_waves_per_eu(AHEAD ? 2 : 4, AHEAD ? 8 : 4)))
void k_pcg_spmv(const int *__restrict__ cols, const double *__restrict__ vals, int nrow, int nnz, int S, int nslab,
                double2 *__restrict__ zpA, double2 *__restrict__ zpB, double *__restrict__ q,
                double *__restrict__ part, const IterState *st_in, IterState *st_out, int self_sum)
{
  __shared__ double lds[48];
  __shared__ IterState N;
  const int lane = threadIdx.x;
  const long long row = (long long)blockIdx.x * S + lane;
  PcgSlots<U> first;
  pcg_fetch<U>(cols, vals, nnz, S, (long long)blockIdx.x * S * nnz, lane, 0, first);  // padding rows hold -1
  if (lane == 0) N = *st_in;
  __syncthreads();
  if (self_sum && !N.done && !N.fresh) {
    double s[2];
    group_sum_rows<2>(part + 1, nslab, 4, s, lds);
    if (lane == 0) pcg_after_update(s[0], s[1], N.rtol, N.bnorm, N.max_its, N.its, N.rnorm, N.rz, N.beta, N.done);
    __syncthreads();
  }
  if (blockIdx.x == 0 && lane == 0) {
    IterState o = N;
    o.fresh = 0;
    *st_out = o;
  }
  if (N.done) return;
  const double beta = N.beta;
  const double2 *zc = N.pbuf ? zpB : zpA;
  double2 *zn = N.pbuf ? zpA : zpB;
  double v[1] = {0.0};
  if (row < nrow) v[0] = pcg_q_row<U, AHEAD>(cols, vals, nnz, S, blockIdx.x, lane, row, zc, beta, zn, q, first);
  block_sum<1>(v, lds);
  if (lane == 0) part[blockIdx.x * 4] = v[0];
}

// alpha from the p.q partials; x += alpha p, r -= alpha q, z = dinv r
// (pcg_update_row); partials r.r, r.z (part[.][1..2]).  The row's vectors are
// asked for before the scalars are formed, where that takes the sums (self_sum) both
// buffers' p because the state says which is the new one.  Past that, where memory
// bounds the kernel, both cost more than they hide: 3,090,903 rows 48.3 us with both,
// 44.0 with one.
__global__ void k_pcg_update(int nrow, int S, int nslab, const double *__restrict__ dinv,
                             double2 *__restrict__ zpA, double2 *__restrict__ zpB, const double *__restrict__ q,
                             double *__restrict__ x, double *__restrict__ r, double *__restrict__ part,
                             const IterState *st_in, IterState *st_out, int self_sum)
{
  __shared__ double lds[32];
  __shared__ IterState N;
  const int lane = threadIdx.x;
  const long long row = (long long)blockIdx.x * S + lane;
  const bool on = row < nrow;
  PcgRow w = {0.0, 0.0, 0.0, 0.0, 0.0};
  double pA = 0.0, pB = 0.0;
  if (on) {
    pcg_row_load(row, dinv, q, x, r, w);
    if (self_sum) {
      pA = zpA[row].y;
      pB = zpB[row].y;
    }
  }
  if (lane == 0) N = *st_in;
  __syncthreads();
  if (self_sum && !N.done) {
    double s[1];
    group_sum_rows<1>(part, nslab, 4, s, lds);
    if (lane == 0) {
      N.alpha = pcg_alpha(N.rz, s[0]);
      N.pbuf ^= 1;
    }
    __syncthreads();
  }
  if (blockIdx.x == 0 && lane == 0) *st_out = N;
  if (N.done) return;
  double2 *zp = N.pbuf ? zpB : zpA;  // the pairs whose p k_pcg_spmv wrote
  w.p = N.pbuf ? pB : pA;
  if (!self_sum && on) w.p = zp[row].y;
  double v[2] = {0.0, 0.0};
  if (on) pcg_update_row(row, N.alpha, w, zp, x, r, v);
  block_sum<2>(v, lds);
  if (lane == 0) {
    part[blockIdx.x * 4 + 1] = v[0];
    part[blockIdx.x * 4 + 2] = v[1];
  }
}

// ---- the same iteration as one persistent kernel ----------------------------
// k_pcg_fused runs up to `its` PCG iterations in one cooperative launch of G
// co-resident workgroups of 256 lanes (one slab each at a time, slabs
// blockIdx.x, +G, ...).  An iteration is q = A p for the own slabs, a grid
// barrier, p.q summed by every workgroup from the slab partials, the vector
// update of the own slabs, a second barrier and the r.r / r.z sums.  Every
// workgroup sums the same partials in the same order as the two-launch
// kernels (256 lanes, slab-strided, then block_sum) and takes the same scalar
// steps, so all of them hold the same scalars, take the same branch at the
// convergence test and match k_pcg_spmv / k_pcg_update bit for bit.  Slab partials: p.q in part[.][0], r.r and r.z in part[.][1..2];
// each is rewritten only after a barrier that every reader of the previous
// value has passed.
constexpr int kFusedLanes = 256;
// Grid barrier words, each on a 256-byte line of its own (index * kBarLine):
// line 0 the release word, line 1 the count of groups arrived, line 2 + g
// the count of arrivals of group g (kBarGroup consecutive workgroups).
constexpr int kBarLine = 64;
constexpr int kBarGroup = 16;
constexpr int kBarMaxGroups = 64;
constexpr int kBarMaxGrid = kBarGroup * kBarMaxGroups;
constexpr size_t kBarBytes = (size_t)(2 + kBarMaxGroups) * kBarLine * sizeof(unsigned);
// Bound on a barrier wait in polls (each polls an agent-scope atomic, then
// sleeps): far above any legitimate wait (the slowest workgroup's phase),
// and a wait that reaches it marks the launch as faulted instead of hanging.
constexpr unsigned kBarSpinLimit = 1u << 22;

// Barrier n (1, 2, ... within a launch; the host zeroes the words before
// it).  After the workgroup barrier, lane 0 arrives at its group's counter
// with a release RMW at agent scope (the L2s of the XCDs are not coherent
// with each other, so this writes the workgroup's stores back); the last
// arrival of the group acquires and arrives at the group count; the last
// group's arrival acquires and publishes n in the release word, which every
// lane 0 polls and then acquires, before the workgroup barrier hands the
// ordering on to the other waves (HIP's own grid sync uses the same chain).
// Two levels keep the same-address atomics to 16 per group counter and one
// per group at the top, and the polls off the counters' lines.  Returns
// false when the wait gave up; the first workgroup to give up leaves the
// fault flag set (fault[0]) and the group count it saw against the count it
// waited for (fault[1], fault[2]; the IterState words after pad0).
__device__ inline bool grid_barrier(unsigned *bar, unsigned n, int *fault, int &ok_lds)
{
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned G = gridDim.x, g = blockIdx.x / kBarGroup;
    const unsigned ngroups = (G + kBarGroup - 1) / kBarGroup;
    const unsigned gsize = (G - g * kBarGroup) < kBarGroup ? (G - g * kBarGroup) : kBarGroup;
    unsigned old = __hip_atomic_fetch_add(&bar[(2 + g) * kBarLine], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    if (old + 1 == n * gsize) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      old = __hip_atomic_fetch_add(&bar[kBarLine], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      if (old + 1 == n * ngroups) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        __hip_atomic_store(&bar[0], n, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    unsigned spins = 0;
    int ok = 1;
    while (__hip_atomic_load(&bar[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < n) {
      if (++spins > kBarSpinLimit ||
          ((spins & 63) == 0 && __hip_atomic_load(fault, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
        ok = 0;
        break;
      }
      __builtin_amdgcn_s_sleep(2);
    }
    if (!ok) {
      __hip_atomic_store(fault + 1, (int)__hip_atomic_load(&bar[kBarLine], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(fault + 2, (int)(n * ngroups), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(fault, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    ok_lds = ok;
  }
  __syncthreads();
  return ok_lds != 0;
}

__global__ __launch_bounds__(kFusedLanes) void k_pcg_fused(
    const int *__restrict__ cols, const double *__restrict__ vals, int nrow, int nnz, int nslab,
    const double *__restrict__ dinv, double *__restrict__ x, double *__restrict__ r, double2 *__restrict__ zpA,
    double2 *__restrict__ zpB, double *__restrict__ q, double *__restrict__ part, IterState *st, unsigned *bar,
    int its)
{
  constexpr int S = kFusedLanes;
  __shared__ double lds[48];
  __shared__ double bc[2];
  __shared__ int ok_lds;
  if (st->done) return;
  const unsigned G = gridDim.x;
  const int lane = threadIdx.x;
  double beta = st->beta, rz = st->rz, alpha = st->alpha, rnorm = st->rnorm;
  const double bnorm = st->bnorm, rtol = st->rtol;
  int pbuf = st->pbuf, n = st->its, done = 0;
  const int max_its = st->max_its;
  int *fault = &st->pad0;
  unsigned arrivals = 0;
  int k = 0;
  for (; k < its && !done; k++) {
    const double2 *zc = pbuf ? zpB : zpA;
    double2 *zn = pbuf ? zpA : zpB;
    for (int slab = blockIdx.x; slab < nslab; slab += G) {
      const long long row = (long long)slab * S + lane;
      double v[1] = {0.0};
      PcgSlots<kU> first;
      pcg_fetch<kU>(cols, vals, nnz, S, (long long)slab * S * nnz, lane, 0, first);
      if (row < nrow) v[0] = pcg_q_row<kU, false>(cols, vals, nnz, S, slab, lane, row, zc, beta, zn, q, first);
      block_sum<1>(v, lds);
      if (lane == 0) part[slab * 4] = v[0];
    }
    if (!grid_barrier(bar, ++arrivals, fault, ok_lds)) return;
    double s1[1], s[2];
    group_sum_rows<1>(part, nslab, 4, s1, lds);
    if (lane == 0) bc[0] = s1[0];
    __syncthreads();
    alpha = pcg_alpha(rz, bc[0]);
    pbuf ^= 1;
    double2 *zp = pbuf ? zpB : zpA;  // = zn
    for (int slab = blockIdx.x; slab < nslab; slab += G) {
      const long long row = (long long)slab * S + lane;
      double v[2] = {0.0, 0.0};
      if (row < nrow) {
        PcgRow w;
        pcg_row_load(row, dinv, q, x, r, w);
        w.p = zp[row].y;
        pcg_update_row(row, alpha, w, zp, x, r, v);
      }
      block_sum<2>(v, lds);
      if (lane == 0) {
        part[slab * 4 + 1] = v[0];
        part[slab * 4 + 2] = v[1];
      }
    }
    if (!grid_barrier(bar, ++arrivals, fault, ok_lds)) return;
    group_sum_rows<2>(part + 1, nslab, 4, s, lds);
    if (lane == 0) {
      bc[0] = s[0];
      bc[1] = s[1];
    }
    __syncthreads();
    pcg_after_update(bc[0], bc[1], rtol, bnorm, max_its, n, rnorm, rz, beta, done);
    __syncthreads();  // bc is rewritten by the next iteration
  }
  // Every workgroup read the state before its first arrival, and workgroup 0
  // writes it only after that barrier completed.
  if (blockIdx.x == 0 && lane == 0 && k > 0) {
    st->its = n;
    st->rnorm = rnorm;
    st->rz = rz;
    st->alpha = alpha;
    st->beta = beta;
    st->pbuf = pbuf;
    st->done = done;
    st->fresh = 0;
  }
}

// ---- the same iteration with the matrix on chip ------------------------------
// k_pcg_resident runs a whole solve in one launch, one workgroup per slab of 256
// rows.  Each lane holds its row: the values and the LDS places of its columns
// (two to a register) for the whole solve, x, r, z and p too (in LDS with LIST).  p
// of the slab's columns (LIST: those it has entries in) lives in LDS: after an update the owners publish z
// as tagged words, and every workgroup forms p = z + beta p for its columns, the
// same bits as the owner.  p.q and {r.r, r.z} go round as tagged
// words too and are summed by every workgroup in the order of the other mappings
// (group_sum_rows: slab-strided, then block_sum).  With the same row arithmetic
// and scalar steps all mappings give the same bits.
//
// Bound by the two exchanges of an iteration and the columns' z between them;
// the two launches per iteration that it replaces were bound by the host's
// launches for small matrices and by reading 12 bytes per entry for larger ones.
// Elasticity systems of N^3 elements with 81 slots, time of a solve by its iterations
// (81 .. 241), us, two launches against this: 2,970 rows 22.7 and 7.4, 14,739 rows 23.6
// and 8.2, 46,875 rows 25.0 and 9.6, 89,373 rows 32.5 and 13.0 (11.7 each beside what
// a solve takes once).
//
// All workgroups have to run at the same time.  They are at most three quarters of what
// the CUs take, two to a CU (one where the LDS of two does not fit): 384 or 192 of 256
// CUs, which leaves a quarter for kernels of other streams that wait for workgroups of
// their own, as the engine's sweeps do (at most 15 CUs each).  Solves of one process
// share that (FairShare).  Beside other work they may still not find their CUs, for
// instance beside another process's solves: they meet before their first exchange, and
// a solve that did not meet, some 10 ms later, is done in the two-launch form, as are
// the mirror's next ones (1, 3, 7, .. 63 of them until one meets again).  After the
// meeting all of them run; the waits are bounded all the same.
constexpr int kResSlots = 81;  // rows of 27 nodes' 3 dofs; five registers for two slots, 203 of 256
                              // (20 to 28 of the others spill, outside the product)
constexpr int kResRest = 63;  // most solves in two launches between attempts
inline int res_cus(int ncu) { return ncu - ncu / 4; }
constexpr int kResOneCuLds = 69 * 1024;  // dynamic LDS up to which two workgroups fit a CU
constexpr int kResMaxLds = 149 * 1024;
constexpr int kResPolls = 1 << 18;  // about 0.2 s
constexpr int kResMaxDevices = 64;
// Spans from which a slab lists the columns it has entries in, in place of keeping
// all: the list costs 20 us a solve and a look-up, and saves asking for columns.
// us an iteration without and with it, spans of 867, 1,359, 2,103 and 6,219 columns:
// 5.3 and 5.5, 6.7 and 6.6, 7.6 and 7.0, 15.9 and 11.6.
constexpr int kResListSpan = 1536;

// Sums NV values over all slabs, valid in every lane: lane 0 of each workgroup
// has posted its own (NV doubles at sums + slab * 8).  False, in every lane, when
// a wait of this workgroup ran out since the solve began (`fail`, LDS).
template <int NV>
__device__ __forceinline__ bool res_collect(const word_t *sums, int nslab, unsigned tag, double (&out)[NV],
                                            double (&lds)[48], double *bc, int *fail)
{
#pragma unroll
  for (int i = 0; i < NV; i++) out[i] = 0.0;
  for (int b = threadIdx.x; b < nslab; b += blockDim.x) {
    word_t w[2 * NV];
    int n = 0;
    for (;;) {
      bool all = true;
#pragma unroll
      for (int i = 0; i < 2 * NV; i++) w[i] = get_word(sums + (long long)b * 8 + i);
#pragma unroll
      for (int i = 0; i < 2 * NV; i++) all = all && (unsigned)(w[i] >> 32) == tag;
      if (all) break;
      if (++n > kResPolls) {
        *fail = 1;
        break;
      }
    }
#pragma unroll
    for (int i = 0; i < NV; i++) out[i] += word_double(w[2 * i], w[2 * i + 1]);
  }
  block_sum<NV>(out, lds);
  if (threadIdx.x == 0)
#pragma unroll
    for (int i = 0; i < NV; i++) bc[i] = out[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NV; i++) out[i] = bc[i];
  return __builtin_amdgcn_readfirstlane(*fail) == 0;
}

extern __shared__ __attribute__((aligned(16))) double res_p[];

// A product that is rounded before it is summed (not contracted into the sum).
__device__ __forceinline__ double rounded(double v)
{
  asm volatile("" : "+v"(v));
  return v;
}

// zw: two words per row (z of the last update), sums: 16 words per slab, all
// zero on entry (no iteration's tag; two words of the first slab's are for the
// meeting); zp[row].x is the first z, .y receives x.  stay_away: call the meeting off.
template <bool LIST>
__global__ __launch_bounds__(256, 2) void k_pcg_resident(const int *__restrict__ cols, const double *__restrict__ vals,
                                                         int nrow, int nnz, int nslab, int lds_rows,
                                                         const double *__restrict__ dinv, const double *__restrict__ x0,
                                                         const double *__restrict__ r0, double2 *__restrict__ zp,
                                                         word_t *zw, word_t *sums, IterState *st, int stay_away)
{
  __shared__ double lds[48];
  __shared__ double bc[2];
  __shared__ double s_row[LIST ? 5 : 1][256];  // x, dinv, r, z and p of the rows, where the registers are full
  __shared__ int s_lo, s_hi, s_fail, s_place, s_wave[4];
  if (st->done) return;
  const int lane = threadIdx.x, slab = blockIdx.x;
  const long long row = (long long)slab * 256 + lane, base = (long long)slab * 256 * nnz;
  const bool on = row < nrow;
  if (lane == 0) {
    s_lo = nrow;
    s_hi = -1;
    s_fail = 0;
  }
  __syncthreads();
  // the row up to its first -1, column places two to a register; the slots
  // after it add -0.0 * res_p[nneed] = -0.0, which changes no sum
  double v[kResSlots];
  unsigned o[(kResSlots + 1) / 2];
  unsigned short *need = reinterpret_cast<unsigned short *>(res_p + lds_rows + 1);
  const int *rc = cols + base + lane;
  const double *rv = vals + base + lane;
  int cnt = 0, lo = nrow, hi = -1;
  bool more = on;
#pragma unroll 1
  for (int u0 = 0; u0 < nnz; u0 += 9) {
    int c[9];
#pragma unroll
    for (int u = 0; u < 9; u++) c[u] = (on && u0 + u < nnz) ? rc[(u0 + u) * 256] : -1;
#pragma unroll
    for (int u = 0; u < 9; u++) {
      more = more && c[u] != -1;
      lo = more ? min(lo, c[u]) : lo;
      hi = more ? max(hi, c[u]) : hi;
      cnt += more ? 1 : 0;
    }
  }
  if (cnt > 0) {
    atomicMin(&s_lo, lo);
    atomicMax(&s_hi, hi);
  }
  __syncthreads();
  lo = __builtin_amdgcn_readfirstlane(s_lo);
  hi = __builtin_amdgcn_readfirstlane(s_hi);
  if (hi - lo >= lds_rows) {  // (the host sized the LDS by the widest slab)
    if (lane == 0) {
      meet_off(sums + 6);
      st->pad0 = 1;
    }
    return;
  }
  if (lane == 0) {
    if (stay_away) meet_off(sums + 6);
    s_place = meet_arrive(sums + 6, nslab);
  }
  // with LIST only the columns that the slab has entries in get a place, else all
  // between the lowest and the highest: they are marked in bytes (neighbouring rows
  // share columns, so that an atomic on bits would meet 64 lanes at a word), then
  // as bits, 32 columns a word: a column's place is its rank, and need lists them.
  // In res_p's place until p is there.
  unsigned *bits = reinterpret_cast<unsigned *>(res_p);
  const int nw = LIST && hi >= lo ? (hi - lo) / 32 + 1 : 0;
  unsigned char *mark = reinterpret_cast<unsigned char *>(bits + nw);
  unsigned short *rank = reinterpret_cast<unsigned short *>(mark + 32 * nw);
  for (int w = lane; w < 8 * nw; w += 256) reinterpret_cast<unsigned *>(mark)[w] = 0;
  __syncthreads();
#pragma unroll 1
  for (int u0 = 0; u0 < (LIST ? nnz : 0); u0 += 9) {
    int c[9];
#pragma unroll
    for (int u = 0; u < 9; u++) c[u] = u0 + u < cnt ? rc[(u0 + u) * 256] - lo : -1;
#pragma unroll
    for (int u = 0; u < 9; u++)
      if (c[u] >= 0) mark[c[u]] = 1;
  }
  __syncthreads();
  for (int w = 2 * (lane >> 6); w < nw; w += 8) {
    const int e = 32 * w + (lane & 63);
    const unsigned long long b = __ballot(e < 32 * nw && mark[min(e, 32 * nw - 1)] != 0);
    if ((lane & 63) == 0) {
      bits[w] = (unsigned)b;
      if (w + 1 < nw) bits[w + 1] = (unsigned)(b >> 32);
    }
  }
  __syncthreads();
  const int per = (nw + 255) / 256;
  int mine = 0;
  for (int w = lane * per; w < min((lane + 1) * per, nw); w++) mine += __popc(bits[w]);
  int at = mine;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int t = __shfl_up(at, off, 64);
    if ((lane & 63) >= off) at += t;
  }
  if ((lane & 63) == 63) s_wave[lane >> 6] = at;
  __syncthreads();
  at -= mine;
  for (int w = 0; w < (lane >> 6); w++) at += s_wave[w];
  const int nneed = LIST ? s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3] : max(hi - lo + 1, 0);
  for (int w = lane * per; w < min((lane + 1) * per, nw); w++) {
    for (unsigned b = bits[w]; b; b &= b - 1) {
      const int e = w * 32 + __ffs(b) - 1;
      rank[e] = (unsigned short)at;
      need[at++] = (unsigned short)e;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u0 = 0; u0 < kResSlots; u0 += 9) {
#pragma unroll
    for (int u = u0; u < u0 + 9; u++) {
      unsigned c = nneed;
      v[u] = -0.0;
      if (u < cnt) {
        c = rc[u * 256] - lo;
        if (LIST) c = rank[c];
        v[u] = rv[u * 256];
      }
      if (u & 1) o[u / 2] |= c << 16;
      else o[u / 2] = c;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();  // the tables make way for p
  int most = cnt;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) most = max(most, __shfl_xor(most, off, 64));
  most = __builtin_amdgcn_readfirstlane(most);
  double xi = on ? x0[row] : 0.0, di = on ? dinv[row] : 0.0, ri = on ? r0[row] : 0.0, zi = on ? zp[row].x : 0.0;
  double pi = 0.0;
  if constexpr (LIST) {
    s_row[0][lane] = xi;
    s_row[1][lane] = di;
    s_row[2][lane] = ri;
    s_row[3][lane] = zi;
    s_row[4][lane] = pi;
  }
  for (int e = lane; e <= nneed; e += 256) res_p[e] = 0.0;
  if (lane == 0 && !meet_wait(sums + 6, s_place, kMeetPolls)) s_fail = 1;
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(s_fail)) {
    if (lane == 0) st->pad0 = 1;
    return;
  }
  const double bnorm = st->bnorm, rtol = st->rtol;
  const int max_its = st->max_its;
  double rz = st->rz, beta = 0.0, alpha = 0.0, rnorm = st->rnorm;
  int n = 0, done = 0;
#pragma unroll 1
  for (;;) {
    if (n > 0) {
      double s[2];
      if (!res_collect<2>(sums + (long long)nslab * 8, nslab, (unsigned)n, s, lds, bc, &s_fail)) break;
      int its = n - 1;
      pcg_after_update(s[0], s[1], rtol, bnorm, max_its, its, rnorm, rz, beta, done);
      if (__builtin_amdgcn_readfirstlane(done)) break;
    }
    // p = z + beta p for the slab's columns, four per lane and trip
    for (int e0 = lane; e0 < nneed; e0 += 4 * 256) {
      double z[4];
      int listed[4];
      if constexpr (LIST) {
#pragma unroll
        for (int i = 0; i < 4; i++) listed[i] = lo + need[min(e0 + 256 * i, nneed - 1)];
      }
      const auto col = [&](int i) {
        if constexpr (LIST) return listed[i];
        else return min(lo + e0 + 256 * i, hi);
      };
      if (n == 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) z[i] = zp[col(i)].x;
      } else {
        word_t a[4], b[4];
        int m = 0;
        for (;;) {
          bool all = true;
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const word_t *w = zw + 2LL * col(i);
            a[i] = get_word(w);
            b[i] = get_word(w + 1);
          }
#pragma unroll
          for (int i = 0; i < 4; i++)
            all = all && (unsigned)(a[i] >> 32) == (unsigned)n && (unsigned)(b[i] >> 32) == (unsigned)n;
          if (all) break;
          if (++m > kResPolls) {
            s_fail = 1;
            break;
          }
        }
#pragma unroll
        for (int i = 0; i < 4; i++) z[i] = word_double(a[i], b[i]);
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (e0 + 256 * i < nneed) res_p[e0 + 256 * i] = fma(beta, res_p[e0 + 256 * i], z[i]);
    }
    if constexpr (LIST) s_row[4][lane] = fma(beta, s_row[4][lane], s_row[3][lane]);
    else pi = fma(beta, pi, zi);
    __syncthreads();
    // (o is taken apart anew each time: the places would not fit the registers)
#pragma unroll
    for (int u = 0; u < (kResSlots + 1) / 2; u++) asm volatile("" : "+v"(o[u]));
    double qi = 0.0;
#pragma unroll
    for (int u0 = 0; u0 < kResSlots; u0 += 9) {
      if (u0 < most) {
        double t[9];
#pragma unroll
        for (int u = 0; u < 9; u++) t[u] = res_p[((u0 + u) & 1) ? o[(u0 + u) / 2] >> 16 : o[(u0 + u) / 2] & 0xffffu];
#pragma unroll
        for (int u = 0; u < 9; u++) qi = fma(v[u0 + u], t[u], qi);
      }
    }
    const unsigned tag = (unsigned)n + 1u;
    if constexpr (LIST) pi = s_row[4][lane];
    double s1[1] = {rounded(pi * qi)};
    block_sum<1>(s1, lds);
    if (lane == 0) put_double(sums + (long long)slab * 8, tag, s1[0]);
    if (!res_collect<1>(sums, nslab, tag, s1, lds, bc, &s_fail)) break;
    alpha = pcg_alpha(rz, s1[0]);
    if constexpr (LIST) {
      xi = s_row[0][lane];
      di = s_row[1][lane];
      ri = s_row[2][lane];
      pi = s_row[4][lane];
    }
    xi = fma(alpha, pi, xi);
    ri = fma(-alpha, qi, ri);
    zi = di * ri;
    if constexpr (LIST) {
      s_row[0][lane] = xi;
      s_row[2][lane] = ri;
      s_row[3][lane] = zi;
    }
    if (on) put_double(zw + 2 * row, tag, zi);
    double s2[2] = {rounded(ri * ri), rounded(ri * zi)};  // (zero beyond the last row)
    block_sum<2>(s2, lds);
    if (lane == 0) {
      put_double(sums + (long long)(nslab + slab) * 8, tag, s2[0]);
      put_double(sums + (long long)(nslab + slab) * 8 + 2, tag, s2[1]);
    }
    n++;
  }
  if (s_fail) {
    if (lane == 0) st->pad0 = 1;  // (any of them may; the host reads it after the kernel)
    return;
  }
  if (on) zp[row].y = LIST ? s_row[0][lane] : xi;
  if (slab == 0 && lane == 0) {
    st->its = n;
    st->rnorm = rnorm;
    st->rz = rz;
    st->alpha = alpha;
    st->beta = beta;
    st->done = done;
    st->fresh = 0;
  }
}

// Its LDS for slabs spanning `rows` columns: p and a zero, and the columns' list.
static size_t res_lds(int rows) { return (size_t)(rows + 1) * sizeof(double) + (size_t)rows * sizeof(short); }

// The exchange sums of k_pcg_resident (its z words are zeroed by k_pcg_init).
__global__ void k_res_zero(word_t *sums, int n)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) sums[i] = 0;
}

// x after a resident solve that succeeded.
__global__ void k_res_take(const IterState *st, const double2 *__restrict__ zp, double *__restrict__ x, int n)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && !st->fresh && !st->pad0) x[i] = zp[i].y;
}

// Zeroes the barrier words of k_pcg_fused (a kernel, not a memset node).
__global__ void k_bar_reset(unsigned *bar)
{
  if (threadIdx.x < 2 + kBarMaxGroups) bar[threadIdx.x * kBarLine] = 0u;
}

// x = 0 (a kernel, not a memset node, so that the solve can sit in a graph)
__global__ void k_zero(double *__restrict__ x, int n)
{
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = 0.0;
}

// PCG work vectors of one solve
struct PcgVecs {
  double *r;
  double2 *zpA, *zpB;  // {z, p} pairs, two buffers
  double *q, *part;
  IterState *st;   // two copies (the two-launch iteration passes the state between them)
  unsigned *bar;   // grid-barrier words of k_pcg_fused
};

// ---- between the host's row-major layout and the slabs ----------------------
// PLACE: rows of `rm` (row-major) into the slabs at `sl`, whose rows beyond `rows`
// get `pad`; else the reverse.  64 rows by 16 slots per trip through the LDS, so
// that both sides are read and written in runs of 64 to 512 bytes.  Bound by the
// host's copies (28 GB/s in, 17 out), which move 12 bytes per entry as the loops
// on the host did that this replaces: 14,688 rows of 81 slots up 6.5 ms before
// and 0.55 now, down 3.3 and 0.87.
constexpr int kPlaceSlots = 16;
template <typename T, bool PLACE>
__global__ __launch_bounds__(256) void k_ell_place(T *__restrict__ rm, int rows, int nnz, int S, T pad,
                                                   T *__restrict__ sl)
{
  __shared__ T tile[64][kPlaceSlots + 1];
  const int tid = threadIdx.x, per = S / 64;
  const int r0 = blockIdx.x * 64;  // first row of the tile, S a multiple of 64
  T *slab = sl + (long long)(blockIdx.x / per) * S * nnz + (blockIdx.x % per) * 64;
  T *row = rm + (long long)r0 * nnz;
  for (int j0 = blockIdx.y * kPlaceSlots; j0 < nnz; j0 += gridDim.y * kPlaceSlots) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int jr = tid % kPlaceSlots, rr = tid / kPlaceSlots + 16 * i;  // along a row
      const int js = tid / 64 + 4 * i, rs = tid % 64;                    // along a slot
      if (PLACE) {
        tile[rr][jr] = (r0 + rr < rows && j0 + jr < nnz) ? row[(long long)rr * nnz + j0 + jr] : pad;
      } else {
        tile[rs][js] = (j0 + js < nnz) ? slab[(long long)(j0 + js) * S + rs] : pad;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int jr = tid % kPlaceSlots, rr = tid / kPlaceSlots + 16 * i;
      const int js = tid / 64 + 4 * i, rs = tid % 64;
      if (PLACE) {
        if (j0 + js < nnz) slab[(long long)(j0 + js) * S + rs] = tile[rs][js];
      } else {
        if (r0 + rr < rows && j0 + jr < nnz) row[(long long)rr * nnz + j0 + jr] = tile[rr][jr];
      }
    }
    __syncthreads();
  }
}

// Of each row up to its first -1: the inverse of the diagonal (1 / 0 = inf where
// there is none, like the reference), and the most columns that the rows of one
// slab span into *band.
__global__ void k_ell_scan(const int *__restrict__ cols, const double *__restrict__ vals, int nrow, int ncol, int nnz,
                           int S, double *__restrict__ dinv, int *band)
{
  __shared__ int s_lo, s_hi;
  const int lane = threadIdx.x;
  const long long row = (long long)blockIdx.x * S + lane, base = (long long)blockIdx.x * S * nnz + lane;
  if (lane == 0) {
    s_lo = ncol;
    s_hi = -1;
  }
  __syncthreads();
  if (row < nrow) {
    double d = 0.0;
    int lo = ncol, hi = -1;
    bool found = false, more = true;
    for (int j0 = 0; j0 < nnz && more; j0 += 9) {
      int c[9];
#pragma unroll
      for (int u = 0; u < 9; u++) c[u] = j0 + u < nnz ? cols[base + (long long)(j0 + u) * S] : -1;
#pragma unroll
      for (int u = 0; u < 9; u++) {
        more = more && c[u] != -1;
        if (!more) continue;
        lo = min(lo, c[u]);
        hi = max(hi, c[u]);
        if (!found && c[u] == row) {
          found = true;
          d = vals[base + (long long)(j0 + u) * S];
        }
      }
    }
    dinv[row] = 1 / d;
    atomicMin(&s_lo, lo);
    atomicMax(&s_hi, hi);
  }
  __syncthreads();
  if (lane == 0 && band) atomicMax(band, max(s_hi - s_lo + 1, 1));
}

__global__ void k_zero_int(int *p, int n)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

}  // namespace

struct ell_device_ {
  int nrow, ncol, nnz, S, nslab;
  int device;  // HIP device the mirror lives on
  int *cols;
  double *vals, *dinv;
  double *x, *b, *r, *q, *part;
  double2 *zpA, *zpB;  // PCG {z, p} pairs
  IterState *st;
  unsigned *bar;
  char *stage;     // row-major entries on their way in or out (null until the first)
  pthread_mutex_t stage_mu;  // of downloads, which may overlap
  int band;        // most columns that a slab's rows span (0: not known)
  int ncu;         // CUs of the device
  // k_pcg_resident: solves to do otherwise before the next attempt, and how many that
  // was last time; solves that stayed, and that were given up; tests: never meet
  int res_rest, res_rested, res_stayed, res_left, res_away;
  int fused_its;   // 0: two launches per PCG iteration; n > 0: k_pcg_fused, n iterations per launch
  int fused_grid;  // co-resident workgroups of k_pcg_fused (set with fused_its)
  hipStream_t stream;
};

// The kernels read x[col] for every column id, so each must be -1 or a
// column of the matrix (ell_add_val never stores anything else).
static int check_cols(const ell_matrix *m)
{
  const size_t n = (size_t)m->nrow * m->nnz;
  const int *c = m->cols;
  const unsigned top = (unsigned)m->ncol;  // c + 1 as unsigned: 0 for -1, past top for what is out of range
  unsigned bad = 0;
  for (size_t e = 0; e < n; e++) bad |= (unsigned)c[e] + 1u > top;
  if (!bad) return 0;
  for (size_t e = 0; e < n; e++)
    if ((unsigned)c[e] + 1u > top) {
      fprintf(stderr, "madmax_amd: ell column id %d at slot %zu outside [-1, %d)\n", c[e], e, m->ncol);
      break;
    }
  return 1;
}

// Slabs whose row-major entries (cols and vals, 12 bytes) are staged on the
// device at a time: up to 64 MiB, at least one slab.
static int stage_slabs(const ell_device *d)
{
  const size_t slab = (size_t)d->S * d->nnz * 12, most = ((size_t)64 << 20) / (slab ? slab : 1);
  return most < 1 ? 1 : most < (size_t)d->nslab ? (int)most : d->nslab;
}

static size_t stage_bytes(const ell_device *d) { return (size_t)stage_slabs(d) * d->S * d->nnz * 12 + 8; }

static dim3 place_grid(const ell_device *d, int slabs)
{
  const int strips = (d->nnz + kPlaceSlots - 1) / kPlaceSlots;
  return dim3(slabs * (d->S / 64), strips < 1024 ? strips : 1024);
}

static int upload(ell_device *d, const ell_matrix *m)
{
  if (d->nrow == 0 || d->nnz == 0) {
    if (d->nrow) {
      k_ell_scan<<<d->nslab, d->S, 0, d->stream>>>(d->cols, d->vals, d->nrow, d->ncol, 0, d->S, d->dinv, nullptr);
      MM_HIP(hipGetLastError());
      MM_HIP(hipStreamSynchronize(d->stream));
    }
    return 0;
  }
  const int cs = stage_slabs(d);
  const size_t chunk = (size_t)cs * d->S * d->nnz;
  if (!d->stage) MM_HIP(hipMalloc((void **)&d->stage, stage_bytes(d)));
  double *sv = reinterpret_cast<double *>(d->stage);
  int *sc = reinterpret_cast<int *>(sv + chunk), *band = sc + chunk;
  k_zero_int<<<1, 64, 0, d->stream>>>(band, 1);
  for (int s = 0; s < d->nslab; s += cs) {
    const int slabs = d->nslab - s < cs ? d->nslab - s : cs;
    const size_t r0 = (size_t)s * d->S, left = (size_t)d->nrow - r0;
    const size_t rows = left < (size_t)slabs * d->S ? left : (size_t)slabs * d->S;
    const size_t n = rows * d->nnz, at = r0 * d->nnz;
    MM_HIP(hipMemcpyAsync(sc, m->cols + at, n * sizeof(int), hipMemcpyHostToDevice, d->stream));
    MM_HIP(hipMemcpyAsync(sv, m->vals + at, n * sizeof(double), hipMemcpyHostToDevice, d->stream));
    k_ell_place<int, true><<<place_grid(d, slabs), 256, 0, d->stream>>>(sc, (int)rows, d->nnz, d->S, -1, d->cols + at);
    k_ell_place<double, true>
        <<<place_grid(d, slabs), 256, 0, d->stream>>>(sv, (int)rows, d->nnz, d->S, 0.0, d->vals + at);
    MM_HIP(hipGetLastError());
  }
  k_ell_scan<<<d->nslab, d->S, 0, d->stream>>>(d->cols, d->vals, d->nrow, d->ncol, d->nnz, d->S, d->dinv, band);
  MM_HIP(hipGetLastError());
  MM_HIP(hipMemcpyAsync(&d->band, band, sizeof(int), hipMemcpyDeviceToHost, d->stream));
  MM_HIP(hipStreamSynchronize(d->stream));
  return 0;
}

extern "C" int ell_device_create(const ell_matrix *m, int slab_rows, ell_device **out)
{
  if (m == NULL || out == NULL || m->cols == NULL || m->vals == NULL) return 1;
  if (m->nrow < 0 || m->nnz < 0 || m->ncol < 0) return 2;
  int S = slab_rows > 0 ? slab_rows : 256;
  if (S % 64 != 0 || S > 1024) return 1;
  if (check_cols(m)) return 1;
  ell_device *d = (ell_device *)calloc(1, sizeof(ell_device));
  if (!d) return 2;
  pthread_mutex_init(&d->stage_mu, nullptr);
  d->nrow = m->nrow;
  d->ncol = m->ncol;
  d->nnz = m->nnz;
  d->S = S;
  d->nslab = (m->nrow + S - 1) / S;
  if (hipGetDevice(&d->device) != hipSuccess ||
      hipDeviceGetAttribute(&d->ncu, hipDeviceAttributeMultiprocessorCount, d->device) != hipSuccess) {
    free(d);
    return MM_ERR_HIP;
  }
  const size_t slots = (size_t)d->nslab * S * d->nnz;
  const size_t nv = (size_t)(d->nslab ? d->nslab : 1) * S;
  const size_t nvc = (size_t)(m->ncol > (int)nv ? m->ncol : nv);
  int rc = 0;
#define ALLOC(ptr, bytes)                                                   \
  if (hipMalloc((void **)&(ptr), (bytes) ? (bytes) : 8) != hipSuccess) { \
    rc = MM_ERR_HIP;                                                         \
    goto fail;                                                               \
  }
  if (hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking) != hipSuccess) {
    free(d);
    return MM_ERR_HIP;
  }
  ALLOC(d->cols, slots * sizeof(int));
  ALLOC(d->vals, slots * sizeof(double));
  ALLOC(d->dinv, nv * sizeof(double));
  ALLOC(d->x, nvc * sizeof(double));
  ALLOC(d->b, nv * sizeof(double));
  ALLOC(d->r, nv * sizeof(double));
  ALLOC(d->zpA, nvc * sizeof(double2));
  ALLOC(d->zpB, nvc * sizeof(double2));
  ALLOC(d->q, nv * sizeof(double));
  ALLOC(d->part, (size_t)(d->nslab + 1) * 4 * sizeof(double));
  ALLOC(d->st, 2 * sizeof(IterState));
  ALLOC(d->bar, kBarBytes);
#undef ALLOC
  if (hipMemsetAsync(d->st, 0, 2 * sizeof(IterState), d->stream) != hipSuccess) {
    rc = MM_ERR_HIP;
    goto fail;
  }
  rc = upload(d, m);
  if (rc) goto fail;
  *out = d;
  return 0;
fail:
  ell_device_destroy(d);
  return rc;
}

extern "C" int ell_device_update(ell_device *d, const ell_matrix *m)
{
  if (!d || !m || m->nrow != d->nrow || m->nnz != d->nnz || m->ncol != d->ncol) return 1;
  if (check_cols(m)) return 1;
  return upload(d, m);
}

// (Through the mirror's stage: memory allocated and freed by each call would make it
// wait for all streams of the device, 39 ms beside an engine at work in place of 2.)
extern "C" int ell_device_download(const ell_device *d, int *cols, double *vals)
{
  if (!d || !cols || !vals) return 1;
  if (d->nrow == 0 || d->nnz == 0) return 0;
  ell_device *m = const_cast<ell_device *>(d);
  pthread_mutex_lock(&m->stage_mu);
  hipError_t e = hipSuccess;
  if (!m->stage) e = hipMalloc((void **)&m->stage, stage_bytes(d));
  const int cs = stage_slabs(d);
  const size_t chunk = (size_t)cs * d->S * d->nnz;
  double *sv = reinterpret_cast<double *>(m->stage);
  int *sc = reinterpret_cast<int *>(sv + chunk);
  for (int s = 0; s < d->nslab && e == hipSuccess; s += cs) {
    const int slabs = d->nslab - s < cs ? d->nslab - s : cs;
    const size_t r0 = (size_t)s * d->S, left = (size_t)d->nrow - r0;
    const size_t rows = left < (size_t)slabs * d->S ? left : (size_t)slabs * d->S;
    const size_t n = rows * d->nnz, at = r0 * d->nnz;
    k_ell_place<int, false><<<place_grid(d, slabs), 256, 0, d->stream>>>(sc, (int)rows, d->nnz, d->S, -1, d->cols + at);
    k_ell_place<double, false>
        <<<place_grid(d, slabs), 256, 0, d->stream>>>(sv, (int)rows, d->nnz, d->S, 0.0, d->vals + at);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(cols + at, sc, n * sizeof(int), hipMemcpyDeviceToHost, d->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(vals + at, sv, n * sizeof(double), hipMemcpyDeviceToHost, d->stream);
  }
  if (e == hipSuccess) e = hipStreamSynchronize(d->stream);
  pthread_mutex_unlock(&m->stage_mu);
  MM_HIP(e);
  return 0;
}

extern "C" int ell_device_time_mvp(ell_device *d, int reps, double *ms)
{
  if (!d || !ms || reps < 1) return 1;
  *ms = 0.0;
  if (d->nrow == 0) return 0;
  hipEvent_t a = nullptr, b = nullptr;
  MM_HIP(hipEventCreate(&a));
  if (hipEventCreate(&b) != hipSuccess) {
    (void)hipEventDestroy(a);
    return MM_ERR_HIP;
  }
  int rc = 0;
  k_spmv64_exact<<<d->nslab, d->S, 0, d->stream>>>(d->cols, d->vals, d->nrow, d->nnz, d->S, d->x, d->q);
  float t = 0.f;
  if (hipEventRecord(a, d->stream) != hipSuccess) rc = MM_ERR_HIP;
  for (int i = 0; i < reps && !rc; i++)
    k_spmv64_exact<<<d->nslab, d->S, 0, d->stream>>>(d->cols, d->vals, d->nrow, d->nnz, d->S, d->x, d->q);
  if (!rc && (hipGetLastError() != hipSuccess || hipEventRecord(b, d->stream) != hipSuccess ||
              hipEventSynchronize(b) != hipSuccess || hipEventElapsedTime(&t, a, b) != hipSuccess))
    rc = MM_ERR_HIP;
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  if (!rc) *ms = (double)t / reps;
  return rc;
}

extern "C" int ell_device_mvp(ell_device *d, const double *x, double *y)
{
  if (!d || !x || !y) return 1;
  if (d->nrow == 0) return 0;
  MM_HIP(hipMemcpyAsync(d->x, x, d->ncol * sizeof(double), hipMemcpyHostToDevice, d->stream));
  k_spmv64_exact<<<d->nslab, d->S, 0, d->stream>>>(d->cols, d->vals, d->nrow, d->nnz, d->S, d->x, d->q);
  MM_HIP(hipGetLastError());
  MM_HIP(hipMemcpyAsync(y, d->q, d->nrow * sizeof(double), hipMemcpyDeviceToHost, d->stream));
  MM_HIP(hipStreamSynchronize(d->stream));
  return 0;
}

static int set_state(ell_device *d, IterState *st, int max_its, double rtol, double min_err)
{
  IterState h;
  memset(&h, 0, sizeof(h));
  h.max_its = max_its;
  h.rtol = rtol;
  h.min_err = min_err;
  MM_HIP(hipMemcpyAsync(st, &h, sizeof(h), hipMemcpyHostToDevice, d->stream));
  return 0;
}

static int get_state(ell_device *d, const IterState *st, IterState *h)
{
  MM_HIP(hipMemcpyAsync(h, st, sizeof(*h), hipMemcpyDeviceToHost, d->stream));
  MM_HIP(hipStreamSynchronize(d->stream));
  return 0;
}

extern "C" int ell_device_solve_jacobi(ell_device *d, ell_solver *solver, const double *b, double *x)
{
  if (!d || !b || !x) return 1;
  if (d->nrow != d->ncol) return 1;
  if (d->nrow == 0) return 0;
  int rc = set_state(d, d->st, MAX_ITS, 0.0, MIN_ERR);
  if (rc) return rc;
  MM_HIP(hipMemcpyAsync(d->x, x, d->nrow * sizeof(double), hipMemcpyHostToDevice, d->stream));
  MM_HIP(hipMemcpyAsync(d->b, b, d->nrow * sizeof(double), hipMemcpyHostToDevice, d->stream));
  IterState h;
  for (;;) {
    for (int k = 0; k < 64; k++) {
      k_jac_res<<<d->nslab, d->S, 0, d->stream>>>(d->cols, d->vals, d->nrow, d->nnz, d->S, d->x, d->b,
                                                  d->r, d->part, d->st);
      k_reduce<<<1, 256, 0, d->stream>>>(d->part, d->nslab, RED_JAC, d->st);
      k_jac_upd<<<d->nslab, d->S, 0, d->stream>>>(d->nrow, d->S, d->dinv, d->r, d->x, d->st);
    }
    MM_HIP(hipGetLastError());
    rc = get_state(d, d->st, &h);
    if (rc) return rc;
    if (h.done) break;
  }
  MM_HIP(hipMemcpyAsync(x, d->x, d->nrow * sizeof(double), hipMemcpyDeviceToHost, d->stream));
  MM_HIP(hipStreamSynchronize(d->stream));
  if (solver) {
    solver->its = h.its;
    solver->err = h.err;
  }
  return 0;
}

// What resident solves of this process hold together of a device, in halves of a CU.
static ShareGate &res_gate(int device)
{
  static ShareGate g[kResMaxDevices];
  return g[device];
}

// Jacobi-PCG on the device mirror with b and x (initial guess in, solution
// out) in device memory and the work vectors V; the host polls the
// iteration state every 32 iterations.  Returns 0 when converged, 5 when
// max_its was reached.
static int pcg_run(ell_device *d, const PcgVecs &V, ell_solver *solver, const double *b, double *x,
                   bool may_stay = true)
{
  // the matrix on chip (k_pcg_resident) where the columns that a slab spans fit
  // the LDS and the workgroups the GPU; it was the faster at every size it takes
  const int span = d->band > 0 ? d->band : d->nrow, res_rows = span > 64 ? span : 64;  // (its tables want as much)
  const bool pairs = res_lds(res_rows) <= (size_t)kResOneCuLds;  // two workgroups to a CU
  bool resident = may_stay && d->fused_its == 0 && d->S == 256 && d->nnz <= kResSlots && d->device < kResMaxDevices &&
                  res_lds(res_rows) <= (size_t)kResMaxLds && d->nslab <= (pairs ? 2 : 1) * res_cus(d->ncu);
  if (resident && d->res_rest > 0) {
    d->res_rest--;
    resident = false;
  }
  const int max_its = (solver && solver->max_its > 0) ? solver->max_its : MAX_ITS;
  const double rtol = (solver && solver->min_err > 0) ? solver->min_err : MIN_ERR;
  int rc = set_state(d, V.st, max_its, rtol, 0.0);
  if (rc) return rc;
  k_pcg_init<<<d->nslab, d->S, 0, d->stream>>>(d->cols, d->vals, d->nrow, d->nnz, d->S, x, b, d->dinv, V.r,
                                               V.zpA, V.zpB, V.part);
  k_reduce<<<1, 256, 0, d->stream>>>(V.part, d->nslab, RED_INIT, V.st);
  MM_HIP(hipGetLastError());
  IterState h;
  if (resident) {
    {
      FairShare share(res_gate(d->device), pairs ? d->nslab : 2 * d->nslab, 2 * res_cus(d->ncu));
      word_t *zw = reinterpret_cast<word_t *>(V.zpB), *sums = reinterpret_cast<word_t *>(V.q);
      k_res_zero<<<(16 * d->nslab + 255) / 256, 256, 0, d->stream>>>(sums, 16 * d->nslab);
      const auto solve = span > kResListSpan ? k_pcg_resident<true> : k_pcg_resident<false>;
      solve<<<d->nslab, 256, res_lds(res_rows), d->stream>>>(d->cols, d->vals, d->nrow, d->nnz, d->nslab, res_rows,
                                                             d->dinv, x, V.r, V.zpA, zw, sums, V.st, d->res_away);
      k_res_take<<<(d->nrow + 255) / 256, 256, 0, d->stream>>>(V.st, V.zpA, x, d->nrow);
      MM_HIP(hipGetLastError());
      rc = get_state(d, V.st, &h);
      if (rc) return rc;
    }
    if (h.pad0) {  // no meeting, or a wait that ran out: x is as it was
      d->res_left++;
      d->res_rest = d->res_rested = d->res_rested < kResRest ? 2 * d->res_rested + 1 : kResRest;
      return pcg_run(d, V, solver, b, x, false);
    }
    d->res_stayed++;
    d->res_rested = 0;
  } else {
    rc = get_state(d, V.st, &h);
    if (rc) return rc;
  }
  if (h.bnorm == 0.0) {  // zero right-hand side: the solution is zero
    k_zero<<<(d->nrow + 255) / 256, 256, 0, d->stream>>>(x, d->nrow);
    MM_HIP(hipGetLastError());
  }
  while (!h.done && d->fused_its > 0) {
    k_bar_reset<<<1, 128, 0, d->stream>>>(V.bar);
    MM_HIP(hipGetLastError());
    const int *cols = d->cols;
    const double *vals = d->vals, *dinv = d->dinv;
    int nrow = d->nrow, nnz = d->nnz, nslab = d->nslab, its = d->fused_its;
    double *xv = x, *r = V.r, *q = V.q, *part = V.part;
    double2 *zpA = V.zpA, *zpB = V.zpB;
    IterState *st = V.st;
    unsigned *bar = V.bar;
    void *args[] = {&cols, &vals, &nrow, &nnz, &nslab, &dinv, &xv, &r, &zpA, &zpB, &q, &part, &st, &bar, &its};
    MM_HIP(hipLaunchCooperativeKernel((const void *)k_pcg_fused, dim3(d->fused_grid), dim3(kFusedLanes), args, 0,
                                      d->stream));
    rc = get_state(d, V.st, &h);
    if (rc) return rc;
    if (h.pad0) {
      fprintf(stderr,
              "madmax_amd: k_pcg_fused: a grid barrier wait gave up at %d of %d group arrivals (%d workgroups)\n",
              h.pad1, h.pad2, d->fused_grid);
      return MM_ERR_HIP;
    }
  }
  // the state passes st[0] -> st[1] -> st[0]; up to kSelfSumSlabs slabs two
  // launches per iteration, beyond that a one-workgroup k_reduce before each
  const int self_sum = d->nslab <= kSelfSumSlabs ? 1 : 0;
  const auto spmv = d->nslab <= kAheadSlabs && d->S <= 256 ? k_pcg_spmv<kAhead, true> : k_pcg_spmv<kU, false>;
  while (!h.done) {
    for (int k = 0; k < 32; k++) {
      spmv<<<d->nslab, d->S, 0, d->stream>>>(d->cols, d->vals, d->nrow, d->nnz, d->S, d->nslab, V.zpA, V.zpB, V.q,
                                             V.part, V.st, V.st + 1, self_sum);
      if (!self_sum) k_reduce<<<1, 256, 0, d->stream>>>(V.part, d->nslab, RED_PQ, V.st + 1);
      k_pcg_update<<<d->nslab, d->S, 0, d->stream>>>(d->nrow, d->S, d->nslab, d->dinv, V.zpA, V.zpB, V.q, x,
                                                     V.r, V.part, V.st + 1, V.st, self_sum);
      if (!self_sum) k_reduce<<<1, 256, 0, d->stream>>>(V.part, d->nslab, RED_RR, V.st);
    }
    MM_HIP(hipGetLastError());
    rc = get_state(d, V.st, &h);
    if (rc) return rc;
  }
  MM_HIP(hipStreamSynchronize(d->stream));
  const double relres = (h.bnorm == 0.0) ? 0.0 : h.rnorm / h.bnorm;
  if (solver) {
    solver->its = h.its;
    solver->err = relres;
  }
  return (h.bnorm == 0.0 || h.rnorm <= rtol * h.bnorm) ? 0 : MM_NOT_CONVERGED;
}

extern "C" int ell_device_set_pcg_fused(ell_device *d, int its_per_launch)
{
  if (!d || its_per_launch < 0) return 1;
  if (its_per_launch == 0) {
    d->fused_its = 0;
    return 0;
  }
  if (d->S != kFusedLanes || d->nslab == 0) return 1;
  int coop = 0, ncu = 0, per_cu = 0;
  MM_HIP(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, d->device));
  if (!coop) return 1;
  MM_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, d->device));
  MM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k_pcg_fused, kFusedLanes, 0));
  if (ncu < 1 || per_cu < 1) return 1;
  // Half of what fits: a grid at the full occupancy limit needs every wave
  // slot of every CU free at once, and the launch admits it even when some
  // are not (its barrier waits then run out).  Workgroups loop over slabs,
  // so a smaller grid only lengthens each one's share.
  long long cap = (long long)ncu * (per_cu > 1 ? per_cu / 2 : 1);
  if (cap > kBarMaxGrid) cap = kBarMaxGrid;
  d->fused_grid = (int)(d->nslab < cap ? d->nslab : cap);
  d->fused_its = its_per_launch;
  return 0;
}

extern "C" int ell_device_solve_pcg(ell_device *d, ell_solver *solver, const double *b, double *x)
{
  if (!d || !b || !x) return 1;
  if (d->nrow != d->ncol) return 1;
  if (d->nrow == 0) return 0;
  MM_HIP(hipMemcpyAsync(d->x, x, d->nrow * sizeof(double), hipMemcpyHostToDevice, d->stream));
  MM_HIP(hipMemcpyAsync(d->b, b, d->nrow * sizeof(double), hipMemcpyHostToDevice, d->stream));
  const PcgVecs V{d->r, d->zpA, d->zpB, d->q, d->part, d->st, d->bar};
  const int rc = pcg_run(d, V, solver, d->b, d->x);
  if (rc != 0 && rc != MM_NOT_CONVERGED) return rc;
  MM_HIP(hipMemcpyAsync(x, d->x, d->nrow * sizeof(double), hipMemcpyDeviceToHost, d->stream));
  MM_HIP(hipStreamSynchronize(d->stream));
  return rc;
}

// ---- internal: a device ELL filled by kernels (fe.hip) --------------------

int mm::ell_device_alloc(int nrow, int nnz, int S, ell_device **out)
{
  if (!out || nrow < 0 || nnz < 1 || S % 64 != 0 || S < 64 || S > 1024) return MM_ERR_ARG;
  ell_device *d = (ell_device *)calloc(1, sizeof(ell_device));
  if (!d) return MM_ERR_ALLOC;
  pthread_mutex_init(&d->stage_mu, nullptr);
  d->nrow = d->ncol = nrow;
  d->nnz = nnz;
  d->S = S;
  d->nslab = (nrow + S - 1) / S;
  if (hipGetDevice(&d->device) != hipSuccess ||
      hipDeviceGetAttribute(&d->ncu, hipDeviceAttributeMultiprocessorCount, d->device) != hipSuccess) {
    free(d);
    return MM_ERR_HIP;
  }
  const size_t slots = (size_t)d->nslab * S * nnz;
  const size_t nv = (size_t)(d->nslab ? d->nslab : 1) * S;
  int rc = 0;
#define ALLOC(ptr, bytes)                                                   \
  if (hipMalloc((void **)&(ptr), (bytes) ? (bytes) : 8) != hipSuccess) { \
    rc = MM_ERR_HIP;                                                         \
    goto fail;                                                               \
  }
  if (hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking) != hipSuccess) {
    free(d);
    return MM_ERR_HIP;
  }
  ALLOC(d->cols, slots * sizeof(int));
  ALLOC(d->vals, slots * sizeof(double));
  ALLOC(d->dinv, nv * sizeof(double));
  ALLOC(d->x, nv * sizeof(double));
  ALLOC(d->b, nv * sizeof(double));
  ALLOC(d->r, nv * sizeof(double));
  ALLOC(d->zpA, nv * sizeof(double2));
  ALLOC(d->zpB, nv * sizeof(double2));
  ALLOC(d->q, nv * sizeof(double));
  ALLOC(d->part, (size_t)(d->nslab + 1) * 4 * sizeof(double));
  ALLOC(d->st, 2 * sizeof(IterState));
  ALLOC(d->bar, kBarBytes);
#undef ALLOC
  if (hipMemsetAsync(d->cols, 0xff, slots * sizeof(int), d->stream) != hipSuccess ||
      hipMemsetAsync(d->vals, 0, slots * sizeof(double), d->stream) != hipSuccess ||
      hipMemsetAsync(d->st, 0, 2 * sizeof(IterState), d->stream) != hipSuccess ||
      hipStreamSynchronize(d->stream) != hipSuccess) {
    rc = MM_ERR_HIP;
    goto fail;
  }
  *out = d;
  return 0;
fail:
  ell_device_destroy(d);
  return rc;
}

void mm::ell_device_arrays(ell_device *d, int **cols, double **vals, double **dinv, int *S, hipStream_t *s)
{
  *cols = d->cols;
  *vals = d->vals;
  *dinv = d->dinv;
  *S = d->S;
  *s = d->stream;
}

void mm::ell_device_set_band(ell_device *d, long long band) { d->band = band < d->nrow ? (int)band : 0; }

int mm::ell_device_pcg_device(ell_device *d, ell_solver *solver, const double *b, double *x)
{
  if (!d || !b || !x) return MM_ERR_ARG;
  if (d->nrow == 0) return 0;
  const PcgVecs V{d->r, d->zpA, d->zpB, d->q, d->part, d->st, d->bar};
  return pcg_run(d, V, solver, b, x);
}

extern "C" int ell_device_pcg_counts(const ell_device *d, int *counts)
{
  if (!d || !counts) return MM_ERR_ARG;
  counts[0] = d->res_stayed;
  counts[1] = d->res_left;
  counts[2] = d->res_rest;
  return 0;
}

extern "C" int ell_device_set_stay_away(ell_device *d, int on)
{
  if (!d) return MM_ERR_ARG;
  d->res_away = on ? 1 : 0;
  return 0;
}

// ---- the same solve without any allocation ----------------------------------
// The PCG work vectors, partial sums and iteration state of
// ell_device_solve_pcg_noalloc live in this file-scope array: six vectors of
// ELL_NOALLOC_MAX_ROWS doubles, the partials of up to ELL_NOALLOC_MAX_ROWS / 64
// slabs, two IterState copies and the fused kernel's barrier words (about
// 48.5 MiB, held on every GPU the library runs on until the process ends).
// Host code never uses the array's name as an address: the per-device
// address comes from hipGetSymbolAddress.
namespace {
constexpr size_t kNaRows = ELL_NOALLOC_MAX_ROWS;
constexpr size_t kNaPart = (kNaRows / 64 + 1) * 4;
constexpr size_t kNaState = (2 * sizeof(IterState) + 7) / 8;
constexpr size_t kNaBar = kBarBytes / 8;  // the grid-barrier words of k_pcg_fused
constexpr size_t kNaDoubles = 6 * kNaRows + kNaPart + kNaState + kNaBar;
constexpr int kNaMaxDevices = 64;
}  // namespace

static __device__ __align__(256) double scratch[kNaDoubles];

static std::mutex g_na_mu;
static double *g_na_ptr[kNaMaxDevices];

// Address of `scratch` on `device`, looked up once per device with that
// device current.
static int noalloc_scratch(int device, double **out)
{
  if (device < 0 || device >= kNaMaxDevices) return MM_ERR_ARG;
  std::lock_guard<std::mutex> lk(g_na_mu);
  if (!g_na_ptr[device]) {
    int cur = -1;
    MM_HIP(hipGetDevice(&cur));
    if (cur != device) MM_HIP(hipSetDevice(device));
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != device) MM_HIP(hipSetDevice(cur));
    if (e != hipSuccess || !p) {
      fprintf(stderr, "madmax_amd: hipGetSymbolAddress(scratch) failed: %s\n", hipGetErrorName(e));
      return MM_ERR_HIP;
    }
    g_na_ptr[device] = (double *)p;
  }
  *out = g_na_ptr[device];
  return 0;
}

extern "C" int ell_device_solve_pcg_noalloc(ell_device *d, ell_solver *solver, const double *b, double *x)
{
  if (!d || !b || !x) return 1;
  if (d->nrow != d->ncol) return 1;
  if ((size_t)d->nrow > kNaRows) {
    fprintf(stderr, "madmax_amd: ell_device_solve_pcg_noalloc: %d rows exceed the %zu-row scratch\n", d->nrow,
            kNaRows);
    return 1;
  }
  if (d->nrow == 0) return 0;
  double *sp = nullptr;
  const int rc = noalloc_scratch(d->device, &sp);
  if (rc) return rc;
  // r, then the two pair buffers (2 rows' worth each, 16-byte aligned), q, the
  // partials, the two states and the barrier words
  const PcgVecs V{sp, reinterpret_cast<double2 *>(sp + kNaRows), reinterpret_cast<double2 *>(sp + 3 * kNaRows),
                  sp + 5 * kNaRows, sp + 6 * kNaRows, reinterpret_cast<IterState *>(sp + 6 * kNaRows + kNaPart),
                  reinterpret_cast<unsigned *>(sp + 6 * kNaRows + kNaPart + kNaState)};
  return pcg_run(d, V, solver, b, x);
}

extern "C" int ell_device_destroy(ell_device *d)
{
  if (!d) return 1;
  if (d->stream) (void)hipStreamSynchronize(d->stream);
  (void)hipFree(d->cols);
  (void)hipFree(d->vals);
  (void)hipFree(d->dinv);
  (void)hipFree(d->x);
  (void)hipFree(d->b);
  (void)hipFree(d->r);
  (void)hipFree(d->zpA);
  (void)hipFree(d->zpB);
  (void)hipFree(d->q);
  (void)hipFree(d->part);
  (void)hipFree(d->st);
  (void)hipFree(d->bar);
  (void)hipFree(d->stage);
  if (d->stream) (void)hipStreamDestroy(d->stream);
  free(d);
  return 0;
}

// ---- reference entry points running on the GPU ------------------------------

// src/ell.c:127-141
extern "C" int ell_mvp(ell_matrix *m, double *x, double *y)
{
  if (m == NULL || x == NULL || y == NULL) return 1;
  ell_device *d = NULL;
  int rc = ell_device_create(m, 0, &d);
  if (rc) return rc;
  rc = ell_device_mvp(d, x, y);
  ell_device_destroy(d);
  return rc;
}

// src/ell.c:143-184
extern "C" int ell_solve_jacobi(ell_solver *solver, ell_matrix *m, double *b, double *x)
{
  if (m == NULL || b == NULL || x == NULL) return 1;
  ell_device *d = NULL;
  int rc = ell_device_create(m, 0, &d);
  if (rc) return rc;
  rc = ell_device_solve_jacobi(d, solver, b, x);
  ell_device_destroy(d);
  return rc;
}

extern "C" int ell_solve_pcg(ell_solver *solver, ell_matrix *m, double *b, double *x)
{
  if (m == NULL || b == NULL || x == NULL) return 1;
  ell_device *d = NULL;
  int rc = ell_device_create(m, 0, &d);
  if (rc) return rc;
  rc = ell_device_solve_pcg(d, solver, b, x);
  ell_device_destroy(d);
  return rc;
}
