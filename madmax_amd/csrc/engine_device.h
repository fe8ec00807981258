// engine_device.h -- device code shared by the solver kernels of the RVE engine
// (engine_kernels.hip, engine_sweep.hip): the per-slab partial sums and the
// scalar steps of the phase machine.
#pragma once

#include <hip/hip_runtime.h>

#include "mm_device.h"
#include "mm_internal.h"

namespace mm {

// Per-slab partial sums of the launch that produced them, summed over the
// RVE's slabs in slab order (group_sum_cols): every workgroup of the consuming
// launch forms the same totals.  A slab has kPart partial values, value i
// at part[i * part_stride + slab] (value-major, so that a sum over an RVE's
// slabs reads contiguous memory).  Values:
//   [0, K)      p.q            (A -> B)
//   [K, 3K)     r.r, r.z       (B -> A)
//   [3K, 7K)    residual norms (R -> A)
//   [0, 12K)    averages       (R -> A), never pending with the others
struct SlabPart {
  double *p;
  long long s;
  __device__ __forceinline__ double &operator[](int i) const { return p[(size_t)i * s]; }
};
__device__ __forceinline__ SlabPart slab_part(const EngPtrs &P, int slab)
{
  return SlabPart{P.part + slab, P.part_stride};
}

// The words of load case k of a resident sweep (sweep_region), ni interior nodes.
struct SweepWords {
  word_t *w[3], *sum;
};
template <typename TS>
__device__ __forceinline__ SweepWords sweep_words(const EngPtrs &P, int nslab, int K, int first_slab, int k,
                                                  long long ni)
{
  const long long b0 = sweep_region(nslab, P.SN, K, (int)sizeof(TS), first_slab, k);
  SweepWords X;
  X.w[0] = reinterpret_cast<word_t *>((char *)P.q + b0);
  X.w[1] = reinterpret_cast<word_t *>((char *)P.p + b0);
  X.w[2] = reinterpret_cast<word_t *>((char *)P.d + b0);
  X.sum = X.w[2] + ni * (long long)(sizeof(TS) / 4);
  return X;
}

// MI355X dispatches workgroup i to XCD i % 8.  The solver grids are a
// multiple of 8 and workgroup i processes slab (i % 8) * (grid / 8) + i / 8,
// so each XCD walks one contiguous run of slabs and the z rows that
// neighbouring slabs of an RVE share stay in that XCD's L2.
constexpr int kXcd = 8;
// Largest grid of kernel R (a multiple of 8; k_step_r loops over the slabs).
constexpr int kRGrid = 2048;
__device__ __forceinline__ int xcd_slab()
{
  const int per = gridDim.x / kXcd;
  return (blockIdx.x % kXcd) * per + blockIdx.x / kXcd;
}

// Solver launches run over the list of slabs being solved (act_list[0] of
// them, ascending from act_list[1]); the grid is a power of two >= 64 that
// covers the list.  The list is split in 8 contiguous parts, one per XCD, so
// neighbouring slabs of an RVE share an L2.  Returns false for workgroups
// beyond the list.
__device__ __forceinline__ bool active_in(const int *list, int &slab)
{
  const int n = list[0];
  const int per = (n + kXcd - 1) / kXcd;
  const int j = blockIdx.x / kXcd;
  const int i = (blockIdx.x % kXcd) * per + j;
  if (j >= per || i >= n) return false;
  slab = list[1 + i];
  return true;
}
__device__ __forceinline__ bool active_slab(const EngPtrs &P, int &slab) { return active_in(P.act_list, slab); }

// Zeroes the slab's share of the words that the ranks of a resident sweep
// exchange (tag 0 is no iteration's).
template <typename TS, int K>
__device__ void sweep_words_zero(const EngPtrs &P, const RveDev *R, int slab)
{
  const int ls = slab - R->first_slab, bd = (int)blockDim.x, cw = R->scw, cz = cw / R->sty;
  const int nixy = (R->nx - 2) * (R->ny - 2), niz = R->nz - 2, ni = nixy * niz;
  // the planes that ranks exchange: the first and last of each share, or, where
  // the rows are shared too, all
  const int nw = R->sty > 1 ? ni : 2 * cz * nixy;
#pragma unroll 1
  for (int k = 0; k < K; k++) {
    const SweepWords X = sweep_words<TS>(P, R->nslab, K, R->first_slab, k, ni);
    for (int i = ls * bd + (int)threadIdx.x; i < nw; i += R->nslab * bd) {
      int at = i;
      if (R->sty == 1) {
        const int pl = i / nixy, r = pl >> 1;
        at = ((pl & 1) ? (r + 1) * niz / cz - 1 : r * niz / cz) * nixy + i - pl * nixy;
      }
#pragma unroll
      for (int d = 0; d < 3; d++)
#pragma unroll
        for (int h = 0; h < (int)(sizeof(TS) / 4); h++) X.w[d][(long long)h * ni + at] = 0;
    }
    if (ls == 0)
      for (int i = threadIdx.x; i < 16 * cw; i += bd) X.sum[i] = 0;  // (the meeting's words: sweep_end)
  }
}

// The words of the meetings: load case k's are two, k times `step` on from the first.
struct MeetWords {
  word_t *w;
  long long step;
};
template <typename TS, int K>
__device__ __forceinline__ MeetWords sweep_meeting(const EngPtrs &P, const RveDev *R)
{
  const long long ni = (long long)(R->nx - 2) * (R->ny - 2) * (R->nz - 2);
  return {sweep_words<TS>(P, R->nslab, K, R->first_slab, 0, ni).sum + 16 * R->scw,
          (long long)R->nslab * 3 * P.SN * (int)sizeof(TS) / 8};
}
// Which load cases' workgroups met in the launch (bit k); and parts them again.
template <typename TS, int K>
__device__ __forceinline__ unsigned sweep_met(const EngPtrs &P, const RveDev *R)
{
  const MeetWords m = sweep_meeting<TS, K>(P, R);
  word_t w[K];
  unsigned met = 0;
#pragma unroll
  for (int k = 0; k < K; k++) w[k] = m.w[k * m.step + 1];
#pragma unroll
  for (int k = 0; k < K; k++) met |= (w[k] == kMeetGo ? 1u : 0u) << k;
  return met;
}
template <typename TS, int K>
__device__ __forceinline__ void sweep_part(const EngPtrs &P, const RveDev *R)
{
  const MeetWords m = sweep_meeting<TS, K>(P, R);
  for (int k = 0; k < K; k++) m.w[k * m.step] = m.w[k * m.step + 1] = 0;
}

// Whether a resident RVE's state st[0] is ready for the residual: it wants its
// first one, or the sweep has run for every load case that needed it.
template <typename TS, int K>
__device__ __forceinline__ bool sweep_ran(const EngPtrs &P, const RveDev *R)
{
  const SolveState *S = &R->st[0];
  if (S->phase != PH_INNER) return S->phase == PH_RES;
  return !R->smeet || (~(S->done_in | sweep_met<TS, K>(P, R)) & ((1u << K) - 1u)) == 0;
}

// A resident RVE's state between launches, by one lane, after the residual (if
// any).  The end of a sweep: its iteration count is the largest of the load cases'
// (as inner_check counts).  Load cases whose cluster did not meet are left for the
// next launch; the host counts those without a meeting and puts the RVE on kernels
// A and B after a few.
template <typename TS, int K>
__device__ void sweep_end(const EngPtrs &P, int slot, RveDev *R, SolveState &N)
{
  const int phase = N.phase, meets = R->smeet;
  bool left = false;
  if (phase == PH_INNER) {
    unsigned ran = ~0u;
    if (meets) ran = sweep_met<TS, K>(P, R);
    for (int k = 0; k < K; k++) {
      if ((N.done_in >> k) & 1u) continue;
      if ((ran >> k) & 1u) N.its = max(N.its, R->lits[k]);
      else left = true;
    }
    if (meets) {
      const unsigned run = ~N.done_in & ((1u << K) - 1u);
      P.out[slot].met = R->met += __popc(run & ran);
      P.out[slot].missed = R->missed += __popc(run & ~ran);
      N.done_in |= ran;
    }
  }
  if (meets && (phase == PH_INNER || phase == PH_RES)) sweep_part<TS, K>(P, R);
  if (phase == PH_INNER && !left) {
    N.its_total += N.its;
    N.sweep += 1;
    N.phase = PH_RESRED;
  } else if (phase == PH_RES) {
    N.phase = PH_RESRED;
  } else if (phase == PH_AVG) {
    N.phase = PH_AVGRED;
  }
}

// Start of a refinement sweep from the reduced residual norms s4 =
// {||r64||^2, ||r||^2, r.z, ||r_cold||^2} per load case (FP64 residual r64,
// its rounding r, cold-start right-hand side r_cold).
template <int K>
__device__ void start_sweep(SolveState &N, const double (&s4)[4 * K], const RveDev *R,
                            const SolveParams &sp)
{
  const bool need_cold = (R->warm || R->affine) && N.sweep == 0;
  unsigned done_out = 0;
  for (int k = 0; k < K; k++) {
    const double rn = sqrt(s4[k]);
    N.rnorm[k] = rn;
    if (N.sweep == 0) N.r0[k] = need_cold ? sqrt(s4[3 * K + k]) : rn;
    const bool conv = (k >= R->nload) || N.r0[k] == 0.0 || rn <= sp.rtol * N.r0[k] ||
                      rn < sp.abs_tol || N.sweep >= sp.max_sweeps + R->again;
    if (conv) done_out |= 1u << k;
    // absolute target of this sweep: inner_rtol of the sweep's right-hand
    // side, but no tighter than what the outer tolerance still needs
    const double cap = (N.r0[k] > 0.0 && rn > 0.0) ? 0.5 * sp.rtol * N.r0[k] / rn : 0.0;
    N.bnorm_in[k] = fmax(sp.inner_rtol, cap) * sqrt(s4[K + k]);
    N.beta[k] = 0.0;
    N.rz[k] = s4[2 * K + k];
  }
  const unsigned all = (1u << K) - 1u;
  N.done_out = done_out;
  if ((done_out & all) == all) {
    N.phase = PH_AVG;
  } else {
    N.done_in = done_out;
    N.its = 0;
    N.phase = PH_INNER;
  }
}

// End of a PCG iteration from the reduced s2 = {r.r, r.z}: each load case
// stops at its own sweep target; the sweep ends (x += d, then a new FP64
// residual) when all have, or at max_inner_its.  Returns true at sweep end.
template <int K>
__device__ bool inner_check(SolveState &N, const double (&s2)[2 * K], const SolveParams &sp)
{
  N.its += 1;
  unsigned done = N.done_in;
  const unsigned all = (1u << K) - 1u;
  for (int k = 0; k < K; k++) {
    const double rr = s2[k], rz = s2[K + k];
    if ((done >> k) & 1u) {
      N.beta[k] = 0.0;
      continue;
    }
    if (sqrt(rr) <= N.bnorm_in[k] || N.rz[k] == 0.0) {
      done |= 1u << k;
      N.beta[k] = 0.0;
    } else {
      N.beta[k] = rz / N.rz[k];
      N.rz[k] = rz;
    }
  }
  N.done_in = done;
  if ((done & all) == all || N.its >= sp.max_inner_its) {
    N.its_total += N.its;
    N.sweep += 1;
    N.phase = PH_RES;
    return true;
  }
  return false;
}

// Volume averages and tangent of a finished RVE (micro/src/homogenize.c:
// 344-368, :80) from the averaging partials; run by one workgroup.  Bound by its
// chain of memory round trips: each wave sums every so many of the 12 K values, a
// lane per slab, and a lane forms each output.  Four values at a time over the
// workgroup and one lane for the outputs took 38 us for one 10^3
// cell and 110 for 24 cells up to 30^3; this takes 10 and 20.
template <int K>
__device__ void finish_rve(const EngPtrs &P, int slot, const RveDev *R, SolveState &N, const SolveParams &sp)
{
  __shared__ double avg[MM_MAX_RHS][12];
  const double *p0 = slab_part(P, R->first_slab).p;
  const int tid = threadIdx.x, ln = tid & 63, nslab = R->nslab;
  const double vol = R->vol;
#pragma unroll 1
  for (int i0 = 4 * (tid >> 6); i0 < 12 * K; i0 += 4 * ((int)blockDim.x >> 6)) {
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int b = ln; b < nslab; b += 64)
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] += p0[(size_t)(i0 + i) * P.part_stride + b];
    int q;
    const double s = wave_sum4(v, q);
    if ((ln & 15) == 0) avg[(i0 + q) / 12][(i0 + q) % 12] = s / vol;
  }
  __syncthreads();
  RveOut *o = P.out + slot;
  const int mode = R->tangent_mode;
  for (int t = tid; t < 12 * K; t += blockDim.x) {
    const int k = t / 12, i = t - 12 * k;
    if (i < 6) o->strain[k][i] = avg[k][i];
    else o->stress[k][i - 6] = avg[k][i];
  }
  for (int t = tid; t < 36; t += blockDim.x) {
    const int j = t / 6, i = t - 6 * j;  // c[j * 6 + i]: d stress j / d strain i
    double c = 0.0;
    if (mode == MM_TANGENT_UNIT && K >= 6) {
      c = avg[i][6 + j] / R->load[i][i];
    } else if (mode == MM_TANGENT_FD && K >= 7) {
      c = (avg[i + 1][6 + j] - avg[0][6 + j]) / (R->load[i + 1][i] - R->load[0][i]);
    }
    o->c[t] = c;
  }
  __threadfence_system();  // each lane's outputs, before lane 0 says that they are there
  __syncthreads();
  if (tid != 0) return;
  double rel = 0.0;
  bool ok = true;
  for (int k = 0; k < K && k < R->nload; k++) {
    const double r0 = N.r0[k], rn = N.rnorm[k];
    rel = fmax(rel, (r0 > 0.0) ? rn / r0 : 0.0);
    if (!(r0 == 0.0 || rn <= sp.rtol * r0 || rn < sp.abs_tol)) ok = false;
  }
  o->residual_rel = rel;
  o->its_total = N.its_total;
  o->sweeps = N.sweep - R->idle;
  o->status = ok ? MM_OK : MM_NOT_CONVERGED;
  N.status = o->status;
  N.phase = PH_DONE;
  __threadfence_system();
  o->phase = PH_DONE;
  __threadfence_system();
}

}  // namespace mm
