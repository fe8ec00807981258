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
                      rn < sp.abs_tol || N.sweep >= sp.max_sweeps;
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
// 344-368, :80) from the averaging partials; run by one workgroup.
template <int K, int L>
__device__ void finish_rve(const EngPtrs &P, int slot, const RveDev *R, SolveState &N,
                           const SolveParams &sp, double (&lds)[L])
{
  __shared__ double tot[MM_MAX_RHS][12];
  const double *p0 = slab_part(P, R->first_slab).p;
#pragma unroll 1
  for (int k = 0; k < K; k++) group_sum_cols_lds<12>(p0, R->nslab, P.part_stride, k * 12, &tot[k][0], lds);
  __shared__ double sig[MM_MAX_RHS][6];
  if (threadIdx.x != 0) return;
  RveOut *o = P.out + slot;
  double rel = 0.0;
  bool ok = true;
#pragma unroll 1
  for (int k = 0; k < K; k++) {
#pragma unroll 1
    for (int i = 0; i < 12; i++) {
      const double s = tot[k][i] / R->vol;
      if (i < 6) o->strain[k][i] = s;
      else {
        o->stress[k][i - 6] = s;
        sig[k][i - 6] = s;
      }
    }
    if (k < R->nload) {
      const double r0 = N.r0[k], rn = N.rnorm[k];
      rel = fmax(rel, (r0 > 0.0) ? rn / r0 : 0.0);
      if (!(r0 == 0.0 || rn <= sp.rtol * r0 || rn < sp.abs_tol)) ok = false;
    }
  }
  for (int i = 0; i < 36; i++) o->c[i] = 0.0;
  if (R->tangent_mode == MM_TANGENT_UNIT && K >= 6) {
    for (int i = 0; i < 6; i++)
      for (int j = 0; j < 6; j++) o->c[j * 6 + i] = sig[i][j] / R->load[i][i];
  } else if (R->tangent_mode == MM_TANGENT_FD && K >= 7) {
    for (int i = 0; i < 6; i++)
      for (int j = 0; j < 6; j++)
        o->c[j * 6 + i] = (sig[i + 1][j] - sig[0][j]) / (R->load[i + 1][i] - R->load[0][i]);
  }
  o->residual_rel = rel;
  o->its_total = N.its_total;
  o->sweeps = N.sweep;
  o->status = ok ? MM_OK : MM_NOT_CONVERGED;
  N.status = o->status;
  N.phase = PH_DONE;
  __threadfence_system();
  o->phase = PH_DONE;
  __threadfence_system();
}

}  // namespace mm
