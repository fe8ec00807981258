// mm_device.h -- device helpers shared by the HIP kernels: deterministic
// block and group reductions (fixed summation order, no atomics on values).
#pragma once

#include <hip/hip_runtime.h>

namespace mm {

// Two 32-bit halves of a double moved together.
typedef unsigned halves_t __attribute__((ext_vector_type(2)));
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v)
{
  const halves_t b = __builtin_bit_cast(halves_t, v);
  halves_t m;
  m.x = __builtin_amdgcn_update_dpp(0, b.x, CTRL, 0xf, 0xf, true);
  m.y = __builtin_amdgcn_update_dpp(0, b.y, CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, m);
}
// a with its upper half of lanes replaced by b's lower half, plus b with its
// lower half replaced by a's upper half (OFF 32; of each 32 lanes for OFF 16):
// lane l < OFF has a[l] + a[l + OFF], lane l + OFF the same of b.
template <int OFF>
__device__ __forceinline__ double halve(double a, double b)
{
  const halves_t x = __builtin_bit_cast(halves_t, a), y = __builtin_bit_cast(halves_t, b);
  halves_t lo, hi, p, q;
  if constexpr (OFF == 32) {
    lo = __builtin_amdgcn_permlane32_swap(x.x, y.x, false, false);
    hi = __builtin_amdgcn_permlane32_swap(x.y, y.y, false, false);
  } else {
    lo = __builtin_amdgcn_permlane16_swap(x.x, y.x, false, false);
    hi = __builtin_amdgcn_permlane16_swap(x.y, y.y, false, false);
  }
  p.x = lo.x;
  p.y = hi.x;
  q.x = lo.y;
  q.y = hi.y;
  return __builtin_bit_cast(double, p) + __builtin_bit_cast(double, q);
}

// Sums four values over a wave (lanes 32, 16, 8, 4, 2 and 1 apart); lanes 0, 32, 16
// and 48 return the sum of value q = 0, 1, 2 and 3.
__device__ __forceinline__ double wave_sum4(const double (&v)[4], int &q)
{
  const int lane = threadIdx.x & 63;
  double t = halve<16>(halve<32>(v[0], v[1]), halve<32>(v[2], v[3]));
  t += dpp_move<0x108>(t);  // row_shl:8, 4, 2, 1: lane l takes lane l + 8 ... of its 16
  t += dpp_move<0x104>(t);
  t += dpp_move<0x102>(t);
  t += dpp_move<0x101>(t);
  q = (lane >> 5) + 2 * ((lane >> 4) & 1);
  return t;
}

// Sums NV values over the block in a fixed order; returns the sum of value i in
// thread i < NV.  lds holds 16 doubles per value (blockDim.x <= 1024); its size
// is checked at compile time.  Each wave adds lanes 32, 16, 8, 4, 2 and 1 apart,
// then lane i of wave 0 the waves' value i in order.  The first two steps put two and four values
// beside each other in one register, so NV values take about 1.5 NV + 4 adds, and
// the moves between lanes are DPP and permlane swaps in the vector unit: through
// the LDS (ds_bpermute) a step's round trip is some 100 cycles.  An iteration of
// k_pcg_resident, with four such sums in a row, took 8.6 us for 2,970 rows with
// shuffles and a serial sum of the waves, and takes 7.0.
template <int NV, int L>
__device__ inline double block_sum_lane(const double (&v)[NV], double (&lds)[L])
{
  static_assert(L >= NV * 16 && NV <= 64, "block_sum: LDS scratch too small");
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
#pragma unroll
  for (int i = 0; i < NV; i += 4) {
    const double v4[4] = {v[i], v[i + 1 < NV ? i + 1 : i], v[i + 2 < NV ? i + 2 : i], v[i + 3 < NV ? i + 3 : i]};
    int q;
    const double t = wave_sum4(v4, q);
    if ((lane & 15) == 0 && i + q < NV) lds[(i + q) * 16 + wid] = t;
    __builtin_amdgcn_sched_barrier(0);  // (NV sums at a time would take many registers)
  }
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x < 64) {
    const double *p = lds + min(lane, NV - 1) * 16;
    for (int w = 0; w < nw; w += 4) {  // (all 16 places of a value exist)
      const double t[4] = {p[w], p[w + 1], p[w + 2], p[w + 3]};
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (w + k < nw) s += t[k];
    }
  }
  __syncthreads();
  return s;
}
// The same with all sums in v, valid in the first wave.
template <int NV, int L>
__device__ inline void block_sum(double (&v)[NV], double (&lds)[L])
{
  const halves_t b = __builtin_bit_cast(halves_t, block_sum_lane<NV>(v, lds));
#pragma unroll
  for (int i = 0; i < NV; i++) {
    halves_t r;
    r.x = __builtin_amdgcn_readlane(b.x, i);
    r.y = __builtin_amdgcn_readlane(b.y, i);
    v[i] = __builtin_bit_cast(double, r);
  }
}

// Run by every thread of a workgroup: sums partial values off .. off+NV-1
// over nslab slabs written by an earlier launch (visible at kernel start, so
// plain cached loads).  Value i of slab b is p0[(off + i) * vstride + b]:
// each value's partials are contiguous, so a workgroup reads nslab * 8 bytes
// per value, not one cache line per slab.  Lane-strided in slab order, then
// block_sum; the total is valid in thread 0, and every workgroup that calls
// it over the same partials obtains the same bits.
template <int NV, int L>
__device__ inline void group_sum_cols(const double *p0, int nslab, long long vstride, int off, double (&out)[NV],
                                      double (&lds)[L])
{
#pragma unroll
  for (int i = 0; i < NV; i++) out[i] = 0.0;
  for (int b = threadIdx.x; b < nslab; b += blockDim.x)
#pragma unroll
    for (int i = 0; i < NV; i++) out[i] += p0[(size_t)(off + i) * vstride + b];
  block_sum<NV>(out, lds);
}
// The sum of value i in thread i < NV.
template <int NV, int L>
__device__ inline double group_sum_cols_lane(const double *p0, int nslab, long long vstride, int off,
                                             double (&lds)[L])
{
  double v[NV];
#pragma unroll
  for (int i = 0; i < NV; i++) v[i] = 0.0;
  for (int b = threadIdx.x; b < nslab; b += blockDim.x)
#pragma unroll
    for (int i = 0; i < NV; i++) v[i] += p0[(size_t)(off + i) * vstride + b];
  return block_sum_lane<NV>(v, lds);
}

// group_sum_cols four values at a time, the totals written to out[] (LDS,
// valid in every thread after the call); the same bits with fewer live
// registers.
template <int NV, int L>
__device__ inline void group_sum_cols_lds(const double *p0, int nslab, long long vstride, int off, double *out,
                                          double (&lds)[L])
{
#pragma unroll 1
  for (int c = 0; c < NV; c += 4) {
    double v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = 0.0;
    for (int b = threadIdx.x; b < nslab; b += blockDim.x)
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (c + i < NV) v[i] += p0[(size_t)(off + c + i) * vstride + b];
    block_sum<4>(v, lds);
    if (threadIdx.x == 0)
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (c + i < NV) out[c + i] = v[i];
  }
  __syncthreads();
}

// The same over row-major partials: value i of slab b at p0[b * stride + i].
template <int NV, int L>
__device__ inline void group_sum_rows(const double *p0, int nslab, int stride, double (&out)[NV],
                                      double (&lds)[L])
{
#pragma unroll
  for (int i = 0; i < NV; i++) out[i] = 0.0;
  for (int b = threadIdx.x; b < nslab; b += blockDim.x)
#pragma unroll
    for (int i = 0; i < NV; i++) out[i] += p0[(size_t)b * stride + i];
  block_sum<NV>(out, lds);
}

// Words that workgroups of a running kernel pass to each other: 32 bits of
// payload under a 32-bit tag, one 64-bit relaxed atomic access at agent scope
// each way.  A reader polls the word until it carries the tag it waits for, so
// payload and readiness arrive together and no fence (an L2 write-back or
// invalidate) is needed.  A word may be rewritten once its reader is known to
// have read it.
typedef unsigned long long word_t;
__device__ __forceinline__ void put_word(word_t *p, unsigned tag, unsigned bits)
{
  __hip_atomic_store(p, ((word_t)tag << 32) | bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ word_t get_word(const word_t *p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A double as two words, and back.
__device__ __forceinline__ void put_double(word_t *p, unsigned tag, double v)
{
  const word_t b = __builtin_bit_cast(word_t, v);
  put_word(p, tag, (unsigned)b);
  put_word(p + 1, tag, (unsigned)(b >> 32));
}
__device__ __forceinline__ double word_double(word_t lo, word_t hi)
{
  return __builtin_bit_cast(double, (hi << 32) | (lo & 0xffffffffull));
}

// Workgroups that are to wait for each other meet first, at two words that are zero
// before: the last to arrive lets them go; the first calls it off when some stay away
// for long, in which case all leave, also those that come later.  Its wait covers
// kernels before this one that still run; it differs from one attempt to the next, so
// that two groups on different streams that keep each other from the CUs do not go on
// doing so.  Run by one lane of each workgroup.
constexpr word_t kMeetGo = 1, kMeetOff = 2;
constexpr int kMeetPolls = 1 << 14;     // some 10 ms, plus as much at random
constexpr int kMeetPatience = 1 << 18;  // some 0.2 s, for groups that leave the others room
__device__ __forceinline__ void meet_set(word_t *meet, word_t to)
{
  word_t none = 0;
  __hip_atomic_compare_exchange_strong(&meet[1], &none, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void meet_off(word_t *meet) { meet_set(meet, kMeetOff); }
// Returns the place among those that arrived (0: the first).
__device__ __forceinline__ int meet_arrive(word_t *meet, int count)
{
  const int n = (int)__hip_atomic_fetch_add(&meet[0], (word_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (n + 1 == count) meet_set(meet, kMeetGo);
  return n;
}
__device__ __forceinline__ bool meet_wait(word_t *meet, int place, int polls)
{
  const int most = place == 0 ? polls + (int)(clock64() & (polls - 1)) : 4 * polls;
  for (int i = 0;; i++) {
    const word_t m = get_word(&meet[1]);
    if (m != 0) return m == kMeetGo;
    if (i >= most) meet_off(meet);
    __builtin_amdgcn_s_sleep(8);
  }
}

}  // namespace mm
