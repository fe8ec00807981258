// engine_sweep.hip -- a whole PCG sweep of an RVE load case on chip.
//
// One workgroup, or a cluster of scw workgroups that split the RVE's interior
// z-planes and, where whole planes are too much, their rows, runs every PCG
// iteration of one sweep of one load case in a single launch: z in LDS (the
// tile's own and the nodes around it), p, q and d in registers, the dictionary
// blocks in LDS.  See RveDev::scw for which RVEs.
//
// Why: kernels A and B move eleven vector passes per iteration through HBM and
// are two to four launches; here an iteration moves only the nodes between ranks
// and the partial sums.  What bounds it: vector issue (of some 250 instructions
// per node and iteration 162 are the multiply-adds of its rows) and, for
// clusters, two exchanges of 2.5 us.  One 30^3 load case (4 ranks of 8 planes,
// FP32) takes 25 us per iteration; kernels A, B and R took 640 us for 768 of
// them, 53 per 64.  Measured on the way there, same case:
//   z neighbours read from LDS, one per key: 38 us; x-neighbours through DPP: 31
//   (LDS reads per node 81 -> 27 dwords);
//   1,024 lanes at 128 VGPRs, items of 4 planes: 32 us (spills, dictionary reads
//   shared by half as many nodes);
//   two workgroups per CU, items of 3 planes: 67 us per 60 load cases (bound by
//   the dictionary's LDS reads);
//   waiting for r.r / r.z before w = A z instead of behind it: 31 us;
//   the planes above and below one by one: 243 multiply-adds, 27.8 to 30.7 us.
// Whole solves (rtol 1e-10), kernels A and B and this: 128 x 30^3 tangents 187 and
// 57 ms, 64 uneven cells 8^3 .. 32^3 50 and 12 ms, 24 x 20^3 in FP64 25.5 and 5.2
// ms, one 10^3 4.7 and 0.67.
// Sharing the rows: 32 x 33 x 36 x 40 tangents 122 and 42 ms, 4 x 60^3 93 and 32;
// one load case of 48^3 7.9 and 3.6 ms, of 100^3 50 and 14, 74 us
// an iteration by kernels A, S, B and R and 20 here.
#include <hip/hip_runtime.h>

#include "engine_device.h"
#include "mm_device.h"
#include "mm_internal.h"
#include "sweep_geo.h"

namespace mm {

namespace {

// The RVE's fields are the same in every lane but read through vector memory;
// readfirstlane keeps them, and every address formed from them, scalar.
__device__ __forceinline__ int scalar(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ SweepGeo sweep_geo_of(const RveDev *R, int rk)
{
  return sweep_geo(scalar(R->nx), scalar(R->ny), scalar(R->nz), scalar(R->scw), scalar(R->sty), scalar(R->slp),
                   scalar(R->snch), rk);
}

// Three consecutive values: one 96-bit LDS read in FP32.
typedef float lds_f3 __attribute__((ext_vector_type(3), aligned(4)));
__device__ __forceinline__ void lds_read3(const float *p, float (&v)[3])
{
  const lds_f3 t = *(const __attribute__((address_space(3))) lds_f3 *)p;
  v[0] = t.x;
  v[1] = t.y;
  v[2] = t.z;
}
__device__ __forceinline__ void lds_read3(const double *p, double (&v)[3])
{
#pragma unroll
  for (int d = 0; d < 3; d++) v[d] = ((const __attribute__((address_space(3))) double *)p)[d];
}

// w[d] += a[e][d] * (x[e][d] of the lane before, DX = 0, or after, DX = 2), e = 0,
// 1, 2 in turn: the shift rides on the multiply-add.  (x may come straight from
// a vector instruction, which a DPP read must not follow within two cycles.)
template <int DX>
__device__ __forceinline__ void fma_lane_x(const float (&a)[3][3], const float *const (&x)[3][3], float (&w)[3])
{
#define MM_FMAC_DPP(SHIFT)                                                             \
  asm("s_nop 1\n\t"                                                                    \
      "v_fmac_f32_dpp %0, %3, %12 " SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
      "v_fmac_f32_dpp %1, %4, %13 " SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
      "v_fmac_f32_dpp %2, %5, %14 " SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
      "v_fmac_f32_dpp %0, %6, %15 " SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
      "v_fmac_f32_dpp %1, %7, %16 " SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
      "v_fmac_f32_dpp %2, %8, %17 " SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
      "v_fmac_f32_dpp %0, %9, %18 " SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
      "v_fmac_f32_dpp %1, %10, %19 " SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
      "v_fmac_f32_dpp %2, %11, %20 " SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:1"     \
      : "+v"(w[0]), "+v"(w[1]), "+v"(w[2])                                               \
      : "v"(*x[0][0]), "v"(*x[0][1]), "v"(*x[0][2]), "v"(*x[1][0]), "v"(*x[1][1]), "v"(*x[1][2]), "v"(*x[2][0]), \
        "v"(*x[2][1]), "v"(*x[2][2]), "v"(a[0][0]), "v"(a[0][1]), "v"(a[0][2]), "v"(a[1][0]), "v"(a[1][1]),      \
        "v"(a[1][2]), "v"(a[2][0]), "v"(a[2][1]), "v"(a[2][2]))
  if constexpr (DX == 0) MM_FMAC_DPP("wave_shr:1");
  else MM_FMAC_DPP("wave_shl:1");
#undef MM_FMAC_DPP
}
template <int DX>
__device__ __forceinline__ double lane_x(double v)
{
  constexpr int shift = DX == 0 ? 0x138 : 0x130;  // wave_shr:1, wave_shl:1
  const int2 b = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_update_dpp(0, b.x, shift, 0xf, 0xf, true),
                                              __builtin_amdgcn_update_dpp(0, b.y, shift, 0xf, 0xf, true)));
}
template <int DX>
__device__ __forceinline__ void fma_lane_x(const double (&a)[3][3], const double *const (&x)[3][3], double (&w)[3])
{
#pragma unroll
  for (int e = 0; e < 3; e++) {
    // (x[e] names one or two values)
    const double x0 = lane_x<DX>(*x[e][0]);
    const double x1 = x[e][1] == x[e][0] ? x0 : lane_x<DX>(*x[e][1]);
    const double x2 = x[e][2] == x[e][0] ? x0 : x[e][2] == x[e][1] ? x1 : lane_x<DX>(*x[e][2]);
    w[0] = fma(a[e][0], x0, w[0]);
    w[1] = fma(a[e][1], x1, w[1]);
    w[2] = fma(a[e][2], x2, w[2]);
  }
}

// w += the block Db times x of the x-neighbour DX (1: the column itself), for LP
// nodes of the lane's column; x(l, e, d): the value that row e, column d multiplies.
template <typename TS, int LP, int DX, typename X>
__device__ __forceinline__ void sweep_key(const TS *Db, const X &x, TS (&w)[LP][3])
{
  constexpr int blk = sweep_dict_block((int)sizeof(TS));
  TS a[3][3];  // [d'][d]
#pragma unroll
  for (int e = 0; e < 3; e++) lds_read3(Db + DX * blk + e * (blk / 3), a[e]);
#pragma unroll
  for (int l = 0; l < LP; l++) {
    const TS *v[3][3];
#pragma unroll
    for (int e = 0; e < 3; e++)
#pragma unroll
      for (int d = 0; d < 3; d++) v[e][d] = &x(l, e, d);
    if constexpr (DX != 1) {
      fma_lane_x<DX>(a, v, w[l]);
    } else {
#pragma unroll
      for (int e = 0; e < 3; e++)
#pragma unroll
        for (int d = 0; d < 3; d++) w[l][d] = fma(a[e][d], *v[e][d], w[l][d]);
    }
  }
}

// w += the nine blocks of the columns at dy, of which the lane's has the rows x
// (from the plane below the first node): those of the node's own plane, then the planes below and above together.  The cell is the
// same mirrored in z (the phases do not vary along z), so the block below is the
// block above with the signs of its xz, yz, zx and zy entries changed: of z above
// and below, the sum goes with the others and the difference with these.  That
// takes 162 multiply-adds and 18 adds per node in place of 243, two thirds of the
// dictionary's reads, and reads a column's z once.
template <typename TS, int LP>
__device__ __forceinline__ void sweep_rows(const TS (&x)[LP + 2][3], const TS *dict, int dy, TS (&w)[LP][3])
{
  constexpr int blk = sweep_dict_block((int)sizeof(TS));
  {
    const TS *Db = dict + (3 * dy + 9) * blk;
    const auto own = [&](int l, int e, int) -> const TS & { return x[l + 1][e]; };
    sweep_key<TS, LP, 0>(Db, own, w);
    sweep_key<TS, LP, 1>(Db, own, w);
    sweep_key<TS, LP, 2>(Db, own, w);
  }
  TS s[LP][3], t[LP][3];
#pragma unroll
  for (int l = 0; l < LP; l++)
#pragma unroll
    for (int e = 0; e < 3; e++) {
      s[l][e] = x[l + 2][e] + x[l][e];
      t[l][e] = x[l + 2][e] - x[l][e];
    }
  const TS *Db = dict + (3 * dy + 18) * blk;
  const auto pair = [&](int l, int e, int d) -> const TS & { return (e == 2) == (d == 2) ? s[l][e] : t[l][e]; };
  sweep_key<TS, LP, 0>(Db, pair, w);
  sweep_key<TS, LP, 1>(Db, pair, w);
  sweep_key<TS, LP, 2>(Db, pair, w);
}

// The same for rows in LDS from zr.
template <typename TS, int LP>
__device__ __forceinline__ void sweep_strip(const TS *zr, int ps, const TS *dict, int dy, TS (&w)[LP][3])
{
  TS x[LP + 2][3];
#pragma unroll
  for (int l = 0; l < LP + 2; l++) lds_read3(zr + l * ps, x[l]);
  sweep_rows<TS, LP>(x, dict, dy, w);
}

// The LDS dictionary of an RVE, by `lanes` lanes: the blocks of the 16 patterns
// that repeat along z, rounded from the FP64 dictionary D (the values of the
// solver dictionary), and an entry of zeros.
template <typename TS>
__device__ __forceinline__ void sweep_dict_load(TS *dict, const double *D, int lanes)
{
  constexpr int stride = sweep_dict_stride((int)sizeof(TS)), blk = sweep_dict_block((int)sizeof(TS));
  for (int i = threadIdx.x; i < stride; i += lanes) dict[16 * stride + i] = (TS)0;
  for (int i = threadIdx.x; i < 16 * 27 * 9; i += lanes) {
    const int e = i / (27 * 9), o = i - e * (27 * 9), key = o / 9, j = o - key * 9;
    dict[e * stride + key * blk + (j / 3) * (blk / 3) + j % 3] =
        (TS)D[(size_t)(e * 17) * kDictEntry + key * kDictBlk + (j / 3) * 4 + j % 3];
  }
}

// Bound on a wait in polls (half a minute or more).  A rank waits for the
// slowest of its cluster to run one phase, or, before its first exchange, for a
// rank that has no CU yet: until a running sweep ends.  A wait that reaches the
// bound ends the sweep without an update.
constexpr int kSweepPolls = 1 << 25;

// A double moved between lanes (0 where no lane supplies one).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_get(double v)
{
  const int2 b = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_update_dpp(0, b.x, CTRL, ROWS, 0xf, true),
                                              __builtin_amdgcn_update_dpp(0, b.y, CTRL, ROWS, 0xf, true)));
}

// Sums NV values over the workgroup: valid in every lane, one barrier.  buf
// (NV * 8 doubles) must not be rewritten before the next barrier.
template <int NV>
__device__ __forceinline__ void lanes_sum(double (&v)[NV], double *buf)
{
#pragma unroll
  for (int i = 0; i < NV; i++) {
    v[i] += dpp_get<0x111, 0xf>(v[i]);  // row_shr:1, 2, 4, 8: lane 15 of each row has its sum
    v[i] += dpp_get<0x112, 0xf>(v[i]);
    v[i] += dpp_get<0x114, 0xf>(v[i]);
    v[i] += dpp_get<0x118, 0xf>(v[i]);
    v[i] += dpp_get<0x142, 0xa>(v[i]);  // row_bcast:15 into rows 1 and 3
    v[i] += dpp_get<0x143, 0xc>(v[i]);  // row_bcast:31 into rows 2 and 3: lane 63 has the total
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 63)
#pragma unroll
    for (int i = 0; i < NV; i++) buf[i * (kSweepLanes / 64) + wid] = v[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NV; i++) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kSweepLanes / 64; w++) s += buf[i * (kSweepLanes / 64) + w];
    v[i] = s;
  }
}

// (A word that the ranks of a cluster exchange is rewritten only after a sum
// over the cluster that its reader joined after reading it.)

// Sums NV values over the workgroups of a cluster: lane 0 posts the workgroup's
// own, every wave then collects all of them and adds them in rank order, so
// that every lane of every rank has the same bits.  Collecting returns false
// when the wait ran out.
template <int NV>
__device__ __forceinline__ void cluster_post(const double (&v)[NV], word_t *sum, int rk, unsigned tag)
{
  if (threadIdx.x == 0)
#pragma unroll
    for (int i = 0; i < NV; i++) put_double(sum + rk * 8 + 2 * i, tag, v[i]);
}
template <int NV>
__device__ __forceinline__ bool cluster_collect(double (&v)[NV], const word_t *sum, int cw, unsigned tag)
{
  const int lane = threadIdx.x & 63;
  const bool mine = lane < cw * 2 * NV;
  const word_t *src = sum + (mine ? (lane / (2 * NV)) * 8 + lane % (2 * NV) : 0);
  word_t w = 0;
  int n = 0;
  for (;;) {
    if (mine) w = get_word(src);
    if (__all(!mine || (unsigned)(w >> 32) == tag)) break;
    if (++n > kSweepPolls) return false;
  }
  const unsigned bits = (unsigned)w;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    double s = 0.0;
    for (int r = 0; r < cw; r++) {
      const unsigned lo = __builtin_amdgcn_readlane(bits, r * 2 * NV + 2 * i);
      const unsigned hi = __builtin_amdgcn_readlane(bits, r * 2 * NV + 2 * i + 1);
      s += __builtin_bit_cast(double, ((word_t)hi << 32) | lo);
    }
    v[i] = s;
  }
  return true;
}

// The same for clusters of more ranks than fit a wave's lanes: lane r collects
// rank r's and the workgroup adds them (lanes_sum, a barrier).
template <int NV>
__device__ __forceinline__ bool cluster_collect_many(double (&v)[NV], const word_t *sum, int cw, unsigned tag,
                                                     double *buf)
{
  const bool mine = (int)threadIdx.x < cw;
  const word_t *src = sum + (mine ? (int)threadIdx.x * 8 : 0);
  word_t w[2 * NV];
  bool ok = true;
  int n = 0;
  for (;;) {
    bool all = true;
#pragma unroll
    for (int i = 0; i < 2 * NV; i++) w[i] = get_word(src + i);
#pragma unroll
    for (int i = 0; i < 2 * NV; i++) all = all && (unsigned)(w[i] >> 32) == tag;
    if (!mine || all) break;
    if (++n > kSweepPolls) {
      ok = false;
      break;
    }
  }
#pragma unroll
  for (int i = 0; i < NV; i++) v[i] = mine ? word_double(w[2 * i], w[2 * i + 1]) : 0.0;
  lanes_sum<NV>(v, buf);
  return ok;
}
template <int NV>
__device__ __forceinline__ bool cluster_sum(double (&v)[NV], const word_t *sum, int cw, unsigned tag, double *buf)
{
  if (cw > kSweepFreeRanks) return cluster_collect_many<NV>(v, sum, cw, tag, buf);
  return cluster_collect<NV>(v, sum, cw, tag);
}

// Publishes a node's three rows as the words of interior node at.
__device__ __forceinline__ void put_node(const SweepWords &X, int ni, int at, unsigned tag, const float (&x)[3])
{
#pragma unroll
  for (int d = 0; d < 3; d++) put_word(X.w[d] + at, tag, __builtin_bit_cast(unsigned, x[d]));
}
__device__ __forceinline__ void put_node(const SweepWords &X, int ni, int at, unsigned tag, const double (&x)[3])
{
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const word_t b = __builtin_bit_cast(word_t, x[d]);
    put_word(X.w[d] + at, tag, (unsigned)b);
    put_word(X.w[d] + ni + at, tag, (unsigned)(b >> 32));
  }
}
__device__ __forceinline__ void word_node(const word_t *w, float *dst)
{
#pragma unroll
  for (int d = 0; d < 3; d++) dst[d] = __builtin_bit_cast(float, (unsigned)w[d]);
}
__device__ __forceinline__ void word_node(const word_t *w, double *dst)
{
#pragma unroll
  for (int d = 0; d < 3; d++) dst[d] = word_double(w[2 * d], w[2 * d + 1]);
}

// The nodes beside the tile (sweep_place) <- the words that the neighbouring ranks
// published under `tag`.  U nodes of either side per trip, all their words asked
// for together, again until each carries the tag.
template <typename TS>
__device__ __forceinline__ bool get_halo(const SweepGeo &g, TS *zl, const SweepWords &X, unsigned tag)
{
  constexpr int H = (int)(sizeof(TS) / 4), W = 3 * H, U = H == 1 ? 2 : 1;
  const SweepHalo h = sweep_halo(g);
  const word_t none = (word_t)tag << 32;
  bool ok = true;
  int c0 = threadIdx.x;
  asm volatile("" : "+v"(c0));  // the places are formed here, not kept from one iteration to the next
  for (; c0 < h.n; c0 += U * kSweepLanes) {
    int at[U], dst[U], dat[U], ddst[U];
    bool lo[U], hi[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      sweep_place(g, h.r0, h.n1, h.n, c0 + u * kSweepLanes, at[u], dst[u], dat[u], ddst[u], lo[u], hi[u]);
    }
    word_t a[U][W], b[U][W];
    int m = 0;
    for (;;) {
      bool all = true;
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int i = 0; i < W; i++) {
          const word_t *w = X.w[i / H] + (long long)(i % H) * g.ni + at[u];
          a[u][i] = lo[u] ? get_word(w) : none;
          b[u][i] = hi[u] ? get_word(w + dat[u]) : none;
        }
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int i = 0; i < W; i++)
          all = all && (unsigned)(a[u][i] >> 32) == tag && (unsigned)(b[u][i] >> 32) == tag;
      if (all) break;
      if (++m > kSweepPolls) {
        ok = false;
        break;
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (lo[u]) word_node(a[u], zl + dst[u] * 3);
      if (hi[u]) word_node(b[u], zl + (dst[u] + ddst[u]) * 3);
    }
  }
  return ok;
}

// Item j of lane tid.
__device__ __forceinline__ SweepItem sweep_item_of(const SweepGeo &g, int tid, int j)
{
  return sweep_item(g, scalar((tid >> 6) + j * (kSweepLanes / 64)), tid & 63);
}

// The sweep of one load case on this workgroup's tile; zl holds z = dinv r of
// the sweep's right-hand side.  An item is one interior column times lp planes,
// LP >= lp of its nodes' rows in registers, one lane each; a wave takes strips
// of kSweepStrip consecutive positions, so that the x-neighbours of a node are
// the lanes beside it and come from them (DPP) instead of LDS.  The recurrences
// are kernel A's and kernel B's (r = z / dinv formed for the dots); the row sums
// (sweep_strip) and the dot products are grouped differently.  Returns the
// iterations taken.
template <typename TS, int LP>
__device__ __forceinline__ int sweep_case(const EngPtrs &P, const SweepGeo &g, int fs, int K, int k, TS *zl,
                                          const TS *dict, double *red, int *s_fail, const SweepWords &X, double rz,
                                          double tgt, int max_its)
{
  constexpr int NI = kSweepItems;
  const int tid = threadIdx.x, SN = P.SN, RS = 3 * SN;
  TS p[NI][LP][3], q[NI][LP][3], dd[NI][LP][3];
  int z0[NI], d0[NI], cnt[NI], wd[NI];
  unsigned put[NI];  // sweep_put
#pragma unroll
  for (int j = 0; j < NI; j++) {
    const SweepItem it = sweep_item_of(g, tid, j);
    cnt[j] = scalar(it.cnt);
    put[j] = sweep_put(g, it);
    wd[j] = it.word;
    z0[j] = it.lds * 3;
    // the phases do not vary along z: one pattern per column; lanes without a
    // node take the zero entry, so that their q, r and dot products are zero
    const int pat = P.npat[(long long)(fs + (it.node >> P.sn_shift)) * SN + (it.node & (SN - 1))] & 15;
    d0[j] = (it.on ? pat : 16) * sweep_dict_stride((int)sizeof(TS));
#pragma unroll
    for (int l = 0; l < LP; l++)
#pragma unroll
      for (int d = 0; d < 3; d++) p[j][l][d] = q[j][l][d] = dd[j][l][d] = (TS)0;
  }
  const int ps0 = g.pw * 3;
  const word_t *sum2 = X.sum + 8 * g.cw;
  double v2[2] = {0.0, 0.0};
  int n = 0;
#pragma unroll 1
  for (;;) {
    double v1[1] = {0.0}, beta = 0.0;
    TS b;
    bool done = false;
    // opaque per iteration: the addresses that follow from these are formed
    // where they are used and not kept in registers
    int ps = ps0;
    asm volatile("" : "+s"(ps));
#pragma unroll
    for (int j = 0; j < NI; j++) asm volatile("" : "+v"(z0[j]), "+v"(wd[j]), "+v"(put[j]));
#pragma unroll
    for (int j = 0; j < NI; j++) {
      if (j > 0 && cnt[j] == 0) continue;
      TS w[LP][3];
#pragma unroll
      for (int l = 0; l < LP; l++)
#pragma unroll
        for (int d = 0; d < 3; d++) w[l][d] = (TS)0;
      const TS *zr = zl + z0[j] - g.rsx * 3, *Db = dict + d0[j];
#pragma unroll 1
      for (int dy = 0; dy < 3; dy++) sweep_strip<TS, LP>(zr + dy * g.rsx * 3, ps, Db, dy, w);
      if (j == 0) {
        // w = A z needs neither r.r nor r.z of the last update: their sums over
        // the cluster, posted before it, have arrived by now
        if (n > 0) {
          if (g.cw > 1 && !cluster_sum<2>(v2, sum2, g.cw, (unsigned)n, red + 4 * (kSweepLanes / 64))) *s_fail = 1;
          done = scalar(sqrt(v2[0]) <= tgt || rz == 0.0 || n >= max_its) != 0;
          if (done) break;
          beta = v2[1] / rz;
          rz = v2[1];
        }
        b = (TS)beta;
      }
      TS x[LP][3];
#pragma unroll
      for (int l = 0; l < LP; l++) lds_read3(zl + z0[j] + (l + 1) * ps, x[l]);
#pragma unroll
      for (int l = 0; l < LP; l++) {
        if (l >= cnt[j]) break;
#pragma unroll
        for (int d = 0; d < 3; d++) {
          p[j][l][d] = fma(b, p[j][l][d], x[l][d]);
          q[j][l][d] = fma(b, q[j][l][d], w[l][d]);
          v1[0] = fma((double)p[j][l][d], (double)q[j][l][d], v1[0]);
        }
      }
    }
    if (done) break;
    const unsigned tag = (unsigned)n + 1u;
    lanes_sum<1>(v1, red);
    if (g.cw > 1) {
      cluster_post<1>(v1, X.sum, g.rk, tag);
      if (!cluster_sum<1>(v1, X.sum, g.cw, tag, red + 3 * (kSweepLanes / 64))) *s_fail = 1;
    }
    const TS al = (TS)((v1[0] == 0.0) ? 0.0 : rz / v1[0]);
    v2[0] = v2[1] = 0.0;
#pragma unroll
    for (int j = 0; j < NI; j++) {
      if (j > 0 && cnt[j] == 0) continue;
      TS dg[3], yg[3];  // the column's dinv and its reciprocal, after its blocks
      lds_read3(dict + d0[j] + 27 * sweep_dict_block((int)sizeof(TS)), dg);
      lds_read3(dict + d0[j] + 27 * sweep_dict_block((int)sizeof(TS)) + sweep_dict_block((int)sizeof(TS)) / 3, yg);
      TS x[LP][3];
#pragma unroll
      for (int l = 0; l < LP; l++) lds_read3(zl + z0[j] + (l + 1) * ps, x[l]);
#pragma unroll
      for (int l = 0; l < LP; l++) {
        if (l >= cnt[j]) break;
#pragma unroll
        for (int d = 0; d < 3; d++) {
          dd[j][l][d] = fma(al, p[j][l][d], dd[j][l][d]);
          const TS zi = fma(-al, dg[d] * q[j][l][d], x[l][d]);
          x[l][d] = zi;
          // r = z / dinv: the quotient from the reciprocal and its exact
          // remainder, correctly rounded (Markstein)
          TS r = zi * yg[d];
          r = fma(fma(-r, dg[d], zi), yg[d], r);
          v2[0] = fma((double)r, (double)r, v2[0]);
          v2[1] = fma((double)r, (double)zi, v2[1]);
        }
        if ((int)put[j] < 0) {
#pragma unroll
          for (int d = 0; d < 3; d++) zl[z0[j] + (l + 1) * ps + d] = x[l][d];
          if ((put[j] >> l) & 1u) put_node(X, g.ni, wd[j] + l * g.nixy, tag, x[l]);
        }
      }
    }
    lanes_sum<2>(v2, red + kSweepLanes / 64);  // its barrier also ends the writes of z
    n++;
    if (g.cw > 1) {
      cluster_post<2>(v2, X.sum + 8 * g.cw, g.rk, tag);
      if (!get_halo<TS>(g, zl, X, tag)) *s_fail = 1;
      __syncthreads();
      if (scalar(*s_fail)) return n;  // a wait ran out: no update; the residual shows it
    }
  }
  if (g.cw > 1) {
    __syncthreads();
    if (scalar(*s_fail)) return n;
  }
  int t2 = tid;
  asm volatile("" : "+v"(t2));  // the items' nodes are formed again, not kept
#pragma unroll
  for (int j = 0; j < NI; j++) {
    const SweepItem it = sweep_item_of(g, t2, j);
#pragma unroll
    for (int l = 0; l < LP; l++)
      if (it.on && l < it.cnt) {
        const int m = it.node + l * g.nxy;
        double *xo = P.x64 + ((long long)(fs + (m >> P.sn_shift)) * K + k) * RS + 3 * (m & (SN - 1));
#pragma unroll
        for (int d = 0; d < 3; d++) xo[d] += (double)dd[j][l][d];
      }
  }
  return n;
}

// sweep_case for the tile's item length.
template <typename TS>
struct SweepRun {
  const EngPtrs &P;
  const SweepGeo &g;
  int fs, K, k;
  TS *zl;
  const TS *dict;
  double *red;
  int *fail;
  const SweepWords &X;
  double rz, tgt;
  int max_its;
  template <int LP>
  __device__ __forceinline__ int go() const
  {
    if constexpr (LP > 2)
      if (g.lp <= sweep_shorter(LP)) return go<sweep_shorter(LP)>();
    return sweep_case<TS, LP>(P, g, fs, K, k, zl, dict, red, fail, X, rz, tgt, max_its);
  }
};

extern __shared__ __attribute__((aligned(16))) double sweep_dyn[];

}  // namespace

// The resident RVEs' kernel A (reads st[2], writes st[0]).  Workgroups take the
// entries of the unit list (RVE slot, load case * 256 + rank) by ticket, in list
// order: the ranks of a cluster are consecutive entries, so the started
// workgroups form whole clusters but for the last one, the whole ones finish
// without waiting for anyone else, and their places go to the missing ranks
// (also beside other such launches: each leaves at most one cluster of at most
// sweep_free_ranks workgroups waiting, and the GPU has more places than the
// queues' launches can fill with those).  A cluster waits only before it has
// started (meet_wait), a larger one not for long.
// The residual follows (k_sweep_res), and kernel R passes the state on.
template <typename TS, int K>
__global__ __launch_bounds__(kSweepLanes) void k_sweep(EngPtrs P, SolveParams sp)
{
  __shared__ double lds[64];
  __shared__ double red[6 * (kSweepLanes / 64)];
  __shared__ double tot[4 * K];
  __shared__ SolveState N;
  __shared__ int s_unit, s_fail;
  const int tid = threadIdx.x;
  if (tid == 0) {
    s_unit = (int)__hip_atomic_fetch_add(P.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_fail = 0;
  }
  __syncthreads();
  const int u = scalar(s_unit);
  if (u >= P.units[0].x) return;
  const int slot = scalar(P.units[1 + u].x);
  const int case_rank = scalar(P.units[1 + u].y);
  const int k = case_rank / kSweepUnitRanks, rk = case_rank % kSweepUnitRanks;
  RveDev *R = P.rves + slot;
  const int phase0 = R->st[2].phase;
  const bool writer = k == 0 && rk == 0;
  if (phase0 == PH_AVGRED) {
    if (!writer) return;
    if (tid == 0) N = R->st[2];
    __syncthreads();
    finish_rve<K>(P, slot, R, N, sp);
    if (tid == 0) R->st[0] = N;
    return;
  }
  if (tid == 0) N = R->st[2];
  if (phase0 == PH_RESRED) {
    group_sum_cols_lds<4 * K>(slab_part(P, R->first_slab).p, R->nslab, P.part_stride, 3 * K, tot, lds);
    if (tid == 0) start_sweep<K>(N, *reinterpret_cast<const double(*)[4 * K]>(tot), R, sp);
  }
  __syncthreads();
  if (writer && tid == 0) R->st[0] = N;
  if (N.phase != PH_INNER || ((N.done_in >> k) & 1u)) return;

  const SweepGeo g = sweep_geo_of(R, rk);
  const int SN = P.SN, RS = 3 * SN, fs = scalar(R->first_slab), tsz = (int)sizeof(TS);
  const SweepWords X = sweep_words<TS>(P, scalar(R->nslab), K, fs, k, g.ni);
  const int meets = scalar(R->smeet);
  if (meets) {
    if (tid == 0) {
      word_t *meet = X.sum + 16 * g.cw;
      if ((sp.meet_off >> k) & 1u) meet_off(meet);
      s_unit = meet_wait(meet, meet_arrive(meet, g.cw), meets == kSweepMeetLarge ? kMeetPolls : kMeetPatience) ? 1 : 0;
    }
    __syncthreads();
    if (scalar(s_unit) == 0) return;
  }
  TS *dict = reinterpret_cast<TS *>(sweep_dyn);
  TS *zl = reinterpret_cast<TS *>(reinterpret_cast<unsigned char *>(sweep_dyn) + sweep_dict_bytes(tsz));
  const double *D = P.dict64 + (size_t)slot * kDictPat * kDictEntry;
  sweep_dict_load<TS>(dict, D, kSweepLanes);
  for (int i = tid; i < 16 * 3; i += kSweepLanes) {
    const int e = i / 3, d = i - e * 3;
    // the solver's dinv of a node of that pattern, and its reciprocal
    const TS dg = (TS)(1.0 / D[(size_t)(e * 17) * kDictEntry + 13 * kDictBlk + d * 4 + d]);
    TS *o = dict + e * sweep_dict_stride(tsz) + 27 * sweep_dict_block(tsz) + d;
    o[0] = dg;
    o[sweep_dict_block(tsz) / 3] = (TS)1 / dg;
  }
  const int zlen = sweep_lds_planes(tsz, g.lp, g.nch) * g.pw * 3;
  for (int i = tid; i < zlen; i += kSweepLanes) zl[i] = (TS)0;
  __syncthreads();
  for (int s = 0; s < g.np + 2; s++) {
    const int z = g.zs - 1 + s;
    if (z == 0 || z == R->nz - 1) continue;
    for (int c = tid; c < (g.nr + 2) * g.nix; c += kSweepLanes) {
      const int r = c / g.nix, ix = c - r * g.nix;
      if ((r == 0 && !g.ylo) || (r == g.nr + 1 && !g.yhi)) continue;
      const int m = (ix + 1) + (g.ys + r) * g.nx + z * g.nxy;
      const TS *src = (const TS *)P.z + ((long long)(fs + (m >> P.sn_shift)) * K + k) * RS + 3 * (m & (SN - 1));
      TS *dst = zl + (s * g.pw + 1 + r * g.rsx + ix) * 3;
#pragma unroll
      for (int d = 0; d < 3; d++) dst[d] = src[d];
    }
  }
  __syncthreads();
  const double rz = N.rz[k], tgt = N.bnorm_in[k];
  int n;
  const SweepRun<TS> run{P, g, fs, K, k, zl, dict, red, &s_fail, X, rz, tgt, sp.max_inner_its};
  n = run.template go<sweep_max_planes((int)sizeof(TS))>();
  if (rk == 0 && tid == 0) R->lits[k] = n;
}

// The resident RVEs' FP64 residual (kernel R does the others'), between sweeps:
// r = -K x64, z = dinv r, the partial sums of kernel R, and the words of the next
// sweep zeroed.  The state is still k_sweep's (st[0]); kernel R passes it on.
//
// Workgroup b of an RVE takes items b * kResWaves + wave, + nslab * kResWaves, ..:
// a strip of 62 positions of a plane's rows, kResPlanes nodes of each column and
// one load case, with the sweep's product (sweep_rows) on rows read from memory.
// x-neighbours come from the lanes beside, the dictionary from LDS.  Bound by
// vector issue (180 FP64 operations per node, and 54 moves between lanes).  Kernel
// R gathers 27 neighbours per node through L1, 81 reads in place of 13.5, and took
// 22 us for one 10^3 cell with 6 load cases and 100 for 24 cells of 12^3 .. 30^3
// with 7; this takes 14 and, with the boundary part twice, 82.
constexpr int kResWaves = 4;
constexpr int kResPlanes = 4;

template <typename TS, int K>
__global__ __launch_bounds__(64 * kResWaves) void k_sweep_res(EngPtrs P)
{
  __shared__ double acc[kResWaves][4 * K];
  int slab;
  if (!active_slab(P, slab)) return;
  slab = scalar(slab);
  const int slot = scalar(P.slab_rve[slab]);
  if (slot < 0) return;
  const RveDev *R = P.rves + slot;
  if (scalar(R->scw) == 0 || !sweep_ran<TS, K>(P, R)) return;
  const bool cold = scalar((R->warm || R->affine) && R->st[0].phase == PH_RES && R->st[0].sweep == 0) != 0;
  const int tid = threadIdx.x, ln = tid & 63, wv = tid >> 6;
  const int nx = scalar(R->nx), ny = scalar(R->ny), nz = scalar(R->nz), nxy = nx * ny;
  const int fs = scalar(R->first_slab), nslab = scalar(R->nslab), nload = scalar(R->nload);
  const int SN = P.SN, RS = 3 * SN, b = slab - fs;
  const int npos = nx * (ny - 2), nstrip = (npos + kSweepStrip - 1) / kSweepStrip;
  const int nrun = (nz - 2 + kResPlanes - 1) / kResPlanes, items = nstrip * nrun * nload;
  if (R->scw > 1) sweep_words_zero<TS, K>(P, R, slab);
  double *dict = sweep_dyn;
  for (int i = tid; i < kResWaves * 4 * K; i += 64 * kResWaves) (&acc[0][0])[i] = 0.0;
  if (b * kResWaves < items) sweep_dict_load<double>(dict, P.dict64 + (size_t)slot * kDictPat * kDictEntry, 64 * kResWaves);
  __syncthreads();
#pragma unroll 1
  for (int it = scalar(b * kResWaves + wv); it < items; it += nslab * kResWaves) {
    const int k = it % nload, u = it / nload, run = u % nrun, st = u / nrun;
    const int zf = 1 + run * kResPlanes, cnt = min(kResPlanes, nz - 1 - zf);
    const int pos = st * kSweepStrip + ln - 1, pc = min(max(pos, 0), npos - 1);
    const int iy = pc / nx, ix = pc - iy * nx;  // row iy + 1 of the plane
    const bool bx = ix == 0 || ix == nx - 1;
    const bool on = ln >= 1 && ln <= kSweepStrip && pos < npos && !bx;
    const int n0 = ix + (iy + 1) * nx + zf * nxy;
    const int pat = P.npat[(long long)(fs + (n0 >> P.sn_shift)) * SN + (n0 & (SN - 1))] & 15;
    const double *Db = dict + (on ? pat : 16) * sweep_dict_stride(8);
    double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for (int pass = 0; pass <= (cold ? 1 : 0); pass++) {  // pass 1: the boundary nodes' part alone
      double w[kResPlanes][3];
#pragma unroll
      for (int l = 0; l < kResPlanes; l++)
#pragma unroll
        for (int d = 0; d < 3; d++) w[l][d] = 0.0;
#pragma unroll 1
      for (int dy = 0; dy < 3; dy++) {
        const bool column = pass == 0 || bx || iy + dy == 0 || iy + dy == ny - 1;
        double x[kResPlanes + 2][3];
#pragma unroll
        for (int l = 0; l < kResPlanes + 2; l++) {
          const int z = min(zf - 1 + l, nz - 1), m = n0 + (dy - 1) * nx + (z - zf) * nxy;
          const double *src = P.x64 + ((long long)(fs + (m >> P.sn_shift)) * K + k) * RS + 3 * (m & (SN - 1));
          const bool keep = column || z == 0 || z == nz - 1;
#pragma unroll
          for (int d = 0; d < 3; d++) x[l][d] = keep ? src[d] : 0.0;
        }
        sweep_rows<double, kResPlanes>(x, Db, dy, w);
      }
#pragma unroll
      for (int l = 0; l < kResPlanes; l++) {
        if (!on || l >= cnt) continue;
        const int m = n0 + l * nxy;
        const long long sl = fs + (m >> P.sn_shift);
        const int row = 3 * (m & (SN - 1));
        const TS *dinv = (const TS *)P.dinv + sl * RS + row;
        TS *z = (TS *)P.z + (sl * K + k) * RS + row;
#pragma unroll
        for (int d = 0; d < 3; d++) {
          const double r64 = -w[l][d];
          if (pass == 0) {
            const TS r = (TS)r64, zi = dinv[d] * r;
            z[d] = zi;
            v[0] = fma(r64, r64, v[0]);
            v[1] = fma((double)r, (double)r, v[1]);
            v[2] = fma((double)r, (double)zi, v[2]);
          } else {
            v[3] = fma(r64, r64, v[3]);
          }
        }
      }
    }
    int q;
    const double t = wave_sum4(v, q);
    if ((ln & 15) == 0) acc[wv][q * K + k] += t;
  }
  __syncthreads();
  if (tid < 4 * K) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < kResWaves; w++) t += acc[w][tid];
    slab_part(P, slab)[3 * K + tid] = t;
  }
}

template <typename TS, int K>
static int launch_sweep_res(const EngPtrs &P, int grid, hipStream_t s)
{
  if (grid <= 0) return MM_ERR_ARG;
  k_sweep_res<TS, K><<<grid, 64 * kResWaves, sweep_dict_bytes(8), s>>>(P);
  MM_HIP(hipGetLastError());
  return 0;
}

template <typename TS, int K>
static int launch_sweep(const EngPtrs &P, const SolveParams &sp, hipStream_t s)
{
  if (P.u_grid <= 0 || P.u_lds <= 0 || P.u_lds > kSweepMaxLds) return MM_ERR_ARG;
  k_sweep<TS, K><<<P.u_grid, kSweepLanes, P.u_lds, s>>>(P, sp);
  MM_HIP(hipGetLastError());
  return 0;
}

#define MM_SWEEP_DISPATCH(FP64, K, F, ...)       \
  do {                                           \
    if (FP64) {                                  \
      switch (K) {                               \
        case 1: return F<double, 1>(__VA_ARGS__); \
        case 6: return F<double, 6>(__VA_ARGS__); \
        case 7: return F<double, 7>(__VA_ARGS__); \
        default: return MM_ERR_ARG;              \
      }                                          \
    }                                            \
    switch (K) {                                 \
      case 1: return F<float, 1>(__VA_ARGS__);   \
      case 6: return F<float, 6>(__VA_ARGS__);   \
      case 7: return F<float, 7>(__VA_ARGS__);   \
      default: return MM_ERR_ARG;                \
    }                                            \
  } while (0)

int eng_launch_sweep(bool fp64, int K, const EngPtrs &P, const SolveParams &sp, hipStream_t s)
{
  MM_SWEEP_DISPATCH(fp64, K, launch_sweep, P, sp, s);
}

int eng_launch_sweep_res(bool fp64, int K, const EngPtrs &P, int grid, hipStream_t s)
{
  MM_SWEEP_DISPATCH(fp64, K, launch_sweep_res, P, grid, s);
}

}  // namespace mm
