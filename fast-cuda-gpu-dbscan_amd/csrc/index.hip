// Grid-index build on gfx950: the MI355X replacement for the reference's
// tree index (indexing.cu:23-118, main.cu:166-340).
//
//   k_bbox        per-instance bounding box (main.cu:166-181 does it on the
//                 host, initialised to 0 / 999999999; here +-inf)
//   k_grid_setup  cell width, cells per axis, key space per instance
//                 (main.cu:184-207 bin width + eps check, main.cu:209-244 tree
//                 metadata: replaced by a flat grid); with one instance done
//                 by the last workgroup of k_bbox
//   k_cellkey(_hist)  per-point cell key (insertData, indexing.cu:107-118)
//   radix sort    LDS radix sort of (key, id), stable (thrust::sort_by_key,
//                 main.cu:332-333)
//   CSR           wavefront ballot/mbcnt compaction of key changes into cell
//                 ranges (INDEXING_ADJUSTMENT's per-leaf equal_range,
//                 indexing.cu:23-51), and the table of columns
//   k_gather      cell-sorted SoA coordinates (FP64 + fixed-point)
//   k_rows        the windows of each cell's 3^(D-1) neighbour columns that
//                 cover its stencil (cells of side eps/2, a 5^D stencil;
//                 searchPoints' level-by-level descent, dbscan.cu:390-474)
#include "internal.h"
#include "kernels.h"

#include <algorithm>
#include <type_traits>
#include <cmath>

namespace dclust {

// ------------------------------------------------------------------ fill --
static int fill_grid(int64_t n) {
  int64_t b = (n + 255) / 256;
  if (b > 4096) b = 4096;
  if (b < 1) b = 1;
  return (int)b;
}

// Start of a run, one launch: control counters, statistics stripes, the sort's
// group counts and the bounding-box stripes (per instance and stripe: 0..2 min
// as ordered keys starting at the largest key, 3..5 max, 6 max |x|, 7
// non-finite flag, all starting at 0).  What the call brings (input, output,
// the parameters of a single instance) is taken from `src` (pinned host
// memory) in a captured run, whose replays read what the host left there,
// else from `v`.
constexpr int64_t kGroupWords = ((int64_t)kSortPasses * kSortGroups << kDigitBits) / 2;
__global__ __launch_bounds__(256) void k_init_head(Dev d, const Call* src, Call v) {
  constexpr int kInstWords = sizeof(Inst) / 8;
  const int64_t nb = (int64_t)d.ninst * kBoxStripes * 8;
  const int64_t ns = (int64_t)kStatStride * kStripes;
  const int64_t ni = d.ninst == 1 ? kInstWords : d.ninst;
  const int64_t tot = nb + ns + C_NCTL + ni + kGroupWords;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < tot;
       i += (int64_t)gridDim.x * blockDim.x) {
    if (i < nb) {
      d.bbox[i] = (i & 7) < 3 ? ~0ull : 0ull;
    } else if (i < nb + ns) {
      d.stat[i - nb] = 0;
    } else if (i < nb + ns + C_NCTL) {
      const int c = (int)(i - nb - ns);
      long long w = 0;
      if (c == C_XYZ) w = reinterpret_cast<long long>(src ? src->xyz : v.xyz);
      if (c == C_LABELS) w = reinterpret_cast<long long>(src ? src->labels : v.labels);
      if (c == C_T_START) w = (long long)__builtin_amdgcn_s_memrealtime();
      d.ctl[c] = w;
    } else if (i >= tot - kGroupWords) {
      reinterpret_cast<unsigned long long*>(d.dgrp)[i - (tot - kGroupWords)] = 0ull;
    } else {
      const int64_t k = i - nb - ns - C_NCTL;
      if (d.ninst == 1) {
        // (src is null or not for the whole launch; v stays in the kernel's
        // argument memory)
        const unsigned long long* from =
            reinterpret_cast<const unsigned long long*>(src ? &src->inst : &v.inst);
        reinterpret_cast<unsigned long long*>(d.inst)[k] = from[k];
      } else {
        d.inst[k].err = 0;  // (the table may be last run's)
      }
    }
  }
}

void launch_init_head(const Dev& d, const Call* src, const Call& v, hipStream_t s) {
  const int64_t tot = (int64_t)d.ninst * kBoxStripes * 8 + (int64_t)kStatStride * kStripes + C_NCTL +
                      std::max<int64_t>(d.ninst, sizeof(Inst) / 8) + kGroupWords;
  hipLaunchKernelGGL(k_init_head, dim3(fill_grid(tot)), dim3(256), 0, s, d, src, v);
}

// The counters after the grid set-up of an eager run (a run's last kernel
// reads them back itself).
__global__ __launch_bounds__(1024) void k_readback(Dev d, long long* out) { readback(d, out); }

void launch_readback(const Dev& d, long long* out, hipStream_t s) {
  hipLaunchKernelGGL(k_readback, dim3(1), dim3(1024), 0, s, d, out);
}

// ------------------------------------------------------------------ bbox --

// One block per chunk (chunks never straddle instances).  Block reduction,
// then one ordered-u64 atomic min/max per axis.  Non-finite input sets the
// instance error.
// Points of a chunk per thread step: the loads of kChunkU points (strided
// by the block) are issued before any is used, so their latencies overlap.
constexpr int kChunkU = 4;

template <int D>
__device__ __forceinline__ void bbox_points(const double* p0, int64_t np, double (&mn)[3],
                                            double (&mx)[3], double& ma, bool& bad) {
  for (int64_t i0 = threadIdx.x; i0 < np; i0 += kChunkU * 256) {
    double v[kChunkU][D];
#pragma unroll
    for (int u = 0; u < kChunkU; ++u) {
      // past the end: the chunk's last point again (min and max unchanged)
      const int64_t i = i0 + u * 256 < np ? i0 + u * 256 : np - 1;
#pragma unroll
      for (int k = 0; k < D; ++k) v[u][k] = p0[i * D + k];
    }
#pragma unroll
    for (int u = 0; u < kChunkU; ++u)
#pragma unroll
      for (int k = 0; k < D; ++k) {
        bad |= !isfinite(v[u][k]);
        mn[k] = fmin(mn[k], v[u][k]);
        mx[k] = fmax(mx[k], v[u][k]);
        ma = fmax(ma, fabs(v[u][k]));
      }
  }
}

__device__ void setup_instance(Inst& I, const unsigned long long (&bb)[8],
                               unsigned long long& cells, unsigned long long& keys,
                               long long& lines);
__device__ void setup_totals(const Dev& d, unsigned long long cells, unsigned long long keys,
                             long long lines, int err);

// (a call of one instance has no separate grid set-up: the workgroup that
// finishes last does it, from coherent loads of the stripes, which saves a
// launch of one workgroup that took 11 to 19 us)
__global__ __launch_bounds__(256, 6) void k_bbox(Dev d) {
  Chunk ch;
  if (d.ninst != 1) {
    ch = d.chunks[blockIdx.x];
  } else {  // an equal share of the points
    const int64_t per = (d.n + gridDim.x - 1) / gridDim.x, lo = blockIdx.x * per;
    ch.inst = 0;
    ch.begin = lo < d.n ? lo : d.n - 1;
    ch.end = lo + per < d.n ? lo + per : d.n;
  }
  const Inst& I = d.inst[ch.inst];
  const int dim = I.dim;
  double mn[3] = {INFINITY, INFINITY, INFINITY};
  double mx[3] = {-INFINITY, -INFINITY, -INFINITY};
  double ma = 0.0;
  bool bad = false;
  const double* p0 = in_xyz(d) + I.xyz_off + (ch.begin - I.pt_begin) * dim;
  if (dim == 3)
    bbox_points<3>(p0, ch.end - ch.begin, mn, mx, ma, bad);
  else
    bbox_points<2>(p0, ch.end - ch.begin, mn, mx, ma, bad);
  __shared__ double s_red[4][7];
  __shared__ int s_bad;
  if (threadIdx.x == 0) s_bad = 0;
  for (int k = 0; k < 3; ++k) {
    mn[k] = wave_min(mn[k]);
    mx[k] = wave_max(mx[k]);
  }
  ma = wave_max(ma);
  bool wb = ballot(bad) != 0;
  __syncthreads();
  const int wv = threadIdx.x >> 6;
  if (lane_id() == 0) {
    for (int k = 0; k < 3; ++k) {
      s_red[wv][k] = mn[k];
      s_red[wv][3 + k] = mx[k];
    }
    s_red[wv][6] = ma;
    if (wb) atomicOr(&s_bad, 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w)
      for (int k = 0; k < 3; ++k) {
        s_red[0][k] = fmin(s_red[0][k], s_red[w][k]);
        s_red[0][3 + k] = fmax(s_red[0][3 + k], s_red[w][3 + k]);
        s_red[0][6] = fmax(s_red[0][6], s_red[w][6]);
      }
    unsigned long long* bb =
        d.bbox + ((int64_t)ch.inst * kBoxStripes +
                  (d.ninst != 1 ? (ch.begin - I.pt_begin) / kChunk : blockIdx.x) % kBoxStripes) * 8;
    for (int k = 0; k < dim; ++k) {
      atomicMin(&bb[k], ord_d(s_red[0][k]));
      atomicMax(&bb[3 + k], ord_d(s_red[0][3 + k]));
    }
    atomicMax(&bb[6], ord_d(s_red[0][6]));
    if (s_bad) atomicOr((unsigned long long*)&bb[7], 1ULL);
  }
  if (d.ninst != 1) return;
  __shared__ int s_last;
  if (threadIdx.x == 0) {
    // the stripes' atomics before the count: both are done at device scope,
    // so it is enough that they have completed (a device-wide fence per
    // workgroup writes L2 back: 4 M points 65 us with it, 22 without).  The
    // wait orders nothing but accesses that bypass the XCD's L2, so within this
    // kernel the stripes may be written by device-scope atomics and read by
    // device-scope atomic loads only: a plain store would stay in one XCD's L2.
    // (The language gives no such order; this relies on gfx950's vmcnt, which
    // counts an atomic without a result until it is done at its scope.)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // counted in stripes first: one address takes about 10 ns per workgroup
    const unsigned G = gridDim.x, g = blockIdx.x % kStripes;
    s_last = 0;
    if (atomicAdd((unsigned long long*)&d.stat[g * kStatStride + C_BOXES], 1ull) + 1 ==
        (G - g + kStripes - 1) / kStripes)
      s_last = atomicAdd((unsigned long long*)&d.ctl[C_BOXES], 1ull) + 1 ==
               (G < (unsigned)kStripes ? G : (unsigned)kStripes);
  }
  __syncthreads();
  if (!s_last || threadIdx.x >= 64) return;
  unsigned long long bx[8];
  static_assert(kBoxStripes <= 64, "one lane per stripe");
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const unsigned long long none = k < 3 ? ~0ull : 0ull;
    bx[k] = threadIdx.x < kBoxStripes
                ? __hip_atomic_load(&d.bbox[threadIdx.x * 8 + k], __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT)
                : none;
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) bx[k] = k < 3 ? wave_min(bx[k]) : wave_max(bx[k]);
  if (threadIdx.x == 0) {
    Inst J = d.inst[0];
    unsigned long long cells, keys;
    long long lines;
    setup_instance(J, bx, cells, keys, lines);
    J.key_base = 0;
    J.line_base = 0;
    d.inst[0] = J;
    setup_totals(d, cells, keys, lines, J.err);
  }
}

// ------------------------------------------------------------ grid setup --
// Cells are cubes of width w = (eps/2)*(1+2^-20).  Two consequences:
//  * every cell is a clique: its diagonal sqrt(D)*w <= 0.87*eps, so any two
//    of its points are neighbours with a wide margin (FP64 rounding of the
//    box test and of d^2 is far below that margin);
//  * every eps-neighbour of a point lies in the 5^D cells around its cell
//    (|dx| <= eps < 2w, and the cell function is monotone, so the
//    rounding of floor(fl(fl(x-mn)*inv_w)) -- below 5*2^-53 per cell --
//    cannot move a neighbour further than the 2^-20 margin allows).
// PARTITION_SIZE r is validated as the reference does (min extent / r must
// be >= eps, main.cu:204-207, else DCLUST_E_BINWIDTH); it does not change
// the grid, whose resolution is fixed by eps (DBSCAN labels do not depend on
// the index).  Axes are limited to 2^21 cells (3-D) / 2^31 (2-D), i.e. an
// extent of about 2^20 eps; larger inputs get DCLUST_E_CAPACITY.
//
// FP32 form: distances are formed from fixed-point coordinates in units of
// w*2^-29 (29 fraction bits, wrapping every 8 cells; stencil differences
// stay below 3 cells < 2^31 units).  The FP32 squared distance D2 differs
// from the exact squared distance (same units) by at most 5*2^-24 relative
// (int->float conversion, square, two fused adds) plus the quantisation of
// the coordinates.  Pairs with |D2 - eps^2| <= band are re-decided with the
// exact FP64 predicate; band is 8 ulp = 2^-20 relative unless the bound
// above (plus the box-test slack from coordinate magnitude) requires more,
// in which case it is widened to twice the bound.
//
// Per instance this also sets the column-table base: the dense column table
// (one entry per possible column) locates a neighbour column in O(1).
__device__ void setup_instance(Inst& I, const unsigned long long (&bb)[8],
                               unsigned long long& cells, unsigned long long& keys,
                               long long& lines) {
  const int dim = I.dim;
  double mn[3] = {0, 0, 0}, mx[3] = {0, 0, 0};
  double emin = INFINITY;
  bool empty = I.pt_end <= I.pt_begin;
  // (constant indexes throughout: the arrays stay in registers)
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (k < dim && !empty) {
      mn[k] = unord_d(bb[k]);
      mx[k] = unord_d(bb[3 + k]);
    }
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (k < dim) emin = fmin(emin, mx[k] - mn[k]);
  I.maxabs = empty ? 0.0 : unord_d(bb[6]);
  if (bb[7]) {
    // DCLUST_E_PARAM: non-finite input.  The instance keeps a one-cell
    // grid (every point in cell 0) so that every kernel stays in bounds;
    // its result is discarded.
    I.err = -1;
#pragma unroll
    for (int k = 0; k < 3; ++k) mn[k] = mx[k] = 0.0;
    I.maxabs = 0.0;
  }
  if (I.r > 0) {
    double wr = emin / (double)I.r;
    if (!(wr >= I.eps) && I.err == 0 && !empty) I.err = -2;  // DCLUST_E_BINWIDTH
  }
  // coordinates so large that FP64 cannot resolve eps
  if (I.maxabs > I.eps * 0x1p40 && I.err == 0) I.err = -1;
  double w = 0.5 * I.eps * (1.0 + 0x1p-20);
  const double cap = dim == 3 ? 2097152.0 : 2147483647.0;
  for (;;) {
    // an oversized input keeps a valid (coarser) grid so that every
    // kernel stays in bounds; its result is discarded (error set)
    double inv = 1.0 / w;
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (k < dim && floor((mx[k] - mn[k]) * inv) + 1.0 > cap) ok = false;
    if (ok) break;
    if (I.err == 0) I.err = -6;  // DCLUST_E_CAPACITY
    w *= 2.0;
  }
  I.w = w;
  I.inv_w = 1.0 / w;
  cells = 1;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    I.mn[k] = k < dim ? mn[k] : 0.0;
    I.nk[k] = 1;
    if (k < dim) {
      double t = floor(cell_t(mx[k], mn[k], I.inv_w));
      I.nk[k] = (int32_t)t + 1;
      cells *= (unsigned long long)I.nk[k];
    }
  }
  const long long bx = ((long long)I.nk[0] + 1) / 2, by = ((long long)I.nk[1] + 1) / 2;
  I.cstride = dim == 3 ? by + 1 : 1;
  lines = bx * I.cstride;
  I.nlines = lines;
  I.nzl = dim == 3 ? (long long)I.nk[2] << 2 : (long long)I.nk[1] << 1;
  I.inv_nzl = 1.0 / (double)I.nzl;
  keys = (unsigned long long)lines * (unsigned long long)I.nzl;
  // FP32 guard band (units of w * 2^-29)
  const double gs = I.inv_w * 0x1p29;
  const double es = I.eps * gs;
  const double e2 = es * es;
  const double u = 0x1p-24;
  double bound = 5.0 * u * (1.0 + 4.0 * u);
  bound += 2.0 * 1.7320508075688772 * 2.5 / es + 6.25 * 3.0 / e2;  // quantisation
  bound += 8.0 * 0x1p-52 * (I.maxabs / I.eps + 1.0);             // box slack
  double band = 0x1p-20;
  if (bound > 0.5 * band) band = 2.0 * bound;
  float fin = (float)(e2 * (1.0 - band));
  if ((double)fin > e2 * (1.0 - band)) fin = __int_as_float(__float_as_int(fin) - 1);
  float fout = (float)(e2 * (1.0 + band));
  if ((double)fout < e2 * (1.0 + band)) fout = __int_as_float(__float_as_int(fout) + 1);
  I.d2_in = fin;
  I.d2_out = fout;
  I.d2_mid = (float)e2;
  // The FP64 predicate compares squares: where eps^2 rounds to infinity or has
  // lost bits to underflow (0 below 1.6e-162, where only the box test is left),
  // the fixed-point distances say nothing about it.  Then every pair is inside
  // the band, so that nothing is joined or left out by them.
  if (!(I.eps2 >= 0x1p-1000 && I.eps2 <= 0x1.fffffffffffffp1023)) {
    I.d2_in = -1.f;
    I.d2_out = INFINITY;
  }
}

// The call's totals: key width, columns, errors.
__device__ void setup_totals(const Dev& d, unsigned long long cells, unsigned long long keys,
                             long long lines, int err) {
  d.ctl[C_ERR] = err != 0;
  d.ctl[C_NLINES] = lines;
  if (cells > kMaxKeySpace || keys == ~0ull) {
    // the keys would not fit the sort: the whole call fails (instances of a
    // batch share one key space), and every later kernel returns at once
    d.ctl[C_KEYOVF] = 1;
    d.ctl[C_ERR] = 1;
    d.ctl[C_ABANDON] = 1;
    d.ctl[C_KEYBITS] = 8;
  } else {
    d.ctl[C_KEYBITS] = key_bits_for(keys);
    if (err && d.err_stops) d.ctl[C_ABANDON] = 1;
  }
}

// Grid set-up of a batch, one workgroup: per instance, then the scans of key
// and column bases over the instances.
__global__ __launch_bounds__(1024) void k_grid_setup(Dev d) {
  __shared__ unsigned long long s_scan[1024];
  __shared__ unsigned long long s_scanc[1024];
  __shared__ long long s_scanl[1024];
  __shared__ unsigned long long s_carry, s_carryc;
  __shared__ long long s_carryl;
  __shared__ int s_err;
  if (threadIdx.x == 0) {
    s_carry = 0;
    s_carryc = 0;
    s_carryl = 0;
    s_err = 0;
  }
  __syncthreads();
  for (int base = 0; base < d.ninst; base += blockDim.x) {
    const int i = base + threadIdx.x;
    unsigned long long cells = 0;  // at most 2^63 (3 axes of at most 2^21 cells)
    unsigned long long keys = 0;   // at most 2^63 + 2^43
    long long lines = 0;
    if (i < d.ninst) {
      Inst I = d.inst[i];
      unsigned long long bb[8];
      {
        const unsigned long long* bs = d.bbox + (int64_t)i * kBoxStripes * 8;
#pragma unroll
        for (int k = 0; k < 8; ++k) bb[k] = k < 3 ? ~0ull : 0ull;
        // (as many stripes as the instance has chunks: with all 32 this read
        // was most of the 33 us of 256 instances, 45 of 400 tiny ones)
        const int64_t chunks = (I.pt_end - I.pt_begin + kChunk - 1) / kChunk;
        const int ns = chunks < kBoxStripes ? (int)chunks : kBoxStripes;
#pragma unroll 4
        for (int st = 0; st < ns; ++st)
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const unsigned long long v = bs[st * 8 + k];
            bb[k] = k < 3 ? (v < bb[k] ? v : bb[k]) : (v > bb[k] ? v : bb[k]);
          }
      }
      setup_instance(I, bb, cells, keys, lines);
      d.inst[i] = I;
      if (I.err) atomicOr(&s_err, 1);
    }
    s_scan[threadIdx.x] = keys;
    s_scanc[threadIdx.x] = cells;
    s_scanl[threadIdx.x] = lines;
    __syncthreads();
    // inclusive Hillis-Steele scans over the block
    // (the key-space sums saturate: a total beyond 2^63 fails the call below)
    for (int o = 1; o < (int)blockDim.x; o <<= 1) {
      unsigned long long v = threadIdx.x >= (unsigned)o ? s_scan[threadIdx.x - o] : 0;
      unsigned long long vc = threadIdx.x >= (unsigned)o ? s_scanc[threadIdx.x - o] : 0;
      long long vl = threadIdx.x >= (unsigned)o ? s_scanl[threadIdx.x - o] : 0;
      __syncthreads();
      s_scan[threadIdx.x] = sat_add(s_scan[threadIdx.x], v);
      s_scanc[threadIdx.x] = sat_add(s_scanc[threadIdx.x], vc);
      s_scanl[threadIdx.x] += vl;
      __syncthreads();
    }
    if (i < d.ninst) {
      d.inst[i].key_base = (int64_t)(sat_add(s_carry, s_scan[threadIdx.x]) - keys);
      d.inst[i].line_base = s_carryl + s_scanl[threadIdx.x] - lines;
    }
    __syncthreads();
    if (threadIdx.x == blockDim.x - 1) {
      s_carry = sat_add(s_carry, s_scan[threadIdx.x]);
      s_carryc = sat_add(s_carryc, s_scanc[threadIdx.x]);
      s_carryl += s_scanl[threadIdx.x];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) setup_totals(d, s_carryc, s_carry, s_carryl, s_err);
}

// --------------------------------------------------------------- cellkey --
// Forms of the sort keys.  Up to 32 bits: 32-bit keys beside 32-bit ids.  Up
// to 36 bits, ids of 28 bits: the key's lower four bits ride in the id's
// upper four (only the first pass looks at them, so the later passes count
// from the keys alone), and a pass still moves 8 bytes a point where a 64-bit
// key moves 12.
// Above that 64-bit keys; the buffers are viewed as any of them.  The host
// picks the form from the key bits it knows (the grid set-up's, or the largest
// so far for a captured graph: a replay whose keys are wider is abandoned by
// k_csr_count, so a truncated key is never used).
template <int KF>
using SortKey = typename std::conditional<KF == 64, uint64_t, uint32_t>::type;
template <int KF>
__device__ __forceinline__ SortKey<KF>* key_buf(const Dev& d, int b) {
  return reinterpret_cast<SortKey<KF>*>(d.key[b]);
}
constexpr uint32_t kIdMask = (1u << 28) - 1;  // of the 36-bit form
static_assert(kMaxCells <= (int64_t)kIdMask + 1, "every id fits the 36-bit form");
// the whole key of a sort entry
template <int KF>
__device__ __forceinline__ uint64_t entry_key(SortKey<KF> k, int32_t v) {
  return KF == 36 ? (uint64_t)k << 4 | (uint32_t)v >> 28 : (uint64_t)k;
}
template <int KF>
__device__ __forceinline__ uint32_t entry_digit(SortKey<KF> k, int32_t v, int shift,
                                                uint32_t mask) {
  return (uint32_t)(entry_key<KF>(k, v) >> shift) & mask;
}

__device__ __forceinline__ int32_t cell_index(double x, const Inst& I, int k) {
  double t = floor(cell_t(x, I.mn[k], I.inv_w));
  int32_t c = (t >= 0.0) ? (int32_t)fmin(t, (double)(I.nk[k] - 1)) : 0;
  return c;
}

// ------------------------------------------------------------ radix sort --
// LSD radix sort by digits of at most 9 bits, two launches a pass.  Every
// workgroup owns one contiguous range of the entries, so the digit counts are
// few ([workgroups][512], added up in groups as they are made), and its tiles
// write one after the other to neighbouring places, whose partial lines its L2
// joins.  Buffer parity: the number of passes.
//
// Bound by the bytes it moves, in runs of a few dozen bytes, at the larger sizes
// and by launches and each workgroup's chain of barriers at the smaller.  Per
// pass, 32 M points of 33 bits: count 29 us, scatter 147 to 177 (four passes);
// 4 M of 32 bits 6 + 26 (four).  Before (8-bit digits, one tile of
// 2048 keys a workgroup, counts [256][n / 2048]) 88 + 43 + 233 (five passes of
// 64-bit keys) and 15 + 6 + 22.  Interleaving the tiles of neighbouring
// workgroups instead (one tile each) took longer, 225 us a scatter.
constexpr int RS_T = 512;
constexpr int RS_D = 1 << kDigitBits;  // a thread per digit
static_assert(RS_T == RS_D, "one digit per thread");

// The fewest passes of at most 9 bits, of widths as equal as they can be; the
// wider digits come last, where the entries already have long runs.
__device__ __forceinline__ int sort_passes(const Dev& d) {
  return ((int)d.ctl[C_KEYBITS] + kDigitBits - 1) / kDigitBits;
}
struct SortDigit {
  int shift, width;
};
__device__ __forceinline__ SortDigit sort_digit(const Dev& d, int pass, int passes) {
  const int bits = (int)d.ctl[C_KEYBITS], w = bits / passes, first_wide = passes - bits % passes;
  SortDigit g;
  g.shift = pass * w + (pass > first_wide ? pass - first_wide : 0);
  g.width = w + (pass >= first_wide);
  return g;
}

// Entries of workgroup b of nblk.
__device__ __forceinline__ void sort_range(int64_t n, int b, int nblk, int64_t& lo, int64_t& hi) {
  const int64_t per = ((n + nblk - 1) / nblk + 63) & ~63LL;
  lo = b * per < n ? b * per : n;
  hi = lo + per < n ? lo + per : n;
}

// Workgroups of one XCD own neighbouring ranges.
__device__ __forceinline__ int sort_block(int nblk) {
  const int b = blockIdx.x;
  return nblk % 8 == 0 ? (b & 7) * (nblk / 8) + (b >> 3) : b;
}

// lanes of the wave with the same digit among the `valid` ones
__device__ __forceinline__ unsigned long long match_digit(uint32_t dg, int width, bool valid) {
  unsigned long long peers = ballot(valid);
#pragma unroll
  for (int b = 0; b < kDigitBits; ++b) {
    if (b < width) {
      const bool bit = (dg >> b) & 1;
      const unsigned long long m = ballot(bit);
      peers &= bit ? m : ~m;
    }
  }
  return peers;
}

// Digit counts of each workgroup's range.  The lanes of a wave count in
// kHistCopies copies in turn: the upper digits of clustered points are few, and
// their atomics on one address would queue (32 M points, one copy: 28 us for
// the lower digits and 130 for the upper).
constexpr int kHistCopies = 8;
__device__ __forceinline__ void hist_clear(uint32_t (&h)[RS_D * kHistCopies]) {
#pragma unroll
  for (int c = 0; c < kHistCopies; ++c) h[c * RS_T + threadIdx.x] = 0;
  __syncthreads();
}
// (also to the counts of the workgroup's group, which start at zero)
__device__ __forceinline__ void hist_store(const Dev& d, uint32_t (&h)[RS_D * kHistCopies],
                                           int pass, int b) {
  __syncthreads();
  uint32_t sum = 0;
#pragma unroll
  for (int c = 0; c < kHistCopies; ++c) sum += h[threadIdx.x * kHistCopies + c];
  d.hist[(int64_t)b * RS_D + threadIdx.x] = sum;
  if (sum)
    atomicAdd(&d.dgrp[(pass * kSortGroups + b / kSortGroup) * RS_D + threadIdx.x], sum);
}

template <int D, int KF, int T, typename F>
__device__ __forceinline__ void cellkey_points(const Dev& d, const Inst& I, int64_t begin,
                                               int64_t end, const F& count) {
  const double* p0 = in_xyz(d) + I.xyz_off + (begin - I.pt_begin) * D;
  const int64_t np = end - begin;
  for (int64_t i0 = threadIdx.x; i0 < np; i0 += kChunkU * T) {
    double v[kChunkU][D];
#pragma unroll
    for (int u = 0; u < kChunkU; ++u) {
      const int64_t i = i0 + u * T < np ? i0 + u * T : np - 1;
#pragma unroll
      for (int k = 0; k < D; ++k) v[u][k] = p0[i * D + k];
    }
#pragma unroll
    for (int u = 0; u < kChunkU; ++u) {
      const int64_t i = i0 + u * T;
      if (i < np) {
        const int32_t cx = cell_index(v[u][0], I, 0), cl = cell_index(v[u][D - 1], I, D - 1);
        uint64_t lin;  // (unsigned: an instance may have a few keys above 2^63)
        if (D == 3) {
          const int32_t cy = cell_index(v[u][1], I, 1);
          lin = (uint64_t)((cx >> 1) * I.cstride + (cy >> 1)) * (uint64_t)I.nzl +
                (uint64_t)(cl * 4LL + (cx & 1) * 2 + (cy & 1));
        } else {
          lin = (uint64_t)((cx >> 1) * I.nzl + cl * 2LL + (cx & 1));
        }
        const uint64_t key = (uint64_t)I.key_base + lin;
        key_buf<KF>(d, 0)[begin + i] = (SortKey<KF>)(KF == 36 ? key >> 4 : key);
        // (the first pass knows the ids, which are the positions)
        if (KF == 36)
          d.val[0][begin + i] = (int32_t)((uint32_t)(begin + i) | (uint32_t)key << 28);
        count((uint32_t)key);
      }
    }
  }
}

template <int KF, int T, typename F>
__device__ __forceinline__ void cellkeys(const Dev& d, int inst, int64_t begin, int64_t end,
                                         const F& count) {
  // a copy: the key stores could alias the instance table as far as the
  // compiler knows, which would reload its fields after every store
  const Inst I = d.inst[inst];
  if (I.dim == 3)
    cellkey_points<3, KF, T>(d, I, begin, end, count);
  else
    cellkey_points<2, KF, T>(d, I, begin, end, count);
}

// Keys of a batch, a chunk of one instance per workgroup.
template <int KF>
__global__ __launch_bounds__(256) void k_cellkey(Dev d) {
  const Chunk ch = d.chunks[blockIdx.x];
  cellkeys<KF, 256>(d, ch.inst, ch.begin, ch.end, [](uint32_t) {});
}

// Keys of a single instance, and the first pass's digit counts: a workgroup
// takes its range of the sort.
template <int KF>
__global__ __launch_bounds__(RS_T) void k_cellkey_hist(Dev d, int nblk) {
  const uint32_t mask = (1u << sort_digit(d, 0, sort_passes(d)).width) - 1;
  __shared__ uint32_t h[RS_D * kHistCopies];
  hist_clear(h);
  const int b = sort_block(nblk);
  int64_t lo, hi;
  sort_range(d.n, b, nblk, lo, hi);
  const int copy = threadIdx.x & (kHistCopies - 1);
  cellkeys<KF, RS_T>(d, 0, lo, hi,
                     [&](uint32_t k) { atomicAdd(&h[(k & mask) * kHistCopies + copy], 1u); });
  hist_store(d, h, 0, b);
}

template <int KF>
__global__ __launch_bounds__(RS_T) void k_rs_hist(Dev d, int pass, int nblk) {
  const int np = sort_passes(d);
  if (pass >= np) return;
  const SortDigit P = sort_digit(d, pass, np);
  const SortKey<KF>* kin = key_buf<KF>(d, pass & 1);
  const int32_t* vin = d.val[pass & 1];
  const int shift = P.shift;
  const uint32_t mask = (1u << P.width) - 1;
  const bool ids = KF == 36 && shift < 4;
  __shared__ uint32_t h[RS_D * kHistCopies];
  hist_clear(h);
  const int copy = threadIdx.x & (kHistCopies - 1);
  const int b = sort_block(nblk);
  int64_t lo, hi;
  sort_range(d.n, b, nblk, lo, hi);
  constexpr int U = 8;
  for (int64_t i0 = lo + threadIdx.x; i0 < hi; i0 += U * RS_T) {
    SortKey<KF> k[U];
    int32_t v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t i = i0 + u * RS_T < hi ? i0 + u * RS_T : lo;
      k[u] = kin[i];
      v[u] = ids ? vin[i] : 0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i0 + u * RS_T < hi) 
        atomicAdd(&h[entry_digit<KF>(k[u], v[u], shift, mask) * kHistCopies + copy], 1u);
  }
  hist_store(d, h, pass, b);
}

// Exclusive scan over the workgroup's RS_T threads (a barrier inside; s_w is
// free again after the caller's next barrier).
__device__ __forceinline__ uint32_t sort_scan(uint32_t v, uint32_t (&s_w)[RS_T / 64]) {
  const uint32_t inc = wave_incl_scan(v);
  const int wv = threadIdx.x >> 6;
  if (lane_id() == 63) s_w[wv] = inc;
  __syncthreads();
  uint32_t e = inc - v;
#pragma unroll
  for (int w = 0; w < RS_T / 64; ++w) e += w < wv ? s_w[w] : 0u;
  return e;
}

// Stable scatter, tile by tile of RS_T * NI entries.  Each wave owns a
// contiguous run of 64 * NI entries of the tile and ranks them round by round
// (64 consecutive entries per round, lanes in order) against counters of its
// own in LDS, with no barrier between rounds (a wave's LDS accesses complete
// in order); one barrier later each digit's counts of the waves before it and
// the tile's local starts turn the ranks into positions, so equal digits keep
// their order.  The tile is staged in LDS in local digit order and written
// out in runs per digit.  The counts of the workgroups before come from the
// groups and from the rows of the own group, at most 48 loads a thread (a scan
// of all rows in a launch of its own took 5 us a pass).
template <int KF, int NI>
__global__ __launch_bounds__(RS_T, 4) void k_rs_scatter(Dev d, int pass, int nblk) {
  using KT = SortKey<KF>;
  constexpr int TILE = RS_T * NI, NW = RS_T / 64;
  const int np = sort_passes(d);
  if (pass >= np) return;
  const SortDigit P = sort_digit(d, pass, np);
  const KT* kin = key_buf<KF>(d, pass & 1);
  const int32_t* vin = d.val[pass & 1];
  KT* kout = key_buf<KF>(d, (pass & 1) ^ 1);
  int32_t* vout = d.val[(pass & 1) ^ 1];
  const bool ids = KF != 36 && pass == 0;  // the ids are the positions
  const int shift = P.shift;
  const uint32_t mask = (1u << P.width) - 1;
  __shared__ KT s_k[TILE];
  __shared__ int32_t s_v[TILE];
  __shared__ uint32_t s_gd[RS_D];
  __shared__ uint16_t s_wc[NW][RS_D];
  __shared__ uint32_t s_w0[NW], s_w1[NW];
  const int tid = threadIdx.x, wv = tid >> 6;
  const int b = sort_block(nblk);
  int64_t lo, hi;
  sort_range(d.n, b, nblk, lo, hi);
  // where this workgroup's next entry of digit tid goes
  uint32_t pre = 0, tot = 0;
  const int grp = b / kSortGroup;
#pragma unroll
  for (int q = 0; q < kSortGroups; ++q) {
    const uint32_t c = d.dgrp[(pass * kSortGroups + q) * RS_D + tid];
    tot += c;
    pre += q < grp ? c : 0u;
  }
  for (int q0 = grp * kSortGroup; q0 < b; q0 += 16) {
    uint32_t c[16];  // (rows past the own one are read, not counted: one trip)
#pragma unroll
    for (int u = 0; u < 16; ++u) c[u] = d.hist[(int64_t)(q0 + u < b ? q0 + u : b) * RS_D + tid];
#pragma unroll
    for (int u = 0; u < 16; ++u) pre += q0 + u < b ? c[u] : 0u;
  }
  uint32_t goff = sort_scan(tot, s_w1) + pre;
  // (32-bit places from here on: ids are 32-bit too)
  kin += lo;
  vin += lo;
  const uint32_t len = (uint32_t)(hi - lo);
  KT kr[NI];
  int32_t vr[NI];
  auto load = [&](uint32_t t0) {
    const uint32_t w0 = t0 + wv * (64 * NI) + lane_id();
#pragma unroll
    for (int r = 0; r < NI; ++r) {
      const uint32_t i = w0 + r * 64 < len ? w0 + r * 64 : 0u;
      kr[r] = kin[i];
      vr[r] = ids ? (int32_t)(lo + i) : vin[i];
    }
  };
  if (len > 0) load(0);
  for (uint32_t t0 = 0; t0 < len; t0 += TILE) {
    const uint32_t w0 = t0 + wv * (64 * NI) + lane_id();
#pragma unroll
    for (int q = 0; q < RS_D / 64; ++q) s_wc[wv][q * 64 + lane_id()] = 0;
    uint32_t lr[NI / 2];  // (two 16-bit ranks a register)
#pragma unroll
    for (int r = 0; r < NI; ++r) {
      const bool v = w0 + r * 64 < len;
      const uint32_t dg = entry_digit<KF>(kr[r], vr[r], shift, mask);
      const unsigned long long peers = match_digit(dg, P.width, v);
      const uint32_t rank = mbcnt(peers);
      const uint32_t base = s_wc[wv][dg];
      if (v && rank == 0) s_wc[wv][dg] = (uint16_t)(base + (uint32_t)__popcll(peers));
      lr[r / 2] = r & 1 ? lr[r / 2] | (base + rank) << 16 : base + rank;
    }
    __syncthreads();
    uint32_t cw[NW], c = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      cw[w] = s_wc[w][tid];
      c += cw[w];
    }
    uint32_t lst = sort_scan(c, s_w0);
    s_gd[tid] = goff - lst;
    goff += c;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      s_wc[w][tid] = (uint16_t)lst;
      lst += cw[w];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NI; ++r) {
      if (w0 + r * 64 < len) {
        const uint32_t lp = s_wc[wv][entry_digit<KF>(kr[r], vr[r], shift, mask)] +
                            (r & 1 ? lr[r / 2] >> 16 : lr[r / 2] & 0xffffu);
        s_k[lp] = kr[r];
        s_v[lp] = vr[r];
      }
    }
    __syncthreads();
    // the next tile's entries travel while this one is written out
    if (t0 + TILE < len) load(t0 + TILE);
    // every slot is read (past the tile's end the reads are unused), the
    // stores are guarded
    const uint32_t tn = len - t0 < TILE ? len - t0 : TILE;
#pragma unroll 4
    for (int r = 0; r < NI; ++r) {
      const uint32_t l = r * RS_T + tid;
      const KT k = s_k[l];
      const int32_t v = s_v[l];
      const uint32_t g = s_gd[entry_digit<KF>(k, v, shift, mask)] + l;
      if (l < tn) {
        kout[g] = k;
        vout[g] = v;
      }
    }
  }
}

// ------------------------------------------------------- CSR compaction --
// Flag = sorted key differs from its predecessor.  Pass 1 counts flags per
// 2048-key tile with ballot/popcount; a single block scans the tile counts;
// pass 2 ranks flags inside the tile with mbcnt and writes the cell ranges.
constexpr int CS_T = 256;
constexpr int CS_I = 8;
constexpr int CS_TILE = CS_T * CS_I;

// Sorted keys i and i - 1 of each of a thread's rounds, loaded before any
// is used (indices clamped into the array) so that the loads are in flight
// together; key i starts a cell when i < n and it differs from key i - 1.
template <int KF, int NI>
__device__ __forceinline__ void load_key_pairs(const Dev& d, int64_t t0, uint64_t (&k)[NI],
                                               uint64_t (&kp)[NI]) {
  const int par = sort_passes(d) & 1;
  const SortKey<KF>* key = key_buf<KF>(d, par);
  const int32_t* val = d.val[par];
#pragma unroll
  for (int r = 0; r < NI; ++r) {
    const int64_t i = t0 + r * CS_T + threadIdx.x;
    const int64_t ic = i < d.n ? i : 0, ip = ic > 0 ? ic - 1 : 0;
    k[r] = entry_key<KF>(key[ic], KF == 36 ? val[ic] : 0);
    kp[r] = entry_key<KF>(key[ip], KF == 36 ? val[ip] : 0);
  }
}

// (also, in a captured run, whose radix passes and column table are fixed: a
// key wider than the passes cover leaves the keys unsorted, and more columns
// than the table has would be searched for slowly, so the run is abandoned:
// every later kernel returns at once and the host runs the call again;
// counting unsorted keys here is harmless)
template <int KF>
__global__ __launch_bounds__(CS_T) void k_csr_count(Dev d, int bits) {
  if (blockIdx.x == 0 && threadIdx.x == 0 &&
      (d.ctl[C_KEYBITS] > bits ||
       (d.line_cap > 0 && d.line_cap < kMaxLineTable && d.ctl[C_NLINES] > d.line_cap)))
    d.ctl[C_ABANDON] = 1;
  if (abandoned(d)) return;
  // the column table, cleared by the whole grid (which is larger than the
  // tiles need when there are few)
  const long long P = d.ctl[C_NLINES];
  if (P <= d.line_cap)
    for (int64_t i = (int64_t)blockIdx.x * CS_T + threadIdx.x; i < P;
         i += (int64_t)gridDim.x * CS_T)
      d.lines[i] = make_int2(-1, -1);
  const int64_t t0 = (int64_t)blockIdx.x * CS_TILE;
  if (t0 >= d.n) return;
  uint64_t kr[CS_I], kp[CS_I];
  load_key_pairs<KF, CS_I>(d, t0, kr, kp);
  int c = 0;
#pragma unroll
  for (int r = 0; r < CS_I; ++r) {
    const int64_t i = t0 + r * CS_T + threadIdx.x;
    c += __popcll(ballot(i < d.n && (i == 0 || kr[r] != kp[r])));
  }
  __shared__ int s[4];
  if (lane_id() == 0) s[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) d.scan_tmp[blockIdx.x] = s[0] + s[1] + s[2] + s[3];
}

// exclusive scan of nb int64 values in place by one block
__global__ __launch_bounds__(1024) void k_scan_top(int64_t* v, int nb) {
  __shared__ int64_t s[1024];
  const int per = (nb + 1023) / 1024;
  const int b0 = threadIdx.x * per;
  int64_t sum = 0;
  for (int j = 0; j < per; ++j)
    if (b0 + j < nb) sum += v[b0 + j];
  s[threadIdx.x] = sum;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    int64_t u = threadIdx.x >= (unsigned)o ? s[threadIdx.x - o] : 0;
    __syncthreads();
    s[threadIdx.x] += u;
    __syncthreads();
  }
  int64_t run = s[threadIdx.x] - sum;
  for (int j = 0; j < per; ++j)
    if (b0 + j < nb) {
      int64_t x = v[b0 + j];
      v[b0 + j] = run;
      run += x;
    }
}

// instance owning a key: last i with key_base <= key
__device__ __forceinline__ int32_t inst_of_key(const Dev& d, uint64_t key, int lo, int hi) {
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if ((uint64_t)d.inst[mid].key_base <= key) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Column (within the instance) and place in the column of a key, decoded once
// per cell.  By the stored reciprocal: an instance has fewer than 2^42 columns,
// so the rounded quotient is off by less than 2^-9 and its floor by one at
// most.  Unsigned up to the remainder: 2^21 cells along each of three axes have
// keys up to 2^63 + 2^43.  (With integer divisions, unrolled and 64-bit ones among them,
// k_csr_write took 13 us on 100 k points, 37 on 4 M, 127 on 32 M; 12, 33, 115 now.)
__device__ __forceinline__ void split_key(const Inst& I, uint64_t key, int64_t& col,
                                          uint32_t& zl) {
  const uint64_t rel = key - (uint64_t)I.key_base;
  int64_t q = (int64_t)((double)rel * I.inv_nzl);
  int64_t r = (int64_t)(rel - (uint64_t)q * (uint64_t)I.nzl);
  if (r < 0) {
    --q;
    r += I.nzl;
  } else if (r >= I.nzl) {
    ++q;
    r -= I.nzl;
  }
  col = q;
  zl = (uint32_t)r;
}

// Sum of the block counts v[0..b) (`scanned` false: they are counts; true:
// already their exclusive prefix), by the whole workgroup of 256.  Where
// there are at most kScanInline blocks every block sums its own prefix, which
// takes fewer microseconds than a launch that scans them all.
constexpr int kScanInline = 2048;
__device__ __forceinline__ int64_t block_prefix(const int64_t* v, int b, bool scanned) {
  __shared__ int64_t s_part[4];
  if (scanned) return v[b];
  int64_t sum = 0;
  for (int i = threadIdx.x; i < b; i += 256) sum += v[i];
  sum = wave_sum(sum);
  if (lane_id() == 0) s_part[threadIdx.x >> 6] = sum;
  __syncthreads();
  sum = s_part[0] + s_part[1] + s_part[2] + s_part[3];
  __syncthreads();
  return sum;
}

// Also fills the column table: a cell whose predecessor's key lies below its
// column's first key starts the column and ends the one before.
template <int KF>
__global__ __launch_bounds__(CS_T) void k_csr_write(Dev d, bool scanned) {
  if (abandoned(d)) return;
  const bool table = d.ctl[C_NLINES] <= d.line_cap;
  const int64_t t0 = (int64_t)blockIdx.x * CS_TILE;
  __shared__ int s_w[CS_I][4];
  const int wv = threadIdx.x >> 6;
  uint64_t kr[CS_I], kp[CS_I];
  load_key_pairs<KF, CS_I>(d, t0, kr, kp);
  // every round's instance, column and place, from the
  // instance table before the first store (the stores could alias it as far
  // as the compiler knows, which would hold each round's reads behind the
  // previous round's stores)
  // (the tile's keys are sorted: they lie in the instances of its first and
  // last key, in a batch mostly one; 7 M points in 256 instances 113 us with a
  // search per cell, 71 now)
  int i_lo = 0, i_hi = 0;
  if (d.ninst != 1) {
    const int64_t last = t0 + CS_TILE < d.n ? t0 + CS_TILE - 1 : d.n - 1;
    const int par = sort_passes(d) & 1;
    const SortKey<KF>* key = key_buf<KF>(d, par);
    const int32_t* val = d.val[par];
    i_lo = inst_of_key(d, entry_key<KF>(key[t0], KF == 36 ? val[t0] : 0), 0, d.ninst - 1);
    i_hi = inst_of_key(d, entry_key<KF>(key[last], KF == 36 ? val[last] : 0), i_lo, d.ninst - 1);
  }
  int32_t ir[CS_I];
  uint32_t zr[CS_I], cr[CS_I];
#pragma unroll
  for (int r = 0; r < CS_I; ++r) {
    ir[r] = 0;
    zr[r] = 0;
    cr[r] = 0;
    const int64_t i = t0 + r * CS_T + threadIdx.x;
    if (i < d.n && (i == 0 || kr[r] != kp[r])) {
      ir[r] = inst_of_key(d, kr[r], i_lo, i_hi);
      const Inst& I = d.inst[ir[r]];
      int64_t col;
      split_key(I, kr[r], col, zr[r]);
      cr[r] = (uint32_t)(I.line_base + col);
    }
  }
  // flags of every round and wave first: one barrier, not three a round
#pragma unroll
  for (int r = 0; r < CS_I; ++r) {
    const int64_t i = t0 + r * CS_T + threadIdx.x;
    const unsigned long long m = ballot(i < d.n && (i == 0 || kr[r] != kp[r]));
    if (lane_id() == 0) s_w[r][wv] = __popcll(m);
  }
  int64_t run = block_prefix(d.scan_tmp, blockIdx.x, scanned);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < CS_I; ++r) {
    int64_t i = t0 + r * CS_T + threadIdx.x;
    bool inr = i < d.n;
    const uint64_t k = kr[r];
    const bool f = inr && (i == 0 || k != kp[r]);
    int64_t pre = run;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      pre += w < wv ? s_w[r][w] : 0;
      run += s_w[r][w];
    }
    int64_t cid = pre + mbcnt(ballot(f)) + (f ? 1 : 0) - 1;  // inclusive - 1
    if (inr) {
      d.cell_of[i] = (int32_t)cid;
      if (f) {
        d.cell_start[cid] = (int32_t)i;
        d.cell_key[cid] = k;
        d.cell_inst[cid] = ir[r];
        d.cell_col[cid] = cr[r];
        d.cell_zl[cid] = zr[r];
        if (table && (i == 0 || kp[r] < k - zr[r])) {
          d.lines[cr[r]].x = (int32_t)cid;
          if (i > 0) {
            // (the previous key's instance: this one, or one before it)
            const int32_t pi = kp[r] >= (uint64_t)d.inst[ir[r]].key_base
                                   ? ir[r]
                                   : inst_of_key(d, kp[r], 0, ir[r] - 1);
            const Inst& I = d.inst[pi];
            int64_t col;
            uint32_t zl;
            split_key(I, kp[r], col, zl);
            d.lines[I.line_base + col].y = (int32_t)cid;
          }
        }
      }
      if (i == d.n - 1) {
        // (the last point's cell started in this tile or before)
        if (table) {
          const Inst& I = d.inst[inst_of_key(d, k, i_lo, i_hi)];
          int64_t col;
          uint32_t zl;
          split_key(I, k, col, zl);
          d.lines[I.line_base + col].y = (int32_t)cid + 1;
        }
        d.cell_start[cid + 1] = (int32_t)d.n;
        d.ctl[C_NCELL] = cid + 1;
      }
    }
  }
}

// ---------------------------------------------------------------- gather --
// One point: its whole row is loaded before anything is stored (a store
// could alias the row as far as the compiler knows, which would otherwise
// hold each coordinate's random-access load until the previous store).
template <int D>
__device__ __forceinline__ void gather_point(const Dev& d, const Inst& I, const double* xyz,
                                             int64_t i, int32_t src) {
  const int64_t off = I.xyz_off + ((int64_t)src - I.pt_begin) * D;
  const double* p = xyz + off;
  double x[D], mn[D];
#pragma unroll
  for (int k = 0; k < D; ++k) {
    x[k] = p[k];
    mn[k] = I.mn[k];
  }
  const double inv_w = I.inv_w;
  if (!d.X) d.xrow[i] = p;  // the FP32 form's way back to FP64 rows
#pragma unroll
  for (int k = 0; k < D; ++k) {
    if (d.X) d.X[3 * i + k] = x[k];  // the FP64 form's sorted copy
    const double t = cell_t(x[k], mn[k], inv_w);  // same rounding as the key
    const double f = floor(t * 0x1p29);           // exact scaling by 2^29
    d.G[3 * i + k] = (uint32_t)(unsigned long long)(long long)f;  // wraps mod 8 cells
  }
  d.orig[i] = src;
}

// Also the run's state: cluster flags (none), and per expansion wave (`waves`
// is 0 without seed lists) its pair count and the start of its seeding
// segment of the cells.
__global__ __launch_bounds__(256) void k_gather(Dev d, int64_t waves, uint32_t id_mask) {
  if (abandoned(d)) return;
  const int64_t nf = (d.n + 63) / 64, C = d.ctl[C_NCELL];
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nf || i < waves;
       i += (int64_t)gridDim.x * blockDim.x) {
    if (i < nf) d.flag[i] = 0ull;
    if (i < waves) {
      d.pair_cnt[i] = 0;
      d.seg_pos[i] = C * i / waves;
    }
  }
  const int32_t* vsrc = d.val[sort_passes(d) & 1];
  const double* xyz = in_xyz(d);
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < d.n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t src = (int32_t)((uint32_t)vsrc[i] & id_mask);
    const Inst& I = *inst_of_cell(d, d.ninst == 1 ? 0 : d.cell_of[i]);
    if (I.dim == 3)
      gather_point<3>(d, I, xyz, i, src);
    else
      gather_point<2>(d, I, xyz, i, src);
  }
}

// ------------------------------------------------------------------ rows --
// Three lower bounds lo[j] = first index in [lo[j], hi[j]) with a[i] >= v[j],
// in lockstep (the loads of the three searches overlap), a quarter of the
// range per step: a chain of loads half as long as by halves, which is what
// the few columns left to k_rows_global take (22 us with halves, 18 now, on
// calls of 262 k to 1.5 M points).
template <typename T>
__device__ __forceinline__ void lower_bound3(const T* a, int32_t (&lo)[3], int32_t (&hi)[3],
                                             const T (&v)[3]) {
  const auto cut = [](int32_t l, int32_t h, int i) {  // pivot i of 1..3, in [l, h)
    return l + (int32_t)(((uint64_t)(uint32_t)(h - l) * (uint32_t)i) >> 2);
  };
  for (;;) {
    T km[3][3];
    bool any = false;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
      for (int i = 0; i < 3; ++i)
        km[j][i] = lo[j] < hi[j] ? a[cut(lo[j], hi[j], i + 1)] : (T)0;
      any |= lo[j] < hi[j];
    }
    if (!any) return;
#pragma unroll
    for (int j = 0; j < 3; ++j)
      if (lo[j] < hi[j]) {
        const int32_t l = lo[j], h = hi[j];
        const int c = (km[j][0] < v[j]) + (km[j][1] < v[j]) + (km[j][2] < v[j]);
        if (c > 0) lo[j] = cut(l, h, c) + 1;
        if (c < 3) hi[j] = cut(l, h, c + 1);
      }
  }
}

// Rows of the cells.  One wavefront per (tile of 64 consecutive cells, group
// g): 3-D group g holds the three columns with block offset g - 1 along axis
// 0 (consecutive columns); 2-D has one group (g = 0), its three columns
// being consecutive too.  The tile's cells lie in a few consecutive columns
// (cells are sorted, so the first and last lanes bound them), and so do
// their neighbour columns: the column table gives the range of cells those
// hold, and the wave copies the cells' sort keys, relative to the span's
// first column, into LDS with coalesced loads, padded with ~0 to a larger
// power of two and four slots more.  A window then starts at the first key >=
// its own first key, found by a branchless binary search of a depth uniform
// over the wave, and its slot bits come from the keys that follow (four per
// step).  4 M 3-D points: 205 + 57 us with k_rows_global, where 25 lines per
// cell took 274 + 28 (and 320 MB of rows instead of 240).  A tile whose cells do not fit the LDS slots (one that crosses an
// axis-0 boundary, long or sparse columns, two instances of a batch, no
// column table) is listed for k_rows_global.
constexpr int RW_LINES = 512;  // column-table entries of a tile's span (at most)
constexpr int RW_CELLS = 512;  // cell keys staged per wavefront (a power of two)
constexpr int RW_SLOTS = RW_CELLS + 4;

// Rows of one (tile, group) from LDS; false when the tile does not fit (then
// nothing is written).  Tiles of one instance only, so the instance's fields
// are wave-uniform (scalar loads).
__device__ __forceinline__ bool rows_staged(const Dev& d, int64_t tile, int g, int32_t C,
                                            uint32_t* ck, int32_t* cs) {
  const int lane = lane_id();
  const int32_t c = (int32_t)(tile * 64 + lane);
  const bool act = c < C;
  const int32_t cc = act ? c : C - 1;
  const int nact = __popcll(ballot(act));
  int32_t iid = 0;
  if (d.ninst != 1) {
    const int32_t v = d.cell_inst[cc];
    iid = rfl_i(v);
    if (iid != rl_i(v, nact - 1)) return false;
  }
  const Inst& I = d.inst[iid];
  const bool d3 = I.dim == 3;
  if (!d3 && g > 0) return true;  // (2-D rows are those of group 0)
  const int ls = d3 ? 2 : 1;      // log2 of a column's cells per step
  const int64_t nzl = I.nzl;
  const int32_t nz = (int32_t)(nzl >> ls);
  const int64_t shift = d3 ? (g - 1) * I.cstride : 0;
  // columns of the tile, and of its neighbours in this group, within the
  // instance
  const int64_t own = (int64_t)d.cell_col[cc] - I.line_base;
  const uint32_t z = d.cell_zl[cc] >> ls;
  int64_t lmin = rl_l(own, 0) + shift - 1, lmax = rl_l(own, nact - 1) + shift + 1;
  lmin = lmin < 0 ? 0 : lmin;
  lmax = lmax >= I.nlines ? I.nlines - 1 : lmax;
  if (lmax - lmin >= RW_LINES) return false;
  const int span = lmax >= lmin ? (int)(lmax - lmin + 1) : 0;
  // relative keys of the span must fit below the ~0 padding
  if ((unsigned long long)span * (unsigned long long)nzl >= 0xfffffff0ull) return false;
  const int64_t gl = I.line_base + lmin;  // first column-table entry of the span
  // Staged cells: [cb[j], cb[j] + sn[j]) one after the other.  A tile within
  // one column needs only the steps its cells reach of each of the (at most)
  // three neighbour columns, found by six lanes' binary searches at once
  // (long columns would not fit whole).  Any other tile takes the cells of
  // the whole span: [first start, last end) of its non-empty columns (the
  // columns are in cell order: the first and last non-empty entries).
  int32_t cb[3] = {0, 0, 0}, sn[3] = {0, 0, 0};
  int ncz;
  const bool one = rl_l(own, 0) == rl_l(own, nact - 1);
  if (one) {
    const uint32_t z0 = rl_u(z, 0), z1 = rl_u(z, nact - 1);  // (cells are sorted)
    const uint32_t lo0 = (z0 >= 2 ? z0 - 2 : 0) << ls;
    // lane 2j: first cell of column j at or above lo0; lane 2j + 1: first cell
    // above the last place of step z1 + 2
    int32_t at = 0, hi = 0;
    if (lane < 2 * span) {
      const int2 e = d.lines[gl + (lane >> 1)];
      if (e.x >= 0) {
        at = e.x;
        hi = e.y;
      }
    }
    const unsigned long long key1 = (((unsigned long long)z1 + 3ull) << ls);
    while (ballot(at < hi)) {
      if (at < hi) {
        const int32_t mid = (at + hi) >> 1;
        const uint32_t v = d.cell_zl[mid];
        if ((lane & 1) ? (unsigned long long)v < key1 : v < lo0)
          at = mid + 1;
        else
          hi = mid;
      }
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      cb[j] = rl_i(at, 2 * j);
      sn[j] = rl_i(at, 2 * j + 1) - cb[j];
    }
    ncz = sn[0] + sn[1] + sn[2];
  } else {
    int32_t cmin = -1, cmax = -1;
    // the entries' loads are all issued before the first is used
    int2 ev[RW_LINES / 64];
#pragma unroll
    for (int k = 0; k < RW_LINES / 64; ++k) {
      const int i = lane + 64 * k;
      ev[k] = make_int2(-1, -1);
      if (i < span) ev[k] = d.lines[gl + i];
    }
#pragma unroll
    for (int k = 0; k < RW_LINES / 64; ++k) {
      if (64 * k < span) {
        const int2 e = ev[k];
        const unsigned long long m = ballot(e.x >= 0 && e.y > e.x);
        if (m) {
          if (cmin < 0) cmin = rl_i(e.x, __ffsll((long long)m) - 1);
          cmax = rl_i(e.y, 63 - __clzll((long long)m));
        }
      }
    }
    cb[0] = cmin < 0 ? 0 : cmin;
    ncz = sn[0] = cmin >= 0 ? cmax - cmin : 0;
  }
  if (ncz >= RW_CELLS) return false;
  const int n0 = sn[0], n01 = sn[0] + sn[1];
  // a power of two > ncz: the last slot is always a ~0 sentinel, so the
  // search (which reaches index pad - 2 at most) is exact
  const int pad = 1 << (32 - __clz(ncz));
  // keys relative to kbase fit 32 bits, so the low halves of the keys are
  // enough (little-endian), all loaded before the first is stored
  const uint32_t kbase = (uint32_t)(I.key_base + lmin * nzl);
  const uint32_t* key_lo = reinterpret_cast<const uint32_t*>(d.cell_key);
  uint32_t kv[RW_CELLS / 64];
  int32_t sv[RW_CELLS / 64];  // and the cells' ends, for the windows' point counts
#pragma unroll
  for (int k = 0; k < RW_CELLS / 64; ++k) {
    const int i = lane + 64 * k;
    kv[k] = 0u;
    sv[k] = 0;
    const int32_t ci = i < n0 ? cb[0] + i : (i < n01 ? cb[1] + (i - n0) : cb[2] + (i - n01));
    if (i < ncz) {
      kv[k] = key_lo[2 * (int64_t)ci];
      sv[k] = d.cell_start[ci + 1];
    }
  }
#pragma unroll
  for (int k = 0; k < RW_CELLS / 64; ++k) {
    const int i = lane + 64 * k;
    if (i < pad) {
      ck[i] = i < ncz ? kv[k] - kbase : 0xffffffffu;
      cs[i] = sv[k];
    }
  }
  if (lane < 4) ck[pad + lane] = 0xffffffffu;
  wave_sync();
  // windows: first key, key past the end, and the key of slot 0 (which may
  // lie below the column: modulo 2^32); a column outside the instance gets an
  // empty window
  const uint32_t zlo = z >= 2 ? z - 2 : 0;
  const uint32_t zhi = z + 2u < (uint32_t)nz ? z + 2u : (uint32_t)nz - 1u;
  uint32_t klo[3], kend[3], kwin[3];
  int32_t pos[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int64_t col = own + shift + j - 1 - lmin;
    const bool ok = act && col >= 0 && col < span;
    const uint32_t base = (uint32_t)(col * nzl);
    klo[j] = ok ? base + (zlo << ls) : 0u;
    kend[j] = ok ? base + ((zhi + 1) << ls) : 0u;
    kwin[j] = base + (z << ls) - (2u << ls);
    pos[j] = -1;  // last index with key < klo
  }
  for (int h = pad >> 1; h > 0; h >>= 1) {
    uint32_t v[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) v[j] = ck[pos[j] + h];
#pragma unroll
    for (int j = 0; j < 3; ++j) pos[j] = v[j] < klo[j] ? pos[j] + h : pos[j];
  }
  uint32_t m[3] = {0u, 0u, 0u};
  int32_t q[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) q[j] = pos[j] + 1;
  for (;;) {
    // (q stays at or below pad: the keys from ncz on end every window)
    uint32_t v[3][4];
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[j][i] = ck[q[j] + i];
    bool more = false;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (v[j][i] < kend[j]) m[j] |= 1u << (v[j][i] - kwin[j]);
      if (v[j][3] < kend[j]) {
        q[j] += 4;
        more = true;
      }
    }
    if (!ballot(more)) break;
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int r = d3 ? 3 * g + j : j;
    const int f = pos[j] + 1, nc = __popc(m[j]);
    // (the windows of a one-column tile lie in segment lmin + k, k = the
    // window's column - lmin)
    const int k = one ? (int)(own + shift + j - 1 - lmin) : 0;
    const int32_t first = f + (k <= 0 ? cb[0] : (k == 1 ? cb[1] - n0 : cb[2] - n01));
    int32_t np = 0;
    if (act && m[j]) np = cs[f + nc - 1] - d.cell_start[first];
    if (act) d.rows[(int64_t)r * d.rstride + c] = make_row(first, m[j], np);
  }
  return true;
}

__global__ __launch_bounds__(256, 8) void k_rows(Dev d) {
  if (abandoned(d)) return;
  __shared__ uint32_t s_ck[4][RW_SLOTS];
  __shared__ int32_t s_cs[4][RW_CELLS];
  const int32_t C = (int32_t)d.ctl[C_NCELL];
  const bool table = d.ctl[C_NLINES] <= d.line_cap;
  const int wv = threadIdx.x >> 6;
  // work item: tile * 3 + group; the four waves of a workgroup take four
  // consecutive items per step (the steps are uniform over the workgroup, as
  // the list append wants)
  const int64_t items = (((int64_t)C + 63) >> 6) * 3;
  for (int64_t base = (int64_t)blockIdx.x * 4; base < items; base += (int64_t)gridDim.x * 4) {
    const int64_t it = base + wv;
    bool left = false;
    if (it < items) {
      const int64_t tile = it / 3;
      left = !(table && rows_staged(d, tile, (int)(it - tile * 3), C, s_ck[wv], s_cs[wv]));
    }
    block_append(lane_id() == 0 && left, (int32_t)it, d.rows_fb);
  }
}

// The (tile, group) pairs k_rows left: one lane per cell, the column's cell
// range from the column table (or by two lower bounds over all cell keys
// when there is none), then the first cell of the window by binary search
// over cell_zl in global memory and its slot bits from the cells that
// follow, the three columns in lockstep so that their loads overlap.
__global__ __launch_bounds__(256) void k_rows_global(Dev d) {
  if (abandoned(d)) return;
  __shared__ long long s_pre[kStripes + 1];
  const long long nit = slist_prefix(d.rows_fb, s_pre);
  const int32_t C = (int32_t)d.ctl[C_NCELL];
  const bool table = d.ctl[C_NLINES] <= d.line_cap;
  const int wv = threadIdx.x >> 6, lane = lane_id();
  for (long long w = (long long)blockIdx.x * 4 + wv; w < nit; w += (long long)gridDim.x * 4) {
    const int64_t it = slist_at(d.rows_fb, s_pre, w);
    const int64_t tile = it / 3;
    const int g = (int)(it - tile * 3);
    const int32_t c = (int32_t)(tile * 64 + lane);
    const int32_t cc = c < C ? c : C - 1;
    const Inst& I = *inst_of_cell(d, cc);
    const bool d3 = I.dim == 3;
    const bool act = c < C && (d3 || g == 0);
    const int ls = d3 ? 2 : 1;
    const int64_t nzl = I.nzl;
    const int32_t nz = (int32_t)(nzl >> ls);
    const int64_t shift = d3 ? (g - 1) * I.cstride : 0;
    const uint32_t zl = d.cell_zl[cc], z = zl >> ls;
    const uint64_t key0 = d.cell_key[cc] - zl;  // first key of the cell's column
    const int64_t own = table ? (int64_t)d.cell_col[cc] - I.line_base
                              : (int64_t)((key0 - (uint64_t)I.key_base) / (uint64_t)nzl);
    int32_t st[3], en[3];
    bool ok[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int64_t col = own + shift + j - 1;
      ok[j] = act && col >= 0 && col < I.nlines;
      st[j] = en[j] = 0;
      if (ok[j] && table) {
        const int2 lr = d.lines[I.line_base + col];
        if (lr.x >= 0) {
          st[j] = lr.x;
          en[j] = lr.y;
        }
      }
    }
    if (!table) {
      int32_t lo[3], hi[3];
      uint64_t k0[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        k0[j] = key0 + (uint64_t)((shift + j - 1) * nzl);
        lo[j] = 0;
        hi[j] = ok[j] ? C : 0;
      }
      lower_bound3(d.cell_key, lo, hi, k0);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        st[j] = lo[j];
        hi[j] = ok[j] ? C : lo[j];
        k0[j] += (uint64_t)nzl;
      }
      lower_bound3(d.cell_key, lo, hi, k0);
#pragma unroll
      for (int j = 0; j < 3; ++j) en[j] = ok[j] ? lo[j] : st[j];
    }
    const uint32_t zlo = z >= 2 ? z - 2 : 0;
    const uint32_t zhi = z + 2u < (uint32_t)nz ? z + 2u : (uint32_t)nz - 1u;
    int32_t q[3], hi[3];
    uint32_t lov[3], m[3] = {0u, 0u, 0u};
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      q[j] = st[j];
      hi[j] = en[j];
      lov[j] = zlo << ls;
    }
    lower_bound3(d.cell_zl, q, hi, lov);
    // (the last place of a window may be the last 32-bit value: compared
    // inclusively)
    const uint32_t last = (zhi << ls) + ((1u << ls) - 1u), win = (z << ls) - (2u << ls);
    int32_t first[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) first[j] = q[j];
    for (;;) {
      uint32_t v[3][4];
      bool in[3][4], more = false;
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          in[j][i] = q[j] + i < en[j];
          v[j][i] = in[j][i] ? d.cell_zl[q[j] + i] : 0u;
        }
#pragma unroll
      for (int j = 0; j < 3; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (in[j][i] && v[j][i] <= last) m[j] |= 1u << (v[j][i] - win);
        if (in[j][3] && v[j][3] <= last) {
          q[j] += 4;
          more = true;
        } else {
          q[j] = en[j];
        }
      }
      if (!ballot(more)) break;
    }
    if (act) {
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const int r = d3 ? 3 * g + j : j;
        int32_t np = 0;
        if (m[j]) np = d.cell_start[first[j] + __popc(m[j])] - d.cell_start[first[j]];
        d.rows[(int64_t)r * d.rstride + c] = make_row(first[j], m[j], np);
      }
    }
  }
}

// Neighbourhood sizes (on request): non-empty cells and candidate points of
// every cell's 5^D stencil.
template <int D>
__device__ void nbr_stats_cell(const Dev& d, int32_t c, long long& cand, long long& nbrc) {
  const int local = (int)(d.cell_zl[c] & (Win<D>::nl - 1));
  const RowsOf rows = rows_of(d, c);
  long long pts = 0;
  for (int r = 0; r < Win<D>::rows; ++r) {
    const uint2 row = rows[r];
    uint32_t m = row.y & (D == 3 ? row_valid<3>(r / 3 - 1, r % 3 - 1, local)
                                 : row_valid<2>(r - 1, 0, local));
    nbrc += __popc(m);
    while (m) {
      const int32_t q = slot_cell(row, __ffs(m) - 1);
      m &= m - 1;
      pts += d.cell_start[q + 1] - d.cell_start[q];
    }
  }
  cand += pts * (d.cell_start[c + 1] - d.cell_start[c]);
}

__global__ __launch_bounds__(256) void k_nbr_stats(Dev d) {
  if (abandoned(d)) return;
  const int32_t C = (int32_t)d.ctl[C_NCELL];
  long long cand = 0, nbrc = 0;
  for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < C;
       c += (int64_t)gridDim.x * blockDim.x) {
    if (inst_of_cell(d, c)->dim == 3)
      nbr_stats_cell<3>(d, (int32_t)c, cand, nbrc);
    else
      nbr_stats_cell<2>(d, (int32_t)c, cand, nbrc);
  }
  stat_add(d, C_CAND, cand);
  stat_add(d, C_NBRC, nbrc);
}

// ------------------------------------------------------------- launchers --
void launch_index_head(const Dev& d, int nchunks, hipStream_t s) {
  // (one instance: 1024 points and more a workgroup, a step of its threads)
  const int64_t shares = std::max<int64_t>(1, std::min<int64_t>(2048, (d.n + 1023) / 1024));
  hipLaunchKernelGGL(k_bbox, dim3(d.ninst == 1 ? (unsigned)shares : nchunks), dim3(256), 0, s, d);
  if (d.ninst != 1) hipLaunchKernelGGL(k_grid_setup, dim3(1), dim3(1024), 0, s, d);
}

// Workgroups and entries per thread of the radix passes over n entries: at most
// kSortGrid workgroups (two per CU; with 768 or 1024 the scatters of 4 M points took 129 and 134 us), and
// the largest tile of which each still gets one and a half or more, so that one
// tile's loads run beside another's write-out.  Scatter of all passes, us, at
// 2 / 4 / 8 / 16 entries per thread: 10 k points 12 / 15 / 17 / -, 262 k
// 26 / 30 / 41 / 45, 614 k 37 / 43 / 54 / 84, 1 M 32 / 38 / 45 / 69, 1.5 M
// 44 / 45 / 60 / 55, 4 M 152 / 112 / 96 / 126, 8 M (batch) 233 / 178 / 171 / 156,
// 32 M - / 833 / 692 / 622.  (64-bit keys stop at 8: the tile has 12 bytes an
// entry.)
struct SortShape {
  int blocks, items;
};
SortShape sort_shape(int form, int64_t n) {
  SortShape s;
  s.items = form == 64 ? 8 : 16;
  while (s.items > 2 && 2 * n < 3LL * kSortGrid * RS_T * s.items) s.items /= 2;
  const int64_t tile = (int64_t)RS_T * s.items;
  s.blocks = (int)std::max<int64_t>(1, std::min<int64_t>(kSortGrid, (n + tile - 1) / tile));
  if (s.blocks >= 64) s.blocks &= ~7;  // (XCD-wise ranges)
  return s;
}

constexpr int kClearGrid = 1024;

template <int KF, int NI>
static void radix_passes(const Dev& d, int passes, int nblk, hipStream_t s) {
  for (int p = 0; p < passes; ++p) {
    if (p > 0 || d.ninst != 1)
      hipLaunchKernelGGL(k_rs_hist<KF>, dim3(nblk), dim3(RS_T), 0, s, d, p, nblk);
    hipLaunchKernelGGL((k_rs_scatter<KF, NI>), dim3(nblk), dim3(RS_T), 0, s, d, p, nblk);
  }
}

template <int KF>
static void index_sort(const Dev& d, int64_t n, int nchunks, int bits, hipStream_t s) {
  const int passes = (bits + kDigitBits - 1) / kDigitBits;
  const SortShape sh = sort_shape(KF, n);
  if (d.ninst == 1)
    hipLaunchKernelGGL(k_cellkey_hist<KF>, dim3(sh.blocks), dim3(RS_T), 0, s, d, sh.blocks);
  else
    hipLaunchKernelGGL(k_cellkey<KF>, dim3(nchunks), dim3(256), 0, s, d);
  if (sh.items == 2)
    radix_passes<KF, 2>(d, passes, sh.blocks, s);
  else if (sh.items == 4)
    radix_passes<KF, 4>(d, passes, sh.blocks, s);
  else if (KF == 64 || sh.items == 8)
    radix_passes<KF, 8>(d, passes, sh.blocks, s);
  else
    radix_passes<KF, KF == 64 ? 8 : 16>(d, passes, sh.blocks, s);
  const int ncs = (int)((n + CS_TILE - 1) / CS_TILE);
  // (the grid also clears the column table: not too small for a large one)
  const int ncc = std::max(ncs, d.line_cap > (1 << 16) ? kClearGrid : 1);
  hipLaunchKernelGGL(k_csr_count<KF>, dim3(ncc), dim3(CS_T), 0, s, d,
                     std::min(KF, kDigitBits * passes));
  const bool scan = ncs > kScanInline;
  if (scan)
    hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, s, d.scan_tmp, ncs);
  hipLaunchKernelGGL(k_csr_write<KF>, dim3(ncs), dim3(CS_T), 0, s, d, scan);
}

// the sort's form for keys of `bits` bits over n points
static int sort_form(int64_t n, int bits) {
  return bits <= 32 ? 32 : bits <= 36 && n <= (int64_t)kIdMask + 1 ? 36 : 64;
}

void launch_index_sort(const Dev& d, int64_t n, int nchunks, int bits, hipStream_t s) {
  const int form = sort_form(n, bits);
  if (form == 32)
    index_sort<32>(d, n, nchunks, bits, s);
  else if (form == 36)
    index_sort<36>(d, n, nchunks, bits, s);
  else
    index_sort<64>(d, n, nchunks, bits, s);
}

void launch_gather(const Dev& d, int64_t n, int64_t waves, int bits, hipStream_t s) {
  // random-access gather: more blocks in flight than a fill needs
  const int64_t gb = (n + 255) / 256;
  hipLaunchKernelGGL(k_gather, dim3((int)std::max<int64_t>(1, std::min<int64_t>(16384, gb))),
                     dim3(256), 0, s, d, waves, sort_form(n, bits) == 36 ? kIdMask : ~0u);
}

// Row pass grid: one wavefront per (tile of 64 cells, group) for up
// to n cells, at most kRowGrid workgroups (the steps loop beyond).
constexpr int64_t kRowGrid = 16384;
int64_t row_blocks(int64_t n) {
  return std::max<int64_t>(1, std::min<int64_t>(kRowGrid, (((n + 63) / 64) * 3 + 3) / 4));
}
int64_t row_list_cap(int64_t n) {
  const int64_t items = ((n + 63) / 64) * 3;
  const int64_t g = row_blocks(n);
  const int64_t steps = (items + 4 * g - 1) / (4 * g);
  return (g + kStripes - 1) / kStripes * 4 * steps;  // appends per stripe, at most
}

void launch_rows(const Dev& d, int64_t n, int grid_cells, hipStream_t s) {
  hipLaunchKernelGGL(k_rows, dim3((unsigned)row_blocks(n)), dim3(256), 0, s, d);
  // the tiles left over, one wavefront each: enough waves for the list
  const int64_t gb = std::max<int64_t>(1, std::min<int64_t>(4LL * grid_cells, (n + 255) / 256));
  hipLaunchKernelGGL(k_rows_global, dim3((unsigned)gb), dim3(256), 0, s, d);
  if (d.nbr_stats) hipLaunchKernelGGL(k_nbr_stats, dim3((unsigned)gb), dim3(256), 0, s, d);
}

// digit counts of the workgroups: room for any form of the keys
int64_t sort_hist_entries(int64_t n) {
  return (int64_t)RS_D * std::max(sort_shape(32, n).blocks,
                                  std::max(sort_shape(36, n).blocks, sort_shape(64, n).blocks));
}
int64_t scan_tmp_entries(int64_t n) { return (n + CS_TILE - 1) / CS_TILE + 16; }

}  // namespace dclust
