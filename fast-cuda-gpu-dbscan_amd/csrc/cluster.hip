// Clustering kernels on gfx950: the MI355X replacement for the reference's
// expansion kernel and host merge loop.
//
// Grid: cells of side (eps/2)(1+2^-20), so every cell is a clique (all its
// points are mutual neighbours) and every neighbour of a point lies in the
// 5^D stencil of cells around its cell.  The stencil is covered by windows of
// 3^(D-1) neighbour columns of cells ("rows", internal.h).
//
//   k_core, k_core_rest, k_core_crowd   one lane per point, then several (a
//                wavefront where the candidates are many): neighbour count with early exit
//                at minpts -> core flag.  (dbscan.cu:331-369 counts while it
//                expands; here the count is its own pass, so every later
//                kernel knows which points are core.)  A cell holding
//                >= minpts points is all core without a distance test.  A
//                point that stays below minpts has seen all its neighbours
//                and records them for the border pass.
//   k_rep, k_adj   the near graph over core cells: two cells at most one
//                apart along every axis are linked when their representatives
//                (one core point each) are certainly joined.
//   k_link_local, k_link_cross   components of the near graph by union-find,
//                in LDS over runs of cells, then in global memory.
//   k_expand     the same components by persistent seed-list expansion
//                (dbscan.cu:254-387) over cells, for calls that give the
//                reference's launch values (MAX_SEEDS, THREAD_BLOCKS,
//                THREAD_COUNT, EXTRA_COLLISION_SIZE): each wavefront owns a
//                seed list of cells in LDS and pops up to 64 of them at once,
//                one per lane; each lane
//                claims the adjacent unclaimed cells of its cell with one CAS
//                each (MarkAsCandidate, dbscan.cu:189-222) and pushes them;
//                cells already claimed by another chain become collision
//                pairs in the wave's own buffer (extraCollision,
//                dbscan.cu:202-211).  Seed-list overflow and lists left when
//                a wave's budget runs out go to a correction queue that the
//                next pass expands, instead of being dropped
//                (dbscan.cu:196-199).
//   k_merge_lds / k_union_pairs / k_flatten   GPU atomic union-find over
//                chain ids (MonitorSeedPoints' CPU BFS over the collision
//                matrix and thrust::replace relabels, dbscan.cu:60-125).
//   k_comp, k_far, k_far_pairs   pairs of stencil cells in two components are
//                decided exactly and united.
//   k_roots_final / k_keys / k_border / rank scan / k_output (_split, _place)
//                canonical labels:
//                cluster id = rank of the component's minimum core input
//                index; border = minimum id over adjacent cores; noise = 0
//                (GetDbscanResult, dbscan.cu:225-251, writes sorted labels
//                instead; this writes per-point labels).
//
// Neighbour predicate P(p,q), FP64 form (exactly the reference oracle's,
// cpu-dbscan/dbscan_rtree_exp.cpp:351-358,420-438 and Rtree.h:1573-1587):
// closed box fl(p-eps) <= q <= fl(p+eps) on every axis, and
// fl(fl(fl(dx0^2) + fl(dx1^2)) [+ fl(dx2^2)]) <= fl(eps*eps).  This file is
// compiled with -ffp-contract=off so no FMA is formed.  d^2 is symmetric in
// p and q (fl(p-q) = -fl(q-p)); only the box test can differ between the two
// directions.  Two core points are joined when d^2 <= eps^2 and the box test
// holds from at least one side (the oracle's union runs from every core
// point, cpu-dbscan/dbscan_rtree_exp.cpp:379-404).
#include <algorithm>
#include <climits>

#include "internal.h"
#include "kernels.h"
#include "stencil.h"

namespace dclust {

constexpr int kCoreBatch = 4;  // neighbour-count candidates loaded per lane step
                               // (latency bound: residency pays more than longer batches)

struct Tally {  // per-lane event counts (summed per wave by stat_add)
  int band = 0, flip = 0, asym = 0, eval = 0;
  int rows = 0, ranges = 0;  // stencil work (algorithmic bytes)
};

// FP32 squared distance from fixed-point coordinates (units of w*2^-29).
// Differences are exact in wrapped int32 arithmetic because two stencil
// points are less than three cells apart on every axis.
template <int D>
__device__ __forceinline__ float d2fix(const uint32_t* a, const uint32_t* b) {
  float f = (float)(int32_t)(b[0] - a[0]);
  float s = f * f;
#pragma unroll
  for (int k = 1; k < D; ++k) {
    float g = (float)(int32_t)(b[k] - a[k]);
    s = __builtin_fmaf(g, g, s);
  }
  return s;
}

// FP32 squared distance (fixed point) from point g to the box [lo, hi] of
// points of one cell (no wrap inside a cell).  Never above d2fix(g, q) for
// any q in the box, so d2box > d2_out rules out every pair.
template <int D>
__device__ __forceinline__ float d2box(const uint32_t* g, const uint32_t* lo, const uint32_t* hi) {
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    int32_t a = (int32_t)(lo[k] - g[k]);
    int32_t b = (int32_t)(g[k] - hi[k]);
    int32_t gap = a > 0 ? a : (b > 0 ? b : 0);
    float f = (float)gap;
    s = __builtin_fmaf(f, f, s);
  }
  return s;
}

// Scalar parameters of one instance, read once per lane.
struct Par {
  double eps, eps2;
  float d2_in, d2_out, d2_mid;
  int minpts;
  __device__ __forceinline__ explicit Par(const Inst& I)
      : eps(I.eps), eps2(I.eps2), d2_in(I.d2_in), d2_out(I.d2_out), d2_mid(I.d2_mid),
        minpts(I.minpts) {}
};

// Core-core relation of the pair (a, b): d^2 <= eps^2 and the box test from
// at least one side.  FP32 form: decided by the fixed-point distance outside
// the guard band, exactly in FP64 inside it.
template <int D, bool F32>
__device__ __forceinline__ bool edge_pair(const Dev& d, const Par& P, int32_t a, int32_t b,
                                          const uint32_t* ag, const uint32_t* bg,
                                          const double* ax, const double* bx, Tally& t) {
  double xa[D], xb[D];
  if (F32) {
    const float s = d2fix<D>(ag, bg);
    if (s < P.d2_in) return true;
    if (s > P.d2_out) return false;
    t.band++;
    load_x<D, F32>(d, a, xa);
    load_x<D, F32>(d, b, xb);
  } else {
#pragma unroll
    for (int k = 0; k < D; ++k) {
      xa[k] = ax[k];
      xb[k] = bx[k];
    }
  }
  const double dd = d2_64<D>(xa, xb);
  if (!(dd <= P.eps2)) return false;
  const bool f = box_64<D>(xa, xb, P.eps), r = box_64<D>(xb, xa, P.eps);
  t.asym += (f != r) && a < b;
  return f || r;
}

// Per-lane dispatch on the instance dimension (a wavefront can straddle two
// instances of a batch).
#define DCLUST_BY_DIM(act, dim, CALL3, CALL2)      \
  do {                                             \
    if (ballot((act) && (dim) == 3)) {             \
      if ((act) && (dim) == 3) { CALL3; }          \
    }                                              \
    if (ballot((act) && (dim) == 2)) {             \
      if ((act) && (dim) == 2) { CALL2; }          \
    }                                              \
  } while (0)


// ------------------------------------------------------------------ core --
// Neighbour counts in three kernels.
//
//   k_core        one lane per point.  A cell of >= minpts points is all core,
//                 and a point whose rows hold fewer than minpts points in all
//                 (the rows carry the counts) is not core.  Else the points of the cells around the point's cell (4 x 4
//                 x 3 of them in 3-D: the middle steps of its own column's
//                 window and of those towards the sides of the block that the
//                 cell lies on) are counted until minpts, kCoreBudget of them
//                 at most.  That settles most core points; the others are
//                 listed for k_core_rest.  The count needs no records, and in the FP32 form no
//                 guard band (a pair inside it is left to the list), so the
//                 kernel is small enough for full residency.
//   k_core_rest   two or four lanes per listed point: the exact count over all
//                 of its rows with early exit at minpts.  Every candidate with
//                 d^2 <= eps^2 (either box direction) is recorded, so a point
//                 that ends non-core holds all its neighbours outside its own
//                 cell (records are kept slot by slot, so that neighbouring
//                 points write neighbouring words).
//   k_core_crowd  one wavefront per listed point with more than kCoreCrowd
//                 candidates (a few lanes would take as long as the rest of the
//                 launch); in the FP32 form first four lanes per point that a pair
//                 inside the guard band may decide, by the exact predicate.  (Few
//                 of those in most data, but every point of a lattice whose
//                 spacing is eps: a wavefront each took 1538 of the 1894 us of a
//                 call on 1 M such points, 110 of 505 now.)
//
// Both passes over points are bound by the rows and coordinates they fetch at
// random: neighbouring points name the same ones, so each XCD takes runs of
// kXcdRun workgroups of points, and the lists of k_core are walked on the XCD
// that filled them.  k_core / k_core_rest / k_core_crowd, us: 4 M 3-D points,
// FP32 form, 144 / 123 / 15 (with whole eighths of the points per XCD, lists
// walked in order and a lane per listed point 162 / 204 / 5); the batch of 7 M
// points 198 / 179 / 18 (233 / 270 / 33); 262 k dense 3-D points, FP64 form,
// 29 / 47 / 10 (31 / 110 / 18); 100 k 3-D points, FP32 form, 14 / 15 / 4 (13 /
// 47 / 4).  Lists walked with whole eighths per XCD suit the batch but not one
// clustered instance, whose work then sits on few XCDs (4 M: 214 us).
//
// A row's points are consecutive; those of the few cells of a row outside the
// 5^D stencil fail the distance test.  The non-empty point ranges of a point
// wait in a queue of its own in LDS, so that its lanes go on to the next range
// as soon as they are done with one, whatever the others are at.
constexpr int kXcdRun = 64;
// points from which two lanes share a listed point instead of four: with fewer,
// the chain of loads of one point sets the time (262 k points 47 us against
// 67), with more the work does (4 M 166 against 145; 614 k 27 against 26)
constexpr int64_t kRestQuad = 1 << 19;
constexpr int kCoreBudget = 64;   // candidates k_core tests per point
constexpr int kCoreCrowd = 512;   // candidates from which a wavefront takes a point

// Rows from the cell's own column outwards: block offsets in units of the
// near sides' (ax, ay); the first four (two in 2-D) are the near ones.
template <int D>
__device__ __forceinline__ int core_row(int i, int ax, int ay) {
  constexpr int oa[9] = {0, 1, 0, 1, -1, 0, -1, 1, -1}, ob[9] = {0, 0, 1, 1, 0, -1, 1, -1, -1};
  if (D == 2) return Win<2>::own + (i == 0 ? 0 : (i == 1 ? ax : -ax));
  return Win<3>::own + 3 * oa[i] * ax + ob[i] * ay;
}
template <int D>
__device__ __forceinline__ void near_sides(int local, int& ax, int& ay) {
  ax = D == 3 ? (local & 2 ? 1 : -1) : (local & 1 ? 1 : -1);
  ay = D == 3 ? (local & 1 ? 1 : -1) : 0;
}

// Certain neighbours of p among the points of the near rows' middle steps,
// its own cell's (`own` = qe - qs) included, until minpts or the budget; -1
// when all rows together hold fewer than minpts points.
template <int D, bool F32>
__device__ int core_near(const Dev& d, const Par& P, int32_t p, int32_t c, int32_t qs,
                         int32_t own, int2* queue, Tally& t) {
  constexpr int NN = D == 3 ? 4 : 2;
  constexpr int nl = Win<D>::nl;
  constexpr int B = kCoreBatch;
  constexpr uint32_t kLow = (1u << nl) - 1u, kMid = ((1u << (3 * nl)) - 1u) << nl;
  int ax, ay;
  near_sides<D>((int)(d.cell_zl[c] & (nl - 1)), ax, ay);
  const RowsOf rows = rows_of(d, c);
  uint2 row[Win<D>::rows];
#pragma unroll
  for (int r = 0; r < Win<D>::rows; ++r) row[r] = rows[core_row<D>(r, ax, ay)];
  uint32_t tot = 0u;
  bool many = false;
#pragma unroll
  for (int r = 0; r < Win<D>::rows; ++r) {
    tot += row_count(row[r]);
    many |= row_count(row[r]) == kRowCount;
  }
  t.rows += Win<D>::rows;
  if (!many && (int)tot < P.minpts) return -1;
  uint32_t pg[D];
  double px[D];
  if (F32)
    load_g<D>(d, p, pg);
  else
    load_x<D, F32>(d, p, px);
  int32_t a[NN], e[NN];
#pragma unroll
  for (int r = 0; r < NN; ++r) {
    const int32_t m0 = (int32_t)row[r].x + __popc(row[r].y & kLow);
    const int32_t n = __popc(row[r].y & kMid);
    a[r] = e[r] = 0;
    if (n) {
      a[r] = d.cell_start[m0];
      e[r] = d.cell_start[m0 + n];
    }
  }
  int nq = 0;
#pragma unroll
  for (int r = 0; r < NN; ++r)
    if (e[r] > a[r]) queue[256 * nq++] = make_int2(a[r], e[r]);
  t.ranges += nq;
  int cnt = own, j = 0, left = kCoreBudget;
  int2 cur = make_int2(0, 0);
  while (cnt < P.minpts && left > 0 && (cur.x < cur.y || j < nq)) {
    if (cur.x >= cur.y) cur = queue[256 * j++];
    int32_t qi[B];
    uint32_t cg[B][D];
    double cx[B][D];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      // past the end: a point of the own cell, which is not counted
      qi[u] = cur.x + u < cur.y ? cur.x + u : qs;
      if (F32)
        load_g<D>(d, qi[u], cg[u]);
      else
        load_x<D, F32>(d, qi[u], cx[u]);
    }
#pragma unroll
    for (int u = 0; u < B; ++u) {
      bool in;
      if (F32)
        in = d2fix<D>(pg, cg[u]) < P.d2_in;
      else
        in = d2_64<D>(px, cx[u]) <= P.eps2 && box_64<D>(px, cx[u], P.eps);
      cnt += in && (uint32_t)(qi[u] - qs) >= (uint32_t)own;
    }
    t.eval += cur.y - cur.x < B ? cur.y - cur.x : B;
    cur.x += B;
    left -= B;
  }
  return cnt;
}

template <bool F32>
__global__ __launch_bounds__(256, F32 ? 8 : 6) void k_core(Dev d) {
  if (abandoned(d)) return;
  stamp(d, C_T_CORE0);
  __shared__ int2 s_queue[4 * 256];
  const int64_t pl = (int64_t)xcd_runs<kXcdRun>(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const bool act = pl < d.n;
  const int32_t p = act ? (int32_t)pl : 0;
  int32_t c = 0, qs = 0, own = 0;
  int dim = 0;
  const Inst* I = d.inst;
  if (act) {
    c = d.cell_of[p];
    qs = d.cell_start[c];
    own = d.cell_start[c + 1] - qs;
    I = inst_of_cell(d, c);
    dim = I->dim;
  }
  Tally t;
  const Par P(*I);
  int cnt = own;  // the own cell is a clique, p itself included
  const bool search = act && own < P.minpts;
  DCLUST_BY_DIM(search, dim, (cnt = core_near<3, F32>(d, P, p, c, qs, own, s_queue + threadIdx.x, t)),
                (cnt = core_near<2, F32>(d, P, p, c, qs, own, s_queue + threadIdx.x, t)));
  const bool isc = cnt >= P.minpts;
  if (act) d.core[p] = isc;
  if (cnt < 0) d.rec_n[p] = kRecFew;
  block_append(act && !isc && cnt >= 0, p, d.core_rest);
  block_append(cnt < 0, p, d.border_pts);
  stat_add(d, C_EVAL, t.eval);
  stat_add(d, C_CORE_ROWS, t.rows);
  stat_add(d, C_CORE_RANGES, t.ranges);
}

// The exact predicate of the pair (p, q): `sym` d^2 <= eps^2, `fwd` the box
// test from p's side as well.
template <int D, bool F32>
__device__ __forceinline__ void core_pred(const Dev& d, const Par& P, int32_t p, int32_t q,
                                          const uint32_t* pg, const uint32_t* qg,
                                          const double* px, const double* qx, bool& sym,
                                          bool& fwd, Tally& t) {
  if (F32) {
    const float sd = d2fix<D>(pg, qg);
    sym = fwd = sd < P.d2_in;
    if (!(sd < P.d2_in) && !(sd > P.d2_out)) {
      double ax[D], bx[D];
      load_x<D, F32>(d, p, ax);
      load_x<D, F32>(d, q, bx);
      sym = d2_64<D>(ax, bx) <= P.eps2;
      fwd = sym && box_64<D>(ax, bx, P.eps);
      t.band++;
      t.flip += fwd != (sd <= P.d2_mid);
    }
  } else {
    sym = d2_64<D>(px, qx) <= P.eps2;
    fwd = sym && box_64<D>(px, qx, P.eps);
  }
}

// Block offsets of row i in units of the near sides (core_row for an i that is
// not a constant; 1 + offset in two bits).
template <int D>
__device__ __forceinline__ void row_sides(int i, int& oa, int& ob) {
  constexpr uint32_t a3 = 0x08499u, b3 = 0x021A5u, a2 = 0x09u;
  oa = (int)(((D == 3 ? a3 : a2) >> (2 * i)) & 3u) - 1;
  ob = D == 3 ? (int)((b3 >> (2 * i)) & 3u) - 1 : 0;
}

// Squared distances (fixed-point units) from a point to what its rows hold, by
// axis: to the blocks on the near and the far side, and to the cells one and
// two steps below and above.  The cells of a row beyond eps of the point are
// those of its first and last steps, so what is left is again one range of
// points: 132 of the 180 cells of a 3-D stencil's rows on average.  The
// distances use the arithmetic of d2fix, so d2_out bounds them.
template <int D>
struct Reach {
  float xn, xf, yn, yf, below1, below2, above1, above2;
  __device__ __forceinline__ Reach(const uint32_t* g, int local) {
    constexpr uint32_t W = 1u << kFixBits, F = W - 1u;
    const uint32_t fx = g[0] & F, fl = g[D - 1] & F;
    const bool lx = D == 3 ? (local & 2) : (local & 1);
    xn = sq(lx ? W - fx : fx);
    xf = sq(lx ? W + fx : 2u * W - fx);
    yn = yf = 0.f;
    if (D == 3) {
      const uint32_t fy = g[1] & F;
      yn = sq(local & 1 ? W - fy : fy);
      yf = sq(local & 1 ? W + fy : 2u * W - fy);
    }
    below1 = sq(fl);
    below2 = sq(fl + W);
    above1 = sq(W - fl);
    above2 = sq(2u * W - fl);
  }
  static __device__ __forceinline__ float sq(uint32_t v) {
    const float f = (float)(int32_t)v;
    return f * f;
  }
  // slots of the row on sides (oa, ob) that the point may reach
  __device__ __forceinline__ uint32_t slots(int oa, int ob, float d2_out) const {
    constexpr int nl = Win<D>::nl;
    const float s = (oa == 0 ? 0.f : oa > 0 ? xn : xf) + (ob == 0 ? 0.f : ob > 0 ? yn : yf);
    const int lo = s + below2 <= d2_out ? 0 : s + below1 <= d2_out ? 1 : 2;
    const int hi = s + above2 <= d2_out ? 5 : s + above1 <= d2_out ? 4 : 3;
    return s > d2_out ? 0u : ((1u << (hi * nl)) - 1u) & ~((1u << (lo * nl)) - 1u);
  }
};

// points of the row's cells in a run of slots: [a, e)
__device__ __forceinline__ void row_points_in(const Dev& d, uint2 row, uint32_t slots, int32_t& a,
                                              int32_t& e) {
  a = e = 0;
  const uint32_t in = row.y & slots;
  if (in) {
    const int32_t m0 = (int32_t)row.x + __popc(row.y & ((slots & (0u - slots)) - 1u));
    a = d.cell_start[m0];
    e = d.cell_start[m0 + __popc(in)];
  }
}

// Count of p over all of its rows by the Q lanes that share it.  0:
// not core, 1: core, 2: left to a wavefront (many candidates), 3: in the FP32
// form, left to the exact test (`exact`) for a pair inside the guard band that
// the others do not make up for: it costs 20 registers.
template <int D, bool F32, int Q, bool exact>
__device__ int core_rest(const Dev& d, const Par& P, int32_t p, int R,
                         int2* ranges, int32_t* lrec, Tally& t) {
  constexpr int NR = Win<D>::rows, NK = (NR + Q - 1) / Q;
  constexpr int B = 8 / Q;
  const int sub = lane_id() & (Q - 1), q0 = lane_id() & ~(Q - 1);
  // the group's bits of a ballot
  const auto mine = [&](unsigned long long m) {
    return ((q0 & 32 ? (uint32_t)(m >> 32) : (uint32_t)m) >> (q0 & 31)) & ((1u << Q) - 1u);
  };
  const uint32_t below = (1u << sub) - 1u;
  const int32_t c = d.cell_of[p];
  const int32_t qs = d.cell_start[c], own = d.cell_start[c + 1] - qs;
  int ax, ay;
  const int local = (int)(d.cell_zl[c] & (Win<D>::nl - 1));
  near_sides<D>(local, ax, ay);
  uint32_t pg[D];
  load_g<D>(d, p, pg);
  const RowsOf rows = rows_of(d, c);
  int32_t a[NK], e[NK];
  {
    uint2 row[NK];
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      const int r = k * Q + sub;
      row[k] = make_uint2(0u, 0u);
      if (r < NR) {
        int oa, ob;
        row_sides<D>(r, oa, ob);
        row[k] = rows[Win<D>::own + (D == 3 ? 3 * oa * ax + ob * ay : oa * ax)];
      }
    }
    const Reach<D> reach(pg, local);
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      int oa, ob;
      row_sides<D>(k * Q + sub, oa, ob);
      row_points_in(d, row[k], reach.slots(oa, ob, P.d2_out), a[k], e[k]);
    }
  }
  int nq = 0;
  int32_t tot = 0;  // (the own cell's points included)
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    const uint32_t m = mine(ballot(e[k] > a[k]));
    if (e[k] > a[k]) ranges[nq + __popc(m & below)] = make_int2(a[k], e[k]);
    nq += __popc(m);
    tot += e[k] - a[k];
  }
#pragma unroll
  for (int o = 1; o < Q; o <<= 1) tot += __shfl_xor(tot, o, 64);
  if (sub == 0) {
    t.rows += NR;
    t.ranges += nq;
  }
  if (tot > kCoreCrowd) return 2;
  wave_sync();  // the ranges, before the lanes read each other's
  int nrec = 0;
  double px[D];
  if (!F32) load_x<D, F32>(d, p, px);
  // the ranges one after the other, the lanes side by side
  bool band = false;
  int cnt = own, j = 0;  // cnt: own + nrec, less what only one box test finds
  int2 cur = ranges[0];
  int32_t at = cur.x + sub;
  for (int32_t i0 = sub; i0 - sub < tot && cnt < P.minpts; i0 += Q * B) {
    int32_t qi[B];
    uint32_t cg[B][D];
    double cx[B][D];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      while (at >= cur.y && j + 1 < nq) {
        at -= cur.y;
        cur = ranges[++j];
        at += cur.x;
      }
      // past the end: a point of the own cell, which is not counted
      qi[u] = i0 + u * Q < tot ? at : qs;
      at += Q;
      if (F32)
        load_g<D>(d, qi[u], cg[u]);
      else
        load_x<D, F32>(d, qi[u], cx[u]);
    }
#pragma unroll
    for (int u = 0; u < B; ++u) {
      bool sym = false, fwd = false;
      if ((uint32_t)(qi[u] - qs) >= (uint32_t)own) {
        if (F32 && !exact) {
          const float sd = d2fix<D>(pg, cg[u]);
          sym = fwd = sd < P.d2_in;
          band |= !(sd < P.d2_in) && !(sd > P.d2_out);
        } else {
          core_pred<D, F32>(d, P, p, qi[u], pg, cg[u], px, cx[u], sym, fwd, t);
        }
        ++t.eval;
      }
      const uint32_t m = mine(ballot(sym));
      const int slot = nrec + __popc(m & below);
      if (sym && slot < R) lrec[slot] = qi[u];
      nrec += __popc(m);
      cnt += __popc(m);
      if (!F32 || exact)
        if (const unsigned long long one = ballot(sym && !fwd)) cnt -= __popc(mine(one));
    }
  }
  if (cnt >= P.minpts) return 1;
  if (F32 && !exact && mine(ballot(band))) return 3;
  wave_sync();
  for (int i = sub; i < nrec && i < R; i += Q) d.rec[(int64_t)i * d.n + p] = lrec[i];
  if (sub == 0) d.rec_n[p] = (uint8_t)(nrec <= R ? nrec : kRecNone);
  return 0;
}

// Entry of Dev::core_crowd: a point, and whether four lanes take it.
constexpr int32_t kBandPoint = 1 << 28;

// LDS of a k_core_rest workgroup (k_core_crowd: Q = 4): per point nine ranges, and R record slots
// (one more: fewer bank conflicts)
static size_t core_lds(int R, int Q) {
  return 256 / Q * (kMaxRows * sizeof(int2) + (R + 1) * 4);
}

template <bool F32, int Q>
__global__ __launch_bounds__(256, (F32 ? 7 : 5) + (Q == 4)) void k_core_rest(Dev d) {
  if (abandoned(d)) return;
  extern __shared__ int2 s_core[];
  constexpr int PB = 256 / Q;  // points of a workgroup
  const Stripe L(d.core_rest);
  const int R = d.rec_stride;
  const int pt = threadIdx.x / Q;
  const bool lead = threadIdx.x % Q == 0;
  int2* ranges = s_core + pt * kMaxRows;
  int32_t* lrec = reinterpret_cast<int32_t*>(s_core + PB * kMaxRows) + pt * (R + 1);
  Tally t;
  for (int64_t i0 = L.first(PB); i0 < L.n; i0 += L.step(PB)) {
    const int64_t i = i0 + pt;
    const bool act = i < L.n;
    const int32_t p = act ? L.data[i] : 0;
    const Inst* I = d.inst;
    int dim = 0;
    if (act) {
      if (d.ninst != 1) I = inst_of_cell(d, d.cell_of[p]);
      dim = I->dim;
    }
    const Par P(*I);
    int res = 0;
    DCLUST_BY_DIM(act, dim, (res = core_rest<3, F32, Q, false>(d, P, p, R, ranges, lrec, t)),
                  (res = core_rest<2, F32, Q, false>(d, P, p, R, ranges, lrec, t)));
    if (act && lead && res == 1) d.core[p] = 1;
    block_append(act && lead && res == 0, p, d.border_pts);
    block_append(act && lead && res >= 2, p | (res == 3 ? kBandPoint : 0), d.core_crowd);
  }
  stat_add(d, C_EVAL, t.eval);
  stat_add(d, C_CORE_ROWS, t.rows);
  stat_add(d, C_CORE_RANGES, t.ranges);
}

template <int D, bool F32>
__device__ bool core_wave(const Dev& d, const Par& P, int32_t p, int R, Tally& t) {
  constexpr int NR = Win<D>::rows;
  const int lane = lane_id();
  const int32_t c = d.cell_of[p];
  const int32_t qs = d.cell_start[c], own = d.cell_start[c + 1] - qs;
  int ax, ay;
  const int local = (int)(d.cell_zl[c] & (Win<D>::nl - 1));
  near_sides<D>(local, ax, ay);
  const RowsOf rows = rows_of(d, c);
  uint32_t pg[D];
  double px[D];
  load_g<D>(d, p, pg);
  if (!F32) load_x<D, F32>(d, p, px);
  const Reach<D> reach(pg, local);
  int cnt = own, nrec = 0;
  for (int r = 0; r < NR && cnt < P.minpts; ++r) {
    int32_t a, e;
    int oa, ob;
    row_sides<D>(r, oa, ob);
    row_points_in(d, rows[Win<D>::own + (D == 3 ? 3 * oa * ax + ob * ay : oa * ax)],
                  reach.slots(oa, ob, P.d2_out), a, e);
    for (; a < e && cnt < P.minpts; a += 64) {
      const int32_t q = a + lane < e ? a + lane : qs;
      uint32_t qg[D];
      double qx[D];
      if (F32)
        load_g<D>(d, q, qg);
      else
        load_x<D, F32>(d, q, qx);
      bool sym = false, fwd = false;
      if ((uint32_t)(q - qs) >= (uint32_t)own) {
        core_pred<D, F32>(d, P, p, q, pg, qg, px, qx, sym, fwd, t);
        ++t.eval;
      }
      cnt += __popcll(ballot(fwd));
      const unsigned long long m = ballot(sym);
      const int slot = nrec + mbcnt(m);
      if (sym && slot < R) d.rec[(int64_t)slot * d.n + p] = q;
      nrec += __popcll(m);
    }
  }
  if (lane == 0) d.rec_n[p] = (uint8_t)(nrec <= R ? nrec : kRecNone);
  return cnt >= P.minpts;
}

// The listed points that a pair inside the guard band may decide.
__device__ __forceinline__ void core_band(const Dev& d, const Stripe& L, int2* s_core, Tally& t) {
  constexpr int Q = 4, PB = 256 / Q;
  const int R = d.rec_stride;
  const int pt = threadIdx.x / Q;
  const bool lead = threadIdx.x % Q == 0;
  int2* ranges = s_core + pt * kMaxRows;
  int32_t* lrec = reinterpret_cast<int32_t*>(s_core + PB * kMaxRows) + pt * (R + 1);
  for (int64_t i0 = L.first(PB); i0 < L.n; i0 += L.step(PB)) {
    const int32_t e = i0 + pt < L.n ? L.data[i0 + pt] : 0;
    const bool act = (e & kBandPoint) != 0;
    if (!__syncthreads_or(act)) continue;
    const int32_t p = act ? e & ~kBandPoint : 0;
    const Inst* I = d.inst;
    int dim = 0;
    if (act) {
      if (d.ninst != 1) I = inst_of_cell(d, d.cell_of[p]);
      dim = I->dim;
    }
    const Par P(*I);
    int res = 0;
    DCLUST_BY_DIM(act, dim, (res = core_rest<3, true, Q, true>(d, P, p, R, ranges, lrec, t)),
                  (res = core_rest<2, true, Q, true>(d, P, p, R, ranges, lrec, t)));
    if (act && lead && res == 1) d.core[p] = 1;
    block_append(act && lead && res == 0, p, d.border_pts);
  }
}

template <bool F32>
__global__ __launch_bounds__(256) void k_core_crowd(Dev d) {
  if (abandoned(d)) return;
  extern __shared__ int2 s_core[];
  const Stripe L(d.core_crowd);
  const int R = d.rec_stride;
  Tally t;
  if constexpr (F32) core_band(d, L, s_core, t);
  // (a wavefront's next 64 entries at once)
  const int64_t step = L.step(4);
  for (int64_t i = L.first(4) + (threadIdx.x >> 6); i < L.n; i += 64 * step) {
    const int64_t il = i + lane_id() * step;
    const int32_t el = il < L.n ? L.data[il] : kBandPoint;
    for (unsigned long long m = ballot(!(el & kBandPoint)); m; m &= m - 1) {
      const int32_t p = rl_i(el, __ffsll((long long)m) - 1);
      const Inst& I = *inst_of_cell(d, d.ninst == 1 ? 0 : d.cell_of[p]);
      const Par P(I);
      const bool isc = I.dim == 3 ? core_wave<3, F32>(d, P, p, R, t)
                                  : core_wave<2, F32>(d, P, p, R, t);
      if (lane_id() == 0) {
        if (isc) {
          d.core[p] = 1;
        } else {
          const SList& B = d.border_pts;
          const int s = blockIdx.x & (kStripes - 1);
          B.data[s * B.cap + (int64_t)atomicAdd(&B.cnt[s * kStatStride], 1ull)] = p;
        }
      }
    }
  }
  stat_add(d, C_EVAL, t.eval);
  stat_add(d, C_BAND_CORE, t.band);
  stat_add(d, C_BAND, t.band);
  stat_add(d, C_FLIP, t.flip);
}

// ----------------------------------------------------------- near graph --
// Workgroups of the kernels that walk the list of core cells (grid-stride).
constexpr int kListGrid = 4096;

// Every core cell is represented by its first core point (the sort is
// stable, so that is also its smallest core input index).  One lane per cell
// writes the representative's coordinates and sorted index in one 16-byte
// record (w = kNoRep for a cell without core points), resets the cell's
// state of the clustering phases and lists the core cells.
constexpr uint32_t kNoRep = 0xffffffffu;

__global__ __launch_bounds__(1024) void k_rep(Dev d) {
  if (abandoned(d)) return;
  stamp(d, C_T_CORE1);
  const int64_t C = d.ctl[C_NCELL];
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c - threadIdx.x >= C) return;  // (block-uniform)
  const bool in = c < C;
  const int64_t cc = in ? c : 0;
  const int32_t q0 = d.cell_start[cc], q1 = d.cell_start[cc + 1];
  const int minpts = inst_of_cell(d, cc)->minpts;
  // core points: all of a cell of minpts points, else its fewer than minpts
  // flags, one after the other (262 k 3-D points: 11 us with minpts 32, 13 with
  // 64, 53 with 512, 188 with 2000, a thirtieth of such a call)
  int32_t ncore = q1 - q0, first = q0;
  if (ncore < minpts) {
    ncore = 0;
    for (int32_t q = q1 - 1; q >= q0; --q)
      if (d.core[q]) {
        ++ncore;
        first = q;
      }
  }
  const bool hc = in && ncore > 0;
  uint4 r = make_uint4(0u, 0u, 0u, kNoRep);
  if (hc) {
    const int32_t q = first;
    r = make_uint4(d.G[3 * (int64_t)q], d.G[3 * (int64_t)q + 1], d.G[3 * (int64_t)q + 2],
                   (uint32_t)q);
  }
  // (the forest covers every cell: the chain merge walks all of it, and the
  // relabel pass reads entry 0 for points that are not core; without seed
  // lists k_link_local starts it, and nothing else reads the rest of a cell
  // without core points: 4 M points 57 us with everything written, 50 now)
  if (in) {
    d.rep[c] = r;
    d.cell_comp[c] = -1;
    d.amask[c] = 0u;
    if (d.chains) {
      d.parent[c] = (int32_t)c;
      d.cell_label[c] = kUnclaimed;
    }
    if (hc || d.chains) {
      d.cell_ncore[c] = ncore;
      d.compmin[c] = kNoKey;
    }
  }
  block_append(hc, (int32_t)c, d.core_cells);
  // core points, those of light cells, all-core cells and heavy cells: one
  // atomic per workgroup and counter (counted by every wave of k_core
  // instead, these took 1.0 of its 1.6 ms on 32 M points)
  const int nc = hc ? ncore : 0, m = in ? q1 - q0 : 0;
  const int sums[4] = {wave_sum(nc), wave_sum(m <= kHeavy ? nc : 0),
                       (int)__popcll(ballot(in && m >= minpts)),
                       (int)__popcll(ballot(m > kHeavy))};
  __shared__ int s_sum[16][4];
  if (lane_id() == 0)
    for (int k = 0; k < 4; ++k) s_sum[threadIdx.x >> 6][k] = sums[k];
  __syncthreads();
  if (threadIdx.x < 4) {
    constexpr int ctr[4] = {C_NCORE, C_NADJPTS, C_DENSE, C_NHEAVY};
    int t = 0;
    for (int w = 0; w < 16; ++w) t += s_sum[w][threadIdx.x];
    if (t)
      atomicAdd((unsigned long long*)&d.stat[(blockIdx.x & (kStripes - 1)) * kStatStride +
                                             ctr[threadIdx.x]],
                (unsigned long long)t);
  }
}

// Near graph: near bit b of a core cell's mask is set when the near cell at
// its offset holds a representative that is certainly joined to its own
// (fixed-point distance below the guard band, which implies the FP64
// predicate in both directions).  Each pair is tested once, by the cell for
// which the offset is positive (bits above kNearOwn).
// The graph need not hold every adjacent pair: whatever pair it
// leaves in two components is decided exactly by the pass over component
// borders (k_far, k_far_pairs).  Inside a cluster the first pair of points
// nearly always joins (of 7.3 M near cell pairs of the 4 M point 3-D
// workload 92 % are joined, with 1.15 point tests per pair), so one 16-byte
// load and one distance per pair take the place of a scan of both cells'
// points: 55 + 58 us with k_rep, where testing every near pair to the end
// took 289 us there, 77 + 90 us on 1 M 2-D points (here 20) and 2.2 ms on
// 32 M points in dense blobs (cells of more than 32 points wave by wave).
// Representatives of three consecutive steps (below, at and above the cell)
// at one place of a row, tested against `ag`: bits b0, b0 + 1, b0 + 2.
template <int D>
__device__ __forceinline__ void near_line(const Dev& d, float d2_in, const uint32_t* ag,
                                          uint2 row, int place, int b0, uint32_t& m, Tally& t) {
  constexpr int nl = Win<D>::nl;
  uint4 b4[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int s = (k + 1) * nl + place;
    b4[k].w = kNoRep;
    if ((row.y >> s) & 1u) b4[k] = d.rep[slot_cell(row, s)];
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const uint32_t bg[3] = {b4[k].x, b4[k].y, b4[k].z};
    if (b4[k].w != kNoRep) {
      ++t.eval;
      if (d2fix<D>(ag, bg) < d2_in) m |= 1u << (b0 + k);
    }
  }
}

template <int D>
__device__ __forceinline__ uint32_t near_bits(const Dev& d, float d2_in, int32_t A, Tally& t) {
  const uint4 a4 = d.rep[A];
  const uint32_t ag[3] = {a4.x, a4.y, a4.z};
  const int local = (int)(d.cell_zl[A] & (Win<D>::nl - 1));
  const RowsOf rows = rows_of(d, A);
  uint32_t m = 0;
  if (D == 2) {
    const uint2 own = rows[1], up = rows[1 + local];  // dx = 1 lies in block lx
    near_line<2>(d, d2_in, ag, up, local ^ 1, 21, m, t);
    const int s = 3 * 2 + local;  // dx = 0, one step up
    if ((own.y >> s) & 1u) {
      const uint4 b4 = d.rep[slot_cell(own, s)];
      const uint32_t bg[3] = {b4.x, b4.y, b4.z};
      if (b4.w != kNoRep) {
        ++t.eval;
        if (d2fix<2>(ag, bg) < d2_in) m |= 1u << 14;
      }
    }
  } else {
    const int lx = local >> 1, ly = local & 1;
    // dx = 1 lies in block row lx; dy = 0 and the dy towards the cell's own
    // block in block column 0, the other dy in block column nb; dx = 0,
    // dy = 1 in block column ly
    const int nb = ly ? 1 : -1;
    const uint2 own = rows[4], x0 = rows[4 + 3 * lx], xb = rows[4 + 3 * lx + nb],
                y1 = rows[4 + ly];
    const int xo = (lx ^ 1) * 2;
    near_line<3>(d, d2_in, ag, x0, xo + ly, 21, m, t);
    near_line<3>(d, d2_in, ag, x0, xo + (ly ^ 1), 21 - 3 * nb, m, t);
    near_line<3>(d, d2_in, ag, xb, xo + (ly ^ 1), 21 + 3 * nb, m, t);
    near_line<3>(d, d2_in, ag, y1, lx * 2 + (ly ^ 1), 15, m, t);
    const int s = 3 * 4 + local;  // dx = dy = 0, one step up
    if ((own.y >> s) & 1u) {
      const uint4 b4 = d.rep[slot_cell(own, s)];
      const uint32_t bg[3] = {b4.x, b4.y, b4.z};
      if (b4.w != kNoRep) {
        ++t.eval;
        if (d2fix<3>(ag, bg) < d2_in) m |= 1u << 14;
      }
    }
  }
  return m;
}

// Near cell of A at near bit b (one of A's mask bits).
__device__ __forceinline__ int32_t near_cell(const RowsOf& rows, int dim, int local, int b) {
  int row, slot;
  if (dim == 3)
    near_slot<3>(b, local, row, slot);
  else
    near_slot<2>(b, local, row, slot);
  return slot_cell(rows[row], slot);
}
__device__ __forceinline__ int local_of(const Dev& d, int32_t c, int dim) {
  return (int)(d.cell_zl[c] & (dim == 3 ? 3u : 1u));
}

// The rows that hold a cell's forward near cells (bits above kNearOwn), loaded
// once: the loops over mask bits then wait for no row.
struct NearRows {
  uint32_t ox, oy, x0x, x0y, xbx, xby, y1x, y1y;
  int dim, local, gb;  // gb: the group of three bits whose row is xb
};
__device__ __forceinline__ NearRows near_rows(const Dev& d, int32_t A, int dim) {
  const RowsOf rows = rows_of(d, A);
  const int local = local_of(d, A, dim);
  const int lx = local >> 1, nb = local & 1 ? 1 : -1;
  const bool d3 = dim == 3;
  const uint2 own = rows[d3 ? 4 : 1], x0 = rows[d3 ? 4 + 3 * lx : 1 + local],
              xb = rows[d3 ? 4 + 3 * lx + nb : 1 + local], y1 = rows[d3 ? 4 + (local & 1) : 1];
  return NearRows{own.x, own.y, x0.x, x0.y, xb.x, xb.y, y1.x, y1.y, dim, local, d3 ? 7 + nb : -1};
}
__device__ __forceinline__ uint32_t pick(bool c, uint32_t a, uint32_t b) {
  const uint32_t m = 0u - (uint32_t)c;  // (a ?: of two fields goes through scratch)
  return (a & m) | (b & ~m);
}
// forward near cell at bit b
__device__ __forceinline__ int32_t near_cell(const NearRows& n, int b) {
  const int g = (b * 11) >> 5;  // b / 3 for b < 27
  int row, slot;
  if (n.dim == 3)
    near_slot<3>(b, n.local, row, slot);
  else
    near_slot<2>(b, n.local, row, slot);
  uint2 r;
  r.x = pick(g == 4, n.ox, pick(g == 5, n.y1x, pick(g == n.gb, n.xbx, n.x0x)));
  r.y = pick(g == 4, n.oy, pick(g == 5, n.y1y, pick(g == n.gb, n.xby, n.x0y)));
  return slot_cell(r, slot);
}

// One lane per core cell.  For the expansion by seed lists each bit of A is
// also set in the other cell's mask, at the opposite offset.
__global__ __launch_bounds__(256) void k_adj(Dev d) {
  if (abandoned(d)) return;
  const Stripe L(d.core_cells);
  Tally t;
  long long edges = 0;
  for (int64_t i0 = L.first(256); i0 < L.n; i0 += L.step(256)) {
    const int64_t i = i0 + threadIdx.x;
    const bool act = i < L.n;
    const int32_t A = act ? L.data[i] : 0;
    int dim = 0;
    float d2_in = 0.f;
    if (act) {
      const Inst* I = inst_of_cell(d, A);
      dim = I->dim;
      d2_in = I->d2_in;
    }
    uint32_t m = 0;
    DCLUST_BY_DIM(act, dim, (m = near_bits<3>(d, d2_in, A, t)),
                  (m = near_bits<2>(d, d2_in, A, t)));
    if (!d.chains) {
      edges += 2 * __popc(m);
      if (act) d.amask[A] = m;
    } else if (m) {
      const RowsOf rows = rows_of(d, A);
      const int local = local_of(d, A, dim);
      atomicOr(&d.amask[A], m);
      while (m) {
        const int b = __ffs(m) - 1;
        m &= m - 1;
        atomicOr(&d.amask[near_cell(rows, dim, local, b)], 1u << (2 * kNearOwn - b));
      }
    }
  }
  stat_add(d, C_ADJ_TESTS, t.eval);
  if (!d.chains) stat_add(d, C_EDGES, edges);
}

// Components of the near graph without seed lists, in two kernels.
// k_link_local: a workgroup takes a run of consecutive cells and unites the
// pairs inside it in an LDS copy of the forest, then writes every cell's
// root; the bits that leave the run stay in the masks.  k_link_cross unites
// those in global memory, between roots only.  (All pairs in global memory
// took 1.65-2.1 ms on the 4 M point 3-D workload, against 61 + 64 us: cells
// of a cluster hook each other link by link into chains that every find then
// walks with loads past the L2, which is not coherent across XCDs.  Without
// its table of pairs k_link_cross took 150 us, and 114 with links by id
// instead of uf_order.)
//
// A thread unites the pairs of its cells one after the other, so short runs
// and many workgroups pay until the pairs between runs weigh more: runs of at
// least 4096 cells on 512 workgroups took 104 + 61 us on the 4 M points, 57 +
// 10 on 100 k (15 + 17 now), 30 + 13 on 1 M 2-D points (10 + 15); 8192
// workgroups 65 + 78 on the 4 M.
//
// k_link_cross walks the whole list, neighbouring workgroups on neighbouring
// entries: with the entries of a stripe on one XCD its plain loads find parents
// that are stale in that L2, and it took 121 us.
constexpr int kLinkCells = 16384;  // cells of one LDS forest (64 KiB)
constexpr int kLinkMin = 1024;     // least cells of a run
constexpr int kLinkGrid = 2048;    // workgroups

__device__ __forceinline__ int32_t lds_find(int32_t* par, int32_t x) {
  for (;;) {
    int32_t p = par[x];
    if (p == x) return x;
    int32_t gp = par[p];
    if (gp != p) par[x] = gp;
    x = p;
  }
}

// unites the sets of a and b; returns their root
__device__ __forceinline__ int32_t lds_union(int32_t* par, int32_t a, int32_t b) {
  a = lds_find(par, a);
  b = lds_find(par, b);
  while (a != b) {
    if (uf_order(a) < uf_order(b)) {
      const int32_t t = a;
      a = b;
      b = t;
    }
    const int32_t old = atomicCAS(&par[a], a, b);
    if (old == a || old == b) return b;
    a = lds_find(par, old);
    b = lds_find(par, b);
  }
  return a;
}

__global__ __launch_bounds__(1024) void k_link_local(Dev d) {
  if (abandoned(d)) return;
  __shared__ int32_t par[kLinkCells];
  const int32_t C = (int32_t)d.ctl[C_NCELL];
  // cells per run: the workgroups share the cells, in whole wavefronts
  int32_t K = (C + (int32_t)gridDim.x - 1) / (int32_t)gridDim.x;
  K = (K + 1023) & ~1023;
  K = K < kLinkMin ? kLinkMin : (K > kLinkCells ? kLinkCells : K);
  for (int64_t c0 = (int64_t)blockIdx.x * K; c0 < C; c0 += (int64_t)gridDim.x * K) {
    const int32_t nc = (int32_t)(C - c0 < K ? C - c0 : K);
    for (int i = threadIdx.x; i < nc; i += 1024) par[i] = i;
    __syncthreads();
    for (int i = threadIdx.x; i < nc; i += 1024) {
      const int32_t A = (int32_t)c0 + i;
      uint32_t m = d.amask[A];
      if (!m) continue;
      const NearRows near = near_rows(d, A, inst_of_cell(d, A)->dim);
      uint32_t ext = 0u;
      int32_t root = i;
      while (m) {
        const int b = __ffs(m) - 1;
        m &= m - 1;
        const int32_t B = near_cell(near, b) - (int32_t)c0;
        if (B >= 0 && B < nc)
          root = lds_union(par, root, B);
        else
          ext |= 1u << b;
      }
      d.amask[A] = ext;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nc; i += 1024) {
      int32_t r = i;
      while (par[r] != r) r = par[r];
      d.parent[c0 + i] = (int32_t)c0 + r;
    }
    __syncthreads();
  }
}

constexpr int kLinkSeen = 256;  // root pairs a wavefront remembers

__global__ __launch_bounds__(256) void k_link_cross(Dev d) {
  if (abandoned(d)) return;
  __shared__ long long s_pre[kStripes + 1];
  __shared__ unsigned long long s_seen[4][kLinkSeen];
  __shared__ uint8_t s_tag[4][kLinkSeen];
  const int lane = lane_id(), wv = threadIdx.x >> 6;
  unsigned long long* seen = s_seen[wv];
  uint8_t* tag = s_tag[wv];
  for (int i = lane; i < kLinkSeen; i += 64) seen[i] = ~0ull;
  const long long n = slist_prefix(d.core_cells, s_pre);
  for (long long i0 = (long long)blockIdx.x * 256; i0 < n; i0 += (long long)gridDim.x * 256) {
    const long long i = i0 + threadIdx.x;
    const int32_t A = i < n ? slist_at(d.core_cells, s_pre, i) : -1;
    uint32_t m = A >= 0 ? d.amask[A] : 0u;
    const int32_t pa = m ? d.parent[A] : 0;
    const NearRows near = near_rows(d, m ? A : 0, inst_of_cell(d, m ? A : 0)->dim);
    while (ballot(m != 0u)) {
      int32_t pb = -1;
      if (m) {
        const int b = __ffs(m) - 1;
        m &= m - 1;
        pb = d.parent[near_cell(near, b)];
      }
      // neighbouring cells mostly name the same two roots: a pair in the
      // wave's table is left out, and of the lanes that hold the same pair
      // now, the one whose id survives in the pair's tag slot unites it
      const unsigned long long key = ((unsigned long long)(uint32_t)pa << 32) | (uint32_t)pb;
      const int h = (int)(((uint32_t)pa * 0x9E3779B1u ^ (uint32_t)pb * 0x85EBCA6Bu) >> 24);
      bool nw = pb >= 0 && seen[h] != key;
      if (nw) tag[h] = (uint8_t)lane;
      wave_sync();
      const int w = nw ? (int)tag[h] : lane;
      const uint32_t wlo = (uint32_t)__shfl((int)(uint32_t)key, w, 64);
      const uint32_t whi = (uint32_t)__shfl((int)(uint32_t)(key >> 32), w, 64);
      if (w != lane && (((unsigned long long)whi << 32) | wlo) == key) nw = false;
      if (nw) {
        seen[h] = key;
        uf_union(d.parent, pa, pb);
      }
      wave_sync();
    }
  }
}

// Component of every core cell (the root of its chain, or of the cell
// itself without seed lists), the component minima of the core input index,
// and the list of the roots.
__global__ __launch_bounds__(256) void k_comp(Dev d) {
  if (abandoned(d)) return;
  const Stripe L(d.core_cells);
  for (int64_t i0 = L.first(256); i0 < L.n; i0 += L.step(256)) {
    const int64_t i = i0 + threadIdx.x;
    const bool act = i < L.n;
    const int32_t A = act ? L.data[i] : 0;
    int32_t comp = -1, cmin = kNoKey;
    if (act) {
      cmin = d.orig[d.rep[A].w];
      comp = uf_find(d.parent, d.chains ? d.cell_label[A] : A);
      d.cell_comp[A] = comp;
    }
    // the wave's leading component: one atomic; the other lanes: one each,
    // unless the minimum (a plain load is at worst too large) is already
    // lower
    const unsigned long long ma = ballot(act);
    if (ma) {
      const int32_t lead = rl_i(comp, __ffsll((long long)ma) - 1);
      const bool mine = act && comp == lead;
      const int32_t v = wave_min(mine ? cmin : kNoKey);
      if (lane_id() == 0 && v < d.compmin[lead]) atomicMin(&d.compmin[lead], v);
      if (act && !mine && cmin < d.compmin[comp]) atomicMin(&d.compmin[comp], cmin);
    }
    block_append(act && comp == A, A, d.near_roots);
  }
}

// --------------------------------------------------- component borders --
// Distance (fixed-point units) from a point at fraction f of its cell to
// the cell o cells away along one axis (0 for o = 0).
__device__ __forceinline__ float cell_gap(int o, int32_t f) {
  const int32_t g = o > 0 ? (o << kFixBits) - f : (o < 0 ? f + ((-o - 1) << kFixBits) : 0);
  return (float)g;
}

// Distance (fixed-point units) from a point at fraction f of its cell to
// the far side of the cell o cells away along one axis.
__device__ __forceinline__ float cell_far(int o, int32_t f) {
  constexpr int32_t W = 1 << kFixBits;
  const int32_t g = o > 0 ? (o + 1) * W - f : (o < 0 ? f - o * W : (f > W - f ? f : W - f));
  return (float)g;
}

// Is some core point of A (points [qs, qe)) joined to some core point of B
// (points [b0, b1), holding at least one core point)?  off = offset of B's
// cell from A's.  A's core points are tried in turn: skipped when B's cell
// box lies beyond eps of the point, accepted without a test when B's whole
// box lies inside the guard band around it (every point of B is then
// joined to it), else tested against B's core points.  The box distances
// use the same fixed-point arithmetic as the distance, so they bound it.
template <int D, bool F32>
__device__ bool cells_joined(const Dev& d, const Par& P, int32_t qs, int32_t qe, bool allc,
                             int32_t b0, int32_t b1, int off0, int off1, int offl, Tally& t,
                             long long& freeb) {
  constexpr uint32_t kFrac = (1u << kFixBits) - 1u;
  const int off[3] = {off0, D == 3 ? off1 : offl, offl};
  for (int32_t a = qs; a < qe; ++a) {
    // the flag and the coordinates are loaded together
    uint32_t ag[D];
    load_g<D>(d, a, ag);
    if (!allc && !d.core[a]) continue;
    float g2 = 0.f, h2 = 0.f;
#pragma unroll
    for (int x = 0; x < D; ++x) {
      const int32_t f = (int32_t)(ag[x] & kFrac);
      const float e = cell_gap(off[x], f), fe = cell_far(off[x], f);
      g2 = __builtin_fmaf(e, e, g2);
      h2 = __builtin_fmaf(fe, fe, h2);
    }
    if (g2 > P.d2_out) continue;
    if (h2 < P.d2_in) {
      ++freeb;
      return true;
    }
    double ax[D];
#pragma unroll
    for (int x = 0; x < D; ++x) ax[x] = F32 ? 0.0 : d.X[3 * (int64_t)a + x];
    for (int32_t q0 = b0; q0 < b1; q0 += 4) {
      bool cf[4];
      uint32_t qg[4][D];
      double qx[4][D];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool in = q0 + j < b1;
        const int32_t q = in ? q0 + j : b0;
        // (coordinates loaded with the flag, not after it)
        cf[j] = in && d.core[q];
#pragma unroll
        for (int x = 0; x < D; ++x) {
          qg[j][x] = F32 ? d.G[3 * (int64_t)q + x] : 0u;
          qx[j][x] = !F32 ? d.X[3 * (int64_t)q + x] : 0.0;
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (cf[j]) {
          ++t.eval;
          if (edge_pair<D, F32>(d, P, a, q0 + j, ag, qg[j], ax, qx[j], t)) return true;
        }
      }
    }
  }
  return false;
}

// Core cell A, one lane: the stencil cells above A (each unordered pair is
// taken by its lower cell) with core points in another component, `sel`, and
// which of those pairs have a heavy cell, `heavy`, by slot of A's own row and
// the rows above it.  (Deciding them here held the lanes of the listing at 5
// waves per SIMD with 32 spilled registers: 158 us on the 4 M point 3-D
// workload, against 65 + 24 with k_far_pairs.)
constexpr int kFarRows = Win<3>::rows - Win<3>::own;
struct FarCell {
  uint2 row[kFarRows];
  uint32_t sel[kFarRows], heavy[kFarRows];
};
template <int D>
__device__ __forceinline__ void far_cell(const Dev& d, int32_t A, int32_t compA, bool heavyA,
                                         FarCell& f) {
  constexpr int NU = Win<D>::rows - Win<D>::own;  // own row and those above
  constexpr int nl = Win<D>::nl;
  const int local = (int)(d.cell_zl[A] & (nl - 1));
  const RowsOf rows = rows_of(d, A);
#pragma unroll
  for (int j = 0; j < NU; ++j) f.row[j] = rows[Win<D>::own + j];
  // cells with core points in another component, by place in each window's
  // cells (cell_comp is -1 for a cell without core points); the windows'
  // cells are consecutive, so their components are loaded four at a time (up
  // to three entries past the last cell may be read: the array has them)
  uint32_t other[NU];
#pragma unroll
  for (int j = 0; j < NU; ++j) {
    const int n = row_cells(f.row[j]);
    const int32_t* cp = d.cell_comp + (int64_t)f.row[j].x;
    other[j] = 0u;
#pragma unroll
    for (int q = 0; q < Win<D>::slots; q += 4)
      if (q < n) {
        const int32_t k[4] = {cp[q], cp[q + 1], cp[q + 2], cp[q + 3]};
#pragma unroll
        for (int u = 0; u < 4; ++u)
          other[j] |= (k[u] >= 0 && k[u] != compA) ? 1u << (q + u) : 0u;
      }
    other[j] &= (1u << n) - 1u;
  }
#pragma unroll
  for (int j = 0; j < NU; ++j) {
    if (!other[j]) continue;
    const int r = Win<D>::own + j;
    const int a = D == 3 ? r / 3 - 1 : r - 1, b = D == 3 ? r % 3 - 1 : 0;
    uint32_t todo = f.row[j].y & row_valid<D>(a, b, local);
    if (j == 0) todo &= ~0u << (2 * nl + local + 1);  // above A in its own column
    while (todo) {
      const int s = __ffs(todo) - 1;
      todo &= todo - 1;
      const int place = __popc(f.row[j].y & ((1u << s) - 1u));
      if (!((other[j] >> place) & 1u)) continue;
      const int32_t B = (int32_t)f.row[j].x + place;
      f.sel[j] |= 1u << s;
      if (heavyA || d.cell_start[B + 1] - d.cell_start[B] > kHeavy) f.heavy[j] |= 1u << s;
    }
  }
}

// Stores the pairs of a wavefront's cells, `tot` in all, this lane's `mine` of
// them from number `first` on (its light or its heavy ones), and returns how
// many found room.  One atomic for the wavefront's pairs: the sub-list of its
// own first, then whichever have room, so that a list takes as many pairs as it
// holds from however few wavefronts, and a full one costs a single look at its
// counters.  k_far with an atomic for each pair, on the sub-list of the
// workgroup, and now: 2566 and 184 us on a 3-D lattice of 1 M points with eps
// 1.5 spacings, 948 and 115 on a 2-D one with eps one spacing, 61 and 45 on the
// 4 M point 3-D workload.
__device__ __forceinline__ int far_store(const PairList& L, const FarCell& f, int32_t A,
                                         bool heavy, int first, int mine, int tot) {
  const int lane = lane_id();
  int done = 0;
  int st = (int)((blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) & (kStripes - 1));
  unsigned long long tried = 0;
  for (;;) {
    long long at = 0;
    if (lane == 0)
      at = (long long)atomicAdd(&L.cnt[st * kStatStride], (unsigned long long)(tot - done));
    at = rl_l(at, 0);
    const long long room = (long long)L.cap - at;
    const int take = room <= 0 ? 0 : (room < tot - done ? (int)room : tot - done);
    if (take > 0 && mine > 0 && first < done + take && first + mine > done) {
      int2* to = L.data + st * L.cap + at;
      int k = first - done;
#pragma unroll
      for (int j = 0; j < kFarRows; ++j) {
        uint32_t m = f.sel[j] & (heavy ? f.heavy[j] : ~f.heavy[j]);
        while (m) {
          const int s = __ffs(m) - 1;
          m &= m - 1;
          if (k >= 0 && k < take) to[k] = make_int2(A, slot_cell(f.row[j], s));
          ++k;
        }
      }
    }
    done += take;
    if (done == tot) break;
    tried |= 1ull << st;
    const unsigned long long open =
        ballot((long long)__hip_atomic_load(&L.cnt[lane * kStatStride], __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT) < (long long)L.cap) &
        ~tried;
    if (!open) break;
    const unsigned long long above = open & (~0ull << st);  // (st itself is not open)
    st = __ffsll((long long)(above ? above : open)) - 1;
  }
  return done;
}

// A listed cell of Dev::far_over: its index, and which pairs were not stored.
constexpr int32_t kOverLight = 1 << 28, kOverHeavy = 1 << 29, kOverCell = kOverLight - 1;
static_assert(kMaxCells <= (1LL << 28), "a cell index has 28 bits");

__global__ __launch_bounds__(256, 8) void k_far(Dev d) {
  if (abandoned(d)) return;
  __shared__ long long s_pre[kStripes + 1];
  const long long n = slist_prefix(d.core_cells, s_pre);
  for (long long i0 = (long long)blockIdx.x * 256; i0 < n; i0 += (long long)gridDim.x * 256) {
    const long long i = i0 + threadIdx.x;
    const bool act = i < n;
    int32_t A = 0, comp = 0;
    int dim = 0;
    bool heavy = false;
    if (act) {
      A = slist_at(d.core_cells, s_pre, i);
      dim = inst_of_cell(d, A)->dim;
      comp = d.cell_comp[A];
      heavy = d.cell_start[A + 1] - d.cell_start[A] > kHeavy;
    }
    FarCell f;
#pragma unroll
    for (int j = 0; j < kFarRows; ++j) {
      f.row[j] = make_uint2(0u, 0u);
      f.sel[j] = f.heavy[j] = 0u;
    }
    DCLUST_BY_DIM(act, dim, far_cell<3>(d, A, comp, heavy, f), far_cell<2>(d, A, comp, heavy, f));
    int nl = 0, nh = 0;
#pragma unroll
    for (int j = 0; j < kFarRows; ++j) {
      nl += __popc(f.sel[j] & ~f.heavy[j]);
      nh += __popc(f.heavy[j]);
    }
    if (!ballot((nl | nh) != 0)) continue;
    // (a lane has at most 100 pairs, so both counts of the wave fit one word)
    const uint32_t both = (uint32_t)nl | (uint32_t)nh << 16;
    const uint32_t incl = wave_incl_scan(both), before = incl - both, all = rl_u(incl, 63);
    const int tl = (int)(all & 0xffffu), th = (int)(all >> 16);
    const int fl = (int)(before & 0xffffu), fh = (int)(before >> 16);
    const int sl = tl ? far_store(d.far_light, f, A, false, fl, nl, tl) : 0;
    const int sh = th ? far_store(d.far_heavy, f, A, true, fh, nh, th) : 0;
    // cells with pairs that found no room
    const int32_t left = (nl && fl + nl > sl ? kOverLight : 0) | (nh && fh + nh > sh ? kOverHeavy : 0);
    if (const unsigned long long m = ballot(left != 0)) {
      const int st = blockIdx.x & (kStripes - 1);
      long long at = 0;
      if (lane_id() == 0)
        at = (long long)atomicAdd(&d.far_over.cnt[st * kStatStride],
                                  (unsigned long long)__popcll(m));
      at = rl_l(at, 0);
      if (left) d.far_over.data[st * d.far_over.cap + at + mbcnt(m)] = A | left;
    }
  }
}

// Is some core point of A joined to some core point of B?  The whole
// wavefront: 64 points of A and 64 of B at a time, one of each per lane.
// B's points beyond eps of the box of A's are dropped, then A's points
// beyond eps of the box of those left; the rest are tried in turn (broadcast
// from their lane) against all lanes, until one joins.
template <int D, bool F32>
__device__ bool wave_joined(const Dev& d, const Par& P, int32_t A, int32_t B, Tally& t) {
  const int lane = lane_id();
  const int32_t a0 = d.cell_start[A], a1 = d.cell_start[A + 1];
  const int32_t b0 = d.cell_start[B], b1 = d.cell_start[B + 1];
  for (int32_t ac = a0; ac < a1; ac += 64) {
    const int32_t p = ac + lane < a1 ? ac + lane : a0;
    const bool av = ac + lane < a1 && d.core[p];
    if (!ballot(av)) continue;
    uint32_t ag[D], alo[D], ahi[D];
    double ax[D];
#pragma unroll
    for (int k = 0; k < D; ++k) {
      ag[k] = d.G[3 * (int64_t)p + k];
      ax[k] = F32 ? 0.0 : d.X[3 * (int64_t)p + k];
    }
    // (coordinates of one cell's points do not wrap against each other)
#pragma unroll
    for (int k = 0; k < D; ++k) {
      alo[k] = wave_min(av ? ag[k] : 0xffffffffu);
      ahi[k] = wave_max(av ? ag[k] : 0u);
    }
    for (int32_t bc = b0; bc < b1; bc += 64) {
      const int32_t q = bc + lane < b1 ? bc + lane : b0;
      uint32_t bg[D], blo[D], bhi[D];
      double bx[D];
#pragma unroll
      for (int k = 0; k < D; ++k) {
        bg[k] = d.G[3 * (int64_t)q + k];
        bx[k] = F32 ? 0.0 : d.X[3 * (int64_t)q + k];
      }
      const bool bv = bc + lane < b1 && d.core[q] && !(d2box<D>(bg, alo, ahi) > P.d2_out);
      if (!ballot(bv)) continue;
#pragma unroll
      for (int k = 0; k < D; ++k) {
        blo[k] = wave_min(bv ? bg[k] : 0xffffffffu);
        bhi[k] = wave_max(bv ? bg[k] : 0u);
      }
      unsigned long long m = ballot(av && !(d2box<D>(ag, blo, bhi) > P.d2_out));
      while (m) {
        const int l = __ffsll((long long)m) - 1;
        m &= m - 1;
        uint32_t ug[D];
        double ux[D];
#pragma unroll
        for (int k = 0; k < D; ++k) {
          ug[k] = rl_u(ag[k], l);
          ux[k] = F32 ? 0.0 : rl_d(ax[k], l);
        }
        bool hit = false;
        if (bv) {
          ++t.eval;
          hit = edge_pair<D, F32>(d, P, ac + l, q, ug, bg, ux, bx, t);
        }
        if (ballot(hit)) return true;
      }
    }
  }
  return false;
}

// Prefix of a pair list's sub-list lengths (as stored) in LDS.
__device__ __forceinline__ long long pairs_prefix(const PairList& L, long long* s_pre) {
  if (threadIdx.x < kStripes) {
    const long long v = (long long)L.cnt[threadIdx.x * kStatStride];
    const long long incl = wave_incl_scan(v < L.cap ? v : (long long)L.cap);
    s_pre[threadIdx.x + 1] = incl;
    if (threadIdx.x == 0) s_pre[0] = 0;
  }
  __syncthreads();
  return s_pre[kStripes];
}
__device__ __forceinline__ int2 pairs_at(const PairList& L, const long long* s_pre, long long i) {
  int lo = 0, hi = kStripes - 1;  // last sub-list whose range starts at or before i
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (s_pre[mid] <= i) lo = mid; else hi = mid - 1;
  }
  return L.data[(int64_t)lo * L.cap + (i - s_pre[lo])];
}

// Offset of cell B from cell A of its stencil along axis k (the cells'
// coordinates modulo 8 are the top bits of their points').
__device__ __forceinline__ int cell_offset(const uint4& a, const uint4& b, int k) {
  const uint32_t x = k == 0 ? a.x : (k == 1 ? a.y : a.z);
  const uint32_t y = k == 0 ? b.x : (k == 1 ? b.y : b.z);
  return (int32_t)(((y >> kFixBits) - (x >> kFixBits)) << kFixBits) >> kFixBits;
}

// One pair, one lane: decided exactly unless its components have been united
// meanwhile; joined, they are united (lock-free union-find).
template <bool F32>
__device__ __forceinline__ void far_light(const Dev& d, int32_t A, int32_t B, Tally& t,
                                          long long& freeb, long long& joins) {
  const Inst& I = *inst_of_cell(d, A);
  const int32_t qs = d.cell_start[A], qe = d.cell_start[A + 1];
  const int32_t b0 = d.cell_start[B], b1 = d.cell_start[B + 1];
  const bool allc = d.cell_ncore[A] == qe - qs;
  const uint4 ra4 = d.rep[A], rb4 = d.rep[B];
  const int32_t ra = uf_find_cached(d.parent, d.cell_comp[A]);
  const int32_t rb = uf_find_cached(d.parent, d.cell_comp[B]);
  if (ra == rb) return;
  const Par P(I);
  const int o0 = cell_offset(ra4, rb4, 0), o1 = cell_offset(ra4, rb4, 1);
  const bool j =
      I.dim == 3 ? cells_joined<3, F32>(d, P, qs, qe, allc, b0, b1, o0, o1,
                                        cell_offset(ra4, rb4, 2), t, freeb)
                 : cells_joined<2, F32>(d, P, qs, qe, allc, b0, b1, o0, 0, o1, t, freeb);
  if (j) {
    uf_union(d.parent, ra, rb);
    ++joins;
  }
}

// One pair, the whole wavefront (wave-uniform: every lane walks the same path,
// lane 0's roots are taken).
template <bool F32>
__device__ __forceinline__ void far_heavy(const Dev& d, int32_t A, int32_t B, Tally& t,
                                          long long& joins) {
  const int32_t ra = rfl_i(uf_find_cached(d.parent, d.cell_comp[A]));
  const int32_t rb = rfl_i(uf_find_cached(d.parent, d.cell_comp[B]));
  if (ra == rb) return;
  const Inst& I = *inst_of_cell(d, A);
  const Par P(I);
  const bool j = I.dim == 3 ? wave_joined<3, F32>(d, P, A, B, t)
                            : wave_joined<2, F32>(d, P, A, B, t);
  if (j && lane_id() == 0) {
    uf_union(d.parent, ra, rb);
    ++joins;
  }
}

// The light or the heavy pairs of core cell A (when a list had no room for
// all of them), in turn.
template <int D, typename F>
__device__ __forceinline__ void far_cell_pairs(const Dev& d, int32_t A, bool heavy,
                                               const F& decide) {
  const int local = (int)(d.cell_zl[A] & (Win<D>::nl - 1));
  const int32_t comp = d.cell_comp[A];
  const bool heavyA = d.cell_start[A + 1] - d.cell_start[A] > kHeavy;
  for (int r = Win<D>::own; r < Win<D>::rows; ++r) {
    const uint2 row = rows_of(d, A)[r];
    uint32_t todo = row.y & (D == 3 ? row_valid<3>(r / 3 - 1, r % 3 - 1, local)
                                    : row_valid<2>(r - 1, 0, local));
    while (todo) {
      const int32_t B = slot_cell(row, __ffs(todo) - 1);
      todo &= todo - 1;
      if (B <= A || d.cell_comp[B] < 0 || d.cell_comp[B] == comp) continue;
      if ((heavyA || d.cell_start[B + 1] - d.cell_start[B] > kHeavy) == heavy) decide(B);
    }
  }
}

// The listed pairs: light ones one lane each, those with a heavy cell one
// wavefront each.  Then the cells whose pairs found their list full, in the
// same way, a cell's pairs one after the other: the unions of the first then
// settle most of the rest.  (Two sheets of 100 k points in 288 cells, just over
// eps apart: 2.1 s when few sub-lists took all pairs and a lane each decided
// those of a cell again, 69 us now.)
template <bool F32>
__global__ __launch_bounds__(256, 4) void k_far_pairs(Dev d) {
  if (abandoned(d)) return;
  __shared__ long long s_pre[kStripes + 1];
  Tally t;
  long long freeb = 0, joins = 0;
  const long long nl = pairs_prefix(d.far_light, s_pre);
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < nl;
       i += (long long)gridDim.x * 256) {
    const int2 pr = pairs_at(d.far_light, s_pre, i);
    far_light<F32>(d, pr.x, pr.y, t, freeb, joins);
  }
  __syncthreads();  // the prefix is rewritten
  const long long nh = pairs_prefix(d.far_heavy, s_pre);
  for (long long i = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); i < nh;
       i += (long long)gridDim.x * 4) {
    const int2 pr = pairs_at(d.far_heavy, s_pre, i);
    far_heavy<F32>(d, rfl_i(pr.x), rfl_i(pr.y), t, joins);
  }
  __syncthreads();
  const long long no = slist_prefix(d.far_over, s_pre);
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < no;
       i += (long long)gridDim.x * 256) {
    const int32_t e = slist_at(d.far_over, s_pre, i), A = e & kOverCell;
    if (!(e & kOverLight)) continue;
    const auto light = [&](int32_t B) { far_light<F32>(d, A, B, t, freeb, joins); };
    if (inst_of_cell(d, A)->dim == 3)
      far_cell_pairs<3>(d, A, false, light);
    else
      far_cell_pairs<2>(d, A, false, light);
  }
  for (long long i = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); i < no;
       i += (long long)gridDim.x * 4) {
    const int32_t e = rfl_i(slist_at(d.far_over, s_pre, i)), A = e & kOverCell;
    if (!(e & kOverHeavy)) continue;
    const auto heavy = [&](int32_t B) { far_heavy<F32>(d, A, rfl_i(B), t, joins); };
    if (inst_of_cell(d, A)->dim == 3)
      far_cell_pairs<3>(d, A, true, heavy);
    else
      far_cell_pairs<2>(d, A, true, heavy);
  }
  stat_add(d, C_BAND, t.band);
  stat_add(d, C_ASYM, t.asym);
  stat_add(d, C_FAR_TESTS, t.eval);
  stat_add(d, C_ADJ_FREE, freeb);
  stat_add(d, C_FAR_JOINS, joins);
}

// Final roots of the near components (the only component ids) after the
// unions across their borders, and their minima moved to them.  The walk
// writes nothing but each near root's own entry: a path-halving write of
// another thread's walk could otherwise replace a root that its owner has just
// stored with an inner ancestor, and a later read of "the root" would get
// that.  (uf_order keeps the walks short, so no compressing pass precedes.)
__global__ __launch_bounds__(256) void k_roots_final(Dev d) {
  if (abandoned(d)) return;
  const Stripe L(d.near_roots);
  for (int64_t i = L.first(256) + threadIdx.x; i < L.n; i += L.step(256)) {
    const int32_t c = L.data[i];
    const int32_t m = d.compmin[c];
    const int32_t r = uf_root(d.parent, c);
    d.parent[c] = r;
    if (r != c && m < d.compmin[r]) atomicMin(&d.compmin[r], m);
  }
}

// ---------------------------------------------------------------- expand --
// Persistent expansion pass.  Wave w scans its own contiguous segment of
// the cells for unclaimed cells with core points and starts a new chain at
// each (device-side seeding; the reference pops host-side seeds,
// dbscan.cu:142-160); it also drains the correction queue left by the
// previous pass.  A wave pops up to 64 cells of its list at once, one per
// lane; lane l walks the adjacency bits of its cell: an unclaimed neighbour
// is claimed for the cell's chain (CAS) and pushed, a neighbour of another
// chain is a collision pair.  After `budget` cells a wave hands its list to
// the next pass and exits, so one long chain cannot hold a pass; a wave also
// exits when its list is empty and no seed source is left.  Every wave
// reaches the end of the kernel: there is no inter-wave waiting.
constexpr int kSeen = 256;   // per-wave table of recently recorded collision pairs

// The cells one wave popped in a round (one per lane).
struct PopStage {
  uint2 rows[kMaxRows][64];  // windows
  uint32_t mask[64];         // near bits
  int32_t own[64];           // chain
  int32_t pre[64];           // exclusive prefix of the mask bit counts
  uint8_t kind[64];          // place in the block (bits 0-1), 2-D (bit 2)
};

__global__ __launch_bounds__(256) void k_expand(Dev d, int pass, int S, int budget) {
  extern __shared__ int32_t s_lists[];
  __shared__ unsigned long long s_seen[4][kSeen];
  __shared__ uint8_t s_tag[4][kSeen];  // per-wave dedup slots of one step
  __shared__ PopStage s_pop[4];         // per-wave popped cells of a round
  if (d.ctl[C_IDLE] || abandoned(d)) return;
  const int lane = lane_id(), wv = threadIdx.x >> 6;
  const int nwb = blockDim.x >> 6;
  const int64_t gw = (int64_t)xcd_block(blockIdx.x, gridDim.x) * nwb + wv;
  const int64_t W = (int64_t)gridDim.x * nwb;
  const int32_t C = (int32_t)d.ctl[C_NCELL];
  int32_t* list = s_lists + wv * S;
  unsigned long long* seen = s_seen[wv];
  uint8_t* tag = s_tag[wv];
  PopStage& pst = s_pop[wv];
  int32_t* qout = d.q[(pass + 1) & 1];
  unsigned long long* qout_n = (unsigned long long*)&d.ctl[C_Q0_N + ((pass + 1) & 1)];
  const int32_t* qin = d.q[pass & 1];
  unsigned long long* qin_head = (unsigned long long*)&d.ctl[C_Q0_HEAD + (pass & 1)];
  const long long qn = pass > 0 ? d.ctl[C_Q0_N + (pass & 1)] : 0;
  bool qlive = qn > 0;
  const int pcap = d.pair_per;
  int2* pbuf = d.pairs + gw * (int64_t)pcap;
  const int pc0 = rfl_i(d.pair_cnt[gw]);  // pairs recorded by earlier passes
  int pc = pc0;
  for (int i = lane; i < kSeen; i += 64) seen[i] = ~0ull;
  wave_sync();
  const unsigned long long t_begin = __builtin_amdgcn_s_memrealtime();
  // the seeding cursor over this wave's segment of cells persists across passes
  // (cell indices, below 2^31; the per-pass counters are bounded by the
  // pop budget: 32-bit, which keeps the wave-uniform state in fewer
  // scalar registers)
  int32_t seg = (int32_t)d.seg_pos[gw];
  const int32_t seg_end = (int32_t)((int64_t)C * (gw + 1) / W);
  int left = budget;
  int sl = 0;  // seed-list length (wave-uniform)
  int pops = 0, ovf = 0, edges = 0, seeds = 0, rounds = 0;
  int32_t cur = -1;    // chain of the cells in the list when not mixed
  bool mixed = false;  // the list holds queue cells (chains read per cell)
  for (;;) {
    if (left <= 0) {
      if (sl > 0) {
        long long base = 0;
        if (lane == 0) base = (long long)atomicAdd(qout_n, (unsigned long long)sl);
        base = __shfl(base, 0, 64);
        for (int i = lane; i < sl; i += 64) qout[base + i] = list[i];
      }
      break;
    }
    if (sl == 0) {
      bool got = false;
      if (qlive) {
        const int take = S < 64 ? S : 64;  // a refill fits the seed list
        long long base = 0;
        if (lane == 0) base = (long long)atomicAdd(qin_head, (unsigned long long)take);
        base = __shfl(base, 0, 64);
        if (base < qn) {
          const int cnt = (int)((qn - base) < take ? (qn - base) : take);
          if (lane < cnt) list[lane] = qin[base + lane];
          sl = cnt;
          got = true;
          mixed = true;  // queue cells: chains of other waves
        } else {
          qlive = false;
        }
      }
      while (!got && seg < seg_end) {
        const int32_t i = seg + lane;
        // both loads together (seg < seg_end, so seg is a cell)
        const int32_t ic = i < seg_end ? i : seg;
        const int32_t nco = d.cell_ncore[ic], lb = d.cell_label[ic];
        const bool cand = i < seg_end && nco > 0 && lb == kUnclaimed;
        unsigned long long m = ballot(cand);
        while (m) {
          const int l = __ffsll((long long)m) - 1;
          int ok = 0;
          if (lane == 0) {
            // a chain is named by its seed cell: unique, below the cell
            // count, and no shared counter to contend on
            const int32_t id = (int32_t)(seg + l);
            ok = atomicCAS(&d.cell_label[seg + l], kUnclaimed, id) == kUnclaimed;
          }
          ok = __shfl(ok, 0, 64);
          if (ok) {
            if (lane == 0) list[0] = (int32_t)(seg + l);
            ++seeds;
            sl = 1;
            got = true;
            cur = (int32_t)(seg + l);
            mixed = false;
            seg = seg + l + 1;
            break;
          }
          m &= m - 1;
        }
        if (!got) seg += 64;
      }
      if (!got) break;
      wave_sync();
    }
    // pop the top P cells, one per lane
    const int P = sl < 64 ? (sl < left ? sl : left) : (64 < left ? 64 : left);
    const bool act = lane < P;
    const int32_t A = act ? list[sl - P + lane] : 0;
    wave_sync();  // popped before the pushes below overwrite the slots
    sl -= P;
    left -= P;
    pops += P;
    ++rounds;
    int32_t own = 0;
    uint32_t m0 = 0u;
    int dim = 3;
    if (act) {
      // A list filled only by this wave's seeding and pushes holds cells of
      // its current chain alone (a new chain is seeded only into an empty
      // list).  After a refill from the queue the chain is read: coherently,
      // since the claim may have been made moments ago on another XCD, whose
      // L2 is not coherent with this one for plain loads.
      own = mixed ? __hip_atomic_load(&d.cell_label[A], __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT)
                  : cur;
      m0 = d.amask[A];
      dim = inst_of_cell(d, A)->dim;
    }
    // the popped cells' chains, masks and windows go to LDS (the windows
    // loaded together with the label and mask), and their adjacency bits are
    // dealt out evenly: item t of the round is bit k of the mask of lane
    // src, where src is the last lane whose bit prefix is at most t; a round
    // then takes ceil(bits / (64 T)) steps instead of the most bits of one
    // lane / T
    {
      // all nine loads in flight before the first LDS write
      const RowsOf rows = rows_of(d, A);
      uint2 rv[kMaxRows];
#pragma unroll
      for (int r = 0; r < kMaxRows; ++r)
        rv[r] = act && (dim == 3 || r < 3) ? rows[r] : make_uint2(0u, 0u);
      pst.kind[lane] = (uint8_t)(local_of(d, A, dim) | (dim == 3 ? 0 : 4));
#pragma unroll
      for (int r = 0; r < kMaxRows; ++r) pst.rows[r][lane] = rv[r];
    }
    const int nb = __popc(m0);
    edges += nb;
    const int incl = wave_incl_scan(nb);
    const int total = rfl_i(__shfl(incl, 63, 64));
    pst.own[lane] = own;
    pst.mask[lane] = m0;
    pst.pre[lane] = incl - nb;
    wave_sync();
    constexpr int T = 8;  // items per lane step
    for (int base = 0; base < total; base += 64 * T) {
      // sub-steps of 64 items that hold any (wave-uniform: a small round,
      // the usual case late in a chain, skips the empty ones)
      const int nsub = (total - base + 63) >> 6 < T ? (total - base + 63) >> 6 : T;
      int32_t tg[T], ow[T];
      bool v[T];
#pragma unroll
      for (int j = 0; j < T; ++j) {
        v[j] = false;
        tg[j] = 0;
        ow[j] = 0;
        if (j >= nsub) continue;
        const int t = base + j * 64 + lane;
        v[j] = t < total;
        int src = 0;
#pragma unroll
        for (int st = 32; st >= 1; st >>= 1)
          if (pst.pre[src + st] <= t) src += st;
        // bit k of the source mask: its k-th set bit
        int k = t - pst.pre[src];
        uint32_t m = pst.mask[src];
        int b = 0;
#pragma unroll
        for (int w = 16; w >= 1; w >>= 1) {
          const int c = __popc(m & ((1u << w) - 1u));
          if (k >= c) {
            k -= c;
            m >>= w;
            b += w;
          }
        }
        if (v[j]) {
          const int kind = pst.kind[src];
          int row, slot;
          if (kind < 4)
            near_slot<3>(b, kind, row, slot);
          else
            near_slot<2>(b, kind & 3, row, slot);
          tg[j] = slot_cell(pst.rows[row][src], slot);
        }
        ow[j] = pst.own[src];
      }
      // a plain load can only be stale as kUnclaimed (a label is written
      // once), so only those cells pay for a CAS
      int32_t lab[T];
#pragma unroll
      for (int j = 0; j < T; ++j) lab[j] = (j < nsub && v[j]) ? d.cell_label[tg[j]] : ow[j];
      // the claims are all issued before any result is used, so that they
      // are in flight together
      bool cl[T], need[T];
      int32_t old[T];
#pragma unroll
      for (int j = 0; j < T; ++j) {
        need[j] = j < nsub && v[j] && lab[j] == kUnclaimed;
        old[j] = lab[j];
      }
#pragma unroll
      for (int j = 0; j < T; ++j)
        if (need[j]) old[j] = atomicCAS(&d.cell_label[tg[j]], kUnclaimed, ow[j]);
#pragma unroll
      for (int j = 0; j < T; ++j) {
        cl[j] = need[j] && old[j] == kUnclaimed;
        lab[j] = cl[j] ? ow[j] : old[j];
      }
#pragma unroll
      for (int j = 0; j < T; ++j) {
        if (j >= nsub) break;
        // pushes: one slot range per step
        const unsigned long long mc = ballot(cl[j]);
        if (mc) {
          const int pos = sl + mbcnt(mc);
          if (cl[j]) {
            if (pos < S) {
              list[pos] = tg[j];
            } else {
              const unsigned long long qi = atomicAdd(qout_n, 1ull);
              qout[qi] = tg[j];
              ++ovf;
            }
          }
          sl += __popcll(mc);
          sl = sl < S ? sl : S;
        }
        // collisions, recorded by all lanes at once: a pair already in the
        // wave's table of recent pairs is skipped; among the lanes of this
        // step with the same pair, the one whose id survives in the tag slot
        // of the pair's hash records it (a lane whose hash slot was won by a
        // different pair records its own; a rare duplicate is harmless)
        const bool coll = v[j] && lab[j] != ow[j];
        if (ballot(coll)) {
          const unsigned long long key =
              ((unsigned long long)(uint32_t)ow[j] << 32) | (uint32_t)lab[j];
          const int h =
              (int)(((uint32_t)ow[j] * 0x9E3779B1u ^ (uint32_t)lab[j] * 0x85EBCA6Bu) >> 24);
          bool nw = coll && seen[h] != key;
          if (nw) tag[h] = (uint8_t)lane;
          wave_sync();
          const int w = nw ? (int)tag[h] : lane;
          const uint32_t wlo = (uint32_t)__shfl((int)(uint32_t)key, w, 64);
          const uint32_t whi = (uint32_t)__shfl((int)(uint32_t)(key >> 32), w, 64);
          if (nw && w != lane && (((unsigned long long)whi << 32) | wlo) == key) nw = false;
          const unsigned long long mn = ballot(nw);
          if (nw) {
            seen[h] = key;
            const int slot = pc + (int)mbcnt(mn);
            if (slot < pcap)
              pbuf[slot] = make_int2(ow[j], lab[j]);
            else
              uf_union(d.parent, ow[j], lab[j]);  // buffer full: merge inline
          }
          pc += __popcll(mn);
        }
      }
    }
    wave_sync();
  }
  if (lane == 0) {
    // device clock -> microseconds of this wave's life
    const unsigned long long us = (__builtin_amdgcn_s_memrealtime() - t_begin) / kClockMHz;
    d.pair_cnt[gw] = pc;
    d.seg_pos[gw] = seg;
    if (seg < seg_end) atomicAdd((unsigned long long*)&d.ctl[C_SEGS_LEFT], 1ull);
    if (pc > pc0) atomicAdd((unsigned long long*)&d.ctl[C_NPAIR], (unsigned long long)(pc - pc0));
    atomicAdd((unsigned long long*)&d.ctl[C_BUSY_SUM], us);
    atomicMax((unsigned long long*)&d.ctl[C_BUSY_MAX], us);
    atomicAdd((unsigned long long*)&d.ctl[C_POPS], (unsigned long long)pops);
    atomicMax((unsigned long long*)&d.ctl[C_POPS_MAX], (unsigned long long)pops);
    atomicMax((unsigned long long*)&d.ctl[C_SEEDS_MAX], (unsigned long long)seeds);
    atomicMax((unsigned long long*)&d.ctl[C_ROUNDS_MAX], (unsigned long long)rounds);
    if (pops) atomicMax((unsigned long long*)&d.ctl[C_LASTPASS], (unsigned long long)(pass + 1));
  }
  stat_add(d, C_OVF, ovf);
  stat_add(d, C_EDGES, edges);
  stat_add(d, C_NCHAIN, lane == 0 ? seeds : 0);  // seeds is wave-uniform
}



// Resets the counters of the queue that pass `pass` fills and of the head
// of the queue it drains, and marks the pass idle when nothing is pending.
__global__ void k_pass_prep(Dev d, int pass) {
  // nothing left by the previous pass: the waves of this one return at once
  d.ctl[C_IDLE] = pass > 0 && d.ctl[C_Q0_N + (pass & 1)] == 0 && d.ctl[C_SEGS_LEFT] == 0;
  d.ctl[C_Q0_N + ((pass + 1) & 1)] = 0;
  d.ctl[C_Q0_HEAD + (pass & 1)] = 0;
  d.ctl[C_SEGS_LEFT] = 0;
}

// After a pass: queue entries no wave took (every wave spent its budget)
// are appended to the queue of the next pass.  One block.  With `check` =
// the number of passes (after the last pass of a captured run), work still
// pending afterwards (queue or seeding segments) marks the run as abandoned,
// and the kernels after the expansion return at once (the host runs the call
// again).
__global__ __launch_bounds__(256) void k_pass_carry(Dev d, int pass, int check) {
  __shared__ long long s_base;
  long long qn = 0, head = 0;
  if (!abandoned(d) && pass > 0) {
    qn = d.ctl[C_Q0_N + (pass & 1)];
    head = d.ctl[C_Q0_HEAD + (pass & 1)];
  }
  if (head < qn) {  // block-uniform: every thread read the same two counters
    if (threadIdx.x == 0)
      s_base = (long long)atomicAdd((unsigned long long*)&d.ctl[C_Q0_N + ((pass + 1) & 1)],
                                    (unsigned long long)(qn - head));
    __syncthreads();
    const int32_t* qin = d.q[pass & 1];
    int32_t* qout = d.q[(pass + 1) & 1];
    for (long long i = head + threadIdx.x; i < qn; i += blockDim.x)
      qout[s_base + (i - head)] = qin[i];
  }
  if (check > 0 && threadIdx.x == 0) {
    // coherent loads: the add above went to L2, past this CU's cache
    const long long left = __hip_atomic_load(&d.ctl[C_Q0_N + (check & 1)], __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
    const long long segs = __hip_atomic_load(&d.ctl[C_SEGS_LEFT], __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
    if (left != 0 || segs != 0) d.ctl[C_ABANDON] = 1;
  }
}

// ----------------------------------------------------------------- merge --
// Chain ids are seed cell indices.  When the id space fits in LDS (up to
// 32768 cells), one workgroup merges every recorded pair on an LDS copy of
// the chain forest with LDS atomics and writes the flattened roots back.
// Otherwise the pairs are merged in global memory by the whole grid (the
// ids are spread over the cell range, so the unions rarely share a cache
// line).
constexpr int kLdsChains = 32768;  // 128 KiB of LDS (gfx950 allows 160 KiB per workgroup)
constexpr int kMergeChunk = 4096;  // pair buffers scanned at a time (16 KiB of LDS)

// number of expansion waves whose pair buffers are in use
__device__ __forceinline__ int64_t pair_waves(const Dev& d) { return d.pair_cap / d.pair_per; }

__global__ __launch_bounds__(1024) void k_merge_lds(Dev d) {
  if (abandoned(d)) return;
  __shared__ int32_t par[kLdsChains];
  __shared__ int32_t s_pre[kMergeChunk + 1];
  __shared__ int32_t s_wsum[16];
  const long long nc = chain_ids(d);
  if (nc > kLdsChains) return;
  // parent may already hold inline merges (pairs past a full buffer)
  for (int i = threadIdx.x; i < nc; i += blockDim.x) par[i] = d.parent[i];
  // the pair buffers of kMergeChunk expansion waves at a time: their counts
  // are scanned in LDS, then every thread takes pairs by flat index, so the
  // buffers are read in parallel
  const int64_t nw = pair_waves(d);
  const int per = d.pair_per;
  const int lane = lane_id(), wv = threadIdx.x >> 6;
  for (int64_t w0 = 0; w0 < nw; w0 += kMergeChunk) {
    const int nb = (int)((nw - w0) < kMergeChunk ? (nw - w0) : kMergeChunk);
    // per thread: kMergeChunk / 1024 consecutive buffers
    constexpr int kPer = kMergeChunk / 1024;
    int cnt[kPer];
    int sum = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int b = threadIdx.x * kPer + j;
      cnt[j] = b < nb ? min(d.pair_cnt[w0 + b], per) : 0;
      sum += cnt[j];
    }
    const int incl = wave_incl_scan(sum);
    if (lane == 63) s_wsum[wv] = incl;
    __syncthreads();
    int off = incl - sum;
    for (int w = 0; w < wv; ++w) off += s_wsum[w];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      s_pre[threadIdx.x * kPer + j] = off;
      off += cnt[j];
    }
    if (threadIdx.x == blockDim.x - 1) s_pre[kMergeChunk] = off;
    __syncthreads();
    const int tot = s_pre[kMergeChunk];
    // kBatch pairs per thread at a time: fixed-step searches for their
    // buffers, then their loads, all independent, before the unions
    constexpr int kBatch = 8;
    for (int f0 = 0; f0 < tot; f0 += (int)blockDim.x * kBatch) {
      int2 pr[kBatch];
#pragma unroll
      for (int j = 0; j < kBatch; ++j) {
        const int f = f0 + j * (int)blockDim.x + (int)threadIdx.x;
        // last buffer whose range starts at or before f (s_pre[0] = 0)
        int lo = 0;
#pragma unroll
        for (int step = kMergeChunk / 2; step >= 1; step >>= 1)
          if (s_pre[lo + step] <= f) lo += step;
        pr[j] = f < tot ? d.pairs[(w0 + lo) * per + (f - s_pre[lo])] : make_int2(0, 0);
      }
#pragma unroll
      for (int j = 0; j < kBatch; ++j) {
        lds_union(par, pr[j].x, pr[j].y);
      }
    }
    __syncthreads();  // s_pre is rewritten by the next chunk
  }
  for (int i = threadIdx.x; i < nc; i += blockDim.x) {
    int32_t r = i;
    while (par[r] != r) r = par[r];
    d.parent[i] = r;
  }
}

__global__ __launch_bounds__(256) void k_union_pairs(Dev d) {
  if (abandoned(d)) return;
  if (chain_ids(d) <= kLdsChains) return;
  const int64_t nw = pair_waves(d);
  const int64_t wid = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;
  const int64_t nwv = ((int64_t)gridDim.x * blockDim.x) >> 6;
  for (int64_t w = wid; w < nw; w += nwv) {
    const int cnt = min(d.pair_cnt[w], d.pair_per);
    for (int k = lane_id(); k < cnt; k += 64) {
      int2 p = d.pairs[w * d.pair_per + k];
      uf_union(d.parent, p.x, p.y);
    }
  }
}

__global__ __launch_bounds__(256) void k_flatten(Dev d) {
  if (abandoned(d)) return;
  const long long nc = chain_ids(d);
  if (nc <= kLdsChains) return;
  for (long long c = blockIdx.x * (long long)blockDim.x + threadIdx.x; c < nc;
       c += (long long)gridDim.x * blockDim.x)
    d.parent[c] = uf_find(d.parent, (int32_t)c);
}

// Points per thread step of the per-point relabel passes: each level of
// their dependent loads is issued for all of them before the next level,
// and nothing is stored until every load is done, so the latencies overlap.
constexpr int kRelU = 4;

// Keys of the core points (k_border, which reads them, gives the others
// theirs).
__global__ __launch_bounds__(256) void k_keys(Dev d) {
  if (abandoned(d)) return;
  for (int64_t i0 = blockIdx.x * (int64_t)(kRelU * 256); i0 < d.n;
       i0 += (int64_t)gridDim.x * (kRelU * 256)) {
    int64_t ic[kRelU];
    bool cr[kRelU];
    int32_t c[kRelU], o[kRelU], li[kRelU], pr[kRelU], k[kRelU];
#pragma unroll
    for (int u = 0; u < kRelU; ++u) {
      const int64_t i = i0 + u * 256 + threadIdx.x;
      ic[u] = i < d.n ? i : 0;
      cr[u] = i < d.n && d.core[ic[u]];
      c[u] = d.cell_of[ic[u]];
      o[u] = d.orig[ic[u]];
    }
    // (a core point's cell has a component; the others read entry 0)
#pragma unroll
    for (int u = 0; u < kRelU; ++u) li[u] = cr[u] ? d.cell_comp[c[u]] : 0;
#pragma unroll
    for (int u = 0; u < kRelU; ++u) pr[u] = d.parent[li[u]];
#pragma unroll
    for (int u = 0; u < kRelU; ++u) k[u] = d.compmin[pr[u]];
#pragma unroll
    for (int u = 0; u < kRelU; ++u) {
      if (cr[u]) {
        d.keyv[ic[u]] = k[u];
        if (o[u] == k[u]) atomicOr(&d.flag[k[u] >> 6], 1ull << (k[u] & 63));
      }
    }
  }
}

// ---------------------------------------------------------------- border --
// P(q -> p) for a core point q and a non-core point p, evaluated from the
// core point's side as its expansion in the reference oracle would.
template <int D, bool F32>
__device__ __forceinline__ bool pred_to(const Dev& d, const Par& P, int32_t q, int32_t p,
                                        const uint32_t* pg, const double* px, Tally& t) {
  double qx[D];
  if (F32) {
    uint32_t qg[D];
    load_g<D>(d, q, qg);
    const float s = d2fix<D>(qg, pg);
    if (s < P.d2_in) return true;
    if (s > P.d2_out) return false;
    t.band++;
    double ax[D];
    load_x<D, F32>(d, q, qx);
    load_x<D, F32>(d, p, ax);
    const bool ex = box_64<D>(qx, ax, P.eps) && d2_64<D>(qx, ax) <= P.eps2;
    t.flip += ex != (s <= P.d2_mid);
    return ex;
  }
  load_x<D, F32>(d, q, qx);
  return box_64<D>(qx, px, P.eps) && d2_64<D>(qx, px) <= P.eps2;
}

// Component key of a core cell.
__device__ __forceinline__ int32_t comp_key(const Dev& d, int32_t comp) {
  return d.compmin[d.parent[comp]];
}

// The smallest component key below `best` over the core points q of p's rows
// with P(q -> p): a cell without core points, or with a key that is no
// smaller, is passed over as a whole.
template <int D, bool F32>
__device__ int32_t border_scan(const Dev& d, const Par& P, int32_t p, int32_t c, int32_t best,
                               const uint32_t* pg, const double* px, Tally& t) {
  constexpr int NR = Win<D>::rows;
  const RowsOf rows = rows_of(d, c);
  // rows with a core cell among their first four cells, or with more cells:
  // the loads of all rows in flight together
  uint32_t todo = 0u;
  {
    uint2 row[NR];
    int32_t k[NR][4];
#pragma unroll
    for (int r = 0; r < NR; ++r) row[r] = rows[r];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int n = row_cells(row[r]);
#pragma unroll
      for (int u = 0; u < 4; ++u) k[r][u] = -1;
      if (n) {
        const int32_t* cp = d.cell_comp + (int64_t)row[r].x;
#pragma unroll
        for (int u = 0; u < 4; ++u) k[r][u] = cp[u];
      }
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int n = row_cells(row[r]);
      bool any = n > 4;
#pragma unroll
      for (int u = 0; u < 4; ++u) any |= u < n && k[r][u] >= 0;
      todo |= any ? 1u << r : 0u;
    }
  }
  while (todo) {
    const int r = __ffs(todo) - 1;
    todo &= todo - 1;
    const uint2 row = rows[r];
    const int n = row_cells(row);
    for (int i = 0; i < n; ++i) {
      const int32_t B = (int32_t)row.x + i;
      const int32_t comp = d.cell_comp[B];
      if (comp < 0 || B == c) continue;
      const int32_t key = comp_key(d, comp);
      if (key >= best) continue;
      const int32_t b1 = d.cell_start[B + 1];
      for (int32_t q = d.cell_start[B]; q < b1; ++q)
        if (d.core[q] && pred_to<D, F32>(d, P, q, p, pg, px, t)) {
          best = key;
          break;
        }
    }
  }
  return best;
}

// Smallest component key over the core points q with P(q -> p): the own
// cell (a clique), then the recorded neighbours, or the rows' core cells
// when there are no records.
template <int D, bool F32>
__device__ int32_t border_lane(const Dev& d, const Par& P, int32_t p, int32_t c, Tally& t,
                               long long& ovf) {
  const int32_t comp = d.cell_comp[c];
  const int n = (int)d.rec_n[p];
  int32_t best = comp >= 0 ? comp_key(d, comp) : kNoKey;
  uint32_t pg[D];
  double px[D];
  if (F32)
    load_g<D>(d, p, pg);
  else
    load_x<D, F32>(d, p, px);
  if (n >= kRecFew) {
    ovf += n == kRecNone;
    return border_scan<D, F32>(d, P, p, c, best, pg, px, t);
  }
  // four records at a time: their indices, then their core flags and keys,
  // each level of loads issued together
  const int32_t* rec = d.rec + p;
  for (int j0 = 0; j0 < n; j0 += 4) {
    int32_t q[4], k[4];
    bool cq[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) q[u] = j0 + u < n ? rec[(int64_t)(j0 + u) * d.n] : p;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      cq[u] = j0 + u < n && d.core[q[u]];
      k[u] = d.keyv[q[u]];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (cq[u] && k[u] < best && pred_to<D, F32>(d, P, q[u], p, pg, px, t)) best = k[u];
  }
  return best;
}

// One lane per non-core point (the list k_core fills; a wave's points are
// consecutive ones of one workgroup there, in cell order).
template <bool F32>
__global__ __launch_bounds__(256) void k_border(Dev d) {
  if (abandoned(d)) return;
  const Stripe L(d.border_pts);
  Tally t;
  long long ovf = 0, noise = 0;
  for (int64_t i0 = L.first(256); i0 < L.n; i0 += L.step(256)) {
    const int64_t i = i0 + threadIdx.x;
    const bool act = i < L.n;
    const int32_t p = act ? L.data[i] : 0;
    int32_t c = 0;
    int dim = 0;
    const Inst* I = d.inst;
    if (act) {
      c = d.cell_of[p];
      I = inst_of_cell(d, c);
      dim = I->dim;
    }
    int32_t best = kNoKey;
    const Par P(*I);
    DCLUST_BY_DIM(act, dim, (best = border_lane<3, F32>(d, P, p, c, t, ovf)),
                  (best = border_lane<2, F32>(d, P, p, c, t, ovf)));
    if (act) d.keyv[p] = best;
    noise += act && best == kNoKey;
  }
  stat_add(d, C_BAND, t.band);
  stat_add(d, C_FLIP, t.flip);
  stat_add(d, C_RECOVF, ovf);
  stat_add(d, C_NNOISE, noise);
}

// ------------------------------------------------------------ rank + out --
// Ranks of the clusters: the flags of their smallest core input indices are
// bits, so rank(k) = the flags before k's word (a scan over N/64 words: small
// enough to stay in L2 for the random reads of the labels, where one entry per
// point was not) + the bits below k in its word.
constexpr int kOutWindows = 512;  // windows of the labels, at most
constexpr int kOutPad = 16;       // a window's cursor has a cache line of its own
constexpr int kRankOne = 1 << 13;  // words that one workgroup ranks
constexpr int RK_T = 256;
constexpr int RK_I = 4;
constexpr int RK_TILE = RK_T * RK_I;  // words per workgroup

// (`cursor`: k_output_split's, started here, or null)
__global__ __launch_bounds__(RK_T) void k_rank_count(Dev d, uint32_t* cursor) {
  if (abandoned(d)) return;
  if (cursor && blockIdx.x == 0)
    for (int i = threadIdx.x; i < kOutWindows; i += RK_T) cursor[i * kOutPad] = 0;
  const int64_t nf = (d.n + 63) / 64, t0 = (int64_t)blockIdx.x * RK_TILE;
  int c = 0;
#pragma unroll
  for (int r = 0; r < RK_I; ++r) {
    const int64_t i = t0 + r * RK_T + threadIdx.x;
    if (i < nf) c += __popcll(d.flag[i]);
  }
  c = wave_sum(c);
  __shared__ int s[4];
  if (lane_id() == 0) s[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) d.scan_tmp[blockIdx.x] = s[0] + s[1] + s[2] + s[3];
}

__global__ __launch_bounds__(RK_T) void k_rank_write(Dev d) {
  if (abandoned(d)) return;
  const int64_t nf = (d.n + 63) / 64, t0 = (int64_t)blockIdx.x * RK_TILE;
  __shared__ int s_w[4];
  __shared__ int64_t s_p[4];
  // flags of the workgroups before (a count for 65536 points)
  int64_t pre = 0;
  for (int i = threadIdx.x; i < (int)blockIdx.x; i += RK_T) pre += d.scan_tmp[i];
  pre = wave_sum(pre);
  // RK_I consecutive words per thread
  int c[RK_I], sum = 0;
#pragma unroll
  for (int r = 0; r < RK_I; ++r) {
    const int64_t i = t0 + (int64_t)threadIdx.x * RK_I + r;
    c[r] = i < nf ? __popcll(d.flag[i]) : 0;
    sum += c[r];
  }
  const int incl = wave_incl_scan(sum), wv = threadIdx.x >> 6;
  if (lane_id() == 63) {
    s_w[wv] = incl;
    s_p[wv] = pre;
  }
  __syncthreads();
  int run = (int)(s_p[0] + s_p[1] + s_p[2] + s_p[3]) + incl - sum;
  for (int w = 0; w < wv; ++w) run += s_w[w];
#pragma unroll
  for (int r = 0; r < RK_I; ++r) {
    const int64_t i = t0 + (int64_t)threadIdx.x * RK_I + r;
    if (i < nf) d.rank[i] = run;
    run += c[r];
    if (i == nf - 1) d.ctl[C_NCLUST] = run;
  }
}

// The two in one for at most 2^19 points, a launch less: 4 us for 100 k points
// and 6 for 262 k where the two take 9, but 11 for 614 k and 16 for 1 M.
__global__ __launch_bounds__(1024) void k_rank_one(Dev d) {
  if (abandoned(d)) return;
  constexpr int W = kRankOne / 1024;
  const int nf = (int)((d.n + 63) / 64), w0 = threadIdx.x * W, wv = threadIdx.x >> 6;
  __shared__ int s_w[16];
  int c[W], sum = 0;
#pragma unroll
  for (int r = 0; r < W; ++r) c[r] = w0 + r < nf ? __popcll(d.flag[w0 + r]) : 0;
#pragma unroll
  for (int r = 0; r < W; ++r) sum += c[r];
  const int incl = wave_incl_scan(sum);
  if (lane_id() == 63) s_w[wv] = incl;
  __syncthreads();
  int run = incl - sum;
  for (int w = 0; w < wv; ++w) run += s_w[w];
#pragma unroll
  for (int r = 0; r < W; ++r) {
    if (w0 + r < nf) d.rank[w0 + r] = run;
    run += c[r];
  }
  if (threadIdx.x == 1023) d.ctl[C_NCLUST] = run;
}

// flags before input index k
__device__ __forceinline__ int32_t rank_of(const Dev& d, int64_t k) {
  return d.rank[k >> 6] + __popcll(d.flag[k >> 6] & ((1ull << (k & 63)) - 1ull));
}

// Labels of NI points from i0 on, RS apart, and their input indices (an index
// past the end reads point 0).
template <int NI, int RS>
__device__ __forceinline__ void point_labels(const Dev& d, int64_t i0, int32_t (&o)[NI],
                                            int32_t (&lab)[NI]) {
  int32_t k[NI], rb[NI];
  int64_t pb[NI];
#pragma unroll
  for (int u = 0; u < NI; ++u) {
    const int64_t ic = i0 + u * RS < d.n ? i0 + u * RS : 0;
    o[u] = d.orig[ic];
    k[u] = d.keyv[ic];
    pb[u] = inst_of_cell(d, d.ninst == 1 ? 0 : d.cell_of[ic])->pt_begin;
  }
#pragma unroll
  for (int u = 0; u < NI; ++u) {
    lab[u] = rank_of(d, k[u] == kNoKey ? 0 : k[u]);
    rb[u] = d.ninst == 1 ? 0 : rank_of(d, pb[u]);
  }
#pragma unroll
  for (int u = 0; u < NI; ++u) lab[u] = k[u] == kNoKey ? 0 : lab[u] - rb[u] + 1;
}

// A run's last kernel has a workgroup more that reads the counters back (`out`
// not null: in a launch of their own 5 us a call); it does so in an abandoned
// run too, where it is the only one that works.
__device__ __forceinline__ bool reads_back(const Dev& d, long long* out) {
  if (!out || blockIdx.x != gridDim.x - 1) return false;
  readback(d, out);
  return true;
}

__global__ __launch_bounds__(256) void k_output(Dev d, long long* out) {
  if (reads_back(d, out) || abandoned(d)) return;
  int32_t* labels = out_labels(d);
  const int G = out ? gridDim.x - 1 : gridDim.x;
  for (int64_t i0 = blockIdx.x * (int64_t)(kRelU * 256) + threadIdx.x; i0 - threadIdx.x < d.n;
       i0 += (int64_t)G * (kRelU * 256)) {
    int32_t o[kRelU], lab[kRelU];
    point_labels<kRelU, 256>(d, i0, o, lab);
#pragma unroll
    for (int u = 0; u < kRelU; ++u)
      if (i0 + u * 256 < d.n) labels[o[u]] = lab[u];
  }
}

// The labels of a large call in two steps.  Written one by one in sorted order
// each 4-byte label is a partial line of its own (32 M points: 815 us, 2.5 TB/s
// of 64-byte writes).  k_output_split sorts tiles of (input index, label) pairs
// by window of the labels in LDS and appends them window by window (the input
// indices are a permutation, so a window's place and size are known, and the
// order inside it does not matter); k_output_place writes each window on one
// XCD, whose L2 joins its lines.
//
// k_output against the two steps, us: 1 M points 14 / 20, 1.5 M 22 / 24, 4 M 74
// / 41, 7 M in a batch 101 / 98, 32 M 815 / 289.  A part is gathered from its
// whole window, so the windows stay below kOutWindow labels; larger calls
// (above 67 M points) keep the one step.
constexpr int kOutItems = 16;
constexpr int64_t kOutSplit = 1 << 21;
constexpr int64_t kOutWindow = 1 << 17;
__global__ __launch_bounds__(512, 4) void k_output_split(Dev d, int shift, uint32_t* cursor,
                                                      uint2* pairs) {
  if (abandoned(d)) return;
  constexpr int T = 512, NI = kOutItems;
  static_assert(T == kOutWindows, "a thread per window");
  __shared__ uint2 s_p[T * NI];
  __shared__ uint32_t s_cnt[T], s_dst[T], s_w[T / 64];
  const int tid = threadIdx.x, wv = tid >> 6;
  s_cnt[tid] = 0;
  const int64_t t0 = (int64_t)blockIdx.x * (T * NI);
  int32_t o[NI], lab[NI];
#pragma unroll
  for (int h = 0; h < NI; h += kRelU) {
    int32_t ho[kRelU], hl[kRelU];
    point_labels<kRelU, T>(d, t0 + tid + h * T, ho, hl);
#pragma unroll
    for (int u = 0; u < kRelU; ++u) {
      o[h + u] = ho[u];
      lab[h + u] = hl[u];
    }
  }
  __syncthreads();
  uint32_t at[NI];
#pragma unroll
  for (int u = 0; u < NI; ++u)
    at[u] = t0 + u * T + tid < d.n ? atomicAdd(&s_cnt[o[u] >> shift], 1u) : 0u;
  __syncthreads();
  const uint32_t c = s_cnt[tid];
  const uint32_t base = c ? atomicAdd(&cursor[tid * kOutPad], c) : 0u;
  const uint32_t inc = wave_incl_scan(c);
  if (lane_id() == 63) s_w[wv] = inc;
  __syncthreads();
  uint32_t lst = inc - c;
  for (int w = 0; w < wv; ++w) lst += s_w[w];
  s_cnt[tid] = lst;
  s_dst[tid] = ((uint32_t)tid << shift) + base - lst;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NI; ++u)
    if (t0 + u * T + tid < d.n)
      s_p[s_cnt[o[u] >> shift] + at[u]] = make_uint2((uint32_t)o[u], (uint32_t)lab[u]);
  __syncthreads();
  const int tn = (int)(d.n - t0 < T * NI ? d.n - t0 : T * NI);
#pragma unroll 4
  for (int u = 0; u < NI; ++u) {
    const int l = u * T + tid;
    if (l < tn) {
      const uint2 p = s_p[l];
      pairs[s_dst[p.x >> shift] + (uint32_t)l] = p;
    }
  }
}

// A workgroup gathers PART labels, a part of a window, in LDS and writes them
// in order (written from the pairs directly, the scattered 4-byte requests took
// 236 us on 32 M points).
template <int PART, int T>
__global__ __launch_bounds__(T) void k_output_place(Dev d, int shift, const uint2* pairs,
                                                    long long* out) {
  if (reads_back(d, out) || abandoned(d)) return;
  __shared__ int32_t s_l[PART];
  constexpr int U = 8;
  const int64_t first = (int64_t)xcd_runs<8>(blockIdx.x, out ? gridDim.x - 1 : gridDim.x) * PART;
  const int64_t w0 = first >> shift << shift;
  const int64_t w1 = w0 + (1LL << shift) < d.n ? w0 + (1LL << shift) : d.n;
  for (int64_t i0 = w0 + threadIdx.x; i0 < w1; i0 += T * U) {
    uint2 p[U];
#pragma unroll
    for (int u = 0; u < U; ++u) p[u] = pairs[i0 + u * T < w1 ? i0 + u * T : w0];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t l = p[u].x - (uint32_t)first;
      if (i0 + u * T < w1 && l < (uint32_t)PART) s_l[l] = (int32_t)p[u].y;
    }
  }
  __syncthreads();
  int32_t* labels = out_labels(d) + first;
  const int np = (int)(d.n - first < PART ? d.n - first : PART);
  for (int l = threadIdx.x; l < np; l += T) labels[l] = s_l[l];
}

// ------------------------------------------------------------- launchers --
// one lane per point, grid a multiple of 8 (XCD remap)
static int point_grid(int64_t n) {
  int64_t b = (n + 255) / 256;
  b = (b + 7) / 8 * 8;
  return (int)(b < 8 ? 8 : b);
}

int64_t point_blocks(int64_t n) { return point_grid(n); }
int64_t cell_blocks(int64_t n) { return (n + 1023) / 1024; }

// walkers of a list of up to n items, a lane each; k_core_rest takes several
static int list_grid(int64_t n) {
  return std::min(kListGrid, (point_grid(n) + kStripes - 1) / kStripes * kStripes);
}

template <bool F32, int Q>
static void core_kernels(const Dev& d, hipStream_t s) {
  hipLaunchKernelGGL(k_core<F32>, dim3(point_grid(d.n)), dim3(256), 0, s, d);
  hipLaunchKernelGGL((k_core_rest<F32, Q>), dim3(list_grid(d.n * Q)), dim3(256),
                     core_lds(d.rec_stride, Q), s, d);
  hipLaunchKernelGGL(k_core_crowd<F32>, dim3(list_grid(d.n)), dim3(256),
                     F32 ? core_lds(d.rec_stride, 4) : 0, s, d);
}

void launch_core(const Dev& d, bool f32, hipStream_t s) {
  if (d.n < kRestQuad)
    f32 ? core_kernels<true, 4>(d, s) : core_kernels<false, 4>(d, s);
  else
    f32 ? core_kernels<true, 2>(d, s) : core_kernels<false, 2>(d, s);
}

void launch_near(const Dev& d, hipStream_t s) {
  hipLaunchKernelGGL(k_rep, dim3((unsigned)cell_blocks(d.n)), dim3(1024), 0, s, d);
  hipLaunchKernelGGL(k_adj, dim3(list_grid(d.n)), dim3(256), 0, s, d);
}

void launch_link(const Dev& d, hipStream_t s) {
  const int64_t runs = (d.n + kLinkMin - 1) / kLinkMin;
  hipLaunchKernelGGL(k_link_local, dim3((unsigned)std::min<int64_t>(kLinkGrid, runs)), dim3(1024),
                     0, s, d);
  hipLaunchKernelGGL(k_link_cross, dim3(list_grid(d.n)), dim3(256), 0, s, d);
}

void launch_comp(const Dev& d, hipStream_t s) {
  hipLaunchKernelGGL(k_comp, dim3(list_grid(d.n)), dim3(256), 0, s, d);
}

void launch_pass_prep(const Dev& d, int pass, hipStream_t s) {
  hipLaunchKernelGGL(k_pass_prep, dim3(1), dim3(1), 0, s, d, pass);
}

void launch_pass_carry(const Dev& d, int pass, int check, hipStream_t s) {
  hipLaunchKernelGGL(k_pass_carry, dim3(1), dim3(256), 0, s, d, pass, check);
}

void launch_expand(const Dev& d, int pass, int grid, int seeds, int threads, int budget,
                   hipStream_t s) {
  size_t lds = (size_t)(threads / 64) * seeds * sizeof(int32_t);
  hipLaunchKernelGGL(k_expand, dim3(grid), dim3(threads), lds, s, d, pass, seeds, budget);
}

int expand_blocks_per_cu(int seeds, int threads) {
  int nb = 0;
  size_t lds = (size_t)(threads / 64) * seeds * sizeof(int32_t);
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_expand, threads, lds);
  if (e != hipSuccess || nb < 1) nb = 1;
  return nb;
}

void launch_merge(const Dev& d, int grid, hipStream_t s) {
  hipLaunchKernelGGL(k_merge_lds, dim3(1), dim3(1024), 0, s, d);
  hipLaunchKernelGGL(k_union_pairs, dim3(grid), dim3(256), 0, s, d);
  hipLaunchKernelGGL(k_flatten, dim3(grid), dim3(256), 0, s, d);
}

void launch_far(const Dev& d, bool f32, int grid, hipStream_t s) {
  hipLaunchKernelGGL(k_far, dim3(list_grid(d.n)), dim3(256), 0, s, d);
  if (f32)
    hipLaunchKernelGGL(k_far_pairs<true>, dim3(grid), dim3(256), 0, s, d);
  else
    hipLaunchKernelGGL(k_far_pairs<false>, dim3(grid), dim3(256), 0, s, d);
  hipLaunchKernelGGL(k_roots_final, dim3(list_grid(d.n)), dim3(256), 0, s, d);
}

void launch_border(const Dev& d, bool f32, hipStream_t s) {
  int g2 = (int)((d.n + 255) / 256);
  if (g2 > 4096) g2 = 4096;
  if (g2 < 1) g2 = 1;
  hipLaunchKernelGGL(k_keys, dim3(g2), dim3(256), 0, s, d);
  if (f32)
    hipLaunchKernelGGL(k_border<true>, dim3(list_grid(d.n)), dim3(256), 0, s, d);
  else
    hipLaunchKernelGGL(k_border<false>, dim3(list_grid(d.n)), dim3(256), 0, s, d);
}

// core flags to input order (on request, after a run)
__global__ __launch_bounds__(256) void k_core_out(const uint8_t* core, const int32_t* orig,
                                                  int64_t n, uint8_t* out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    out[orig[i]] = core[i];
}

void launch_core_out(const uint8_t* core, const int32_t* orig, int64_t n, uint8_t* out,
                     hipStream_t s) {
  int g = (int)((n + 255) / 256);
  if (g > 4096) g = 4096;
  if (g < 1) g = 1;
  hipLaunchKernelGGL(k_core_out, dim3(g), dim3(256), 0, s, core, orig, n, out);
}

void launch_relabel(const Dev& d, int64_t n, long long* out, hipStream_t s) {
  const unsigned rb = out ? 1 : 0;  // (the workgroup that reads the counters back)
  const int nb = (int)(((n + 63) / 64 + RK_TILE - 1) / RK_TILE);
  const bool split = n >= kOutSplit && n <= kOutWindows * kOutWindow;
  if ((n + 63) / 64 <= kRankOne) {
    hipLaunchKernelGGL(k_rank_one, dim3(1), dim3(1024), 0, s, d);
  } else {
    hipLaunchKernelGGL(k_rank_count, dim3(nb), dim3(RK_T), 0, s, d, split ? d.hist : nullptr);
    hipLaunchKernelGGL(k_rank_write, dim3(nb), dim3(RK_T), 0, s, d);
  }
  int g2 = (int)((n + 255) / 256);
  if (g2 > 4096) g2 = 4096;
  if (g2 < 1) g2 = 1;
  if (split) {
    int shift = 0;
    while ((n - 1) >> shift >= kOutWindows) ++shift;
    uint2* pairs = reinterpret_cast<uint2*>(d.key[0]);  // (the representatives are done with)
    hipLaunchKernelGGL(k_output_split, dim3((unsigned)((n + 512 * kOutItems - 1) / (512 * kOutItems))),
                       dim3(512), 0, s, d, shift, d.hist, pairs);
    // (a window smaller than the part it is gathered in shares its workgroup)
    if (shift > 13)
      hipLaunchKernelGGL((k_output_place<32768, 1024>), dim3((unsigned)((n + 32767) / 32768) + rb),
                         dim3(1024), 0, s, d, std::max(shift, 15), pairs, out);
    else
      hipLaunchKernelGGL((k_output_place<8192, 512>), dim3((unsigned)((n + 8191) / 8192) + rb),
                         dim3(512), 0, s, d, 13, pairs, out);
  } else {
    hipLaunchKernelGGL(k_output, dim3(g2 + rb), dim3(256), 0, s, d, out);
  }
}

}  // namespace dclust
