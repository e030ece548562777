// Internal device/host definitions shared by the HIP translation units.
//
// Data layout in HBM (all arrays live in the handle's arena, sized for the
// largest run seen so far and reused):
//   input   xyz       caller's row-major FP64 rows, instances back to back
//   sort    key[2]    u32 or u64 cell keys (ping-pong), val[2] i32 point ids
//   CSR     cell_start[C+1], cell_key[C], cell_inst[C], cell_col[C], cell_zl[C],
//           rows[3^(D-1)][C] (windows of the neighbour columns),
//           cell_ncore[C], cell_label[C] (chain), amask[C] (near graph), rep[C]
//   points  (cell-sorted)  X[N][3] FP64 (FP64 form only), G[N][3] u32 fixed-point
//           coordinates (29 fraction bits per cell, wrapping mod 8 cells),
//           orig[N], cell_of[N], core[N] u8, rec[N][R] + rec_n[N] (the
//           neighbours of each non-core point)
//   merge   parent[] union-find over cells, compmin[N], pairs[waves][E] int2
//   output  keyv[N] (component min input index), a flag bit per input index,
//           rank[N/64]
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace dclust {

constexpr int32_t kUnclaimed = -1;
constexpr int32_t kNoKey = 0x7fffffff;
constexpr int kFixBits = 29;  // fixed-point fraction bits per cell width
constexpr int kMaxRows = 9;   // 3^(D-1) neighbour columns for D <= 3
// points (and so cells) of a call: below this, because the 36-bit sort form
// keeps point ids in 28 bits
constexpr int64_t kMaxCells = 1LL << 28;
constexpr int kHeavy = 32;    // cells with more points are "heavy" (a wavefront per border pair)
// Neighbour records kept per non-core point, at most.  A bound on memory, not a
// measured optimum: 32 slots are 128 of the 400 or so bytes a point takes, and
// 16 keep the fixed region's capacity.  A non-core point has fewer than minpts
// neighbours, so records cover minpts up to 33 (17); above that the points with
// more neighbours are scanned again by k_border: 262 k 3-D points 37 us with
// minpts 33, 352 with 64, 701 with 128; without allocation, 100 k points 9 us
// with minpts 16, 81 with 24.
constexpr int kRecSlots = 32;
constexpr int kRecSlotsFixed = 16;  // in the fixed region of no-allocation runs
// rec_n of a point without records, whose rows are scanned instead: fewer
// than minpts points in all, or more neighbours than slots
constexpr int kRecFew = 254;
constexpr int kRecNone = 255;

// Cell order.  A column is the cells of a 2 x 2 block of the first two axes
// (3-D; of two cells of the first axis in 2-D) along the whole last axis.
// Cells are sorted by column, then by position along the last axis, then by
// place in the block (`local`, 2 bits in 3-D, 1 in 2-D: x & 1, then y & 1).
// So the 5^D stencil of a cell is covered by the same window of five steps
// along the last axis in 3^(D-1) neighbouring columns, and each window is a
// run of consecutive cells.  Row r of a cell is the window of the column with
// block offsets (a, b): r = 3(a+1) + b+1 in 3-D, r = a+1 in 2-D.  It holds the
// window's first cell, one bit per window slot: slot = step * nl + local, step
// 0..4 from two below the cell, nl = 2^(D-1) cells of a column per step, and
// above the 20 slot bits the number of the window's points (at most
// kRowCount).  The cell in slot s is first + (number of bits below s).  (One line per
// pair of offsets along the first two axes, as before, took 25 searches per
// cell instead of 9 and 100 bytes per cell instead of 72.)
template <int D>
struct Win {
  static constexpr int nl = 1 << (D - 1);
  static constexpr int rows = D == 3 ? 9 : 3;
  static constexpr int own = D == 3 ? 4 : 1;  // row of the cell's own column
  static constexpr int slots = 5 * nl;
  // local bits of all five steps from those of one
  static constexpr uint32_t steps = D == 3 ? 0x11111u : 0x155u;
};

constexpr uint32_t kRowBits = (1u << 20) - 1u;
constexpr uint32_t kRowCount = (1u << 12) - 1u;  // this many points or more

// Cells of block offset a that lie within two cells of a cell at place l of
// its block, along one axis (bit 0: place 0, bit 1: place 1).
__host__ __device__ __forceinline__ constexpr uint32_t axis_valid(int a, int l) {
  return a == 0 ? 3u : (a > 0 ? (l ? 3u : 1u) : (l ? 2u : 3u));
}

// Slots of row (a, b) inside the 5^D stencil of a cell at `local`.
template <int D>
__host__ __device__ __forceinline__ constexpr uint32_t row_valid(int a, int b, int local) {
  if (D == 2) return axis_valid(a, local & 1) * Win<2>::steps;
  const uint32_t vx = axis_valid(a, local >> 1), vy = axis_valid(b, local & 1);
  return ((vx & 1u ? vy : 0u) | (vx & 2u ? vy << 2 : 0u)) * Win<3>::steps;
}

// Near cells: at most one cell away along every axis.  Offset (dx, dy, dz)
// has the bit (dx+1)*9 + (dy+1)*3 + dz+1 of a cell's near mask (2-D: dy = 0);
// the opposite offset has bit 26 - b.
constexpr int kNearOwn = 13;

// Row and slot of near bit b for a cell at `local`.
template <int D>
__host__ __device__ __forceinline__ constexpr void near_slot(int b, int local, int& row,
                                                             int& slot) {
  const int dx = (b * 57) >> 9;           // b / 9 for b < 27
  const int r9 = b - 9 * dx;
  const int dy = (r9 * 11) >> 5;          // r9 / 3 for r9 < 9
  const int dz = r9 - 3 * dy;
  if (D == 2) {
    const int tx = (local & 1) + dx - 1;  // -1..2
    row = 1 + (tx >> 1);
    slot = (dz + 1) * 2 + (tx & 1);
  } else {
    const int tx = (local >> 1) + dx - 1, ty = (local & 1) + dy - 1;
    row = 4 + 3 * (tx >> 1) + (ty >> 1);
    slot = (dz + 1) * 4 + (tx & 1) * 2 + (ty & 1);
  }
}

namespace tables {
// every offset of the 5^D stencil lies in exactly one valid slot, and the
// near bits name the slots of their offsets
template <int D>
constexpr bool windows_ok() {
  for (int local = 0; local < Win<D>::nl; ++local) {
    const int lx = D == 3 ? local >> 1 : local, ly = D == 3 ? local & 1 : 0;
    int count = 0;
    for (int a = -1; a <= 1; ++a)
      for (int b = D == 3 ? -1 : 0; b <= (D == 3 ? 1 : 0); ++b)
        for (int s = 0; s < Win<D>::slots; ++s) {
          const int l = s % Win<D>::nl, dz = s / Win<D>::nl - 2;
          const int dx = 2 * a + (D == 3 ? l >> 1 : l) - lx;
          const int dy = D == 3 ? 2 * b + (l & 1) - ly : 0;
          const bool in = dx >= -2 && dx <= 2 && dy >= -2 && dy <= 2;
          if (in != (((row_valid<D>(a, b, local) >> s) & 1u) != 0)) return false;
          count += in;
          if (dx < -1 || dx > 1 || dy < -1 || dy > 1 || dz < -1 || dz > 1) continue;
          int row = 0, slot = 0;
          near_slot<D>((dx + 1) * 9 + (dy + 1) * 3 + dz + 1, local, row, slot);
          if (row != (D == 3 ? 3 * (a + 1) + b + 1 : a + 1) || slot != s) return false;
        }
    if (count != (D == 3 ? 125 : 25)) return false;
  }
  return true;
}
static_assert(windows_ok<2>() && windows_ok<3>(), "stencil windows");
}  // namespace tables

// Per-instance parameters and derived grid (device table, one per instance).
struct Inst {
  double mn[3];    // grid origin = bounding-box minimum
  double inv_w;    // 1 / cell width: cell(x) = floor(fl(fl(x - mn) * inv_w))
  double w;        // cell width
  double eps;      // EPS
  double eps2;     // fl(eps * eps), the oracle's threshold
  double maxabs;   // max |coordinate| (FP error bounds)
  float d2_in;     // FP32 form: D2 <  d2_in  -> neighbour
  float d2_out;    // FP32 form: D2 >  d2_out -> not a neighbour
  float d2_mid;    // FP32 form: rounded eps^2 in fixed-point units
  int32_t dim;
  int32_t minpts;
  int32_t r;       // PARTITION_SIZE (0 = auto)
  int32_t nk[3];   // cells per axis
  int32_t err;     // per-instance error code (DCLUST_E_*)
  int64_t key_base;            // first key of this instance's cell space
  int64_t line_base;           // first entry of this instance's column table
  int64_t nlines;              // its columns
  int64_t nzl;                 // keys of a column: cells along the last axis * nl
  int64_t cstride;             // columns per step of the first axis' blocks (3-D: one
                               // more than there are, so that the column before the
                               // first and after the last of a step is always empty)
  double inv_nzl;              // fl(1 / nzl)
  int64_t pt_begin, pt_end;    // global point-index range
  int64_t xyz_off;             // element offset of the first coordinate
};

// column table entries (8 bytes each) above which neighbour columns are found
// by binary search instead
constexpr long long kMaxLineTable = 1LL << 26;  // 512 MiB at most

// Chunk of at most kChunk points of one instance (work list of the per-point
// kernels that need the instance, so no point->instance search is needed;
// host-built, for a batch).
constexpr int64_t kChunk = 4096;
struct Chunk {
  int32_t inst;
  int32_t pad;
  int64_t begin, end;
};

// Control block (int64 counters in device memory).
enum Ctl : int {
  C_KEYBITS = 0,
  C_NCELL,
  C_NCHAIN,     // chains started (a chain id is its seed cell's index)
  C_NPAIR,
  C_Q0_N,
  C_Q1_N,
  C_Q0_HEAD,
  C_Q1_HEAD,
  C_NCORE,
  C_NNOISE,
  C_NCLUST,
  C_CAND,
  C_NBRC,
  C_BAND,
  C_FLIP,
  C_ASYM,
  C_EVAL,
  C_OVF,
  C_ERR,
  C_BAND_CORE,
  C_POPS,       // cells expanded
  C_BUSY_SUM,  // expansion: sum over waves of their lifetime (us)
  C_BUSY_MAX,
  C_SEGS_LEFT,  // expansion waves whose seeding segment is not finished
  C_NLINES,     // total column-table entries
  C_DENSE,      // cells resolved as all-core without distance tests
  C_NHEAVY,     // heavy cells (more than kHeavy points)
  C_NADJPTS,    // core points of light cells
  C_NCORECELLS, // cells with core points (listed in Dev::core_cells)
  C_EDGES,      // joined pairs of the near graph, from both sides
  C_RECOVF,     // non-core points whose neighbour record overflowed
  C_ADJ_TESTS,  // representative pairs tested for the near graph
  C_ADJ_FREE,   // border pairs joined without a test (cell inside the eps ball)
  C_FAR_TESTS,  // pair tests of the border-pair passes
  C_FAR_JOINS,  // border pairs that joined two components
  C_LASTPASS,   // 1 + the last expansion pass that popped a cell
  C_POPS_MAX,   // most cells popped by one expansion wave in one pass
  C_SEEDS_MAX,  // most chains started by one expansion wave in one pass
  C_ABANDON,    // expansion left work pending in a run with a fixed pass
                // count: the kernels after it return at once
  C_IDLE,       // nothing pending for the current expansion pass
  C_ROUNDS_MAX, // most pop rounds of one expansion wave in one pass
  C_KEYOVF,     // the cell-key space of the whole call exceeds 2^63 keys
  // work counts of the neighbour kernels (their algorithmic bytes)
  C_CORE_ROWS,    // neighbour counts: rows read
  C_CORE_RANGES,  // neighbour counts: non-empty point ranges of them
  C_NROWSFB,      // row work items left to the global-memory pass (Dev::rows_fb)
  C_NBORDERPTS,   // non-core points (listed in Dev::border_pts)
  C_NCOREREST,    // points left by the first count pass (Dev::core_rest)
  C_NCORECROWD,   // those taken by a wavefront each (Dev::core_crowd)
  C_NROOTS,       // near components (listed in Dev::near_roots)
  C_NFARLIGHT,    // pairs across components (listed in Dev::far_light)
  C_NFARHEAVY,    // those with a heavy cell (listed in Dev::far_heavy)
  C_NFAROVER,     // cells with pairs that found no room there (Dev::far_over)
  C_BOXES,        // chunks whose bounding box is done (one instance)
  // this call's input and output (addresses), written by the run's first kernel
  C_XYZ,
  C_LABELS,
  // device clock (kClockMHz) at the start of the run, of the neighbour counts
  // and of what follows them
  C_T_START,
  C_T_CORE0,
  C_T_CORE1,
  C_NCTL
};
static_assert(C_T_CORE1 < C_NCTL, "control block too small");

// Cell-key space: the sort key of a cell is its instance's key base plus its
// place in the cell order, and the
// cells of all instances of a call must number at most 2^63.  Sums are
// saturating, so an overflowing total stays above the limit.  (The keys
// themselves number a little more: odd axes are rounded up to whole blocks,
// and every step of blocks has one empty column.)
constexpr unsigned long long kMaxKeySpace = 1ull << 63;
__host__ __device__ __forceinline__ unsigned long long sat_add(unsigned long long a,
                                                                unsigned long long b) {
  const unsigned long long s = a + b;
  return s < a ? ~0ull : s;
}
// Radix-sort key width for a key space of `total` keys.
__host__ __device__ __forceinline__ int key_bits_for(unsigned long long total) {
  int bits = 1;
  while (bits < 64 && (1ull << bits) < total) ++bits;
  return bits;
}

// Statistics counters are striped: a wave adds to one of kStripes copies.
// The copies of one counter lie kStatStride counters apart, so that they are
// on different cache lines (atomics on one line are taken one after the
// other, about 1 ns each).
constexpr int kStripes = 64;
constexpr int kStatStride = 64;
static_assert(C_NCTL <= kStatStride, "counter stripe too short");

// A work list filled by many workgroups: kStripes sub-lists (workgroup b
// appends to sub-list b % kStripes, with its own counter), so that the
// appends do not serialise on one address.  Element i of the whole list is
// found through the prefix of the sub-list counts.  The counters live in
// the striped statistics array, so the host reads the total like a counter.
struct SList {
  int32_t* data;             // [kStripes][cap]
  unsigned long long* cnt;   // [kStripes], kStatStride apart
  int64_t cap;
};

// The same for pairs of cells; a counter may exceed cap (the pairs past it
// were not stored).
struct PairList {
  int2* data;                // [kStripes][cap]
  unsigned long long* cnt;   // [kStripes], kStatStride apart
  int64_t cap;
};

// Radix sort: the fewest passes of digits of at most kDigitBits bits that cover
// the key, each of which scatters (index.hip).
constexpr int kDigitBits = 9;  // of a radix pass, at most
constexpr int kSortPasses = 8;  // of up to 64 bits
constexpr int kSortGrid = 512;  // workgroups of the sort, at most
constexpr int kSortGroup = 32;  // of which so many add to one group's counts
constexpr int kSortGroups = kSortGrid / kSortGroup;

// Bounding-box partials: chunk b of an instance reduces into stripe b % kBoxStripes of its
// instance (so that the atomics of many chunks do not meet on one address);
// the grid set-up reduces the stripes.
constexpr int kBoxStripes = 32;

// What a call brings besides its sizes: input and output, and its parameters
// if it has one instance.  They reach the kernels through the control block
// and the instance table, not through Dev: a captured run is replayed for
// calls with other buffers and other parameters.
struct Call {
  const double* xyz;
  int32_t* labels;
  Inst inst;
};
static_assert(sizeof(Inst) % 8 == 0, "the instance table is copied in words");

constexpr int kClockMHz = 100;  // of the constant device clock

// All device pointers of one run, passed to kernels by value.
struct Dev {
  int64_t n;
  int32_t ninst;
  int32_t err_stops;  // 1: an instance's error fails the call, which then writes nothing
  Inst* inst;
  const Chunk* chunks;
  unsigned long long* bbox;  // [ninst][kBoxStripes][8] ordered-u64 min0..2 max0..2,
                             // max |x|, non-finite flag
  long long* ctl;
  long long* stat;  // [kStripes][kStatStride] statistics counters

  // radix sort
  uint64_t* key[2];
  int32_t* val[2];
  uint32_t* hist;   // [nblk][512] digit counts of the sort's workgroups
  uint32_t* dgrp;   // [kSortPasses][kSortGroups][512] digit counts of its groups

  // CSR
  int32_t* cell_start;  // [N+1]
  uint64_t* cell_key;   // [N]
  uint32_t* cell_col;   // [N] column-table index (when there is a column table)
  uint32_t* cell_zl;    // [N] place in the column: last coordinate * nl + local
  int32_t* cell_inst;   // [N]
  int32_t* cell_ncore;  // [N] core points per cell
  int32_t* cell_label;  // [N] chain owning the cell's core points
  uint32_t* amask;      // [N] near graph: joined near cells, by near bit
  int32_t* cell_comp;   // [N+4] component (root chain) of each core cell, -1 otherwise
  uint4* rep;           // [N] per cell: its first core point's G and sorted index
                        // (over the sort keys, which the CSR pass is the last to read)
  int32_t chains;       // 1: near components by seed-list expansion, 0: by union-find
  SList core_rest;      // points the first count pass leaves (over keyv)
  SList core_crowd;     // those of them with many candidates (over compmin)
  SList border_pts;     // non-core points (border-label lanes)
  SList core_cells;     // cells with core points (near-graph and border-pair lanes)
  SList near_roots;     // roots of the near components
  PairList far_light;   // pairs of cells across components without a heavy cell and
  PairList far_heavy;   // with one (over the sort's point ids, which the gather is the
                        // last to read)
  SList far_over;       // cells with pairs that neither had room for (over keyv)
  uint2* rows;          // [kMaxRows][rstride] neighbour windows (first cell, slot bits and
                        // point count), row-major so that consecutive cells are adjacent
  int64_t rstride;      // >= number of cells
  int32_t* cell_of;     // [N] per sorted point
  int2* lines;          // [line_cap] first / end cell of every column
  int64_t line_cap;     // 0: no column table, windows found by binary search
  int32_t nbr_stats;    // 1: the neighbourhood sizes are summed

  // sorted point data
  double* X;            // [N][3] FP64 form only (null in the FP32 form)
  const double** xrow;  // FP32 form: each point's row of the input
  uint32_t* G;          // [N][3]
  int32_t* orig;
  uint8_t* core;
  int32_t* rec;         // [rec_stride][N] neighbours of non-core points
  uint8_t* rec_n;       // [N] records written, kRecFew or kRecNone
  int32_t rec_stride;   // record slots per point: minpts or more, at most kRecSlots
  int32_t* parent;
  int32_t* compmin;
  int2* pairs;          // [waves][pair_per] collision pairs per expansion wave
  int32_t* pair_cnt;    // [waves] pairs recorded (may exceed pair_per)
  int64_t pair_cap;     // waves * pair_per
  int32_t pair_per;
  int32_t* q[2];
  int64_t* seg_pos;     // [waves] seeding cursor of each expansion wave
  int32_t* keyv;
  SList rows_fb;         // row work items (tile * 3 + group) left to k_rows_global
  unsigned long long* flag;  // [N/64] bit per input index: smallest core point of a cluster
  int32_t* rank;             // [N/64] flags before each word
  int64_t* scan_tmp;  // block sums for scans

  uint8_t* core_out;    // core flags in input order
};

// ------------------------------------------------------------ helpers ----
__device__ __forceinline__ int lane_id() { return __lane_id(); }

__device__ __forceinline__ unsigned long long ballot(bool p) {
  return __ballot(p);
}

__device__ __forceinline__ int mbcnt(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi(
      (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ int rl_i(int v, int l) {
  return __builtin_amdgcn_readlane(v, l);
}
__device__ __forceinline__ uint32_t rl_u(uint32_t v, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
__device__ __forceinline__ double rl_d(double v, int l) {
  long long b = __double_as_longlong(v);
  int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), l);
  int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (uint32_t)lo);
}
__device__ __forceinline__ int64_t rl_l(int64_t v, int l) {
  const int lo = __builtin_amdgcn_readlane((int)(v & 0xffffffffLL), l);
  const int hi = __builtin_amdgcn_readlane((int)(v >> 32), l);
  return (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}
__device__ __forceinline__ int rfl_i(int v) {
  return __builtin_amdgcn_readfirstlane(v);
}

// wave barrier + wavefront-scope fence: orders LDS traffic between lanes of
// one wave (seed-list pushes followed by pops).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class T>
__device__ __forceinline__ T wave_sum(T v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
template <class T>
__device__ __forceinline__ T wave_min(T v) {
  for (int o = 32; o > 0; o >>= 1) {
    T u = __shfl_xor(v, o, 64);
    v = u < v ? u : v;
  }
  return v;
}
template <class T>
__device__ __forceinline__ T wave_max(T v) {
  for (int o = 32; o > 0; o >>= 1) {
    T u = __shfl_xor(v, o, 64);
    v = u > v ? u : v;
  }
  return v;
}
// inclusive prefix sum over the wave
template <class T>
__device__ __forceinline__ T wave_incl_scan(T v) {
  const int l = lane_id();
  for (int o = 1; o < 64; o <<= 1) {
    T u = __shfl_up(v, o, 64);
    if (l >= o) v += u;
  }
  return v;
}

// chain ids are seed cell indices: the id space is the cell count
__device__ __forceinline__ long long chain_ids(const Dev& d) { return d.ctl[C_NCELL]; }

__device__ __forceinline__ const double* in_xyz(const Dev& d) {
  return reinterpret_cast<const double*>(d.ctl[C_XYZ]);
}
__device__ __forceinline__ int32_t* out_labels(const Dev& d) {
  return reinterpret_cast<int32_t*>(d.ctl[C_LABELS]);
}
// the device clock, stamped by one thread of the launch
__device__ __forceinline__ void stamp(const Dev& d, int ctr) {
  if (blockIdx.x == 0 && threadIdx.x == 0) d.ctl[ctr] = (long long)__builtin_amdgcn_s_memrealtime();
}

// set when a run with a fixed number of expansion passes left work pending
__device__ __forceinline__ bool abandoned(const Dev& d) { return d.ctl[C_ABANDON] != 0; }

// Statistics counter update: the wave's sum goes to one of kStripes copies
// of the counter, picked by the wave's position in the launch, so that a
// launch of many waves does not serialise on one address.
// A wave with nothing to add (most waves of most counters) skips the sum;
// small counts are summed in 32 bits (half the shuffles).
__device__ __forceinline__ void stat_add(const Dev& d, int ctr, long long v) {
  if (!ballot(v != 0)) return;
  const long long s = ballot((v >> 24) != 0) ? wave_sum(v) : (long long)wave_sum((int)v);
  if (lane_id() == 0) {
    const unsigned w = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) & (kStripes - 1);
    atomicAdd((unsigned long long*)&d.stat[w * kStatStride + ctr], (unsigned long long)s);
  }
}

// Appends `value` of the threads with `take` to the workgroup's sub-list of
// L, in thread order, with one atomic per workgroup.  Every thread of the
// workgroup calls it.
__device__ __forceinline__ void block_append(bool take, int32_t value, const SList& L) {
  __shared__ int s_cnt[16];
  __shared__ long long s_base;
  const int wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const unsigned long long m = ballot(take);
  if (lane_id() == 0) s_cnt[wv] = __popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    int tot = 0;
    for (int w = 0; w < nw; ++w) tot += s_cnt[w];
    s_base = tot ? (long long)atomicAdd(&L.cnt[(blockIdx.x & (kStripes - 1)) * kStatStride],
                                        (unsigned long long)tot)
                 : 0;
  }
  __syncthreads();
  long long base = s_base;
  for (int w = 0; w < wv; ++w) base += s_cnt[w];
  if (take) L.data[(int64_t)(blockIdx.x & (kStripes - 1)) * L.cap + base + mbcnt(m)] = value;
  __syncthreads();  // s_cnt / s_base are reused by the next call
}

// The part of a list that a workgroup walks: the sub-list that the workgroups
// with its stripe filled, shared by the grid's workgroups of that stripe (the
// grid is a multiple of kStripes).  A stripe is on one XCD, and the kernels
// that fill lists give each XCD one range of points or cells, so a walker
// finds the lists' neighbourhoods in its own L2.  A walker that appends to
// another list appends to the same stripe, so that list needs no more room a
// stripe than this one.
struct Stripe {
  const int32_t* data;
  int64_t n;
  __device__ __forceinline__ explicit Stripe(const SList& L) {
    const int s = blockIdx.x & (kStripes - 1);
    data = L.data + s * L.cap;
    n = (int64_t)L.cnt[s * kStatStride];
  }
  // first item of this workgroup and its stride, `per` items at a time
  __device__ __forceinline__ int64_t first(int per) const {
    return (int64_t)(blockIdx.x / kStripes) * per;
  }
  __device__ __forceinline__ int64_t step(int per) const {
    return (int64_t)(gridDim.x / kStripes) * per;
  }
};

// The control counters, their stripes added, into the handle's pinned buffer,
// by one workgroup of at least four wavefronts: a lane per counter, a share of
// the stripes per wavefront.
static_assert(C_NCTL <= 64 && kStatStride == 64, "a lane per counter");
__device__ __forceinline__ void readback(const Dev& d, long long* out) {
  __shared__ long long s_sum[16][64];
  const int l = lane_id(), wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  long long v[kStripes / 4], sum = wv == 0 && l < C_NCTL ? d.ctl[l] : 0;
#pragma unroll
  for (int r = 0; r < kStripes / 4; ++r)
    v[r] = wv + r * nw < kStripes ? d.stat[(wv + r * nw) * kStatStride + l] : 0;
#pragma unroll
  for (int r = 0; r < kStripes / 4; ++r) sum += v[r];
  s_sum[wv][l] = sum;
  __syncthreads();
  if (threadIdx.x >= C_NCTL) return;
  sum = 0;
  for (int w = 0; w < nw; ++w) sum += s_sum[w][l];
  out[l] = sum;
}

// Prefix of the sub-list counts of L in LDS (s_pre[kStripes + 1]); returns
// the list length.  Every thread of the workgroup calls it.
__device__ __forceinline__ long long slist_prefix(const SList& L, long long* s_pre) {
  if (threadIdx.x < kStripes) {
    const long long v = (long long)L.cnt[threadIdx.x * kStatStride];
    const long long incl = wave_incl_scan(v);
    s_pre[threadIdx.x + 1] = incl;
    if (threadIdx.x == 0) s_pre[0] = 0;
  }
  __syncthreads();
  return s_pre[kStripes];
}

// Element i (< length) of the list.
__device__ __forceinline__ int32_t slist_at(const SList& L, const long long* s_pre, long long i) {
  int lo = 0, hi = kStripes - 1;  // last sub-list whose range starts at or before i
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (s_pre[mid] <= i) lo = mid; else hi = mid - 1;
  }
  return L.data[(int64_t)lo * L.cap + (i - s_pre[lo])];
}

// Monotone map double -> u64 (for atomic min/max of doubles).
__device__ __forceinline__ unsigned long long ord_d(double x) {
  unsigned long long u = (unsigned long long)__double_as_longlong(x);
  return (u >> 63) ? ~u : (u | 0x8000000000000000ULL);
}
__host__ __device__ inline double unord_d(unsigned long long u) {
  unsigned long long b = (u >> 63) ? (u & 0x7fffffffffffffffULL) : ~u;
  double d;
  __builtin_memcpy(&d, &b, sizeof(d));
  return d;
}

// Blocks of a launch are dealt to the 8 XCDs round-robin (block b runs on
// XCD b % 8).  Remap so that each XCD owns a contiguous range of logical
// blocks: neighbouring work then shares that XCD's L2.  G must be a
// multiple of 8.
__device__ __forceinline__ int xcd_block(int b, int G) {
  int per = G >> 3;
  return (b & 7) * per + (b >> 3);
}

// The same in runs: the XCDs take runs of CH consecutive workgroups in turn,
// so that a clustered input's work spreads over all of them (the last, partial
// round of runs is not remapped).
template <int CH>
__device__ __forceinline__ int xcd_runs(int b, int G) {
  const int q = b >> 3, round = q / CH;
  return (round + 1) * 8 * CH <= G ? round * 8 * CH + (b & 7) * CH + q % CH : b;
}

// State of the one-step (CUDA-DClust) baseline, cell-sorted order.
struct OneStep {
  int32_t* label;     // [n] -1 unclassified, -2 noise, >= 0 chain
  int32_t* state;     // [n] 0 not expanded, 1 expanded, 2 expanded core
  int32_t* seeds;     // [blocks * S] per-chain seed lists
  int32_t* len;       // [blocks] seed-list lengths
  int2* contacts;     // [cap] (chain, chain) contacts between core points
  int32_t* ctr;       // [2] contacts recorded since the last host read (may
                      // exceed cap: the rest were not stored), spare
  int32_t blocks, S, cap, pad;
};

// The rows of one cell.
struct RowsOf {
  const uint2* base;
  int64_t stride;
  __device__ __forceinline__ uint2 operator[](int r) const { return base[(int64_t)r * stride]; }
};
__device__ __forceinline__ RowsOf rows_of(const Dev& d, int64_t c) {
  return RowsOf{d.rows + c, d.rstride};
}
// cells and points of a row's window
__device__ __forceinline__ int row_cells(uint2 row) { return __popc(row.y & kRowBits); }
__device__ __forceinline__ uint32_t row_count(uint2 row) { return row.y >> 20; }
__device__ __forceinline__ uint2 make_row(int32_t first, uint32_t bits, int32_t points) {
  const uint32_t n = (uint32_t)points < kRowCount ? (uint32_t)points : kRowCount;
  return make_uint2(bits ? (uint32_t)first : 0u, bits | (n << 20));
}
// cell in slot s of a row
__device__ __forceinline__ int32_t slot_cell(uint2 row, int s) {
  return (int32_t)row.x + __popc(row.y & ((1u << s) - 1u));
}

// Instance of a cell (a run of one instance reads the table entry directly,
// with no per-cell load).
__device__ __forceinline__ const Inst* inst_of_cell(const Dev& d, int64_t c) {
  return d.ninst == 1 ? d.inst : d.inst + d.cell_inst[c];
}

// Cell index along one axis, shared by key computation, gather and every
// search (the reference computes insert and search bins with different
// formulas, indexing.cu:114 vs indexing.cu:96-101; here there is one).
__device__ __forceinline__ double cell_t(double x, double mn, double inv_w) {
  return (x - mn) * inv_w;
}

// ---- lock-free union-find ----------------------------------------------
// A link only ever replaces a root's self-pointer (by CAS) with a node of
// smaller uf_order, a bijective scramble of the ids, so links cannot close a
// cycle and every value par[x] has held is an ancestor of x.  (Linked by the
// ids themselves, neighbouring sets, whose ids follow the cell order, hook
// each other into chains as long as the row of sets; in scrambled order the
// expected depth is logarithmic.)  A plain load may therefore return a stale
// but still valid ancestor: uf_find_cached walks with plain (L2-cached)
// loads, which is enough to decide "same set" when two walks meet.  A CAS on
// a stale "root" fails and the retry walks with coherent (agent-scope)
// loads, which guarantees progress.
__device__ __forceinline__ uint32_t uf_order(int32_t x) { return (uint32_t)x * 0x9E3779B1u; }

__device__ __forceinline__ int32_t uf_find(int32_t* par, int32_t x) {
  for (;;) {
    int32_t p = __hip_atomic_load(&par[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (p == x) return x;
    int32_t gp = __hip_atomic_load(&par[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (gp != p)
      __hip_atomic_store(&par[x], gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    x = p;
  }
}

// Root of x by a walk that writes nothing (for a pass in which every thread
// stores a root of its own and no unions run).
__device__ __forceinline__ int32_t uf_root(const int32_t* par, int32_t x) {
  for (;;) {
    const int32_t p = par[x];
    if (p == x) return x;
    x = p;
  }
}

__device__ __forceinline__ int32_t uf_find_cached(int32_t* par, int32_t x) {
  for (;;) {
    int32_t p = par[x];
    if (p == x) return x;
    int32_t gp = par[p];
    if (gp != p) par[x] = gp;  // path halving: gp is an ancestor of x
    x = p;
  }
}

__device__ __forceinline__ void uf_union(int32_t* par, int32_t a, int32_t b) {
  a = uf_find_cached(par, a);
  b = uf_find_cached(par, b);
  for (;;) {
    if (a == b) return;
    if (uf_order(a) < uf_order(b)) {
      int32_t t = a;
      a = b;
      b = t;
    }
    int32_t old = atomicCAS(&par[a], a, b);
    // (a concurrent union of the same two sets: the usual reason to fail)
    if (old == a || old == b) return;
    a = uf_find(par, old);
    b = uf_find(par, b);
  }
}

}  // namespace dclust
