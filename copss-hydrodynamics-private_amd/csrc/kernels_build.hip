// kernels_build.hip -- (a) the neighbour build: element binning, counting
// sort of the particles into cell order (stable by particle id), the
// per-slot list lengths and sliced lists and the element lists of the
// spreading (built brick by brick from LDS-staged cell starts), and the CSR
// emission of the reference's lists for export.
//
// Reference: PointMesh<3>::reinit (point_mesh.C:245-289) with
// build_elem_point_containing_list (:573-648), build_elem_point_neighbor_list
// (:652-799) and build_point_point_neighbor_list (:803-848).  The element
// stencil replaces build_elem_elem_neighbor_list (:293-443); it is computed
// on the host once per context.
#include "ggem_device.h"

namespace ggem {

namespace {

constexpr int kBlock = 256;

inline unsigned blocks_for(int64_t n, int b = kBlock) { return unsigned((n + b - 1) / b); }

// Canonical element of a point: per axis floor((x - min)/h) clamped to
// [0, n-1]; -1 outside [min, max].
__device__ __forceinline__ int64_t locate_dev(const Grid& g, double x, double y, double z) {
  const double v[3] = {x, y, z};
  int64_t c[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (!(v[d] >= g.bmin[d]) || !(v[d] <= g.bmin[d] + g.L[d])) return -1;
    int64_t q = int64_t(floor((v[d] - g.bmin[d]) / g.h[d]));
    q = q < 0 ? 0 : q;
    q = q > g.n[d] - 1 ? g.n[d] - 1 : q;
    c[d] = q;
  }
  return c[0] + int64_t(g.n[0]) * (c[1] + int64_t(g.n[1]) * c[2]);
}

// brick-order cell index of reference element e
__device__ __forceinline__ int64_t elem_cell(const Grid& g, int64_t e) {
  int i, j, k;
  elem_ijk(g, e, i, j, k);
  return cell_index(g, i, j, k);
}

// Elem::contains_point of an axis-aligned hex with libMesh's 1e-6 tolerance
// on the reference element.
__device__ __forceinline__ bool contains_dev(const Grid& g, int64_t e, double x, double y,
                                             double z) {
  int ci, cj, ck;
  elem_ijk(g, e, ci, cj, ck);
  const double v[3] = {x, y, z};
  const int ijk[3] = {ci, cj, ck};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double cen = g.bmin[d] + (double(ijk[d]) + 0.5) * g.h[d];
    const double xi = 2.0 * (v[d] - cen) / g.h[d];
    if (!(fabs(xi) <= 1.0 + 1e-6)) return false;
  }
  return true;
}

// Grid, stencil rows and cell starts seen by one particle or slot: the
// context's own, or those of its system in a batched context (cell starts
// shifted to the system's first element, so element ids stay local).
struct SysView {
  Grid g;
  const StencilRow* rows;
  int nrows;
  const int32_t* cs;  // cell starts from the system's first cell
  int64_t eoff;       // first element id of the system
  int64_t coff;       // first cell index of the system
};

template <bool BATCH>
__device__ __forceinline__ SysView sys_view(const Grid& g, const StencilRow* rows, int nrows,
                                            const int32_t* cs, const SysGrid* sys, const int32_t* sys_of,
                                            int64_t i) {
  if constexpr (BATCH) {
    const SysGrid& S = sys[sys_of[i]];
    return SysView{S.g, rows + S.row_off, S.nrows, cs + S.cell_off, S.elem_off, S.cell_off};
  } else {
    return SysView{g, rows, nrows, cs, 0, 0};
  }
}

template <bool BATCH>
__global__ void k_bin(Grid g, const SysGrid* __restrict__ sys, const int32_t* __restrict__ sys_part,
                      int64_t n, const double* __restrict__ x, int32_t* __restrict__ elem, int use_prev,
                      int32_t* __restrict__ pcell, int32_t* __restrict__ prank, int32_t* __restrict__ count,
                      int32_t* __restrict__ flag) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const SysView v = sys_view<BATCH>(g, nullptr, 0, nullptr, sys, sys_part, i);
  const double px = x[3 * i], py = x[3 * i + 1], pz = x[3 * i + 2];
  int64_t e = -1;
  if (use_prev) {
    const int64_t old = int64_t(elem[i]) - v.eoff;
    if (old >= 0 && old < v.g.n_elem && contains_dev(v.g, old, px, py, pz)) e = old;
  }
  if (e < 0) e = locate_dev(v.g, px, py, pz);
  if (e < 0) {
    atomicOr(flag, 1);
    e = 0;  // keep later kernels in bounds; the host reports the error
  }
  const int64_t c = v.coff + elem_cell(v.g, e);
  elem[i] = int32_t(v.eoff + e);
  pcell[i] = int32_t(c);
  prank[i] = atomicAdd(&count[c], 1);  // a place in the cell, in arrival order
}

// system of each particle from the particle ranges (binary search)
__global__ void k_part_sys(int64_t n, int nsys, const int64_t* __restrict__ part_off,
                           int32_t* __restrict__ sys_part) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int lo = 0, hi = nsys - 1;
  while (lo < hi) {  // last k with part_off[k] <= i
    const int mid = (lo + hi + 1) >> 1;
    if (part_off[mid] <= i) lo = mid;
    else hi = mid - 1;
  }
  sys_part[i] = lo;
}

// Exclusive scan of int32 counts in three phases: per-block scan with block
// totals, a single-block scan of the totals, and the carry-in add.
constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ __forceinline__ int32_t block_exclusive_scan(int32_t v, int32_t* sh, int32_t& total) {
  const int t = threadIdx.x;
  sh[t] = v;
  __syncthreads();
  for (int off = 1; off < kScanThreads; off <<= 1) {
    const int32_t add = (t >= off) ? sh[t - off] : 0;
    __syncthreads();
    sh[t] += add;
    __syncthreads();
  }
  total = sh[kScanThreads - 1];
  const int32_t incl = sh[t];
  __syncthreads();
  return incl - v;
}

// (the counts are left zero for the next build)
__global__ void k_scan_tiles(int32_t* __restrict__ in, int64_t len, int32_t* __restrict__ out,
                             int32_t* __restrict__ tile_sums) {
  __shared__ int32_t sh[kScanThreads];
  const int64_t base = int64_t(blockIdx.x) * kScanTile + int64_t(threadIdx.x) * kScanItems;
  int32_t v[kScanItems];
  int32_t s = 0;
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    v[q] = (base + q < len) ? in[base + q] : 0;
    if (v[q] != 0) in[base + q] = 0;  // (410^3 cells, most of them empty: 418 -> 308 us)
    s += v[q];
  }
  int32_t total;
  int32_t run = block_exclusive_scan(s, sh, total);
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    if (base + q < len) out[base + q] = run;
    run += v[q];
  }
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

__global__ void k_scan_sums(int32_t* __restrict__ sums, int64_t ntiles) {
  __shared__ int32_t sh[kScanThreads];
  int32_t carry = 0;
  for (int64_t c0 = 0; c0 < ntiles; c0 += kScanThreads) {
    const int64_t i = c0 + threadIdx.x;
    const int32_t v = (i < ntiles) ? sums[i] : 0;
    int32_t total;
    const int32_t ex = block_exclusive_scan(v, sh, total);
    if (i < ntiles) sums[i] = ex + carry;
    carry += total;
    __syncthreads();
  }
}

// Carry into one tile per block: the sum of the tiles before it, added up
// by the block itself (a launch less than scanning the sums first; at most
// kScanSelfMax tiles, 8 loads a thread at 2M cells), or the scanned sums'.
constexpr int64_t kScanSelfMax = 4096;
__global__ void k_scan_add(int32_t* __restrict__ out, int64_t len, const int32_t* __restrict__ sums, int scanned,
                           int32_t total_n) {
  __shared__ int32_t sh[kScanThreads / 64];
  int32_t carry = 0;
  if (scanned) {
    carry = sums[blockIdx.x];
  } else {
    for (int t = int(threadIdx.x); t < int(blockIdx.x); t += kScanThreads) carry += sums[t];
    carry = wave_sum(carry);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = carry;
    __syncthreads();
    carry = 0;
#pragma unroll
    for (int w = 0; w < kScanThreads / 64; ++w) carry += sh[w];
  }
  const int64_t base = int64_t(blockIdx.x) * kScanTile;
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    const int64_t i = base + q * kScanThreads + threadIdx.x;
    if (i < len) out[i] += carry;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) out[len] = total_n;
}

// Every particle into its cell's slot range, in arrival order
__global__ void k_place(int64_t n, const int32_t* __restrict__ pcell, const int32_t* __restrict__ prank,
                        const int32_t* __restrict__ cell_start, int32_t* __restrict__ arrived) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) arrived[cell_start[pcell[i]] + prank[i]] = int32_t(i);
}

// Forces of particle p (interleaved) to slot s: SoA and gather records
__device__ __forceinline__ void slot_forces(int64_t n, int64_t s, int64_t p, const double* __restrict__ f,
                                            double* __restrict__ fs, float4* __restrict__ fg32,
                                            double4* __restrict__ fg64) {
  const double fx = f[3 * p], fy = f[3 * p + 1], fz = f[3 * p + 2];
  fs[s] = fx;
  fs[n + s] = fy;
  fs[2 * n + s] = fz;
  fg32[s] = make_float4(float(fx), float(fy), float(fz), 0.f);
  fg64[s] = make_double4(fx, fy, fz, 0.0);
}

// The slot arrays.  A particle's slot is its cell's first plus the cell's
// particles of smaller id (counted, so the order does not depend on the
// arrival); its thread writes all of the slot's records: one pass instead
// of a sort per cell and a pass each for positions, FP32C records and
// forces.  FP32C position record: the FP64 offset from the cell centre
// rounded to FP32, the cell's (i, j, k) packed into the fourth word, so that
// a pair displacement is (cell difference) h + (offset difference), all
// terms small, in FP32.
template <bool BATCH>
__global__ void k_slots(Grid g, const SysGrid* __restrict__ sys, const int32_t* __restrict__ sys_part, int64_t n,
                        const int32_t* __restrict__ arrived, const int32_t* __restrict__ pcell,
                        const int32_t* __restrict__ cell_start, const double* __restrict__ x,
                        const double* __restrict__ f, int32_t* __restrict__ perm, int32_t* __restrict__ slot_of,
                        int32_t* __restrict__ slot_cell, int32_t* __restrict__ sys_slot, double4* __restrict__ x4,
                        float4* __restrict__ pc, double* __restrict__ fs, float4* __restrict__ fg32,
                        double4* __restrict__ fg64) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int32_t p = arrived[t];
  const int32_t c = pcell[p];
  const int32_t a = cell_start[c], b = cell_start[c + 1];
  const double px = x[3 * int64_t(p)], py = x[3 * int64_t(p) + 1], pz = x[3 * int64_t(p) + 2];
  int32_t s = a;
  for (int32_t q = a; q < b; ++q) s += arrived[q] < p ? 1 : 0;
  perm[s] = p;
  slot_of[p] = s;
  slot_cell[s] = c;
  x4[s] = make_double4(px, py, pz, 0.0);
  const SysView v = sys_view<BATCH>(g, nullptr, 0, nullptr, sys, sys_part, p);
  if constexpr (BATCH) sys_slot[s] = sys_part[p];
  int ci, cj, ck;
  cell_ijk(v.g, c - v.coff, ci, cj, ck);
  const double cx = v.g.bmin[0] + (double(ci) + 0.5) * v.g.h[0];
  const double cy = v.g.bmin[1] + (double(cj) + 0.5) * v.g.h[1];
  const double cz = v.g.bmin[2] + (double(ck) + 0.5) * v.g.h[2];
  const uint32_t packed = uint32_t(ci) | (uint32_t(cj) << kCellBitsX) | (uint32_t(ck) << (kCellBitsX + kCellBitsY));
  pc[s] = make_float4(float(px - cx), float(py - cy), float(pz - cz), __uint_as_float(packed));
  slot_forces(n, s, p, f, fs, fg32, fg64);
}

// Forces (interleaved, particle order) -> slot SoA and gather records.
__global__ void k_gather_forces(int64_t n, const int32_t* __restrict__ perm, const double* __restrict__ f,
                                double* __restrict__ fs, float4* __restrict__ fg32, double4* __restrict__ fg64) {
  const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (s < n) slot_forces(n, s, perm[s], f, fs, fg32, fg64);
}

// ---- per-brick list builds: the brick's box cells staged in LDS ----
//
// One workgroup per brick of 8 x 8 x 8 cells.  The cell starts of the
// brick's box (the brick widened by the stencil reach) go to LDS once:
// per box cell the first slot of its grid cell and the particles of the
// box cells before it.  Each target (slot or element) of the brick then
// walks its stencil rows through LDS (box_walk_flat, box_walk_rec) or has a
// wave test the records against the stencil (wave_records), all in
// for_each_segment's order, so the lists and counts equal those of the walks
// over the global cell starts, which serve bricks whose box does not fit the
// LDS tables.
constexpr int kBrickThreads = 256;

struct BrickArgs {
  Grid g;
  const StencilRow* rows;
  int nrows;
  int32_t reach[3];
  const int32_t* cs;         // cell starts, brick order, all systems
  const int32_t* slot_cell;  // brick-order cell of each slot
  const SysGrid* sys;        // batched contexts (null: one system)
  const int32_t* sys_slot;
  int walk;                  // list_walk (list fill)
  int32_t cells_cap;         // box cells and stencil rows the LDS tables hold
  int32_t rows_cap;
  int32_t recs_cap;          // records of a brick the list fill's tables hold
  int32_t* cnt;              // [n] list lengths by slot
  int64_t* box_cnt;          // census of the staged records (k_brick_count)
  int64_t* box_ecnt;
  int32_t* box_tgt;
  // slots whose list is the one their particle kept (GGEM_COMPAT_STALE_LISTS)
  const uint8_t* stale;      // [n] or null
  const int64_t* keep_off;   // kept lists by particle (reference order)
  const int32_t* keep_ids;
  const int32_t* slot_of;
  const int32_t* perm;
};

// grid, rows and box of the brick whose first slot is sb
template <bool BATCH>
__device__ __forceinline__ SysView brick_view(const BrickArgs& a, int64_t brick, int64_t sb, BoxGeom& B) {
  const SysView v = sys_view<BATCH>(a.g, a.rows, a.nrows, a.cs, a.sys, a.sys_slot, sb);
  if constexpr (BATCH) B.init(v.g, v.coff, a.sys[a.sys_slot[sb]].reach, brick);
  else B.init(v.g, 0, a.reach, brick);
  return v;
}

__device__ __forceinline__ bool brick_staged(const BrickArgs& a, const BoxGeom& B) {
  return B.nbc <= a.cells_cap && B.fits();
}

// Slot with periodic shift code and packed box cell of every record of the
// box, after stage_box_cells; ends with a barrier.
__device__ __forceinline__ void stage_box_entries(const BoxGeom& B, const int32_t* first, const int32_t* cst,
                                                  uint32_t* rent, uint32_t* rcell) {
  for (int q = int(threadIdx.x); q < B.nbc; q += kBrickThreads) {
    const int r0 = cst[q], e = cst[q + 1];
    if (r0 == e) continue;
    int x, y, z;
    B.xyz(q, x, y, z);
    const uint32_t hi = B.shift_code(x, y, z) << kSlotBits, cell = box_pack(x, y, z);
    for (int r = r0; r < e; ++r) {
      rent[r] = uint32_t(first[q] + (r - r0)) | hi;
      rcell[r] = cell;
    }
  }
  __syncthreads();
}

constexpr int kBoxSortMax = 2048;  // targets of a brick ordered in LDS

// List lengths of the brick's slots (own element + stencil, minus itself),
// and the census of the staged records: the records of the brick's box
// (box_cnt, 0 where the brick is not staged: no targets, a box over the
// packing or more than kBoxMaxRecs records), its targets longest lists first
// (box_tgt, ties by slot; slot order in bricks that are not staged) and the
// size of its entry layout (box_ecnt: 64 x the longest list of every wave of
// that order).  Every brick writes its box_cnt and box_ecnt.
template <bool BATCH>
__global__ void __launch_bounds__(kBrickThreads) k_brick_count(BrickArgs a) {
  extern __shared__ int32_t cst[];  // [cells_cap + 1], then the stencil rows
  __shared__ int32_t s_w[kBrickThreads / 64];
  __shared__ __attribute__((aligned(16))) int32_t keys[kBoxSortMax];  // list lengths in slot order
  __shared__ int32_t skeys[kBoxSortMax];                              // the same, longest first
  __shared__ int64_t s_e[kBrickThreads / 64];
  const int64_t brick = blockIdx.x;
  const int64_t c0 = brick * kBrickCells;
  const int32_t sb = a.cs[c0], se = a.cs[c0 + kBrickCells];
  const int nt = se - sb;
  if (nt <= 0) {  // uniform over the block
    if (threadIdx.x == 0) a.box_cnt[brick] = a.box_ecnt[brick] = 0;
    return;
  }
  BoxGeom B;
  const SysView v = brick_view<BATCH>(a, brick, sb, B);
  const bool order = nt <= kBoxSortMax;
  int total = 0;
  if (brick_staged(a, B) && v.nrows <= a.rows_cap) {
    BoxRow* rt = reinterpret_cast<BoxRow*>(cst + ((a.cells_cap + 2) & ~1));
    stage_box_rows(B, v.rows, v.nrows, rt);
    stage_box_cells<kBrickThreads>(B, a.cs, nullptr, cst, s_w);
    total = cst[B.nbc];
    const int nl = walk_lanes<kBrickThreads>(nt);  // lanes per slot, each a range of the rows
    const int sub = int(threadIdx.x) & (nl - 1);
    const int r0 = v.nrows * sub / nl, r1 = v.nrows * (sub + 1) / nl;
    for (int i = int(threadIdx.x) / nl; i < nt; i += kBrickThreads / nl) {
      int ci, cj, ck;
      cell_ijk(v.g, a.slot_cell[sb + i] - v.coff, ci, cj, ck);
      int c = 0;
      box_walk_flat(rt, cst, r0, r1, B.box_cell(ci, cj, ck), [&](int p, int q) { c += q - p; });
      c = group_sum(c, nl) - 1;
      if (sub == 0) {
        a.cnt[sb + i] = c;
        if (order) keys[i] = c;
      }
    }
  } else {
    for (int i = int(threadIdx.x); i < nt; i += kBrickThreads) {
      int ci, cj, ck;
      cell_ijk(v.g, a.slot_cell[sb + i] - v.coff, ci, cj, ck);
      int c = -1;
      for_each_segment(v.g, v.rows, v.nrows, v.cs, ci, cj, ck, [&](int32_t p, int32_t q, uint32_t) { c += q - p; });
      a.cnt[sb + i] = c;
      if (order) keys[i] = c;
    }
  }
  const bool staged = total > 0 && total <= kBoxMaxRecs;
  const bool sorted = staged && order;
  if (order)
    for (int i = nt + int(threadIdx.x); i < ((nt + 3) & ~3); i += kBrickThreads) keys[i] = -1;  // (kBoxSortMax is 4k)
  __syncthreads();
  if (sorted) {
    const int4* k4 = reinterpret_cast<const int4*>(keys);
    for (int i = int(threadIdx.x); i < nt; i += kBrickThreads) {
      const int ki = keys[i];
      int r = 0;  // lengths that come before: longer ones, and equal ones of smaller slot
      for (int j = 0; j < nt; j += 4) {
        const int4 k = k4[j >> 2];
        r += (k.x > ki || (k.x == ki && j < i)) ? 1 : 0;
        r += (k.y > ki || (k.y == ki && j + 1 < i)) ? 1 : 0;
        r += (k.z > ki || (k.z == ki && j + 2 < i)) ? 1 : 0;
        r += (k.w > ki || (k.w == ki && j + 3 < i)) ? 1 : 0;
      }
      skeys[r] = ki;
      a.box_tgt[sb + r] = sb + i;
    }
    __syncthreads();
  } else {
    for (int i = int(threadIdx.x); i < nt; i += kBrickThreads) a.box_tgt[sb + i] = sb + i;
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int64_t esum = 0;
  const int nw = (nt + 63) / 64;
  for (int w = wv; w < nw; w += kBrickThreads / 64) {
    const int i = 64 * w + lane;
    const int c = i < nt ? (sorted ? skeys[i] : order ? keys[i] : a.cnt[sb + i]) : 0;
    esum += 64 * int64_t(wave_max(c));
  }
  if (lane == 0) s_e[wv] = esum;
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t e = 0;
#pragma unroll
    for (int w = 0; w < kBrickThreads / 64; ++w) e += s_e[w];
    a.box_ecnt[brick] = e;
    a.box_cnt[brick] = staged ? total : 0;
  }
}

// Slice lengths (64 x the longest list of each wave of 64 slots) and the
// pair total from the list lengths (one atomic per block of 1024).
constexpr int kSliceBlock = 1024;
__global__ void __launch_bounds__(kSliceBlock) k_slice_len(const int32_t* __restrict__ cnt, int64_t n,
                                                           int64_t* __restrict__ slice_len,
                                                           unsigned long long* __restrict__ total) {
  __shared__ int64_t s_sum[kSliceBlock / 64];
  const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t c = s < n ? cnt[s] : 0;
  int64_t mx = c, sum = c;
  for (int off = 32; off > 0; off >>= 1) {
    mx = max(mx, (int64_t)__shfl_down(mx, off, 64));
    sum += __shfl_down(sum, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    const int64_t q = s >> 6;
    if (q * 64 < n) slice_len[q] = mx * 64;
    s_sum[threadIdx.x >> 6] = sum;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t b = 0;
    for (int w = 0; w < kSliceBlock / 64; ++w) b += s_sum[w];
    if (b) atomicAdd(total, (unsigned long long)b);
  }
}

// The lists of the brick's slots in the sliced layout.  In a staged brick a
// list is its records in record order (rows in stencil order, x ascending
// through the box, slots ascending within a cell).  The record tables hold what
// the build's fullest staged brick has: sized for kBoxMaxRecs they leave six
// blocks to a CU (400,000 beads, 18 a brick, 21 rows: 301 us, now 218).
template <bool BATCH>
__global__ void __launch_bounds__(kBrickThreads) k_brick_fill_ell(BrickArgs a, const int64_t* __restrict__ slice_off,
                                                                  uint32_t* __restrict__ ell) {
  extern __shared__ int32_t lds[];
  __shared__ int32_t s_w[kBrickThreads / 64];
  int32_t* first = lds;                                                 // [cells_cap]
  int32_t* cst = lds + a.cells_cap;                                     // [cells_cap + 1]
  uint32_t* rent = reinterpret_cast<uint32_t*>(cst + a.cells_cap + 1);  // [recs_cap]
  uint32_t* rcell = rent + a.recs_cap;                                  // [recs_cap]
  BoxStencil st;
  st.ok = false;
  st.t = reinterpret_cast<uint16_t*>(rcell + a.recs_cap);               // [kStencilTab]
  const int64_t brick = blockIdx.x;
  const int64_t c0 = brick * kBrickCells;
  const int32_t sb = a.cs[c0], se = a.cs[c0 + kBrickCells];
  if (sb >= se) return;
  BoxGeom B;
  const SysView v = brick_view<BATCH>(a, brick, sb, B);
  const bool waves = wave_walk(se - sb, v.nrows, a.walk);
  int i0, i1;
  brick_share(se - sb, waves, i0, i1);
  if (i0 >= i1) return;  // uniform over the block
  bool recs = false;
  if (brick_staged(a, B)) {
    if (waves) st.init(B, v.rows, v.nrows);
    stage_box_cells<kBrickThreads>(B, a.cs, first, cst, s_w);
    recs = cst[B.nbc] <= a.recs_cap;
    if (recs) {
      stage_box_entries(B, first, cst, rent, rcell);
    }
  }
  if (waves && recs && !a.stale && st.ok) {
    // one wave per slot over the records of its z layers, 64 at a time
    for (int i = i0 + int(threadIdx.x >> 6); i < i1; i += kBrickThreads / 64) {
      const int32_t s = __builtin_amdgcn_readfirstlane(sb + i);
      int ci, cj, ck;
      cell_ijk(v.g, a.slot_cell[s] - v.coff, ci, cj, ck);
      const int q = B.box_cell(ci, cj, ck), self = cst[q] + (s - first[q]);
      const uint32_t kb = 0x808080u - box_pack(ci - B.ox, cj - B.oy, ck - B.oz);
      uint32_t* out = ell + slice_off[s >> 6] + (s & 63);
      wave_records(
          B, st, cst, ck - B.oz, [&](int r) { return r != self && st.has(rcell[r] + kb); },
          [&](int r, int k) { out[int64_t(k) * kSlice] = rent[r]; });
    }
    return;
  }
  for (int32_t s = sb + i0 + int32_t(threadIdx.x); s < sb + i1; s += kBrickThreads) {
    int ci, cj, ck;
    cell_ijk(v.g, a.slot_cell[s] - v.coff, ci, cj, ck);
    uint32_t* out = ell + slice_off[s >> 6] + (s & 63);
    if (a.stale && a.stale[s]) {  // the particle's kept list, slots by the current order
      const int32_t p = a.perm[s];
      for (int64_t q = a.keep_off[p], e = a.keep_off[p + 1]; q < e; ++q, out += kSlice)
        *out = uint32_t(a.slot_of[a.keep_ids[q]]);
      continue;
    }
    if (recs) {
      const int q = B.box_cell(ci, cj, ck);
      const int self = cst[q] + (s - first[q]);
      box_walk_rec(B, v.rows, v.nrows, cst, q, [&](int r) {
        if (r == self) return;
        *out = rent[r];
        out += kSlice;
      });
    } else {
      for_each_segment(v.g, v.rows, v.nrows, v.cs, ci, cj, ck, [&](int32_t p, int32_t q, uint32_t code) {
        const uint32_t hi = code << kSlotBits;
        for (int32_t t = p; t < q; ++t) {
          if (t == s) continue;
          *out = uint32_t(t) | hi;
          out += kSlice;
        }
      });
    }
  }
}

// Element lists of the spreading by brick (one system): element = cell,
// the own element is part of its stencil and nothing is excluded.  Every
// brick has elements, particles or not.
__global__ void __launch_bounds__(kBrickThreads) k_brick_elist_count(BrickArgs a, int64_t* __restrict__ cnt) {
  extern __shared__ int32_t cst[];  // [cells_cap + 1], then the stencil rows
  __shared__ int32_t s_w[kBrickThreads / 64];
  BoxGeom B;
  B.init(a.g, 0, a.reach, blockIdx.x);
  const bool staged = brick_staged(a, B) && a.nrows <= a.rows_cap;
  BoxRow* rt = reinterpret_cast<BoxRow*>(cst + ((a.cells_cap + 2) & ~1));
  if (staged) {
    stage_box_rows(B, a.rows, a.nrows, rt);
    stage_box_cells<kBrickThreads>(B, a.cs, nullptr, cst, s_w);
  }
  for (int l = int(threadIdx.x); l < kBrickCells; l += kBrickThreads) {
    int ci, cj, ck;
    int64_t e;
    if (!brick_elem(B, l, ci, cj, ck, e)) continue;
    int64_t c = 0;
    if (staged)
      box_walk_flat(rt, cst, 0, a.nrows, B.box_cell(ci, cj, ck), [&](int p, int q) { c += q - p; });
    else
      for_each_segment(a.g, a.rows, a.nrows, a.cs, ci, cj, ck, [&](int32_t p, int32_t q, uint32_t) { c += q - p; });
    cnt[e] = c;
  }
}

// The element lists, a wave per x-row of eight elements of a brick over the
// records of the z layers in reach, 64 at a time: the eight elements share a
// record's (dj, dk) row of the stencil and differ by one in x, and the
// matching lanes write one run of an element's list.  (69,120 elements and
// 6,400 beads in a slit: 36 us, with k_elist_fill's lane per element 83 us;
// launch_elist_fill says which where.)
// Bricks over kBoxMaxRecs records walk the rows with a lane per element, in
// the same order; boxes over the packing walk the global cell starts.
__global__ void __launch_bounds__(kBrickThreads) k_brick_elist_fill(BrickArgs a, const int64_t* __restrict__ off,
                                                                    uint32_t* __restrict__ elist) {
  extern __shared__ int32_t lds[];
  __shared__ int32_t s_w[kBrickThreads / 64];
  int32_t* first = lds;                                                 // [cells_cap]
  int32_t* cst = lds + a.cells_cap;                                     // [cells_cap + 1]
  uint32_t* rent = reinterpret_cast<uint32_t*>(cst + a.cells_cap + 1);  // [kBoxMaxRecs]
  uint32_t* rcell = rent + kBoxMaxRecs;                                 // [kBoxMaxRecs]
  BoxStencil st;
  st.t = reinterpret_cast<uint16_t*>(rcell + kBoxMaxRecs);              // [kStencilTab]
  BoxGeom B;
  B.init(a.g, 0, a.reach, blockIdx.x);
  // this block's share of the brick's 64 rows (gridDim.y blocks per brick)
  constexpr int E = 1 << kBrickBits;
  const int row0 = E * E * int(blockIdx.y) / int(gridDim.y), row1 = E * E * (int(blockIdx.y) + 1) / int(gridDim.y);
  if (!brick_staged(a, B)) {
    for (int l = E * row0 + int(threadIdx.x); l < E * row1; l += kBrickThreads) {
      int ci, cj, ck;
      int64_t e;
      if (!brick_elem(B, l, ci, cj, ck, e)) continue;
      uint32_t* out = elist + off[e];
      for_each_segment(a.g, a.rows, a.nrows, a.cs, ci, cj, ck, [&](int32_t p, int32_t q, uint32_t code) {
        for (int32_t t = p; t < q; ++t) *out++ = uint32_t(t) | (code << kSlotBits);
      });
    }
    return;
  }
  st.init(B, a.rows, a.nrows);
  stage_box_cells<kBrickThreads>(B, a.cs, first, cst, s_w);
  if (cst[B.nbc] > kBoxMaxRecs || !st.ok) {  // uniform over the block
    for (int l = E * row0 + int(threadIdx.x); l < E * row1; l += kBrickThreads) {
      int ci, cj, ck;
      int64_t e;
      if (!brick_elem(B, l, ci, cj, ck, e)) continue;
      uint32_t* out = elist + off[e];
      box_walk_rows(B, a.rows, 0, a.nrows, B.box_cell(ci, cj, ck), [&](int q0, int q1) {
        for (int q = q0; q <= q1; ++q) {
          int x, y, z;
          B.xyz(q, x, y, z);
          const uint32_t hi = B.shift_code(x, y, z) << kSlotBits;
          for (int32_t t = first[q], te = t + (cst[q + 1] - cst[q]); t < te; ++t) *out++ = uint32_t(t) | hi;
        }
      });
    }
    return;
  }
  stage_box_entries(B, first, cst, rent, rcell);
  const int lane = int(threadIdx.x) & 63, exy = B.ex * B.ey;
  for (int row = row0 + int(threadIdx.x >> 6); row < row1; row += kBrickThreads / 64) {
    int ci, cj, ck;
    int64_t e0;
    if (!brick_elem(B, E * row, ci, cj, ck, e0)) continue;  // (uniform over the wave)
    const int ne = min(E, B.n[0] - ci), bz = ck - B.oz;
    const uint32_t kb = 0x808080u - box_pack(ci - B.ox, cj - B.oy, bz);
    uint32_t* out[E];
#pragma unroll
    for (int x = 0; x < E; ++x) out[x] = elist + off[e0 + min(x, ne - 1)];
    for (int b = cst[(bz - st.rz) * exy], r1 = cst[(bz + st.rz + 1) * exy]; b < r1; b += 64) {
      const int r = b + lane;
      uint32_t w = 0x00FFu, dx = 0, ent = 0;
      if (r < r1) {
        const uint32_t d = rcell[r] + kb;
        w = st.row(d);
        dx = d & 0xffu;
        ent = rent[r];
      }
      const uint32_t lo = w & 0xffu, hi = w >> 8;
#pragma unroll
      for (int x = 0; x < E; ++x) {
        if (x >= ne) break;
        const bool in = dx >= lo + uint32_t(x) && dx <= hi + uint32_t(x);
        const uint64_t m = __ballot(in);
        if (in) out[x][__popcll(m & ((uint64_t(1) << lane) - 1))] = ent;
        out[x] += __popcll(m);
      }
    }
  }
}

// The element lists, a lane per element walking its stencil rows through the
// global cell starts: the lists of a block's consecutive elements form one
// output range, which is assembled in LDS and written with whole lines (direct
// stores when it exceeds the buffer).
constexpr int kElistLds = 10240;
__global__ void __launch_bounds__(kBlock) k_elist_fill(Grid g, const StencilRow* __restrict__ rows, int nrows,
                                                      const int32_t* __restrict__ cell_start,
                                                      const int64_t* __restrict__ off,
                                                      uint32_t* __restrict__ elist) {
  __shared__ uint32_t buf[kElistLds];
  const int64_t e0 = int64_t(blockIdx.x) * kBlock, e_end = min(e0 + int64_t(kBlock), g.n_elem);
  const int64_t base = off[e0], total = off[e_end] - base;
  const bool fits = total <= kElistLds;  // uniform over the block
  const int64_t e = e0 + threadIdx.x;
  if (e < g.n_elem) {
    int ci, cj, ck;
    elem_ijk(g, e, ci, cj, ck);
    int64_t k = off[e] - base;
    for_each_segment(g, rows, nrows, cell_start, ci, cj, ck, [&](int32_t a, int32_t b, uint32_t code) {
      const uint32_t hi = code << kSlotBits;
      for (int32_t t = a; t < b; ++t, ++k) {
        if (fits) buf[k] = uint32_t(t) | hi;
        else elist[base + k] = uint32_t(t) | hi;
      }
    });
  }
  if (!fits) return;
  __syncthreads();
  for (int64_t i = threadIdx.x; i < total; i += kBlock) elist[base + i] = buf[i];
}

// Exclusive scan of int64 values (three phases, as the int32 scan).
constexpr int kScan64Threads = 256;
constexpr int kScan64Items = 4;
constexpr int kScan64Tile = kScan64Threads * kScan64Items;

__device__ __forceinline__ int64_t block_exclusive_scan64(int64_t v, int64_t* sh, int64_t& total) {
  const int t = threadIdx.x;
  sh[t] = v;
  __syncthreads();
  for (int off = 1; off < kScan64Threads; off <<= 1) {
    const int64_t add = (t >= off) ? sh[t - off] : 0;
    __syncthreads();
    sh[t] += add;
    __syncthreads();
  }
  total = sh[kScan64Threads - 1];
  const int64_t incl = sh[t];
  __syncthreads();
  return incl - v;
}

__global__ void k_scan64_tiles(const int64_t* __restrict__ in, int64_t len, int64_t* __restrict__ out,
                               int64_t* __restrict__ tile_sums) {
  __shared__ int64_t sh[kScan64Threads];
  const int64_t base = int64_t(blockIdx.x) * kScan64Tile + int64_t(threadIdx.x) * kScan64Items;
  int64_t v[kScan64Items];
  int64_t s = 0;
#pragma unroll
  for (int q = 0; q < kScan64Items; ++q) {
    v[q] = (base + q < len) ? in[base + q] : 0;
    s += v[q];
  }
  int64_t total;
  int64_t run = block_exclusive_scan64(s, sh, total);
#pragma unroll
  for (int q = 0; q < kScan64Items; ++q) {
    if (base + q < len) out[base + q] = run;
    run += v[q];
  }
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

__global__ void k_scan64_sums(int64_t* __restrict__ sums, int64_t ntiles) {
  __shared__ int64_t sh[kScan64Threads];
  int64_t carry = 0;
  for (int64_t c0 = 0; c0 < ntiles; c0 += kScan64Threads) {
    const int64_t i = c0 + threadIdx.x;
    const int64_t v = (i < ntiles) ? sums[i] : 0;
    int64_t total;
    const int64_t ex = block_exclusive_scan64(v, sh, total);
    if (i < ntiles) sums[i] = ex + carry;
    carry += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) sums[ntiles] = carry;
}

__global__ void k_scan64_add(int64_t* __restrict__ out, int64_t len, const int64_t* __restrict__ sums,
                             int64_t ntiles) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < len) out[i] += sums[i / kScan64Tile];
  if (i == 0) out[len] = sums[ntiles];
}

// What a build leaves to the host, in one launch (up to kSizesBricks bricks):
// block 0 scans the records per brick, block 1 the entries per brick, block 2
// the slice lengths (a null input is left to launch_scan64), block 3 the maxima over the bricks
// (records, targets, unstaged bricks with targets, bricks with targets), the
// out-of-domain flag and the pair count, which it clears for the next build;
// block 4 lists the quad pair sums' blocks.  The results go straight to
// pinned host memory.
constexpr int kSizesThreads = 1024;
constexpr int kSizesItems = 4;
constexpr int64_t kSizesMax = 65536;  // most slices one block scans (16 rounds)
// More bricks than this go through k_size_tiles and k_size_fill instead: one
// block takes 4 us for every 1,024 of them
constexpr int64_t kSizesBricks = 4096;
struct SizesArgs {
  const int64_t* in[3];
  int64_t* out[3];
  int64_t len[3];
  const int32_t* cs;
  const int64_t* box_cnt;
  int64_t nbricks;
  int32_t* flag;
  int64_t* pairs;
  QuadItem* work;
  int64_t* host;  // [10] flag, pairs, records, entries, list slots, the maxima (4), work items
};
// Exclusive scan of in[len] by one block, the total to out[len] and *host
__device__ __forceinline__ void scan_sizes(const int64_t* __restrict__ in, int64_t* __restrict__ out, int64_t len,
                                           int64_t* host) {
  constexpr int NW = kSizesThreads / 64;
  __shared__ int64_t sh[NW];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int64_t carry = 0;
  for (int64_t c0 = 0; c0 < len; c0 += kSizesThreads * kSizesItems) {
    const int64_t base = c0 + int64_t(threadIdx.x) * kSizesItems;
    int64_t v[kSizesItems], mine = 0;
#pragma unroll
    for (int q = 0; q < kSizesItems; ++q) {
      v[q] = base + q < len ? in[base + q] : 0;
      mine += v[q];
    }
    int64_t incl = mine;
    for (int o = 1; o < 64; o <<= 1) {
      const int64_t y = __shfl_up(incl, o, 64);
      if (lane >= o) incl += y;
    }
    if (lane == 63) sh[wv] = incl;
    __syncthreads();
    int64_t run = carry + incl - mine, total = 0;
    for (int w = 0; w < NW; ++w) {
      if (w < wv) run += sh[w];
      total += sh[w];
    }
    carry += total;
#pragma unroll
    for (int q = 0; q < kSizesItems; ++q) {
      if (base + q < len) out[base + q] = run;
      run += v[q];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[len] = *host = carry;
}

__global__ void __launch_bounds__(kSizesThreads) k_build_sizes(SizesArgs a) {
  __shared__ int64_t sh[kSizesThreads / 64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  constexpr int NW = kSizesThreads / 64;
  if (blockIdx.x == 4) {
    __shared__ int32_t s_n[NW];
    int carry = 0;
    int64_t rcarry = 0;
    for (int64_t c0 = 0; c0 < a.nbricks; c0 += kSizesThreads) {
      const int64_t k = c0 + threadIdx.x;
      const int sb = k < a.nbricks ? a.cs[k * kBrickCells] : 0;
      const int nt = k < a.nbricks ? a.cs[(k + 1) * kBrickCells] - sb : 0;
      const int64_t nrec = k < a.nbricks ? a.box_cnt[k] : 0;
      const int m = quad_shares(nt);
      int incl = m;
      int64_t rincl = nrec;
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o, 64);
        const int64_t r = __shfl_up(rincl, o, 64);
        if (lane >= o) {
          incl += y;
          rincl += r;
        }
      }
      if (lane == 63) {
        s_n[wv] = incl;
        sh[wv] = rincl;
      }
      __syncthreads();
      int at = carry + incl - m;
      int64_t r0 = rcarry + rincl - nrec;
      for (int w = 0; w < NW; ++w) {
        if (w < wv) {
          at += s_n[w];
          r0 += sh[w];
        }
        carry += s_n[w];
        rcarry += sh[w];
      }
      for (int y = 0; y < m; ++y) {
        const int t0 = int(int64_t(nt) * y / m), t1 = int(int64_t(nt) * (y + 1) / m);
        a.work[at + y] = QuadItem{sb + t0, t1 - t0, r0 | (nrec << kItemRecShift)};
      }
      __syncthreads();
    }
    if (threadIdx.x == 0) a.host[9] = carry;
    return;
  }
  if (blockIdx.x < 3) {
    if (a.in[blockIdx.x]) scan_sizes(a.in[blockIdx.x], a.out[blockIdx.x], a.len[blockIdx.x], a.host + 2 + blockIdx.x);
    return;
  }
  int mr = 0, mt = 0, nu = 0, nf = 0;
  for (int64_t k = threadIdx.x; k < a.nbricks; k += kSizesThreads) {
    const int nt = a.cs[(k + 1) * kBrickCells] - a.cs[k * kBrickCells];
    const int nr = int(a.box_cnt[k]);
    mr = max(mr, nr);
    mt = max(mt, nt);
    nu += nt > 0 && nr == 0 ? 1 : 0;
    nf += nt > 0 ? 1 : 0;
  }
  mr = wave_max(mr);
  mt = wave_max(mt);
  nu = wave_sum(nu);
  nf = wave_sum(nf);
  __shared__ int32_t s_m[4][NW];
  if (lane == 0) {
    s_m[0][wv] = mr;
    s_m[1][wv] = mt;
    s_m[2][wv] = nu;
    s_m[3][wv] = nf;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < NW; ++w) {
      mr = max(mr, s_m[0][w]);
      mt = max(mt, s_m[1][w]);
      nu += s_m[2][w];
      nf += s_m[3][w];
    }
    a.host[0] = *a.flag;
    a.host[1] = *a.pairs;
    a.host[5] = mr;
    a.host[6] = mt;
    a.host[7] = nu;
    a.host[8] = nf;
    *a.flag = 0;
    *a.pairs = 0;
  }
}

// The sizes of a mesh of many bricks, by tiles of kSizesThreads bricks: each
// tile's totals (k_size_tiles), then each block adds up the tiles before its
// own and writes its bricks' offsets and work items; the last tile's block
// writes the totals as k_build_sizes does, and one more block scans the
// slices.  (300^3 elements, 54,872 bricks: one block each 212 us, by tiles 14
// us; 410^3, 140,608 bricks: 533 and 16 us.)
struct SizeTile {
  int64_t rec, ent;
  int32_t items, max_rec, max_tgt, unstaged, full;
};
__device__ __forceinline__ int64_t wave_sum64(int64_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
// brick k: targets, records, entries and quad work items (none past the end)
struct BrickSize {
  int sb, nt;
  int64_t rec, ent;
};
__device__ __forceinline__ BrickSize brick_size(const SizesArgs& a, int64_t k) {
  BrickSize b{0, 0, 0, 0};
  if (k < a.nbricks) {
    b.sb = a.cs[k * kBrickCells];
    b.nt = a.cs[(k + 1) * kBrickCells] - b.sb;
    b.rec = a.box_cnt[k];
    b.ent = a.in[1][k];
  }
  return b;
}
// x summed up over a wave's lanes before and with this one
template <class T>
__device__ __forceinline__ T wave_scan(T x) {
  const int lane = threadIdx.x & 63;
  for (int o = 1; o < 64; o <<= 1) {
    const T y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  return x;
}

__global__ void __launch_bounds__(kSizesThreads) k_size_tiles(SizesArgs a, SizeTile* __restrict__ tiles) {
  constexpr int NW = kSizesThreads / 64;
  __shared__ SizeTile s_t[NW];
  const BrickSize b = brick_size(a, int64_t(blockIdx.x) * kSizesThreads + threadIdx.x);
  SizeTile t;
  t.rec = wave_sum64(b.rec);
  t.ent = wave_sum64(b.ent);
  t.items = wave_sum(quad_shares(b.nt));
  t.max_rec = wave_max(int(b.rec));
  t.max_tgt = wave_max(b.nt);
  t.unstaged = wave_sum(b.nt > 0 && b.rec == 0 ? 1 : 0);
  t.full = wave_sum(b.nt > 0 ? 1 : 0);
  if ((threadIdx.x & 63) == 0) s_t[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < NW; ++w) {
    t.rec += s_t[w].rec;
    t.ent += s_t[w].ent;
    t.items += s_t[w].items;
    t.max_rec = max(t.max_rec, s_t[w].max_rec);
    t.max_tgt = max(t.max_tgt, s_t[w].max_tgt);
    t.unstaged += s_t[w].unstaged;
    t.full += s_t[w].full;
  }
  tiles[blockIdx.x] = t;
}

__global__ void __launch_bounds__(kSizesThreads) k_size_fill(SizesArgs a, const SizeTile* __restrict__ tiles,
                                                             int ntiles) {
  constexpr int NW = kSizesThreads / 64;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, tile = int(blockIdx.x);
  if (tile == ntiles) {
    if (a.in[2]) scan_sizes(a.in[2], a.out[2], a.len[2], a.host + 4);
    return;
  }
  // the tiles before this one; the last tile's block takes all tiles' maxima
  const bool last = tile == ntiles - 1;
  int64_t rec = 0, ent = 0;
  int items = 0, mr = 0, mt = 0, nu = 0, nf = 0;
  for (int k = int(threadIdx.x); k < (last ? ntiles : tile); k += kSizesThreads) {
    const SizeTile t = tiles[k];
    if (k < tile) {
      rec += t.rec;
      ent += t.ent;
      items += t.items;
    }
    mr = max(mr, t.max_rec);
    mt = max(mt, t.max_tgt);
    nu += t.unstaged;
    nf += t.full;
  }
  const int64_t k = int64_t(tile) * kSizesThreads + threadIdx.x;
  const BrickSize b = brick_size(a, k);
  const int m = quad_shares(b.nt);
  const int64_t rincl = wave_scan(b.rec), eincl = wave_scan(b.ent);
  const int iincl = wave_scan(m);
  __shared__ int64_t s_r[2][NW], s_e[2][NW];
  __shared__ int32_t s_i[2][NW], s_m[4][NW];
  rec = wave_sum64(rec);
  ent = wave_sum64(ent);
  items = wave_sum(items);
  mr = wave_max(mr);
  mt = wave_max(mt);
  nu = wave_sum(nu);
  nf = wave_sum(nf);
  if (lane == 63) {
    s_r[0][wv] = rec, s_r[1][wv] = rincl;
    s_e[0][wv] = ent, s_e[1][wv] = eincl;
    s_i[0][wv] = items, s_i[1][wv] = iincl;
    s_m[0][wv] = mr, s_m[1][wv] = mt, s_m[2][wv] = nu, s_m[3][wv] = nf;
  }
  __syncthreads();
  int64_t r0 = rincl - b.rec, e0 = eincl - b.ent;
  int at = iincl - m;
  for (int w = 0; w < NW; ++w) {
    r0 += s_r[0][w] + (w < wv ? s_r[1][w] : 0);
    e0 += s_e[0][w] + (w < wv ? s_e[1][w] : 0);
    at += s_i[0][w] + (w < wv ? s_i[1][w] : 0);
  }
  if (k < a.nbricks) {
    a.out[0][k] = r0;
    a.out[1][k] = e0;
  }
  for (int y = 0; y < m; ++y) {
    const int t0 = int(int64_t(b.nt) * y / m), t1 = int(int64_t(b.nt) * (y + 1) / m);
    a.work[at + y] = QuadItem{b.sb + t0, t1 - t0, r0 | (b.rec << kItemRecShift)};
  }
  if (!last || threadIdx.x != kSizesThreads - 1) return;  // (its offsets end at the totals)
  for (int w = 0; w < NW; ++w) {
    mr = max(mr, s_m[0][w]);
    mt = max(mt, s_m[1][w]);
  }
  nu = nf = 0;
  for (int w = 0; w < NW; ++w) {
    nu += s_m[2][w];
    nf += s_m[3][w];
  }
  a.out[0][a.nbricks] = a.host[2] = r0 + b.rec;
  a.out[1][a.nbricks] = a.host[3] = e0 + b.ent;
  a.host[0] = *a.flag;
  a.host[1] = *a.pairs;
  a.host[5] = mr;
  a.host[6] = mt;
  a.host[7] = nu;
  a.host[8] = nf;
  a.host[9] = at + m;
  *a.flag = 0;
  *a.pairs = 0;
}

// Neighbour count of every particle (own element + stencil, minus itself).
__global__ void k_count_pairs(Grid g, const StencilRow* __restrict__ rows, int nrows,
                              const int32_t* __restrict__ cell_start,
                              const int32_t* __restrict__ slot_cell,
                              const int32_t* __restrict__ perm, int64_t n,
                              int64_t* __restrict__ counts, unsigned long long* __restrict__ total) {
  const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  int64_t cnt = 0;
  if (s < n) {
    int ci, cj, ck;
    cell_ijk(g, slot_cell[s], ci, cj, ck);
    for_each_segment(g, rows, nrows, cell_start, ci, cj, ck,
                     [&](int32_t a, int32_t b, uint32_t) { cnt += b - a; });
    cnt -= 1;
    if (counts) counts[perm[s]] = cnt;
  }
  // wave reduction then one atomic per wave
  for (int off = 32; off > 0; off >>= 1) cnt += __shfl_down(cnt, off, 64);
  if ((threadIdx.x & 63) == 0 && cnt) atomicAdd(total, (unsigned long long)cnt);
}

// Reference order of a particle list: own element's particles (ascending id,
// itself removed), then the other stencil elements by ascending element id,
// each by ascending particle id.  Slots within a cell are in particle-id
// order; the tail (cells of the stencil other than the own) is sorted by
// (element id, particle id).  c: brick-order index of cell (ci, cj, ck).
__device__ void emit_list(const Grid& g, const StencilRow* rows, int nrows, const int32_t* cell_start,
                          int ci, int cj, int ck, int64_t c, int32_t self_slot, const int32_t* perm,
                          const int32_t* elem, int32_t* out) {
  const int32_t oa = cell_start[c], ob = cell_start[c + 1];
  int64_t w = 0;
  for (int32_t t = oa; t < ob; ++t)
    if (t != self_slot) out[w++] = t;
  const int64_t head = w;
  for_each_segment(g, rows, nrows, cell_start, ci, cj, ck, [&](int32_t a, int32_t b, uint32_t) {
    for (int32_t t = a; t < b; ++t)
      if (t < oa || t >= ob) out[w++] = t;
  });
  auto key = [&](int32_t t) {
    const int32_t p = perm[t];
    return (uint64_t(uint32_t(elem[p])) << 32) | uint32_t(p);
  };
  for (int64_t q = head + 1; q < w; ++q) {  // insertion sort of the tail
    const int32_t v = out[q];
    const uint64_t kv = key(v);
    int64_t t = q - 1;
    while (t >= head && key(out[t]) > kv) {
      out[t + 1] = out[t];
      --t;
    }
    out[t + 1] = v;
  }
  for (int64_t q = 0; q < w; ++q) out[q] = perm[out[q]];
}

__global__ void k_fill_csr(Grid g, const StencilRow* __restrict__ rows, int nrows,
                           const int32_t* __restrict__ cell_start,
                           const int32_t* __restrict__ slot_cell, const int32_t* __restrict__ perm,
                           const int32_t* __restrict__ elem, int64_t n, const int64_t* __restrict__ offsets,
                           int32_t* __restrict__ ids) {
  const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const int32_t p = perm[s];
  const int64_t c = slot_cell[s];
  int ci, cj, ck;
  cell_ijk(g, c, ci, cj, ck);
  emit_list(g, rows, nrows, cell_start, ci, cj, ck, c, int32_t(s), perm, elem, ids + offsets[p]);
}

// e runs over reference element ids
__global__ void k_elem_point(Grid g, const StencilRow* __restrict__ rows, int nrows,
                             const int32_t* __restrict__ cell_start,
                             const int32_t* __restrict__ perm, const int32_t* __restrict__ elem,
                             int64_t e0, int64_t ne, int64_t* __restrict__ offsets, int32_t* __restrict__ ids,
                             int pass) {
  const int64_t q = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q >= ne) return;
  const int64_t e = e0 + q;
  int ci, cj, ck;
  elem_ijk(g, e, ci, cj, ck);
  if (pass == 0) {
    int64_t cnt = 0;
    for_each_segment(g, rows, nrows, cell_start, ci, cj, ck,
                     [&](int32_t a, int32_t b, uint32_t) { cnt += b - a; });
    offsets[q + 1] = cnt;
  } else {
    emit_list(g, rows, nrows, cell_start, ci, cj, ck, cell_index(g, ci, cj, ck), -1, perm, elem,
              ids + offsets[q]);
  }
}

// PointMesh::reinit(false) (point_mesh.C:245-289 without the list
// update): the slot positions take the particles' new positions; the FP32C
// records are relative to the centre of the cell now holding the particle
// (floor, clamped), the lists, elements and slot order stay.
__global__ void k_update_slots(Grid g, int64_t n, const int32_t* __restrict__ perm, const double* __restrict__ x,
                               double4* __restrict__ x4, float4* __restrict__ pc) {
  const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const int64_t p = perm[s];
  const double v[3] = {x[3 * p], x[3 * p + 1], x[3 * p + 2]};
  int c[3];
  float o[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    double q = floor((v[d] - g.bmin[d]) / g.h[d]);
    q = q < 0.0 ? 0.0 : (q > double(g.n[d] - 1) ? double(g.n[d] - 1) : q);
    c[d] = int(q);
    o[d] = float(v[d] - (g.bmin[d] + (q + 0.5) * g.h[d]));
  }
  x4[s] = make_double4(v[0], v[1], v[2], 0.0);
  const uint32_t packed = uint32_t(c[0]) | (uint32_t(c[1]) << kCellBitsX) | (uint32_t(c[2]) << (kCellBitsX + kCellBitsY));
  pc[s] = make_float4(o[0], o[1], o[2], __uint_as_float(packed));
}

// PointParticle::set_neighbor_list (point_particle.h:189-194): a slot whose
// new list is empty keeps its particle's previous list (keep_off null: no
// previous lists).
__global__ void k_stale_patch(int64_t n, const int32_t* __restrict__ perm, const int64_t* __restrict__ keep_off,
                              int32_t* __restrict__ cnt, uint8_t* __restrict__ stale, int32_t* __restrict__ flag) {
  const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (s >= n) return;
  uint8_t st = 0;
  if (keep_off && cnt[s] == 0) {
    const int64_t p = perm[s];
    const int64_t m = keep_off[p + 1] - keep_off[p];
    if (m > 0) {
      cnt[s] = int32_t(m);
      st = 1;
      atomicOr(flag, 1);
    }
  }
  stale[s] = st;
}

// list length of every particle, by particle id
__global__ void k_counts_by_particle(int64_t n, const int32_t* __restrict__ slot_of, const int32_t* __restrict__ cnt,
                                     int64_t* __restrict__ out) {
  const int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p < n) out[p] = cnt[slot_of[p]];
}

// every particle's list in the reference's order: the kept one, or the
// stencil list of this build
__global__ void k_fill_keep(Grid g, const StencilRow* __restrict__ rows, int nrows,
                            const int32_t* __restrict__ cell_start, const int32_t* __restrict__ slot_cell,
                            const int32_t* __restrict__ perm, const int32_t* __restrict__ elem, int64_t n,
                            const uint8_t* __restrict__ stale, const int64_t* __restrict__ old_off,
                            const int32_t* __restrict__ old_ids, const int64_t* __restrict__ off,
                            int32_t* __restrict__ ids) {
  const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const int32_t p = perm[s];
  if (stale[s]) {
    for (int64_t q = old_off[p], w = off[p]; q < old_off[p + 1]; ++q, ++w) ids[w] = old_ids[q];
    return;
  }
  const int64_t c = slot_cell[s];
  int ci, cj, ck;
  cell_ijk(g, c, ci, cj, ck);
  emit_list(g, rows, nrows, cell_start, ci, cj, ck, c, int32_t(s), perm, elem, ids + off[p]);
}

__global__ void k_locate(Grid g, int64_t m, const double* __restrict__ pts, int32_t* __restrict__ elem,
                         int32_t* __restrict__ outside) {
  const int64_t q = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q >= m) return;
  const int32_t e = int32_t(locate_dev(g, pts[3 * q], pts[3 * q + 1], pts[3 * q + 2]));
  elem[q] = e;
  if (e < 0 && outside) atomicOr(outside, 1);
}

}  // namespace

hipError_t launch_clear_counters(ggem_ctx* ctx) {
  hipError_t e = hipMemsetAsync(ctx->cell_count, 0, sizeof(int32_t) * ctx->grid.n_cells, ctx->stream);
  if (e == hipSuccess) e = hipMemsetAsync(ctx->flag, 0, sizeof(int32_t), ctx->stream);
  if (e == hipSuccess) e = hipMemsetAsync(ctx->pairs_d, 0, sizeof(int64_t), ctx->stream);
  return e;
}

hipError_t launch_bin(ggem_ctx* ctx, bool hysteresis) {
  if (ctx->n == 0) return hipSuccess;
  ProfScope ps(ctx, "bin");
  if (ctx->nsys > 1)
    hipLaunchKernelGGL(k_bin<true>, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->grid,
                       ctx->sys_d, ctx->sys_part, ctx->n, ctx->x_in, ctx->elem, hysteresis ? 1 : 0,
                       ctx->pcell, ctx->prank, ctx->cell_count, ctx->flag);
  else
    hipLaunchKernelGGL(k_bin<false>, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->grid,
                       nullptr, nullptr, ctx->n, ctx->x_in, ctx->elem, hysteresis ? 1 : 0, ctx->pcell, ctx->prank,
                       ctx->cell_count, ctx->flag);
  return hipGetLastError();
}

hipError_t launch_scan(ggem_ctx* ctx) {
  const int64_t len = ctx->grid.n_cells;
  const int64_t ntiles = (len + kScanTile - 1) / kScanTile;
  ProfScope ps(ctx, "scan");
  hipLaunchKernelGGL(k_scan_tiles, dim3(unsigned(ntiles)), dim3(kScanThreads), 0, ctx->stream,
                     ctx->cell_count, len, ctx->cell_start, ctx->scan_tmp);
  const int scanned = ntiles > kScanSelfMax ? 1 : 0;
  if (scanned)
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kScanThreads), 0, ctx->stream, ctx->scan_tmp, ntiles);
  hipLaunchKernelGGL(k_scan_add, dim3(unsigned(ntiles)), dim3(kScanThreads), 0, ctx->stream, ctx->cell_start,
                     len, ctx->scan_tmp, scanned, int32_t(ctx->n));
  return hipGetLastError();
}

hipError_t launch_place(ggem_ctx* ctx) {
  if (ctx->n == 0) return hipSuccess;
  ProfScope ps(ctx, "place_sort");
  hipLaunchKernelGGL(k_place, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->n, ctx->pcell, ctx->prank,
                     ctx->cell_start, ctx->arrived);
  if (ctx->nsys > 1)
    hipLaunchKernelGGL(k_slots<true>, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->grid, ctx->sys_d,
                       ctx->sys_part, ctx->n, ctx->arrived, ctx->pcell, ctx->cell_start, ctx->x_in, ctx->f_in,
                       ctx->perm, ctx->slot_of, ctx->slot_cell, ctx->sys_slot, ctx->x4, ctx->pc32, ctx->fs, ctx->fg32,
                       ctx->fg64);
  else
    hipLaunchKernelGGL(k_slots<false>, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->grid, nullptr,
                       nullptr, ctx->n, ctx->arrived, ctx->pcell, ctx->cell_start, ctx->x_in, ctx->f_in, ctx->perm,
                       ctx->slot_of, ctx->slot_cell, nullptr, ctx->x4, ctx->pc32, ctx->fs, ctx->fg32, ctx->fg64);
  return hipGetLastError();
}

hipError_t launch_gather_forces(ggem_ctx* ctx) {
  if (ctx->n == 0) return hipSuccess;
  ProfScope ps(ctx, "gather_forces");
  hipLaunchKernelGGL(k_gather_forces, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->n,
                     ctx->perm, ctx->f_in, ctx->fs, ctx->fg32, ctx->fg64);
  return hipGetLastError();
}

BrickArgs brick_args(const ggem_ctx* ctx) {
  BrickArgs a;
  a.g = ctx->grid;
  a.rows = ctx->rows_d;
  a.nrows = ctx->n_rows;
  a.walk = list_walk(ctx);
  for (int d = 0; d < 3; ++d) a.reach[d] = ctx->reach[d];
  a.cs = ctx->cell_start;
  a.slot_cell = ctx->slot_cell;
  a.sys = ctx->nsys > 1 ? ctx->sys_d : nullptr;
  a.sys_slot = ctx->nsys > 1 ? ctx->sys_slot : nullptr;
  // LDS tables sized for the largest box of any system
  auto cells = [](const int32_t* r) {
    return ((1 << kBrickBits) + 2 * r[0]) * ((1 << kBrickBits) + 2 * r[1]) * ((1 << kBrickBits) + 2 * r[2]);
  };
  int cap = cells(ctx->reach);
  for (int k = 0; k < ctx->nsys && ctx->nsys > 1; ++k) cap = std::max(cap, cells(ctx->sys_h[k].reach));
  a.cells_cap = std::min(cap, kBoxMaxCells);
  a.rows_cap = box_rows_cap(ctx);
  a.recs_cap = ctx->max_recs;
  a.cnt = ctx->nbr_cnt;
  a.box_cnt = ctx->box_cnt;
  a.box_ecnt = ctx->box_ecnt;
  a.box_tgt = ctx->box_tgt;
  a.stale = ctx->stale_lists ? ctx->stale_slot : nullptr;
  a.keep_off = ctx->keep_off;
  a.keep_ids = ctx->keep_ids;
  a.slot_of = ctx->slot_of;
  a.perm = ctx->perm;
  return a;
}

unsigned brick_count(const ggem_ctx* ctx) { return unsigned(ctx->grid.n_cells >> (3 * kBrickBits)); }

hipError_t launch_slice_len(ggem_ctx* ctx) {
  hipLaunchKernelGGL(k_slice_len, dim3(blocks_for(ctx->n, kSliceBlock)), dim3(kSliceBlock), 0, ctx->stream,
                     ctx->nbr_cnt, ctx->n, ctx->slice_len, reinterpret_cast<unsigned long long*>(ctx->pairs_d));
  return hipGetLastError();
}

hipError_t launch_count_lists(ggem_ctx* ctx) {
  ProfScope ps(ctx, "count_lists");
  const BrickArgs a = brick_args(ctx);
  const size_t lds = sizeof(int32_t) * size_t((a.cells_cap + 2) & ~1) + sizeof(BoxRow) * size_t(a.rows_cap);
  if (a.sys)
    hipLaunchKernelGGL(k_brick_count<true>, dim3(brick_count(ctx)), dim3(kBrickThreads), lds, ctx->stream, a);
  else
    hipLaunchKernelGGL(k_brick_count<false>, dim3(brick_count(ctx)), dim3(kBrickThreads), lds, ctx->stream, a);
  return ctx->n > 0 ? launch_slice_len(ctx) : hipGetLastError();
}

size_t size_tile_bytes(const ggem_ctx* ctx) {
  const int64_t nb = int64_t(brick_count(ctx));
  return nb > kSizesBricks ? sizeof(SizeTile) * size_t((nb + kSizesThreads - 1) / kSizesThreads) : 0;
}

hipError_t launch_build_sizes(ggem_ctx* ctx, int64_t* host) {
  const int64_t nb = int64_t(brick_count(ctx)), nsl = (ctx->n + kSlice - 1) / kSlice;
  SizesArgs a;
  a.in[0] = ctx->box_cnt;
  a.in[1] = ctx->box_ecnt;
  a.in[2] = nsl > 0 && nsl <= kSizesMax ? ctx->slice_len : nullptr;
  a.out[0] = ctx->box_off;
  a.out[1] = ctx->box_eoff;
  a.out[2] = ctx->slice_off;
  a.len[0] = a.len[1] = nb;
  a.len[2] = nsl;
  if (!a.in[2]) {
    host[4] = nsl == 0 ? 0 : -1;  // no particles: no slices; many: read back by the caller
    if (nsl > 0) {
      const hipError_t e = launch_scan64(ctx, ctx->slice_len, nsl, ctx->slice_off);
      if (e != hipSuccess) return e;
    }
  }
  a.cs = ctx->cell_start;
  a.box_cnt = ctx->box_cnt;
  a.nbricks = nb;
  a.flag = ctx->flag;
  a.pairs = ctx->pairs_d;
  a.work = ctx->quad_work;
  a.host = host;
  ProfScope ps(ctx, "build_sizes");
  if (nb > kSizesBricks) {
    const unsigned ntiles = unsigned((nb + kSizesThreads - 1) / kSizesThreads);
    if (ctx->size_tiles_cap < size_tile_bytes(ctx)) return hipErrorInvalidValue;
    SizeTile* const tiles = reinterpret_cast<SizeTile*>(ctx->size_tiles);
    hipLaunchKernelGGL(k_size_tiles, dim3(ntiles), dim3(kSizesThreads), 0, ctx->stream, a, tiles);
    hipLaunchKernelGGL(k_size_fill, dim3(ntiles + 1), dim3(kSizesThreads), 0, ctx->stream, a, tiles, int(ntiles));
  } else {
    hipLaunchKernelGGL(k_build_sizes, dim3(5), dim3(kSizesThreads), 0, ctx->stream, a);
  }
  return hipGetLastError();
}

hipError_t launch_scan64(ggem_ctx* ctx, const int64_t* in, int64_t len, int64_t* out) {
  const int64_t ntiles = (len + kScan64Tile - 1) / kScan64Tile;
  if (ctx->scan64_tmp_len < ntiles + 1) return hipErrorInvalidValue;
  ProfScope ps(ctx, "scan64");
  if (ntiles > 0)
    hipLaunchKernelGGL(k_scan64_tiles, dim3(unsigned(ntiles)), dim3(kScan64Threads), 0, ctx->stream, in,
                       len, out, ctx->scan64_tmp);
  hipLaunchKernelGGL(k_scan64_sums, dim3(1), dim3(kScan64Threads), 0, ctx->stream, ctx->scan64_tmp,
                     ntiles);
  hipLaunchKernelGGL(k_scan64_add, dim3(blocks_for(len + 1)), dim3(kBlock), 0, ctx->stream, out, len,
                     ctx->scan64_tmp, ntiles);
  return hipGetLastError();
}

hipError_t launch_fill_ell(ggem_ctx* ctx) {
  if (ctx->n == 0) return hipSuccess;
  ProfScope ps(ctx, "fill_ell");
  const BrickArgs a = brick_args(ctx);
  const size_t lds =
      sizeof(int32_t) * (2 * size_t(a.cells_cap) + 1 + 2 * size_t(a.recs_cap)) + sizeof(uint16_t) * kStencilTab;
  const unsigned split = brick_split(ctx);
  if (a.sys)
    hipLaunchKernelGGL(k_brick_fill_ell<true>, dim3(brick_count(ctx), split), dim3(kBrickThreads), lds, ctx->stream, a,
                       ctx->slice_off, ctx->ell);
  else
    hipLaunchKernelGGL(k_brick_fill_ell<false>, dim3(brick_count(ctx), split), dim3(kBrickThreads), lds, ctx->stream,
                       a, ctx->slice_off, ctx->ell);
  return hipGetLastError();
}

hipError_t launch_part_sys(ggem_ctx* ctx) {
  if (ctx->n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_part_sys, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->n, ctx->nsys,
                     ctx->part_off_d, ctx->sys_part);
  return hipGetLastError();
}

hipError_t launch_elist_count(ggem_ctx* ctx) {
  ProfScope ps(ctx, "elist_count");
  const BrickArgs a = brick_args(ctx);
  const size_t lds = sizeof(int32_t) * size_t((a.cells_cap + 2) & ~1) + sizeof(BoxRow) * size_t(a.rows_cap);
  hipLaunchKernelGGL(k_brick_elist_count, dim3(brick_count(ctx)), dim3(kBrickThreads), lds, ctx->stream, a,
                     ctx->elist_off);
  return hipGetLastError();
}

hipError_t launch_elist_fill(ggem_ctx* ctx) {
  ProfScope ps(ctx, "elist_fill");
  // A lane per element or a wave per eight (k_brick_elist_fill), by the beads
  // of a brick for each stencil row: a wave reads its z layers' records for
  // eight elements' rows, a lane its rows alone, and lanes win where rows are
  // few or hold many beads, if there are elements enough.  Wave -> lane, us:
  //   rows (element)  beads a brick    700 bricks and more  340 to 512  125 and fewer
  //   69 (2.0)            45           89 -> 189            -           36 -> 92
  //   29 (3.1)            39           65 -> 86             56 -> 50    27 -> 39
  //   21 (3.9)            80           102 -> 125           43 -> 44    23 -> 34
  //   21 (3.9)           175 to 200    93 -> 86             56 -> 47    28 -> 43
  //   21 (3.9)           244           499 -> 371 (4,096)   97 -> 57    37 -> 45
  //   13 (5.0)           200           93 -> 46             -           29 -> 23
  //    9 (6.0)           500           -                    51 -> 29    27 -> 25
  const unsigned nb = brick_count(ctx);
  if (ctx->n_rows <= 16 || (nb >= 256 && ctx->n > 8 * int64_t(ctx->n_rows) * nb)) {
    hipLaunchKernelGGL(k_elist_fill, dim3(blocks_for(ctx->grid.n_elem)), dim3(kBlock), 0, ctx->stream, ctx->grid,
                       ctx->rows_d, ctx->n_rows, ctx->cell_start, ctx->elist_off, ctx->elist);
    return hipGetLastError();
  }
  const BrickArgs a = brick_args(ctx);
  const size_t lds =
      sizeof(int32_t) * (2 * size_t(a.cells_cap) + 1 + 2 * size_t(kBoxMaxRecs)) + sizeof(uint16_t) * kStencilTab;
  // few bricks: several blocks each, to reach every CU (of 512 to 1,023
  // bricks two where the walk outweighs a second staging: 80 beads a brick
  // and 29 rows 70 -> 58 us, 10 beads and 69 rows 44 -> 59)
  const bool one = nb >= 1024 || (nb >= 512 && 2 * ctx->n < 3 * int64_t(ctx->n_rows) * nb);
  const unsigned split = one ? 1u : nb >= 256 ? 2u : 4u;
  hipLaunchKernelGGL(k_brick_elist_fill, dim3(nb, split), dim3(kBrickThreads), lds, ctx->stream, a, ctx->elist_off,
                     ctx->elist);
  return hipGetLastError();
}

hipError_t launch_count_pairs(ggem_ctx* ctx, int64_t* counts_d) {
  ctx->counters_clear = false;
  hipError_t e = hipMemsetAsync(ctx->pairs_d, 0, sizeof(int64_t), ctx->stream);
  if (e != hipSuccess || ctx->n == 0) return e;
  hipLaunchKernelGGL(k_count_pairs, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->grid,
                     ctx->rows_d, ctx->n_rows, ctx->cell_start, ctx->slot_cell, ctx->perm, ctx->n,
                     counts_d, reinterpret_cast<unsigned long long*>(ctx->pairs_d));
  return hipGetLastError();
}

hipError_t launch_fill_csr(ggem_ctx* ctx, const int64_t* offsets_d, int32_t* ids_d) {
  if (ctx->n == 0) return hipSuccess;
  ProfScope ps(ctx, "fill_csr");
  hipLaunchKernelGGL(k_fill_csr, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->grid,
                     ctx->rows_d, ctx->n_rows, ctx->cell_start, ctx->slot_cell, ctx->perm, ctx->elem, ctx->n,
                     offsets_d, ids_d);
  return hipGetLastError();
}

hipError_t launch_elem_point_csr(ggem_ctx* ctx, int64_t e0, int64_t ne, int64_t* offsets_d,
                                 int32_t* ids_d, int pass) {
  if (ne == 0) return hipSuccess;
  hipLaunchKernelGGL(k_elem_point, dim3(blocks_for(ne)), dim3(kBlock), 0, ctx->stream, ctx->grid,
                     ctx->rows_d, ctx->n_rows, ctx->cell_start, ctx->perm, ctx->elem, e0, ne, offsets_d, ids_d,
                     pass);
  return hipGetLastError();
}

hipError_t launch_update_slots(ggem_ctx* ctx) {
  if (ctx->n == 0) return hipSuccess;
  ProfScope ps(ctx, "update_slots");
  hipLaunchKernelGGL(k_update_slots, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->grid, ctx->n,
                     ctx->perm, ctx->x_in, ctx->x4, ctx->pc32);
  return hipGetLastError();
}

hipError_t launch_stale_patch(ggem_ctx* ctx, bool have_kept) {
  ctx->counters_clear = false;
  hipError_t e = hipMemsetAsync(ctx->flag, 0, sizeof(int32_t), ctx->stream);
  if (e == hipSuccess) e = hipMemsetAsync(ctx->pairs_d, 0, sizeof(int64_t), ctx->stream);
  if (e != hipSuccess || ctx->n == 0) return e;
  ProfScope ps(ctx, "stale_lists");
  hipLaunchKernelGGL(k_stale_patch, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->n, ctx->perm,
                     have_kept ? ctx->keep_off : nullptr, ctx->nbr_cnt, ctx->stale_slot, ctx->flag);
  return launch_slice_len(ctx);
}

hipError_t launch_counts_by_particle(ggem_ctx* ctx, int64_t* out) {
  if (ctx->n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_counts_by_particle, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->n,
                     ctx->slot_of, ctx->nbr_cnt, out);
  return hipGetLastError();
}

hipError_t launch_fill_keep(ggem_ctx* ctx, const int64_t* old_off, const int32_t* old_ids, const int64_t* off,
                            int32_t* ids) {
  if (ctx->n == 0) return hipSuccess;
  ProfScope ps(ctx, "stale_lists");
  hipLaunchKernelGGL(k_fill_keep, dim3(blocks_for(ctx->n)), dim3(kBlock), 0, ctx->stream, ctx->grid, ctx->rows_d,
                     ctx->n_rows, ctx->cell_start, ctx->slot_cell, ctx->perm, ctx->elem, ctx->n, ctx->stale_slot,
                     old_off, old_ids, off, ids);
  return hipGetLastError();
}

hipError_t launch_locate(ggem_ctx* ctx, int64_t m, const double* pts, int32_t* elem, int32_t* outside) {
  if (m == 0) return hipSuccess;
  hipLaunchKernelGGL(k_locate, dim3(blocks_for(m)), dim3(kBlock), 0, ctx->stream, ctx->grid, m, pts,
                     elem, outside);
  return hipGetLastError();
}

}  // namespace ggem
