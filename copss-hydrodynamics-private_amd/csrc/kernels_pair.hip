// kernels_pair.hip -- (b) the local regularized-Stokeslet pair sum
// u_i = sum_{j in nbr(i)} G_reg(x_j - x_i) f_j, and the mobility and
// Chebyshev applications built on it.
//
// Reference: GGEMStokes::local_solution_bead (ggem_stokes.C:427-503),
// local_solution_field (:360-424), green_tensor_local_regularized
// (:304-357), global_self_exclusion (:506-523), the velocity combination of
// PMSystemStokes::compute_point_velocity (pm_system_stokes.C:441-457) and the
// Chebyshev vector updates (brownian_system.C:1037-1041, :1093-1101).
//
// The targets' neighbour lists are stored sliced by wave (entry k of lane l
// of slice q at slice_off[q] + 64k + l): every list access of a wave is one
// coalesced transaction.  Positions do not move between neighbour builds,
// so pair tensors are evaluated once per build and streamed by every later
// application (the local velocity, each Chebyshev term, M y).  FP64:
// k_tensors stores G = A I + sgn w w^T, w = sqrt(|Bx|) x_ij (32 bytes per
// entry) in list order and k_apply streams them, gathering one operand
// record per neighbour.  FP32C, one operand: per brick of cells the
// neighbours' records are staged in LDS and the entries stream a 2-byte
// record number (k_box_fill, k_apply_box, k_apply_quad, below).  FP32C,
// several operands: k_apply_quad, four lanes per target, and in dense bricks
// k_apply_box_nr, one.  The explicit minimum image, bricks that are not
// staged: k_apply evaluates (A, Bx) per pair from the coefficient table in
// LDS.  Blocks are
// renumbered per XCD so a chip partition keeps a contiguous stretch of
// cells and their neighbours in its L2.
//
// FP64: the reference's formula with libm-class erf/exp.  FP32C: x_ij from
// the cell-relative FP32 position records ((cell difference) h + offset
// difference), (A, Bx) from a piecewise polynomial in r^2, partial sums in
// FP32 merged every 8 neighbours into a Kahan accumulator; the epilogue
// (combination, recurrence) runs in FP64.
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "ggem_device.h"

namespace ggem {

namespace {

constexpr int kBlock = 256;
constexpr int kMergeEvery = 8;

inline unsigned blocks_for(int64_t n, int b = kBlock) { return unsigned((n + b - 1) / b); }

struct PairArgs {
  Grid g;
  GGEMConst k;
  GGEMConst32 k32;
  const double4* x4;
  const int32_t* cnt;
  const int64_t* slice_off;
  const uint32_t* ell;
  const int32_t* perm;
  const double* fs;  // own forces (FP64 SoA) for the mobility epilogue
  int64_t n;
  double bsign;
  const SysGrid* sys;       // batched contexts: grid of each system
  const int32_t* sys_slot;  // and system of each slot
  const float4* pc32;       // FP32C position records (cell-relative offsets, packed cell)
  int32_t xcd;              // renumber blocks per XCD (xcd_block)
  int32_t exact;            // explicit minimum image (no list shift codes)
  const float4* tab;        // FP32C (A, Bx) as a piecewise polynomial in r^2, 4 float4 per interval
  CoefTab ct;
};

// FP32C (A, Bx) at s = r^2 from the interval table (copied to LDS): the
// interval and y = 2 (s - mid)/d are formed exactly (widths are powers of
// two), then two degree-7 Horner chains; past the cut-off the last
// interval is zero.  One body for every FP32C kernel, so they all
// evaluate bit-identical tensors.
// The interval of s and y in it.  The last interval (index t.n - 1) is the
// zero one: its pairs are skipped by every FP32C pair sum (fp32c_kept),
// which add exactly the same terms in the same order whether they store the
// kept pairs or test each entry.
__device__ __forceinline__ int fp32c_interval(const CoefTab& t, float s, float& y) {
  const bool r2 = s >= t.s1;
  const float base = r2 ? t.s1 : 0.f;
  const float inv = r2 ? t.inv2 : t.inv1;
  const float d = r2 ? t.d2 : t.d1;
  const int j = min(int((s - base) * inv), r2 ? t.n2 : t.n1 - 1);
  const float mid = __builtin_fmaf(float(j) + 0.5f, d, base);
  y = (s - mid) * (2.f * inv);
  return (r2 ? t.n1 : 0) + j;
}
__device__ __forceinline__ bool fp32c_kept(const CoefTab& t, int i) { return i < t.n - 1; }
// fp32c_interval for a table of one width (n2 = 0, so s1 lies at or past
// the cut): the same arithmetic below s1; s >= s1 gives the zero interval
__device__ __forceinline__ int fp32c_interval1(const CoefTab& t, float s, float& y) {
  const int j = min(int(s * t.inv1), t.n1);
  const float mid = __builtin_fmaf(float(j) + 0.5f, t.d1, 0.f);
  y = (s - mid) * (2.f * t.inv1);
  return j;
}

// (A, Bx) at y in interval i of the table's LDS copy (load_tab: the four
// coefficient quadruples of an interval padded to kTabStride, so that lanes
// at different intervals spread over the LDS banks and the four reads
// share one address)
constexpr int kTabStride = 5;
__device__ __forceinline__ void fp32c_eval(const float4* __restrict__ tab, int i, float y, float& A, float& Bx) {
  const float4* t = tab + __mul24(i, kTabStride);  // (a full-rate multiply)
  const float4 a0 = t[0], a1 = t[1], b0 = t[2], b1 = t[3];
  float pa = __builtin_fmaf(a1.w, y, a1.z);
  pa = __builtin_fmaf(pa, y, a1.y);
  pa = __builtin_fmaf(pa, y, a1.x);
  pa = __builtin_fmaf(pa, y, a0.w);
  pa = __builtin_fmaf(pa, y, a0.z);
  pa = __builtin_fmaf(pa, y, a0.y);
  A = __builtin_fmaf(pa, y, a0.x);
  float pb = __builtin_fmaf(b1.w, y, b1.z);
  pb = __builtin_fmaf(pb, y, b1.y);
  pb = __builtin_fmaf(pb, y, b1.x);
  pb = __builtin_fmaf(pb, y, b0.w);
  pb = __builtin_fmaf(pb, y, b0.z);
  pb = __builtin_fmaf(pb, y, b0.y);
  Bx = __builtin_fmaf(pb, y, b0.x);
}

// r^2 of an FP32C displacement, one fixed evaluation order
__device__ __forceinline__ float fp32c_r2(float dx, float dy, float dz) {
  return __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
}

// p += A f + Bx (x . f) x with every product fused explicitly, so that no
// kernel is left a choice of contraction: all FP32C pair sums add
// bit-identical terms
__device__ __forceinline__ void fp32c_acc(float A, float Bx, float dx, float dy, float dz, float fx, float fy,
                                          float fz, float& p0, float& p1, float& p2) {
  const float b = Bx * __builtin_fmaf(dz, fz, __builtin_fmaf(dy, fy, dx * fx));
  p0 += __builtin_fmaf(A, fx, b * dx);
  p1 += __builtin_fmaf(A, fy, b * dy);
  p2 += __builtin_fmaf(A, fz, b * dz);
}

// G f = A f + sgn (w . f) w with the stored FP64 (A, w) = c, every product
// fused explicitly, so that all FP64 pair sums add bit-identical terms
__device__ __forceinline__ void fp64_acc(const double4& c, double sg, const double4& f, double& p0, double& p1,
                                         double& p2) {
  const double wf = sg * __builtin_fma(c.w, f.z, __builtin_fma(c.z, f.y, c.y * f.x));
  p0 += __builtin_fma(c.x, f.x, wf * c.y);
  p1 += __builtin_fma(c.x, f.y, wf * c.z);
  p2 += __builtin_fma(c.x, f.z, wf * c.w);
}

// the interval table into LDS: quadruple c of interval i (a.tab[4 i + c])
// to dst[kTabStride i + c] (the whole block takes part)
__device__ __forceinline__ void load_tab(float4* dst, const PairArgs& a) {
  for (int q = threadIdx.x; q < 4 * a.ct.n; q += blockDim.x) dst[kTabStride * (q >> 2) + (q & 3)] = a.tab[q];
}

// Launch shapes the autotuner chooses from (index 0 is the default); every
// shape computes the same per-slot arithmetic, so results do not depend on
// the choice.
struct Shape {
  int block, xcd;
};
constexpr Shape kApplyShapes[] = {{256, 1}, {128, 1}, {512, 1}, {64, 1}, {256, 0}};
constexpr int kNApply = sizeof(kApplyShapes) / sizeof(kApplyShapes[0]);
constexpr Shape kTensorShapes[] = {{256, 1}, {128, 1}, {512, 1}, {64, 1}};
constexpr int kNTensor = sizeof(kTensorShapes) / sizeof(kTensorShapes[0]);

__device__ __forceinline__ int64_t block_index(int xcd) {
  return xcd ? xcd_block(blockIdx.x, gridDim.x) : int64_t(blockIdx.x);
}

// Grid of a slot's system.
template <bool BATCH>
__device__ __forceinline__ const Grid& slot_grid(const PairArgs& a, int64_t s) {
  if constexpr (BATCH) return a.sys[a.sys_slot[s]].g;
  else return a.g;
}

template <class T>
struct V4;
template <>
struct V4<float> {
  using type = float4;
};
template <>
struct V4<double> {
  using type = double4;
};

// FP64 pair tensors of all list entries: (A, w) with G = A I + sgn w w^T.
// gridDim.y threads share a slot's entries (every gridDim.y-th one each):
// one entry is a chain of a gather, two erf and two exp, so a few thousand
// slots with one thread each left the chip idle (3,001 beads: 65 us, with
// eight threads a slot 12.5 us).
template <bool EXACT, bool BATCH, int BLK>
__global__ void __launch_bounds__(BLK) k_tensors(PairArgs a, double4* __restrict__ c64) {
  const int64_t s = block_index(a.xcd) * BLK + threadIdx.x;
  if (s >= a.n) return;
  const Grid& g = slot_grid<BATCH>(a, s);
  const int cnt = a.cnt[s];
  const int64_t base = a.slice_off[s >> 6] + (s & 63);
  const uint32_t* lst = a.ell + base;
  const double4 xs = a.x4[s];
  const int k0 = int(blockIdx.y), dk = int(gridDim.y), last = cnt - 1;
  if (k0 > last) return;
  uint32_t e1 = lst[uint32_t(k0) * uint32_t(kSlice)];
  uint32_t e2 = lst[uint32_t(min(k0 + dk, last)) * uint32_t(kSlice)];
  double4 xa = a.x4[e1 & kSlotMask];
  for (int k = k0; k < cnt; k += dk) {
    const uint32_t e = e1;
    const double4 xt = xa;
    e1 = e2;
    xa = a.x4[e1 & kSlotMask];
    e2 = lst[uint32_t(min(k + 2 * dk, last)) * uint32_t(kSlice)];
    double dx, dy, dz;
    pair_disp<EXACT>(g, xs, xt, e >> kSlotBits, dx, dy, dz);
    const int64_t o = base + int64_t(k) * kSlice;
    double A, Bx;
    green_coef_f64(a.k, dx * dx + dy * dy + dz * dz, A, Bx);
    const double sb = sqrt(fabs(Bx));
    c64[o] = make_double4(A, sb * dx, sb * dy, sb * dz);
  }
}

// What the epilogue of a target slot reads once for all its components.
struct EpiTarget {
  double da, db, ck, cm1, c0;  // EPI_CHEB
};
template <int EPI>
__device__ __forceinline__ EpiTarget epi_target(const PairArgs& a, int64_t s, const ChebEpi& epi) {
  EpiTarget T{epi.da, epi.db, epi.c, epi.cm1, epi.c0};
  if (EPI == EPI_CHEB && epi.dpar) {
    const double* pp = epi.dpar + int64_t(epi.sys ? epi.sys[s] : 0) * epi.pstride;
    T.da = pp[0];
    T.db = pp[1];
    T.ck = pp[2 + epi.term];
    if (epi.ymask & 1) T.cm1 = pp[epi.term];
    if (epi.ymask & 2) T.c0 = pp[1 + epi.term];
  }
  return T;
}

// What the epilogue of component q of target slot s and operand r reads
// besides the pair sum: a kernel with a short pair loop loads it ahead.
struct EpiIn {
  double xv;  // own force, own component of the operand
  double xm;  // u_glob; x_{k-1}
  double y, my;
  int64_t p;  // EPI_LOCAL, EPI_MOBILITY: particle of the slot
};
template <int EPI>
__device__ __forceinline__ EpiIn epi_in(const PairArgs& a, int64_t s, int r, int q,
                                        const double* __restrict__ xsoa, const ChebEpi& epi,
                                        const double* __restrict__ u_glob) {
  EpiIn I{0.0, 0.0, 0.0, 0.0, 0};
  if constexpr (EPI == EPI_LOCAL || EPI == EPI_MOBILITY) {
    I.xv = a.fs[q * a.n + s];  // forces are the operand: own force from the FP64 store
    I.p = a.perm[s];
    if (EPI == EPI_MOBILITY && u_glob) I.xm = u_glob[3 * I.p + q];
  } else {
    const int64_t idx = int64_t(r) * 3 * a.n + int64_t(q) * a.n + s;
    I.xv = xsoa[idx];
    if constexpr (EPI == EPI_REF) {
      if (epi.ref.term != 0) {
        I.y = epi.y[idx];
        I.my = epi.ref.my[idx];
        I.xm = epi.xm1.soa[idx];
      }
    } else if (epi.kind > 1) {
      I.xm = epi.xm1.soa[idx];
      if (epi.ymask) I.y = epi.y[idx];
    }
  }
  return I;
}

// Epilogue of component q of the pair sum of target slot s for operand r, m
// the sum (see Epi) and I = epi_in(...); the value of the new vector
// (EPI_CHEB, EPI_REF), whose gather record is left to epi_record.
template <int EPI>
__device__ __forceinline__ double epi_component(const PairArgs& a, const EpiTarget& T, const EpiIn& I, int64_t s,
                                                int r, int q, double m, const SlotVec& v, const ChebEpi& epi,
                                                double* __restrict__ out, double (&dots)[3]) {
  const int64_t n = a.n;
  if constexpr (EPI == EPI_LOCAL || EPI == EPI_MOBILITY) {
    const double fo = I.xv;
    double u = m;
    if (a.k.point_type == GGEM_LAGRANGIAN_POINT) u += a.k.coeff_2 * fo;  // self term
    if (EPI == EPI_MOBILITY) {
      const double ug = I.xm;
      if (a.k.point_type == GGEM_POLYMER_BEAD) u = ug + u - a.k.coeff_1 * fo + fo;
      else if (a.k.point_type == GGEM_LAGRANGIAN_POINT) u = ug + u;
      else u = 0.0;
    }
    out[3 * I.p + q] = u;
    return u;
  } else {
    const int64_t idx = int64_t(r) * 3 * n + int64_t(q) * n + s;
    const double xv = I.xv;
    if (a.k.point_type == GGEM_POLYMER_BEAD) m = m - a.k.coeff_1 * xv + xv;
    else if (a.k.point_type == GGEM_LAGRANGIAN_POINT) m = m + a.k.coeff_2 * xv;
    else m = 0.0;
    double nv;
    if constexpr (EPI == EPI_REF) {
      const RefEpi& R = epi.ref;
      double y = R.c * xv, my = R.c * m;
      if (R.term == 0) {
        nv = T.db * xv + T.da * m;
        dots[0] += m * xv;
      } else {
        y += I.y;
        my += I.my;
        nv = 2. * T.db * xv + 2. * T.da * m - I.xm;
        dots[0] += my * my;
      }
      dots[1] += y * y;
      dots[2] += xv * xv;
      epi.y[idx] = y;
      R.my[idx] = my;
    } else if (epi.kind == 0) {
      nv = m;
    } else if (epi.kind == 1) {
      nv = T.db * xv + T.da * m;
    } else {
      const double xm = I.xm;
      nv = 2. * T.db * xv + 2. * T.da * m;
      nv += -1.0 * xm;
      if (epi.ymask == 4) {
        epi.y[idx] = I.y + T.ck * nv;
      } else if (epi.ymask) {  // x_{k-1}, x_k and x_{k+1} terms in one update of y
        double add = 0.0;
        if (epi.ymask & 1) add += T.cm1 * xm;
        if (epi.ymask & 2) add += T.c0 * xv;
        if (epi.ymask & 4) add += T.ck * nv;
        epi.y[idx] = I.y + add;
      }
    }
    v.soa[idx] = nv;
    return nv;
  }
}
// gather record of the new vector, operand r of NR
template <int NR, int EPI>
__device__ __forceinline__ void epi_record(int64_t n, int64_t s, int r, double x, double y, double z,
                                           const SlotVec& v) {
  if constexpr (EPI == EPI_CHEB || EPI == EPI_REF) {
    if (v.g32) v.g32[gather_index(false, NR, n, s, r)] = make_float4(float(x), float(y), float(z), 0.f);
    if (v.g64) v.g64[gather_index(true, NR, n, s, r)] = make_double4(x, y, z, 0.0);
  }
}

// Epilogue of the pair sums of target slot s, one thread
template <int NR, int EPI>
__device__ __forceinline__ void apply_epilogue(const PairArgs& a, int64_t s, const double (&acc)[NR][3],
                                               const double* __restrict__ xsoa, const SlotVec& v,
                                               const ChebEpi& epi, const double* __restrict__ u_glob,
                                               double* __restrict__ out, double (&dots)[3]) {
  const EpiTarget T = epi_target<EPI>(a, s, epi);
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    double nv[3];
#pragma unroll
    for (int q = 0; q < 3; ++q)
      nv[q] = epi_component<EPI>(a, T, epi_in<EPI>(a, s, r, q, xsoa, epi, u_glob), s, r, q, acc[r][q], v, epi, out,
                                 dots);
    epi_record<NR, EPI>(a.n, s, r, nv[0], nv[1], nv[2], v);
  }
}

// value of v in lane M of the lane's quad (four consecutive lanes)
template <int M>
__device__ __forceinline__ int quad_get(int v) {
  return __builtin_amdgcn_mov_dpp(v, M * 0x55, 0xf, 0xf, true);
}
template <int M>
__device__ __forceinline__ float quad_get(float v) {
  return __int_as_float(quad_get<M>(__float_as_int(v)));
}
template <int M>
__device__ __forceinline__ double quad_get(double v) {
  return __hiloint2double(quad_get<M>(__double2hiint(v)), quad_get<M>(__double2loint(v)));
}
// p + v of lane 0 + .. + v of lane 3 of the quad, in that order
template <class T>
__device__ __forceinline__ T quad_add(T p, T v) {
  p += quad_get<0>(v);
  p += quad_get<1>(v);
  p += quad_get<2>(v);
  p += quad_get<3>(v);
  return p;
}

// Epilogue of the pair sum of target slot s of a quad whose lanes all hold
// it: lane c < 3 takes component c, with I = epi_in(..., c, ...)
template <int EPI>
__device__ __forceinline__ void quad_epilogue(const PairArgs& a, const EpiTarget& T, const EpiIn& I, int64_t s, int c,
                                              double m0, double m1, double m2, const SlotVec& v, const ChebEpi& epi,
                                              double* __restrict__ out, double (&dots)[3]) {
  double nv = 0.0;
  if (c < 3) nv = epi_component<EPI>(a, T, I, s, 0, c, c == 0 ? m0 : (c == 1 ? m1 : m2), v, epi, out, dots);
  const double x = quad_get<0>(nv), y = quad_get<1>(nv), z = quad_get<2>(nv);
  if (c == 0) epi_record<1, EPI>(a.n, s, 0, x, y, z, v);
}

// the block's sums of three values, on every thread (one barrier pair)
__device__ __forceinline__ void block_add3(double (&t)[3]) {
  __shared__ double sh[3][16];
#pragma unroll
  for (int q = 0; q < 3; ++q)
    for (int o = 32; o > 0; o >>= 1) t[q] += __shfl_down(t[q], o, 64);
  const int nw = int(blockDim.x >> 6);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int q = 0; q < 3; ++q) sh[q][threadIdx.x >> 6] = t[q];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    t[q] = 0.0;
    for (int w = 0; w < nw; ++w) t[q] += sh[q][w];
  }
  __syncthreads();
}

// The estimators and the stopping rule of a reference-mode term from its three
// dot products t (one thread)
__device__ __forceinline__ void ref_rule(const RefEpi& R, const double (&t)[3]) {
  if (R.term == 0) {
    R.st[0] = t[0];
  } else {
    const double aux2 = R.st[0], aux4 = sqrt(R.st[1]), aux3 = sqrt(t[2]) * fabs(R.c), aux1 = t[0];
    double err1 = R.st[4], err2 = R.st[5];
    if (aux2 != 0.0) err1 = sqrt(fabs(aux1 - aux2) / aux2);
    if (aux4 != 0.0) err2 = aux3 / aux4;
    R.st[4] = err1;
    R.st[5] = err2;
    R.st[6] = double(R.term);
    if (R.check) {
      if (err1 <= R.tol) {
        R.st[7] = 1.0;
        *R.stop = 1;
      } else if (err2 <= 1E-9) {
        *R.stop = 1;
      }
    }
  }
  R.st[1] = t[1];
}

// The whole block's sums of the three dot products over parts b0 .. b1 - 1 of
// nb, as load(q nb + b) reads them
template <class Load>
__device__ __forceinline__ void ref_sum(int b0, int b1, int nb, double (&t)[3], Load&& load) {
#pragma unroll
  for (int q = 0; q < 3; ++q) t[q] = 0.0;
  constexpr int U = 4;  // parts in flight per thread and product
  for (int b = b0 + int(threadIdx.x); b < b1; b += U * int(blockDim.x)) {
    double w[U][3];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int bu = min(b + u * int(blockDim.x), b1 - 1);
#pragma unroll
      for (int q = 0; q < 3; ++q) w[u][q] = load(int64_t(q) * nb + bu);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (b + u * int(blockDim.x) < b1)
#pragma unroll
        for (int q = 0; q < 3; ++q) t[q] += w[u][q];
  }
  block_add3(t);
}

// The decision by the launch's last block to finish: every block's parts t go
// to memory past the XCD's L2 (agent scope), and the last block adds all of
// them (in block order, whichever block that is) and applies the stopping
// rule.  Tickets are drawn in kRefGroups groups, a group's last block drawing
// one of the top: a single ticket's atomics follow one another at 11 ns each
// (700 blocks: 8 us).
__device__ __forceinline__ void ref_tickets(const RefEpi& R, double (&t)[3]) {
  __shared__ int s_last;
  const int nb = int(gridDim.x), id = int(blockIdx.x);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < 3; ++q)
      __hip_atomic_store(R.part + int64_t(q) * nb + id, t[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int g = id % kRefGroups, groups = min(nb, kRefGroups), in_group = (nb - g + kRefGroups - 1) / kRefGroups;
    bool last = __hip_atomic_fetch_add(R.ticket + 1 + g, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == in_group - 1;
    if (last) last = __hip_atomic_fetch_add(R.ticket, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == groups - 1;
    s_last = last;
  }
  __syncthreads();
  if (!s_last) return;  // uniform over the block
  ref_sum(0, nb, nb, t, [&](int64_t i) {
    return __hip_atomic_load(R.part + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  });
  if (threadIdx.x <= kRefGroups) R.ticket[threadIdx.x] = 0;  // (blocks have 64 threads or more)
  if (threadIdx.x == 0) ref_rule(R, t);
}

// End of a reference-mode launch, the whole block with its parts of the
// three dot products: the decision in the launch itself where it has few
// blocks (one launch per term instead of six: per-term dot products, gather
// records and the deciding kernel were 16 us of the 66 us a term took for
// 25,600 chain beads), else the parts left to k_ref_decide (null ticket).
__device__ __forceinline__ void ref_finish(const ChebEpi& epi, const double (&dots)[3]) {
  const RefEpi& R = epi.ref;
  double t[3] = {dots[0], dots[1], dots[2]};
  block_add3(t);
  if (R.ticket) {
    ref_tickets(R, t);
  } else if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < 3; ++q) R.part[int64_t(q) * gridDim.x + blockIdx.x] = t[q];
  }
}

// The decision of a launch of many blocks, over the nb parts it left (nothing
// after the stop): a ticket's release writes the XCD's L2 back, 20 to 40 ns a
// block while the pair sums' results are in it.  Per term, one more launch
// against tickets, us: 3,000 beads (125 blocks) 13.4 and 12.8; 8,000 (343)
// 14.5 and 17.6; 26,000 (1,000) 16.8 and 34.5; 120,000 (4,096) 37 and 131;
// 400,000 (50,653) 227 and 1,267.  One block for every kRefDecideParts parts.
constexpr int kRefDecideThreads = 1024, kRefDecideParts = 8192;
__global__ void __launch_bounds__(kRefDecideThreads) k_ref_decide(RefEpi R, const double* __restrict__ parts, int nb) {
  if (*R.stop) return;  // uniform over the grid: set by the block that finishes last
  const int b0 = int(int64_t(nb) * blockIdx.x / gridDim.x), b1 = int(int64_t(nb) * (blockIdx.x + 1) / gridDim.x);
  double t[3];
  ref_sum(b0, b1, nb, t, [&](int64_t i) { return parts[i]; });
  if (gridDim.x > 1) ref_tickets(R, t);
  else if (threadIdx.x == 0) ref_rule(R, t);
}

// Output of one target: m = sum over its list of G_ij x_j for NR operand
// vectors, then the epilogue.
template <int P, int NR, int EPI, int BLK>
__global__ void __launch_bounds__(BLK) k_apply(PairArgs a, const void* __restrict__ coef_raw,
                                                 const double4* __restrict__ xg64,
                                                 const float4* __restrict__ xg32,
                                                 const double* __restrict__ xsoa, SlotVec v,
                                                 ChebEpi epi, const double* __restrict__ u_glob,
                                                 double* __restrict__ out) {
  // (the tensor pointer is untyped in the signature: a type computed from
  // the header's unnamed precision enum would be mangled differently by the
  // host and device compilations; FP32C keeps no tensors)
  if (epi.skip && *epi.skip) return;  // uniform over the grid
  const int64_t s = block_index(a.xcd) * BLK + threadIdx.x;
  const float4* tab = nullptr;
  if constexpr (P != GGEM_FP64) {
    __shared__ float4 s_tab[kTabStride * kTabMaxIntervals];
    load_tab(s_tab, a);
    __syncthreads();
    tab = s_tab;
  }
  double dots[3] = {0.0, 0.0, 0.0};
  auto body = [&]() {
  const int cnt = a.cnt[s];
  const int64_t base = a.slice_off[s >> 6] + (s & 63);
  const uint32_t* lst = a.ell + base;
  double acc[NR][3];
  // Groups of U entries: the entries of the next group are loaded one group
  // ahead, and the U tensors and operand records of a group are all
  // requested before the first is used (memory-level parallelism for the
  // dependent gathers).  The summation order is the list order.
  constexpr int U = NR >= 4 ? 1 : (NR == 2 ? 2 : 4);
  const int last = cnt > 0 ? cnt - 1 : 0;

  if constexpr (P == GGEM_FP64) {
    uint32_t en[U];
#pragma unroll
    for (int i = 0; i < U; ++i) en[i] = cnt > 0 ? lst[uint32_t(min(i, last)) * uint32_t(kSlice)] : 0u;
    const double4* __restrict__ cf = static_cast<const double4*>(coef_raw) + base;
    const double4* __restrict__ xg = xg64;
    const double sg = a.bsign;
    double ps[NR][3];
#pragma unroll
    for (int r = 0; r < NR; ++r) ps[r][0] = ps[r][1] = ps[r][2] = 0.0;
    // G f = A f + sgn (w . f) w with the stored (A, w)
    auto pair_acc = [&](const double4& c, const double4* f) {
#pragma unroll
      for (int r = 0; r < NR; ++r) fp64_acc(c, sg, f[r], ps[r][0], ps[r][1], ps[r][2]);
    };
    int k = 0;
    for (; k + U <= cnt; k += U) {
      uint32_t e[U];
      double4 c[U];
#pragma unroll
      for (int i = 0; i < U; ++i) {
        e[i] = en[i];
        en[i] = lst[uint32_t(min(k + U + i, last)) * uint32_t(kSlice)];
        c[i] = cf[int64_t(k + i) * kSlice];
      }
      double4 f[U][NR];
#pragma unroll
      for (int i = 0; i < U; ++i)
#pragma unroll
        for (int r = 0; r < NR; ++r) f[i][r] = xg[gather_index(true, NR, a.n, e[i] & kSlotMask, r)];
#pragma unroll
      for (int i = 0; i < U; ++i) pair_acc(c[i], f[i]);
    }
#pragma unroll
    for (int i = 0; i < U - 1; ++i) {
      if (k + i < cnt) {  // entries en[0 .. cnt - k)
        double4 f[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) f[r] = xg[gather_index(true, NR, a.n, en[i] & kSlotMask, r)];
        pair_acc(cf[int64_t(k + i) * kSlice], f);
      }
    }
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int q = 0; q < 3; ++q) acc[r][q] = ps[r][q];
  } else {
    // FP32C: G f = A f + Bx (x . f) x with x_ij from the cell-relative FP32
    // positions, x_ij = (cell_t - cell_s + shift) h + (offset_t - offset_s)
    // per axis, and (A, Bx) from the table at r^2
    const float4* __restrict__ xg = xg32;
    const float4* __restrict__ pc = a.pc32;
    const Grid& g = a.sys ? a.sys[a.sys_slot[s]].g : a.g;
    uint32_t en[U];  // entries of the next group
#pragma unroll
    for (int i = 0; i < U; ++i) en[i] = cnt > 0 ? lst[uint32_t(min(i, last)) * uint32_t(kSlice)] : 0u;
    const float hx = float(g.h[0]), hy = float(g.h[1]), hz = float(g.h[2]);
    const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
    const float Lx = float(g.L[0]), Ly = float(g.L[1]), Lz = float(g.L[2]);
    const int px = g.periodic[0], py = g.periodic[1], pz = g.periodic[2];
    const float4 po = pc[s];
    const uint32_t co = __float_as_uint(po.w);
    const int io = int(co & ((1u << kCellBitsX) - 1));
    const int jo = int((co >> kCellBitsX) & ((1u << kCellBitsY) - 1));
    const int ko = int(co >> (kCellBitsX + kCellBitsY));
    float ps[NR][3];
    KahanF kh[NR][3];
#pragma unroll
    for (int r = 0; r < NR; ++r) ps[r][0] = ps[r][1] = ps[r][2] = 0.f;
    auto disp = [&](uint32_t e, const float4& pt, float& dx, float& dy, float& dz) {
      const uint32_t ct = __float_as_uint(pt.w);
      int di = int(ct & ((1u << kCellBitsX) - 1)) - io;
      int dj = int((ct >> kCellBitsX) & ((1u << kCellBitsY) - 1)) - jo;
      int dk = int(ct >> (kCellBitsX + kCellBitsY)) - ko;
      const uint32_t code = e >> kSlotBits;
      if (!a.exact) {  // the entry's single periodic shift, in cells
        di += (int(code & 1u) - int((code >> 1) & 1u)) * nx;
        dj += (int((code >> 2) & 1u) - int((code >> 3) & 1u)) * ny;
        dk += (int((code >> 4) & 1u) - int((code >> 5) & 1u)) * nz;
      } else {  // the nearest image of the cell difference, exact in integers
        if (px) di = 2 * di > nx ? di - nx : (2 * di < -nx ? di + nx : di);
        if (py) dj = 2 * dj > ny ? dj - ny : (2 * dj < -ny ? dj + ny : dj);
        if (pz) dk = 2 * dk > nz ? dk - nz : (2 * dk < -nz ? dk + nz : dk);
      }
      dx = __builtin_fmaf(float(di), hx, pt.x - po.x);
      dy = __builtin_fmaf(float(dj), hy, pt.y - po.y);
      dz = __builtin_fmaf(float(dk), hz, pt.z - po.z);
      if (a.exact) {  // minimum image (pm_periodic_boundary.C:350-374)
        if (px) dx = dx <= -0.5f * Lx ? dx + Lx : (dx > 0.5f * Lx ? dx - Lx : dx);
        if (py) dy = dy <= -0.5f * Ly ? dy + Ly : (dy > 0.5f * Ly ? dy - Ly : dy);
        if (pz) dz = dz <= -0.5f * Lz ? dz + Lz : (dz > 0.5f * Lz ? dz - Lz : dz);
      }
    };
    // kept pairs are summed and merged every kMergeEvery of them; the zero
    // interval's pairs are skipped (nk counts the kept ones)
    int nk = 0;
    auto merge = [&]() {
      if ((nk & (kMergeEvery - 1)) == 0) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            kh[r][q].add(ps[r][q]);
            ps[r][q] = 0.f;
          }
      }
    };
    auto pair_acc = [&](uint32_t e, const float4& pt, const float4* f) {
      float dx, dy, dz;
      disp(e, pt, dx, dy, dz);
      float y;
      const int it = fp32c_interval(a.ct, fp32c_r2(dx, dy, dz), y);
      if (!fp32c_kept(a.ct, it)) return;
      float A, Bx;
      fp32c_eval(tab, it, y, A, Bx);
#pragma unroll
      for (int r = 0; r < NR; ++r) fp32c_acc(A, Bx, dx, dy, dz, f[r].x, f[r].y, f[r].z, ps[r][0], ps[r][1], ps[r][2]);
      ++nk;
      merge();
    };
    int k = 0;
    for (; k + U <= cnt; k += U) {
      uint32_t c[U];
      float4 pt[U];
#pragma unroll
      for (int i = 0; i < U; ++i) {
        c[i] = en[i];
        en[i] = lst[uint32_t(min(k + U + i, last)) * uint32_t(kSlice)];
      }
      float4 f[U][NR];
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const uint32_t t = c[i] & kSlotMask;
        pt[i] = pc[t];
#pragma unroll
        for (int r = 0; r < NR; ++r) f[i][r] = xg[gather_index(false, NR, a.n, t, r)];
      }
#pragma unroll
      for (int i = 0; i < U; ++i) pair_acc(c[i], pt[i], f[i]);
    }
#pragma unroll
    for (int i = 0; i < U - 1; ++i) {
      if (k + i < cnt) {  // entries en[0 .. cnt - k)
        const uint32_t t = en[i] & kSlotMask;
        float4 f[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) f[r] = xg[gather_index(false, NR, a.n, t, r)];
        pair_acc(en[i], pc[t], f);
      }
    }
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        kh[r][q].add(ps[r][q]);
        acc[r][q] = kh[r][q].value();
      }
  }

  apply_epilogue<NR, EPI>(a, s, acc, xsoa, v, epi, u_glob, out, dots);
  };
  if (s < a.n) body();
  if constexpr (EPI == EPI_REF) ref_finish(epi, dots);
}


// ---- FP32C pair sum with the neighbour records staged in LDS ----
//
// One workgroup per brick of 8 x 8 x 8 cells.  The brick's box is the brick
// widened by the stencil reach (periodic images unwrapped); each particle of
// the box is one record, in box order: box cells x-major through the box,
// particles of a cell in slot order, so a stencil run of box cells is one
// range of records.  Once per list build k_box_fill writes every staged
// brick's records (slot, cell-relative FP32 position with the packed box
// cell) and finds each target's among them in list order (wave_records,
// box_walk_rec): per kept entry the neighbour's record number (16 bits).
// k_apply_box copies the records, their operands and the coefficient table
// to LDS and streams the record numbers (2 bytes per pair): per pair the
// neighbour from LDS and (A, Bx) from the table at the displacement, a
// group of entries at a time (records first, then intervals, then tensors
// and sums) so that the LDS reads of a group overlap.  The summation order
// (list order) and the arithmetic are k_apply's; the displacement (box_t -
// box_s) h + (offset_t - offset_s) has the same integer cell difference as
// the list entry's periodic shift gives, so the results are bit-identical.
// A brick whose box holds more than kBoxMaxRecs records reads its list and
// gathers the neighbours' records from global memory.
constexpr int kBoxThreads = 256;
// FP64 with a lane per target in dense bricks or few (dense64): threads for
// twice 256 targets.  A block of 256 goes round a second time in every brick
// with more (23 of 100 at 244 targets a brick), with a few lanes and at the
// latency of a whole list; the further threads cost nothing there and help to
// stage.  125,000 beads: 41.6 -> 35.2 us per application, and 34.2 us with the
// tensors loaded a group ahead (211 MB at 6.1 TB/s).
// FP32C is not bound by that latency (1M beads: 82.7 us either way).
constexpr int kDenseThreads = 512;
// A target's packed entry base: the offset of its entry 0 (below 2^40), its
// own record number (12 bits) and, in staged bricks, its count of stored
// (kept) entries (12 bits; a staged box holds at most kBoxMaxRecs records).
constexpr int kBaseBits = 40;
constexpr int64_t kBaseMask = (int64_t(1) << kBaseBits) - 1;
constexpr int kSelfShift = kBaseBits, kKeptShift = kBaseBits + 12;
constexpr uint64_t kField12 = 0xFFFu;

struct BoxArgs {
  const int32_t* cs;     // cell starts, brick order
  int32_t reach[3];      // stencil reach of a plain context
  const int64_t* off;    // [n_bricks + 1] first record of each brick
  const int64_t* eoff;   // [n_bricks + 1] first entry of each brick
  const int32_t* tgt;    // [n] slots of each brick, longest lists first (staged bricks)
  int64_t* base;         // [n] entry 0 of the target at each position of tgt (low kBaseBits),
                         // its own record in a staged brick (above)
  uint32_t* slot;        // [records] slot of each record
  float4* pos;           // [records] offset xyz, packed box cell
  uint16_t* idx;         // [entries] neighbour's record number (staged bricks): FP32C brick layout,
                         // FP64 the lists' slice layout
  int32_t cells_cap;     // k_box_fill: box cells, waves and records of a brick its LDS tables hold
  int32_t waves_cap;
  int32_t recs_cap;
  int32_t fp64;          // FP64: every pair stored, at its list position
  uint32_t* ell;         // FP64: the lists themselves, written along (null: already filled)
  const StencilRow* rows;  // stencil rows (a batched context: all systems', SysGrid::row_off)
  int32_t nrows;
  int walk;  // list_walk
};

// What the staged pair sums read of the layout (their kernel arguments
// stay small)
struct BoxView {
  const int32_t* cs;
  int32_t reach[3];
  const int64_t* off;
  const int32_t* tgt;
  const int64_t* base;
  const uint32_t* slot;
  const float4* pos;
  const uint16_t* idx;
  const QuadItem* work;  // k_apply_quad: what every block sums
};

// Entry layout of a brick: its targets in the order tgt, in waves of 64;
// entry k of the target at position i = 64 w + l lies at
// eoff + 64 (W_0 + .. + W_{w-1}) + 64 k + l, W_w being the longest list of
// wave w.  Staged bricks order their targets by list length, longest first
// (ties by slot), so the lanes of a wave do similar work.
constexpr int kBoxMaxWaves = kBoxMaxTargets / 64;  // waves of one brick

// Box of the brick holding first_slot (the slot picks the system of a
// batched context).
__device__ __forceinline__ void box_init(BoxGeom& B, const PairArgs& a, const int32_t* reach, int64_t brick,
                                         int64_t first_slot) {
  if (a.sys) {
    const SysGrid* S = a.sys + a.sys_slot[first_slot];
    B.init(S->g, S->cell_off, S->reach, brick);
  } else {
    B.init(a.g, 0, reach, brick);
  }
}

// Records of staged bricks, the entry layout of every brick's targets, and
// in staged bricks each entry's neighbour record number.  Launches that walk by
// lanes alone have an instance without the wave walk, whose registers cost them
// 8% (1M beads, 72 targets a brick: 272 -> 250 us).
template <bool BATCH, bool WAVES>
__global__ void __launch_bounds__(kBoxThreads) k_box_fill(PairArgs a, BoxArgs b) {
  extern __shared__ float4 dyn[];
  float4* rpos = dyn;                                                  // [recs_cap] records of a staged brick
  int32_t* cfirst = reinterpret_cast<int32_t*>(rpos + b.recs_cap);     // [cells_cap] first slot of each box cell
  int32_t* cst = cfirst + b.cells_cap;                                 // [cells_cap + 1] record start of each box cell
  int32_t* wpre = cst + b.cells_cap + 1;                               // [waves_cap + 1] entry rows before each wave
  __shared__ int32_t s_w[kBoxThreads / 64];
  __shared__ uint16_t s_st[kStencilTab];
  uint32_t* rent = reinterpret_cast<uint32_t*>(wpre + b.waves_cap + 1);  // [recs_cap] list entry of each record (ell)
  const int64_t brick = blockIdx.x;
  const int64_t c0 = brick * kBrickCells;
  const int32_t sb = b.cs[c0], se = b.cs[c0 + kBrickCells];
  if (sb >= se) return;
  const int nt = se - sb;
  const StencilRow* rows = b.rows;
  int nrows = b.nrows;
  if constexpr (BATCH) {
    const SysGrid& S = a.sys[a.sys_slot[sb]];
    rows += S.row_off;
    nrows = S.nrows;
  }
  const bool waves = WAVES && wave_walk(nt, nrows, b.walk);
  int t0, t1;  // this block's share of the targets
  brick_share(nt, waves, t0, t1);
  if (t0 >= t1) return;  // uniform over the block
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t r0 = b.off[brick];
  const int nrec = int(b.off[brick + 1] - r0);
  BoxGeom B;
  box_init(B, a, b.reach, brick, sb);
  BoxStencil st;
  st.t = s_st;
  st.ok = false;
  if (nrec > 0) {
    if (waves) st.init(B, rows, nrows);
    // (1) first slots and record starts of the box cells (the total is nrec),
    // (2) the records: record i lies in the last box cell whose start is <= i
    stage_box_cells<kBoxThreads>(B, b.cs, cfirst, cst, s_w);
    int top = 1;  // largest power of two below nbc
    while (2 * top < B.nbc) top *= 2;
    constexpr int G = 4;  // records per thread and step, their searches and loads interleaved
    for (int i0 = int(threadIdx.x); i0 < nrec; i0 += G * kBoxThreads) {
      int lo[G], ii[G];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        ii[u] = min(i0 + u * kBoxThreads, nrec - 1);
        lo[u] = 0;
      }
      for (int step = top; step > 0; step >>= 1)
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const int m = lo[u] + step;
          if (m < B.nbc && cst[m] <= ii[u]) lo[u] = m;
        }
      int64_t t[G];
      float4 p[G];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        t[u] = int64_t(cfirst[lo[u]]) + (ii[u] - cst[lo[u]]);
        p[u] = a.pc32[t[u]];
      }
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int i = i0 + u * kBoxThreads;
        if (i >= nrec) break;
        int x, y, z;
        B.xyz(lo[u], x, y, z);
        const uint32_t packed = box_pack(x, y, z);
        const float4 rec = make_float4(p[u].x, p[u].y, p[u].z, __uint_as_float(packed));
        if (t0 == 0) {
          b.slot[r0 + i] = uint32_t(t[u]);
          b.pos[r0 + i] = rec;
        }
        rpos[i] = rec;
        if (b.ell) rent[i] = uint32_t(t[u]) | (B.shift_code(x, y, z) << kSlotBits);
      }
    }
  }
  // (3) the entry layout: the longest list of every wave of the order,
  // exclusive prefix (the host keeps nt within kBoxMaxWaves waves)
  const int nw = (nt + 63) / 64;
  for (int w = wv; w < nw; w += kBoxThreads / 64) {
    const int i = 64 * w + lane;
    const int m = wave_max(i < nt ? a.cnt[b.tgt[sb + i]] : 0);
    if (lane == 0) wpre[w] = m;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int run = 0;
    for (int w = 0; w < nw; ++w) {
      const int m = wpre[w];
      wpre[w] = run;
      run += m;
    }
  }
  __syncthreads();
  // (4) the entries of the staged bricks' targets, in record order: the
  // neighbour's record number of every kept pair (outside the table's zero
  // interval at the FP32C displacement, formed exactly as the list-order
  // kernel forms it); FP64: of every pair, at its position in the lists'
  // slice layout.  The targets of other bricks keep their entry offset only.
  const float hx = B.h[0], hy = B.h[1], hz = B.h[2];
  const bool all = b.fp64 != 0;
  struct Target {
    float4 po;
    uint32_t kb;
    int q, z, self;
  };
  auto target = [&](int64_t s) {
    Target T;
    T.po = a.pc32[s];
    const uint32_t co = __float_as_uint(T.po.w);
    const int x = int(co & ((1u << kCellBitsX) - 1)) - B.ox;
    const int y = int((co >> kCellBitsX) & ((1u << kCellBitsY) - 1)) - B.oy;
    T.z = int(co >> (kCellBitsX + kCellBitsY)) - B.oz;
    T.kb = 0x808080u - box_pack(x, y, T.z);
    T.q = (T.z * B.ey + y) * B.ex + x;
    T.self = cst[T.q] + int(s - cfirst[T.q]);  // the target's own record
    return T;
  };
  auto keeps = [&](const Target& T, const float4& pt) {
    float di, dj, dk;
    box_diff(__float_as_uint(pt.w), T.kb, di, dj, dk);
    const float dx = __builtin_fmaf(di, hx, pt.x - T.po.x);
    const float dy = __builtin_fmaf(dj, hy, pt.y - T.po.y);
    const float dz = __builtin_fmaf(dk, hz, pt.z - T.po.z);
    float y;
    return fp32c_kept(a.ct, fp32c_interval(a.ct, fp32c_r2(dx, dy, dz), y));
  };
  auto entries = [&](int64_t s, int64_t bb) { return b.idx + (all ? a.slice_off[s >> 6] + (s & 63) : bb); };
  auto packed = [&](const Target& T, int64_t bb, int kept) {
    return all ? bb : bb | (int64_t(T.self) << kSelfShift) | (int64_t(kept) << kKeptShift);
  };
  if (waves && nrec > 0 && st.ok) {
    for (int i = t0 + wv; i < t1; i += kBoxThreads / 64) {  // one wave per target
      const int32_t s = __builtin_amdgcn_readfirstlane(b.tgt[sb + i]);
      const int64_t bb = b.eoff[brick] + 64 * int64_t(wpre[i >> 6]) + (i & 63);
      const Target T = target(s);
      uint16_t* __restrict__ out = entries(s, bb);
      uint32_t* __restrict__ lst = b.ell ? b.ell + a.slice_off[s >> 6] + (s & 63) : nullptr;
      const int kept = wave_records(
          B, st, cst, T.z,
          [&](int r) {
            const float4 pt = rpos[r];
            return r != T.self && st.has(__float_as_uint(pt.w) + T.kb) && (all || keeps(T, pt));
          },
          [&](int r, int k) {
            out[int64_t(k) * kSlice] = uint16_t(r);
            if (lst) lst[int64_t(k) * kSlice] = rent[r];
          });
      if (lane == 0) b.base[sb + i] = packed(T, bb, kept);
    }
    return;
  }
  for (int i = t0 + int(threadIdx.x); i < t1; i += kBoxThreads) {
    const int64_t s = b.tgt[sb + i];
    const int64_t bb = b.eoff[brick] + 64 * int64_t(wpre[i >> 6]) + (i & 63);
    if (nrec == 0) {
      b.base[sb + i] = bb;  // unstaged brick: the pair sum reads its list
      continue;
    }
    const Target T = target(s);
    uint16_t* out = entries(s, bb);
    uint32_t* lst = b.ell ? b.ell + a.slice_off[s >> 6] + (s & 63) : nullptr;
    int kept = 0;
    box_walk_rec(B, rows, nrows, cst, T.q, [&](int r) {
      if (r == T.self || !(all || keeps(T, rpos[r]))) return;
      *out = uint16_t(r);
      out += kSlice;
      if (lst) {
        *lst = rent[r];
        lst += kSlice;
      }
      ++kept;
    });
    b.base[sb + i] = packed(T, bb, kept);
  }
}

// pair sum of slot s through global gathers (FP32C, one operand; the
// coefficient table in LDS)
__device__ __forceinline__ void fp32c_pairs_global(const PairArgs& a, int64_t s, const float4* __restrict__ tab,
                                                   const float4* __restrict__ xg, double (&acc)[1][3]) {
  const int cnt = a.cnt[s];
  const int64_t base = a.slice_off[s >> 6] + (s & 63);
  const Grid& g = a.sys ? a.sys[a.sys_slot[s]].g : a.g;
  const float hx = float(g.h[0]), hy = float(g.h[1]), hz = float(g.h[2]);
  const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
  const float4 po = a.pc32[s];
  const uint32_t co = __float_as_uint(po.w);
  const int io = int(co & ((1u << kCellBitsX) - 1));
  const int jo = int((co >> kCellBitsX) & ((1u << kCellBitsY) - 1));
  const int ko = int(co >> (kCellBitsX + kCellBitsY));
  float ps[3] = {0.f, 0.f, 0.f};
  KahanF kh[3];
  int nk = 0;  // kept pairs so far
  for (int k = 0; k < cnt; ++k) {
    const uint32_t e = a.ell[base + int64_t(k) * kSlice];
    const uint32_t t = e & kSlotMask;
    const float4 pt = a.pc32[t];
    const float4 f = xg[t];
    const uint32_t ct = __float_as_uint(pt.w);
    const uint32_t code = e >> kSlotBits;
    const int di = int(ct & ((1u << kCellBitsX) - 1)) - io + (int(code & 1u) - int((code >> 1) & 1u)) * nx;
    const int dj = int((ct >> kCellBitsX) & ((1u << kCellBitsY) - 1)) - jo +
                   (int((code >> 2) & 1u) - int((code >> 3) & 1u)) * ny;
    const int dk = int(ct >> (kCellBitsX + kCellBitsY)) - ko + (int((code >> 4) & 1u) - int((code >> 5) & 1u)) * nz;
    const float dx = __builtin_fmaf(float(di), hx, pt.x - po.x);
    const float dy = __builtin_fmaf(float(dj), hy, pt.y - po.y);
    const float dz = __builtin_fmaf(float(dk), hz, pt.z - po.z);
    float y;
    const int it = fp32c_interval(a.ct, fp32c_r2(dx, dy, dz), y);
    if (!fp32c_kept(a.ct, it)) continue;  // the zero interval
    float A, Bx;
    fp32c_eval(tab, it, y, A, Bx);
    fp32c_acc(A, Bx, dx, dy, dz, f.x, f.y, f.z, ps[0], ps[1], ps[2]);
    if ((++nk & (kMergeEvery - 1)) == 0) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        kh[q].add(ps[q]);
        ps[q] = 0.f;
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    kh[q].add(ps[q]);
    acc[0][q] = kh[q].value();
  }
}

template <int EPI, bool ONE>  // ONE: the table has one interval width
__global__ void __launch_bounds__(kBoxThreads) k_apply_box(PairArgs a, BoxView b, const float4* __restrict__ xg,
                                                          const double* __restrict__ xsoa, SlotVec v, ChebEpi epi,
                                                          const double* __restrict__ u_glob,
                                                          double* __restrict__ out) {
  extern __shared__ float4 lds[];
  if (epi.skip && *epi.skip) return;  // uniform over the grid
  const int64_t brick = block_index(a.xcd);
  const int64_t c0 = brick * kBrickCells;
  const int32_t sb = b.cs[c0], se = b.cs[c0 + kBrickCells];
  double dots[3] = {0.0, 0.0, 0.0};
  if (sb >= se) {  // no targets (uniform over the block)
    if constexpr (EPI == EPI_REF) ref_finish(epi, dots);
    return;
  }
  const int64_t r0 = b.off[brick];
  const int nrec = int(b.off[brick + 1] - r0);
  const int nt = se - sb;
  float4* s_tab = lds;                         // coefficient table
  float4* rpos = lds + kTabStride * a.ct.n;    // [nrec] offset xyz, packed box cell
  float4* rval = rpos + nrec;         // [nrec] operand
  load_tab(s_tab, a);
  if (nrec == 0) {
    __syncthreads();
    for (int i = int(threadIdx.x); i < nt; i += kBoxThreads) {
      const int64_t s = b.tgt[sb + i];
      double acc[1][3];
      fp32c_pairs_global(a, s, s_tab, xg, acc);
      apply_epilogue<1, EPI>(a, s, acc, xsoa, v, epi, u_glob, out, dots);
    }
    if constexpr (EPI == EPI_REF) ref_finish(epi, dots);
    return;
  }
  {
    // four records in flight per thread, then the remainder one at a time
    int i = int(threadIdx.x);
    for (; i + 3 * kBoxThreads < nrec; i += 4 * kBoxThreads) {
      const uint32_t t0 = b.slot[r0 + i], t1 = b.slot[r0 + i + kBoxThreads];
      const uint32_t t2 = b.slot[r0 + i + 2 * kBoxThreads], t3 = b.slot[r0 + i + 3 * kBoxThreads];
      const float4 p0 = b.pos[r0 + i], p1 = b.pos[r0 + i + kBoxThreads];
      const float4 p2 = b.pos[r0 + i + 2 * kBoxThreads], p3 = b.pos[r0 + i + 3 * kBoxThreads];
      const float4 f0 = xg[t0], f1 = xg[t1], f2 = xg[t2], f3 = xg[t3];
      rpos[i] = p0;
      rpos[i + kBoxThreads] = p1;
      rpos[i + 2 * kBoxThreads] = p2;
      rpos[i + 3 * kBoxThreads] = p3;
      rval[i] = f0;
      rval[i + kBoxThreads] = f1;
      rval[i + 2 * kBoxThreads] = f2;
      rval[i + 3 * kBoxThreads] = f3;
    }
    for (; i < nrec; i += kBoxThreads) {
      rpos[i] = b.pos[r0 + i];
      rval[i] = xg[b.slot[r0 + i]];
    }
  }
  __syncthreads();
  BoxGeom B;
  box_init(B, a, b.reach, brick, sb);
  const float hx = B.h[0], hy = B.h[1], hz = B.h[2];
  constexpr int U = 4;  // entries per group, the next group's record numbers loaded one ahead
  for (int i = int(threadIdx.x); i < nt; i += kBoxThreads) {
    const int64_t s = b.tgt[sb + i];
    const int64_t bpk = b.base[sb + i];
    const int64_t base = bpk & kBaseMask;
    const float4 po = rpos[int((uint64_t(bpk) >> kSelfShift) & kField12)];  // the target's own record
    const uint32_t kb = 0x808080u - __float_as_uint(po.w);
    const int cnt = int((uint64_t(bpk) >> kKeptShift) & kField12);  // stored (kept) entries
    float ps[3] = {0.f, 0.f, 0.f};
    KahanF kh[3];
    // displacement to record rec and its interval in the table (every
    // stored entry is a kept pair)
    auto disp = [&](const float4& pt, float& dx, float& dy, float& dz, float& y) {
      float di, dj, dk;
      box_diff(__float_as_uint(pt.w), kb, di, dj, dk);
      dx = __builtin_fmaf(di, hx, pt.x - po.x);
      dy = __builtin_fmaf(dj, hy, pt.y - po.y);
      dz = __builtin_fmaf(dk, hz, pt.z - po.z);
      return ONE ? fp32c_interval1(a.ct, fp32c_r2(dx, dy, dz), y) : fp32c_interval(a.ct, fp32c_r2(dx, dy, dz), y);
    };
    auto merge = [&](int k) {
      if ((k & (kMergeEvery - 1)) == kMergeEvery - 1) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          kh[q].add(ps[q]);
          ps[q] = 0.f;
        }
      }
    };
    auto one = [&](uint32_t rec, int k) {
      const float4 pt = rpos[rec];
      const float4 f = rval[rec];
      float dx, dy, dz, y, A, Bx;
      const int it = disp(pt, dx, dy, dz, y);
      fp32c_eval(s_tab, it, y, A, Bx);
      fp32c_acc(A, Bx, dx, dy, dz, f.x, f.y, f.z, ps[0], ps[1], ps[2]);
      merge(k);
    };
    if (cnt > 0) {  // an empty list has no storage
      const uint16_t* __restrict__ ci = b.idx + base;
      const int last = cnt - 1;
      uint32_t en[U];  // record numbers of the next group
#pragma unroll
      for (int u = 0; u < U; ++u) en[u] = ci[int64_t(min(u, last)) * kSlice];
      int k = 0;
      for (; k + U <= cnt; k += U) {
        uint32_t c[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          c[u] = en[u];
          en[u] = ci[int64_t(min(k + U + u, last)) * kSlice];
        }
        // a group: its records, then displacements and intervals, then the
        // tensors from the table and the sums in list order
        float4 pt[U], f[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          pt[u] = rpos[c[u]];
          f[u] = rval[c[u]];
        }
        float dx[U], dy[U], dz[U], y[U];
        int it[U];
#pragma unroll
        for (int u = 0; u < U; ++u) it[u] = disp(pt[u], dx[u], dy[u], dz[u], y[u]);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          float A, Bx;
          fp32c_eval(s_tab, it[u], y[u], A, Bx);
          fp32c_acc(A, Bx, dx[u], dy[u], dz[u], f[u].x, f[u].y, f[u].z, ps[0], ps[1], ps[2]);
          merge(k + u);
        }
      }
#pragma unroll
      for (int u = 0; u < U - 1; ++u)
        if (k + u < cnt) one(en[u], k + u);  // entries en[0 .. cnt - k)
    }
    double acc[1][3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      kh[q].add(ps[q]);
      acc[0][q] = kh[q].value();
    }
    apply_epilogue<1, EPI>(a, s, acc, xsoa, v, epi, u_glob, out, dots);
  }
  if constexpr (EPI == EPI_REF) ref_finish(epi, dots);
}


// The staged pair sum with four lanes (a quad) per target, for NR operands
// (in which bricks: quad_lanes).
// One operand: lane c takes entries c, c + 4, ...; the four terms of a step
// are added in list order by every lane (quad_add).  Several operands: lane c
// forms the displacement and the tensor of its entry, then the quad goes
// through the four entries together and lane c sums operands c, c + 4, ...
// (NR = 2: c mod 2).  Sums, merge points and epilogue are k_apply's for NR
// operands, bit for bit.  A block takes one item of the work list, a brick's share
// of about kQuadShare targets.
// A lane per target leaves most of a block idle in bricks with few targets
// (20,000 beads: 39 of 256 lanes) and walks each list alone: one operand 9.1
// -> 6.6 us per application there, 30 -> 21 us for chains in a slit (25,600
// beads).  Several operands used to gather from global memory, a lane per
// target: eight of 20,000 beads 34.8 -> 12.8 us, four of 272,000 beads in 64
// suspensions 176 -> 128 us (16 records staged per target, three blocks per
// CU in LDS).
// A block of 39 targets is a chain of dependent loads, not work: the item
// word holds what took two more loads, and the first target's words, record
// numbers and epilogue inputs are requested while the records are staged
// (20,000 beads 6.6 -> 5.6 us, chains 21.9 -> 21.1 us).
template <int EPI, bool ONE, int NR>
__global__ void __launch_bounds__(kBoxThreads) k_apply_quad(PairArgs a, BoxView b, const float4* __restrict__ xg,
                                                           const double* __restrict__ xsoa, SlotVec v, ChebEpi epi,
                                                           const double* __restrict__ u_glob,
                                                           double* __restrict__ out) {
  extern __shared__ float4 lds[];
  const QuadItem item = b.work[block_index(a.xcd)];
  if ((epi.skip && *epi.skip) || item.nt <= 0) return;  // uniform over the grid (every item has targets)
  const int nt = item.nt, nrec = int(item.rec >> kItemRecShift);
  const int64_t r0 = item.rec & kItemRecMask;
  double dots[3] = {0.0, 0.0, 0.0};
  const int c = int(threadIdx.x) & 3;
  constexpr int PER = NR <= 4 ? 1 : NR / 4;  // operands per lane
  const int op = NR == 1 ? 0 : (NR == 2 ? (c & 1) : c);
  float4* s_tab = lds;                       // coefficient table
  float4* rpos = lds + kTabStride * a.ct.n;  // [nrec] offset xyz, packed box cell
  float4* rval = rpos + nrec;                // [nrec][NR] operands
  float hx = float(a.g.h[0]), hy = float(a.g.h[1]), hz = float(a.g.h[2]);
  if (a.sys) {
    const SysGrid* S = a.sys + a.sys_slot[item.t0];
    hx = float(S->g.h[0]);
    hy = float(S->g.h[1]);
    hz = float(S->g.h[2]);
  }
  if (nrec == 0) {  // not staged (one operand only)
    load_tab(s_tab, a);
    __syncthreads();
    if constexpr (NR == 1)
      for (int j = int(threadIdx.x); j < nt; j += kBoxThreads) {
        const int64_t sj = b.tgt[item.t0 + j];
        double acc[1][3];
        fp32c_pairs_global(a, sj, s_tab, xg, acc);
        apply_epilogue<1, EPI>(a, sj, acc, xsoa, v, epi, u_glob, out, dots);
      }
    if constexpr (EPI == EPI_REF) ref_finish(epi, dots);
    return;
  }
  // A target's words, its first record numbers and what its epilogue reads;
  // the first target's are on their way while the records are staged.
  int i = int(threadIdx.x) >> 2;
  int32_t s = 0;
  int64_t bpk = 0;
  const uint16_t* __restrict__ ci = b.idx;
  int cnt = 0, last = 0;
  uint32_t e0 = 0, e1 = 0;
  const EpiTarget T = epi_target<EPI>(a, item.t0, epi);  // (a brick's targets are of one system)
  constexpr int NC = NR == 1 ? 1 : 3;  // components per lane
  EpiIn in[PER][NC];
  auto words = [&]() {
    if (i >= nt) return;
    s = b.tgt[item.t0 + i];
    bpk = b.base[item.t0 + i];
  };
  auto ahead = [&]() {
    if (i >= nt) return;
    ci = b.idx + (bpk & kBaseMask);
    cnt = int((uint64_t(bpk) >> kKeptShift) & kField12);  // stored (kept) entries
    last = cnt - 1;
    if (cnt > 0) {
      e0 = ci[int64_t(min(c, last)) * kSlice];
      if (NR == 1) e1 = ci[int64_t(min(c + 4, last)) * kSlice];
    }
#pragma unroll
    for (int r = 0; r < PER; ++r)
#pragma unroll
      for (int q = 0; q < NC; ++q)
        in[r][q] = epi_in<EPI>(a, s, op + 4 * r, NR == 1 ? min(c, 2) : q, xsoa, epi, u_glob);
  };
  words();
  load_tab(s_tab, a);
  {
    // positions, then operands: U loads in flight per thread, neighbouring
    // threads on neighbouring words of a record
    constexpr int U = NR == 1 ? 2 : 8;  // (eight operand sets: 4 or 8 within 2 %)
    const uint32_t* __restrict__ slot = b.slot + r0;
    const float4* __restrict__ pos = b.pos + r0;
    const int nv = nrec * NR;
    uint32_t t[U];
    int j0 = int(threadIdx.x);
#pragma unroll
    for (int u = 0; u < U; ++u) t[u] = slot[min(j0 + u * kBoxThreads, nv - 1) / NR];
    ahead();
    while (j0 < nv) {
      float4 f[U];
#pragma unroll
      for (int u = 0; u < U; ++u) f[u] = xg[int64_t(t[u]) * NR + min(j0 + u * kBoxThreads, nv - 1) % NR];
      if constexpr (NR == 1) {
        static_assert(U == 2);
        const int j1 = j0 + kBoxThreads;
        const float4 p0 = pos[j0], p1 = pos[min(j1, nv - 1)];
        rpos[j0] = p0;
        if (j1 < nv) rpos[j1] = p1;
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (j0 + u * kBoxThreads < nv) rval[j0 + u * kBoxThreads] = f[u];
      j0 += U * kBoxThreads;
#pragma unroll
      for (int u = 0; u < U; ++u) t[u] = slot[min(j0 + u * kBoxThreads, nv - 1) / NR];
    }
    if constexpr (NR > 1)
      for (int j = int(threadIdx.x); j < nrec; j += kBoxThreads) rpos[j] = pos[j];
  }
  __syncthreads();
  while (i < nt) {
    const float4 po = rpos[int((uint64_t(bpk) >> kSelfShift) & kField12)];  // the target's own record
    const uint32_t kb = 0x808080u - __float_as_uint(po.w);
    float ps[PER][3];
    KahanF kh[PER][3];
#pragma unroll
    for (int r = 0; r < PER; ++r) ps[r][0] = ps[r][1] = ps[r][2] = 0.f;
    auto merge = [&]() {
#pragma unroll
      for (int r = 0; r < PER; ++r)
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          kh[r][q].add(ps[r][q]);
          ps[r][q] = 0.f;
        }
    };
    struct Geo {
      float dx, dy, dz, A, Bx;
    };
    auto geometry = [&](const float4& pt) {
      Geo g;
      float di, dj, dk, y;
      box_diff(__float_as_uint(pt.w), kb, di, dj, dk);
      g.dx = __builtin_fmaf(di, hx, pt.x - po.x);
      g.dy = __builtin_fmaf(dj, hy, pt.y - po.y);
      g.dz = __builtin_fmaf(dk, hz, pt.z - po.z);
      const float r2 = fp32c_r2(g.dx, g.dy, g.dz);
      const int it = ONE ? fp32c_interval1(a.ct, r2, y) : fp32c_interval(a.ct, r2, y);
      fp32c_eval(s_tab, it, y, g.A, g.Bx);
      return g;
    };
    static_assert(kMergeEvery == 8, "a merge every two steps of the quad");
    if constexpr (NR == 1) {
      auto term = [&](const Geo& g, const float4& f, bool in, float& x, float& y, float& z) {
        x = y = z = 0.f;
        fp32c_acc(g.A, g.Bx, g.dx, g.dy, g.dz, f.x, f.y, f.z, x, y, z);
        if (!in) x = y = z = 0.f;
      };
      // two steps (eight entries) at a time, their record numbers loaded one ahead
      int k = 0;
      auto steps = [&](bool in0, bool in1) {
        const float4 p0 = rpos[e0], p1 = rpos[e1], f0 = rval[e0], f1 = rval[e1];
        e0 = ci[int64_t(min(k + 8 + c, last)) * kSlice];
        e1 = ci[int64_t(min(k + 12 + c, last)) * kSlice];
        const Geo g0 = geometry(p0), g1 = geometry(p1);
        float x0, y0_, z0, x1, y1_, z1;
        term(g0, f0, in0, x0, y0_, z0);
        term(g1, f1, in1, x1, y1_, z1);
        ps[0][0] = quad_add(quad_add(ps[0][0], x0), x1);
        ps[0][1] = quad_add(quad_add(ps[0][1], y0_), y1_);
        ps[0][2] = quad_add(quad_add(ps[0][2], z0), z1);
        merge();
      };
      for (; k + 8 <= cnt; k += 8) steps(true, true);
      if (k < cnt) steps(k + c < cnt, k + 4 + c < cnt);
    } else {
      for (int k = 0; k < cnt; k += 4) {
        const int e = int(e0);
        e0 = ci[int64_t(min(k + 4 + c, last)) * kSlice];
        const Geo g = geometry(rpos[e]);
        auto entry = [&](auto M) {
          constexpr int m = decltype(M)::value;
          if (k + m < cnt) {  // uniform over the quad
            const int em = quad_get<m>(e);
            const Geo gm{quad_get<m>(g.dx), quad_get<m>(g.dy), quad_get<m>(g.dz), quad_get<m>(g.A),
                         quad_get<m>(g.Bx)};
#pragma unroll
            for (int r = 0; r < PER; ++r) {
              const float4 f = rval[em * NR + op + 4 * r];
              fp32c_acc(gm.A, gm.Bx, gm.dx, gm.dy, gm.dz, f.x, f.y, f.z, ps[r][0], ps[r][1], ps[r][2]);
            }
          }
        };
        entry(std::integral_constant<int, 0>{});
        entry(std::integral_constant<int, 1>{});
        entry(std::integral_constant<int, 2>{});
        entry(std::integral_constant<int, 3>{});
        if ((k & 4) && k + 4 <= cnt) merge();
      }
    }
    double acc[PER][3];
#pragma unroll
    for (int r = 0; r < PER; ++r)
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        kh[r][q].add(ps[r][q]);
        acc[r][q] = kh[r][q].value();
      }
    if constexpr (NR == 1) {
      quad_epilogue<EPI>(a, T, in[0][0], s, c, acc[0][0], acc[0][1], acc[0][2], v, epi, out, dots);
    } else if (c < NR) {
#pragma unroll
      for (int r = 0; r < PER; ++r) {
        double nv[3];
#pragma unroll
        for (int q = 0; q < 3; ++q)
          nv[q] = epi_component<EPI>(a, T, in[r][q], s, op + 4 * r, q, acc[r][q], v, epi, out, dots);
        epi_record<NR, EPI>(a.n, s, op + 4 * r, nv[0], nv[1], nv[2], v);
      }
    }
    i += kBoxThreads / 4;
    words();
    ahead();
  }
  if constexpr (EPI == EPI_REF) ref_finish(epi, dots);
}

// k_apply_box for NR = 2 and 4 operands, for dense bricks (quad_lanes): a lane
// per target, the box's positions and the operands' records in LDS, a plane
// per operand ([NR][nrec]: the lanes of a wave read one operand of records at
// random, which a plane spreads over all banks), each kept pair's tensor
// formed once for all NR.  Sums, merge points and epilogue are k_apply's for
// NR operands, bit for bit.  Every brick with targets is staged.
template <int EPI, bool ONE, int NR>
__global__ void __launch_bounds__(kBoxThreads) k_apply_box_nr(PairArgs a, BoxView b, const float4* __restrict__ xg,
                                                             const double* __restrict__ xsoa, SlotVec v, ChebEpi epi,
                                                             const double* __restrict__ u_glob,
                                                             double* __restrict__ out) {
  static_assert(NR > 1 && EPI != EPI_REF, "one operand: k_apply_box");
  extern __shared__ float4 lds[];
  if (epi.skip && *epi.skip) return;  // uniform over the grid
  const int64_t brick = block_index(a.xcd);
  const int64_t c0 = brick * kBrickCells;
  const int32_t sb = b.cs[c0], se = b.cs[c0 + kBrickCells];
  if (sb >= se) return;  // no targets (uniform over the block)
  const int64_t r0 = b.off[brick];
  const int nrec = int(b.off[brick + 1] - r0);
  const int nt = se - sb;
  if (nrec == 0) return;  // not staged: never launched so (uniform over the block)
  float4* s_tab = lds;                       // coefficient table
  float4* rpos = lds + kTabStride * a.ct.n;  // [nrec] offset xyz, packed box cell
  float4* rval = rpos + nrec;                // [NR][nrec] operands
  load_tab(s_tab, a);
  for (int i = int(threadIdx.x); i < nrec; i += kBoxThreads) {
    const uint32_t t = b.slot[r0 + i];
    rpos[i] = b.pos[r0 + i];
#pragma unroll
    for (int r = 0; r < NR; ++r) rval[r * nrec + i] = xg[gather_index(false, NR, a.n, t, r)];
  }
  __syncthreads();
  BoxGeom B;
  box_init(B, a, b.reach, brick, sb);
  const float hx = B.h[0], hy = B.h[1], hz = B.h[2];
  constexpr int U = 2;  // entries per group, the next group's record numbers loaded one ahead
  for (int i = int(threadIdx.x); i < nt; i += kBoxThreads) {
    const int64_t s = b.tgt[sb + i];
    const int64_t bpk = b.base[sb + i];
    const float4 po = rpos[int((uint64_t(bpk) >> kSelfShift) & kField12)];  // the target's own record
    const uint32_t kb = 0x808080u - __float_as_uint(po.w);
    const int cnt = int((uint64_t(bpk) >> kKeptShift) & kField12);  // stored (kept) entries
    float ps[NR][3];
    KahanF kh[NR][3];
#pragma unroll
    for (int r = 0; r < NR; ++r) ps[r][0] = ps[r][1] = ps[r][2] = 0.f;
    auto disp = [&](const float4& pt, float& dx, float& dy, float& dz, float& y) {
      float di, dj, dk;
      box_diff(__float_as_uint(pt.w), kb, di, dj, dk);
      dx = __builtin_fmaf(di, hx, pt.x - po.x);
      dy = __builtin_fmaf(dj, hy, pt.y - po.y);
      dz = __builtin_fmaf(dk, hz, pt.z - po.z);
      return ONE ? fp32c_interval1(a.ct, fp32c_r2(dx, dy, dz), y) : fp32c_interval(a.ct, fp32c_r2(dx, dy, dz), y);
    };
    auto add = [&](int it, float y, float dx, float dy, float dz, const float4* f, int k) {
      float A, Bx;
      fp32c_eval(s_tab, it, y, A, Bx);
#pragma unroll
      for (int r = 0; r < NR; ++r) fp32c_acc(A, Bx, dx, dy, dz, f[r].x, f[r].y, f[r].z, ps[r][0], ps[r][1], ps[r][2]);
      if ((k & (kMergeEvery - 1)) == kMergeEvery - 1) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            kh[r][q].add(ps[r][q]);
            ps[r][q] = 0.f;
          }
      }
    };
    if (cnt > 0) {  // an empty list has no storage
      const uint16_t* __restrict__ ci = b.idx + (bpk & kBaseMask);
      const int last = cnt - 1;
      uint32_t en[U];
#pragma unroll
      for (int u = 0; u < U; ++u) en[u] = ci[int64_t(min(u, last)) * kSlice];
      for (int k = 0; k < cnt; k += U) {
        float4 pt[U], f[U][NR];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t c = en[u];
          en[u] = ci[int64_t(min(k + U + u, last)) * kSlice];
          pt[u] = rpos[c];
#pragma unroll
          for (int r = 0; r < NR; ++r) f[u][r] = rval[r * nrec + c];
        }
        float dx[U], dy[U], dz[U], y[U];
        int it[U];
#pragma unroll
        for (int u = 0; u < U; ++u) it[u] = disp(pt[u], dx[u], dy[u], dz[u], y[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (u == 0 || k + u < cnt) add(it[u], y[u], dx[u], dy[u], dz[u], f[u], k + u);
      }
    }
    double acc[NR][3];
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        kh[r][q].add(ps[r][q]);
        acc[r][q] = kh[r][q].value();
      }
    double dots[3];  // (EPI_REF only)
    apply_epilogue<NR, EPI>(a, s, acc, xsoa, v, epi, u_glob, out, dots);
  }
}

// k_apply_box64 (below) with four lanes per target: lane c takes entries c,
// c + 4, ...; the four terms of a step are added in list order by every lane.
template <int EPI>
__global__ void __launch_bounds__(kBoxThreads) k_apply_quad64(PairArgs a, BoxView b, const double4* __restrict__ c64,
                                                             const double4* __restrict__ xg,
                                                             const double* __restrict__ xsoa, SlotVec v, ChebEpi epi,
                                                             const double* __restrict__ u_glob,
                                                             double* __restrict__ out) {
  extern __shared__ double4 lds64[];
  const QuadItem item = b.work[block_index(a.xcd)];
  if ((epi.skip && *epi.skip) || item.nt <= 0) return;  // uniform over the grid (every item has targets)
  const int nt = item.nt, nrec = int(item.rec >> kItemRecShift);
  const int64_t r0 = item.rec & kItemRecMask;
  double dots[3] = {0.0, 0.0, 0.0};
  double4* rval = lds64;  // [nrec] operand
  const double sg = a.bsign;
  const int c = int(threadIdx.x) & 3;
  constexpr int U = 2;  // steps per group, the next group's tensors and record numbers loaded one ahead
  // A target's words, its first tensors and what its epilogue reads; the
  // first target's are on their way while the operands are staged.
  int i = int(threadIdx.x) >> 2;
  int cnt = 0;
  int64_t base = 0;
  double4 tn[U];
  uint32_t en[U];
  const EpiTarget T = epi_target<EPI>(a, item.t0, epi);  // (a brick's targets are of one system)
  EpiIn in{};
  auto words = [&]() {
    if (i >= nt) return;
    const int64_t s = item.t0 + i;
    cnt = a.cnt[s];
    base = a.slice_off[s >> 6] + (s & 63);
  };
  auto ahead = [&]() {
    if (i >= nt) return;
    if (nrec > 0 && cnt > 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t e = base + int64_t(min(4 * u + c, cnt - 1)) * kSlice;
        en[u] = b.idx[e];
        tn[u] = c64[e];
      }
    }
    const int64_t s = item.t0 + i;
    in = epi_in<EPI>(a, s, 0, min(c, 2), xsoa, epi, u_glob);
  };
  words();
  {
    constexpr int G = 2;  // records in flight per thread
    const uint32_t* __restrict__ slot = b.slot + r0;
    uint32_t t[G];
    int j0 = int(threadIdx.x);
    if (nrec > 0)
#pragma unroll
      for (int u = 0; u < G; ++u) t[u] = slot[min(j0 + u * kBoxThreads, nrec - 1)];
    ahead();
    while (j0 < nrec) {
      double4 f[G];
#pragma unroll
      for (int u = 0; u < G; ++u) f[u] = xg[t[u]];
#pragma unroll
      for (int u = 0; u < G; ++u)
        if (j0 + u * kBoxThreads < nrec) rval[j0 + u * kBoxThreads] = f[u];
      j0 += G * kBoxThreads;
#pragma unroll
      for (int u = 0; u < G; ++u) t[u] = slot[min(j0 + u * kBoxThreads, nrec - 1)];
    }
  }
  __syncthreads();
  while (i < nt) {
    const int64_t s = item.t0 + i;
    const int last = cnt - 1;
    double ps[3] = {0.0, 0.0, 0.0};
    const double4* __restrict__ cf = c64 + base;
    auto sum = [&](const double4& t, const double4& f, bool in) {
      double x = 0.0, y = 0.0, z = 0.0;
      fp64_acc(t, sg, f, x, y, z);
      if (!in) x = y = z = 0.0;
      ps[0] = quad_add(ps[0], x);
      ps[1] = quad_add(ps[1], y);
      ps[2] = quad_add(ps[2], z);
    };
    if (nrec > 0 && cnt > 0) {
      const uint16_t* __restrict__ ci = b.idx + base;
      for (int k = 0; k < cnt; k += 4 * U) {
        double4 t[U], f[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          t[u] = tn[u];
          f[u] = rval[en[u]];
          const int64_t e = int64_t(min(k + 4 * (U + u) + c, last)) * kSlice;
          en[u] = ci[e];
          tn[u] = cf[e];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) sum(t[u], f[u], k + 4 * u + c < cnt);
      }
    } else {
      for (int k = 0; k < cnt; k += 4) {
        const int64_t e = int64_t(min(k + c, last)) * kSlice;
        sum(cf[e], xg[a.ell[base + e] & kSlotMask], k + c < cnt);
      }
    }
    quad_epilogue<EPI>(a, T, in, s, c, ps[0], ps[1], ps[2], v, epi, out, dots);
    i += kBoxThreads / 4;
    words();
    ahead();
  }
  if constexpr (EPI == EPI_REF) ref_finish(epi, dots);
}

// FP64 pair sum with the operand records staged in LDS: one workgroup per
// brick, its targets in slot order; per entry the stored tensor (list
// layout) and the neighbour's record number in the brick's box (the same
// layout), the operand read from LDS.  List order and fp64_acc as in
// k_apply, so the sums are bit-identical.  A brick that is not staged
// gathers the operands from global memory.
template <int EPI, int NT>
__global__ void __launch_bounds__(NT) k_apply_box64(PairArgs a, BoxView b, const double4* __restrict__ c64,
                                                            const double4* __restrict__ xg,
                                                            const double* __restrict__ xsoa, SlotVec v, ChebEpi epi,
                                                            const double* __restrict__ u_glob,
                                                            double* __restrict__ out) {
  extern __shared__ double4 lds64[];
  if (epi.skip && *epi.skip) return;  // uniform over the grid
  const int64_t brick = block_index(a.xcd);
  const int64_t c0 = brick * kBrickCells;
  const int32_t sb = b.cs[c0], se = b.cs[c0 + kBrickCells];
  double dots[3] = {0.0, 0.0, 0.0};
  if (sb >= se) {  // no targets (uniform over the block)
    if constexpr (EPI == EPI_REF) ref_finish(epi, dots);
    return;
  }
  const int64_t r0 = b.off[brick];
  const int nrec = int(b.off[brick + 1] - r0);
  const int nt = se - sb;
  double4* rval = lds64;  // [nrec] operand
  if (nrec > 0) {
    // four records in flight per thread, then the remainder one at a time
    int i = int(threadIdx.x);
    for (; i + 3 * NT < nrec; i += 4 * NT) {
      const uint32_t t0 = b.slot[r0 + i], t1 = b.slot[r0 + i + NT];
      const uint32_t t2 = b.slot[r0 + i + 2 * NT], t3 = b.slot[r0 + i + 3 * NT];
      const double4 f0 = xg[t0], f1 = xg[t1], f2 = xg[t2], f3 = xg[t3];
      rval[i] = f0;
      rval[i + NT] = f1;
      rval[i + 2 * NT] = f2;
      rval[i + 3 * NT] = f3;
    }
    for (; i < nrec; i += NT) rval[i] = xg[b.slot[r0 + i]];
    __syncthreads();
  }
  const double sg = a.bsign;
  constexpr int U = 2;  // entries per group, the next group's tensors and record numbers loaded one ahead (4: 34.0)
  for (int i = int(threadIdx.x); i < nt; i += NT) {
    const int64_t s = sb + i;
    const int cnt = a.cnt[s];
    const int64_t base = a.slice_off[s >> 6] + (s & 63);
    const double4* __restrict__ cf = c64 + base;
    double ps[3] = {0.0, 0.0, 0.0};
    if (cnt > 0 && nrec > 0) {
      const uint16_t* __restrict__ ci = b.idx + base;
      const int last = cnt - 1;
      uint32_t en[U];
      double4 cn[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        en[u] = ci[int64_t(min(u, last)) * kSlice];
        cn[u] = cf[int64_t(min(u, last)) * kSlice];
      }
      int k = 0;
      for (; k + U <= cnt; k += U) {
        double4 c[U], f[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          c[u] = cn[u];
          f[u] = rval[en[u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          en[u] = ci[int64_t(min(k + U + u, last)) * kSlice];
          cn[u] = cf[int64_t(min(k + U + u, last)) * kSlice];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) fp64_acc(c[u], sg, f[u], ps[0], ps[1], ps[2]);
      }
#pragma unroll
      for (int u = 0; u < U - 1; ++u)
        if (k + u < cnt) fp64_acc(cn[u], sg, rval[en[u]], ps[0], ps[1], ps[2]);
    } else if (cnt > 0) {
      const uint32_t* __restrict__ lst = a.ell + base;
      for (int k = 0; k < cnt; ++k)
        fp64_acc(cf[int64_t(k) * kSlice], sg, xg[lst[int64_t(k) * kSlice] & kSlotMask], ps[0], ps[1], ps[2]);
    }
    const double acc[1][3] = {{ps[0], ps[1], ps[2]}};
    apply_epilogue<1, EPI>(a, s, acc, xsoa, v, epi, u_glob, out, dots);
  }
  if constexpr (EPI == EPI_REF) ref_finish(epi, dots);
}

// Field points: sum over the element's particle list, own element
// included, no exclusion (ggem_stokes.C:396-420), full minimum image.
// kPointLanes lanes share a point: lane l walks the stencil rows l, l +
// kPointLanes, ... (a chain of dependent loads) and leaves their particles in
// the point's list in LDS, then the lanes take the list's entries in turn, so
// that the tensors, two erf and two exp each, are evaluated on full lanes; the
// lanes' sums are added pairwise.  100,000 points of the 20,000-bead
// suspension (29 rows, 9.5 particles a point), FP64: a lane per point 210 us,
// sixteen that sum as they walk 125 us, with the lists 60 us.  A point with
// more than kPointList particles is summed on the walk.  Points without an
// element (elem < 0, the caller reports them) are skipped.
constexpr int kPointLanes = 16, kPointList = 128;
template <int P>
__global__ void __launch_bounds__(kBlock) k_pair_points(PairArgs a, const StencilRow* __restrict__ rows,
                                                       int nrows, const int32_t* __restrict__ cell_start,
                                                       const float4* __restrict__ fg32,
                                                       const double4* __restrict__ fg64, int64_t m,
                                                       const double* __restrict__ pts,
                                                       const int32_t* __restrict__ elem,
                                                       double* __restrict__ u) {
  __shared__ int32_t s_list[kBlock / kPointLanes][kPointList];
  const int64_t q = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) / kPointLanes;
  const int l = int(threadIdx.x) & (kPointLanes - 1);
  if (q >= m || elem[q] < 0) return;  // (a point's lanes together)
  int32_t* const list = s_list[threadIdx.x / kPointLanes];
  int ci, cj, ck;
  elem_ijk(a.g, elem[q], ci, cj, ck);
  const double4 xq = make_double4(pts[3 * q], pts[3 * q + 1], pts[3 * q + 2], 0.0);
  double us[3] = {0.0, 0.0, 0.0};
  KahanF kx, ky, kz;
  auto add = [&](int32_t t) {
    double dx, dy, dz;
    pair_disp<true>(a.g, xq, a.x4[t], 0u, dx, dy, dz);
    if (P == GGEM_FP64) {
      const double4 f = fg64[t];
      green_acc_f64(a.k, dx, dy, dz, f.x, f.y, f.z, us[0], us[1], us[2]);
    } else {
      const float4 f = fg32[t];
      const float fx = float(dx), fy = float(dy), fz = float(dz);
      float A, Bx;
      green_coef_f32(a.k32, fx * fx + fy * fy + fz * fz, A, Bx);
      const float B = Bx * (fx * f.x + fy * f.y + fz * f.z);
      kx.add(A * f.x + B * fx);
      ky.add(A * f.y + B * fy);
      kz.add(A * f.z + B * fz);
    }
  };
  auto walk = [&](auto&& seg) {
    for_each_segment(a.g, rows, nrows, cell_start, ci, cj, ck, seg, l, kPointLanes);
  };
  int mine = 0;
  walk([&](int32_t lo, int32_t hi, uint32_t) { mine += hi - lo; });
  int incl = mine;
#pragma unroll
  for (int o = 1; o < kPointLanes; o <<= 1) {
    const int y = __shfl_up(incl, o, kPointLanes);
    if (l >= o) incl += y;
  }
  const int total = __shfl(incl, kPointLanes - 1, kPointLanes);
  if (total <= kPointList) {
    int at = incl - mine;
    walk([&](int32_t lo, int32_t hi, uint32_t) {
      for (int32_t t = lo; t < hi; ++t) list[at++] = t;
    });
    wave_lds_sync();  // (a point's lanes are in one wave)
    for (int j = l; j < total; j += kPointLanes) add(list[j]);
  } else {
    walk([&](int32_t lo, int32_t hi, uint32_t) {
      for (int32_t t = lo; t < hi; ++t) add(t);
    });
  }
  if (P != GGEM_FP64) {
    us[0] = kx.value();
    us[1] = ky.value();
    us[2] = kz.value();
  }
#pragma unroll
  for (int o = 1; o < kPointLanes; o <<= 1)
#pragma unroll
    for (int d = 0; d < 3; ++d) us[d] += __shfl_xor(us[d], o, 64);
  if (l < 3) u[3 * q + l] = l == 0 ? us[0] : (l == 1 ? us[1] : us[2]);
}

// erfcx fit (see erfcx_f32): coefficients of Q in x = 2t/t_max - 1,
// t_max = 1/(1 + 0.45/2), least squares with relative weights on
// z in [0.45, 1e4].
constexpr float kErfcxTmax = 0.816326530612f;
constexpr float kErfcxC[kErfcxDeg + 1] = {
    4.52274475e-01f,  2.40276895e-01f, 8.51269019e-02f,  1.35228369e-02f,
    -3.15813629e-03f, -1.64298252e-03f, 2.09066292e-04f, 1.94463725e-04f,
    -2.89952557e-05f, -1.94542224e-05f, 3.23959705e-06f};

PairArgs make_args(const ggem_ctx* ctx) {
  PairArgs a;
  a.g = ctx->grid;
  a.k = ctx->gc;
  a.k32.eps = float(ctx->gc.eps);
  a.k32.alpha = float(ctx->gc.alpha);
  a.k32.ksi = float(ctx->gc.ksi);
  a.k32.two_alpha_sqrt_pi = float(ctx->gc.two_alpha_sqrt_pi);
  a.k32.two_ksi_sqrt_pi = float(ctx->gc.two_ksi_sqrt_pi);
  a.k32.coeff_2 = float(ctx->gc.coeff_2);
  a.k32.erf_switch = 0.5f;
  a.k32.erfcx_scale = 2.0f / kErfcxTmax;
  for (int i = 0; i <= kErfcxDeg; ++i) a.k32.erfcx_c[i] = kErfcxC[i];
  a.x4 = ctx->x4;
  a.cnt = ctx->nbr_cnt;
  a.slice_off = ctx->slice_off;
  a.ell = ctx->ell;
  a.perm = ctx->perm;
  a.fs = ctx->fs;
  a.n = ctx->n;
  a.bsign = double(ctx->bsign);
  a.sys = ctx->sys_d;
  a.sys_slot = ctx->sys_slot;
  a.pc32 = ctx->pc32;
  a.xcd = 1;
  a.exact = explicit_minimg(ctx);
  a.tab = ctx->tab32;
  a.ct = ctx->tab;
  return a;
}

template <int P, int NR, int EPI, int BLK>
void launch_kb(ggem_ctx* ctx, const PairArgs& a, const double4* g64, const float4* g32, const double* soa,
               const SlotVec& v, const ChebEpi& epi, const double* u_glob, double* out) {
  if constexpr (P == GGEM_FP64)
    hipLaunchKernelGGL((k_apply<P, NR, EPI, BLK>), dim3(blocks_for(a.n, BLK)), dim3(BLK), 0, ctx->stream, a,
                       ctx->coef64, g64, g32, soa, v, epi, u_glob, out);
  else
    hipLaunchKernelGGL((k_apply<P, NR, EPI, BLK>), dim3(blocks_for(a.n, BLK)), dim3(BLK), 0, ctx->stream, a,
                       nullptr, g64, g32, soa, v, epi, u_glob, out);
}

BoxArgs box_args(const ggem_ctx* ctx) {
  BoxArgs b;
  b.cs = ctx->cell_start;
  for (int d = 0; d < 3; ++d) b.reach[d] = ctx->reach[d];
  b.rows = ctx->rows_d;
  b.nrows = ctx->n_rows;
  b.cells_cap = b.waves_cap = b.recs_cap = 0;
  b.off = ctx->box_off;
  b.eoff = ctx->box_eoff;
  b.tgt = ctx->box_tgt;
  b.base = ctx->box_base;
  b.slot = ctx->box_slot;
  b.pos = ctx->box_pos;
  b.idx = ctx->box_idx;
  b.fp64 = ctx->box_fp64 ? 1 : 0;
  b.ell = nullptr;
  b.walk = list_walk(ctx);
  return b;
}

BoxView box_view(const ggem_ctx* ctx) {
  BoxView b;
  b.cs = ctx->cell_start;
  for (int d = 0; d < 3; ++d) b.reach[d] = ctx->reach[d];
  b.off = ctx->box_off;
  b.tgt = ctx->box_tgt;
  b.base = ctx->box_base;
  b.slot = ctx->box_slot;
  b.pos = ctx->box_pos;
  b.idx = ctx->box_idx;
  b.work = ctx->quad_work;
  return b;
}

unsigned n_bricks(const ggem_ctx* ctx) { return unsigned(ctx->grid.n_cells >> (3 * kBrickBits)); }

// Four lanes per target (k_apply_quad, k_apply_quad64) or one (k_apply_box,
// k_apply_box64), by the mean number of targets of the bricks that have
// any.  One operand, one lane -> four, us per application:
//   targets a brick     13 (h = 2)  20         33 (h = 2)  59          117         176         244
//   FP32C               13.2->10.0  9.3->7.7   15.1->9.5   10.7->9.0   13.6->11.8  16.1->16.5  26.2->25.4
//   FP64                10.9->10.3  8.3->7.3   10.6->9.8   9.6->9.8    16.6->17.0  24.3->26.3  43.9->45.7
// and 87 -> 122 us at 1M beads (244, FP32C): there the lanes are busy either
// way and the sums on every lane of a quad only cost.  FP64 streams its
// tensors and gains by the split only where few beads leave CUs idle.  Quads,
// a lane per target in blocks of 256 and of 512, us per application:
//   beads      targets:  quads 256  512    targets:  quads 256  512
//   12,000     23 (3.9)   7.7  8.1  8.3     96        8.8 10.4 10.2
//              188       14.1 18.6 13.9
//   22,000     17 (2.5)   9.4  9.1   -      43 (2.0) 12.8   -  14.1
//   30,000     17 (2.5)  11.2 10.4 11.5     59       11.9 11.2 10.5
//              240       18.7 23.7 16.6
//   120,000    29 (3.9)  19.3 16.2 21.7     55 (3.1) 24.8 21.8 22.5
//              120       26.0 23.1 23.9     234      41.1 41.6 37.0
//   400,000    18 (2.5)  70.0 55.8 90.2     50 (3.9) 46.1 35.6 42.6
//              182        132  119  120     231       158  150  137
//   1,000,000  20 (3.1)   183  152  254     46 (3.9)  142  114  147
// FP32C with several operands, quads -> one lane (k_apply_box_nr; 8 as 4 + 4;
// * as 2 + 2, the records of 4 exceed the LDS), us per application:
//   beads    targets   2 operands      4 operands      8 operands
//   25,000     49      11.8 -> 14.6    13.3 -> 19.4    18.5 -> 36.9
//             200      14.4 -> 17.4    17.3 -> 23.0    32.1 -> 43.7
//   50,000     98      14.8 -> 15.8    17.7 -> 21.6    33.1 -> 41.9
//             146      18.3 -> 19.5    29.6 -> 27.8    56.4 -> 53.5
//             231      42.3 -> 34.8    82.5 -> 67.1*   161 -> 132*
//   65,536     49      17.8 -> 16.6    21.9 -> 32.0    33.4 -> 61.3
//              90      18.2 -> 16.2    23.2 -> 22.4    43.4 -> 42.0
//             191      23.8 -> 20.1    39.1 -> 27.8    76.2 -> 53.1
//   100,000    58      22.9 -> 21.2    27.8 -> 39.6    64.3 -> 76.2
//             100      22.5 -> 18.2    28.4 -> 26.4    58.9 -> 49.9
//             195      28.7 -> 21.6    52.2 -> 30.4    102 -> 57.1
//             292      64.9 -> 42.2    127 -> 80.8*    252 -> 160*
// A quad block stages its brick's records for about 64 targets, a lane block
// for all of them: quads lose where bricks use the threads of a lane block (45
// targets at two operands, 95 at four) and the lanes fill the chip (beads, or
// beads times targets a brick where the staging decides).
// FP32C with one operand, quads -> one lane over many beads:
//   beads    element (records a target)  targets: us per application
//   100,000  3.1 (5.4)  58: 15.0 -> 15.9;  3.9 (3.4)  46: 13.3 -> 13.0  100: 15.0 -> 13.9
//   200,000  2.0 (11)   41: 32 -> 42;      3.9        49: 19.7 -> 18.5   91: 22.4 -> 20.1
//   400,000  3.1        38: 37 -> 35;      3.9        50: 31.4 -> 27.9   98: 37.3 -> 29.2
//   800,000  2.0        41: 119 -> 140;    3.1  36: 67 -> 62  3.9  46: 57 -> 50  137: 69 -> 50
// The chip is full either way there, and what counts is how many of a lane
// block's threads the staging of a target's records keeps busy: targets a
// brick over records a target.
bool quad_lanes(const ggem_ctx* ctx, int precision, int nr) {
  const int64_t n = ctx->n, b = ctx->full_bricks, recs = ctx->box_recs;
  if (nr == 2) return n < 45 * b || (n < 65536 && n * n < 10000000 * b);
  if (nr > 2) return n < 95 * b || n * n < 6200000 * b;
  if (precision == GGEM_FP32C)
    return n <= 150 * b && (n < 100000 || n * n <= (n < 262144 ? 13 : 6) * b * recs);
  return n < 22000;
}

// FP64 with a lane per target: blocks of 512 threads, where bricks often hold
// more than 256 targets or fewer blocks than two per CU leave wave slots free;
// elsewhere most of their threads would have no target (the table above)
bool dense64(const ggem_ctx* ctx) {
  return ctx->n > 200 * int64_t(ctx->full_bricks) || n_bricks(ctx) <= 512;
}

size_t box_lds(const ggem_ctx* ctx, int nr) {
  return sizeof(float4) * (kTabStride * size_t(ctx->tab.n) + size_t(ctx->box_max) * size_t(1 + nr));
}

template <int EPI, int NR>
hipError_t launch_quad(ggem_ctx* ctx, PairArgs a, const float4* xg, const double* soa, const SlotVec& v,
                       const ChebEpi& epi, const double* u_glob, double* out) {
  const dim3 grid(unsigned(ctx->quad_items));
  if (ctx->tab.n2 == 0)
    hipLaunchKernelGGL((k_apply_quad<EPI, true, NR>), grid, dim3(kBoxThreads), box_lds(ctx, NR), ctx->stream, a,
                       box_view(ctx), xg, soa, v, epi, u_glob, out);
  else
    hipLaunchKernelGGL((k_apply_quad<EPI, false, NR>), grid, dim3(kBoxThreads), box_lds(ctx, NR), ctx->stream, a,
                       box_view(ctx), xg, soa, v, epi, u_glob, out);
  return hipGetLastError();
}

template <int EPI>
hipError_t launch_box(ggem_ctx* ctx, PairArgs a, const float4* xg, const double* soa, const SlotVec& v,
                      const ChebEpi& epi, const double* u_glob, double* out) {
  if (!ctx->box_valid || ctx->box_fp64 || ctx->box_max <= 0 || ctx->box_max > kBoxMaxRecs)
    return hipErrorInvalidConfiguration;
  a.xcd = 1;
  if (quad_lanes(ctx, GGEM_FP32C, 1)) return launch_quad<EPI, 1>(ctx, a, xg, soa, v, epi, u_glob, out);
  const size_t lds = box_lds(ctx, 1);
  if (ctx->tab.n2 == 0)
    hipLaunchKernelGGL((k_apply_box<EPI, true>), dim3(n_bricks(ctx)), dim3(kBoxThreads), lds, ctx->stream, a,
                       box_view(ctx), xg, soa, v, epi, u_glob, out);
  else
    hipLaunchKernelGGL((k_apply_box<EPI, false>), dim3(n_bricks(ctx)), dim3(kBoxThreads), lds, ctx->stream, a,
                       box_view(ctx), xg, soa, v, epi, u_glob, out);
  return hipGetLastError();
}

// staged FP32C pair sum of NR > 1 operands: every brick with targets staged
// and the box's positions and NR operand tables within the block's LDS
constexpr size_t kBoxNrLds = 81920;  // two blocks per CU
bool box_nr_ready(const ggem_ctx* ctx, int nr) {
  return (nr == 2 || nr == 4 || nr == 8) && ctx->box_valid && !ctx->box_fp64 && !ctx->box_unstaged &&
         ctx->box_max > 0 && ctx->box_max <= kBoxMaxRecs && box_lds(ctx, nr) <= kBoxNrLds;
}

template <int EPI, int NR>
hipError_t launch_box_nr(ggem_ctx* ctx, PairArgs a, const float4* xg, const double* soa, const SlotVec& v,
                         const ChebEpi& epi, const double* u_glob, double* out) {
  if (!box_nr_ready(ctx, NR)) return hipErrorInvalidConfiguration;
  a.xcd = 1;
  if constexpr (NR <= 4)
    if (!quad_lanes(ctx, GGEM_FP32C, NR)) {
      const size_t lds = box_lds(ctx, NR);
      if (ctx->tab.n2 == 0)
        hipLaunchKernelGGL((k_apply_box_nr<EPI, true, NR>), dim3(n_bricks(ctx)), dim3(kBoxThreads), lds, ctx->stream,
                           a, box_view(ctx), xg, soa, v, epi, u_glob, out);
      else
        hipLaunchKernelGGL((k_apply_box_nr<EPI, false, NR>), dim3(n_bricks(ctx)), dim3(kBoxThreads), lds,
                           ctx->stream, a, box_view(ctx), xg, soa, v, epi, u_glob, out);
      return hipGetLastError();
    }
  return launch_quad<EPI, NR>(ctx, a, xg, soa, v, epi, u_glob, out);
}

template <int EPI>
hipError_t launch_box64(ggem_ctx* ctx, PairArgs a, const double4* xg, const double* soa, const SlotVec& v,
                        const ChebEpi& epi, const double* u_glob, double* out) {
  if (!ctx->box_valid || !ctx->box_fp64 || ctx->box_max <= 0 || ctx->box_max > kBoxMaxRecs || !ctx->coef64_valid)
    return hipErrorInvalidConfiguration;
  a.xcd = 1;
  const size_t lds = size_t(ctx->box_max) * sizeof(double4);
  if (quad_lanes(ctx, GGEM_FP64, 1))
    hipLaunchKernelGGL((k_apply_quad64<EPI>), dim3(unsigned(ctx->quad_items)), dim3(kBoxThreads), lds, ctx->stream, a,
                       box_view(ctx), ctx->coef64, xg, soa, v, epi, u_glob, out);
  else if (dense64(ctx))
    hipLaunchKernelGGL((k_apply_box64<EPI, kDenseThreads>), dim3(n_bricks(ctx)), dim3(kDenseThreads), lds, ctx->stream,
                       a, box_view(ctx), ctx->coef64, xg, soa, v, epi, u_glob, out);
  else
    hipLaunchKernelGGL((k_apply_box64<EPI, kBoxThreads>), dim3(n_bricks(ctx)), dim3(kBoxThreads), lds, ctx->stream, a,
                       box_view(ctx), ctx->coef64, xg, soa, v, epi, u_glob, out);
  return hipGetLastError();
}

// candidate index of the staged-record kernels (one operand, after the
// block shapes of k_apply); it is the default where some brick is staged
constexpr int kBoxShape = kNApply;
bool box_ready(const ggem_ctx* ctx, int precision, int nr) {
  if (nr > 1) return precision == GGEM_FP32C && box_nr_ready(ctx, nr);
  if (!ctx->box_valid || ctx->box_max <= 0) return false;
  return precision == GGEM_FP32C ? !ctx->box_fp64 : (ctx->box_fp64 && ctx->coef64_valid);
}
// The staged kernel by default wherever it applies, except in many sparse
// bricks for several operands and for FP64 (whose lists are there): a block's
// cost is then the block, not its few targets, while the list-order kernel
// fills its waves.  Several operands by bricks
// with targets over the records of each, and bricks enough for the blocks to
// outweigh a wave that walks its lists alone; quads -> list order, us:
//   beads (bricks)    element  2 operands      4               8
//   5,000 (3,500)     2.0      12.3 -> 10.2    12.6 -> 13.0    15.8 -> 18.9
//   10,000 (7,000)    2.0      17.9 -> 10.3    19.0 -> 12.9    25.1 -> 18.8
//   14,000 (1,750)    3.1      10.4 -> 12.0    -               -
//   30,000 (1,728)    2.0      15.6 -> 22.4    17.0 -> 33.0    26.9 -> 53.0
//   65,000 (9,261)    2.0      30.4 -> 17.5    33.6 -> 25.6    46.3 -> 38.7
//   100,000 (5,832)   2.0      32.4 -> 30.2    36.4 -> 48.2    63.4 -> 73.9
//   100,000 (5,832)   3.1      25.1 -> 18.6    29.0 -> 29.4    43.5 -> 44.1
//   140,000 (8,000)   3.9      30.2 -> 18.4    34.5 -> 26.6    52.4 -> 45.3
//   300,000 (10,648)  2.0      68.1 -> 69.6    90.4 -> 115     -
//   300,000 (39,304)  2.0      109 -> 37.4     123 -> 60.8     -
// FP64 by targets a brick; lanes -> list order, us per application (in a
// convergence-checked term, whose every block also leaves its dot products):
//   beads      element  targets
//   60,000     2.0        9: 20.5 -> 13.5            18: 17.2 -> 18.9
//              3.1       18: 12.9 -> 11.9 (27 -> 17) 27: 12.5 -> 13.6
//   400,000    2.0        9: 95.5 -> 43.7 (250 -> 54 at 8)  18: 89.6 -> 87.6
//              3.1       18: 49.8 -> 35.7 (122 -> 50)       29: 41.5 -> 42.8
//   1,000,000  3.1       20:  152 -> 97  (355 -> 129)       28:  134 -> 127
bool sparse_bricks(const ggem_ctx* ctx, int nr) {
  const int64_t b = ctx->full_bricks;
  if (nr == 1) return b >= 2500 && ctx->n < 20 * b;
  return b >= (nr == 2 ? 3000 : nr == 4 ? 4500 : 6000) && b * b > (nr == 2 ? 33 : nr == 4 ? 65 : 100) * ctx->box_recs;
}
int apply_default(const ggem_ctx* ctx, int precision, int nr) {
  if (!box_ready(ctx, precision, nr)) return 0;
  const bool sparse = nr > 1 ? quad_lanes(ctx, precision, nr) && sparse_bricks(ctx, nr)
                             : precision == GGEM_FP64 && sparse_bricks(ctx, nr);
  return sparse ? 0 : kBoxShape;
}
int apply_candidates(const ggem_ctx* ctx, int precision, int nr) {
  return box_ready(ctx, precision, nr) ? kNApply + 1 : kNApply;
}
// A pick is kept by operand count and size alone: the staged shape it names
// may not apply to the present lists (positions moved on kept lists, fuller
// boxes); the list-order kernel serves then.
int apply_pick(const ggem_ctx* ctx, int precision, int nr, int c) {
  return c == kBoxShape && !box_ready(ctx, precision, nr) ? 0 : c;
}

// one apply launch in candidate shape c
template <int P, int NR, int EPI>
hipError_t launch_k(ggem_ctx* ctx, PairArgs a, int c, const double4* g64, const float4* g32, const double* soa,
                    const SlotVec& v, const ChebEpi& epi, const double* u_glob, double* out) {
  if (c == kBoxShape) {
    if constexpr (P == GGEM_FP32C && NR == 1) return launch_box<EPI>(ctx, a, g32, soa, v, epi, u_glob, out);
    if constexpr (P == GGEM_FP32C && NR > 1)
      return launch_box_nr<EPI, NR>(ctx, a, g32, soa, v, epi, u_glob, out);
    if constexpr (P == GGEM_FP64 && NR == 1) return launch_box64<EPI>(ctx, a, g64, soa, v, epi, u_glob, out);
    return hipErrorInvalidConfiguration;
  }
  if (c < 0 || c >= kNApply) return hipErrorInvalidValue;
  const Shape sh = kApplyShapes[c];
  a.xcd = sh.xcd;
  switch (sh.block) {
    case 64: launch_kb<P, NR, EPI, 64>(ctx, a, g64, g32, soa, v, epi, u_glob, out); break;
    case 128: launch_kb<P, NR, EPI, 128>(ctx, a, g64, g32, soa, v, epi, u_glob, out); break;
    case 512: launch_kb<P, NR, EPI, 512>(ctx, a, g64, g32, soa, v, epi, u_glob, out); break;
    default: launch_kb<P, NR, EPI, 256>(ctx, a, g64, g32, soa, v, epi, u_glob, out); break;
  }
  return hipGetLastError();
}

template <int P>
hipError_t launch_cheb_nr(ggem_ctx* ctx, const PairArgs& a, int c, int nr, const double4* g64, const float4* g32,
                          const double* soa, const SlotVec& v, const ChebEpi& epi) {
  switch (nr) {
    case 1: return launch_k<P, 1, EPI_CHEB>(ctx, a, c, g64, g32, soa, v, epi, nullptr, nullptr);
    case 2: return launch_k<P, 2, EPI_CHEB>(ctx, a, c, g64, g32, soa, v, epi, nullptr, nullptr);
    case 4: return launch_k<P, 4, EPI_CHEB>(ctx, a, c, g64, g32, soa, v, epi, nullptr, nullptr);
    default: return launch_k<P, 8, EPI_CHEB>(ctx, a, c, g64, g32, soa, v, epi, nullptr, nullptr);
  }
}

template <bool E, bool B, int BLK>
void launch_tb(ggem_ctx* ctx, const PairArgs& a) {
  // threads per slot: 2^18 threads fill the chip
  const unsigned split = unsigned(std::min<int64_t>(8, std::max<int64_t>(1, (int64_t(1) << 18) / a.n)));
  hipLaunchKernelGGL((k_tensors<E, B, BLK>), dim3(blocks_for(a.n, BLK), split), dim3(BLK), 0, ctx->stream, a,
                     ctx->coef64);
}

template <bool E, bool B>
hipError_t launch_t(ggem_ctx* ctx, PairArgs a, int c) {
  if (c < 0 || c >= kNTensor) return hipErrorInvalidValue;
  const Shape sh = kTensorShapes[c];
  a.xcd = sh.xcd;
  switch (sh.block) {
    case 64: launch_tb<E, B, 64>(ctx, a); break;
    case 128: launch_tb<E, B, 128>(ctx, a); break;
    case 512: launch_tb<E, B, 512>(ctx, a); break;
    default: launch_tb<E, B, 256>(ctx, a); break;
  }
  return hipGetLastError();
}

hipError_t launch_t_any(ggem_ctx* ctx, const PairArgs& a, int c) {
  const bool ex = explicit_minimg(ctx), bt = ctx->nsys > 1;
  if (bt) return ex ? launch_t<true, true>(ctx, a, c) : launch_t<false, true>(ctx, a, c);
  return ex ? launch_t<true, false>(ctx, a, c) : launch_t<false, false>(ctx, a, c);
}

}  // namespace

hipError_t launch_pair_tensors(ggem_ctx* ctx, int precision) {
  if (precision != GGEM_FP64) return hipErrorInvalidValue;  // FP32C evaluates its table in the pair sums
  if (ctx->n == 0) return hipSuccess;
  const PairArgs a = make_args(ctx);
  auto run = [&](int c) { return launch_t_any(ctx, a, c); };
  const int c = tune_pick(ctx, tune_key("tensors", precision, ctx->nsys > 1, ctx->n), kNTensor, run);
  ProfScope ps(ctx, "tensors_fp64");
  return run(c);
}

bool box_supported(const ggem_ctx* ctx) { return ctx->n > 0 && !explicit_minimg(ctx); }

hipError_t launch_box_fill(ggem_ctx* ctx, bool with_lists) {
  ProfScope ps(ctx, "box_fill");
  BoxArgs b = box_args(ctx);
  // LDS tables sized for the largest box and the most crowded brick
  auto cells = [](const int32_t* r) {
    return ((1 << kBrickBits) + 2 * r[0]) * ((1 << kBrickBits) + 2 * r[1]) * ((1 << kBrickBits) + 2 * r[2]);
  };
  int cap = cells(ctx->reach);
  for (int k = 0; k < ctx->nsys && ctx->nsys > 1; ++k) cap = std::max(cap, cells(ctx->sys_h[k].reach));
  b.cells_cap = std::min(cap, kBoxMaxCells);
  b.waves_cap = (ctx->max_targets + 63) / 64;
  b.recs_cap = ctx->max_recs;
  if (b.waves_cap > kBoxMaxWaves || b.recs_cap > kBoxMaxRecs) return hipErrorInvalidValue;
  const unsigned split = brick_split(ctx);
  b.ell = with_lists ? ctx->ell : nullptr;
  const size_t lds = sizeof(float4) * size_t(b.recs_cap) + sizeof(int32_t) * (2 * size_t(b.cells_cap) + b.waves_cap + 2) +
                     (with_lists ? sizeof(uint32_t) * size_t(b.recs_cap) : 0);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(n_bricks(ctx), split), dim3(kBoxThreads), lds, ctx->stream, make_args(ctx), b);
  };
  if (ctx->nsys > 1)
    b.walk == kWalkLanes ? launch(k_box_fill<true, false>) : launch(k_box_fill<true, true>);
  else
    b.walk == kWalkLanes ? launch(k_box_fill<false, false>) : launch(k_box_fill<false, true>);
  return hipGetLastError();
}

hipError_t launch_pair_beads(ggem_ctx* ctx, int precision, int epi, const double* u_glob, double* out) {
  if (ctx->n == 0) return hipSuccess;
  const PairArgs a = make_args(ctx);
  const SlotVec none{nullptr, nullptr, nullptr};
  const ChebEpi no_epi{0, 0.0, 0.0, 0.0, none, nullptr};
  auto run = [&](int c) {
    if (precision == GGEM_FP64)
      return epi == EPI_LOCAL
                 ? launch_k<GGEM_FP64, 1, EPI_LOCAL>(ctx, a, c, ctx->fg64, ctx->fg32, nullptr, none, no_epi, u_glob, out)
                 : launch_k<GGEM_FP64, 1, EPI_MOBILITY>(ctx, a, c, ctx->fg64, ctx->fg32, nullptr, none, no_epi, u_glob,
                                                        out);
    return epi == EPI_LOCAL
               ? launch_k<GGEM_FP32C, 1, EPI_LOCAL>(ctx, a, c, ctx->fg64, ctx->fg32, nullptr, none, no_epi, u_glob, out)
               : launch_k<GGEM_FP32C, 1, EPI_MOBILITY>(ctx, a, c, ctx->fg64, ctx->fg32, nullptr, none, no_epi, u_glob,
                                                       out);
  };
  // both epilogues write out[] only: idempotent, so the shape can be tuned here
  const int c = apply_pick(ctx, precision, 1,
                           tune_pick(ctx, tune_key("pair_beads", precision, epi, ctx->n),
                                     apply_candidates(ctx, precision, 1), run, apply_default(ctx, precision, 1)));
  ProfScope ps(ctx, precision == GGEM_FP64 ? "pair_beads_fp64" : "pair_beads_fp32c");
  return run(c);
}

hipError_t launch_pair_points(ggem_ctx* ctx, int precision, int64_t m, const double* pts,
                              const int32_t* elem, double* u) {
  const PairArgs a = make_args(ctx);
  ProfScope ps(ctx, precision == GGEM_FP64 ? "pair_points_fp64" : "pair_points_fp32c");
  // a launch of 2^32 threads or more comes out short: up to 2^27 points each
  constexpr int64_t kMost = (int64_t(1) << 31) / kPointLanes;
  for (int64_t q = 0; q < m; q += kMost) {
    const int64_t k = std::min(kMost, m - q);
    const dim3 grid(blocks_for(k * kPointLanes));
    if (precision == GGEM_FP64)
      hipLaunchKernelGGL(k_pair_points<GGEM_FP64>, grid, dim3(kBlock), 0, ctx->stream, a, ctx->rows_d, ctx->n_rows,
                         ctx->cell_start, ctx->fg32, ctx->fg64, k, pts + 3 * q, elem + q, u + 3 * q);
    else
      hipLaunchKernelGGL(k_pair_points<GGEM_FP32C>, grid, dim3(kBlock), 0, ctx->stream, a, ctx->rows_d, ctx->n_rows,
                         ctx->cell_start, ctx->fg32, ctx->fg64, k, pts + 3 * q, elem + q, u + 3 * q);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

int64_t apply_ref_parts(const ggem_ctx* ctx) {
  const int64_t nb =
      std::max<int64_t>(blocks_for(ctx->n, 64), std::max<int64_t>(n_bricks(ctx), ctx->quad_items));
  return 3 * (nb + (nb + kRefDecideParts - 1) / kRefDecideParts);
}

// operands of the next launch of `left`: the largest power of two up to 8,
// halved while only a smaller one fits the staged kernel's LDS, and 4 at once
// where a lane per target sums them (quad_lanes)
int apply_chunk(const ggem_ctx* ctx, int precision, int left) {
  int nr = left >= 8 ? 8 : left >= 4 ? 4 : left >= 2 ? 2 : 1;
  if (precision == GGEM_FP32C)
    for (int m = nr == 8 && !quad_lanes(ctx, precision, nr) ? 4 : nr; m > 1; m /= 2)
      if (box_nr_ready(ctx, m)) return m;
  return nr;
}
uint64_t apply_plan(const ggem_ctx* ctx, int precision) {
  uint64_t plan = 0;
  for (int nr = 1; nr <= 8; nr *= 2)
    plan = (plan << 6) | (uint64_t(apply_chunk(ctx, precision, nr)) << 2) |
           (apply_default(ctx, precision, nr) == kBoxShape ? 2u : 0u) | (quad_lanes(ctx, precision, nr) ? 1u : 0u);
  return plan << 1 | (dense64(ctx) ? 1u : 0u);
}
bool apply_reads_lists(const ggem_ctx* ctx, int precision, int nrhs) {
  if (ctx->tune.on) return true;
  for (int left = nrhs; left > 0;) {
    const int nr = apply_chunk(ctx, precision, left);
    if (apply_default(ctx, precision, nr) != kBoxShape || ctx->box_unstaged) return true;
    left -= nr;
  }
  return false;
}

// Most blocks of a reference-mode launch that decide by tickets (k_ref_decide:
// both sides)
constexpr int64_t kRefTicketBlocks = 128;

hipError_t launch_apply_ref(ggem_ctx* ctx, int precision, const SlotVec& x, const SlotVec& v, const ChebEpi& epi) {
  if (ctx->n == 0) return hipSuccess;
  const PairArgs a = make_args(ctx);
  // (the term updates y in place: the pick of plain applications serves)
  const int c = apply_pick(ctx, precision, 1,
                           tune_lookup(ctx, tune_key("apply", precision, 1, ctx->n), apply_default(ctx, precision, 1)));
  ChebEpi e = epi;
  int64_t nb = 0;
  if (c == kBoxShape) nb = quad_lanes(ctx, precision, 1) ? ctx->quad_items : int64_t(n_bricks(ctx));
  else if (c >= 0 && c < kNApply) nb = blocks_for(ctx->n, kApplyShapes[c].block);
  if (nb > kRefTicketBlocks) e.ref.ticket = nullptr;
  ProfScope ps(ctx, precision == GGEM_FP64 ? "apply_fp64" : "apply_fp32c");
  const hipError_t err =
      precision == GGEM_FP64
          ? launch_k<GGEM_FP64, 1, EPI_REF>(ctx, a, c, x.g64, x.g32, x.soa, v, e, nullptr, nullptr)
          : launch_k<GGEM_FP32C, 1, EPI_REF>(ctx, a, c, x.g64, x.g32, x.soa, v, e, nullptr, nullptr);
  if (err != hipSuccess || e.ref.ticket) return err;
  RefEpi r = epi.ref;  // (the deciding blocks' own parts after the launch's)
  r.part += 3 * nb;
  hipLaunchKernelGGL(k_ref_decide, dim3(unsigned((nb + kRefDecideParts - 1) / kRefDecideParts)),
                     dim3(kRefDecideThreads), 0, ctx->stream, r, epi.ref.part, int(nb));
  return hipGetLastError();
}

hipError_t launch_apply(ggem_ctx* ctx, int precision, int nrhs, const SlotVec& x, const SlotVec& v,
                        const ChebEpi& epi) {
  if (ctx->n == 0) return hipSuccess;
  const PairArgs a = make_args(ctx);
  const int64_t n = ctx->n, stride = 3 * n;
  struct Chunk {
    int nr;
    ChebEpi e;
    SlotVec vv;
    const double4* g64;
    const float4* g32;
    const double* soa;
  };
  std::vector<Chunk> chunks;
  for (int done = 0; done < nrhs;) {
    const int nr = apply_chunk(ctx, precision, nrhs - done);
    ChebEpi e = epi;
    if (e.xm1.soa) e.xm1.soa += done * stride;
    if (e.y) e.y += done * stride;
    SlotVec vv{v.soa + done * stride, v.g32 ? v.g32 + done * n : nullptr, v.g64 ? v.g64 + done * n : nullptr};
    chunks.push_back({nr, e, vv, x.g64 ? x.g64 + done * n : nullptr, x.g32 ? x.g32 + done * n : nullptr,
                      x.soa + done * stride});
    done += nr;
  }
  auto run = [&](const Chunk& k, int c) {
    return precision == GGEM_FP64 ? launch_cheb_nr<GGEM_FP64>(ctx, a, c, k.nr, k.g64, k.g32, k.soa, k.vv, k.e)
                                  : launch_cheb_nr<GGEM_FP32C>(ctx, a, c, k.nr, k.g64, k.g32, k.soa, k.vv, k.e);
  };
  // shapes: tuned on launches that only write v (kinds 0 and 1 with v not
  // aliasing x); the recurrence step (kind 2 updates y and overwrites
  // x_{k-1}) reuses the pick of its operand count
  std::vector<int> pick(chunks.size());
  for (size_t i = 0; i < chunks.size(); ++i) {
    const std::string key = tune_key("apply", precision, chunks[i].nr, n);
    const int dflt = apply_default(ctx, precision, chunks[i].nr);
    if (epi.kind != 2 && v.soa != x.soa)
      pick[i] = tune_pick(ctx, key, apply_candidates(ctx, precision, chunks[i].nr),
                          [&](int c) { return run(chunks[i], c); }, dflt);
    else
      pick[i] = tune_lookup(ctx, key, dflt);
    pick[i] = apply_pick(ctx, precision, chunks[i].nr, pick[i]);
  }
  ProfScope ps(ctx, precision == GGEM_FP64 ? "apply_fp64" : "apply_fp32c");
  for (size_t i = 0; i < chunks.size(); ++i) {
    const hipError_t e = run(chunks[i], pick[i]);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace ggem
