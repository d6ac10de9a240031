// ice3_kernels.hip -- HIP kernels for gfx950 and the C ABI of libice3_hip.so
// (declared in include/ice3.h).
//
// Layout: every field is float64 (nlev, ld), columns contiguous, so a 64-lane
// wavefront that owns 64 consecutive columns reads one level of a field as a
// single 512-byte coalesced transaction.
//
// Kernels:
//   k_ice_adjust   one thread per (level, column) point, pointwise ICE_ADJUST;
//   k_adjust_sedim one thread per column: ICE_ADJUST and the sedimentation in one
//                  top-down walk (the FP64 fused step over many columns);
//   k_sedim<R>     (ice3_sedim.hip) the statistical sedimentation and the surface
//                  precipitation, a wavefront per 64 columns, species and half, or
//   k_sedim_walk<R>  one thread per column (few levels, many columns);
//   k_micro<R>     persistent, one workgroup per compute unit, lookup tables in LDS:
//                  the ICE4 time-split microphysics, total tendencies and negativity
//                  correction per point, with the points of long time splittings
//                  compacted into full wavefronts (ballot, LDS parking);
//   k_sg_network   (ice3_surrogate.hip) the learned surrogate of k_micro: features and range
//                  check per point, the MLP on the bf16 matrix cores, decode, water and sign
//                  checks per point.  Points it rejects are queued for k_micro_segments, the
//                  plain FP64 microphysics over the queue.
// rain_ice is k_sedim then k_micro on one stream; the fused time step is
// k_ice_adjust, k_sedim, k_micro, or k_adjust_sedim, k_micro.  R is the arithmetic of the process rates
// and lookups (double, or float for the mixed path).
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>

#include "../../include/ice3.h"
#include "ice3_params.h"
#include "ice3_physics.hpp"
#include "ice3_stages.hpp"
#include "ice3_mlp.hpp"
#include "ice3_sedim.hpp"
#include "ice3_surrogate.hpp"

namespace ice3 {

// ------------------------------------------------------------------ kernels

__global__ void __launch_bounds__(256) k_ice_adjust(AdjustArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.ncol) return;
  adjust_at(a, i, (size_t)blockIdx.y * a.ld + i);
}

// ICE_ADJUST with the OCND2 branch: one thread per point, blockIdx.y the level (the layer
// thickness reads the heights of the level above).
__global__ void __launch_bounds__(256) k_ice_adjust_ocnd2(AdjustArgs a, Ocnd2Args x) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.ncol) return;
  adjust_at<true>(a, i, (size_t)blockIdx.y * a.ld + i, (int)blockIdx.y, &x);
}

// ICE_ADJUST of fields (ncol, nlev) with the vertical contiguous (the JAX components' arrays as
// they are): one thread per point in memory order, a.ld = 1.  The stage is pointwise, so it is
// bound by HBM as k_ice_adjust is, and the arrays need no transposing pass: 65,536 columns of
// 90 levels through the drop-in 0.30 ms (5.4 TB/s), against 1.12 ms with 19 transposing copies before
// k_ice_adjust.
template <bool OCND2, bool HAIL>
__global__ void __launch_bounds__(256) k_ice_adjust_rows(AdjustArgs a, Ocnd2Args x, unsigned npts) {
  const size_t j = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (j >= npts) return;
  const unsigned c = (unsigned)j / (unsigned)a.nlev;
  const size_t c0 = (size_t)c * a.nlev;
  adjust_at<OCND2, HAIL>(a, (int)c, j, (int)(j - c0), &x, nullptr, c0);
}

// The FP64 fused step's ICE_ADJUST and sedimentation in one column walk: the adjustment's
// memory traffic overlaps the sedimentation's FP64 arithmetic.
__global__ void __launch_bounds__(64) k_adjust_sedim(AdjustArgs aa, SedimArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.ncol) return;
  adjust_sedim_column<double>(aa, a, i);
}

// ---- hail (KRR=7), FP64: ICE_ADJUST with the hail heat capacity (one thread per point),
// and that and the sedimentation with hail in one column walk for the fused step; the
// microphysics is k_micro<double, false, true> (k_micro_points<double, false, true> when the
// context sets another sub-step cap).
__global__ void __launch_bounds__(256) k_ice_adjust_hail(AdjustArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.ncol) return;
  adjust_at<false, true>(a, i, (size_t)blockIdx.y * a.ld + i);
}

__global__ void __launch_bounds__(64) k_adjust_sedim_hail(AdjustArgs aa, SedimArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.ncol) return;
  adjust_sedim_column<double, true>(aa, a, i);
}

// Sum of v over the 64 lanes of the wavefront (every lane gets the total).
__device__ __forceinline__ unsigned long long wave_sum(unsigned long long v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

// ---- k_count_nonfinite: input validation (ice3_count_nonfinite).  blockIdx.y is the
// field; each thread takes one column (grid-stride) and walks the field's rows, so that a
// wavefront's loads are 64 consecutive doubles.  A value is non-finite when its exponent
// bits are all ones (NaN or an infinity).  Only a wavefront that found some adds to the
// field's counter.
struct CountArgs {
  const double *f[ICE3_MAX_CHECK_FIELDS];
  int rows[ICE3_MAX_CHECK_FIELDS];
  int ncol, ld;
  unsigned long long *counts;
};

__global__ void __launch_bounds__(256) k_count_nonfinite(CountArgs a) {
  const int q = blockIdx.y;
  const double *__restrict__ f = a.f[q];
  const int rows = a.rows[q];
  unsigned long long n = 0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < a.ncol; i += gridDim.x * blockDim.x)
#pragma unroll 8
    for (int r = 0; r < rows; ++r) {
      const unsigned long long b = __double_as_longlong(f[(size_t)r * a.ld + i]);
      n += (b & 0x7ff0000000000000ull) == 0x7ff0000000000000ull;
    }
  if (__ballot(n != 0) == 0ull) return;  // uniform: every lane of the wavefront sees it
  n = wave_sum(n);
  if ((threadIdx.x & 63) == 0) atomicAdd(&a.counts[q], n);
}

// The kernels' division, value by value (ice3_divide, a test hook).
__global__ void __launch_bounds__(256) k_divide(int n, const double *a, const double *b, double *q) {
  const unsigned e = blockIdx.x * 256 + threadIdx.x;
  if (e < (unsigned)n) q[e] = a[e] / by(b[e]);
}

// ---- k_transpose: fields (rows, cols) -> (cols, rows), all the fields of a call in one launch.
// A workgroup takes TR_ROWS rows (model columns) and up to TR_COLS of their values (levels): a
// run of memory that it reads in order, and writes through LDS in rows of TR_ROWS doubles (two
// whole cache lines).  Each thread issues TR_BATCH loads before its first wait.  The odd LDS row
// stride leaves both sides free of bank conflicts.  Bound by HBM: 22 fields of 65,536 x 90 in 382
// us, 5.4 TB/s (22 torch copies: 36 us each, 2.6 TB/s).
constexpr int TR_ROWS = 32, TR_COLS = 128, TR_BATCH = 8;
struct TransposeArgs {
  const double *src[ICE3_MAX_CHECK_FIELDS];
  double *dst[ICE3_MAX_CHECK_FIELDS];
  int rows, cols, col_tiles;
};

__global__ void __launch_bounds__(256) k_transpose(TransposeArgs a) {
  __shared__ double tile[TR_ROWS][TR_COLS + 1];
  const double *__restrict__ src = a.src[blockIdx.y];
  double *__restrict__ dst = a.dst[blockIdx.y];
  const int rt = blockIdx.x / a.col_tiles, ct = blockIdx.x - rt * a.col_tiles;
  const int r0 = rt * TR_ROWS, c0 = ct * TR_COLS;
  const int nr = a.rows - r0 < TR_ROWS ? a.rows - r0 : TR_ROWS;
  const int nc = a.cols - c0 < TR_COLS ? a.cols - c0 : TR_COLS;
  const int n = nr * nc, dr = 256 / nc, dc = 256 - dr * nc;  // a step of 256 values, in rows and the rest
  int r = threadIdx.x / nc, c = threadIdx.x - r * nc;
  for (int e0 = 0; e0 < n; e0 += 256 * TR_BATCH) {
    double v[TR_BATCH];
    int o[TR_BATCH];
#pragma unroll
    for (int q = 0; q < TR_BATCH; ++q) {
      o[q] = e0 + q * 256 + (int)threadIdx.x < n ? r * (TR_COLS + 1) + c : -1;
      v[q] = o[q] >= 0 ? src[(size_t)(r0 + r) * a.cols + c0 + c] : 0.;
      r += dr;
      c += dc;
      if (c >= nc) {
        c -= nc;
        ++r;
      }
    }
#pragma unroll
    for (int q = 0; q < TR_BATCH; ++q)
      if (o[q] >= 0) (&tile[0][0])[o[q]] = v[q];
  }
  __syncthreads();
  const int wr = threadIdx.x & (TR_ROWS - 1);
  if (wr < nr)
    for (int wc = threadIdx.x / TR_ROWS; wc < nc; wc += 256 / TR_ROWS)
      dst[(size_t)(c0 + wc) * a.rows + r0 + wr] = tile[wr][wc];
}

// ---- k_sedim_split: ICE4_SEDIMENTATION with CSEDIM='SPLI' (micro/mode_ice4_sedimentation.F90:
// 196-219, micro/mode_ice4_sedimentation_split.F90), FP64.
//
// Each species of a column is integrated in sub-steps of one common length, the largest that
// keeps every level's CFL number under XSPLIT_MAXCFL, until the time step is spent.  One
// wavefront holds one column in registers, level k in lane k % 64, slot k / 64 (L slots):
// a sub-step's fluxes are computed by all lanes at once, its length is a minimum over the
// wavefront, and the flux entering level k from above comes from the next lane.  A workgroup
// of SPLIT_COLS wavefronts takes as many adjacent columns: their inputs are read in rows of
// SPLIT_COLS doubles, every load issued before the first wait, and handed through LDS to the
// columns' wavefronts, up to SPLIT_BATCH fields at a time; the outputs go back the same way.  The
// two workgroups that take the halves of a 16-column row run on the same XCD, so that the row's
// cache lines are fetched once.  While a wavefront's
// state fits 128 registers (one slot, or two without hail) two workgroups share a compute
// unit, one's loads overlapping the other's sub-steps.
// 65,536 columns of 90 levels: 484 us, the VALU 69 % busy and 2.6 TB/s, 504 with each batch's loads
// waited for before the next batch's were issued (10,007 columns: 81, 88).
constexpr int SPLIT_COLS = 8, SPLIT_BATCH = 8;
template <int L, bool HAIL> constexpr int split_wpe() { return L == 1 || (L == 2 && !HAIL) ? 4 : 2; }
constexpr int SPLIT_MAX_SUBSTEPS = 1 << 16;  // per species and column; the reference has no
                                             // bound (its loop ends when the time is spent)

// Lane moves of an FP64 value inside the VALU, as two dword moves: a DPP move (lanes whose
// source lane is outside the wavefront keep old) and the gfx950 permlane swaps, which give
// a the lower and b the upper 16-lane rows of each 32-lane half (16) or the lower and upper
// halves (32) of the wavefront.  Every lane of the wavefront must be active.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v, double old) {
  const int lo = __builtin_amdgcn_update_dpp((int)__double2loint(old), (int)__double2loint(v), CTRL,
                                             0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp((int)__double2hiint(old), (int)__double2hiint(v), CTRL,
                                             0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
constexpr int DPP_QUAD_1032 = 0xB1, DPP_QUAD_2301 = 0x4E, DPP_ROW_MIRROR = 0x140,
              DPP_ROW_HALF_MIRROR = 0x141, DPP_WAVE_SHL1 = 0x130;
__device__ __forceinline__ void swap16_f64(double v, double &a, double &b) {
  const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
  a = __hiloint2double(h[0], l[0]);
  b = __hiloint2double(h[1], l[1]);
}
__device__ __forceinline__ void swap32_f64(double v, double &a, double &b) {
  const auto l = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
  a = __hiloint2double(h[0], l[0]);
  b = __hiloint2double(h[1], l[1]);
}

// Minimum over the wavefront, in every lane: within quads, half-rows and rows by DPP, then
// across rows and halves by the permlane swaps (min is exact, so the order is immaterial).
__device__ __forceinline__ double wave_min(double v) {
  v = dmin(v, dpp_f64<DPP_QUAD_1032>(v, v));
  v = dmin(v, dpp_f64<DPP_QUAD_2301>(v, v));
  v = dmin(v, dpp_f64<DPP_ROW_HALF_MIRROR>(v, v));
  v = dmin(v, dpp_f64<DPP_ROW_MIRROR>(v, v));
  double a, b;
  swap16_f64(v, a, b);
  v = dmin(a, b);
  swap32_f64(v, a, b);
  return dmin(a, b);
}

// Lane 0's value, in a scalar register.
__device__ __forceinline__ double lane0_f64(double v) {
  return __hiloint2double(__builtin_amdgcn_readlane((int)__double2hiint(v), 0),
                          __builtin_amdgcn_readlane((int)__double2loint(v), 0));
}

// Column group of block b: blocks b and b + 8 of a full group of 16 blocks, which the
// dispatcher sends to the same XCD, take the two halves of a 16-column row; the blocks of the
// last, partial group keep their order.
__device__ __forceinline__ int split_group(int b, int nblk) {
  if (b >= (nblk & ~15)) return b;
  return (b & ~15) + ((b & 7) << 1) + ((b >> 3) & 1);
}

// The elements this thread carries between memory and LDS: rows of the workgroup's SPLIT_COLS
// columns from c0 on (outside the domain element 0, to be dropped).
template <int L> struct SplitRows {
  size_t idx[L];
  bool in[L];
  __device__ __forceinline__ SplitRows(const SplitArgs &a, int c0) {
#pragma unroll
    for (int p = 0; p < L; ++p) {
      const int e = threadIdx.x + p * 64 * SPLIT_COLS, k = e / SPLIT_COLS, col = c0 + e - k * SPLIT_COLS;
      in[p] = k < a.nlev && col < a.ncol;
      idx[p] = in[p] ? (size_t)k * a.ld + col : 0;
    }
  }
};

// Issue the loads of NF fields, unconditionally, so that none waits for another.
template <int L, int NF>
__device__ __forceinline__ void split_issue(const SplitRows<L> &rows, const double *const (&f)[NF],
                                            double (&x)[NF][L]) {
#pragma unroll
  for (int g = 0; g < NF; ++g)
#pragma unroll
    for (int p = 0; p < L; ++p) x[g][p] = f[g][rows.idx[p]];
}

// Hand NF loaded fields (field f times scale[f]) over through LDS: v[f][q] of this lane receives
// level lane + 64 q of its wavefront's column (0 outside the domain).  Every thread of the
// workgroup calls it.  With KEEP, fields 1 to 3 are also stored as read into a.keep[0..2] (when
// set), in the same rows.
template <int L, int NF, bool KEEP = false>
__device__ __forceinline__ void split_exchange(double (*tile)[L * 64][SPLIT_COLS + 1],
                                               const SplitArgs &a, const SplitRows<L> &rows,
                                               const double (&x)[NF][L], const double (&scale)[NF],
                                               double (&v)[NF][L]) {
  __syncthreads();  // the previous batch has been read from the tile
#pragma unroll
  for (int g = 0; g < NF; ++g)
#pragma unroll
    for (int p = 0; p < L; ++p) {
      const int e = threadIdx.x + p * 64 * SPLIT_COLS, k = e / SPLIT_COLS;
      tile[g][k][e - k * SPLIT_COLS] = rows.in[p] ? x[g][p] * scale[g] : 0.;
    }
  if constexpr (KEEP) {
    if (a.keep[0]) {  // uniform
#pragma unroll
      for (int g = 0; g < 3; ++g)
#pragma unroll
        for (int p = 0; p < L; ++p)
          if (rows.in[p]) a.keep[g][rows.idx[p]] = x[g + 1][p];
    }
  }
  __syncthreads();
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int g = 0; g < NF; ++g)
#pragma unroll
    for (int q = 0; q < L; ++q) v[g][q] = tile[g][lane + 64 * q][w];
}

// Mass flux ZWSED of species JRR at mixing ratio r above its threshold; rf is the density
// factor rho^(1-XCEXVT) (pristine ice) or rho^(XEXSED-XCEXVT) (the power-law species), fixed
// over the sub-steps (micro/mode_ice4_sedimentation_split.F90:574-578,630-633,747-749).
template <int JRR>
__device__ __forceinline__ double split_flux(double r, double rho, double rf) {
  if constexpr (JRR == 4) {
    return P.XFSEDI * r * rf *
           rpow<double>(dmax(0.05E6, -0.15319E6 - 0.021454E6 * rlog<double>(rho * r)), P.XEXCSEDI);
  } else {
    constexpr double fsed = JRR == 3 ? P.XFSEDR : (JRR == 5 ? P.XFSEDS : (JRR == 6 ? P.XFSEDG : P.XFSEDH));
    constexpr double exsed = JRR == 3 ? P.XEXSEDR : (JRR == 5 ? P.XEXSEDS : (JRR == 6 ? P.XEXSEDG : P.XEXSEDH));
    return fsed * rpow<double>(r, exsed) * rf;
  }
}

// INTERNAL_SEDIM_SPLI (micro/mode_ice4_sedimentation_split.F90:359-849) of species JRR for the
// wavefront's column: r (the state at t on entry, the working state after), s (the source,
// updated); returns the surface rate PINPRX.  Sets *capped when the sub-step cap is reached.
template <int L, int JRR>
__device__ __forceinline__ double split_species(const SplitArgs &a, int lane, const double (&rho)[L],
                                                const double (&dz)[L], const double (&oorhodz)[L],
                                                double (&r)[L], double (&s)[L], bool *capped) {
  constexpr double thr = JRR == 4 ? (P.XRTMIN[4] > 1.0E-7 ? P.XRTMIN[4] : 1.0E-7) : P.XRTMIN[JRR];
  const double dt = a.dt, zinv = 1. / by(dt);
  bool any = false;
#pragma unroll
  for (int q = 0; q < L; ++q) any = any || (lane + 64 * q < a.nlev && r[q] > thr);
  // nothing above the fall threshold: one sub-step of dt changes no source (:786-826)
  if (!__any(any)) return 0.;
  double prs[L], rf[L];
#pragma unroll
  for (int q = 0; q < L; ++q) {
    prs[q] = s[q] - r[q] * zinv;  // external tendency (:241-253)
    rf[q] = lane + 64 * q < a.nlev
                ? rpow<double>(rho[q], JRR == 4 ? 1. - P.XCEXVT
                                                : (JRR == 3 ? P.XEXSEDR : JRR == 5 ? P.XEXSEDS
                                                   : JRR == 6 ? P.XEXSEDG : P.XEXSEDH) - P.XCEXVT)
                : 0.;
  }
  double remaint = dt, inpr = 0.;
  for (int n = 0; remaint > 0.; ++n) {  // wave-uniform: remaint is the column's
    if (n == SPLIT_MAX_SUBSTEPS) {
      *capped = true;
      break;
    }
    double w[L], m = INFINITY;
#pragma unroll
    for (int q = 0; q < L; ++q) {
      const bool in = lane + 64 * q < a.nlev;
      w[q] = in && r[q] > thr ? split_flux<JRR>(r[q], rho[q], rf[q]) : 0.;
      if (in && r[q] > P.XRTMIN[JRR] && w[q] > 1.E-20)
        m = dmin(m, a.maxcfl * rho[q] * r[q] * dz[q] / by(w[q]));  // :795-808
    }
    const double step = dmin(remaint, wave_min(m));
    remaint = remaint - step;  // :814-815
    inpr = inpr + lane0_f64(w[0]) / by(P.XRHOLW) * (step * zinv);
#pragma unroll
    for (int q = 0; q < L; ++q) {  // :820-824; level k + 1 is the next lane (or slot)
      const double next = q + 1 < L ? lane0_f64(w[q + 1 < L ? q + 1 : q]) : 0.;
      const double up = dpp_f64<DPP_WAVE_SHL1>(w[q], next);
      const double mrchange = step * oorhodz[q] * (up - w[q]);
      r[q] = r[q] + mrchange + prs[q] * step;
      s[q] = s[q] + mrchange * zinv;
    }
  }
  return inpr;
}

template <int L, bool HAIL, bool ZZZ>
__global__ void __launch_bounds__(64 * SPLIT_COLS)
    __attribute__((amdgpu_waves_per_eu(split_wpe<L, HAIL>()))) k_sedim_split(SplitArgs a) {
  __shared__ double tile[SPLIT_BATCH][L * 64][SPLIT_COLS + 1];
  constexpr int NV = HAIL ? 8 : 7;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c0 = split_group(blockIdx.x, gridDim.x) * SPLIT_COLS, i = c0 + w;
  const double ts = a.tscale;
  double lv[L], ls[L], r[NV - 3][L], rho[L], dz[L], src[NV][L];
  // batch 1: exn and the state at t of th .. rg; batch 2: hail's state at t, rho, dz and
  // sources; batch 3: the last sources.  RAIN_ICE's L/cph factors of the state at t
  // (rain_ice.F90:335-345) as soon as that state is in.
  constexpr int N2 = HAIL ? 8 : 7, N3 = HAIL ? 3 : 2;
  const SplitRows<L> rows(a, c0);
  double b1[8][L], x1[8][L], x2[N2][L], x3[N3][L];
  {
    const double *const f1[8] = {a.exn, a.t[0], a.t[1], a.t[2], a.t[3], a.t[4], a.t[5], a.t[6]};
    const double *const f2[8] = {a.rhodref, a.dzz, a.src[0], a.src[1], a.src[2], a.src[3],
                                 a.src[4], a.t[7]};
    const double *const f3[3] = {a.src[5], a.src[6], a.src[7]};
    split_issue<L, 8>(rows, f1, x1);
    split_issue<L, N2>(rows, reinterpret_cast<const double *const (&)[N2]>(f2), x2);
    split_issue<L, N3>(rows, reinterpret_cast<const double *const (&)[N3]>(f3), x3);
    const double s1[8] = {1., ts, ts, ts, ts, ts, ts, ts};
    split_exchange<L, 8, true>(tile, a, rows, x1, s1, b1);
  }
  auto factors = [&](const double (&rh_t)[L]) {
#pragma unroll
    for (int q = 0; q < L; ++q) {
      double tq[8];
#pragma unroll
      for (int v = 0; v < 7; ++v) tq[v] = b1[v + 1][q];
      tq[7] = rh_t[q];
      rain_ice_factors<HAIL>(tq, b1[0][q], ls[q], lv[q]);
#pragma unroll
      for (int v = 3; v < 7; ++v) r[v - 3][q] = b1[v + 1][q];
      if constexpr (HAIL) r[4][q] = rh_t[q];
    }
  };
  if constexpr (!HAIL) {
    const double zero[L] = {};
    factors(zero);
  }
  {
    double b2[N2][L];
    const double s2[8] = {1., 1., 1., 1., 1., 1., 1., ts};
    split_exchange<L, N2>(tile, a, rows, x2, reinterpret_cast<const double (&)[N2]>(s2), b2);
    if constexpr (ZZZ) {  // RAIN_ICE's model level height (rain_ice.F90:387-395), in its order
      if (lane == 0 && i < a.ncol) {
        double zzsum = 0.;
        for (int k = a.nlev - 1; k >= 0; --k) {
          zzsum = zzsum + tile[1][k][w];
          a.zzz[(size_t)k * a.ld + i] = zzsum - tile[1][k][w] * 0.5;
        }
      }
    }
    if constexpr (HAIL) factors(b2[7]);
#pragma unroll
    for (int q = 0; q < L; ++q) {
      rho[q] = b2[0][q];
      dz[q] = b2[1][q];
#pragma unroll
      for (int v = 0; v < 5; ++v) src[v][q] = b2[v + 2][q];
    }
  }
  {
    double b3[N3][L];
    const double s3[3] = {1., 1., 1.};
    split_exchange<L, N3>(tile, a, rows, x3, reinterpret_cast<const double (&)[N3]>(s3), b3);
#pragma unroll
    for (int v = 0; v < N3; ++v)
#pragma unroll
      for (int q = 0; q < L; ++q) src[v + 5][q] = b3[v][q];
  }
  double oorhodz[L];
#pragma unroll
  for (int q = 0; q < L; ++q)
    oorhodz[q] = lane + 64 * q < a.nlev ? 1. / by(rho[q] * dz[q]) : 0.;  // ZW (:263)
  if (i < a.ncol) {
    bool capped = false;
    const double pr = split_species<L, 3>(a, lane, rho, dz, oorhodz, r[0], src[IRR], &capped);
    const double pi = split_species<L, 4>(a, lane, rho, dz, oorhodz, r[1], src[IRI], &capped);
    const double ps = split_species<L, 5>(a, lane, rho, dz, oorhodz, r[2], src[IRS], &capped);
    const double pg = split_species<L, 6>(a, lane, rho, dz, oorhodz, r[3], src[IRG], &capped);
    double ph = 0.;
    if constexpr (HAIL) ph = split_species<L, 7>(a, lane, rho, dz, oorhodz, r[4], src[IRH], &capped);
    if (lane == 0) {
      a.inprc[i] = 0.;
      a.inprr[i] = pr;
      a.inpri[i] = pi;
      a.inprs[i] = ps + pi;  // mode_ice4_sedimentation.F90:212
      a.inprg[i] = pg;
      if constexpr (HAIL) a.inprh[i] = ph;
      if (capped && a.capped) atomicAdd(a.capped, 1ull);
    }
#pragma unroll
    for (int q = 0; q < L; ++q) {  // ICE4_CORRECT_NEGATIVITIES (:216-218), every point
      double rh = HAIL ? src[NV - 1][q] : 0.;
      correct_negativities<HAIL>(src[ITH][q], src[IRV][q], src[IRC][q], src[IRR][q], src[IRI][q],
                                 src[IRS][q], src[IRG][q], lv[q], ls[q], &rh);
      if constexpr (HAIL) src[NV - 1][q] = rh;
    }
  }
  // the sources back through LDS, in rows of SPLIT_COLS columns
  __syncthreads();  // every wavefront has read the last batch
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int q = 0; q < L; ++q) tile[v][lane + 64 * q][w] = src[v][q];
  __syncthreads();
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int p = 0; p < L; ++p) {
      const int e = threadIdx.x + p * 64 * SPLIT_COLS, k = e / SPLIT_COLS,
                c = e - k * SPLIT_COLS, col = c0 + c;
      if (k < a.nlev && col < a.ncol) a.dst[v][(size_t)k * a.ld + col] = tile[v][k][c];
    }
}

// ---- k_micro: the ICE4 microphysics, persistent, with the time splitting compacted
// across each wavefront.
//
// Every point makes one hard tendency call, and 42 % of them (on the 512x512x90 synthetic
// workload) then make soft calls, most of them one, a few up to five.  Run one point per
// lane to the end and a wavefront makes as many soft passes as its slowest lane needs,
// nearly all with few lanes active.  Here a wavefront takes 64-point chunks in turn: the hard
// call of all of them, one soft pass over those whose time step goes on, and the stores of
// every point that is then complete (94 %), while the chunk's state is in registers and its
// lines are in the caches.  The few left over are parked in LDS; a soft pass over parked
// points runs when 64 are at hand, or when the park (MicroPark::CAP) would otherwise overflow
// (ballot + prefix count give each its slot).  The per-point arithmetic is that of micro_at,
// only the order in which points are advanced differs, so the results are those of one thread
// per point.
//
// What bounds it: the latency that the wavefronts of a SIMD cannot cover for each other; the
// FP64 VALU issues about two thirds of the cycles.  Parking every unfinished point after its
// hard call, so that soft passes were full, read every input line and wrote every output line
// twice (10 GB at 512x512x90 against 5.3 algorithmic), as their lines had left the L2 by then:
// 2.79 ms in FP64, 2.40 mixed, 3.57 with OCND2, against 2.40, 1.54 and 2.92 now.
//
// Wavefronts per workgroup (one workgroup a compute unit).  FP64: two per SIMD, 233 of 256
// VGPRs.  Mixed: three per SIMD (165 of 168 VGPRs; two per SIMD: 15 % slower).  Hail: two per SIMD
// (256 VGPRs and a few spills: 3.06 ms; one per SIMD: 4.74 in an earlier form).
template <class R, bool HAIL = false> constexpr int micro_waves() { return sizeof(R) == 4 ? 12 : 8; }
// Lookup tables staged in LDS: the ICE3 block; the hail kernel reads the wet-growth kernels
// of hail, which follow it, from device memory.
template <class R, bool HAIL = false> constexpr size_t micro_tab_bytes() {
  return ((size_t)ICE3_T_ICE3 * sizeof(R) + 15) / 16 * 16;
}
// Variables of the time splitting (KRR + 1) and rates kept between tendency calls.
template <bool HAIL> constexpr int micro_nv() { return HAIL ? 8 : 7; }
template <class R, bool HAIL> constexpr int micro_ns() {
  return (int)(sizeof(typename StepStateFor<R, HAIL>::type) / sizeof(R));
}
// Fields of a chunk that its finish reads back from LDS instead of memory: the state at t, the
// sources of rr, ri, rs, rg, and exn, in the mixed path (three wavefronts a SIMD, whose lines do
// not all stay in L2 until then: 9.1 GB, now 7.5).  1.80 -> 1.68 ms at 512x512x90, with 20 park
// slots instead of 49.  In FP64, bound by latency and with 13 slots left, 2.57 -> 2.59 ms, with
// OCND2 3.22 -> 3.33.
template <class R> constexpr int micro_stash() { return sizeof(R) == 4 ? 12 : 0; }
template <class R> constexpr size_t micro_stash_bytes() { return (size_t)micro_stash<R>() * 64 * sizeof(double); }
// Park slots per wavefront: what the LDS holds beside the tables, at most 63 (31 in FP64,
// 20 in the mixed path, 24 with hail).
template <class R, bool HAIL = false> constexpr int micro_park_cap() {
  const size_t slot = (micro_nv<HAIL>() + 2) * sizeof(double) + micro_ns<R, HAIL>() * sizeof(R) +
                      2 * sizeof(int);
  const size_t n = ((160 * 1024 - micro_tab_bytes<R, HAIL>()) / micro_waves<R, HAIL>() -
                    micro_stash_bytes<R>()) / slot;
  return n < 63 ? (int)n : 63;
}

// Points parked by one wavefront: state between tendency calls, one row per field.
// Capacity: what fits the LDS beside the tables (fewer than 64).
template <class R, bool HAIL = false> struct MicroPark {
  static constexpr int NV = micro_nv<HAIL>(), NS = micro_ns<R, HAIL>();
  static constexpr int CAP = micro_park_cap<R, HAIL>();
  double d[NV + 2][CAP];   // vart[NV], cit, time
  R s[NS][CAP];            // StepState (StepStateHail)
  unsigned int q[CAP];     // point index k * ncol + i
  int calls[CAP];
};
static_assert(sizeof(StepState<double>) == 32 * sizeof(double), "StepState layout");
static_assert(sizeof(StepState<float>) == 32 * sizeof(float), "StepState layout");
static_assert(sizeof(StepStateHail<double>) == 43 * sizeof(double), "StepStateHail layout");

template <class R, bool HAIL = false> constexpr size_t micro_lds_bytes() {
  return micro_tab_bytes<R, HAIL>() +
         micro_waves<R, HAIL>() * (sizeof(MicroPark<R, HAIL>) + micro_stash_bytes<R>()) + 16;
}
static_assert(MicroPark<double>::CAP == 31 && MicroPark<float>::CAP == 20 &&
              MicroPark<double, true>::CAP == 24, "park capacity");
static_assert(ICE3_T_ICE3 % 2 == 0, "k_micro stages the tables by pairs");
static_assert(micro_lds_bytes<double>() <= 160 * 1024, "k_micro<double> LDS");
static_assert(2 * micro_nv<false>() - 2 <= micro_stash<float>(), "k_micro<float> stash");
static_assert(micro_lds_bytes<float>() <= 160 * 1024, "k_micro<float> LDS");
static_assert(micro_lds_bytes<double, true>() <= 160 * 1024, "k_micro<double, false, true> LDS");

template <class R, bool HAIL, class SS>
__device__ __forceinline__ void park_store(MicroPark<R, HAIL> &pk, int e, unsigned int q,
                                           const double *vart, double cit, double time,
                                           const SS &S, int calls) {
  constexpr int NV = MicroPark<R, HAIL>::NV, NS = MicroPark<R, HAIL>::NS;
#pragma unroll
  for (int f = 0; f < NV; ++f) pk.d[f][e] = vart[f];
  pk.d[NV][e] = cit;
  pk.d[NV + 1][e] = time;
  const R *sv = reinterpret_cast<const R *>(&S);
#pragma unroll
  for (int f = 0; f < NS; ++f) pk.s[f][e] = sv[f];
  pk.q[e] = q;
  pk.calls[e] = calls;
}

template <class R, bool HAIL, class SS>
__device__ __forceinline__ unsigned int park_load(const MicroPark<R, HAIL> &pk, int e, double *vart,
                                                  double &cit, double &time, SS &S, int &calls) {
  constexpr int NV = MicroPark<R, HAIL>::NV, NS = MicroPark<R, HAIL>::NS;
#pragma unroll
  for (int f = 0; f < NV; ++f) vart[f] = pk.d[f][e];
  cit = pk.d[NV][e];
  time = pk.d[NV + 1][e];
  R *sv = reinterpret_cast<R *>(&S);
#pragma unroll
  for (int f = 0; f < NS; ++f) sv[f] = pk.s[f][e];
  calls = pk.calls[e];
  return pk.q[e];
}

template <class R, bool OCND2 = false, bool HAIL = false>
__global__ void __launch_bounds__((64 * micro_waves<R, HAIL>())) k_micro(MicroArgs a) {
  extern __shared__ __align__(16) unsigned char micro_lds[];
  constexpr int NV = micro_nv<HAIL>();
  R *tab = reinterpret_cast<R *>(micro_lds);
  // the tables, every load issued before the first store (a load and a store at a time take 8 us
  // longer, a fifth of the call on 1,024 columns)
  {
    constexpr int NT = 64 * micro_waves<R, HAIL>(), N2 = ICE3_T_ICE3 / 2, NL = (N2 + NT - 1) / NT;
    typedef double f64x2 __attribute__((ext_vector_type(2)));
    const f64x2 *src = (const f64x2 *)a.tab;
    f64x2 v[NL];
#pragma unroll
    for (int b = 0; b < NL; ++b) {
      const int e = threadIdx.x + b * NT;
      v[b] = src[e < N2 ? e : 0];
    }
#pragma unroll
    for (int b = 0; b < NL; ++b) {
      const int e = threadIdx.x + b * NT;
      if (e < N2) {
        tab[2 * e] = (R)v[b][0];
        tab[2 * e + 1] = (R)v[b][1];
      }
    }
  }
  int *next_chunk = reinterpret_cast<int *>(micro_lds + micro_lds_bytes<R, HAIL>() - 16);
  if (threadIdx.x == 0) *next_chunk = micro_waves<R, HAIL>();
  __syncthreads();
  // hail: the wet-growth kernels of hail from device memory
  const double *htab = HAIL ? a.tab + ICE3_T_ICE3 : nullptr;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  MicroPark<R, HAIL> &pk =
      reinterpret_cast<MicroPark<R, HAIL> *>(micro_lds + micro_tab_bytes<R, HAIL>())[wid];
  constexpr int ST = micro_stash<R>();
  double (*stash)[64] = reinterpret_cast<double (*)[64]>(
      micro_lds + micro_tab_bytes<R, HAIL>() + micro_waves<R, HAIL>() * sizeof(MicroPark<R, HAIL>) +
      wid * micro_stash_bytes<R>());
  const unsigned long long below = (1ull << lane) - 1ull;  // lanes under this one
  const int cpl = (a.ncol + 63) >> 6;                       // chunks per level
  const int nchunk = cpl * a.nlev;
  const double dt = a.dt;
  const PointConst<R> pc_soft{};  // soft calls read no point constants
  int parked = 0;                 // wave-uniform
  bool active = false;            // this lane holds a point whose time step goes on
  unsigned int q = 0;             // that point: index k * ncol + i, offset j
  size_t j = 0;
  StepPointN<NV> p;
  double vart[NV], cit = 0., time = 0.;
  typename StepStateFor<R, HAIL>::type S;
  int calls = 0;
  unsigned int ncalls = 0, ncap = 0, nmicro = 0;  // of this lane: at most 2^18 points (256 CUs) of 2^12 calls
  bool done = false;              // this lane holds a point's end state, to be stored
  double evap3d = 0., rvheni = 0., exnref = 1.;
  // The workgroup's chunks, taken by its wavefronts in turn as they come free (a SIMD favours its
  // oldest wavefront, and with a fixed share each the others ran on alone at the end: 2.56 ms at
  // 512x512x90, 2.40 now; mixed 1.69 and 1.54, OCND2 3.22 and 2.92, hail 3.36 and 3.06).  Few chunks go
  // one to a compute unit before a second to any (1,024 columns: 26.7 us, 7 us more with eight in a
  // row to each); many go in rows of W to a workgroup, whose wavefronts' chunks are then
  // neighbours (mixed path at 512x512x90: 2.6 % faster; FP64 the same).
  constexpr int W = micro_waves<R, HAIL>();
  const int cstep = gridDim.x * W;
  const bool spread = nchunk < 4 * cstep;
  const int c0 = spread ? (int)blockIdx.x : (int)blockIdx.x * W, cw = spread ? (int)gridDim.x : 1;
  for (int n = wid;; n = __builtin_amdgcn_readfirstlane(lane == 0 ? atomicAdd(next_chunk, 1) : 0)) {
    const int c = (n / W) * cstep + (n % W) * cw + c0;
    const bool more = c < nchunk;  // wave-uniform
    if (more) {
      const int k = c / cpl, i = (c - k * cpl) * 64 + lane;
      if (i < a.ncol) {
        q = (unsigned int)k * (unsigned int)a.ncol + (unsigned int)i;
        j = (size_t)k * a.ld + i;
        double t[NV], s[NV];
        micro_load<NV>(a, j, t, s);
        cit = a.src_ci[j];
        // Every input is loaded here, not where the mask or the finish first needs it, a wait for
        // memory later (512x512x90: FP64 2.72 -> 2.56 ms, mixed 1.89 -> 1.81, OCND2 3.37 -> 3.21).
        // exn_ref stays in registers for the finish; the hail kernel has none left.
        const double exn = a.exn[j], rhodref = a.rhodref[j], pabs = a.pabs[j], cldfr = a.cldfr[j],
                     sigs = a.sigs[j];
        MicroOcnd2 xo;
        if constexpr (OCND2) xo = ocnd2_point(a, j);
        if constexpr (!HAIL) exnref = a.exn_ref[j];
        if constexpr (ST != 0) {
#pragma unroll
          for (int f = 0; f < NV; ++f) stash[f][lane] = t[f];
#pragma unroll
          for (int f = 3; f < NV; ++f) stash[NV - 3 + f][lane] = s[f];
          stash[2 * NV - 3][lane] = exn;
        }
        rvheni = 0.;
        evap3d = 0.;
        int st = 0;
        calls = 0;
        if (micro_mask<OCND2, HAIL>(t, a, j)) {
          ++nmicro;
          step_point(dt, exn, rhodref, pabs, cldfr, sigs, s, t, p);
#pragma unroll
          for (int f = 0; f < NV; ++f) vart[f] = t[f];
          time = 0.;
          const PointConst<R> pc = point_const<R>(p.rhodref);
          st = step_call<R, false, OCND2, HAIL>(dt, p, pc, vart, cit, time, S, calls,
                                                DEFAULT_MAX_CALLS, tab, &xo, htab);
          if (st == 0) evap3d = (double)S.rrevav;
        } else {
          micro_nucleation<R, OCND2, HAIL>(a, j, t, cit, rvheni);
#pragma unroll
          for (int f = 0; f < NV; ++f) vart[f] = t[f];
        }
        active = st > 0;
        done = !active;
        ncap += st < 0;
        if (st < 0) calls = -calls;
      }
    }
    // After the chunk's hard call (own): a soft pass over its own unfinished lanes, then the
    // stores of every finished one.  Then soft passes joined by parked points: over a full
    // wavefront while 64 points are at hand, over all of them while they would not fit the park,
    // and over all of them once the chunks are done.
#pragma clang loop unroll(disable)
    for (bool own = more;; own = false) {
      const unsigned long long am = __ballot(active);
      const int nact = __popcll(am), need = 64 - nact;
      const bool pass = own ? nact != 0
                            : (more ? parked >= need || nact + parked > MicroPark<R, HAIL>::CAP : nact + parked != 0);
      if (!own && !pass) break;
      if (!own) {
        if (!active) {
          const int r = __popcll(~am & below);  // rank among the idle lanes
          if (r < parked) {
            q = park_load(pk, parked - 1 - r, vart, cit, time, S, calls);
            const unsigned int k = q / (unsigned int)a.ncol;
            j = (size_t)k * a.ld + (q - k * (unsigned int)a.ncol);
            double t[NV], s[NV];
            micro_load<NV>(a, j, t, s);
            step_point(dt, a.exn[j], a.rhodref[j], a.pabs[j], a.cldfr[j], a.sigs[j], s, t, p);
            if constexpr (!HAIL) exnref = a.exn_ref[j];
            active = true;
            rvheni = 0.;
          }
        }
        parked -= need < parked ? need : parked;
      }
      if (pass && active) {
        const int st = step_call<R, true, OCND2, HAIL>(dt, p, pc_soft, vart, cit, time, S, calls,
                                                       DEFAULT_MAX_CALLS, tab, nullptr, htab);
        active = st > 0;
        done = !active;
        evap3d = st == 0 ? (double)S.rrevav : 0.;
        ncap += st < 0;
        if (st < 0) calls = -calls;
      }
      if (done) {
        ncalls += calls < 0 ? -calls : calls;
        if constexpr (HAIL) exnref = a.exn_ref[j];
        double t[NV], s[NV], exn;
        if (ST != 0 && own) {  // this chunk's points
#pragma unroll
          for (int f = 0; f < NV; ++f) t[f] = stash[f][lane];
#pragma unroll
          for (int f = 3; f < NV; ++f) s[f] = stash[NV - 3 + f][lane];
          exn = stash[2 * NV - 3][lane];
#pragma unroll
          for (int f = 0; f < 3; ++f) s[f] = a.src[f][j];
        } else {
          micro_load<NV>(a, j, t, s);
          exn = a.exn[j];
        }
        micro_finish<HAIL>(a, j, t, s, exn, vart, cit, evap3d, rvheni, calls, exnref);
        done = false;
      }
    }
    if (!more) break;
    // park the points whose time step goes on (parked + their number <= CAP here)
    const unsigned long long am = __ballot(active);
    if (active) {
      park_store(pk, parked + __popcll(am & below), q, vart, cit, time, S, calls);
      active = false;
    }
    parked += __popcll(am);
    // the stores above are read by other lanes of this wavefront in later passes
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  // every lane of the wavefront takes part in the sums (uniform branches)
  const unsigned long long cc = wave_sum(ncap);
  if (cc != 0 && lane == 0 && a.capped) atomicAdd(a.capped, cc);
  if (a.counters) {
    // summed over the workgroup first (in the emptied parks): an addition to an address that every
    // wavefront adds to takes 9 ns, and three of each of 2,048 kept a small call 40 to 55 us longer
    unsigned long long *sum = reinterpret_cast<unsigned long long *>(&pk);
    const unsigned long long n = wave_sum(ncalls), m = wave_sum(nmicro);
    if (lane == 0) {
      sum[0] = n;
      sum[1] = cc;
      sum[2] = m;
    }
    __syncthreads();  // uniform: a.counters is a kernel argument
    if (wid == 0) {   // lane 4 w + f takes sum f of wavefront w
      const int w = lane >> 2, f = lane & 3;
      unsigned long long t = 0;
      if (w < micro_waves<R, HAIL>() && f < 3)
        t = reinterpret_cast<unsigned long long *>(
            micro_lds + micro_tab_bytes<R, HAIL>() + w * sizeof(MicroPark<R, HAIL>))[f];
#pragma unroll
      for (int b = 4; b < 64; b <<= 1) t += __shfl_xor(t, b, 64);
      if (w == 0 && t) atomicAdd(&a.counters[f], t);
    }
  }
}

// The microphysics one thread per point, with the context's sub-step cap a.max_calls read at
// run time (k_micro has the default cap compiled in: the register allocator fails on
// k_micro<double> with a run-time bound).  Launched when a context sets another cap; the
// per-point arithmetic is k_micro's, so the results are the same for the same cap.  With HAIL
// (KRR=7) it is the microphysics of the hail path, with the wet-growth tables of hail.
template <class R, bool OCND2 = false, bool HAIL = false>
__global__ void __launch_bounds__(256) k_micro_points(MicroArgs a) {
  const unsigned int q = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned long long ncalls = 0, ncap = 0, nmicro = 0;
  if (q < (unsigned int)a.nlev * (unsigned int)a.ncol) {
    const unsigned int k = q / (unsigned int)a.ncol;
    const int c = micro_at<R, OCND2, HAIL>(a, (size_t)k * a.ld + (q - k * (unsigned int)a.ncol), a.tab);
    ncalls = c < 0 ? -c : c;
    ncap = c < 0;
    nmicro = c != 0;
  }
  const unsigned long long cc = wave_sum(ncap);
  if (cc != 0 && (threadIdx.x & 63) == 0 && a.capped) atomicAdd(a.capped, cc);
  if (a.counters) {
    const unsigned long long n = wave_sum(ncalls), m = wave_sum(nmicro);
    if ((threadIdx.x & 63) == 0) {
      atomicAdd(&a.counters[0], n);
      atomicAdd(&a.counters[1], cc);
      atomicAdd(&a.counters[2], m);
    }
  }
}

// ICE_ADJUST one thread per point with the record of the branches each point took (the test
// hook of ice3_ice_adjust_branches).
template <bool HAIL>
__global__ void __launch_bounds__(256) k_ice_adjust_branches(AdjustArgs a, unsigned *branches) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.ncol) return;
  const size_t j = (size_t)blockIdx.y * a.ld + i;
  unsigned br = 0;
  adjust_at<false, HAIL>(a, i, j, 0, nullptr, &br);
  branches[j] = br;
}

// The microphysics one thread per point with the branch record of each point (the test
// hook of ice3_rain_ice_branches; the counters of ice3_stats are not kept).
template <bool HAIL>
__global__ void __launch_bounds__(256) k_micro_branches(MicroArgs a) {
  const unsigned int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (unsigned int)a.nlev * (unsigned int)a.ncol) return;
  const unsigned int k = q / (unsigned int)a.ncol;
  const size_t j = (size_t)k * a.ld + (q - k * (unsigned int)a.ncol);
  unsigned br = 0;
  micro_at<double, false, HAIL>(a, j, a.tab, &br);
  a.branches[j] = br;
}

// Plain microphysics over the surrogate's rejected points: SG_PARTS blocks share the points that
// a workgroup of the network stage queued.
template <class R>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) k_micro_segments(MicroArgs a, const unsigned int *queue,
                                                       const unsigned int *qcount, unsigned int seg) {
  const unsigned int n = qcount[blockIdx.x / SG_PARTS];
  const unsigned int *list = queue + (size_t)(blockIdx.x / SG_PARTS) * seg;
  for (unsigned int e = blockIdx.x % SG_PARTS * 64 + threadIdx.x; e < n; e += SG_PARTS * 64)
    if (micro_at<R>(a, (size_t)list[e], a.tab) < 0 && a.capped) atomicAdd(a.capped, 1ull);
}

// Scratch layout of the surrogate step (bytes, 256-aligned blocks).  total is more than the queue
// takes: it is what the interface asks of a work area and measures the allocation-free entry's
// limit by (room for a network input, an output and a reason per point as well; 64 (SG_BLOCKS +
// 1) words and SG_BLOCKS counts are fewer than its 256 x 2049 words beside the points').
struct SgWork {
  size_t queue, qcount, total;
};
static SgWork sg_work_layout(size_t npts) {
  auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
  SgWork w;
  w.queue = 0;
  w.qcount = al((npts + 64 * ((size_t)SG_BLOCKS + 1)) * 4);
  w.total = al(npts * 64) + al(npts * 32) + al(npts) + al((npts + 1 + 256 * 2049) * 4) + 8192;
  return w;
}

// Surrogate features of the points of MicroArgs (training data and tests).
__global__ void __launch_bounds__(256) k_features(MicroArgs m, unsigned int npts,
                                                  const ice3_surrogate_norm *norm, float *raw,
                                                  __bf16 *x, unsigned char *micro) {
  const unsigned int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= npts) return;
  const size_t j = (size_t)(q / m.ncol) * m.ld + q % m.ncol;
  float f[MLP_NFEAT];
  const bool mi = surrogate_features(m, j, f);
  if (micro) micro[q] = mi ? 1 : 0;
  if (raw)
    for (int c = 0; c < MLP_NFEAT; ++c) raw[(size_t)q * MLP_NFEAT + c] = f[c];
  if (x)
    for (int c = 0; c < MLP_IN; ++c)
      x[(size_t)q * MLP_IN + c] =
          (__bf16)(c < MLP_NFEAT ? (f[c] - norm->feat_mean[c]) * norm->feat_scale[c] : 0.f);
}

}  // namespace ice3

// Scratch of the allocation-free surrogate step (ice3_adjust_rain_ice_surrogate_noalloc):
// the same layout as the caller's work area of ice3_adjust_rain_ice_surrogate.  One copy per
// GPU, held until the process ends.  Host code never uses the name: a kernel argument made
// from it would be a host address; ice3_ctx_create takes the device address with
// hipGetSymbolAddress.
static __device__ __align__(256) unsigned char scratch[ICE3_SURROGATE_SCRATCH_BYTES];

// ------------------------------------------------------------------ C ABI

struct ice3_ctx {
  int device;
  int ncu;            // compute units of the device: k_micro runs one workgroup on each
  ice3_params params;
  double *d_tab;
  double h_tab[ICE3_T_TOTAL];
  double *d_tiwmx;    // TIWMX tables of the OCND2 branch (ice3_tiwmx_tables order)
  unsigned long long *d_capped;  // points that hit the sub-step cap since the last status query
  void *d_scratch;    // device address of this device's copy of scratch
  int max_calls;      // sub-step cap per point
  int sedim;          // ICE3_SEDIM_STAT or ICE3_SEDIM_SPLI
  double maxcfl;      // XSPLIT_MAXCFL of the split sedimentation
  void *d_work;       // work area of the fused step with the split sedimentation
  size_t work_bytes;
  int timing;         // record ev[] around the stages of each call
  hipEvent_t ev[7];   // before adjust, after adjust, after sedimentation, then after the
                      // microphysics (plain step: events 3..6 together) or, for the surrogate
                      // step, after the features, the network, the decode and the fallback
};

using namespace ice3;

#define HIPCHK(x)                                 \
  do {                                            \
    if ((x) != hipSuccess) return ICE3_EDEVICE;   \
  } while (0)

extern "C" int ice3_ctx_create(ice3_ctx **out) {
  if (!out) return ICE3_EINVAL;
  ice3_ctx *c = (ice3_ctx *)calloc(1, sizeof(ice3_ctx));
  if (!c) return ICE3_EINVAL;
  ice3_build_params(&c->params, c->h_tab);
  // the kernels carry the constants as literals (P); they must be the host builder's
  if (memcmp(&c->params, &P, sizeof(ice3_params)) != 0) {
    free(c);
    return ICE3_ECONFIG;
  }
  constexpr size_t TIWMX_BYTES = sizeof(double) * ICE3_TW_NTAB * ICE3_TIWMX_N;
  double *tiwmx = (double *)malloc(TIWMX_BYTES);
  if (!tiwmx) {
    free(c);
    return ICE3_EDEVICE;
  }
  ice3_build_tiwmx(&c->params, tiwmx);
  if (hipGetDevice(&c->device) != hipSuccess ||
      hipDeviceGetAttribute(&c->ncu, hipDeviceAttributeMultiprocessorCount, c->device) !=
          hipSuccess || c->ncu <= 0 ||
      hipMalloc((void **)&c->d_tab, sizeof(double) * ICE3_T_TOTAL) != hipSuccess ||
      hipMemcpy(c->d_tab, c->h_tab, sizeof(double) * ICE3_T_TOTAL, hipMemcpyHostToDevice) !=
          hipSuccess ||
      hipMalloc((void **)&c->d_tiwmx, TIWMX_BYTES) != hipSuccess ||
      hipMemcpy(c->d_tiwmx, tiwmx, TIWMX_BYTES, hipMemcpyHostToDevice) !=
          hipSuccess ||
      hipMalloc((void **)&c->d_capped, sizeof(unsigned long long)) != hipSuccess ||
      hipMemset(c->d_capped, 0, sizeof(unsigned long long)) != hipSuccess ||
      hipGetSymbolAddress(&c->d_scratch, HIP_SYMBOL(scratch)) != hipSuccess ||
      c->d_scratch == nullptr) {
    if (c->d_tab) (void)hipFree(c->d_tab);
    if (c->d_tiwmx) (void)hipFree(c->d_tiwmx);
    if (c->d_capped) (void)hipFree(c->d_capped);
    free(tiwmx);
    free(c);
    return ICE3_EDEVICE;
  }
  free(tiwmx);
  c->max_calls = DEFAULT_MAX_CALLS;
  c->sedim = ICE3_SEDIM_STAT;
  c->maxcfl = 0.8;  // PARAM_ICE XSPLIT_MAXCFL default (micro/modd_param_icen.F90:347)
  *out = c;
  return ICE3_OK;
}

extern "C" void ice3_ctx_destroy(ice3_ctx *c) {
  if (!c) return;
  if (c->d_tab) (void)hipFree(c->d_tab);
  if (c->d_tiwmx) (void)hipFree(c->d_tiwmx);
  if (c->d_capped) (void)hipFree(c->d_capped);
  if (c->d_work) (void)hipFree(c->d_work);
  if (c->timing)
    for (int q = 0; q < 7; ++q) (void)hipEventDestroy(c->ev[q]);
  free(c);
}

extern "C" int ice3_stage_timing(ice3_ctx *c, int enable) {
  if (!c) return ICE3_EINVAL;
  if (enable && !c->timing) {
    for (int q = 0; q < 7; ++q) HIPCHK(hipEventCreate(&c->ev[q]));
    c->timing = 1;
  } else if (!enable && c->timing) {
    for (int q = 0; q < 7; ++q) (void)hipEventDestroy(c->ev[q]);
    c->timing = 0;
  }
  return ICE3_OK;
}

extern "C" int ice3_stage_times(ice3_ctx *c, float ms[6]) {
  if (!c || !ms || !c->timing) return ICE3_EINVAL;
  HIPCHK(hipEventSynchronize(c->ev[6]));
  for (int q = 0; q < 6; ++q) HIPCHK(hipEventElapsedTime(&ms[q], c->ev[q], c->ev[q + 1]));
  return ICE3_OK;
}

extern "C" int ice3_ctx_set_substep_cap(ice3_ctx *c, int max_calls) {
  if (!c || max_calls < 1) return ICE3_EINVAL;
  c->max_calls = max_calls;
  return ICE3_OK;
}

extern "C" int ice3_ctx_set_sedimentation(ice3_ctx *c, int scheme, double max_cfl) {
  if (!c || (scheme != ICE3_SEDIM_STAT && scheme != ICE3_SEDIM_SPLI) || !(max_cfl > 0.) ||
      !(max_cfl < INFINITY))
    return ICE3_EINVAL;
  c->sedim = scheme;
  c->maxcfl = max_cfl;
  return ICE3_OK;
}

extern "C" int ice3_ctx_status(ice3_ctx *c, void *stream, unsigned long long *capped) {
  if (!c) return ICE3_EINVAL;
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev != c->device) HIPCHK(hipSetDevice(c->device));
  const hipStream_t s = (hipStream_t)stream;
  unsigned long long h = 0;
  int rc = ICE3_OK;
  if (hipMemcpyAsync(&h, c->d_capped, sizeof h, hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess ||
      (h != 0 && hipMemsetAsync(c->d_capped, 0, sizeof h, s) != hipSuccess) ||
      hipStreamSynchronize(s) != hipSuccess)
    rc = ICE3_EDEVICE;
  if (dev != c->device) (void)hipSetDevice(dev);
  if (rc != ICE3_OK) return rc;
  if (capped) *capped = h;
  return h != 0 ? ICE3_ESUBSTEP : ICE3_OK;
}

// Record stage event q of a timed call (no-op when timing is off).
static int mark(ice3_ctx *c, int q, hipStream_t s) {
  if (c->timing) HIPCHK(hipEventRecord(c->ev[q], s));
  return ICE3_OK;
}
#define MARK(q) do { int rc_ = mark(ctx, (q), s); if (rc_) return rc_; } while (0)

extern "C" const char *ice3_strerror(int code) {
  switch (code) {
    case ICE3_OK: return "ok";
    case ICE3_EINVAL: return "invalid argument (size, stride, precision or NULL pointer)";
    case ICE3_EDEVICE: return "HIP runtime error";
    case ICE3_ESUBSTEP: return "a point reached the sub-step cap of the ICE4 time splitting";
    case ICE3_ECONFIG: return "constants compiled into the kernels differ from the host builder (rebuild)";
    case ICE3_ETOOLARGE:
      return "the problem needs more scratch than the library's static area "
             "(ICE3_SURROGATE_SCRATCH_BYTES); use ice3_adjust_rain_ice_surrogate with a work area";
    default: return "unknown error";
  }
}

static void put(std::string &s, const char *name, const double *v, int n) {
  char b[64];
  snprintf(b, sizeof b, "%s %d", name, n);
  s += b;
  for (int k = 0; k < n; ++k) {
    snprintf(b, sizeof b, " %.17e", v[k]);
    s += b;
  }
  s += "\n";
}

extern "C" long ice3_dump_constants(const ice3_ctx *ctx, char *buf, long buflen) {
  // a NULL context builds the constants on the host only (no device needed)
  static ice3_ctx host;
  const ice3_ctx *c = ctx;
  if (!c) {
    ice3_build_params(&host.params, host.h_tab);
    c = &host;
  }
  const ice3_params &P = c->params;
  std::string s;
#define D(x) put(s, #x, &P.x, 1)
  D(XTT); D(XLVTT); D(XLSTT); D(XLMTT); D(XCPD); D(XCPV); D(XCL); D(XCI); D(XRD); D(XRV);
  D(XEPSILO); D(XALPW); D(XBETAW); D(XGAMW); D(XALPI); D(XBETAI); D(XGAMI); D(XESTT); D(XP00);
  D(XRHOLW); D(XPI); D(XG); D(XMNH_TINY);
  put(s, "XRTMIN", P.XRTMIN + 1, 7);
  put(s, "XFRMIN", P.XFRMIN + 1, 40);
  D(XCEXVT); D(XLBR); D(XLBEXR); D(XLBS); D(XLBEXS); D(XLBG); D(XLBEXG); D(XLBI); D(XLBEXI);
  D(XLBDAS_MAX); D(XDI); D(XBS); D(XCXS); D(XCXG); D(XDG); D(XCONC_LAND);
  D(XCRIAUTC); D(XCRIAUTI); D(XACRIAUTI); D(XBCRIAUTI); D(XT0CRIAUTI); D(XNU10); D(XALPHA1);
  D(XBETA1); D(XNU20); D(XALPHA2); D(XBETA2); D(XMNU0); D(XALPHA3); D(XBETA3); D(XHON);
  D(XSCFAC); D(X0DEPI); D(X2DEPI); D(X0DEPS); D(X1DEPS); D(XEX0DEPS); D(XEX1DEPS); D(X0DEPG);
  D(X1DEPG); D(XEX0DEPG); D(XEX1DEPG); D(XTIMAUTI); D(XTEXAUTI); D(XCOLEXIS); D(XFIAGGS);
  D(XEXIAGGS); D(XTIMAUTC); D(XFCACCR); D(XEXCACCR); D(X0EVAR); D(X1EVAR); D(XEX0EVAR);
  D(XEX1EVAR); D(XEXCRIMSS); D(XCRIMSS); D(XEXCRIMSG); D(XCRIMSG); D(XSRIMCG); D(XEXSRIMCG);
  D(XSRIMCG2); D(XSRIMCG3); D(XEXSRIMCG2); D(XRIMINTP1); D(XRIMINTP2);
  D(XFRACCSS); D(XLBRACCS1); D(XLBRACCS2); D(XLBRACCS3); D(XFSACCRG); D(XLBSACCR1);
  D(XLBSACCR2); D(XLBSACCR3); D(XACCINTP1S); D(XACCINTP2S); D(XACCINTP1R); D(XACCINTP2R);
  D(XFSCVMG); D(XEXRCFRI); D(XRCFRI); D(XEXICFRR); D(XICFRR); D(XFCDRYG); D(XCOLIG);
  D(XCOLEXIG); D(XFIDRYG); D(XCOLSG); D(XCOLEXSG); D(XFSDRYG); D(XLBSDRYG1); D(XLBSDRYG2);
  D(XLBSDRYG3); D(XFRDRYG); D(XLBRDRYG1); D(XLBRDRYG2); D(XLBRDRYG3); D(XDRYINTP1R);
  D(XDRYINTP2R); D(XDRYINTP1S); D(XDRYINTP2S); D(XDRYINTP1G); D(XDRYINTP2G); D(XFSEDR);
  D(XEXSEDR); D(XFSEDS); D(XEXSEDS); D(XFSEDG); D(XEXSEDG); D(XFSEDI); D(XEXCSEDI);
  D(XLBH); D(XLBEXH); D(XCXH); D(XDH); D(XBG); D(XFSEDH); D(XEXSEDH); D(X0DEPH); D(X1DEPH);
  D(XEX0DEPH); D(XEX1DEPH); D(XCOLIH); D(XCOLEXIH); D(XCOLSH); D(XCOLEXSH); D(XCOLGH);
  D(XCOLEXGH); D(XFWETH); D(XFSWETH); D(XLBSWETH1); D(XLBSWETH2); D(XLBSWETH3); D(XFGWETH);
  D(XLBGWETH1); D(XLBGWETH2); D(XLBGWETH3); D(XFRWETH); D(XLBRWETH1); D(XLBRWETH2);
  D(XLBRWETH3); D(XWETINTP1S); D(XWETINTP2S); D(XWETINTP1G); D(XWETINTP2G); D(XWETINTP1R);
  D(XWETINTP2R); D(XWETINTP1H); D(XWETINTP2H);
#undef D
  put(s, "XGAMINC_RIM1", c->h_tab + ICE3_T_RIM1, 80);
  put(s, "XGAMINC_RIM2", c->h_tab + ICE3_T_RIM2, 80);
  put(s, "XGAMINC_RIM4", c->h_tab + ICE3_T_RIM4, 80);
  put(s, "XKER_RACCSS", c->h_tab + ICE3_T_RACCSS, 1600);
  put(s, "XKER_RACCS", c->h_tab + ICE3_T_RACCS, 1600);
  put(s, "XKER_SACCRG", c->h_tab + ICE3_T_SACCRG, 1600);
  put(s, "XKER_SDRYG", c->h_tab + ICE3_T_SDRYG, 3200);
  put(s, "XKER_RDRYG", c->h_tab + ICE3_T_RDRYG, 1600);
  put(s, "XKER_SWETH", c->h_tab + ICE3_T_SWETH, 3200);
  put(s, "XKER_GWETH", c->h_tab + ICE3_T_GWETH, 1600);
  put(s, "XKER_RWETH", c->h_tab + ICE3_T_RWETH, 1600);
  long n = (long)s.size();
  if (buf && buflen > 0) {
    long m = n < buflen - 1 ? n : buflen - 1;
    memcpy(buf, s.data(), (size_t)m);
    buf[m] = 0;
  }
  return n;
}

static bool bad_shape(int ncol, int nlev, int ld, double dt) {
  return ncol <= 0 || nlev <= 0 || ld < ncol || !(dt > 0.) ||
         (double)ld * (double)nlev > 9.0e15 || (double)ncol * (double)nlev > 4294967295.0;
}

// A domain with no column or no level: a valid call with nothing to do (its field pointers
// may be NULL, as an empty array's are).
static bool empty_domain(int ncol, int nlev, int ld, double dt) {
  return (ncol == 0 || nlev == 0) && ncol >= 0 && nlev >= 0 && ld >= ncol && dt > 0.;
}

static bool known_prec(int prec) { return prec == ICE3_PREC_FP64 || prec == ICE3_PREC_MIXED; }

#define NN(p) if (!(p)) return ICE3_EINVAL

extern "C" int ice3_count_nonfinite(int nfield, const double *const *fields, const int *rows,
                                    int ncol, int ld, unsigned long long *counts, void *stream) {
  if (nfield < 0 || nfield > ICE3_MAX_CHECK_FIELDS || ncol < 0 || ld < ncol) return ICE3_EINVAL;
  if (nfield == 0 || ncol == 0) return ICE3_OK;
  if (!fields || !rows || !counts) return ICE3_EINVAL;
  CountArgs a = CountArgs{};
  a.ncol = ncol; a.ld = ld; a.counts = counts;
  int maxrows = 0;
  for (int q = 0; q < nfield; ++q) {
    if (rows[q] < 0 || (rows[q] > 0 && !fields[q])) return ICE3_EINVAL;
    if ((double)rows[q] * (double)ld > 9.0e15) return ICE3_EINVAL;
    a.f[q] = fields[q];
    a.rows[q] = rows[q];
    maxrows = rows[q] > maxrows ? rows[q] : maxrows;
  }
  if (maxrows == 0) return ICE3_OK;
  const int blocks = (ncol + 255) / 256;
  dim3 grid(blocks < 1024 ? blocks : 1024, nfield);
  hipLaunchKernelGGL(k_count_nonfinite, grid, dim3(256), 0, (hipStream_t)stream, a);
  HIPCHK(hipGetLastError());
  return ICE3_OK;
}

extern "C" int ice3_divide(int n, const double *a, const double *b, double *q, void *stream) {
  if (n < 0 || (n > 0 && (!a || !b || !q))) return ICE3_EINVAL;
  if (n == 0) return ICE3_OK;
  hipLaunchKernelGGL(k_divide, dim3((n - 1) / 256 + 1), dim3(256), 0, (hipStream_t)stream, n, a, b, q);
  HIPCHK(hipGetLastError());
  return ICE3_OK;
}

extern "C" int ice3_transpose_fields(int nfield, const double *const *src, double *const *dst, int rows,
                                     int cols, void *stream) {
  if (nfield < 0 || nfield > ICE3_MAX_CHECK_FIELDS || rows < 0 || cols < 0) return ICE3_EINVAL;
  if (nfield == 0 || rows == 0 || cols == 0) return ICE3_OK;
  if (!src || !dst) return ICE3_EINVAL;
  TransposeArgs a = TransposeArgs{};
  for (int q = 0; q < nfield; ++q) {
    NN(src[q]); NN(dst[q]);
    if ((const double *)dst[q] == src[q]) return ICE3_EINVAL;
    a.src[q] = src[q];
    a.dst[q] = dst[q];
  }
  a.rows = rows; a.cols = cols; a.col_tiles = (cols - 1) / TR_COLS + 1;
  const size_t blocks = ((size_t)rows + TR_ROWS - 1) / TR_ROWS * a.col_tiles;
  if (blocks >= (size_t)1 << 24) return ICE3_EINVAL;  // a launch takes fewer than 2^32 threads along an axis
  hipLaunchKernelGGL(k_transpose, dim3((unsigned)blocks, nfield), dim3(256), 0, (hipStream_t)stream, a);
  HIPCHK(hipGetLastError());
  return ICE3_OK;
}

extern "C" int ice3_ice_adjust(ice3_ctx *ctx, int prec, int ncol, int nlev, int ld, double dt,
                               const ice3_ice_adjust_in *in, const ice3_ice_adjust_out *out,
                               void *stream) {
  if (!ctx || !in || !out || !known_prec(prec)) return ICE3_EINVAL;
  if (empty_domain(ncol, nlev, ld, dt)) return ICE3_OK;
  if (bad_shape(ncol, nlev, ld, dt)) return ICE3_EINVAL;
  NN(in->pabs); NN(in->sigs); NN(in->th); NN(in->exn); NN(in->exn_ref); NN(in->rho_dry_ref);
  NN(in->rv); NN(in->rc); NN(in->ri); NN(in->rr); NN(in->rs); NN(in->rg); NN(in->cf_mf);
  NN(in->rc_mf); NN(in->ri_mf); NN(in->rvs); NN(in->rcs); NN(in->ris); NN(in->ths);
  NN(in->sigqsat);
  NN(out->t); NN(out->rv_out); NN(out->rc_out); NN(out->ri_out); NN(out->cldfr);
  NN(out->hlc_hrc); NN(out->hlc_hcf); NN(out->hli_hri); NN(out->hli_hcf); NN(out->cph);
  NN(out->lv); NN(out->ls); NN(out->rvs); NN(out->rcs); NN(out->ris); NN(out->ths);
  if (nlev > 65535) return ICE3_EINVAL;
  AdjustArgs a = AdjustArgs{};  // ris_copy stays NULL
  a.ncol = ncol; a.nlev = nlev; a.ld = ld; a.dt = dt; a.in = *in; a.out = *out;
  dim3 grid((ncol + 255) / 256, nlev);
  hipStream_t s = (hipStream_t)stream;
  MARK(0);
  hipLaunchKernelGGL(k_ice_adjust, grid, dim3(256), 0, s, a);
  HIPCHK(hipGetLastError());
  MARK(1); MARK(2); MARK(3); MARK(4); MARK(5); MARK(6);
  return ICE3_OK;
}

extern "C" int ice3_ice_adjust_ocnd2(ice3_ctx *ctx, int ncol, int nlev, int ld, double dt,
                                     const ice3_ice_adjust_in *in, const ice3_ocnd2_in *in2,
                                     const ice3_ice_adjust_out *out, const ice3_ocnd2_out *out2,
                                     void *stream) {
  if (!ctx || !in || !in2 || !out || !out2) return ICE3_EINVAL;
  if (empty_domain(ncol, nlev, ld, dt)) return ICE3_OK;
  if (bad_shape(ncol, nlev, ld, dt) || nlev < 2 || nlev > 65535) return ICE3_EINVAL;
  NN(in->pabs); NN(in->sigs); NN(in->th); NN(in->exn); NN(in->exn_ref); NN(in->rho_dry_ref);
  NN(in->rv); NN(in->rc); NN(in->ri); NN(in->rr); NN(in->rs); NN(in->rg); NN(in->cf_mf);
  NN(in->rc_mf); NN(in->ri_mf); NN(in->rvs); NN(in->rcs); NN(in->ris); NN(in->ths);
  NN(in->sigqsat); NN(in2->zz); NN(in2->ice_cld_wgt);
  NN(out->t); NN(out->rv_out); NN(out->rc_out); NN(out->ri_out); NN(out->cldfr);
  NN(out->hlc_hrc); NN(out->hlc_hcf); NN(out->hli_hri); NN(out->hli_hcf); NN(out->cph);
  NN(out->lv); NN(out->ls); NN(out->rvs); NN(out->rcs); NN(out->ris); NN(out->ths);
  NN(out2->icldfr); NN(out2->wcldfr); NN(out2->ssio); NN(out2->ssiu); NN(out2->ifr);
  AdjustArgs a = AdjustArgs{};
  a.ncol = ncol; a.nlev = nlev; a.ld = ld; a.dt = dt; a.in = *in; a.out = *out;
  Ocnd2Args x{*in2, *out2, ctx->d_tiwmx};
  dim3 grid((ncol + 255) / 256, nlev);
  hipStream_t s = (hipStream_t)stream;
  MARK(0);
  hipLaunchKernelGGL(k_ice_adjust_ocnd2, grid, dim3(256), 0, s, a, x);
  HIPCHK(hipGetLastError());
  MARK(1); MARK(2); MARK(3); MARK(4); MARK(5); MARK(6);
  return ICE3_OK;
}

// ICE_ADJUST and the statistical sedimentation of the FP64 fused step; aa.rh (with sa.src_rh)
// selects hail.  One column walk when there are enough columns to hide its latency: a lone
// wavefront takes 6 us a level, so that 1,024 to 65,536 columns of 90 levels all take 0.53 to
// 0.60 ms, against 0.08 to 0.44 ms for ICE_ADJUST point by point followed by k_sedim; or levels
// so few that there is little to wait for (sedim_walk_cols).  From 432 columns a compute unit (1.7
// wavefronts per SIMD) on the walk saves more traffic than it waits: at 98,304 columns 0.69 against 0.63 ms, at 106,496 0.71 against 0.69, at 114,688 0.715 against 0.737
// (hail: 0.79 against 0.91), at 131,072 0.75 against 0.82, at 262,144 1.40 against 1.63.
static hipError_t launch_adjust_sedim(const ice3_ctx *ctx, const AdjustArgs &aa, const SedimArgs &sa,
                                      hipStream_t s) {
  const dim3 gw((aa.ncol + 63) / 64), gp((aa.ncol + 255) / 256, aa.nlev);
  if (aa.ncol >= (long long)sedim_walk_cols(SEDIM_FUSED, aa.nlev) * ctx->ncu) {
    if (aa.rh) hipLaunchKernelGGL(k_adjust_sedim_hail, gw, dim3(64), 0, s, aa, sa);
    else hipLaunchKernelGGL(k_adjust_sedim, gw, dim3(64), 0, s, aa, sa);
    return hipGetLastError();
  }
  if (aa.rh) hipLaunchKernelGGL(k_ice_adjust_hail, gp, dim3(256), 0, s, aa);
  else hipLaunchKernelGGL(k_ice_adjust, gp, dim3(256), 0, s, aa);
  const hipError_t e = hipGetLastError();
  return e != hipSuccess ? e : sedim_launch<double>(sa, ctx->ncu, s);
}

extern "C" int ice3_ice_adjust_rows(ice3_ctx *ctx, int ncol, int nlev, double dt,
                                    const ice3_ice_adjust_in *in, const double *rh,
                                    const ice3_ocnd2_in *in2, const ice3_ice_adjust_out *out,
                                    const ice3_ocnd2_out *out2, void *stream) {
  if (!ctx || !in || !out || (in2 == nullptr) != (out2 == nullptr) || (rh && in2)) return ICE3_EINVAL;
  if (empty_domain(ncol, nlev, ncol, dt)) return ICE3_OK;
  if (bad_shape(ncol, nlev, ncol, dt) || nlev > 65535 || (in2 && nlev < 2)) return ICE3_EINVAL;
  NN(in->pabs); NN(in->sigs); NN(in->th); NN(in->exn); NN(in->exn_ref); NN(in->rho_dry_ref);
  NN(in->rv); NN(in->rc); NN(in->ri); NN(in->rr); NN(in->rs); NN(in->rg); NN(in->cf_mf);
  NN(in->rc_mf); NN(in->ri_mf); NN(in->rvs); NN(in->rcs); NN(in->ris); NN(in->ths);
  NN(in->sigqsat);
  NN(out->t); NN(out->rv_out); NN(out->rc_out); NN(out->ri_out); NN(out->cldfr);
  NN(out->hlc_hrc); NN(out->hlc_hcf); NN(out->hli_hri); NN(out->hli_hcf); NN(out->cph);
  NN(out->lv); NN(out->ls); NN(out->rvs); NN(out->rcs); NN(out->ris); NN(out->ths);
  AdjustArgs a = AdjustArgs{};
  a.ncol = ncol; a.nlev = nlev; a.ld = 1; a.dt = dt; a.in = *in; a.out = *out; a.rh = rh;
  Ocnd2Args x = Ocnd2Args{};
  if (in2) {
    NN(in2->zz); NN(in2->ice_cld_wgt);
    NN(out2->icldfr); NN(out2->wcldfr); NN(out2->ssio); NN(out2->ssiu); NN(out2->ifr);
    x = Ocnd2Args{*in2, *out2, ctx->d_tiwmx};
  }
  const unsigned npts = (unsigned)ncol * (unsigned)nlev;
  const dim3 grid((unsigned)(((size_t)npts + 255) / 256));
  hipStream_t s = (hipStream_t)stream;
  MARK(0);
  if (in2) hipLaunchKernelGGL((k_ice_adjust_rows<true, false>), grid, dim3(256), 0, s, a, x, npts);
  else if (rh) hipLaunchKernelGGL((k_ice_adjust_rows<false, true>), grid, dim3(256), 0, s, a, x, npts);
  else hipLaunchKernelGGL((k_ice_adjust_rows<false, false>), grid, dim3(256), 0, s, a, x, npts);
  HIPCHK(hipGetLastError());
  MARK(1); MARK(2); MARK(3); MARK(4); MARK(5); MARK(6);
  return ICE3_OK;
}

// Launch k_micro: one workgroup per compute unit (its LDS holds the tables and the parked
// points, so one workgroup fits a CU).
static hipError_t launch_micro(const ice3_ctx *ctx, int prec, const MicroArgs &m, hipStream_t s) {
  if (m.max_calls != DEFAULT_MAX_CALLS) {  // a context-set cap: the point kernel reads it
    const unsigned int npts = (unsigned int)m.nlev * (unsigned int)m.ncol;
    const dim3 g((npts + 255) / 256);
    if (prec == ICE3_PREC_FP64) hipLaunchKernelGGL(k_micro_points<double>, g, dim3(256), 0, s, m);
    else hipLaunchKernelGGL(k_micro_points<float>, g, dim3(256), 0, s, m);
    return hipGetLastError();
  }
  if (prec == ICE3_PREC_FP64)
    hipLaunchKernelGGL(k_micro<double>, dim3(ctx->ncu), dim3(64 * micro_waves<double>()),
                       micro_lds_bytes<double>(), s, m);
  else
    hipLaunchKernelGGL(k_micro<float>, dim3(ctx->ncu), dim3(64 * micro_waves<float>()),
                       micro_lds_bytes<float>(), s, m);
  return hipGetLastError();
}

// The OCND2 microphysics (FP64): one workgroup per compute unit, or the point kernel when the
// context sets another sub-step cap.
static hipError_t launch_micro_ocnd2(const ice3_ctx *ctx, const MicroArgs &m, hipStream_t s) {
  if (m.max_calls != DEFAULT_MAX_CALLS) {
    const unsigned int npts = (unsigned int)m.nlev * (unsigned int)m.ncol;
    hipLaunchKernelGGL((k_micro_points<double, true>), dim3((npts + 255) / 256), dim3(256), 0, s, m);
  } else {
    hipLaunchKernelGGL((k_micro<double, true>), dim3(ctx->ncu), dim3(64 * micro_waves<double>()),
                       micro_lds_bytes<double>(), s, m);
  }
  return hipGetLastError();
}

// Levels a wavefront of k_sedim_split holds (4 slots per lane).
constexpr int SPLIT_MAX_LEVELS = 4 * 64;

// Whether the context's sedimentation scheme can run nlev levels.
static bool sedim_fits(const ice3_ctx *ctx, int nlev) {
  return ctx->sedim != ICE3_SEDIM_SPLI || nlev <= SPLIT_MAX_LEVELS;
}

template <int L, bool HAIL, bool ZZZ>
static void launch_split_k(const SplitArgs &a, hipStream_t s) {
  hipLaunchKernelGGL((k_sedim_split<L, HAIL, ZZZ>), dim3((a.ncol + SPLIT_COLS - 1) / SPLIT_COLS),
                     dim3(64 * SPLIT_COLS), 0, s, a);
}

template <bool HAIL, bool ZZZ>
static void launch_split_l(const SplitArgs &a, hipStream_t s) {
  switch ((a.nlev + 63) / 64) {
    case 1: launch_split_k<1, HAIL, ZZZ>(a, s); break;
    case 2: launch_split_k<2, HAIL, ZZZ>(a, s); break;
    case 3: launch_split_k<3, HAIL, ZZZ>(a, s); break;
    default: launch_split_k<4, HAIL, ZZZ>(a, s); break;
  }
}

// The split sedimentation (CSEDIM='SPLI') of the stages described by sa (sedimentation) and m
// (the state at t and the th, rv, rc sources); sa.zzz selects the OCND2 model level height,
// sa.src_rh hail.  nlev <= SPLIT_MAX_LEVELS (checked by the entry points).
static hipError_t launch_split(const ice3_ctx *ctx, const SedimArgs &sa, const MicroArgs &m,
                               hipStream_t s, double *const *keep = nullptr) {
  SplitArgs a = split_args(sa, m, ctx->maxcfl, ctx->d_capped);
  if (keep)
    for (int q = 0; q < 3; ++q) a.keep[q] = keep[q];
  if (sa.src_rh) launch_split_l<true, false>(a, s);
  else if (sa.zzz) launch_split_l<false, true>(a, s);
  else launch_split_l<false, false>(a, s);
  return hipGetLastError();
}

// The fused step with the split sedimentation: its negativity correction updates the th, rv
// and rc sources, whose values before it, times dt, are the microphysics' state at t.  The
// split kernel stores them as it reads them into the context's work area (3 fields, grown on
// demand; growing it waits for the device), and m then reads its state at t there.
static int launch_split_keep(ice3_ctx *ctx, int nlev, int ld, const SedimArgs &sa, MicroArgs &m,
                             hipStream_t s) {
  const size_t n = (size_t)nlev * ld;
  const size_t bytes = 3 * n * sizeof(double);
  if (bytes > ctx->work_bytes) {
    HIPCHK(hipDeviceSynchronize());
    if (ctx->d_work) HIPCHK(hipFree(ctx->d_work));
    ctx->d_work = nullptr;
    ctx->work_bytes = 0;
    HIPCHK(hipMalloc(&ctx->d_work, bytes));
    ctx->work_bytes = bytes;
  }
  double *w = (double *)ctx->d_work;
  double *const keep[3] = {w, w + n, w + 2 * n};
  HIPCHK(launch_split(ctx, sa, m, s, keep));
  for (int q = 0; q < 3; ++q) m.t[q] = keep[q];
  return ICE3_OK;
}

// The rain_ice entry points: checks, the sedimentation, the microphysics.  The sources are read
// from src and written to io (and hail->rhs), each from its own array or from the one it is
// written to.  in2 selects OCND2, hail KRR=7.
static hipError_t launch_micro_hail(const ice3_ctx *ctx, const MicroArgs &m, hipStream_t s);

static int rain_ice_call(ice3_ctx *ctx, int prec, int ncol, int nlev, int ld, double dt,
                         const ice3_rain_ice_in *in, const ice3_rain_ocnd2_in *in2,
                         const ice3_rain_ice_src *src, const ice3_rain_ice_inout *io,
                         const ice3_rain_ice_out *out, const ice3_hail *hail,
                         const ice3_stats *stats, void *stream) {
  if (empty_domain(ncol, nlev, ld, dt)) return ICE3_OK;
  if (bad_shape(ncol, nlev, ld, dt) || nlev > 65535) return ICE3_EINVAL;
  NN(in->exn); NN(in->dzz); NN(in->rhodref); NN(in->exn_ref); NN(in->pabs); NN(in->cldfr);
  NN(in->sigs); NN(in->tht); NN(in->rvt); NN(in->rct); NN(in->rrt); NN(in->rit); NN(in->rst);
  NN(in->rgt);
  NN(src->ths); NN(src->rvs); NN(src->rcs); NN(src->rrs); NN(src->ris); NN(src->rss); NN(src->rgs);
  NN(src->ci);
  NN(io->ths); NN(io->rvs); NN(io->rcs); NN(io->rrs); NN(io->ris); NN(io->rss); NN(io->rgs);
  NN(io->ci);
  NN(out->evap3d); NN(out->rainfr); NN(out->inprc); NN(out->inprr); NN(out->inpri);
  NN(out->inprs); NN(out->inprg);
  if (in2) { NN(in2->icldfr); NN(in2->ssio); NN(in2->ssiu); NN(in2->ifr); }
  if (hail) { NN(hail->rht); NN(hail->rhs); NN(hail->inprh); NN(src->rhs); }
  if (!sedim_fits(ctx, nlev)) return ICE3_EINVAL;
  SedimArgs sa;
  MicroArgs m;
  rain_ice_args(ncol, nlev, ld, dt, ctx->d_tab, in, io, out, stats, sa, m);
  sa.src_rr = src->rrs; sa.src_ri = src->ris; sa.src_rs = src->rss; sa.src_rg = src->rgs;
  m.src[ITH] = src->ths; m.src[IRV] = src->rvs; m.src[IRC] = src->rcs; m.src_ci = src->ci;
  m.max_calls = ctx->max_calls; m.capped = ctx->d_capped;
  if (in2) {
    m.icldfr = in2->icldfr; m.ssio = in2->ssio; m.ssiu = in2->ssiu; m.ifr = in2->ifr;
    m.tiwmx = ctx->d_tiwmx;
    sa.zzz = out->rainfr;  // the model level height, read by the microphysics, then overwritten
  }
  if (hail) {
    sa.src_rh = src->rhs; sa.dst_rh = hail->rhs; sa.inprh = hail->inprh;
    m.t[IRH] = hail->rht; m.src[IRH] = hail->rhs; m.dst[IRH] = hail->rhs;
  }
  hipStream_t s = (hipStream_t)stream;
  MARK(0); MARK(1);
  if (ctx->sedim == ICE3_SEDIM_SPLI) {
    HIPCHK(launch_split(ctx, sa, m, s));  // and corrects the th, rv and rc sources
    m.src[ITH] = m.dst[ITH]; m.src[IRV] = m.dst[IRV]; m.src[IRC] = m.dst[IRC];
  } else if (prec == ICE3_PREC_FP64) {
    HIPCHK(sedim_launch<double>(sa, ctx->ncu, s));
  } else {
    HIPCHK(sedim_launch<float>(sa, ctx->ncu, s));
  }
  MARK(2);
  HIPCHK(in2 ? launch_micro_ocnd2(ctx, m, s) : hail ? launch_micro_hail(ctx, m, s) : launch_micro(ctx, prec, m, s));
  MARK(3); MARK(4); MARK(5); MARK(6);
  return ICE3_OK;
}

// The sources of an in-place call.
static ice3_rain_ice_src sources_of(const ice3_rain_ice_inout *io, const double *rhs) {
  return ice3_rain_ice_src{io->ths, io->rvs, io->rcs, io->rrs, io->ris, io->rss, io->rgs, io->ci, rhs};
}

extern "C" int ice3_rain_ice(ice3_ctx *ctx, int prec, int ncol, int nlev, int ld, double dt,
                             const ice3_rain_ice_in *in, const ice3_rain_ice_inout *io,
                             const ice3_rain_ice_out *out, const ice3_stats *stats,
                             void *stream) {
  if (!ctx || !in || !io || !out || !known_prec(prec)) return ICE3_EINVAL;
  const ice3_rain_ice_src src = sources_of(io, nullptr);
  return rain_ice_call(ctx, prec, ncol, nlev, ld, dt, in, nullptr, &src, io, out, nullptr, stats, stream);
}

extern "C" int ice3_rain_ice_ocnd2(ice3_ctx *ctx, int ncol, int nlev, int ld, double dt,
                                   const ice3_rain_ice_in *in, const ice3_rain_ocnd2_in *in2,
                                   const ice3_rain_ice_inout *io, const ice3_rain_ice_out *out,
                                   const ice3_stats *stats, void *stream) {
  if (!ctx || !in || !in2 || !io || !out) return ICE3_EINVAL;
  const ice3_rain_ice_src src = sources_of(io, nullptr);
  return rain_ice_call(ctx, ICE3_PREC_FP64, ncol, nlev, ld, dt, in, in2, &src, io, out, nullptr, stats,
                       stream);
}

extern "C" int ice3_rain_ice_hail(ice3_ctx *ctx, int ncol, int nlev, int ld, double dt,
                                  const ice3_rain_ice_in *in, const ice3_rain_ice_inout *io,
                                  const ice3_rain_ice_out *out, const ice3_hail *hail,
                                  const ice3_stats *stats, void *stream) {
  if (!ctx || !in || !io || !out || !hail) return ICE3_EINVAL;
  const ice3_rain_ice_src src = sources_of(io, hail->rhs);
  return rain_ice_call(ctx, ICE3_PREC_FP64, ncol, nlev, ld, dt, in, nullptr, &src, io, out, hail, stats,
                       stream);
}

// Whether an array of src is an output other than the one of the same name.  The sedimentation's
// wavefronts each write their own species while others still read, and the microphysics writes
// some points while others wait, so such a source would be overwritten before it is read.
static bool crossed_sources(const ice3_rain_ice_src *src, const ice3_rain_ice_inout *io,
                            const ice3_rain_ice_out *out, const ice3_hail *hail) {
  const double *const s[9] = {src->ths, src->rvs, src->rcs, src->rrs, src->ris,
                              src->rss, src->rgs, src->ci,  hail ? src->rhs : nullptr};
  const double *const w[9] = {io->ths, io->rvs, io->rcs, io->rrs, io->ris,
                              io->rss, io->rgs, io->ci,  hail ? hail->rhs : nullptr};
  const double *const o[8] = {out->evap3d, out->rainfr, out->inprc, out->inprr, out->inpri,
                              out->inprs,  out->inprg,  hail ? hail->inprh : nullptr};
  for (int a = 0; a < 9; ++a) {
    if (!s[a]) continue;
    for (int b = 0; b < 9; ++b)
      if (a != b && s[a] == w[b]) return true;
    for (int b = 0; b < 8; ++b)
      if (s[a] == o[b]) return true;
  }
  return false;
}

extern "C" int ice3_rain_ice_from(ice3_ctx *ctx, int prec, int ncol, int nlev, int ld, double dt,
                                  const ice3_rain_ice_in *in, const ice3_rain_ocnd2_in *in2,
                                  const ice3_rain_ice_src *src, const ice3_rain_ice_inout *io,
                                  const ice3_rain_ice_out *out, const ice3_hail *hail,
                                  const ice3_stats *stats, void *stream) {
  if (!ctx || !in || !src || !io || !out || !known_prec(prec) || (in2 && hail) ||
      ((in2 || hail) && prec != ICE3_PREC_FP64))
    return ICE3_EINVAL;
  if (!empty_domain(ncol, nlev, ld, dt) && crossed_sources(src, io, out, hail)) return ICE3_EINVAL;
  return rain_ice_call(ctx, prec, ncol, nlev, ld, dt, in, in2, src, io, out, hail, stats, stream);
}

static bool bad_pipeline_ptrs(const ice3_pipeline_in *in, const ice3_pipeline_out *out) {
  const void *const pin[] = {in->pabs, in->sigs, in->th, in->exn, in->exn_ref, in->rhodref,
                             in->dzz, in->rv, in->rc, in->ri, in->rr, in->rs, in->rg, in->ci,
                             in->cf_mf, in->rc_mf, in->ri_mf, in->ths, in->rvs, in->rcs,
                             in->rrs, in->ris, in->rss, in->rgs, in->sigqsat};
  const void *const pout[] = {out->ths, out->rvs, out->rcs, out->rrs, out->ris, out->rss,
                              out->rgs, out->cldfr, out->hlc_hrc, out->hlc_hcf, out->hli_hri,
                              out->hli_hcf, out->ci, out->evap3d, out->rainfr, out->inprc,
                              out->inprr, out->inpri, out->inprs, out->inprg};
  for (const void *p : pin)
    if (!p) return true;
  for (const void *p : pout)
    if (!p) return true;
  return false;
}

extern "C" int ice3_adjust_rain_ice_stages(ice3_ctx *ctx, int prec, int ncol, int nlev, int ld,
                                           double dt, const ice3_pipeline_in *in,
                                           const ice3_pipeline_out *out,
                                           const ice3_stats *stats, int stages, void *stream) {
  if (!ctx || !in || !out || !known_prec(prec) || stages <= 0 || stages > 7) return ICE3_EINVAL;
  if (empty_domain(ncol, nlev, ld, dt)) return ICE3_OK;
  if (bad_shape(ncol, nlev, ld, dt) || nlev > 65535) return ICE3_EINVAL;
  if (bad_pipeline_ptrs(in, out)) return ICE3_EINVAL;
  if ((stages & ICE3_STAGE_SEDIMENTATION) && !sedim_fits(ctx, nlev)) return ICE3_EINVAL;
  // with SPLI the microphysics' state at t is kept by the sedimentation stage of its call
  if (ctx->sedim == ICE3_SEDIM_SPLI && (stages & ICE3_STAGE_MICROPHYSICS) &&
      !(stages & ICE3_STAGE_SEDIMENTATION))
    return ICE3_EINVAL;
  AdjustArgs aa;
  SedimArgs sa;
  MicroArgs m;
  pipeline_args(ncol, nlev, ld, dt, ctx->d_tab, in, out, stats, aa, sa, m);
  m.max_calls = ctx->max_calls; m.capped = ctx->d_capped;
  hipStream_t s = (hipStream_t)stream;
  const dim3 gp((ncol + 255) / 256, nlev);
  const bool split = ctx->sedim == ICE3_SEDIM_SPLI;
  if ((stages & ICE3_STAGE_ADJUST) && (stages & ICE3_STAGE_SEDIMENTATION)) hand_ris_over(aa, sa);
  MARK(0);
  if (prec == ICE3_PREC_FP64 && !split && (stages & ICE3_STAGE_ADJUST) &&
      (stages & ICE3_STAGE_SEDIMENTATION)) {
    // one column walk for both stages (in the mixed path the float sedimentation is cheap
    // and the two kernels are faster apart)
    HIPCHK(launch_adjust_sedim(ctx, aa, sa, s));
    stages &= ~ICE3_STAGE_SEDIMENTATION;
  } else if (stages & ICE3_STAGE_ADJUST) {
    hipLaunchKernelGGL(k_ice_adjust, gp, dim3(256), 0, s, aa);
    HIPCHK(hipGetLastError());
  }
  MARK(1);
  if (stages & ICE3_STAGE_SEDIMENTATION) {
    if (split && (stages & ICE3_STAGE_MICROPHYSICS)) {
      const int rc = launch_split_keep(ctx, nlev, ld, sa, m, s);
      if (rc != ICE3_OK) return rc;
    } else if (split) {
      HIPCHK(launch_split(ctx, sa, m, s));
    } else if (prec == ICE3_PREC_FP64) {
      HIPCHK(sedim_launch<double>(sa, ctx->ncu, s));
    } else {
      HIPCHK(sedim_launch<float>(sa, ctx->ncu, s));
    }
  }
  MARK(2);
  if (stages & ICE3_STAGE_MICROPHYSICS) {
    HIPCHK(launch_micro(ctx, prec, m, s));
  }
  MARK(3); MARK(4); MARK(5); MARK(6);
  return ICE3_OK;
}

extern "C" int ice3_adjust_rain_ice(ice3_ctx *ctx, int prec, int ncol, int nlev, int ld,
                                    double dt, const ice3_pipeline_in *in,
                                    const ice3_pipeline_out *out, const ice3_stats *stats,
                                    void *stream) {
  return ice3_adjust_rain_ice_stages(ctx, prec, ncol, nlev, ld, dt, in, out, stats,
                                     ICE3_STAGE_ADJUST | ICE3_STAGE_SEDIMENTATION |
                                         ICE3_STAGE_MICROPHYSICS,
                                     stream);
}

extern "C" int ice3_adjust_rain_ice_ocnd2(ice3_ctx *ctx, int ncol, int nlev, int ld, double dt,
                                          const ice3_pipeline_in *in, const ice3_ocnd2_in *in2,
                                          const ice3_pipeline_out *out,
                                          const ice3_ocnd2_out *out2, const ice3_stats *stats,
                                          void *stream) {
  if (!ctx || !in || !in2 || !out || !out2) return ICE3_EINVAL;
  if (empty_domain(ncol, nlev, ld, dt)) return ICE3_OK;
  if (bad_shape(ncol, nlev, ld, dt) || nlev < 2 || nlev > 65535) return ICE3_EINVAL;
  if (bad_pipeline_ptrs(in, out)) return ICE3_EINVAL;
  NN(in2->zz); NN(in2->ice_cld_wgt);
  NN(out2->icldfr); NN(out2->wcldfr); NN(out2->ssio); NN(out2->ssiu); NN(out2->ifr);
  AdjustArgs aa;
  SedimArgs sa;
  MicroArgs m;
  pipeline_args(ncol, nlev, ld, dt, ctx->d_tab, in, out, stats, aa, sa, m);
  m.max_calls = ctx->max_calls; m.capped = ctx->d_capped;
  m.icldfr = out2->icldfr; m.ssio = out2->ssio; m.ssiu = out2->ssiu; m.ifr = out2->ifr;
  m.tiwmx = ctx->d_tiwmx;
  sa.zzz = out->rainfr;  // the model level height, read by the microphysics, then overwritten
  if (!sedim_fits(ctx, nlev)) return ICE3_EINVAL;
  const Ocnd2Args x{*in2, *out2, ctx->d_tiwmx};
  hipStream_t s = (hipStream_t)stream;
  hand_ris_over(aa, sa);
  MARK(0);
  hipLaunchKernelGGL(k_ice_adjust_ocnd2, dim3((ncol + 255) / 256, nlev), dim3(256), 0, s, aa, x);
  HIPCHK(hipGetLastError());
  MARK(1);
  if (ctx->sedim == ICE3_SEDIM_SPLI) {
    const int rc = launch_split_keep(ctx, nlev, ld, sa, m, s);
    if (rc != ICE3_OK) return rc;
  } else {
    HIPCHK(sedim_launch<double>(sa, ctx->ncu, s));
  }
  MARK(2);
  HIPCHK(launch_micro_ocnd2(ctx, m, s));
  MARK(3); MARK(4); MARK(5); MARK(6);
  return ICE3_OK;
}

// ---- hail (KRR=7) entry points, FP64

extern "C" int ice3_ice_adjust_hail(ice3_ctx *ctx, int ncol, int nlev, int ld, double dt,
                                    const ice3_ice_adjust_in *in, const double *rh,
                                    const ice3_ice_adjust_out *out, void *stream) {
  if (!ctx || !in || !out) return ICE3_EINVAL;
  if (empty_domain(ncol, nlev, ld, dt)) return ICE3_OK;
  if (bad_shape(ncol, nlev, ld, dt) || nlev > 65535) return ICE3_EINVAL;
  NN(in->pabs); NN(in->sigs); NN(in->th); NN(in->exn); NN(in->exn_ref); NN(in->rho_dry_ref);
  NN(in->rv); NN(in->rc); NN(in->ri); NN(in->rr); NN(in->rs); NN(in->rg); NN(in->cf_mf);
  NN(in->rc_mf); NN(in->ri_mf); NN(in->rvs); NN(in->rcs); NN(in->ris); NN(in->ths);
  NN(in->sigqsat); NN(rh);
  NN(out->t); NN(out->rv_out); NN(out->rc_out); NN(out->ri_out); NN(out->cldfr);
  NN(out->hlc_hrc); NN(out->hlc_hcf); NN(out->hli_hri); NN(out->hli_hcf); NN(out->cph);
  NN(out->lv); NN(out->ls); NN(out->rvs); NN(out->rcs); NN(out->ris); NN(out->ths);
  AdjustArgs a = AdjustArgs{};
  a.ncol = ncol; a.nlev = nlev; a.ld = ld; a.dt = dt; a.in = *in; a.out = *out; a.rh = rh;
  hipStream_t s = (hipStream_t)stream;
  MARK(0);
  hipLaunchKernelGGL(k_ice_adjust_hail, dim3((ncol + 255) / 256, nlev), dim3(256), 0, s, a);
  HIPCHK(hipGetLastError());
  MARK(1); MARK(2); MARK(3); MARK(4); MARK(5); MARK(6);
  return ICE3_OK;
}

// The hail microphysics (FP64): one workgroup per compute unit, or the point kernel when the
// context sets another sub-step cap (it reads the cap at run time).
static hipError_t launch_micro_hail(const ice3_ctx *ctx, const MicroArgs &m, hipStream_t s) {
  if (m.max_calls != DEFAULT_MAX_CALLS) {
    const unsigned int npts = (unsigned int)m.nlev * (unsigned int)m.ncol;
    hipLaunchKernelGGL((k_micro_points<double, false, true>), dim3((npts + 255) / 256), dim3(256),
                       0, s, m);
  } else {
    hipLaunchKernelGGL((k_micro<double, false, true>), dim3(ctx->ncu),
                       dim3(64 * (micro_waves<double, true>())), (micro_lds_bytes<double, true>()), s, m);
  }
  return hipGetLastError();
}

extern "C" int ice3_ice_adjust_branches(ice3_ctx *ctx, int ncol, int nlev, int ld, double dt,
                                        const ice3_ice_adjust_in *in, const double *rh,
                                        const ice3_ice_adjust_out *out, unsigned *branches,
                                        void *stream) {
  if (!ctx || !in || !out || !branches) return ICE3_EINVAL;
  if (empty_domain(ncol, nlev, ld, dt)) return ICE3_OK;
  if (bad_shape(ncol, nlev, ld, dt) || nlev > 65535) return ICE3_EINVAL;
  NN(in->pabs); NN(in->sigs); NN(in->th); NN(in->exn); NN(in->exn_ref); NN(in->rho_dry_ref);
  NN(in->rv); NN(in->rc); NN(in->ri); NN(in->rr); NN(in->rs); NN(in->rg); NN(in->cf_mf);
  NN(in->rc_mf); NN(in->ri_mf); NN(in->rvs); NN(in->rcs); NN(in->ris); NN(in->ths);
  NN(in->sigqsat);
  NN(out->t); NN(out->rv_out); NN(out->rc_out); NN(out->ri_out); NN(out->cldfr);
  NN(out->hlc_hrc); NN(out->hlc_hcf); NN(out->hli_hri); NN(out->hli_hcf); NN(out->cph);
  NN(out->lv); NN(out->ls); NN(out->rvs); NN(out->rcs); NN(out->ris); NN(out->ths);
  AdjustArgs a = AdjustArgs{};
  a.ncol = ncol; a.nlev = nlev; a.ld = ld; a.dt = dt; a.in = *in; a.out = *out; a.rh = rh;
  const dim3 grid((ncol + 255) / 256, nlev);
  hipStream_t s = (hipStream_t)stream;
  if (rh)
    hipLaunchKernelGGL(k_ice_adjust_branches<true>, grid, dim3(256), 0, s, a, branches);
  else
    hipLaunchKernelGGL(k_ice_adjust_branches<false>, grid, dim3(256), 0, s, a, branches);
  HIPCHK(hipGetLastError());
  return ICE3_OK;
}

extern "C" int ice3_rain_ice_branches(ice3_ctx *ctx, int ncol, int nlev, int ld, double dt,
                                      const ice3_rain_ice_in *in, const ice3_rain_ice_inout *io,
                                      const ice3_rain_ice_out *out, const ice3_hail *hail,
                                      unsigned *branches, void *stream) {
  if (!ctx || !in || !io || !out || !branches) return ICE3_EINVAL;
  if (empty_domain(ncol, nlev, ld, dt)) return ICE3_OK;
  if (bad_shape(ncol, nlev, ld, dt) || nlev > 65535) return ICE3_EINVAL;
  NN(in->exn); NN(in->dzz); NN(in->rhodref); NN(in->exn_ref); NN(in->pabs); NN(in->cldfr);
  NN(in->sigs); NN(in->tht); NN(in->rvt); NN(in->rct); NN(in->rrt); NN(in->rit); NN(in->rst);
  NN(in->rgt);
  NN(io->ths); NN(io->rvs); NN(io->rcs); NN(io->rrs); NN(io->ris); NN(io->rss); NN(io->rgs);
  NN(io->ci);
  NN(out->evap3d); NN(out->rainfr); NN(out->inprc); NN(out->inprr); NN(out->inpri);
  NN(out->inprs); NN(out->inprg);
  if (hail) { NN(hail->rht); NN(hail->rhs); NN(hail->inprh); }
  if (!sedim_fits(ctx, nlev)) return ICE3_EINVAL;
  SedimArgs sa;
  MicroArgs m;
  rain_ice_args(ncol, nlev, ld, dt, ctx->d_tab, in, io, out, nullptr, sa, m);
  m.max_calls = ctx->max_calls; m.capped = ctx->d_capped;
  m.branches = branches;
  if (hail) {
    sa.src_rh = hail->rhs; sa.dst_rh = hail->rhs; sa.inprh = hail->inprh;
    m.t[IRH] = hail->rht; m.src[IRH] = hail->rhs; m.dst[IRH] = hail->rhs;
  }
  hipStream_t s = (hipStream_t)stream;
  if (ctx->sedim == ICE3_SEDIM_SPLI)
    HIPCHK(launch_split(ctx, sa, m, s));
  else
    HIPCHK(sedim_launch<double>(sa, ctx->ncu, s));
  const unsigned int npts = (unsigned int)nlev * (unsigned int)ncol;
  if (hail)
    hipLaunchKernelGGL(k_micro_branches<true>, dim3((npts + 255) / 256), dim3(256), 0, s, m);
  else
    hipLaunchKernelGGL(k_micro_branches<false>, dim3((npts + 255) / 256), dim3(256), 0, s, m);
  HIPCHK(hipGetLastError());
  return ICE3_OK;
}

extern "C" int ice3_adjust_rain_ice_hail(ice3_ctx *ctx, int ncol, int nlev, int ld, double dt,
                                         const ice3_pipeline_in *in, const ice3_pipeline_out *out,
                                         const ice3_pipeline_hail *hail, const ice3_stats *stats,
                                         void *stream) {
  if (!ctx || !in || !out || !hail) return ICE3_EINVAL;
  if (empty_domain(ncol, nlev, ld, dt)) return ICE3_OK;
  if (bad_shape(ncol, nlev, ld, dt) || nlev > 65535) return ICE3_EINVAL;
  if (bad_pipeline_ptrs(in, out)) return ICE3_EINVAL;
  NN(hail->rh); NN(hail->rhs); NN(hail->rhs_out); NN(hail->inprh);
  if ((const double *)hail->rhs_out == hail->rhs) return ICE3_EINVAL;
  AdjustArgs aa;
  SedimArgs sa;
  MicroArgs m;
  pipeline_args(ncol, nlev, ld, dt, ctx->d_tab, in, out, stats, aa, sa, m);
  m.max_calls = ctx->max_calls; m.capped = ctx->d_capped;
  aa.rh = hail->rh;
  sa.src_rh = hail->rhs; sa.dst_rh = hail->rhs_out; sa.inprh = hail->inprh;
  m.t[IRH] = hail->rhs; m.src[IRH] = hail->rhs_out; m.dst[IRH] = hail->rhs_out;
  if (!sedim_fits(ctx, nlev)) return ICE3_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  hand_ris_over(aa, sa);
  MARK(0);
  if (ctx->sedim == ICE3_SEDIM_SPLI) {
    hipLaunchKernelGGL(k_ice_adjust_hail, dim3((ncol + 255) / 256, nlev), dim3(256), 0, s, aa);
    HIPCHK(hipGetLastError());
    MARK(1);
    const int rc = launch_split_keep(ctx, nlev, ld, sa, m, s);
    if (rc != ICE3_OK) return rc;
  } else {
    HIPCHK(launch_adjust_sedim(ctx, aa, sa, s));
    MARK(1);
  }
  MARK(2);
  HIPCHK(launch_micro_hail(ctx, m, s));
  MARK(3); MARK(4); MARK(5); MARK(6);
  return ICE3_OK;
}

extern "C" size_t ice3_surrogate_work_bytes(int ncol, int nlev) {
  if (ncol <= 0 || nlev <= 0) return 0;
  return sg_work_layout((size_t)ncol * nlev).total;
}

// Argument checks of the surrogate step (both entry points); ICE3_OK with *empty set when
// there is nothing to do.
static int surrogate_check(const ice3_ctx *ctx, int ncol, int nlev, int ld, double dt,
                           const ice3_pipeline_in *in, const ice3_pipeline_out *out,
                           const ice3_surrogate *sg, const unsigned long long *sg_counters,
                           bool *empty) {
  *empty = false;
  if (!ctx || !in || !out || !sg || !sg_counters) return ICE3_EINVAL;
  if (empty_domain(ncol, nlev, ld, dt)) {  // the work area is then 0 bytes
    *empty = true;
    return ICE3_OK;
  }
  if (bad_shape(ncol, nlev, ld, dt)) return ICE3_EINVAL;
  if (nlev > 65535 || (double)nlev * ncol >= 4.0e9 || (double)nlev * ld >= 4.0e9)
    return ICE3_EINVAL;
  if (!sg->weights_packed || !sg->params || !sg->norm || !(sg->budget_tol >= 0.f) ||
      !(sg->neg_tol >= 0.f))
    return ICE3_EINVAL;
  if (ctx->sedim != ICE3_SEDIM_STAT) return ICE3_EINVAL;  // trained on the statistical scheme
  if (bad_pipeline_ptrs(in, out)) return ICE3_EINVAL;
  return ICE3_OK;
}

// The surrogate step on a checked problem, with the scratch at work (sg_work_layout).
static int surrogate_step(ice3_ctx *ctx, int ncol, int nlev, int ld, double dt,
                          const ice3_pipeline_in *in, const ice3_pipeline_out *out,
                          const ice3_surrogate *sg, void *work,
                          unsigned long long *sg_counters, const ice3_stats *stats,
                          void *stream) {
  AdjustArgs aa;
  SedimArgs sa;
  MicroArgs m;
  pipeline_args(ncol, nlev, ld, dt, ctx->d_tab, in, out, stats, aa, sa, m);
  m.max_calls = ctx->max_calls; m.capped = ctx->d_capped;
  hipStream_t s = (hipStream_t)stream;
  const unsigned int npts = (unsigned int)nlev * (unsigned int)ncol;
  const SgWork wl = sg_work_layout(npts);
  unsigned char *wb = (unsigned char *)work;
  SurrogateArgs g;
  g.m = m;
  g.npts = npts;
  g.norm = sg->norm;
  g.budget_tol = sg->budget_tol;
  g.neg_tol = sg->neg_tol;
  g.wpk = sg->weights_packed;
  g.params = sg->params;
  g.queue = (unsigned int *)(wb + wl.queue);
  g.counters = sg_counters;
  g.qcount = (unsigned int *)(wb + wl.qcount);
  unsigned int nseg = 0;
  hand_ris_over(aa, sa);
  MARK(0);
  HIPCHK(launch_adjust_sedim(ctx, aa, sa, s));
  MARK(1);
  MARK(2);
  MARK(3);
  HIPCHK(surrogate_network_launch(g, ctx->ncu, &nseg, s));
  MARK(4);
  MARK(5);
  hipLaunchKernelGGL(k_micro_segments<double>, dim3(nseg * SG_PARTS), dim3(64), 0, s, m,
                     (const unsigned int *)g.queue, (const unsigned int *)g.qcount, g.seg);
  HIPCHK(hipGetLastError());
  MARK(6);
  return ICE3_OK;
}

extern "C" int ice3_adjust_rain_ice_surrogate(ice3_ctx *ctx, int ncol, int nlev, int ld,
                                              double dt, const ice3_pipeline_in *in,
                                              const ice3_pipeline_out *out,
                                              const ice3_surrogate *sg, void *work,
                                              unsigned long long *sg_counters,
                                              const ice3_stats *stats, void *stream) {
  bool empty;
  const int rc = surrogate_check(ctx, ncol, nlev, ld, dt, in, out, sg, sg_counters, &empty);
  if (rc != ICE3_OK || empty) return rc;
  if (!work || ((uintptr_t)work & 255) != 0) return ICE3_EINVAL;
  return surrogate_step(ctx, ncol, nlev, ld, dt, in, out, sg, work, sg_counters, stats, stream);
}

extern "C" int ice3_adjust_rain_ice_surrogate_noalloc(ice3_ctx *ctx, int ncol, int nlev, int ld,
                                                      double dt, const ice3_pipeline_in *in,
                                                      const ice3_pipeline_out *out,
                                                      const ice3_surrogate *sg,
                                                      unsigned long long *sg_counters,
                                                      const ice3_stats *stats, void *stream) {
  bool empty;
  const int rc = surrogate_check(ctx, ncol, nlev, ld, dt, in, out, sg, sg_counters, &empty);
  if (rc != ICE3_OK || empty) return rc;
  if (sg_work_layout((size_t)ncol * nlev).total > ICE3_SURROGATE_SCRATCH_BYTES) return ICE3_ETOOLARGE;
  return surrogate_step(ctx, ncol, nlev, ld, dt, in, out, sg, ctx->d_scratch, sg_counters, stats,
                        stream);
}

extern "C" int ice3_surrogate_features(ice3_ctx *ctx, int ncol, int nlev, int ld, double dt,
                                       const ice3_pipeline_in *in, const ice3_pipeline_out *out,
                                       const ice3_surrogate_norm *norm, float *raw, void *x,
                                       unsigned char *micro, void *stream) {
  if (!ctx || !in || !out || (x && !norm)) return ICE3_EINVAL;
  if (empty_domain(ncol, nlev, ld, dt)) return ICE3_OK;
  if (bad_shape(ncol, nlev, ld, dt)) return ICE3_EINVAL;
  if ((double)nlev * ncol >= 4.0e9 || bad_pipeline_ptrs(in, out)) return ICE3_EINVAL;
  AdjustArgs aa;
  SedimArgs sa;
  MicroArgs m;
  pipeline_args(ncol, nlev, ld, dt, ctx->d_tab, in, out, nullptr, aa, sa, m);
  const unsigned int npts = (unsigned int)nlev * (unsigned int)ncol;
  hipLaunchKernelGGL(k_features, dim3((npts + 255) / 256), dim3(256), 0, (hipStream_t)stream, m,
                     npts, norm, raw, (__bf16 *)x, micro);
  HIPCHK(hipGetLastError());
  return ICE3_OK;
}
