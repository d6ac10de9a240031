// ice3_surrogate.hip -- the network stage of the surrogate step.
#include <hip/hip_runtime.h>

#include "ice3_mlp.hpp"
#include "ice3_surrogate.hpp"

namespace ice3 {

// Reasons a point is not taken from the network.
enum { SG_OK = 0, SG_RANGE = 1, SG_NEG = 2, SG_BUDGET = 3, SG_NOMICRO = 4 };

// The network's inputs of a point (bf16, the padding beyond 24 left out; zeros where it does not
// ask the network) and its reason so far.
__device__ __forceinline__ int sg_features(const SurrogateArgs &a, const ice3_surrogate_norm &nm,
                                           size_t j, bf16x8 (&x)[3]) {
  float f[MLP_NFEAT];
  const bool micro = surrogate_features(a.m, j, f);
  bool in = true;
#pragma unroll
  for (int c = 0; c < MLP_NFEAT; ++c) in &= (f[c] >= nm.feat_lo[c]) & (f[c] <= nm.feat_hi[c]);
  const int flag = !micro ? SG_NOMICRO : in ? SG_OK : SG_RANGE;
#pragma unroll
  for (int c = 0; c < 24; ++c)
    x[c / 8][c % 8] = c < MLP_NFEAT ? (__bf16)((f[c] - nm.feat_mean[c]) * nm.feat_scale[c]) : (__bf16)0.f;
  if (flag != SG_OK)
#pragma unroll
    for (int b = 0; b < 3; ++b) x[b] = bf16x8{};
  return flag;
}

// Decode, physical checks, and the results of a point that passes them.
__device__ __forceinline__ int sg_decode_point(const SurrogateArgs &a, const ice3_surrogate_norm &nm,
                                               size_t j, const float *yq) {
  const MicroArgs &m = a.m;
  double out[7], y[7], rsum = 0., rmag = 0.;
#pragma unroll
  for (int v = 0; v < 7; ++v) {
    y[v] = (double)(nm.targ_unit[v] * sinhf(nm.targ_mean[v] + nm.targ_std[v] * yq[v]));
    out[v] = m.src[v][j] + y[v];
    if (v >= 1) { rsum += y[v]; rmag += fabs(y[v]); }
  }
  // water residual against the predicted changes, with a floor of budget_tol times the
  // smallest typical change (median |change| of the training targets)
  double umin = nm.targ_unit[IRV];
#pragma unroll
  for (int v = IRC; v <= IRG; ++v) umin = fmin(umin, (double)nm.targ_unit[v]);
  if (!(fabs(rsum) <= (double)a.budget_tol * (rmag + umin))) return SG_BUDGET;
  out[IRV] -= rsum;  // move the water residual into vapour
  // a source may go negative by neg_tol of (its value + its change + the typical change)
#pragma unroll
  for (int v = IRC; v <= IRG; ++v)
    if (!(out[v] >= -(double)a.neg_tol * (fabs(m.src[v][j]) + fabs(y[v]) + (double)nm.targ_unit[v])))
      return SG_NEG;
  double lvfact, lsfact;
  latent_factors(m, j, lvfact, lsfact);
  correct_negativities(out[ITH], out[IRV], out[IRC], out[IRR], out[IRI], out[IRS], out[IRG],
                       lvfact, lsfact);
  if (!(out[IRV] >= 0.)) return SG_NEG;
  const double cinew =
      fmax(0., m.src_ci[j] + (double)(nm.targ_unit[7] * sinhf(nm.targ_mean[7] + nm.targ_std[7] * yq[7])));
#pragma unroll
  for (int v = 0; v < 7; ++v) m.dst[v][j] = out[v];
  m.ci[j] = cinew;
  m.evap3d[j] = 0.;
  m.rainfr[j] = 1.;
  if (m.calls) m.calls[j] = 0;
  return SG_OK;
}

// ---- k_sg_network: features, range check, network, decode and checks of every point, and the
// queue of those left to the FP64 microphysics.  Persistent grid, one workgroup a compute unit,
// all weights resident in LDS; the wavefronts of a workgroup take its 64-point chunks in turn as
// they come free, a lane a point for features and decode, 32 points at a time through the
// network with their activations in registers, and no barrier between the weights' arrival and
// the final counts.  The network's inputs and outputs (96 bytes a point, written and read)
// never leave LDS.
// Bound by the VALU: of the 36,000 cycles a chunk issues for, the SiLUs take 25,000 (two
// quarter-rate transcendentals, four other operations and half a conversion, 50 cycles a
// wavefront of activations), sinhf of the outputs 3,700 and asinhf of the inputs 2,400.
// 512 x 512 x 90 points take 5.03 ms; three kernels, features 1.01, network 4.24 and decode 1.36
// ms, the first and last of them at the memory's rate, 6.61.  Three wavefronts a SIMD, so that one's
// matrix products and loads run beside the others' SiLUs; a SIMD favours its oldest wavefront, and
// with a fixed share of the chunks each the others ran on alone at the end: 5.83 ms (two
// wavefronts a SIMD 6.13; the ranges and scales read from memory with a branch a feature 6.00).
constexpr int SGN_WAVES = 12, SGN_MT = 2, SGN_PTS = 16 * SGN_MT;
// A point's row in LDS (48 bytes: no bank conflicts): its inputs, bf16, then in their place its
// outputs, fp32.
constexpr int SGN_XROW = 24, SGN_YROW = SGN_XROW / 2;
constexpr size_t SGN_WAVE_LDS = 64 * SGN_XROW * 2;
constexpr size_t SGN_LDS = (size_t)MLP_NW * 2 + MLP_NB * 4 + SGN_WAVES * SGN_WAVE_LDS;
static_assert(SGN_LDS + sizeof(ice3_surrogate_norm) + SGN_WAVES * 20 + 32 <= 160 * 1024, "k_sg_network LDS");
static_assert(MLP_NFEAT <= SGN_XROW && MLP_NTARG <= SGN_YROW, "k_sg_network layout");

__global__ void __launch_bounds__(64 * SGN_WAVES) k_sg_network(SurrogateArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ __attribute__((aligned(16))) ice3_surrogate_norm nm;  // read by every point
  __shared__ unsigned int sCnt[SGN_WAVES][5];
  __shared__ unsigned int sNext, sQueued;  // the next of the workgroup's chunks, points rejected
  if (threadIdx.x == 0) {
    sNext = SGN_WAVES;
    sQueued = 0;
  }
  bf16x8 *sW = (bf16x8 *)smem;
  float *sB = (float *)(smem + MLP_NW * 2);
  const int lane = threadIdx.x % 64, w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int pt = lane % 16, g = lane / 16;  // this lane's point of a tile, and its quarter of the units
  __bf16 *sX = (__bf16 *)(smem + MLP_NW * 2 + MLP_NB * 4 + w * SGN_WAVE_LDS);  // [64][SGN_XROW]
  float *sY = (float *)sX;                                                     // [64][SGN_YROW]
  stage_weights<64 * SGN_WAVES>(sW, sB, (const bf16x8 *)a.wpk, a.params);
  if (threadIdx.x < sizeof(nm) / 4) ((float *)&nm)[threadIdx.x] = ((const float *)a.norm)[threadIdx.x];
  __syncthreads();
  const unsigned int nchunk = (a.npts + 63) / 64;
  unsigned int *queue = a.queue + (size_t)blockIdx.x * a.seg;
  unsigned int cnt[5] = {0, 0, 0, 0, 0};
  for (unsigned int n = w;; n = __builtin_amdgcn_readfirstlane(lane == 0 ? atomicAdd(&sNext, 1u) : 0u)) {
    const unsigned int c = n * gridDim.x + blockIdx.x;
    if (c >= nchunk) break;
    const unsigned int q = c * 64 + lane;
    int flag = -1;
    size_t j = 0;
    {
      bf16x8 x[3] = {bf16x8{}, bf16x8{}, bf16x8{}};
      if (q < a.npts) {
        j = point_offset(a.m, q);
        flag = sg_features(a, nm, j, x);
      }
#pragma unroll
      for (int b = 0; b < 3; ++b) *(bf16x8 *)(sX + lane * SGN_XROW + b * 8) = x[b];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // rows are read across lanes
#pragma unroll 1
    for (int half = 0; half < 64 / SGN_PTS; ++half) {
      f32x4 acc[SGN_MT][MLP_H / 16];
      bf16x8 x0[SGN_MT][1], h[SGN_MT][MLP_H / 32];
#pragma unroll
      for (int mt = 0; mt < SGN_MT; ++mt) {
        x0[mt][0] = bf16x8{};  // the last quarter of the padded inputs
        if (g < 3) x0[mt][0] = *(const bf16x8 *)(sX + (half * SGN_PTS + mt * 16 + pt) * SGN_XROW + 8 * g);
      }
      auto epilogue = [&](int l) {  // bias, SiLU, and the next layer's operands
#pragma unroll
        for (int kk = 0; kk < MLP_H / 32; ++kk) {
          const f32x4 b0 = *(const f32x4 *)(sB + l * MLP_H + kk * 32 + 4 * g);
          const f32x4 b1 = *(const f32x4 *)(sB + l * MLP_H + kk * 32 + 16 + 4 * g);
#pragma unroll
          for (int mt = 0; mt < SGN_MT; ++mt) {
            float v0[4], v1[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              v0[i] = silu(acc[mt][2 * kk][i] + b0[i]);
              v1[i] = silu(acc[mt][2 * kk + 1][i] + b1[i]);
            }
            h[mt][kk] = operand_of(pack4(v0[0], v0[1], v0[2], v0[3]), pack4(v1[0], v1[1], v1[2], v1[3]));
          }
        }
      };
      mlp_product<MLP_IN, MLP_H, MLP_H / 16, SGN_MT>(sW + mlp_woff(0) / 8, x0, acc, lane);
      epilogue(0);
#pragma unroll 1
      for (int l = 1; l <= 3; ++l) {
        mlp_product<MLP_H, MLP_H, MLP_H / 16, SGN_MT>(sW + mlp_woff(l) / 8, h, acc, lane);
        epilogue(l);
      }
      f32x4 out[SGN_MT][1];  // the first 16 of the padded outputs
      mlp_product<MLP_H, 16, MLP_OUT / 16, SGN_MT>(sW + mlp_woff(4) / 8, h, out, lane);
      const f32x4 b = *(const f32x4 *)(sB + 4 * MLP_H + 4 * g);
      if (4 * g < MLP_NTARG)
#pragma unroll
        for (int mt = 0; mt < SGN_MT; ++mt)
          *(f32x4 *)(sY + (half * SGN_PTS + mt * 16 + pt) * SGN_YROW + 4 * g) = out[mt][0] + b;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (flag == SG_OK) {
      float y[MLP_NTARG];
#pragma unroll
      for (int v = 0; v < MLP_NTARG; ++v) y[v] = sY[lane * SGN_YROW + v];
      flag = sg_decode_point(a, nm, j, y);
    }
#pragma unroll
    for (int r = 0; r < 5; ++r) cnt[r] += __popcll(__ballot(flag == r));
    const unsigned long long rej = __ballot(flag > SG_OK);
    if (rej != 0) {  // uniform
      const unsigned int at = __builtin_amdgcn_readfirstlane(
          lane == 0 ? atomicAdd(&sQueued, (unsigned int)__popcll(rej)) : 0u);
      if (flag > SG_OK) queue[at + __popcll(rej & ((1ull << lane) - 1ull))] = (unsigned int)j;
    }
  }
  // the counts, summed over the workgroup first: additions to one address follow one another
  if (lane == 0)
#pragma unroll
    for (int r = 0; r < 5; ++r) sCnt[w][r] = cnt[r];
  __syncthreads();
  if (threadIdx.x == 64) a.qcount[blockIdx.x] = sQueued;
  if (threadIdx.x < 5) {
    unsigned int n = 0;
#pragma unroll
    for (int i = 0; i < SGN_WAVES; ++i) n += sCnt[i][threadIdx.x];
    if (n) atomicAdd(&a.counters[threadIdx.x], (unsigned long long)n);
  }
}

hipError_t surrogate_network_launch(SurrogateArgs &a, int ncu, unsigned int *nseg, hipStream_t s) {
  const unsigned int nchunk = (a.npts + 63) / 64;
  unsigned int nblk = SG_BLOCKS;
  if (nblk > (unsigned int)ncu) nblk = ncu;
  if (nblk > nchunk) nblk = nchunk;
  *nseg = nblk;
  a.seg = (nchunk + nblk - 1) / nblk * 64;
  hipLaunchKernelGGL(k_sg_network, dim3(nblk), dim3(64 * SGN_WAVES), SGN_LDS, s, a);
  return hipGetLastError();
}

}  // namespace ice3
