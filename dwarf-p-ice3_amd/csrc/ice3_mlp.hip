// ice3_mlp.hip -- kernels of the rain_ice surrogate MLP (bf16 matrix cores, fp32
// accumulation): training, with its C ABI (declared in include/ice3.h).
//
//   k_mlp_forward   one 128-point tile per workgroup: 5 layers on v_mfma_f32_16x16x32_bf16
//                   with every weight resident in LDS; saves pre-activations (fp32) and
//                   activations (bf16) for the backward pass; MSE loss and its gradient.
//   k_mlp_backward  one tile per workgroup: dW = H^T dZ and dH = dZ W^T on the matrix
//                   cores, SiLU derivative, bias gradients; one fp32 partial gradient per
//                   workgroup (no atomics: the reduction is deterministic).
//   k_mlp_gradient  both in one kernel, nothing saved between them (the training step).
//   k_mlp_reduce    sum of the partial gradients (and losses).
//   k_mlp_adam      Adam on the fp32 master parameters; rewrites the bf16 row-major and
//                   packed-fragment copies the matrix cores read.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <type_traits>

#include "../../include/ice3.h"
#include "ice3_mlp.hpp"

namespace ice3 {

struct MlpFwdArgs {
  int npts;
  const bf16x8 *wpk;      // packed bf16 weights
  const float *params;    // fp32 master parameters (biases at MLP_NW)
  const __bf16 *x;        // [npts][MLP_IN]
  const float *target;    // [npts][MLP_NTARG] or NULL
  float *y;               // [npts][MLP_NTARG] or NULL
  float *zsave;           // [4][npts][MLP_H] or NULL
  __bf16 *hsave;          // [4][npts][MLP_H] or NULL
  float *dy;              // [npts][MLP_OUT] or NULL
  float *loss_part;       // [gridDim.x] or NULL
  float inv_count;        // 1 / (npts * MLP_NTARG)
};

// bias + activation epilogue of a hidden layer: z -> (save z, h) -> h into sOut
template <int N>
__device__ __forceinline__ void hidden_epilogue(const MlpFwdArgs &a, int l, int p0, int row0,
                                                const f32x4 (&acc)[MLP_MT][N / 16],
                                                const float *sB, __bf16 *sOut, int lane) {
#pragma unroll
  for (int mt = 0; mt < MLP_MT; ++mt)
#pragma unroll
    for (int nn = 0; nn < N / 16; ++nn)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + mt * 16 + 4 * (lane / 16) + i, col = nn * 16 + lane % 16;
        const float z = acc[mt][nn][i] + sB[l * MLP_H + col];
        const __bf16 h = (__bf16)silu(z);
        sOut[row * MLP_HS + col] = h;
        const int p = p0 + row;
        if (a.zsave && p < a.npts) {
          const size_t o = ((size_t)l * a.npts + p) * MLP_H + col;
          a.zsave[o] = z;
          a.hsave[o] = h;
        }
      }
}

__global__ void __launch_bounds__(256) k_mlp_forward(MlpFwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16x8 *sW = (bf16x8 *)smem;                                   // MLP_NW bf16
  float *sB = (float *)(smem + MLP_NW * 2);                      // MLP_NB fp32
  __bf16 *sH = (__bf16 *)(smem + MLP_NW * 2 + MLP_NB * 4);       // [MLP_TILE][MLP_HS]
  __bf16 *sX = sH + MLP_TILE * MLP_HS;                           // [MLP_TILE][MLP_XS]
  __shared__ float sLoss[MLP_WAVES];
  const int lane = threadIdx.x % 64, w = threadIdx.x / 64, row0 = w * MLP_ROWS;
  const int p0 = blockIdx.x * MLP_TILE;
  stage_weights<64 * MLP_WAVES>(sW, sB, a.wpk, a.params);
  // input tile: 4 x 16 bytes per row
  for (int q = threadIdx.x; q < MLP_TILE * 4; q += blockDim.x) {
    const int r = q / 4, c = q % 4, p = p0 + r;
    int4 v = {0, 0, 0, 0};
    if (p < a.npts) v = ((const int4 *)(a.x + (size_t)p * MLP_IN))[c];
    *(int4 *)(sX + r * MLP_XS + c * 8) = v;
  }
  __syncthreads();
  {
    f32x4 acc[MLP_MT][MLP_H / 16];
    mlp_layer<MLP_IN, MLP_H, MLP_XS>(sX, row0, sW + mlp_woff(0) / 8, acc, lane);
    hidden_epilogue<MLP_H>(a, 0, p0, row0, acc, sB, sH, lane);
  }
#pragma unroll 1
  for (int l = 1; l <= 3; ++l) {
    f32x4 acc[MLP_MT][MLP_H / 16];
    mlp_layer<MLP_H, MLP_H, MLP_HS>(sH, row0, sW + mlp_woff(l) / 8, acc, lane);
    hidden_epilogue<MLP_H>(a, l, p0, row0, acc, sB, sH, lane);
  }
  f32x4 acc[MLP_MT][MLP_OUT / 16];
  mlp_layer<MLP_H, MLP_OUT, MLP_HS>(sH, row0, sW + mlp_woff(4) / 8, acc, lane);
  float loss = 0.f;
#pragma unroll
  for (int mt = 0; mt < MLP_MT; ++mt)
#pragma unroll
    for (int nn = 0; nn < MLP_OUT / 16; ++nn)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + mt * 16 + 4 * (lane / 16) + i, col = nn * 16 + lane % 16;
        const int p = p0 + row;
        if (p >= a.npts) continue;
        const float y = acc[mt][nn][i] + sB[4 * MLP_H + col];
        float g = 0.f;
        if (col < MLP_NTARG) {
          if (a.y) a.y[(size_t)p * MLP_NTARG + col] = y;
          if (a.target) {
            const float d = y - a.target[(size_t)p * MLP_NTARG + col];
            loss += d * d;
            g = 2.f * d * a.inv_count;
          }
        }
        if (a.dy) a.dy[(size_t)p * MLP_OUT + col] = g;
      }
  if (a.loss_part) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) loss += __shfl_xor(loss, m, 64);
    if (lane == 0) sLoss[w] = loss;
    __syncthreads();
    if (threadIdx.x == 0) a.loss_part[blockIdx.x] = sLoss[0] + sLoss[1] + sLoss[2] + sLoss[3];
  }
}

constexpr size_t MLP_FWD_LDS = (size_t)MLP_NW * 2 + MLP_NB * 4 + MLP_TILE * MLP_HS * 2 +
                               MLP_TILE * MLP_XS * 2;

struct MlpBwdArgs {
  int npts;
  const __bf16 *wrm;      // row-major bf16 weights
  const __bf16 *x;        // [npts][MLP_IN]
  const float *zsave;     // [4][npts][MLP_H]
  const __bf16 *hsave;    // [4][npts][MLP_H]
  const float *dy;        // [npts][MLP_OUT]
  float *gpart;           // [gridDim.x][MLP_NP]
};

constexpr int BW_S = MLP_H + 8;          // row stride of the backward LDS tiles (bf16)
constexpr int BW_TILE = MLP_H * BW_S;    // elements of one 128 x BW_S tile

// One layer of the backward pass.  On entry sDZ ([point][BW_S], row-major) and sDZT
// ([unit][BW_S], transposed) hold dZ_L in bf16 for the tile; on exit (L > 0) they hold
// dZ_{L-1}.
template <int L>
__device__ __forceinline__ void bwd_layer(const MlpBwdArgs &a, int p0, __bf16 *sW, __bf16 *sDZ,
                                          __bf16 *sDZT, __bf16 *sHT, int lane, int w) {
  constexpr int K = mlp_k(L), N = mlp_n(L);
  float *gp = a.gpart + (size_t)blockIdx.x * MLP_NP;
  // layer input, transposed: sHT[k][p]
  const __bf16 *hin = L == 0 ? a.x : a.hsave + (size_t)(L - 1) * a.npts * MLP_H;
  for (int q = threadIdx.x; q < MLP_TILE * (K / 8); q += blockDim.x) {
    const int r = q / (K / 8), c = q % (K / 8), p = p0 + r;
    bf16x8 v;
    if (p < a.npts) v = *(const bf16x8 *)(hin + (size_t)p * K + c * 8);
    else v = bf16x8{};
#pragma unroll
    for (int i = 0; i < 8; ++i) sHT[(c * 8 + i) * BW_S + r] = v[i];
  }
  if (L > 0)  // W_L row-major: sW[k][n]
    for (int q = threadIdx.x; q < K * (N / 8); q += blockDim.x) {
      const int k = q / (N / 8), c = q % (N / 8);
      *(bf16x8 *)(sW + k * BW_S + c * 8) = *(const bf16x8 *)(a.wrm + mlp_woff(L) + k * N + c * 8);
    }
  __syncthreads();
  // dW_L = H^T dZ (K x N): 16x16 output tiles spread over the waves
  for (int t = w; t < (K / 16) * (N / 16); t += MLP_WAVES) {
    const int m0 = (t / (N / 16)) * 16, n0 = (t % (N / 16)) * 16;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < MLP_TILE / 32; ++kk) {
      const bf16x8 av = *(const bf16x8 *)(sHT + (m0 + lane % 16) * BW_S + kk * 32 + 8 * (lane / 16));
      const bf16x8 bv = *(const bf16x8 *)(sDZT + (n0 + lane % 16) * BW_S + kk * 32 + 8 * (lane / 16));
      acc = mfma_bf16(av, bv, acc);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      gp[mlp_woff(L) + (m0 + 4 * (lane / 16) + i) * N + n0 + lane % 16] = acc[i];
  }
  // bias gradient: column sums of dZ
  for (int n = threadIdx.x; n < N; n += blockDim.x) {
    float s = 0.f;
    for (int p = 0; p < MLP_TILE; ++p) s += (float)sDZT[n * BW_S + p];
    gp[mlp_boff(L) + n] = s;
  }
  if (L == 0) return;
  // dH = dZ W^T (points x K), then dZ_{L-1} = dH * SiLU'(Z_{L-1})
  const int row0 = w * MLP_ROWS;
  f32x4 acc[MLP_MT][K / 16];
#pragma unroll
  for (int mt = 0; mt < MLP_MT; ++mt)
#pragma unroll
    for (int nn = 0; nn < K / 16; ++nn) acc[mt][nn] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < N / 32; ++kk) {
    bf16x8 av[MLP_MT];
#pragma unroll
    for (int mt = 0; mt < MLP_MT; ++mt)
      av[mt] = *(const bf16x8 *)(sDZ + (row0 + mt * 16 + lane % 16) * BW_S + kk * 32 + 8 * (lane / 16));
#pragma unroll
    for (int nn = 0; nn < K / 16; ++nn) {
      const bf16x8 bv = *(const bf16x8 *)(sW + (nn * 16 + lane % 16) * BW_S + kk * 32 + 8 * (lane / 16));
#pragma unroll
      for (int mt = 0; mt < MLP_MT; ++mt) acc[mt][nn] = mfma_bf16(av[mt], bv, acc[mt][nn]);
    }
  }
  const float *zin = a.zsave + (size_t)(L - 1) * a.npts * MLP_H;
#pragma unroll
  for (int mt = 0; mt < MLP_MT; ++mt)
#pragma unroll
    for (int nn = 0; nn < K / 16; ++nn)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + mt * 16 + 4 * (lane / 16) + i, col = nn * 16 + lane % 16;
        const int p = p0 + row;
        acc[mt][nn][i] = p < a.npts ? acc[mt][nn][i] * silu_grad(zin[(size_t)p * MLP_H + col]) : 0.f;
      }
  __syncthreads();  // every wave is done reading sDZ, sDZT, sHT and sW
#pragma unroll
  for (int mt = 0; mt < MLP_MT; ++mt)
#pragma unroll
    for (int nn = 0; nn < K / 16; ++nn)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + mt * 16 + 4 * (lane / 16) + i, col = nn * 16 + lane % 16;
        const __bf16 v = (__bf16)acc[mt][nn][i];
        sDZ[row * BW_S + col] = v;
        sDZT[col * BW_S + row] = v;
      }
  __syncthreads();
}

__global__ void __launch_bounds__(256) k_mlp_backward(MlpBwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __bf16 *sW = (__bf16 *)smem;
  __bf16 *sDZ = sW + BW_TILE;
  __bf16 *sDZT = sDZ + BW_TILE;
  __bf16 *sHT = sDZT + BW_TILE;
  const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
  const int p0 = blockIdx.x * MLP_TILE;
  // dZ_4 = dY (the output layer is linear)
  for (int q = threadIdx.x; q < MLP_TILE * MLP_OUT; q += blockDim.x) {
    const int r = q / MLP_OUT, c = q % MLP_OUT, p = p0 + r;
    const __bf16 v = (__bf16)(p < a.npts ? a.dy[(size_t)p * MLP_OUT + c] : 0.f);
    sDZ[r * BW_S + c] = v;
    sDZT[c * BW_S + r] = v;
  }
  __syncthreads();
  bwd_layer<4>(a, p0, sW, sDZ, sDZT, sHT, lane, w);
  bwd_layer<3>(a, p0, sW, sDZ, sDZT, sHT, lane, w);
  bwd_layer<2>(a, p0, sW, sDZ, sDZT, sHT, lane, w);
  bwd_layer<1>(a, p0, sW, sDZ, sDZT, sHT, lane, w);
  bwd_layer<0>(a, p0, sW, sDZ, sDZT, sHT, lane, w);
}

constexpr size_t MLP_BWD_LDS = (size_t)4 * BW_TILE * 2;

// ---- Forward and backward in one kernel, nothing saved to memory between them.
// A workgroup takes a tile of 128 points, a wavefront 16 of them through every layer, activations
// in registers as in k_sg_network, the pre-activations of the four hidden layers beside them
// (fp32, 128 of 256 registers; the sigmoid is computed a second time rather than kept).  For
// dW = H^T dZ the points are the contraction, so H and dZ of a layer go through LDS transposed;
// dH = W dZ takes dZ from registers.  The backward tiles lie where the forward weights were, the
// weights of a layer one layer ahead of their use.
// 32,768 points (a tile for each compute unit): 43 us a call among calls, 37 and, of the reduction, 10
// as a profiler times the kernels one by one; 208 us of k_mlp_forward (34, with 100 MB of
// pre-activations and activations saved), k_mlp_backward (112) and a serial sum of the partials
// (62).  Bound by the latency of its ten phases between
// barriers at two wavefronts a SIMD, and the 59 MB of partials written and read.
struct MlpGradArgs {
  int npts;
  const bf16x8 *wpk;      // packed bf16 weights
  const __bf16 *wrm;      // row-major bf16 weights
  const float *params;    // fp32 master parameters (biases at MLP_NW)
  const __bf16 *x;        // [npts][MLP_IN]
  const float *target;    // [npts][MLP_NTARG]
  float *gpart;           // [gridDim.x][MLP_NP]
  float *loss_part;       // [gridDim.x]
  float inv_count;        // 1 / (npts * MLP_NTARG)
};

constexpr int GRAD_WAVES = MLP_TILE / 16, GRAD_THREADS = 64 * GRAD_WAVES;

// v: bf16 units u0 .. u0+3 of point col (one point a lane, neighbouring lanes neighbouring points)
// into the transposed tile s[unit][BW_S]; an even lane writes the pairs of the first two units,
// an odd one those of the last two, every bank once.
__device__ __forceinline__ void put_transposed(__bf16 *s, int u0, int col, const u32x2 &v) {
  const bool odd = col & 1;
  const unsigned int own = odd ? v[1] : v[0], send = odd ? v[0] : v[1];
  const unsigned int got = __builtin_amdgcn_update_dpp(0u, send, 0xB1, 0xF, 0xF, true);  // lane ^ 1
  const unsigned int lo = odd ? got : own, hi = odd ? own : got;
  __bf16 *d = s + (u0 + (odd ? 2 : 0)) * BW_S + (col & ~1);
  *(unsigned int *)d = (lo & 0xFFFFu) | (hi << 16);
  *(unsigned int *)(d + BW_S) = (lo >> 16) | (hi & 0xFFFF0000u);
}

// W_L (row-major) to registers, and from there into its padded tile.
template <int L> struct StagedW {
  static constexpr int N = mlp_n(L), NQ = MLP_H * (N / 8) / GRAD_THREADS;
  bf16x8 v[NQ];
  __device__ __forceinline__ void load(const __bf16 *wrm) {
#pragma unroll
    for (int b = 0; b < NQ; ++b)
      v[b] = *(const bf16x8 *)(wrm + mlp_woff(L) + (threadIdx.x + b * GRAD_THREADS) * 8);
  }
  __device__ __forceinline__ void store(__bf16 *sW) const {
#pragma unroll
    for (int b = 0; b < NQ; ++b) {
      const int q = threadIdx.x + b * GRAD_THREADS;
      *(bf16x8 *)(sW + (q / (N / 8)) * BW_S + (q % (N / 8)) * 8) = v[b];
    }
  }
};

// dW_L = H^T dZ and the bias gradient of a tile, to its partial: wavefront w's NT x KT output
// tiles of 16 units of layer L by 16 of its input, from the transposed tiles.
template <int L, int NT, int KT>
__device__ __forceinline__ void grad_weights(float *gp, const __bf16 *sDZT, const __bf16 *sHT,
                                             int n0, int k0, bool bias, int lane) {
  constexpr int N = mlp_n(L);
  const int pt = lane % 16, g = lane / 16;
  f32x4 acc[NT][KT], sum[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    sum[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KT; ++k) acc[n][k] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  bf16x8 ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = (__bf16)1.f;
#pragma unroll
  for (int kk = 0; kk < MLP_TILE / 32; ++kk) {
    bf16x8 dz[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      dz[n] = *(const bf16x8 *)(sDZT + (n0 + n * 16 + pt) * BW_S + kk * 32 + 8 * g);
      if (bias) sum[n] = mfma_bf16(dz[n], ones, sum[n]);
    }
#pragma unroll
    for (int k = 0; k < KT; ++k) {
      const bf16x8 h = *(const bf16x8 *)(sHT + (k0 + k * 16 + pt) * BW_S + kk * 32 + 8 * g);
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[n][k] = mfma_bf16(dz[n], h, acc[n][k]);
    }
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) {
#pragma unroll
    for (int k = 0; k < KT; ++k)
      *(f32x4 *)(gp + mlp_woff(L) + (k0 + k * 16 + pt) * N + n0 + n * 16 + 4 * g) = acc[n][k];
    if (bias && pt == 0) *(f32x4 *)(gp + mlp_boff(L) + n0 + n * 16 + 4 * g) = sum[n];
  }
}

__global__ void __launch_bounds__(GRAD_THREADS) k_mlp_gradient(MlpGradArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16x8 *sWF = (bf16x8 *)smem;                   // forward: every layer's packed weights
  __bf16 *sHT = (__bf16 *)smem;                   // backward, in their place: H^T,
  __bf16 *sW0 = sHT + BW_TILE, *sW1 = sW0 + BW_TILE;  // and the weights of two layers
  float *sB = (float *)(smem + MLP_NW * 2);       // biases
  __bf16 *sDZT = (__bf16 *)(sB + MLP_NB);         // dZ^T
  __shared__ float sLoss[GRAD_WAVES];
  const int lane = threadIdx.x % 64, w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int pt = lane % 16, g = lane / 16;
  const int col = w * 16 + pt, p = blockIdx.x * MLP_TILE + col;  // this lane's point
  const bool live = p < a.npts;
  float *gp = a.gpart + (size_t)blockIdx.x * MLP_NP;
  bf16x8 x0[1][1];
  if (live) x0[0][0] = *(const bf16x8 *)(a.x + (size_t)p * MLP_IN + 8 * g);
  else x0[0][0] = bf16x8{};
  float t[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    t[i] = live && 4 * g < MLP_NTARG ? a.target[(size_t)p * MLP_NTARG + 4 * g + i] : 0.f;
  stage_weights<GRAD_THREADS>(sWF, sB, a.wpk, a.params);
  __syncthreads();

  // forward
  f32x4 z[4][MLP_H / 16];
  u32x2 dz[MLP_H / 16];   // dZ of a layer, bf16, units 16 nn + 4 g .. +3
  {
    bf16x8 h[1][MLP_H / 32];
    f32x4 acc[1][MLP_H / 16];
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      if (l == 0) mlp_product<MLP_IN, MLP_H, MLP_H / 16, 1>(sWF, x0, acc, lane);
      else mlp_product<MLP_H, MLP_H, MLP_H / 16, 1>(sWF + mlp_woff(l) / 8, h, acc, lane);
      u32x2 v[MLP_H / 16];
#pragma unroll
      for (int nn = 0; nn < MLP_H / 16; ++nn) {
        z[l][nn] = acc[0][nn] + *(const f32x4 *)(sB + l * MLP_H + nn * 16 + 4 * g);
        v[nn] = pack4(silu(z[l][nn][0]), silu(z[l][nn][1]), silu(z[l][nn][2]), silu(z[l][nn][3]));
        // opaque to the compiler, which would keep this sigmoid for the backward part (128 registers)
#pragma unroll
        for (int i = 0; i < 4; ++i) asm("" : "+v"(z[l][nn][i]));
      }
#pragma unroll
      for (int kk = 0; kk < MLP_H / 32; ++kk) h[0][kk] = operand_of(v[2 * kk], v[2 * kk + 1]);
    }
    f32x4 out[1][1];  // the first 16 of the padded outputs
    mlp_product<MLP_H, 16, MLP_OUT / 16, 1>(sWF + mlp_woff(4) / 8, h, out, lane);
    const f32x4 b = *(const f32x4 *)(sB + 4 * MLP_H + 4 * g);
    float loss = 0.f, dy[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float d = out[0][0][i] + b[i] - t[i];
      const bool used = live && 4 * g < MLP_NTARG;
      loss += used ? d * d : 0.f;
      dy[i] = used ? 2.f * d * a.inv_count : 0.f;
    }
    dz[0] = pack4(dy[0], dy[1], dy[2], dy[3]);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) loss += __shfl_xor(loss, m, 64);
    if (lane == 0) sLoss[w] = loss;
  }

  // backward: from the layer above's dZ (registers) and its weights, dZ of layer l
  auto dz_below = [&](auto LC, const __bf16 *sW) {
    constexpr int L = decltype(LC)::value, N = mlp_n(L);  // through W_L to layer L - 1
    bf16x8 d[N / 32];
#pragma unroll
    for (int kk = 0; kk < N / 32; ++kk)
      d[kk] = operand_of(dz[2 * kk], L == MLP_LAYERS - 1 ? u32x2{0u, 0u} : dz[2 * kk + 1]);
    f32x4 acc[MLP_H / 16];
#pragma unroll
    for (int nn = 0; nn < MLP_H / 16; ++nn) acc[nn] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < N / 32; ++kk)
#pragma unroll
      for (int nn = 0; nn < MLP_H / 16; ++nn)
        acc[nn] = mfma_bf16(*(const bf16x8 *)(sW + (nn * 16 + pt) * BW_S + kk * 32 + 8 * g), d[kk], acc[nn]);
#pragma unroll
    for (int nn = 0; nn < MLP_H / 16; ++nn) {
      f32x4 v;  // z[L - 1] holds silu'(z) by now
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = live ? acc[nn][i] * z[L - 1][nn][i] : 0.f;
      dz[nn] = pack4(v[0], v[1], v[2], v[3]);
    }
  };
  auto put_dz = [&] {
#pragma unroll
    for (int nn = 0; nn < MLP_H / 16; ++nn) put_transposed(sDZT, nn * 16 + 4 * g, col, dz[nn]);
  };
  auto put_h = [&](f32x4 (&zl)[MLP_H / 16]) {  // H^T of a layer; its z becomes silu'(z)
#pragma unroll
    for (int nn = 0; nn < MLP_H / 16; ++nn) {
      f32x4 h;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = zl[nn][i], s = sigmoid_fast(v);
        h[i] = live ? v * s : 0.f;
        zl[nn][i] = s * (1.f + v * (1.f - s));
      }
      put_transposed(sHT, nn * 16 + 4 * g, col, pack4(h[0], h[1], h[2], h[3]));
    }
  };
  const int n2 = (w % 4) * 32, k4 = (w / 4) * 64;  // this wavefront's 2 x 4 tiles of a hidden layer
  StagedW<4> w4;
  StagedW<3> w3;
  w4.load(a.wrm);
  w3.load(a.wrm);
  __syncthreads();  // the forward weights are read
  if (threadIdx.x == 0) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < GRAD_WAVES; ++i) s += sLoss[i];
    a.loss_part[blockIdx.x] = s;
  }
  w4.store(sW0);
  w3.store(sW1);
  put_h(z[3]);
  put_transposed(sDZT, 4 * g, col, dz[0]);
  __syncthreads();
  // the outputs: 16 of 32 columns, the others' gradients are zero
  grad_weights<4, 1, 1>(gp, sDZT, sHT, 0, w * 16, w == 0, lane);
  *(f32x4 *)(gp + mlp_woff(4) + (w * 16 + pt) * MLP_OUT + 16 + 4 * g) = f32x4{0.f, 0.f, 0.f, 0.f};
  if (threadIdx.x < 16) gp[mlp_boff(4) + 16 + threadIdx.x] = 0.f;
  StagedW<2> w2;
  w2.load(a.wrm);
  dz_below(std::integral_constant<int, 4>{}, sW0);
  __syncthreads();
  put_dz();
  put_h(z[2]);
  w2.store(sW0);
  __syncthreads();
  grad_weights<3, 2, 4>(gp, sDZT, sHT, n2, k4, k4 == 0, lane);
  StagedW<1> w1;
  w1.load(a.wrm);
  dz_below(std::integral_constant<int, 3>{}, sW1);
  __syncthreads();
  put_dz();
  put_h(z[1]);
  w1.store(sW1);
  __syncthreads();
  grad_weights<2, 2, 4>(gp, sDZT, sHT, n2, k4, k4 == 0, lane);
  dz_below(std::integral_constant<int, 2>{}, sW0);
  __syncthreads();
  put_dz();
  put_h(z[0]);
  __syncthreads();
  grad_weights<1, 2, 4>(gp, sDZT, sHT, n2, k4, k4 == 0, lane);
  dz_below(std::integral_constant<int, 1>{}, sW1);
  __syncthreads();
  put_dz();
  const u32x4 xf = __builtin_bit_cast(u32x4, x0[0][0]);
  put_transposed(sHT, 8 * g, col, u32x2{xf[0], xf[1]});
  put_transposed(sHT, 8 * g + 4, col, u32x2{xf[2], xf[3]});
  __syncthreads();
  grad_weights<0, 1, 2>(gp, sDZT, sHT, w * 16, 0, true, lane);
}

constexpr size_t MLP_GRAD_LDS = (size_t)MLP_NW * 2 + MLP_NB * 4 + BW_TILE * 2;
static_assert(3 * BW_TILE * 2 <= MLP_NW * 2, "the backward tiles take the forward weights' place");
static_assert(MLP_GRAD_LDS + GRAD_WAVES * 4 <= 160 * 1024, "k_mlp_gradient LDS");

constexpr int RED_WAVES = 16;

// grad = sum of the tiles' partials; a last block (loss given) sums the tiles' losses.  A workgroup
// sums 64 parameters, each wavefront every RED_WAVES-th tile, in an order that depends on
// the number of tiles alone.  256 tiles: 9.6 us, 6.2 TB/s; 62 us with one thread a parameter, a
// chain of 256 loads.
__global__ void __launch_bounds__(64 * RED_WAVES) k_mlp_reduce(const float *__restrict__ gpart, int nblk,
                                                             float *__restrict__ grad,
                                                             const float *__restrict__ loss_part,
                                                             float *__restrict__ loss) {
  __shared__ float part[RED_WAVES][64];
  const int lane = threadIdx.x % 64, w = threadIdx.x / 64, e = blockIdx.x * 64 + lane;
  const bool last = blockIdx.x * 64 >= MLP_NP;  // uniform
  float s = 0.f;
  if (last) {
    for (int b = threadIdx.x; b < nblk; b += 64 * RED_WAVES) s += loss_part[b];
  } else if (e < MLP_NP) {
#pragma unroll 8
    for (int b = w; b < nblk; b += RED_WAVES) s += gpart[(size_t)b * MLP_NP + e];
  }
  part[w][lane] = s;
  __syncthreads();
  if (w) return;
#pragma unroll
  for (int i = 1; i < RED_WAVES; ++i) s += part[i][lane];
  if (last) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
    if (lane == 0) *loss = s;
  } else if (e < MLP_NP) {
    grad[e] = s;
  }
}

// Layer, row and column of weight element e (row-major per layer).
__device__ __forceinline__ void weight_coords(int e, int &l, int &k, int &n) {
  l = 0;
#pragma unroll
  for (int q = 1; q < MLP_LAYERS; ++q)
    if (e >= mlp_woff(q)) l = q;
  const int r = e - mlp_woff(l);
  k = r / mlp_n(l);
  n = r % mlp_n(l);
}

__global__ void __launch_bounds__(256) k_mlp_adam(int step, float lr, float b1, float b2, float eps,
                                                  float *params, float *m, float *v,
                                                  const float *grad, __bf16 *wrm, __bf16 *wpk) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= MLP_NP) return;
  float p = params[e];
  if (grad) {
    const float g = grad[e];
    const float mm = b1 * m[e] + (1.f - b1) * g;
    const float vv = b2 * v[e] + (1.f - b2) * g * g;
    m[e] = mm;
    v[e] = vv;
    const float mh = mm / (1.f - __powf(b1, (float)step));
    const float vh = vv / (1.f - __powf(b2, (float)step));
    p -= lr * mh / (sqrtf(vh) + eps);
    params[e] = p;
  }
  if (e < MLP_NW) {
    int l, k, n;
    weight_coords(e, l, k, n);
    const __bf16 b = (__bf16)p;
    wrm[e] = b;
    wpk[mlp_pack_index(l, k, n)] = b;
  }
}

}  // namespace ice3

using namespace ice3;

#define HIPCHK(x)                                 \
  do {                                            \
    if ((x) != hipSuccess) return ICE3_EDEVICE;   \
  } while (0)

extern "C" int ice3_mlp_forward(int npts, const void *wpk, const float *params, const void *x,
                                const float *target, float *y, float *zsave, void *hsave,
                                float *dy, float *loss_part, void *stream) {
  if (npts <= 0 || !wpk || !params || !x) return ICE3_EINVAL;
  if ((zsave == nullptr) != (hsave == nullptr) || (zsave && !dy) || (loss_part && !target))
    return ICE3_EINVAL;
  MlpFwdArgs a;
  a.npts = npts; a.wpk = (const bf16x8 *)wpk; a.params = params; a.x = (const __bf16 *)x;
  a.target = target; a.y = y; a.zsave = zsave; a.hsave = (__bf16 *)hsave; a.dy = dy;
  a.loss_part = loss_part; a.inv_count = 1.f / ((float)npts * MLP_NTARG);
  const int nblk = (npts + MLP_TILE - 1) / MLP_TILE;
  hipLaunchKernelGGL(k_mlp_forward, dim3(nblk), dim3(256), MLP_FWD_LDS, (hipStream_t)stream, a);
  HIPCHK(hipGetLastError());
  return ICE3_OK;
}

extern "C" int ice3_mlp_backward(int npts, const void *wrm, const void *x, const float *zsave,
                                 const void *hsave, const float *dy, float *gpart, float *grad,
                                 void *stream) {
  if (npts <= 0 || !wrm || !x || !zsave || !hsave || !dy || !gpart || !grad) return ICE3_EINVAL;
  MlpBwdArgs a;
  a.npts = npts; a.wrm = (const __bf16 *)wrm; a.x = (const __bf16 *)x; a.zsave = zsave;
  a.hsave = (const __bf16 *)hsave; a.dy = dy; a.gpart = gpart;
  const int nblk = (npts + MLP_TILE - 1) / MLP_TILE;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_mlp_backward, dim3(nblk), dim3(256), MLP_BWD_LDS, s, a);
  HIPCHK(hipGetLastError());
  hipLaunchKernelGGL(k_mlp_reduce, dim3((MLP_NP + 63) / 64), dim3(64 * RED_WAVES), 0, s,
                     (const float *)gpart, nblk, grad, (const float *)nullptr, (float *)nullptr);
  HIPCHK(hipGetLastError());
  return ICE3_OK;
}

extern "C" int ice3_mlp_gradient(int npts, const void *wpk, const void *wrm, const float *params,
                                 const void *x, const float *target, float *gpart,
                                 float *loss_part, float *grad, float *loss, void *stream) {
  if (npts <= 0 || !wpk || !wrm || !params || !x || !target || !gpart || !loss_part || !grad || !loss)
    return ICE3_EINVAL;
  if ((uintptr_t)gpart % 16 != 0) return ICE3_EINVAL;  // stored by 16 bytes
  MlpGradArgs a;
  a.npts = npts; a.wpk = (const bf16x8 *)wpk; a.wrm = (const __bf16 *)wrm; a.params = params;
  a.x = (const __bf16 *)x; a.target = target; a.gpart = gpart; a.loss_part = loss_part;
  a.inv_count = 1.f / ((float)npts * MLP_NTARG);
  const int nblk = (npts - 1) / MLP_TILE + 1;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_mlp_gradient, dim3(nblk), dim3(GRAD_THREADS), MLP_GRAD_LDS, s, a);
  HIPCHK(hipGetLastError());
  hipLaunchKernelGGL(k_mlp_reduce, dim3((MLP_NP + 63) / 64 + 1), dim3(64 * RED_WAVES), 0, s,
                     (const float *)gpart, nblk, grad, (const float *)loss_part, loss);
  HIPCHK(hipGetLastError());
  return ICE3_OK;
}

extern "C" int ice3_mlp_adam(int step, float lr, float beta1, float beta2, float eps,
                             float *params, float *m, float *v, const float *grad, void *wrm,
                             void *wpk, void *stream) {
  if (!params || !wrm || !wpk || (grad && (!m || !v || step < 1))) return ICE3_EINVAL;
  hipLaunchKernelGGL(k_mlp_adam, dim3((MLP_NP + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                     step, lr, beta1, beta2, eps, params, m, v, grad, (__bf16 *)wrm,
                     (__bf16 *)wpk);
  HIPCHK(hipGetLastError());
  return ICE3_OK;
}

extern "C" int ice3_mlp_sizes(int *n_params, int *n_weights, int *tile, int *in_width,
                              int *out_width) {
  if (n_params) *n_params = MLP_NP;
  if (n_weights) *n_weights = MLP_NW;
  if (tile) *tile = MLP_TILE;
  if (in_width) *in_width = MLP_IN;
  if (out_width) *out_width = MLP_OUT;
  return ICE3_OK;
}
