// ice3_mlp.hpp -- the per-point MLP of the rain_ice surrogate on CDNA4 matrix cores.
//
// Network: 18 features (padded to MLP_IN = 32) -> 4 hidden layers of 128 units with
// SiLU -> 8 outputs (padded to MLP_OUT = 32).  Weights are bf16 on the matrix cores
// with fp32 accumulation (v_mfma_f32_16x16x32_bf16); master weights, biases and the
// optimiser state are fp32.
//
// Layer l multiplies a (points x K_l) activation tile by W_l (K_l x N_l, row-major).
// Matrix-core operand layouts of v_mfma_f32_16x16x32_bf16 (wave64):
//   A (16 x 32): lane l holds A[l % 16][8*(l/16) + i], i = 0..7
//   B (32 x 16): lane l holds B[8*(l/16) + i][l % 16], i = 0..7
//   D (16 x 16): lane l holds D[4*(l/16) + i][l % 16], i = 0..3
// The forward pass reads W_l as pre-packed B fragments (64 lanes x 8 bf16 per 32x16
// block, so each lane loads 16 contiguous bytes); the backward pass reads the
// row-major copy.
#pragma once
#include <hip/hip_runtime.h>

namespace ice3 {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int MLP_NFEAT = 18;   // features used
constexpr int MLP_NTARG = 8;    // outputs used
constexpr int MLP_IN = 32;      // padded input width
constexpr int MLP_H = 128;      // hidden width
constexpr int MLP_OUT = 32;     // padded output width
constexpr int MLP_LAYERS = 5;
constexpr int MLP_NW = MLP_IN * MLP_H + 3 * MLP_H * MLP_H + MLP_H * MLP_OUT;  // 57344
constexpr int MLP_NB = 4 * MLP_H + MLP_OUT;                                     // 544
constexpr int MLP_NP = MLP_NW + MLP_NB;  // parameters: weights then biases

constexpr int MLP_TILE = 128;                          // points per workgroup tile
constexpr int MLP_WAVES = 4;                           // 256-thread workgroups
constexpr int MLP_MT = MLP_TILE / (16 * MLP_WAVES);    // 16-row m-tiles per wave (2)
constexpr int MLP_ROWS = MLP_TILE / MLP_WAVES;         // rows owned by one wave (32)
constexpr int MLP_HS = MLP_H + 8;                      // padded LDS row strides (bf16)
constexpr int MLP_XS = MLP_IN + 8;
constexpr int MLP_YS = MLP_OUT + 4;                    // fp32 output rows

__host__ __device__ constexpr int mlp_k(int l) { return l == 0 ? MLP_IN : MLP_H; }
__host__ __device__ constexpr int mlp_n(int l) { return l == MLP_LAYERS - 1 ? MLP_OUT : MLP_H; }
__host__ __device__ constexpr int mlp_woff(int l) {
  return l == 0 ? 0 : MLP_IN * MLP_H + (l - 1) * MLP_H * MLP_H;
}
__host__ __device__ constexpr int mlp_boff(int l) { return MLP_NW + l * MLP_H; }

// Offset of row-major element (k, n) of layer l in the packed-fragment copy.
__host__ __device__ inline int mlp_pack_index(int l, int k, int n) {
  const int N = mlp_n(l);
  const int kk = k / 32, kr = k % 32, nn = n / 16, lane = (kr / 8) * 16 + n % 16, i = kr % 8;
  return mlp_woff(l) + ((kk * (N / 16) + nn) * 64 + lane) * 8 + i;
}

__device__ __forceinline__ f32x4 mfma_bf16(const bf16x8 &a, const bf16x8 &b, const f32x4 &c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// SiLU and its derivative from the hardware exp2 and reciprocal (about 1 ulp in fp32;
// the activations are rounded to bf16 afterwards).
__device__ __forceinline__ float sigmoid_fast(float z) {
  return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.44269504f * z));
}
__device__ __forceinline__ float silu(float z) { return z * sigmoid_fast(z); }
__device__ __forceinline__ float silu_grad(float z) {
  const float s = sigmoid_fast(z);
  return s * (1.f + z * (1.f - s));
}

// acc[mt][nn] = In[rows of this wave] (MLP_ROWS x K) * W (K x N), In row-major with row
// stride S (bf16) in LDS, W as packed fragments (LDS).
template <int K, int N, int S>
__device__ __forceinline__ void mlp_layer(const __bf16 *sIn, int row0, const bf16x8 *sWpk,
                                          f32x4 (&acc)[MLP_MT][N / 16], int lane) {
#pragma unroll
  for (int mt = 0; mt < MLP_MT; ++mt)
#pragma unroll
    for (int nn = 0; nn < N / 16; ++nn) acc[mt][nn] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < K / 32; ++kk) {
    bf16x8 a[MLP_MT];
#pragma unroll
    for (int mt = 0; mt < MLP_MT; ++mt)
      a[mt] = *(const bf16x8 *)(sIn + (row0 + mt * 16 + lane % 16) * S + kk * 32 + 8 * (lane / 16));
#pragma unroll
    for (int nn = 0; nn < N / 16; ++nn) {
      const bf16x8 b = sWpk[(kk * (N / 16) + nn) * 64 + lane];
#pragma unroll
      for (int mt = 0; mt < MLP_MT; ++mt) acc[mt][nn] = mfma_bf16(a[mt], b, acc[mt][nn]);
    }
  }
}

// ---- Activations in registers.  With the weights as the first matrix operand and the
// activations as the second (the packed W fragments are the A fragments of W^T), a product of a
// layer leaves lane l with units 4*(l/16) .. +3 of point l % 16 of each 16-unit tile; rounded to
// bf16 that is two dwords, and the next layer's operand wants units 8*(l/16) .. +7 of the same
// point of each 32-unit block.  Two lane swaps a dword pair bring the one to the other, so the
// activations of a wavefront never leave its registers.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ u32x2 pack4(float a, float b, float c, float d) {
  return u32x2{__builtin_bit_cast(unsigned int, bf16x2{(__bf16)a, (__bf16)b}),
               __builtin_bit_cast(unsigned int, bf16x2{(__bf16)c, (__bf16)d})};
}

// The operand fragment of 32 units from its two 16-unit tiles: rows r0..r3 (16 lanes each) of t0
// hold units 0-3, 4-7, 8-11, 12-15, of t1 16-19 .. 28-31; the halves swap gives (t0 r0 r1, t1 r0 r1)
// and (t0 r2 r3, t1 r2 r3), the rows swap units 8r .. 8r+3 and 8r+4 .. 8r+7 in row r.  Every lane
// of the wavefront must be active.
__device__ __forceinline__ bf16x8 operand_of(const u32x2 &t0, const u32x2 &t1) {
  u32x4 f;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const auto h = __builtin_amdgcn_permlane32_swap(t0[q], t1[q], false, false);
    const auto r = __builtin_amdgcn_permlane16_swap(h[0], h[1], false, false);
    f[q] = r[0];
    f[2 + q] = r[1];
  }
  return __builtin_bit_cast(bf16x8, f);
}

// acc[mt][nn]: 16 units (tile nn) x 16 points (tile mt) of W^T X, W as packed fragments in LDS (NT
// unit tiles wide, the first N / 16 of them taken), X as operand fragments.
template <int K, int N, int NT, int MT>
__device__ __forceinline__ void mlp_product(const bf16x8 *sWpk, const bf16x8 (&x)[MT][K / 32],
                                            f32x4 (&acc)[MT][N / 16], int lane) {
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nn = 0; nn < N / 16; ++nn) acc[mt][nn] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < K / 32; ++kk)
#pragma unroll
    for (int nn = 0; nn < N / 16; ++nn) {
      const bf16x8 w = sWpk[(kk * NT + nn) * 64 + lane];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt][nn] = mfma_bf16(w, x[mt][kk], acc[mt][nn]);
    }
}

// All packed weights and biases into LDS with a workgroup of NT threads, every load issued before the
// first store.
template <int NT>
__device__ __forceinline__ void stage_weights(bf16x8 *sW, float *sB, const bf16x8 *__restrict__ wpk,
                                              const float *__restrict__ params) {
  constexpr int NQ = MLP_NW / 8, NL = (NQ + NT - 1) / NT, NBL = (MLP_NB + NT - 1) / NT;
  bf16x8 v[NL];
  float b[NBL];
#pragma unroll
  for (int l = 0; l < NL; ++l) {
    const int q = threadIdx.x + l * NT;
    v[l] = wpk[q < NQ ? q : 0];
  }
#pragma unroll
  for (int l = 0; l < NBL; ++l) {
    const int q = threadIdx.x + l * NT;
    b[l] = params[MLP_NW + (q < MLP_NB ? q : 0)];
  }
#pragma unroll
  for (int l = 0; l < NL; ++l) {
    const int q = threadIdx.x + l * NT;
    if (q < NQ) sW[q] = v[l];
  }
#pragma unroll
  for (int l = 0; l < NBL; ++l) {
    const int q = threadIdx.x + l * NT;
    if (q < MLP_NB) sB[q] = b[l];
  }
}

}  // namespace ice3
