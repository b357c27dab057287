// mlp_core.hpp -- the closure network on BF16 matrix cores: shapes, parameter layout and the
// wave-level building blocks shared by the training kernels (mlp.hip) and the in-stage
// inference (dg_closure.hpp).
//
// Network: x (IN, zero padded) -> 3 x [64, GELU] -> y (OUT, zero padded), all products on
// the BF16 matrix cores (BF16 operands, FP32 accumulation), biases, GELU, loss and Adam in
// FP32.  Inputs are normalised, (x - mu) / sigma, and outputs de-normalised,
// y * scale + shift, in FP32 by the kernels.  Products whose contraction is 32 or more deep
// (every forward layer, the backward products dY W^T) use gfx950's
// v_mfma_f32_16x16x32_bf16; the weight gradients, contracted over a 16-row tile of
// samples, use v_mfma_f32_16x16x16_bf16.
//
// MFMA operand layouts (one wave, lane l, r = l % 16, g = l / 16):
//   16x16x16: A (16 x 16, i x k) lane l supplies A[r][4 g + j], j = 0..3; B (k x n) supplies
//             B[4 g + j][r]
//   16x16x32: A (16 x 32) lane l supplies A[r][8 g + j], j = 0..7; B (32 x 16) supplies
//             B[8 g + j][r]
//   D (16 x 16, FP32, both):            lane l holds D[4 g + j][r], j = 0..3
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace oceano {
namespace mlp {

constexpr int IN = 32, HID = 64, OUT = 32;
// FP32 master parameters, W_l row-major [fan_in][fan_out]
constexpr int W1 = 0, B1 = W1 + IN * HID, W2 = B1 + HID, B2 = W2 + HID * HID, W3 = B2 + HID,
              B3 = W3 + HID * HID, W4 = B3 + HID, B4 = W4 + HID * OUT, NPARAM = B4 + OUT;
// BF16 transposed weights [fan_out][fan_in]: the B operand of the forward products
constexpr int T1 = 0, T2 = T1 + HID * IN, T3 = T2 + HID * HID, T4 = T3 + HID * HID,
              NT = T4 + OUT * HID;
// normalisation block: mu[IN], inv_sigma[IN], scale[OUT], shift[OUT], lo[OUT], hi[OUT]
// (inference saturates the normalised output to [lo, hi]; training does not)
constexpr int NNORM = 2 * IN + 4 * OUT;
constexpr int NLO = 2 * IN + 2 * OUT, NHI = 2 * IN + 3 * OUT;

// de-normalised network output of column o at inference
__device__ inline float output_value(float yn, const float *norm, int o)
{
  yn = fminf(fmaxf(yn, norm[NLO + o]), norm[NHI + o]);
  return yn * norm[2 * IN + o] + norm[2 * IN + OUT + o];
}

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short bf16;

// FP32 -> BF16, round to nearest even (finite inputs)
__host__ __device__ inline bf16 to_bf16(float f)
{
  uint32_t u;
  __builtin_memcpy(&u, &f, 4);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}

__host__ __device__ inline float from_bf16(bf16 h)
{
  const uint32_t u = (uint32_t)h << 16;
  float f;
  __builtin_memcpy(&f, &u, 4);
  return f;
}

__device__ inline f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ inline f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// the 8 consecutive BF16 values at p (16-byte aligned) as an MFMA operand
__device__ inline bf16x8 load8(const bf16 *p) { return *(const bf16x8 *)p; }

// A wave works on tiles of 16 samples with every weight in registers: the B operand of a
// column tile and 32-deep step is 16 consecutive bytes of the transposed weights per lane, so
// one lane holds the whole network in 24 loads of 16 bytes (96 registers), issued at once.  The
// alternative, a copy in LDS, costs each workgroup 24 KiB of staging before its first product:
// the in-stage inference on 2,500 cells took 33.0 us with it, 9.6 us this way.
struct ForwardWeights
{
  bf16x8 w1[HID / 16], w2[HID / 16 * 2], w3[HID / 16 * 2], w4[OUT / 16 * 2];
  float b1[HID / 16], b2[HID / 16], b3[HID / 16], b4[OUT / 16];

  // wt: transposed BF16 weights, p: FP32 parameters (biases), both in global memory
  __device__ __forceinline__ void load(const bf16 *__restrict__ wt, const float *__restrict__ p)
  {
    const int l = threadIdx.x & 63, r = l & 15, k8 = (l >> 4) * 8;
#pragma unroll
    for (int ct = 0; ct < HID / 16; ++ct)
      {
        w1[ct] = load8(wt + T1 + (16 * ct + r) * IN + k8);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
          {
            w2[2 * ct + kk] = load8(wt + T2 + (16 * ct + r) * HID + 32 * kk + k8);
            w3[2 * ct + kk] = load8(wt + T3 + (16 * ct + r) * HID + 32 * kk + k8);
          }
        b1[ct] = p[B1 + 16 * ct + r];
        b2[ct] = p[B2 + 16 * ct + r];
        b3[ct] = p[B3 + 16 * ct + r];
      }
#pragma unroll
    for (int ct = 0; ct < OUT / 16; ++ct)
      {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
          w4[2 * ct + kk] = load8(wt + T4 + (16 * ct + r) * HID + 32 * kk + k8);
        b4[ct] = p[B4 + 16 * ct + r];
      }
  }
};

// row stride of a 16 x 64 activation tile in LDS: 16 bytes of padding spread the 16 rows that an
// operand read touches over the banks
constexpr int LDT = HID + 8;

// orders this wave's LDS writes before its reads by other lanes (the wave owns the tile)
__device__ __forceinline__ void tile_fence()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// acc[ct] = A[16 x 64] W for NC column tiles, A in LDS (row stride LDT); the k order is fixed, so
// a row's result does not depend on the other rows of the tile
template <int NC>
__device__ __forceinline__ void tile_product(const bf16 *A, const bf16x8 (&w)[2 * NC],
                                             f32x4 (&acc)[NC])
{
  const int l = threadIdx.x & 63, r = l & 15, k8 = (l >> 4) * 8;
#pragma unroll
  for (int ct = 0; ct < NC; ++ct)
    acc[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
    {
      const bf16x8 a = load8(A + r * LDT + 32 * kk + k8);
#pragma unroll
      for (int ct = 0; ct < NC; ++ct)
        acc[ct] = mfma32(a, w[2 * ct + kk], acc[ct]);
    }
}

// bias and GELU of a layer: the BF16 activations h of the lane's accumulator entries, also into
// the LDS tile H; slope: the GELU derivatives there (null: not needed)
__device__ __forceinline__ void hidden_layer(const f32x4 (&acc)[HID / 16],
                                             const float (&bias)[HID / 16], bf16 *H,
                                             bf16x4 (*h)[HID / 16], f32x4 (*slope)[HID / 16])
{
  const int l = threadIdx.x & 63, r = l & 15, kq = (l >> 4) * 4;
#pragma unroll
  for (int ct = 0; ct < HID / 16; ++ct)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      {
        const float z = acc[ct][j] + bias[ct];
        const float e = erff(z * 0.70710678118654752f);
        const bf16 v = to_bf16(0.5f * z * (1.0f + e));
        H[(kq + j) * LDT + 16 * ct + r] = v;
        if (h)
          (*h)[ct][j] = (short)v;
        if (slope)
          (*slope)[ct][j] = 0.5f * (1.0f + e) + z * 0.39894228040143268f * expf(-0.5f * z * z);
      }
}

// forward of one tile: x the A operand of its normalised BF16 inputs (row l % 16, inputs
// 8 (l / 16) ..), H two LDS tiles of the wave; out: entries (row 4 (l / 16) + j, output 16 ct +
// l % 16) before de-normalisation.  h, slope (may be null): per hidden layer, see hidden_layer
__device__ __forceinline__ void forward_tile(bf16x8 x, const ForwardWeights &W, bf16 (*H)[16 * LDT],
                                             f32x4 (&out)[OUT / 16],
                                             bf16x4 (*h)[HID / 16] = nullptr,
                                             f32x4 (*slope)[HID / 16] = nullptr)
{
  f32x4 acc[HID / 16];
#pragma unroll
  for (int ct = 0; ct < HID / 16; ++ct)
    acc[ct] = mfma32(x, W.w1[ct], f32x4{0.f, 0.f, 0.f, 0.f});
  hidden_layer(acc, W.b1, H[0], h, slope);
  tile_fence();
  tile_product<HID / 16>(H[0], W.w2, acc);
  hidden_layer(acc, W.b2, H[1], h ? h + 1 : nullptr, slope ? slope + 1 : nullptr);
  tile_fence();
  tile_product<HID / 16>(H[1], W.w3, acc);
  hidden_layer(acc, W.b3, H[0], h ? h + 2 : nullptr, slope ? slope + 2 : nullptr);
  tile_fence();
  tile_product<OUT / 16>(H[0], W.w4, out);
#pragma unroll
  for (int ct = 0; ct < OUT / 16; ++ct)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      out[ct][j] += W.b4[ct];
}

}  // namespace mlp
}  // namespace oceano
