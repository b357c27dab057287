// dg_closure.hpp -- the learned momentum-source correction inside the stage.
//
// Per cell (one lane), from the stage input: the modal coefficients (orthonormal tensor
// Legendre modes) of zeta, hu, hv and the sub-grid statistics (mean, variance, skewness) of
// the bed form the network input; the output holds the modal coefficients of the
// correction tau of hu and hv, which is brought back to nodal values and added to
// M^-1 L_q by the discharge update (a source s in L_q enters as M s, so adding tau after
// the inverse mass is the source term of ShallowWater.h:425-429 with s = tau).  A cell
// that is not active (no sub-grid bathymetry nearby) or whose network output is not finite
// gets tau = 0: the plain sub-grid model.
#pragma once

#include "dg_internal.hpp"
#include "dg_stage.hpp"
#include "mlp_core.hpp"

extern "C" void oc_mlp_device_state(const oc_mlp *m, const float **p, const uint16_t **wt,
                                    const float **norm);

namespace oceano {

struct ClosureArgs
{
  const double *zeta, *q;
  const double *stats;  // [batch][4][lane]: mean, variance, skewness, active flag
  const double *vi;     // [nd][nd] modal <- nodal
  const double *v;      // [nd][nd] nodal <- modal
  const float *p;       // network parameters (biases)
  const uint16_t *wt;   // transposed BF16 weights
  const float *norm;    // normalisation block
  int n_in, n_out;
  double *tau;          // [batch][2][nd][lane]
  float *features;      // [n_cells][n_in] in the caller's cell order (features kernel)
  const int *order;     // slot -> cell
};

template <int P>
__device__ inline void closure_features(const ClosureArgs &C, int batch, int lane,
                                        float (&f)[mlp::IN])
{
  constexpr int ND = (P + 1) * (P + 1);
  static_assert(3 * ND + 3 <= mlp::IN, "closure inputs exceed the network width");
  double z[ND], qx[ND], qy[ND];
#pragma unroll
  for (int k = 0; k < ND; ++k)
    {
      z[k] = C.zeta[vix(batch, 1, 0, ND, k, lane)];
      qx[k] = C.q[vix(batch, 2, 0, ND, k, lane)];
      qy[k] = C.q[vix(batch, 2, 1, ND, k, lane)];
    }
#pragma unroll
  for (int m = 0; m < ND; ++m)
    {
      double a = 0, b = 0, c = 0;
#pragma unroll
      for (int k = 0; k < ND; ++k)
        {
          const double w = C.vi[m * ND + k];
          a += w * z[k];
          b += w * qx[k];
          c += w * qy[k];
        }
      f[m] = float(a);
      f[ND + m] = float(b);
      f[2 * ND + m] = float(c);
    }
#pragma unroll
  for (int s = 0; s < 3; ++s)
    f[3 * ND + s] = float(C.stats[((size_t)batch * 4 + s) * CB + lane]);
#pragma unroll
  for (int i = 3 * ND + 3; i < mlp::IN; ++i)
    f[i] = 0.f;
}

template <int P>
__global__ __launch_bounds__(CB) void k_closure_features(OpArgs O, ClosureArgs C)
{
  const int batch = blockIdx.x, lane = threadIdx.x;
  const int slot = batch * CB + lane;
  if (slot >= O.n_cells)
    return;
  float f[mlp::IN];
  closure_features<P>(C, batch, lane, f);
  const size_t row = (size_t)C.order[slot] * C.n_in;
#pragma unroll
  for (int i = 0; i < mlp::IN; ++i)
    if (i < C.n_in)
      C.features[row + i] = f[i];
}

// The correction of 16 cells per wave and pass.  The lanes are 16 cells x 4 groups: group g < 3
// forms the modal coefficients of field g (zeta, hu, hv), group 3 takes the statistics; after
// the network group g brings half of the nodes of component g / 2 back to nodal values.  A cell
// gets tau = 0 unless it is active and all its outputs are finite.
// Latency bounds it (2,500 cells are 157 waves): 16 cells per wave instead of 64 cells and four
// tiles in turn, weights in registers (ForwardWeights): 33.0 -> 9.6 us.
template <int P>
__global__ __launch_bounds__(CB) void k_closure(OpArgs O, ClosureArgs C)
{
  using namespace mlp;
  constexpr int ND = (P + 1) * (P + 1), TILES = CB / 16;
  static_assert(3 * ND + 3 <= IN && 2 * ND <= OUT, "closure network too narrow");
  __shared__ __attribute__((aligned(16))) bf16 s_x[16 * IN];
  __shared__ __attribute__((aligned(16))) bf16 s_h[2][16 * LDT];
  __shared__ float s_y[16 * OUT];
  const int lane = threadIdx.x, r = lane & 15, g = lane >> 4;
  ForwardWeights W;
  W.load(C.wt, C.p);
  const int n_tiles = (O.n_cells + 15) / 16;
  for (int tile = logical_batch(blockIdx.x, gridDim.x, O.xcd_swizzle); tile < n_tiles;
       tile += gridDim.x)
    {
      const int batch = tile / TILES, cl = (tile % TILES) * 16 + r;
      const bool inside = tile * 16 + r < O.n_cells;
      if (g < 3)
        {
          const double *src = g == 0 ? C.zeta + vix(batch, 1, 0, ND, 0, cl)
                                     : C.q + vix(batch, 2, g - 1, ND, 0, cl);
          double u[ND];
#pragma unroll
          for (int k = 0; k < ND; ++k)
            u[k] = inside ? src[k * CB] : 0.0;
#pragma unroll
          for (int m = 0; m < ND; ++m)
            {
              double a = 0;
#pragma unroll
              for (int k = 0; k < ND; ++k)
                a += C.vi[m * ND + k] * u[k];
              const int i = g * ND + m;
              s_x[r * IN + i] =
                to_bf16(inside ? (float(a) - C.norm[i]) * C.norm[IN + i] : 0.f);
            }
        }
      else
        {
#pragma unroll
          for (int i = 3 * ND; i < IN; ++i)
            {
              float x = 0.f;
              if (i < 3 * ND + 3 && inside)
                x = (float(C.stats[((size_t)batch * 4 + i - 3 * ND) * CB + cl]) - C.norm[i]) *
                    C.norm[IN + i];
              s_x[r * IN + i] = to_bf16(x);
            }
        }
      tile_fence();
      f32x4 out[OUT / 16];
      forward_tile(load8(s_x + r * IN + 8 * g), W, s_h, out);
#pragma unroll
      for (int ct = 0; ct < OUT / 16; ++ct)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          s_y[(4 * g + j) * OUT + 16 * ct + r] = out[ct][j];
      tile_fence();
      const int c = g >> 1;
      double tm[ND];
      bool finite = inside && C.stats[((size_t)batch * 4 + 3) * CB + cl] != 0.0;
#pragma unroll
      for (int m = 0; m < ND; ++m)
        {
          const float y = output_value(s_y[r * OUT + c * ND + m], C.norm, c * ND + m);
          finite = finite && isfinite(y);
          tm[m] = double(y);
        }
      // both components of the cell: groups 0 and 2
      const unsigned long long ok = __ballot(finite);
      finite = ((ok >> r) & (ok >> (r + 32)) & 1ull) != 0;
      constexpr int HALF = (ND + 1) / 2;
      const bool hi = g & 1;
#pragma unroll
      for (int i = 0; i < HALF; ++i)
        {
          constexpr int LAST = ND - 1;
          const int k_hi = HALF + i <= LAST ? HALF + i : LAST;
          double t = 0;
#pragma unroll
          for (int m = 0; m < ND; ++m)
            t += (hi ? C.v[k_hi * ND + m] : C.v[i * ND + m]) * tm[m];
          if (!hi || HALF + i <= LAST)
            C.tau[vix(batch, 2, c, ND, hi ? k_hi : i, cl)] = finite ? t : 0.0;
        }
      tile_fence();
    }
}

// features != nullptr: write the network inputs of every cell (k_closure_features);
// otherwise evaluate the attached network into op->d_closure (k_closure)
template <int P>
int launch_closure(oc_dg *op, const OpArgs &O, const double *zeta, const double *q,
                   float *features, hipStream_t s)
{
  if constexpr (3 * (P + 1) * (P + 1) + 3 > mlp::IN)
    {
      set_error("closure: degree above 2 exceeds the network input width");
      return OC_ERR_ARGUMENT;
    }
  else
    {
      constexpr int ND = (P + 1) * (P + 1);
      ClosureArgs C{};
      C.zeta = zeta;
      C.q = q;
      C.stats = op->d_cstats;
      C.vi = op->d_cvi;
      C.v = op->d_cv;
      C.order = op->d_order;
      C.features = features;
      C.tau = op->d_closure;
      C.n_in = 3 * ND + 3;
      C.n_out = 2 * ND;
      if (features)
        hipLaunchKernelGGL((k_closure_features<P>), dim3(op->NB), dim3(CB), 0, s, O, C);
      else
        {
          oc_mlp_device_state(op->closure_mlp, &C.p, &C.wt, &C.norm);
          // a wave per 16 cells up to 4 waves per SIMD, then each wave keeps its weights for
          // several tiles
          const int tiles = (op->N + 15) / 16;
          hipLaunchKernelGGL((k_closure<P>), dim3(tiles < 4096 ? tiles : 4096), dim3(CB), 0, s, O,
                             C);
        }
      HIP_TRY(hipGetLastError());
      return OC_OK;
    }
}

}  // namespace oceano
