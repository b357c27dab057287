// dg_launch.hpp -- launch sequences of one stage / rhs / apply, per degree.
#pragma once

#include "dg_ark.hpp"
#include "dg_closure.hpp"
#include "dg_internal.hpp"
#include "dg_post.hpp"
#include "dg_stage.hpp"

namespace oceano {
namespace {

struct RkArgs
{
  size_t n;
  const double *k[MAXKI];
  double factor[MAXKI];
  int nk;
  const double *w;
  double *dst;
};

// dst = w + sum_j factor_j k_j, in the reference's order (OceanDG.h:1878-1909); the k
// vectors are stored in KT
template <typename KT>
__global__ void k_rk_update(RkArgs A)
{
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < A.n;
       i += (size_t)gridDim.x * blockDim.x)
    {
      double acc = A.w[i] + A.factor[0] * double(reinterpret_cast<const KT *>(A.k[0])[i]);
      for (int j = 1; j < A.nk; ++j)
        acc += A.factor[j] * double(reinterpret_cast<const KT *>(A.k[j])[i]);
      A.dst[i] = acc;
    }
}


// the arguments of the height and discharge work of one explicit stage
inline void stage_args(const OpArgs &O, uint32_t stage, const double *factor,
                       const double *ri_h, const double *ri_q, const double *ri_v,
                       double *const *ki_h, double *const *ki_q, uint32_t n_ki, double *w_h,
                       double *w_q, double *r_h, double *r_q, int write_scratch, StageArgs &H,
                       StageArgs &Q)
{
  const bool last = (stage == n_ki - 2);
  double *h_dst = last ? w_h : r_h;
  double *q_dst = last ? w_q : r_q;
  // discharge: L_q -> M^-1 L_q -> ki_q[stage+1]; q_dst = w_q + sum_j a_j ki_q[j+1]
  Q = StageArgs{};
  Q.src_h = ri_h;
  Q.src_q = ri_q;
  Q.src_v = ri_v;
  Q.dst = ki_q[stage + 1];
  Q.scratch = write_scratch ? ki_q[0] : nullptr;
  for (uint32_t j = 0; j < stage; ++j)
    Q.kprev[j] = ki_q[j + 1];
  for (uint32_t j = 0; j <= stage; ++j)
    Q.factor[j] = factor[j];
  Q.stage = (int)stage;
  Q.wsol = w_q;
  Q.rk_dst = q_dst;
  // height: L_zeta -> ki_h[stage+1]; front; Jacobi -> h_dst
  H = StageArgs{};
  H.src_h = ri_h;
  H.src_q = ri_q;
  H.dst = ki_h[stage + 1];
  for (uint32_t j = 0; j < stage; ++j)
    H.kprev[j] = ki_h[j + 1];
  for (uint32_t j = 0; j <= stage; ++j)
    H.factor[j] = factor[j];
  H.stage = (int)stage;
  H.wsol = w_h;
  H.rk_dst = h_dst;
  H.scratch = write_scratch ? ki_h[0] : nullptr;
  H.sweeps_blk = O.sweeps;
}

// launch(args) with the argument type that says which terms there are
template <typename Fn>
inline void with_terms(const OpArgs &O, Fn launch)
{
  if (is_plain(O))
    launch(PlainArgs{O});
  else if (is_manning(O))
    launch(ManningArgs{O});
  else
    launch(O);
}

template <int P, typename R>
int launch_stage(oc_dg *op, const OpArgs &O, uint32_t stage, const double *factor,
                 const double *ri_h, const double *ri_q, const double *ri_v,
                 double *const *ki_h, double *const *ki_q, uint32_t n_ki, double *w_h,
                 double *w_q, double *r_h, double *r_q, int write_scratch, hipStream_t s)
{
  const bool last = (stage == n_ki - 2);
  const dim3 grid(op->NB), block(CB);
  double *h_dst = last ? w_h : r_h;
  double *q_dst = last ? w_q : r_q;
  const bool visc = O.nu != 0.0;
  hipEvent_t ev = nullptr;
  StageArgs H, Q;
  stage_args(O, stage, factor, ri_h, ri_q, ri_v, ki_h, ki_q, n_ki, w_h, w_q, r_h, r_q,
             write_scratch, H, Q);
  // the one-pass stage reads neighbour traces of ri while other cells write the outputs:
  // it needs outputs distinct from the inputs (single-stage schemes write w in place)
  const bool alias = (h_dst == ri_h) || (q_dst == ri_q) || (h_dst == ri_q) || (q_dst == ri_h);
  if (!alias)
    {
      timed_begin(op, s, &ev);
      const int items = 2 * op->NB;
      if (visc)
        {
          // paired in FP64 at p <= 2 (RK4 step of 12,800 cells at p = 1 43 -> 35 us, of 51,200 at
          // p = 2 138 -> 129 us); at p >= 3 the cell term's gradients of the velocity fill two
          // waves' registers and the unpaired items at one wave per SIMD are faster (26,000 hanging
          // cells at p = 3: 196 us a step, paired 225; 5,000 at p = 4: 264, paired 279).  FP32 items
          // are unpaired, by the terms there are: 110,000 cells over a flat bed p = 1 103 -> 94 us a
          // step, p = 2 185 -> 168, p = 3 343 -> 310, p = 4 749 -> 654 (FP64 at p >= 3 tests them
          // at run time: there the viscous terms fill the registers either way)
          if constexpr (std::is_same<R, double>::value && P <= 2)
            with_terms(O, [&](auto args) {
              hipLaunchKernelGGL((k_stage_pair<P, R, false, true, 0, decltype(args)>), grid,
                                 dim3(2 * CB), 0, s, args, H, Q);
            });
          else if constexpr (std::is_same<R, float>::value)
            with_terms(O, [&](auto args) {
              hipLaunchKernelGGL((k_stage<P, true, R, 1, decltype(args)>), dim3(items), block, 0, s,
                                 args, H, Q);
            });
          else
            hipLaunchKernelGGL((k_stage<P, true, R, 1>), dim3(items), block, 0, s, O, H, Q);
        }
      else if (op->paired_items)
        {
          constexpr bool C32 = std::is_same<R, float>::value && P <= 3;
          if (C32)
            H.out32 = Q.out32 = op->rk_out32 && !last;
          with_terms(O, [&](auto args) {
            using OA = decltype(args);
            if (C32 && op->rk_in32)
              hipLaunchKernelGGL((k_stage_pair<P, R, C32, false, 0, OA>), grid, dim3(2 * CB), 0, s,
                                 args, H, Q);
            else
              hipLaunchKernelGGL((k_stage_pair<P, R, false, false, 0, OA>), grid, dim3(2 * CB), 0,
                                 s, args, H, Q);
          });
        }
      else
        with_terms(O, [&](auto args) {
          using OA = decltype(args);
          if (op->waves_per_block == 4)
            hipLaunchKernelGGL((k_stage<P, false, R, 4, OA>), dim3((items + 3) / 4), dim3(4 * CB),
                               0, s, args, H, Q);
          else if (op->waves_per_block == 2)
            hipLaunchKernelGGL((k_stage<P, false, R, 2, OA>), dim3((items + 1) / 2), dim3(2 * CB),
                               0, s, args, H, Q);
          else
            hipLaunchKernelGGL((k_stage<P, false, R, 1, OA>), dim3(items), block, 0, s, args, H, Q);
        });
      timed_end(op, s, TK_STAGE, ev);
      HIP_TRY(hipGetLastError());
      if (std::is_same<R, float>::value && defer_depth_solve(P))
        {
          // FP64 depth solve of the cells the FP32 stage left near the depth floor; a wave
          // without such a cell returns at once
          StageArgs D = H;
          for (uint32_t j = 0; j <= stage; ++j)
            D.kprev[j] = ki_h[j + 1];
          timed_begin(op, s, &ev);
          const dim3 dgrid((op->NB + DEFER_BATCHES - 1) / DEFER_BATCHES);
          hipLaunchKernelGGL((k_depth_deferred<P>), dgrid, block, 0, s, O, D);
          timed_end(op, s, TK_HEIGHT_JACOBI, ev);
          HIP_TRY(hipGetLastError());
        }
      return OC_OK;
    }
  // split path: every kernel finishes reading ri before the next one overwrites it
  timed_begin(op, s, &ev);
  hipLaunchKernelGGL((k_height_rhs<P, R>), grid, block, 0, s, O, ri_h, ri_q,
                     ki_h[stage + 1]);
  timed_end(op, s, TK_HEIGHT_RHS, ev);
  timed_begin(op, s, &ev);
  StageArgs A = Q;
  if (visc)
    hipLaunchKernelGGL((k_discharge<P, true, 3, R>), grid, block, 0, s, O, A);
  else
    hipLaunchKernelGGL((k_discharge<P, false, 3, R>), grid, block, 0, s, O, A);
  timed_end(op, s, TK_DISCHARGE, ev);
  RkArgs U{};
  U.n = (size_t)op->NB * CB * 2 * op->nd;
  for (uint32_t j = 0; j <= stage; ++j)
    {
      U.k[j] = ki_q[j + 1];
      U.factor[j] = factor[j];
    }
  U.nk = (int)stage + 1;
  U.w = w_q;
  U.dst = q_dst;
  timed_begin(op, s, &ev);
  hipLaunchKernelGGL(k_rk_update<R>, dim3((U.n + 255) / 256), dim3(256), 0, s, U);
  timed_end(op, s, TK_RK_UPDATE, ev);
  StageArgs J = H;
  for (uint32_t j = 0; j <= stage; ++j)
    J.kprev[j] = ki_h[j + 1];
  timed_begin(op, s, &ev);
  hipLaunchKernelGGL((k_height_jacobi<P, R, R>), grid, block, 0, s, O, J);
  timed_end(op, s, TK_HEIGHT_JACOBI, ev);
  HIP_TRY(hipGetLastError());
  return OC_OK;
}

template <int P, typename R>
int launch_rhs_apply(oc_dg *op, const OpArgs &O, bool invert, const double *src_h,
                     const double *src_q, const double *src_v, double *dst_h, double *dst_q,
                     hipStream_t s)
{
  const dim3 grid(op->NB), block(CB);
  const bool visc = O.nu != 0.0;
  StageArgs S{};
  S.src_h = src_h;
  S.src_q = src_q;
  S.src_v = src_v;
  S.dst = dst_q;
  // FP64: one launch of paired items at p <= 3, viscous at p <= 2 (as the viscous stage).  At p = 4,
  // M^-1 L of 25,538 cells, they measured 46.5 us, but the compiler left two of their builds with
  // register copies that miss the coarse cells of hanging faces (oceano_amd/check_code.py; both wave
  // roles are short of scalar and of vector registers there).  There, and for the FP32 integrals, whose
  // results carry the order of summation of the unpaired items, one launch of unpaired items: 52 us
  // (two launches, one an equation, 77).
  constexpr bool PAIRED = std::is_same<R, double>::value && P <= 3;
  constexpr bool PAIRED_VISC = std::is_same<R, double>::value && P <= 2;
  StageArgs H = S;
  H.dst = dst_h;
  const dim3 pair(2 * CB), items(2 * op->NB);
  with_terms(O, [&](auto args) {
    using OA = decltype(args);
    if constexpr (PAIRED)
      if (!visc)
        {
          if (invert)
            hipLaunchKernelGGL((k_stage_pair<P, R, false, false, 1, OA>), grid, pair, 0, s, args,
                               H, S);
          else
            hipLaunchKernelGGL((k_stage_pair<P, R, false, false, 2, OA>), grid, pair, 0, s, args,
                               H, S);
        }
    if constexpr (!PAIRED)
      if (!visc)
        {
          if (invert)
            hipLaunchKernelGGL((k_stage<P, false, R, 1, OA, 1>), items, block, 0, s, args, H, S);
          else
            hipLaunchKernelGGL((k_stage<P, false, R, 1, OA, 2>), items, block, 0, s, args, H, S);
        }
  });
  if (visc)
    {
      if constexpr (PAIRED_VISC)
        {
          if (invert)
            hipLaunchKernelGGL((k_stage_pair<P, R, false, true, 1>), grid, pair, 0, s, O, H, S);
          else
            hipLaunchKernelGGL((k_stage_pair<P, R, false, true, 2>), grid, pair, 0, s, O, H, S);
        }
      else
        {
          if (invert)
            hipLaunchKernelGGL((k_stage<P, true, R, 1, OpArgs, 1>), items, block, 0, s, O, H, S);
          else
            hipLaunchKernelGGL((k_stage<P, true, R, 1, OpArgs, 2>), items, block, 0, s, O, H, S);
        }
    }
  HIP_TRY(hipGetLastError());
  return OC_OK;
}


}  // namespace
}  // namespace oceano
