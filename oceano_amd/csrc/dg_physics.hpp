// dg_physics.hpp -- pointwise shallow-water model and numerical fluxes (device code).
//
// Restates, for a scalar number type T, the inline functions the reference evaluates at
// every quadrature point:
//   ShallowWater.h:315-336  depth (floor 1e-12) and desingularised velocity
//   ShallowWater.h:381-432  advective/diffusive flux and source (Manning friction,
//                           general wind stress, Coriolis; BottomFriction.h:186-199,
//                           WindStress.h:101-108, Coriolis.h:87-95)
//   ShallowWater.h:476-516  Riemann invariants (absorbing outflow)
//   LaxFriedrichsModified.h:161-230  LLF mass / advective flux, hydrostatic reconstruction
//   NumericalFluxBase.h:103-126      centred strong-form pressure jump
// The faces of the configured meshes are axis-aligned, so the normal is one of +-e_x,
// +-e_y; the functions still take a general normal.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

namespace oceano {

template <typename T>
struct Vec2
{
  T x, y;
};

// 1/sqrt(x) for x > 0 (the depth floor keeps every argument positive): the hardware
// reciprocal square root (relative error at most 5.3e-8) and one third-order step
// y (1 + e / 2 + 3 e^2 / 8), e = 1 - x y^2.  Over 2^20 arguments in [1, 4] and [1e-40, 1e20] the
// error is at most 1.37e-16 (rms 5.4e-17), as with the two Newton-Raphson steps that it
// replaces (1.38e-16), in five instructions, four of them in a chain, for eight, six in a
// chain.  RK4 step of 2,500 channel cells at p = 2 FP64 69 -> 66.5 us, of 97,280 at p = 3 314 ->
// 311 us, additive step of 64,464 148 -> 145 us.
__device__ __forceinline__ double rsqrt_nr(double x)
{
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-(x * y), y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}
// FP32 (mixed path): the hardware reciprocal square root (within 1 ulp), unrefined
__device__ __forceinline__ float rsqrt_nr(float x) { return __builtin_amdgcn_rsqf(x); }

// a b + c d.  FP32: the first product rounded, the second fused.  Which of two products a compiler
// fuses depends on the code around them; written out, the FP32 results of the integrals do not
// change with it
__device__ __forceinline__ double two_products(double a, double b, double c, double d)
{
  return a * b + c * d;
}
__device__ __forceinline__ float two_products(float a, float b, float c, float d)
{
  return __builtin_fmaf(c, d, a * b);
}

// s + a b, the product fused
__device__ __forceinline__ double plus_product(double s, double a, double b) { return s + a * b; }
__device__ __forceinline__ float plus_product(float s, float a, float b)
{
  return __builtin_fmaf(a, b, s);
}

// sqrt(x), x >= 0, through rsqrt_nr
__device__ __forceinline__ double sqrt_nr(double x) { return x > 0.0 ? x * rsqrt_nr(x) : x; }

// The Manning powers h^-0.33333333333 and h^-1.33333333333 of the reference
// (BottomFriction.h:186-212 writes them as exp(a log h)), h >= 1e-12.  Both are a cube root
// times h^(10^-11 / 3): y = h^(-1/3) starts from the FP32 log2 / exp2 (relative error some
// 1e-6) and takes one third-order step y (1 + e / 3 + 2 e^2 / 9), e = 1 - h y^3; the remaining
// exponent enters as 1 + c, c = ln h 10^-11 / 3.  About 20 instructions in place of FP64 exp,
// log and a division (about 170), to the last bits: an RK4 step of the 2,500-cell channel
// at p = 2 101 -> 84 us, an additive step of 64,464 cells 179 -> 168 us.
struct ManningPowers
{
  double y, c;
  __device__ __forceinline__ explicit ManningPowers(double h)
  {
    const float l2 = float(__builtin_amdgcn_frexp_exp(h)) +
                     __builtin_amdgcn_logf(float(__builtin_amdgcn_frexp_mant(h)));
    const double y0 = double(__builtin_amdgcn_exp2f(l2 * -0.33333334f));
    const double e = __builtin_fma(-h, y0 * y0 * y0, 1.0);
    y = __builtin_fma(y0, e * __builtin_fma(e, 2.0 / 9.0, 1.0 / 3.0), y0);
    c = double(l2) * 2.3104906e-12;
  }
  __device__ __forceinline__ double third() const { return __builtin_fma(y, c, y); }
  __device__ __forceinline__ double four_thirds() const
  {
    const double y4 = (y * y) * (y * y);
    return __builtin_fma(y4, c, y4);
  }
};

// Manning friction g n^2 |v| / h^(1/3) (BottomFriction.h:186-199)
__device__ __forceinline__ double manning_coefficient(double g, double n, double h, double vx,
                                                      double vy)
{
  return g * n * n * ManningPowers(h).third() * sqrt_nr(vx * vx + vy * vy);
}
__device__ __forceinline__ float manning_coefficient(float g, float n, float h, float vx,
                                                     float vy)
{
  const float inv_d = 1.f / (exp(log(h) * 0.33333333333f));
  return g * n * n * inv_d * sqrt(two_products(vy, vy, vx, vx));
}

// a . n for the axis-aligned normals of the kernels: with one component of n zero the
// other product is the whole dot product (a.x * 1 + a.y * 0 == a.x for finite a); the
// tests fold at compile time because every normal is a constant of an unrolled face loop
template <typename T>
__host__ __device__ __forceinline__ T dot_n(Vec2<T> a, Vec2<T> n)
{
  if (n.y == T(0))
    return a.x * n.x;
  if (n.x == T(0))
    return a.y * n.y;
  return a.x * n.x + a.y * n.y;
}

// FLAT: the bed is known to be uniform (zb_m == zb_p everywhere)
template <typename T, bool FLAT = false>
struct Phys
{
  T g;
  T cu4;  // Threshold_for_wetdry^4 (ShallowWater.h:295-296)
  T nu;   // constant horizontal viscosity

  __host__ __device__ __forceinline__ T depth(T z, T zb) const
  {
    const T h = z + zb;
    return h > T(1e-12) ? h : T(1e-12);
  }

  // inverse_depth = sqrt(2) h / sqrt(h^4 + max(h^4, cu^4))
  __device__ __forceinline__ T inv_depth(T h) const
  {
    const T h4 = h * h * h * h;
    const T mx = h4 > cu4 ? h4 : cu4;
    return (T(1.4142135623730951) * h) * rsqrt_nr(h4 + mx);
  }

  __device__ __forceinline__ Vec2<T> velocity(T z, Vec2<T> q, T zb) const
  {
    const T s = inv_depth(depth(z, zb));
    return {q.x * s, q.y * s};
  }

  // sqrt(g h) = (g h) / sqrt(g h); g h >= g 1e-12 > 0
  __device__ __forceinline__ T wave_speed(T z, T zb) const
  {
    const T gh = g * depth(z, zb);
    return gh * rsqrt_nr(gh);
  }

  // LaxFriedrichsModified::numerical_massflux_weak
  __device__ __forceinline__ T mass_flux(T z_m, T z_p, Vec2<T> q_m, Vec2<T> q_p, Vec2<T> n,
                                        T zb_m, T zb_p) const
  {
    const Vec2<T> v_m = velocity(z_m, q_m, zb_m);
    const Vec2<T> v_p = velocity(z_p, q_p, zb_p);
    const T lm = std::fabs(dot_n(v_m, n)) + wave_speed(z_m, zb_m);
    const T lp = std::fabs(dot_n(v_p, n)) + wave_speed(z_p, zb_p);
    const T lambda = lp > lm ? lp : lm;
    const T zbs = zb_m < zb_p ? zb_m : zb_p;
    const T hm = depth(z_m, zbs), hp = depth(z_p, zbs);
    const T zcm = z_m > -zbs ? z_m : -zbs;
    const T zcp = z_p > -zbs ? z_p : -zbs;
    return T(0.5) * (dot_n(Vec2<T>{hm * v_m.x, hm * v_m.y}, n) +
                     dot_n(Vec2<T>{hp * v_p.x, hp * v_p.y}, n)) +
           T(0.5) * lambda * (zcm - zcp);
  }

  // LaxFriedrichsModified::numerical_advflux_weak.  BOUNDARY only turns the FP32 rounding of
  // its sums round (two_products): the boundary faces have always been summed so
  template <bool BOUNDARY = false>
  __device__ __forceinline__ Vec2<T> adv_flux(T z_m, T z_p, Vec2<T> q_m, Vec2<T> q_p,
                                             Vec2<T> n, T zb_m, T zb_p) const
  {
    const T s_m = inv_depth(depth(z_m, zb_m)), s_p = inv_depth(depth(z_p, zb_p));
    const Vec2<T> v_m = {q_m.x * s_m, q_m.y * s_m};
    const Vec2<T> v_p = {q_p.x * s_p, q_p.y * s_p};
    const T lm = std::fabs(dot_n(v_m, n)) + wave_speed(z_m, zb_m);
    const T lp = std::fabs(dot_n(v_p, n)) + wave_speed(z_p, zb_p);
    const T lambda = lp > lm ? lp : lm;
    const T zbs = zb_m < zb_p ? zb_m : zb_p;
    const T hm = depth(z_m, zbs), hp = depth(z_p, zbs);
    const Vec2<T> hu_m = {hm * v_m.x, hm * v_m.y};
    const Vec2<T> hu_p = {hp * v_p.x, hp * v_p.y};
    // advective_flux(z, hu, zb*): F[e][d] = hu_e * velocity(z, hu, zb*)_d; with a
    // continuous bathymetry zb* = zb_m = zb_p and the inverse depths are the ones above
    T sm = s_m, sp = s_p;
    if (!FLAT && zb_m != zb_p)
      {
        sm = inv_depth(hm);
        sp = inv_depth(hp);
      }
    const Vec2<T> w_m = {hu_m.x * sm, hu_m.y * sm};
    const Vec2<T> w_p = {hu_p.x * sp, hu_p.y * sp};
    const T wn_m = dot_n(w_m, n);
    const T wn_p = dot_n(w_p, n);
    const T hl = T(0.5) * lambda;
    if (BOUNDARY)
      return {two_products(hl, hu_m.x - hu_p.x, T(0.5), two_products(hu_p.x, wn_p, hu_m.x, wn_m)),
              two_products(hl, hu_m.y - hu_p.y, T(0.5), two_products(hu_p.y, wn_p, hu_m.y, wn_m))};
    return {two_products(T(0.5), two_products(hu_m.x, wn_m, hu_p.x, wn_p), hl, hu_m.x - hu_p.x),
            two_products(T(0.5), two_products(hu_m.y, wn_m, hu_p.y, wn_p), hl, hu_m.y - hu_p.y)};
  }

  // NumericalFluxBase::numerical_presflux_strong, CENTER variant
  __device__ __forceinline__ Vec2<T> pres_flux(T z_m, T z_p, Vec2<T> n, T zb_m, T zb_p) const
  {
    const T zbs = zb_m < zb_p ? zb_m : zb_p;
    const T hp = depth(z_p, zbs), hm = depth(z_m, zbs);
    const T zcm = z_m > -zbs ? z_m : -zbs;
    const T zcp = z_p > -zbs ? z_p : -zbs;
    const T s = g * T(0.25) * (hp + hm) * (zcp - zcm);
    // s * n, with the zero component of an axis-aligned normal left zero
    return {n.x == T(0) ? T(0) : s * n.x, n.y == T(0) ? T(0) : s * n.y};
  }

  __device__ __forceinline__ T riemann_p(T z, Vec2<T> q, Vec2<T> n, T zb) const
  {
    const Vec2<T> v = velocity(z, q, zb);
    return dot_n(v, n) + T(2) * wave_speed(z, zb);
  }
  __device__ __forceinline__ T riemann_m(T z, Vec2<T> q, Vec2<T> n, T zb) const
  {
    const Vec2<T> v = velocity(z, q, zb);
    return dot_n(v, n) - T(2) * wave_speed(z, zb);
  }
};

}  // namespace oceano
