// fl_numerics_fast.hpp -- the per-cell Euler numerics in their fast form.
//
// The same MUSCL-Hancock / HLLC / FORCE formulas as fl_numerics.hpp, written
// for fewer instructions instead of the reference's rounding:
//   - each state's 1/rho is formed once (v_rcp_f64 and one Newton step,
//     within about an ulp) and every quotient by rho becomes a product; other
//     quotients are a * (1/b) the same way (FP32: v_rcp_f32);
//   - square roots take one Goldschmidt step and one correction after
//     v_rsq_f64 (FP32: v_sqrt_f32);
//   - the van Leer slope is its closed form: with r = b/f,
//     (b + f)/2 * 2 min(r, 1)/(1 + r) equals b when 0 < r <= 1 and f when
//     r > 1, i.e. minmod(b, f): no division and no branch (written as the
//     median of b, f and 0 with v_min/v_max and v_med3 it is 1 to 1.5 percent
//     of a sweep faster, but passes a NaN difference over: FP32 1024^2, 16
//     steps, 785 against 796 us, fast FP64 4096^2, 4 steps, 2918 against 2940);
//   - an ideal gas's shock speed a sqrt(1 + q (p*/p - 1)) is one root of
//     gamma/rho (p + q (p* - p)), without the quotient;
//   - multiply-adds are FMAs, written out: the compiler contracts within a
//     basic block only, so left to it the rounding would depend on the kernel
//     that a formula is inlined into, and the step loops, batches and launch
//     shapes would differ in their last bits.
// Results differ from the reference's in the last bits of each operation; the
// FP64 fast path is held to 1e-12 relative L-inf of the reference's results
// over a 100-step run.  FP32 uses these forms always.  Branches (limiter
// signs, flattening threshold, HLLC wave ordering) are the reference's.
// Measured (FP64 HLLC, 4096^2, 4 steps): 2950 us with the quotient forms the
// compiler contracted, 2950 us with these: the same speed, with bits that do
// not depend on the kernel.
#pragma once

#include "fl_numerics.hpp"

namespace fl {
namespace fast {

// Newton steps refining v_rcp_f64: one (about an ulp; tuning builds: 2).
#ifndef FL_FAST_NEWTON
#define FL_FAST_NEWTON 1
#endif

__device__ __forceinline__ double rcp(double b) {
  double r = __builtin_amdgcn_rcp(b);
  double e = __builtin_fma(-b, r, 1.0);
  r = __builtin_fma(r, e, r);
#if FL_FAST_NEWTON > 1
  e = __builtin_fma(-b, r, 1.0);
  r = __builtin_fma(r, e, r);
#endif
  return r;
}
__device__ __forceinline__ float rcp(float b) { return __builtin_amdgcn_rcpf(b); }

// Square root.  FP64 with FL_FAST_SQRT (default): v_rsq_f64, one Goldschmidt
// step and one residual correction (the IEEE sequence's second correction and
// its half-inverse-root refinement left out); +-0 and +inf return x.
// FL_FAST_SQRT=0: the correctly rounded fl::sq.  FP32: v_sqrt_f32.
#ifndef FL_FAST_SQRT
#define FL_FAST_SQRT 1
#endif

__device__ __forceinline__ double sqt(double x) {
#if FL_FAST_SQRT
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y;
  const double h = y * 0.5;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  const double d = __builtin_fma(-g, g, x);
  g = __builtin_fma(d, h, g);
  return __builtin_amdgcn_class(x, 0x260) ? x : g;
#else
  return sq(x);
#endif
}
__device__ __forceinline__ float sqt(float x) { return sq(x); }

template <typename T> __device__ __forceinline__ T div(T a, T b) { return a * rcp(b); }

// Minimum and maximum as single v_min/v_max instructions.  They differ from
// the comparison-based fl::smin/smax only in which operand a NaN or a signed
// zero leaves: a NaN operand yields the other one, as std::min(max, NaN) and
// std::max(0, NaN) do where the reference uses them to clamp.
__device__ __forceinline__ double mn(double a, double b) { return __builtin_fmin(a, b); }
__device__ __forceinline__ double mx(double a, double b) { return __builtin_fmax(a, b); }
__device__ __forceinline__ float mn(float a, float b) { return __builtin_fminf(a, b); }
__device__ __forceinline__ float mx(float a, float b) { return __builtin_fmaxf(a, b); }

// a b + c with one rounding.
__device__ __forceinline__ double fma(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// minmod(a, b); 0 where one of them is NaN, so that a cell that is not a number
// takes no slope from its neighbours to the next.
template <typename T>
__device__ __forceinline__ T minmod(T a, T b) {
  const T m = fabs(a) <= fabs(b) ? a : b;
  return a * b > T(0) ? m : T(0);
}

// Primitive quantities and 1/rho of one conservative state.
template <typename T, int ND> struct PrimR {
  T vel[ND];
  T p;
  T rinv;
};

// FIRST: the velocity component whose square is rounded before the others'
// are added to it (the last, unless said otherwise).
template <typename T, int ND, int FIRST = ND - 1>
__device__ __forceinline__ PrimR<T, ND> prim_of(const T* U, const Material<T>& m) {
  PrimR<T, ND> w;
  w.rinv = fast::rcp(U[0]);
#pragma unroll
  for (int i = 0; i < ND; ++i) w.vel[i] = U[2 + i] * w.rinv;
  T sum = w.vel[FIRST] * w.vel[FIRST];
#pragma unroll
  for (int i = ND - 1; i >= 0; --i)
    if (i != FIRST) sum = fast::fma(w.vel[i], w.vel[i], sum);
  const T e = fast::fma(T(-0.5) * U[0], sum, U[1]);
  w.p = m.corr ? fast::fma(m.gm1, e, -m.gpinf) : m.gm1 * e;
  return w;
}

template <typename T, int ND>
__device__ __forceinline__ Prim<T, ND> as_prim(const PrimR<T, ND>& w) {
  Prim<T, ND> o;
#pragma unroll
  for (int i = 0; i < ND; ++i) o.vel[i] = w.vel[i];
  o.p = w.p;
  return o;
}

template <typename T>
__device__ __forceinline__ T sound_speed(T p, T rinv, const Material<T>& m) {
  if (m.stiff) return fast::sqt(m.gamma * (p + m.p_inf) * rinv);
  return fast::sqt(m.gamma * p * rinv);
}

template <typename T, int ND, int D>
__device__ __forceinline__ void euler_flux(const T* U, const PrimR<T, ND>& w, T* F) {
  const T v = w.vel[D];
  F[0] = U[2 + D];
  F[2 + D] = fast::fma(U[2 + D], v, w.p);
  F[1] = v * (U[1] + w.p);
#pragma unroll
  for (int o = 0; o < ND; ++o)
    if (o != D) F[2 + o] = U[2 + o] * v;
}

template <typename T, int ND>
__device__ __forceinline__ T max_wavespeed(const PrimR<T, ND>& w, const Material<T>& m) {
  T mv = fabs(w.vel[0]);
#pragma unroll
  for (int i = 1; i < ND; ++i) mv = fast::mx(mv, T(fabs(w.vel[i])));
  return mv + fast::sound_speed(w.p, w.rinv, m);
}

// Superbee's limit (superbee_limiter.hpp:72-89) of the ratio a / b.
template <typename T>
__device__ __forceinline__ T superbee(T a, T b) {
  const T r = fast::div(a, b);
  if (r <= T(0) || b == T(0)) return T(0);
  if (r <= T(0.5)) return T(2) * r;
  if (r <= T(1)) return T(1);
  return fast::mn(fast::div(T(2), T(1) + r), fast::mn(r, T(2)));
}

// The limited slope (back + fwrd)/2 * limit(back, fwrd) of one component,
// conservative form (limiting/limiter.hpp:79-97).  van Leer
// (van_leer_limiter.hpp:65-74) in closed form: minmod(back, fwrd).
template <typename T>
__device__ __forceinline__ T slope_cons(int limiter, T back, T fwrd) {
  if (limiter == kLimSuperbee) return (back + fwrd) * T(0.5) * fast::superbee(back, fwrd);
  return fast::minmod(back, fwrd);
}

// Primitive form: the limit of the primitive differences (rb, rf) scales the
// average of the conservative ones (limiting/limiter.hpp:79-97).
template <typename T>
__device__ __forceinline__ T slope_prim(int limiter, T back, T fwrd, T rb, T rf) {
  const T avg = (back + fwrd) * T(0.5);
  if (limiter == kLimSuperbee) return avg * fast::superbee(rb, rf);
  if (!(rb * rf > T(0))) return T(0);
  // 2 min(r, 1) / (1 + r) with r = rb / rf: 2 rb / (rf + rb) or 2 rf / (rf + rb)
  const T m = (fabs(rb) <= fabs(rf)) ? rb : rf;
  return avg * fast::div(T(2) * m, rf + rb);
}

template <typename T>
__device__ __forceinline__ T chi_factor(T p_pprev, T p_prev, T p_next, T p_nnext, T v_prev,
                                        T v_next, const Material<T>& m) {
  const T u_factor = v_prev - v_next;
  const T dp = fabs(p_next - p_prev);
  T pmin = fast::mn(p_next, p_prev);
  if (m.corr) pmin = pmin + m.p_inf;
  // dp / pmin > 0.33 without the quotient: for pmin > 0 it is dp > 0.33 pmin;
  // pmin = 0 gives +inf (dp > 0) or NaN (dp = 0); pmin < 0 a quotient <= 0;
  // a NaN operand fails every comparison.
  const bool flatten = u_factor > T(0) && pmin >= T(0) && dp > T(0.33) * pmin;
  if (!flatten) return T(1);
  const T z = fast::div(dp, T(fabs(p_nnext - p_pprev)));
  const T temp = fast::fma(T(0.75) - z, T(10), T(1));
  return fast::mn(T(1), fast::mx(T(0), temp));
}

// Both evolved face states of one cell (reconstruction/muscl_reconstructor.hpp:
// 99-172), as fl::evolve_faces.
template <typename T, int ND, int D>
__device__ __forceinline__ void evolve_faces(const T* um, const T* u0, const T* up, T chi,
                                             T half_dtdh, int limiter, int form,
                                             const Material<T>& m, T* R, T* L) {
  constexpr int S = 2 + ND;
  T rb[S], rf[S];
  if (form == kFormPrim) {
    const PrimR<T, ND> wm = fast::prim_of<T, ND>(um, m);
    const PrimR<T, ND> w0 = fast::prim_of<T, ND>(u0, m);
    const PrimR<T, ND> wp = fast::prim_of<T, ND>(up, m);
    rb[0] = u0[0] - um[0];
    rf[0] = up[0] - u0[0];
    rb[1] = w0.p - wm.p;
    rf[1] = wp.p - w0.p;
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      rb[2 + i] = w0.vel[i] - wm.vel[i];
      rf[2 + i] = wp.vel[i] - w0.vel[i];
    }
  }
  const T cscale = chi * T(0.5);
  T plus[S], minus[S];
#pragma unroll
  for (int k = 0; k < S; ++k) {
    const T back = u0[k] - um[k];
    const T fwrd = up[k] - u0[k];
    const T lim = (form == kFormPrim) ? fast::slope_prim(limiter, back, fwrd, rb[k], rf[k])
                                      : fast::slope_cons(limiter, back, fwrd);
    plus[k] = fast::fma(lim, cscale, u0[k]);
    minus[k] = fast::fma(-lim, cscale, u0[k]);
  }
  const PrimR<T, ND> wmi = fast::prim_of<T, ND>(minus, m);
  const PrimR<T, ND> wpl = fast::prim_of<T, ND>(plus, m);
  // F(minus) - F(plus)
  const T vm = wmi.vel[D], vp = wpl.vel[D];
  T df[S];
  df[0] = minus[2 + D] - plus[2 + D];
  df[1] = fast::fma(vm, minus[1] + wmi.p, -(vp * (plus[1] + wpl.p)));
#pragma unroll
  for (int i = 0; i < ND; ++i)
    df[2 + i] = i == D ? fast::fma(minus[2 + D], vm, wmi.p) - fast::fma(plus[2 + D], vp, wpl.p)
                       : fast::fma(minus[2 + i], vm, -(plus[2 + i] * vp));
  // FP32 rounds the increment of one of the two states first (x: R, y: L), as
  // FP32 results always have; FP64 rounds once
  constexpr bool f64 = sizeof(T) == 8;
#pragma unroll
  for (int k = 0; k < S; ++k) {
    R[k] = f64 || D == 1 ? fast::fma(df[k], half_dtdh, plus[k]) : plus[k] + df[k] * half_dtdh;
    L[k] = f64 || D == 0 ? fast::fma(df[k], half_dtdh, minus[k]) : minus[k] + df[k] * half_dtdh;
  }
}

// u + side * (the sound speed, or the shock's where p* > p), side = -1 or +1.
// The ideal gas's FP64 form has no quotient; FP32 keeps the one it has, whose
// reciprocal and root are one instruction each.
template <typename T>
__device__ __forceinline__ T hllc_wavespeed(T u, T p, T rinv, T pstar, T sound, T side,
                                            const Material<T>& m) {
  if (pstar <= p) return u + side * sound;
  if (m.corr)
    return u + side * (sound * fast::sqt(fast::fma(
                                   m.q, fast::div(pstar + m.p_inf, p + m.p_inf) - T(1), T(1))));
  if (sizeof(T) == 4 || m.stiff)
    return u + side * (sound * fast::sqt(fast::fma(m.q, fast::div(pstar, p) - T(1), T(1))));
  return u + side * fast::sqt(m.gamma * rinv * fast::fma(m.q, pstar - p, p));
}

// HLLC (flux_method/flux_hllc.hpp:82-245), as fl::hllc_flux.
template <typename T, int ND, int D>
__device__ __forceinline__ void hllc_flux(const T* ul, const T* ur, const Material<T>& m,
                                          T* F) {
  constexpr int S = 2 + ND;
  // (the left state of an FP32 x face sums its squares from vel[0], as FP32
  // results always have)
  const PrimR<T, ND> wl = fast::prim_of<T, ND, sizeof(T) == 4 && D == 0 ? 0 : ND - 1>(ul, m);
  const PrimR<T, ND> wr = fast::prim_of<T, ND>(ur, m);
  const T al = fast::sound_speed(wl.p, wl.rinv, m);
  const T ar = fast::sound_speed(wr.p, wr.rinv, m);
  const T vl = wl.vel[D], vr = wr.vel[D];
  const T p_pvrs =
      T(0.5) * fast::fma(T(-0.25) * fast::fma(ur[2 + D], wr.rinv, -vl) * (ur[0] + ul[0]), al + ar,
                         wl.p + wr.p);
  const T p_star = m.corr ? fast::mx(-m.p_inf, p_pvrs) : fast::mx(T(0), p_pvrs);

  const T wsl = fast::hllc_wavespeed(vl, wl.p, wl.rinv, p_star, al, T(-1), m);
  if (T(0) <= wsl) {
    fast::euler_flux<T, ND, D>(ul, wl, F);
    return;
  }
  const T wsr = fast::hllc_wavespeed(vr, wr.p, wr.rinv, p_star, ar, T(1), m);
  if (T(0) >= wsr) {
    fast::euler_flux<T, ND, D>(ur, wr, F);
    return;
  }
  const T factorl = ul[0] * (wsl - vl);
  const T factorr = ur[0] * (wsr - vr);
  const T ws_star = fast::div(fast::fma(-vr, factorr, fast::fma(vl, factorl, wr.p - wl.p)),
                              fast::fma(ul[0], wsl - vl, -factorr));

  const bool left = T(0) <= ws_star;
  const T* st = left ? ul : ur;
  const PrimR<T, ND>& w = left ? wl : wr;
  const T ws = left ? wsl : wsr;
  const T state_factor = ws - w.vel[D];
  // 1/(ws - ws_star) and 1/state_factor from one reciprocal of their product
  const T rr = fast::rcp((ws - ws_star) * state_factor);
  const T scale_factor = state_factor * state_factor * rr;
  const T inv_sf = (ws - ws_star) * rr;
  // star state minus state
  T d[S];
#pragma unroll
  for (int k = 0; k < S; ++k) d[k] = fast::fma(st[k], scale_factor, -st[k]);
  d[2 + D] = fast::fma(ws_star * st[0], scale_factor, -st[2 + D]);
  d[1] = fast::fma(scale_factor,
                   fast::fma(st[0] * (ws_star - w.vel[D]),
                             fast::fma(w.p * w.rinv, inv_sf, ws_star), st[1]),
                   -st[1]);
#pragma unroll
  for (int i = 0; i < ND; ++i)
    F[2 + i] = i == D ? fast::fma(d[2 + D], ws, fast::fma(st[2 + D], w.vel[D], w.p))
                      : fast::fma(st[2 + i], w.vel[D], d[2 + i] * ws);
  F[0] = fast::fma(d[0], ws, st[2 + D]);
  F[1] = fast::fma(w.vel[D], st[1] + w.p, d[1] * ws);
}

template <typename T, int ND, int D>
__device__ __forceinline__ void force_flux(const T* ul, const T* ur, T dtdh, T dhdt,
                                           const Material<T>& m, T* F) {
  constexpr int S = 2 + ND;
  const PrimR<T, ND> wl = fast::prim_of<T, ND>(ul, m);
  const PrimR<T, ND> wr = fast::prim_of<T, ND>(ur, m);
  T fl[S], fr[S], uri[S];
  fast::euler_flux<T, ND, D>(ul, wl, fl);
  fast::euler_flux<T, ND, D>(ur, wr, fr);
#pragma unroll
  for (int k = 0; k < S; ++k)
    uri[k] = fast::fma(fl[k] - fr[k], dtdh, ul[k] + ur[k]) * T(0.5);
  const PrimR<T, ND> wri = fast::prim_of<T, ND>(uri, m);
  T fri[S];
  fast::euler_flux<T, ND, D>(uri, wri, fri);
#pragma unroll
  for (int k = 0; k < S; ++k) {
    const T lf2 = fast::fma(ul[k] - ur[k], dhdt, fl[k] + fr[k]);
    F[k] = fast::fma(T(0.5), lf2, fri[k]) * T(0.5);
  }
}

template <typename T, int ND, int D>
__device__ __forceinline__ void lax_friedrichs_flux(const T* ul, const T* ur, T dhdt,
                                                    const Material<T>& m, T* F) {
  constexpr int S = 2 + ND;
  const PrimR<T, ND> wl = fast::prim_of<T, ND>(ul, m);
  const PrimR<T, ND> wr = fast::prim_of<T, ND>(ur, m);
  T fl[S], fr[S];
  fast::euler_flux<T, ND, D>(ul, wl, fl);
  fast::euler_flux<T, ND, D>(ur, wr, fr);
#pragma unroll
  for (int k = 0; k < S; ++k)
    F[k] = fast::fma(ul[k] - ur[k], dhdt, fl[k] + fr[k]) * T(0.5);
}

template <typename T, int ND, int D>
__device__ __forceinline__ void richtmyer_flux(const T* ul, const T* ur, T dtdh,
                                               const Material<T>& m, T* F) {
  constexpr int S = 2 + ND;
  const PrimR<T, ND> wl = fast::prim_of<T, ND>(ul, m);
  const PrimR<T, ND> wr = fast::prim_of<T, ND>(ur, m);
  T fl[S], fr[S], uri[S];
  fast::euler_flux<T, ND, D>(ul, wl, fl);
  fast::euler_flux<T, ND, D>(ur, wr, fr);
#pragma unroll
  for (int k = 0; k < S; ++k)
    uri[k] = fast::fma(fl[k] - fr[k], dtdh, ul[k] + ur[k]) * T(0.5);
  const PrimR<T, ND> wri = fast::prim_of<T, ND>(uri, m);
  fast::euler_flux<T, ND, D>(uri, wri, F);
}

template <typename T, int ND, int D, int FLUX>
__device__ __forceinline__ void numerical_flux(const T* ul, const T* ur, T dtdh, T dhdt,
                                               const Material<T>& m, T* F) {
  if constexpr (FLUX == kFluxHllc) {
    fast::hllc_flux<T, ND, D>(ul, ur, m, F);
  } else if constexpr (FLUX == kFluxLaxFriedrichs) {
    fast::lax_friedrichs_flux<T, ND, D>(ul, ur, dhdt, m, F);
  } else if constexpr (FLUX == kFluxRichtmyer) {
    fast::richtmyer_flux<T, ND, D>(ul, ur, dtdh, m, F);
  } else {
    fast::force_flux<T, ND, D>(ul, ur, dtdh, dhdt, m, F);
  }
}

}  // namespace fast
}  // namespace fl
