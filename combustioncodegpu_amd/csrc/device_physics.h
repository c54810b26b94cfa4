// device_physics.h — point-wise physics on the device: NASA-7 thermo,
// Chapman–Enskog/Wilke transport, limiters, the AUSM+ face flux with MUSCL
// reconstruction and the central viscous face flux.  Templated on the
// species count NS (compile time, so all species loops unroll and the
// species table is read with uniform scalar loads) and on the arithmetic
// type R of the flux/transport work (double for the plain path, float for
// the mixed-precision path).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "cfx_types.h"

namespace cfx {

// f(integral_constant<int, I>) for I = 0..N-1, unrolled at compile time.
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// The species table is read through the constant address space: every index
// into it is uniform across the wavefront, so the loads become scalar loads
// into SGPRs instead of vector loads into VGPRs.
template <typename R>
using SpeciesPtrT = const __attribute__((address_space(4))) SpeciesT<R> *;

template <typename R>
__device__ __forceinline__ SpeciesPtrT<R> const_table(const SpeciesDev *p);
template <>
__device__ __forceinline__ SpeciesPtrT<double> const_table<double>(const SpeciesDev *p) {
  return (SpeciesPtrT<double>)&p->d;
}
template <>
__device__ __forceinline__ SpeciesPtrT<float> const_table<float>(const SpeciesDev *p) {
  return (SpeciesPtrT<float>)&p->f;
}

template <typename R>
struct Tiny;
template <>
struct Tiny<double> {
  static constexpr double v = 1e-300;
};
template <>
struct Tiny<float> {
  static constexpr float v = 1e-30f;
};

// Division, reciprocal and square root of the flux work.  FP64: the hardware
// reciprocal (v_rcp_f64) refined by two Newton steps, r <- r + r (1 - b r),
// and the quotient corrected once, q <- q + r (a - b q): within an ulp of the
// IEEE quotient for the normal, finite operands of the flux work (positive
// denominators well inside the exponent range), without the scaling and
// fix-up steps the IEEE sequence spends on special values.  FP32 (mixed
// precision): the hardware reciprocal and square root (v_rcp_f32,
// v_sqrt_f32, 1 ulp), far below the FP32 rounding already accepted there.
template <typename R>
__device__ __forceinline__ R frcp(R a) { return R(1) / a; }
template <>
__device__ __forceinline__ double frcp<double>(double b) {
  double r = __builtin_amdgcn_rcp(b);
  double e = fma(-b, r, 1.0);
  r = fma(r, e, r);
  e = fma(-b, r, 1.0);
  return fma(r, e, r);
}
template <>
__device__ __forceinline__ float frcp<float>(float a) { return __builtin_amdgcn_rcpf(a); }
template <typename R>
__device__ __forceinline__ R fdiv(R a, R b) { return a / b; }
template <>
__device__ __forceinline__ double fdiv<double>(double a, double b) {
  const double r = frcp<double>(b);
  const double q = a * r;
  return fma(r, fma(-b, q, a), q);
}
template <>
__device__ __forceinline__ float fdiv<float>(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
template <typename R>
__device__ __forceinline__ R fsqrt(R a) { return sqrt(a); }
template <>
__device__ __forceinline__ float fsqrt<float>(float a) { return __builtin_amdgcn_sqrtf(a); }
// exp and log of the transport work: the library functions in FP64; in FP32
// e^a = 2^(a log2 e) and ln a = log2(a) ln 2 with the hardware exp2/log2
// (v_exp_f32, v_log_f32), for the moderate arguments of the transport
// (|a| < 10 in exp, temperatures in log) within a few ulp.
template <typename R>
__device__ __forceinline__ R fexp(R a) { return exp(a); }
template <>
__device__ __forceinline__ float fexp<float>(float a) { return __builtin_amdgcn_exp2f(a * 1.4426950408889634f); }
template <typename R>
__device__ __forceinline__ R flog(R a) { return log(a); }
template <>
__device__ __forceinline__ float flog<float>(float a) { return __builtin_amdgcn_logf(a) * 0.6931471805599453f; }

// N quotients or square roots at once, each step over all of them before the next:
// an FP64 chain of dependent operations leaves most issue slots of a wavefront empty
// (two wavefronts share a SIMD in the FP64 kernels), and the compiler keeps the order
// in which chains are written.  The quotients take one Newton step less than fdiv:
// with r within 2^-40 of 1/b the residual correction q + r (a - b q) leaves nothing
// but its own rounding (2^-80 of q), whatever the second step adds.
template <int N, typename R>
__device__ __forceinline__ void fdiv_n(const R *a, const R *b, R *q) {
  R r[N], e[N];
  if constexpr (sizeof(R) == 8) {
#pragma unroll
    for (int n = 0; n < N; ++n) r[n] = __builtin_amdgcn_rcp(b[n]);
#pragma unroll
    for (int n = 0; n < N; ++n) e[n] = fma(-b[n], r[n], R(1));
#pragma unroll
    for (int n = 0; n < N; ++n) r[n] = fma(r[n], e[n], r[n]);
  } else {
#pragma unroll
    for (int n = 0; n < N; ++n) r[n] = frcp<R>(b[n]);
  }
#pragma unroll
  for (int n = 0; n < N; ++n) q[n] = a[n] * r[n];
  if constexpr (sizeof(R) == 8) {
#pragma unroll
    for (int n = 0; n < N; ++n) e[n] = fma(-b[n], q[n], a[n]);
#pragma unroll
    for (int n = 0; n < N; ++n) q[n] = fma(r[n], e[n], q[n]);
  }
}
// sqrt(a) and 1/sqrt(a) of operands well inside the exponent range.  FP64: one
// hardware reciprocal square root, g -> sqrt(a), h -> 1/(2 sqrt(a)) by the coupled
// Newton iteration e = 1/2 - g h, g += g e, h += h e, and two residual corrections
// of g (no scaling and special-value steps, as for fdiv: the root of 0 or infinity
// is NaN, and the caller's to replace where it can occur).
template <int N, typename R>
__device__ __forceinline__ void fsqrt_n(const R *a, R *g, R *rs) {
  if constexpr (sizeof(R) == 8) {
    R h[N], e[N];
#pragma unroll
    for (int n = 0; n < N; ++n) h[n] = __builtin_amdgcn_rsq(a[n]);
#pragma unroll
    for (int n = 0; n < N; ++n) g[n] = a[n] * h[n];
#pragma unroll
    for (int n = 0; n < N; ++n) h[n] = R(0.5) * h[n];
#pragma unroll
    for (int n = 0; n < N; ++n) e[n] = fma(-h[n], g[n], R(0.5));
#pragma unroll
    for (int n = 0; n < N; ++n) g[n] = fma(g[n], e[n], g[n]);
#pragma unroll
    for (int n = 0; n < N; ++n) h[n] = fma(h[n], e[n], h[n]);
#pragma unroll
    for (int n = 0; n < N; ++n) e[n] = fma(-h[n], g[n], R(0.5));
#pragma unroll
    for (int n = 0; n < N; ++n) h[n] = fma(h[n], e[n], h[n]);
#pragma unroll
    for (int it = 0; it < 2; ++it) {
#pragma unroll
      for (int n = 0; n < N; ++n) e[n] = fma(-g[n], g[n], a[n]);
#pragma unroll
      for (int n = 0; n < N; ++n) g[n] = fma(e[n], h[n], g[n]);
    }
#pragma unroll
    for (int n = 0; n < N; ++n) rs[n] = h[n] + h[n];
  } else {
#pragma unroll
    for (int n = 0; n < N; ++n) g[n] = fsqrt<R>(a[n]), rs[n] = frcp<R>(g[n]);
  }
}

// ---------------------------------------------------------------- thermo ---
// h_l(T) and cp_l(T) of one species (Thermo.cu:27-47): NASA-7 polynomial in
// Horner form with the low/high set chosen at t_mid and the linear enthalpy
// extension with frozen cp below t_low.  The coefficients are wave-uniform
// (one record per species); T varies per lane.  Both ranges are evaluated
// with uniform operands and the two results selected per lane: selecting per
// coefficient instead costs a move and a select for each one, or (if the
// compiler folds the select into the loads) a vector load from a per-lane
// address.  The chosen value is bit-for-bit the same.

// Marks v as computed on every lane at this point.  Without it the compiler
// turns the selects below into branches and sinks the polynomial work (and
// its coefficient loads, each with its own wait) into them.
template <typename R>
__device__ __forceinline__ R on_all_lanes(R v) {
  asm volatile("" : "+v"(v));
  return v;
}

// The NASA-7 ranges of a wavefront's temperatures t0, t1: kRangeHi (every species
// in its high set), kRangeLo (every one in its low set, above t_low), kRangeEach
// (each temperature in one of the two), or kRangeAny (some below a t_low, or
// between the species' t_mid).  It chooses where the coefficients are read, never
// the value: the sums are the same ones in the same order, whatever the other
// lanes hold.  (A face on the seam of two tiles is formed in both, next to other
// faces, and its two fluxes have to be the same bits.)  97x61x75 cells with 9
// species and temperatures on both sides of t_low: 21.5 ms per 20 FP64 steps; with a
// sum over the species for the temperatures outside the ranges, beside the
// polynomial of the others, 22.9.
constexpr int kRangeAny = 0, kRangeLo = 1, kRangeHi = 2, kRangeEach = 3;
template <typename R>
__device__ __forceinline__ int thermo_range(SpeciesPtrT<R> sp, R t0, R t1) {
  const R hf = R(sp->hi_from), lf = R(sp->lo_from), lt = R(sp->lo_to);
  const bool h0 = t0 >= hf, h1 = t1 >= hf, l0 = t0 >= lf && t0 < lt, l1 = t1 >= lf && t1 < lt;
  if (__all(h0 && h1)) return kRangeHi;
  if (__all(l0 && l1)) return kRangeLo;
  if (__all((h0 || l0) && (h1 || l1))) return kRangeEach;
  return kRangeAny;
}

// h and cp of one species from its thermo record c, each lane in its own range
template <typename R, typename C>
__device__ __forceinline__ void thermo_h_cp(const C &c, R t, R &h, R &cp) {
  auto p5 = [&](int o) { return R(c[o]) + t * (R(c[o + 1]) + t * (R(c[o + 2]) + t * (R(c[o + 3]) + t * R(c[o + 4])))); };
  const R cp_lo = p5(kThCp), cp_hi = p5(kThCp + 5);
  const R h_lo = t * p5(kThH) + R(c[kThH + 5]);
  const R h_hi = t * p5(kThH + 6) + R(c[kThH + 11]);
  const bool hi = t >= R(c[kThTmid]);
  const R cpp = on_all_lanes<R>(hi ? cp_hi : cp_lo);
  const R hp = on_all_lanes<R>(hi ? h_hi : h_lo);
  const R tl = R(c[kThTlow]);
  const bool below = t < tl;
  cp = below ? R(c[kThCptlow]) : cpp;
  h = below ? R(c[kThHtlow]) + R(c[kThCptlow]) * (t - tl) : hp;
}

template <typename R>
__device__ __forceinline__ void species_h_cp(SpeciesPtrT<R> sp, int l, R t, R &h, R &cp) {
  thermo_h_cp<R>(sp->th[l].v, t, h, cp);
}

// The mixture coefficients of a kernel: a copy of the table in LDS (3 x NS
// records of 8: low sets, high sets, below t_low).  Read as constant memory only a
// few records fit the scalar registers, so that every one or two species wait for a
// scalar load; the LDS copy (broadcast reads) keeps many reads in flight, and lets
// each lane have a range of its own: an FP64 RHS wavefront's AUSM+ phase took
// 3.4k cycles with scalar loads, of which it issued 1.6k.
template <int NS, typename R>
struct ThermoLds {
  SpeciesPtrT<R> sp;
  const R *lds;
  __device__ const R *mix(bool hi) const { return lds + (hi ? NS * 8 : 0); }
  // species l's record at temperature t
  __device__ const R *rec(int l, R t) const {
    return lds + 8 * l + (t < R(sp->t_low[l]) ? 2 * NS * 8 : (t >= R(sp->t_mid[l]) ? NS * 8 : 0));
  }
};

// H_k = sum_l w_l h_{l,k}, k = 0..5, with the coefficients of range rg at
// temperature t (by lane with kRangeEach, by lane and species with kRangeAny), N
// sums at once over the weights w(n, l).  The fused products are written out: left
// to the compiler, a branch may round x0 c0 + x1 c1 the other way round.
template <int NS, int N, typename R, typename TH, typename W>
__device__ __forceinline__ void mixture_sum(const TH &th, int rg, const R *t, W w, R (*H)[6]) {
  auto add = [&](const R *c, int n, int l) {
    const R x = w(n, l);
#pragma unroll
    for (int k = 0; k < 6; ++k) H[n][k] = l == 0 ? x * c[k] : fma(x, c[k], H[n][k]);
  };
  const R hf = R(th.sp->hi_from);
  if (rg == kRangeAny) {
#pragma unroll
    for (int l = 0; l < NS; ++l) {
#pragma unroll
      for (int n = 0; n < N; ++n) {
        add(th.rec(l, t[n]), n, l);
        // (else the branches' sums are merged into one with every record in registers)
        asm volatile("" : "+v"(H[n][0]), "+v"(H[n][1]), "+v"(H[n][2]), "+v"(H[n][3]), "+v"(H[n][4]), "+v"(H[n][5]));
      }
    }
    return;
  }
  if (N > 1 && rg == kRangeEach) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const R *tab = th.mix(t[n] >= hf);
#pragma unroll
      for (int l = 0; l < NS; ++l) add(tab + 8 * l, n, l);
    }
    return;
  }
  const R *tab = th.mix(N == 1 ? t[0] >= hf : rg == kRangeHi);
#pragma unroll
  for (int l = 0; l < NS; ++l)
#pragma unroll
    for (int n = 0; n < N; ++n) add(tab + 8 * l, n, l);
}

// h(T) and cp(T) = dh/dT of a mixture from its summed enthalpy coefficients
// H_k = sum_l Y_l h_{l,k} (k = 0..5, in the layout of the thermo records): cp's
// coefficients are (k + 1) H_k.
// N mixtures in lockstep.
template <int N, typename R>
__device__ __forceinline__ void mixture_h_cp(const R (*C)[6], const R *t, R *h, R *cp) {
#pragma unroll
  for (int n = 0; n < N; ++n) h[n] = C[n][3] + t[n] * C[n][4], cp[n] = R(4) * C[n][3] + t[n] * (R(5) * C[n][4]);
#pragma unroll
  for (int k = 2; k >= 0; --k)
#pragma unroll
    for (int n = 0; n < N; ++n) h[n] = C[n][k] + t[n] * h[n], cp[n] = R(k + 1) * C[n][k] + t[n] * cp[n];
#pragma unroll
  for (int n = 0; n < N; ++n) h[n] = C[n][5] + t[n] * h[n];
}

// sum_l w_l h_l(t), the enthalpy that the diffusive fluxes w_l carry
template <int NS, typename R, typename TH>
__device__ __forceinline__ R carried_enthalpy(const TH &th, R t, const R *w) {
  R H1[1][6];
  mixture_sum<NS, 1, R>(th, thermo_range<R>(th.sp, t, t), &t, [&](int, int l) { return w[l]; }, H1);
  const R *H = H1[0];
  return H[5] + t * (H[0] + t * (H[1] + t * (H[2] + t * (H[3] + t * H[4]))));
}

// cp_l(T) only, frozen below t_low (Thermo.cu:49-63).  Loops over species
// that need only cp read the per-array layout: the cp coefficients of all
// species are contiguous there and arrive in a few wide loads.
template <typename R>
__device__ __forceinline__ R species_cp(SpeciesPtrT<R> sp, int l, R t) {
  auto p5 = [&](const auto &c) { return R(c[0]) + t * (R(c[1]) + t * (R(c[2]) + t * (R(c[3]) + t * R(c[4])))); };
  R cpp;
  if constexpr (sizeof(R) == 4) {
    // both ranges from scalar loads, then a per-lane select
    const R lo = p5(sp->cpc[0][l]), hi = p5(sp->cpc[1][l]);
    cpp = on_all_lanes<R>(t >= R(sp->t_mid[l]) ? hi : lo);
  } else {
    cpp = t >= R(sp->t_mid[l]) ? p5(sp->cpc[1][l]) : p5(sp->cpc[0][l]);
  }
  return t < R(sp->t_low[l]) ? R(sp->cp_tlow[l]) : cpp;
}

// -------------------------------------------------------------- limiters ---
// N limited slopes in lockstep: minmod (Limiter.cuh:13-16), or Van Albada
// (MODE 1).  The slope is 0 where a and b differ in sign, and where one of them is
// NaN, so that a broken point reaches no face beyond its own.  minmod as
// min(max(a, 0), max(b, 0)) + max(min(a, 0), min(b, 0)), of which at most one is not
// 0 and which a NaN leaves at 0 (FP32: each a median); the outer difference of an
// even place is a, of an odd one b, and the terms of the other, which two slopes
// share, are formed once.  256x128x128 cells with 9 species, per evaluation: Van
// Albada 1.13 ms in FP64 and 0.59 mixed (1.09 and 0.58 where NaN went through),
// minmod 1.03 either way.
template <int MODE, int N, typename R>
__device__ __forceinline__ void limiter_n(const R *a, const R *b, R *s) {
  if constexpr (MODE == 1) {
    R ab[N], num[N], den[N];
#pragma unroll
    for (int n = 0; n < N; ++n) ab[n] = a[n] * b[n];
#pragma unroll
    for (int n = 0; n < N; ++n) den[n] = a[n] * a[n] + (b[n] * b[n] + Tiny<R>::v);
#pragma unroll
    for (int n = 0; n < N; ++n) num[n] = ab[n] * (a[n] + b[n]);
    fdiv_n<N, R>(num, den, s);
#pragma unroll
    for (int n = 0; n < N; ++n) s[n] = ab[n] > R(0) ? s[n] : R(0);
  } else {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const R o = n % 2 ? b[n] : a[n], m = n % 2 ? a[n] : b[n];
      const R mp = fmax(m, R(0)), mn = fmin(m, R(0));
      if constexpr (sizeof(R) == 4) s[n] = __builtin_amdgcn_fmed3f(o, R(0), mp) - __builtin_amdgcn_fmed3f(-o, R(0), -mn);
      else s[n] = fmin(fmax(o, R(0)), mp) + fmax(fmin(o, R(0)), mn);
    }
  }
}

// MUSCL kappa = 1/3 on one variable (Reconstruction.cu:26-44), or first
// order.  Both limiters are symmetric (Van Albada up to the rounding of its
// denominator), so the reference's four calls per face reduce to the two limited
// slopes of the two cells: (1-kappa)/4 + (1+kappa)/4 = 1/2.
// N variables in lockstep, q[n][0..3] the four points; MODE: 0 minmod, 1 Van
// Albada, 2 first order.
template <int MODE, int N, typename R>
__device__ __forceinline__ void muscl_n(const R (*q)[4], R *l, R *r) {
  if constexpr (MODE < 2) {
    R a[2 * N], b[2 * N], s[2 * N];
#pragma unroll
    for (int n = 0; n < N; ++n) {
      a[2 * n] = q[n][1] - q[n][0];
      b[2 * n] = a[2 * n + 1] = q[n][2] - q[n][1];
      b[2 * n + 1] = q[n][3] - q[n][2];
    }
    limiter_n<MODE, 2 * N, R>(a, b, s);
#pragma unroll
    for (int n = 0; n < N; ++n) {
      l[n] = q[n][1] + R(0.5) * s[2 * n];
      r[n] = q[n][2] - R(0.5) * s[2 * n + 1];
    }
  } else {
#pragma unroll
    for (int n = 0; n < N; ++n) l[n] = q[n][1], r[n] = q[n][2];
  }
}
// AUSM+ flux (InviscidScheme.cu:39-106) from the reconstructed face states
// pl/pr = (rho,u,v,w,p,Y..) and the face area vector k = 0.5(J_L grad_L +
// J_R grad_R) of the face direction; the face temperature, energy and gamma
// follow Reconstruction.cu:46-89.
template <int NS, typename R, typename TH>
__device__ __forceinline__ void ausm_from_states(SpeciesPtrT<R> sp, const TH &th, const SchemeDev &S, const R *pl,
                                                 const R *pr, R k1, R k2, R k3, R *F) {
  constexpr int NV = 5 + NS;
  // both sides in lockstep (index 0 left, 1 right).  H: specific total
  // enthalpy (E + p) / rho; c2: gamma p / rho, third entry |k|^2
  const R *const P[2] = {pl, pr};
  R H[2], c2[3], x[2], y[2];
#pragma unroll
  for (int n = 0; n < 2; ++n) H[n] = R(0.5) * (P[n][1] * P[n][1] + P[n][2] * P[n][2] + P[n][3] * P[n][3]);
  if constexpr (NS > 0) {
    R w[2] = {R(0), R(0)}, t[2], cp[2];
#pragma unroll
    for (int l = 0; l < NS; ++l)
#pragma unroll
      for (int n = 0; n < 2; ++n) w[n] += P[n][5 + l] * R(sp->inv_mw[l]);
#pragma unroll
    for (int n = 0; n < 2; ++n) w[n] *= R(kRu);  // gas constant of the mixture
#pragma unroll
    for (int n = 0; n < 2; ++n) x[n] = P[n][4], y[n] = P[n][0] * w[n];
    fdiv_n<2, R>(x, y, t);
    const int rg = thermo_range<R>(sp, t[0], t[1]);
    // the mixture's polynomial first (six coefficients, each summed over the
    // species), evaluated once, in place of one enthalpy and one cp polynomial per
    // species
    R C[2][6], h[2];
    mixture_sum<NS, 2, R>(th, rg, t, [&](int n, int l) { return P[n][5 + l]; }, C);
    mixture_h_cp<2, R>(C, t, h, cp);
#pragma unroll
    for (int n = 0; n < 2; ++n) H[n] += h[n];
#pragma unroll
    for (int n = 0; n < 2; ++n) x[n] = cp[n] * (w[n] * t[n]), y[n] = cp[n] - w[n];
    fdiv_n<2, R>(x, y, c2);  // gamma R T
  } else {
    R v[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) x[n] = P[n][4], y[n] = P[n][0];
    fdiv_n<2, R>(x, y, v);
    const R gam = R(S.gamma_air), g1 = R(S.gamma_air / (S.gamma_air - 1));
#pragma unroll
    for (int n = 0; n < 2; ++n) H[n] += g1 * v[n], c2[n] = gam * v[n];
  }
  c2[2] = k1 * k1 + k2 * k2 + k3 * k3;
  R g[3], rs[3];
  fsqrt_n<3, R>(c2, g, rs);
  if constexpr (sizeof(R) == 8) {  // the sound speed of a vacuum
#pragma unroll
    for (int n = 0; n < 2; ++n) g[n] = c2[n] == R(0) ? R(0) : g[n];
  }
  const R gk = g[2], c = R(0.5) * (g[0] + g[1]);
  const R ic = frcp<R>(c) * rs[2];  // 1 / (c |k|)
  R m[2], a[2], b[2];
#pragma unroll
  for (int n = 0; n < 2; ++n) m[n] = (k1 * P[n][1] + k2 * P[n][2] + k3 * P[n][3]) * ic;
  constexpr double alpha = 3 / 16.0;
  // split Mach numbers and pressures; beyond |M| = 1 the pressure split
  // M+-/M is 1 or 0 by the sign of M.  (M +- |M|, and not a maximum: of an infinite
  // M it leaves NaN, so that an infinite velocity reaches the flux on every side)
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const R o = n == 0 ? R(1) : R(-1);
    a[n] = (m[n] + o) * (m[n] + o) * R(0.25);
    b[n] = (m[n] * m[n] - R(1)) * (m[n] * m[n] - R(1));
  }
  const bool sl = fabs(m[0]) > R(1), sr = fabs(m[1]) > R(1);
  const R mlp = sl ? R(0.5) * (m[0] + fabs(m[0])) : a[0] + R(0.125) * b[0];
  const R mrn = sr ? R(0.5) * (m[1] - fabs(m[1])) : -a[1] - R(0.125) * b[1];
  const R plp = sl ? (m[0] > R(0) ? R(1) : R(0)) : a[0] * (R(2) - m[0]) + R(alpha) * m[0] * b[0];
  const R prn = sr ? (m[1] < R(0) ? R(1) : R(0)) : a[1] * (R(2) + m[1]) - R(alpha) * m[1] * b[1];
  const R p_coeff = plp * pl[4] + prn * pr[4];
  const R m_half = mlp + mrn;
  const R mpos = R(0.5) * (m_half + fabs(m_half));
  const R mneg = R(0.5) * (m_half - fabs(m_half));
  const R mass = c * (pl[0] * mpos + pr[0] * mneg);
  const R coeff = mass * gk;
  const bool left = mass >= R(0);
  F[0] = coeff;
  F[1] = coeff * (left ? pl[1] : pr[1]) + p_coeff * k1;
  F[2] = coeff * (left ? pl[2] : pr[2]) + p_coeff * k2;
  F[3] = coeff * (left ? pl[3] : pr[3]) + p_coeff * k3;
  F[4] = coeff * (left ? H[0] : H[1]);
#pragma unroll
  for (int l = 5; l < NV; ++l) F[l] = coeff * (left ? pl[l] : pr[l]);
}

}  // namespace cfx
