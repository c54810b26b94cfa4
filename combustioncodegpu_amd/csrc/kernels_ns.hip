// kernels_ns.hip — the kernels templated on the species count NS, compiled
// once per supported count (-DCFX_NS=n) and precision of the flux work
// (-DCFX_PREC=64: the FP64 set with the update, conversions and ghost fills;
// -DCFX_PREC=32: the FP32 properties and RHS of the mixed-precision path).
// Each build registers its launchers in g_kernels64[n] / g_kernels32[n].
#include <hip/hip_runtime.h>

#include <atomic>

#include "device_physics.h"
#include "kernels.h"
#include "lusgs_plan.h"
#include "mlp.h"
#include "rhs_march.h"
#include "rhs_plane.h"

#ifndef CFX_NS
#error "CFX_NS (species count) must be defined"
#endif
#ifndef CFX_PREC
#error "CFX_PREC (64 or 32) must be defined"
#endif

namespace cfx {

namespace {

constexpr int NS = CFX_NS;
constexpr int NSA = NS > 0 ? NS : 1;  // extent of the per-species arrays
static_assert(NS >= 0 && NS <= kMaxSp, "species count out of range");

__device__ __forceinline__ long long pidx(const GView &B, int i, int j, int k) {
  return (long long)(k + kNgg) * B.sz + (long long)(j + kNgg) * B.sy + (i + kNgg);
}

__device__ __forceinline__ long long interior_pidx(const GView &B, long long q) {
  const unsigned u = (unsigned)q, mx = (unsigned)B.mx, my = (unsigned)B.my;
  const unsigned i = u % mx, r = u / mx;
  return pidx(B, (int)i, (int)(r % my), (int)(r / my));
}

// Mass fraction l at padded point p.  The mixed-precision path keeps no FP64
// copy of Y after the initial upload: there Y_l = (rho Y_l) * (1 / rho) from
// the conserved state, in the update kernel's operation order, which gives
// at every updated point the value the update would have stored.
__device__ __forceinline__ double mass_fraction(const GView &B, long long p, int l) {
  return B.mixed ? B.cv[(5 + l) * B.np + p] * (1.0 / B.cv[p]) : B.yk[l * B.np + p];
}

// Point kernels: workgroup -> (block, first point of its kTpb chunk).
struct PointWork {
  int blk;
  long long base;
};
__device__ __forceinline__ PointWork point_work(const int *__restrict__ off, int nb) {
  const int w = blockIdx.x + off[0];
  const int blk = find_seg(off, nb, w);
  return {blk, (long long)(w - off[blk]) * kTpb};
}

// ------------------------------------------------------------ properties ---
// update_physical_properties (Field.cu:178-210): mixture cp, gamma and speed
// of sound at temperature t and mass fractions Y; cp_l and sum Y_l/W_l are
// returned for the transport.
// FP64: cpl holds a copy of the cp coefficients in LDS (kCpRec per species, the
// low ranges first), from which each lane reads those of its own range (the
// same values).  species_cp reads them from memory behind a branch instead, one
// species after the other: 256x128x128 cells with 9 species 0.30 -> 0.23 ms,
// with the roots of all species at once (floor of its traffic: 0.17).
constexpr int kCpRec = 6;  // 5 coefficients, 16-byte aligned
template <typename R>
__device__ __forceinline__ void mixture_gamma_c(SpeciesPtrT<R> sp, const R *cpl, R t, const R *Y, R *cp, R &winv,
                                                R *out) {
  R cpt = 0;
  winv = 0;
  const bool hi = t >= R(sp->hi_from);
  if (cpl && __all(hi || (t >= R(sp->lo_from) && t < R(sp->lo_to)))) {
    const R *c = cpl + (hi ? NS * kCpRec : 0);
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      const R *x = c + l * kCpRec;
      cp[l] = x[0] + t * (x[1] + t * (x[2] + t * (x[3] + t * x[4])));
    }
  } else {
#pragma unroll
    for (int l = 0; l < NS; ++l) cp[l] = species_cp<R>(sp, l, t);
  }
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    winv += Y[l] * R(sp->inv_mw[l]);
    cpt += Y[l] * cp[l];
  }
  const R Ru = R(kRu);
  const R gam = fdiv<R>(cpt, cpt - Ru * winv);
  out[0] = gam;
  out[1] = fsqrt<R>(gam * Ru * t * winv);
}

// compute_transport_property (Transport.cu:43-96): out = mu, kappa,
// rho*D_1..ns.  The Wilke sums use s_l = sqrt(mu_l) so that sqrt(mu_m/mu_n)
// = s_m/s_n (NS square roots instead of NS^2), and T*^-0.145 =
// T^-0.145 (k/eps_l)^-0.145: one exponential per point, the species factor
// from the table.
// FAST: the roots and their reciprocals of all species at once, and the quotients
// of fdiv_n (within an ulp of the others).
template <typename R, bool FAST = false>
__device__ __forceinline__ void wilke_point(SpeciesPtrT<R> sp, const SchemeDev &S, R t, const R *Y, const R *cp,
                                            R winv, R *out) {
  // Chapman-Enskog species viscosity (Transport.cu:52-57)
  const R tm = fexp<R>(R(-0.145) * flog<R>(t)), st = fsqrt<R>(t);
  R mu_s[NSA], X[NSA], s[NSA], rs[NSA];
  const R imw = frcp<R>(winv);
  auto div = [](R a, R b) {
    R q;
    if constexpr (FAST) fdiv_n<1, R>(&a, &b, &q);
    else q = fdiv<R>(a, b);
    return q;
  };
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    X[l] = Y[l] * imw * R(sp->inv_mw[l]);
    const R tdl = t * R(sp->lj_inv[l]);
    const R a = tdl + R(0.5);
    const R omega = R(1.147) * (tm * R(sp->om145[l])) + frcp<R>(a * a);
    mu_s[l] = div(R(sp->vis_coeff[l]) * st, omega);
    if constexpr (!FAST) {
      s[l] = fsqrt<R>(mu_s[l]);
      rs[l] = frcp<R>(s[l]);
    }
  }
  if constexpr (FAST) fsqrt_n<NSA, R>(mu_s, s, rs);
  // Wilke mixing and Mason-Saxena conductivity (Transport.cu:58-83)
  R mu = 0, kappa = 0;
#pragma unroll
  for (int m = 0; m < NS; ++m) {
    R vt = X[m];
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      if (n == m) continue;
      const R q = R(1) + s[m] * rs[n] * R(sp->wj4[m][n]);
      vt += q * q * R(sp->sqw8[m][n]) * X[n];
    }
    const R lam = mu_s[m] * (cp[m] + R(sp->cond_add[m]));
    mu += div(mu_s[m] * X[m], vt);
    kappa += div(lam * X[m], R(1.065) * vt - R(0.065) * X[m]);
  }
  out[0] = mu;
  out[1] = kappa;
  // constant-Schmidt diffusivity (Transport.cu:85-92, X[l] in the test)
  const R mus = mu * R(S.inv_sc);
#pragma unroll
  for (int l = 0; l < NS; ++l)
    out[2 + l] = fabs(X[l] - R(1)) < R(1e-3) ? mus : div((R(1) - Y[l]) * mu, (R(1) - X[l]) * R(S.sc));
}

// Properties over the padded range, or (2-D) by the points of the plane k = 0,
// whose rows are contiguous: MODE kPropsRing, its properties, and near the faces
// the copies to the ghost planes along k (eliminate_k_gradient, Field.cu:268-292)
// that the ghost fills read; kPropsPlanes, the properties of all planes (those of
// equal points) and every copy.  In R = float (mixed precision) the
// kernel also writes the FP32 copies of the primitives the FP32 RHS reads.
template <typename R, int MODE>
__global__ void __launch_bounds__(kTpb) props_kernel(const BlockView *__restrict__ views, const int *__restrict__ off,
                                                     int nb, const SpeciesDev *__restrict__ spg, SchemeDev S) {
  const SpeciesPtrT<R> sp = const_table<R>(spg);
  const PointWork pw = point_work(off, nb);
  const GView B = gview(views[pw.blk]);
  const long long np = B.np;
  constexpr bool f32 = sizeof(R) == 4;
  __shared__ __attribute__((aligned(16))) R cpl[f32 || NS == 0 ? 1 : 2 * NSA * kCpRec];
  if constexpr (!f32 && NS > 0) {
    for (int n = threadIdx.x; n < 10 * NS; n += kTpb) cpl[n / 5 * kCpRec + n % 5] = sp->cpc[n / (5 * NSA)][n / 5 % NSA][n % 5];
    __syncthreads();
  }
  const long long q = pw.base + threadIdx.x;
  if (q >= (MODE ? B.sz : np)) return;
  const long long p = MODE ? kNgg * B.sz + q : q;
  const R t = R(B.bv[5 * np + p]);
  R out[4 + (NS > 0 ? NS : 0)];
  R Y[NSA];
  if constexpr (NS == 0) {
    const R c_temp = R(S.gamma_air * S.r_air);
    out[0] = R(S.gamma_air);
    out[1] = sqrt(c_temp * t);
    const R mu = R(1.716e-5) * pow(t / R(273), R(1.5)) * R(273 + 111) / (t + R(111));
    out[2] = mu;
    out[3] = mu * c_temp / R(S.gamma_air - 1) * R(S.inv_pr);
  } else {
    R cp[NSA], winv;
    if constexpr (f32) {
      const double ir = 1.0 / B.cv[p];
#pragma unroll
      for (int l = 0; l < NS; ++l) Y[l] = R(B.cv[(5 + l) * np + p] * ir);
    } else {
#pragma unroll
      for (int l = 0; l < NS; ++l) Y[l] = R(B.yk[l * np + p]);
    }
    mixture_gamma_c<R>(sp, f32 ? nullptr : cpl, t, Y, cp, winv, out);
    wilke_point<R, !f32>(sp, S, t, Y, cp, winv, out + 2);
  }
  // loads first (T and Y are already held), then the stores
  double b64[6], c0 = 0;
  if constexpr (f32 || MODE) {
#pragma unroll
    for (int v = 0; v < 6; ++v) b64[v] = B.bv[v * np + p];
  }
  double cvY[NSA];
  if constexpr (MODE && f32) c0 = B.cv[p];
  if constexpr (MODE && NS > 0) {
#pragma unroll
    for (int l = 0; l < NS; ++l) cvY[l] = f32 ? B.cv[(5 + l) * np + p] : double(Y[l]);
  }
  auto put = [&](long long x) {
    if constexpr (f32) {
#pragma unroll
      for (int v = 0; v < 4 + NS; ++v) B.props32[v * np + x] = out[v];
#pragma unroll
      for (int v = 0; v < 6; ++v) B.bv32[v * np + x] = float(b64[v]);
      if constexpr (NS > 0) {
#pragma unroll
        for (int l = 0; l < NS; ++l) B.yk32[l * np + x] = float(Y[l]);
      }
    } else {
#pragma unroll
      for (int v = 0; v < 4 + NS; ++v) B.props[v * np + x] = out[v];
    }
  };
  put(p);
  if constexpr (MODE) {
    const int px = B.px, i = (int)q % px - kNgg, j = (int)q / px - kNgg;
    if (MODE == kPropsRing && i > kNgg && i < B.mx - 1 - kNgg && j > kNgg && j < B.my - 1 - kNgg) return;
#pragma unroll
    for (int g = -kNgg; g <= kNgg; ++g) {
      if (g == 0) continue;
      const long long x = p + g * B.sz;
#pragma unroll
      for (int v = 0; v < 6; ++v) B.bv[v * np + x] = b64[v];
      if constexpr (f32) {  // the mixed path derives Y from cv: rho and rho*Y instead
        B.cv[x] = c0;
#pragma unroll
        for (int l = 0; l < NS; ++l) B.cv[(5 + l) * np + x] = cvY[l];
      } else {
#pragma unroll
        for (int l = 0; l < NS; ++l) B.yk[l * np + x] = cvY[l];
      }
      if (MODE == kPropsPlanes) put(x);
    }
  }
}

template <typename R>
int launch_props(const Batch &b, int mode, const SpeciesDev *sp, const SchemeDev &S, hipStream_t st) {
  if (b.total <= 0) return 0;
  if (mode == kPropsRing)
    props_kernel<R, kPropsRing><<<b.total, kTpb, 0, st>>>(b.views, b.off, b.nb, sp, S);
  else if (mode == kPropsPlanes)
    props_kernel<R, kPropsPlanes><<<b.total, kTpb, 0, st>>>(b.views, b.off, b.nb, sp, S);
  else
    props_kernel<R, kPropsPadded><<<b.total, kTpb, 0, st>>>(b.views, b.off, b.nb, sp, S);
  return (int)hipGetLastError();
}

// ------------------------------------------------------------------- RHS ---
// 2-D.  FP64 with species takes all the registers of 2 waves per SIMD; air and
// FP32 fit twice that.
template <int V, typename R>
int launch_rhs_plane(const Batch &b, int planar, const SpeciesDev *sp, const SchemeDev &S, hipStream_t st) {
  constexpr PlaneTile t = kTiles2[V];
  constexpr int WPE = sizeof(R) == 8 && NS > 0 ? 2 : 4;
  if (b.total <= 0) return 0;
  const int padded = (b.total + 7) / 8 * 8;
  if (planar)
    rhs_plane_kernel<NS, t.tx, t.ty, WPE, R, true><<<padded, 512, 0, st>>>(b.views, b.off, b.nb, padded, sp, S);
  else
    rhs_plane_kernel<NS, t.tx, t.ty, WPE, R, false><<<padded, 512, 0, st>>>(b.views, b.off, b.nb, padded, sp, S);
  return (int)hipGetLastError();
}

// FP64 air fits the registers of two workgroups per CU: 161x113x77 cells 202 ->
// 161 us per evaluation
template <typename R>
constexpr MarchTile march_tile() {
  MarchTile t = sizeof(R) == 8 ? kMarch64 : kMarch32;
  if (NS == 0) t.wpe = 4;
  return t;
}

template <typename R>
int launch_rhs_march(const Batch &b, int chunk, int big, const SpeciesDev *sp, const SchemeDev &S, hipStream_t st) {
  constexpr MarchTile t = march_tile<R>();
  if (b.total <= 0) return 0;
  const int padded = (b.total + 7) / 8 * 8;
  if (big)
    rhs_march_kernel<NS, t.tx, t.ty, t.nt, t.wpe, R, true>
        <<<padded, t.nt, 0, st>>>(b.views, b.off, b.nb, padded, chunk, sp, S);
  else
    rhs_march_kernel<NS, t.tx, t.ty, t.nt, t.wpe, R, false>
        <<<padded, t.nt, 0, st>>>(b.views, b.off, b.nb, padded, chunk, sp, S);
  return (int)hipGetLastError();
}

template <typename R>
int occupancy_rhs_march() {
  constexpr MarchTile t = march_tile<R>();
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, rhs_march_kernel<NS, t.tx, t.ty, t.nt, t.wpe, R, false>, t.nt,
                                                   0) != hipSuccess)
    return 0;
  return n;
}

template <typename R, typename Set>
void register_rhs(Set &k) {
  k.march = launch_rhs_march<R>;
  k.march_occ = occupancy_rhs_march<R>;
  k.plane[0] = launch_rhs_plane<0, R>;
  k.plane[1] = launch_rhs_plane<1, R>;
}

#if CFX_PREC == 64
// ---------------------------------------------------------- total energy ---
// compute_total_energy (Thermo.cu:66-86) from bv/yk/cv at padded point p.
__device__ __forceinline__ void total_energy(const GView &B, SpeciesPtrT<double> sp, const SchemeDev &S,
                                             long long p) {
  const long long np = B.np;
  const double u = B.bv[np + p], v = B.bv[2 * np + p], w = B.bv[3 * np + p];
  double e = 0.5 * B.bv[p] * (u * u + v * v + w * w);
  if constexpr (NS > 0) {
    const double t = B.bv[5 * np + p];
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      double h, cp;
      species_h_cp<double>(sp, l, t, h, cp);
      e += h * B.cv[(5 + l) * np + p];
    }
    e -= B.bv[4 * np + p];
  } else {
    e += B.bv[4 * np + p] / (S.gamma_air - 1);
  }
  B.cv[4 * np + p] = e;
}

// The same total energy from values held in registers (rhoY: the partial
// densities), in total_energy's operation order.
__device__ __forceinline__ double total_energy_of(SpeciesPtrT<double> sp, const SchemeDev &S, double rho, double u,
                                                  double v, double w, double t, double pr, const double *rhoY) {
  double e = 0.5 * rho * (u * u + v * v + w * w);
  if constexpr (NS > 0) {
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      double h, cp;
      species_h_cp<double>(sp, l, t, h, cp);
      e += h * rhoY[l];
    }
    e -= pr;
  } else {
    e += pr / (S.gamma_air - 1);
  }
  return e;
}

// --------------------------------------------------------------- update ---
// update_cv_and_bv (TimeAdvanceFunc.cu:255-290) with the RK stage
// combination q = a*qn + b*(q + dt*dq/J) and the Newton inversion of T
// (Thermo.cu:89-125, stop |dT| <= 1e-10 K unless CFX_Q_NEWTON_REL).
// MIXED selects the FP32 dq.  The loads are issued before the first store:
// the stores go through pointers the compiler must assume alias the loaded
// arrays.
template <bool MIXED>
__global__ void __launch_bounds__(kTpb) update_kernel(const BlockView *__restrict__ views, const int *__restrict__ off,
                                                      int nb, const SpeciesDev *__restrict__ spg, SchemeDev S,
                                                      int stage, const double *__restrict__ dt_dev, int *flags,
                                                      unsigned long long *newton_fail) {
  const SpeciesPtrT<double> sp = const_table<double>(spg);
  constexpr int NV = 5 + NS;
  const PointWork pw = point_work(off, nb);
  const GView B = gview(views[pw.blk]);
  const long long np = B.np, ni = B.ni;
  const long long q = pw.base + threadIdx.x;
  if (q >= ni) return;
  const double A = stage == 1 ? 0.75 : (stage == 2 ? 1.0 / 3.0 : 0.0);
  const double Bc = stage == 1 ? 0.25 : (stage == 2 ? 2.0 / 3.0 : 1.0);
  const bool rel = (S.quirks & CFX_Q_NEWTON_REL) != 0;
  const bool rk3 = S.rk == 3;
  const long long p = interior_pidx(B, q);
  double cur[NV], dqv[NV], qnv[NV];
  // dq and the stage base qn are streamed once per stage: non-temporal
  // accesses keep them from displacing the state in the caches
#pragma unroll
  for (int l = 0; l < NV; ++l) cur[l] = B.cv[l * np + p];
#pragma unroll
  for (int l = 0; l < NV; ++l)
    dqv[l] = MIXED ? (double)__builtin_nontemporal_load(&B.dq32[l * ni + q]) : __builtin_nontemporal_load(&B.dq[l * ni + q]);
  const bool use_qn = rk3 && stage > 0;
  if (use_qn) {
#pragma unroll
    for (int l = 0; l < NV; ++l) qnv[l] = __builtin_nontemporal_load(&B.qn[l * ni + q]);
  }
  const double t_old = B.bv[5 * np + p];
  // LU-SGS: dq already holds the increment
  const double dtj = S.lusgs ? 1.0 : (rk3 ? *dt_dev : B.dt_local[q]) / B.jac[p];
  double c[NV];
#pragma unroll
  for (int l = 0; l < NV; ++l) {
    const double base = use_qn ? qnv[l] : cur[l];
    c[l] = rk3 ? A * base + Bc * (cur[l] + dqv[l] * dtj) : cur[l] + dqv[l] * dtj;
  }
  if (B.mz == 1) c[3] = 0.0;
  // the stage base goes out now (every load of the point has been issued and
  // the Newton iteration reads only scalar memory), which frees cur; the
  // state's stores come after the iteration
  if (rk3 && stage == 0) {
#pragma unroll
    for (int l = 0; l < NV; ++l) __builtin_nontemporal_store(cur[l], &B.qn[l * ni + q]);
  }
  const double rho = c[0];
  const double ir = 1.0 / rho;
  const double u = c[1] * ir, v = c[2] * ir, w = c[3] * ir;
  const double v2 = u * u + v * v + w * w;
  double T, pr;
  double Y[NSA];
  if constexpr (NS > 0) {
    double winv = 0;
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      Y[l] = c[5 + l] * ir;
      winv += Y[l] * sp->inv_mw[l];
    }
    const double R = kRu * winv;
    const double e = c[4] / rho - 0.5 * v2;
    T = t_old;
    double err = 1e30;
    int it = 0;
    const double eps = rel ? 1e-3 : 1e-10;
    while (err > eps && it < 1000) {
      ++it;
      double h = 0, cp = 0;
#pragma unroll
      for (int l = 0; l < NS; ++l) {
        double hl, cpl;
        species_h_cp<double>(sp, l, T, hl, cpl);
        h += hl * Y[l];
        cp += cpl * Y[l];
      }
      const double T1 = T - (h - R * T - e) / (cp - R);
      err = rel ? fabs(1 - T1 / T) : fabs(T1 - T);
      T = T1;
    }
    if (err > eps) atomicAdd(newton_fail, 1ull);
    pr = rho * T * R;
  } else {
    pr = (S.gamma_air - 1) * (c[4] - 0.5 * rho * v2);
    T = pr * ir / S.r_air;
  }
#pragma unroll
  for (int l = 0; l < NV; ++l) B.cv[l * np + p] = c[l];
  if constexpr (NS > 0 && !MIXED) {  // the mixed path derives Y from cv where it needs it
#pragma unroll
    for (int l = 0; l < NS; ++l) B.yk[l * np + p] = Y[l];
  }
  B.bv[p] = rho;
  B.bv[np + p] = u;
  B.bv[2 * np + p] = v;
  B.bv[3 * np + p] = w;
  B.bv[4 * np + p] = pr;
  B.bv[5 * np + p] = T;
  if (!(rho > 0.0) || !(T > 0.0) || !(pr > 0.0) || !isfinite(rho) || !isfinite(T)) atomicOr(flags, 1);
  // apply_outflow (BoundCond.cu:455-487) of the faces folded into the
  // update: a point of the face layer writes its new state into the ghost
  // layers behind it (the same cache lines as its own stores for x faces)
  if (B.fuse_any) {
    const unsigned uq = (unsigned)q, mx = (unsigned)B.mx, my = (unsigned)B.my;
    const int ijk[3] = {(int)(uq % mx), (int)((uq / mx) % my), (int)(uq / (mx * my))};
    const int mm[3] = {B.mx, B.my, B.mz};
    const long long stride[3] = {1, B.sy, B.sz};
    const double bvn[6] = {rho, u, v, w, pr, T};
    for (int a = 0; a < 3; ++a)
      for (int side = 0; side < 2; ++side) {
        if (!B.fuse[2 * a + side] || ijk[a] != (side ? mm[a] - 1 : 0)) continue;
        const long long step = side ? stride[a] : -stride[a];
        for (int g = 1; g <= kNgg; ++g) {
          const long long qg = p + g * step;
#pragma unroll
          for (int l = 0; l < 6; ++l) B.bv[l * np + qg] = bvn[l];
#pragma unroll
          for (int l = 0; l < NV; ++l) B.cv[l * np + qg] = c[l];
          if constexpr (NS > 0 && !MIXED) {
#pragma unroll
            for (int l = 0; l < NS; ++l) B.yk[l * np + qg] = Y[l];
          }
        }
      }
  }
}

// compute_cv_from_bv (Field.cu:150-176) over the padded range
__global__ void __launch_bounds__(kTpb) cv_from_bv_kernel(const BlockView *__restrict__ views,
                                                          const int *__restrict__ off, int nb,
                                                          const SpeciesDev *__restrict__ spg, SchemeDev S) {
  const SpeciesPtrT<double> sp = const_table<double>(spg);
  const PointWork pw = point_work(off, nb);
  const GView B = gview(views[pw.blk]);
  const long long np = B.np;
  const long long p = pw.base + threadIdx.x;
  if (p >= np) return;
  const double rho = B.bv[p];
  B.cv[p] = rho;
  B.cv[np + p] = rho * B.bv[np + p];
  B.cv[2 * np + p] = rho * B.bv[2 * np + p];
  B.cv[3 * np + p] = rho * B.bv[3 * np + p];
#pragma unroll
  for (int l = 0; l < NS; ++l) B.cv[(5 + l) * np + p] = rho * B.yk[l * np + p];
  total_energy(B, sp, S, p);
}

// ------------------------------------------------------------ ghost fill ---
// apply_outflow (BoundCond.cu:455-487) at face point (i, j, k)
__device__ __forceinline__ void bc_outflow_point(const GView &B, const FaceRange &f, int i, int j, int k) {
  int dir[3] = {0, 0, 0};
  dir[f.face] = f.direction;
  const long long np = B.np;
  const long long p = pidx(B, i, j, k);
  // every value of the face point is read before the first store: the
  // stores go to the same arrays, so the compiler could not move a later
  // load above an earlier store and each field would cost a memory round trip
  double bvp[6], cvp[5 + NS], ykp[NSA];
#pragma unroll
  for (int l = 0; l < 6; ++l) bvp[l] = B.bv[l * np + p];
#pragma unroll
  for (int l = 0; l < 5 + NS; ++l) cvp[l] = B.cv[l * np + p];
  if (!B.mixed) {
#pragma unroll
    for (int l = 0; l < NS; ++l) ykp[l] = B.yk[l * np + p];
  }
  for (int g = 1; g <= kNgg; ++g) {
    const long long q = pidx(B, i + g * dir[0], j + g * dir[1], k + g * dir[2]);
#pragma unroll
    for (int l = 0; l < 6; ++l) B.bv[l * np + q] = bvp[l];
#pragma unroll
    for (int l = 0; l < 5 + NS; ++l) B.cv[l * np + q] = cvp[l];
    if (!B.mixed) {
#pragma unroll
      for (int l = 0; l < NS; ++l) B.yk[l * np + q] = ykp[l];
    }
  }
}

// apply_inflow (BoundCond.cu:489-527); the state's total energy is
// precomputed on the host with the same formula as compute_total_energy.
__device__ __forceinline__ void bc_inflow_point(const GView &B, const FaceRange &f, int i, int j, int k,
                                                const InflowDev *__restrict__ in) {
  int dir[3] = {0, 0, 0};
  dir[f.face] = f.direction;
  const long long np = B.np;
  const double rho = in->st[0];
  for (int g = 1; g <= kNgg; ++g) {
    const long long q = pidx(B, i + g * dir[0], j + g * dir[1], k + g * dir[2]);
#pragma unroll
    for (int l = 0; l < 6; ++l) B.bv[l * np + q] = in->st[l];
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      if (!B.mixed) B.yk[l * np + q] = in->y[l];
      B.cv[(5 + l) * np + q] = rho * in->y[l];
    }
    B.cv[q] = rho;
    B.cv[np + q] = rho * in->st[1];
    B.cv[2 * np + q] = rho * in->st[2];
    B.cv[3 * np + q] = rho * in->st[3];
    B.cv[4 * np + q] = in->st[6];
  }
}

__device__ __forceinline__ double mix_mw(SpeciesPtrT<double> sp, const SchemeDev &S, const double *Y) {
  if constexpr (NS == 0) {
    return kRu / S.r_air;
  } else {
    double w = 0;
#pragma unroll
    for (int l = 0; l < NS; ++l) w += Y[l] * sp->inv_mw[l];
    return 1.0 / w;
  }
}

// apply_wall (BoundCond.cu:529-629) over the face's own vertex range (the
// registered range shrunk back by ngg, BoundCond.cu:229-239).
__device__ __forceinline__ void bc_wall_point(const GView &B, const FaceRange &f, int i, int j, int k,
                                              SpeciesPtrT<double> sp, const SchemeDev &S, const WallDev &wl) {
  int dir[3] = {0, 0, 0};
  dir[f.face] = f.direction;
  const long long np = B.np;
  const long long p = pidx(B, i, j, k);
  // every interior value is read before the first store (the stores could
  // alias later loads as far as the compiler knows; one round trip each);
  // interior point g = 1 is the one next to the wall
  long long qi[kNgg], qg[kNgg];
  double Yi[kNgg][NSA], ui[kNgg], vi[kNgg], wi[kNgg], pi[kNgg], ti[kNgg];
#pragma unroll
  for (int g = 0; g < kNgg; ++g) {
    qi[g] = pidx(B, i - (g + 1) * dir[0], j - (g + 1) * dir[1], k - (g + 1) * dir[2]);
    qg[g] = pidx(B, i + (g + 1) * dir[0], j + (g + 1) * dir[1], k + (g + 1) * dir[2]);
#pragma unroll
    for (int l = 0; l < NS; ++l) Yi[g][l] = mass_fraction(B, qi[g], l);
    ui[g] = B.bv[np + qi[g]], vi[g] = B.bv[2 * np + qi[g]], wi[g] = B.bv[3 * np + qi[g]];
    pi[g] = B.bv[4 * np + qi[g]], ti[g] = B.bv[5 * np + qi[g]];
  }
  double t_wall = wl.temperature;
  if (wl.adiabatic) t_wall = ti[0];
  const double pw = pi[0];
  double rY[NSA];
  {
    const double rho = pw * mix_mw(sp, S, Yi[0]) / (t_wall * kRu);
    if (!B.mixed) {
#pragma unroll
      for (int l = 0; l < NS; ++l) B.yk[l * np + p] = Yi[0][l];
    }
    B.bv[p] = rho;
    B.bv[np + p] = 0;
    B.bv[2 * np + p] = 0;
    B.bv[3 * np + p] = 0;
    B.bv[4 * np + p] = pw;
    B.bv[5 * np + p] = t_wall;
    B.cv[p] = rho;
    B.cv[np + p] = 0;
    B.cv[2 * np + p] = 0;
    B.cv[3 * np + p] = 0;
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      rY[l] = Yi[0][l] * rho;
      B.cv[(l + 5) * np + p] = rY[l];
    }
    B.cv[4 * np + p] = total_energy_of(sp, S, rho, 0.0, 0.0, 0.0, t_wall, pw, rY);
  }
#pragma unroll
  for (int g = 0; g < kNgg; ++g) {
    if (!B.mixed) {
#pragma unroll
      for (int l = 0; l < NS; ++l) B.yk[l * np + qg[g]] = Yi[g][l];
    }
    const double mw = mix_mw(sp, S, Yi[g]);
    double t_g = ti[g];
    if (!wl.adiabatic) {
      t_g = 2 * t_wall - ti[g];
      if (t_g <= 0.1 * t_wall) t_g = t_wall;
    }
    const double rho_g = pi[g] * mw / (t_g * kRu);
    B.bv[qg[g]] = rho_g;
    B.bv[np + qg[g]] = -ui[g];
    B.bv[2 * np + qg[g]] = -vi[g];
    B.bv[3 * np + qg[g]] = -wi[g];
    B.bv[4 * np + qg[g]] = pi[g];
    B.bv[5 * np + qg[g]] = t_g;
    B.cv[qg[g]] = rho_g;
    B.cv[np + qg[g]] = -rho_g * ui[g];
    B.cv[2 * np + qg[g]] = -rho_g * vi[g];
    B.cv[3 * np + qg[g]] = -rho_g * wi[g];
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      rY[l] = Yi[g][l] * rho_g;
      B.cv[(l + 5) * np + qg[g]] = rY[l];
    }
    B.cv[4 * np + qg[g]] = total_energy_of(sp, S, rho_g, -ui[g], -vi[g], -wi[g], t_g, pi[g], rY);
  }
}

// Slip wall: the boundary point loses its velocity along the face normal
// n = grad(xi_face)/|grad(xi_face)|; ghost g mirrors interior point g with
// the normal velocity negated and rho, p, T, Y copied.
__device__ __forceinline__ void bc_symmetry_point(const GView &B, const FaceRange &f, int i, int j, int k,
                                                  SpeciesPtrT<double> sp, const SchemeDev &S) {
  int dir[3] = {0, 0, 0};
  dir[f.face] = f.direction;
  const long long np = B.np;
  const long long p = pidx(B, i, j, k);
  // every value is read before the first store (as in the wall condition)
  double n[3];
  for (int c = 0; c < 3; ++c) n[c] = B.metric[(f.face * 3 + c) * np + p];
  double bp[6], rYp[NSA];
#pragma unroll
  for (int l = 0; l < 6; ++l) bp[l] = B.bv[l * np + p];
#pragma unroll
  for (int l = 0; l < NS; ++l) rYp[l] = B.cv[(5 + l) * np + p];
  long long qi[kNgg], qg[kNgg];
  double bi[kNgg][6], Yi[kNgg][NSA];
#pragma unroll
  for (int g = 0; g < kNgg; ++g) {
    qi[g] = pidx(B, i - (g + 1) * dir[0], j - (g + 1) * dir[1], k - (g + 1) * dir[2]);
    qg[g] = pidx(B, i + (g + 1) * dir[0], j + (g + 1) * dir[1], k + (g + 1) * dir[2]);
#pragma unroll
    for (int l = 0; l < 6; ++l) bi[g][l] = B.bv[l * np + qi[g]];
#pragma unroll
    for (int l = 0; l < NS; ++l) Yi[g][l] = mass_fraction(B, qi[g], l);
  }
  const double nn = sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
  n[0] /= nn;
  n[1] /= nn;
  n[2] /= nn;
  {
    const double vn = bp[1] * n[0] + bp[2] * n[1] + bp[3] * n[2];
    for (int c = 0; c < 3; ++c) {
      bp[1 + c] -= vn * n[c];
      B.bv[(1 + c) * np + p] = bp[1 + c];
    }
    for (int c = 0; c < 3; ++c) B.cv[(1 + c) * np + p] = bp[0] * bp[1 + c];
    B.cv[4 * np + p] = total_energy_of(sp, S, bp[0], bp[1], bp[2], bp[3], bp[5], bp[4], rYp);
  }
#pragma unroll
  for (int g = 0; g < kNgg; ++g) {
    const double *b = bi[g];
    const double vn = b[1] * n[0] + b[2] * n[1] + b[3] * n[2];
    double u[3], rY[NSA];
    for (int c = 0; c < 3; ++c) u[c] = b[1 + c] - 2 * vn * n[c];
    B.bv[qg[g]] = b[0];
    for (int c = 0; c < 3; ++c) B.bv[(1 + c) * np + qg[g]] = u[c];
    B.bv[4 * np + qg[g]] = b[4];
    B.bv[5 * np + qg[g]] = b[5];
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      if (!B.mixed) B.yk[l * np + qg[g]] = Yi[g][l];
      rY[l] = b[0] * Yi[g][l];
      B.cv[(5 + l) * np + qg[g]] = rY[l];
    }
    B.cv[qg[g]] = b[0];
    for (int c = 0; c < 3; ++c) B.cv[(1 + c) * np + qg[g]] = b[0] * u[c];
    B.cv[4 * np + qg[g]] = total_energy_of(sp, S, b[0], u[0], u[1], u[2], b[5], b[4], rY);
  }
}

// loop point n of an exchange: the point p of the block and t of the target, and
// whether they are on the shared layer
__device__ __forceinline__ bool exchange_pair(const GView &B, const GView &T, const InnerDev &f, const int n[3],
                                              long long &p, long long &t) {
  int idx[3], d_idx[3], it[3];
  for (int q = 0; q < 3; ++q) {
    d_idx[q] = f.loop_dir[q] * n[q];
    idx[q] = f.rs[q] + d_idx[q];
  }
  for (int q = 0; q < 3; ++q) it[q] = f.ts[q] + f.target_loop_dir[q] * d_idx[f.src_tar[q]];
  p = pidx(B, idx[0], idx[1], idx[2]);
  t = pidx(T, it[0], it[1], it[2]);
  return idx[f.face] == (f.direction > 0 ? f.rs[f.face] : f.re[f.face]);
}

// inner_communication (Field.cu:213-266) with the face loop of
// Mesh.cpp:905-917 at loop point n: shared-face points are averaged between
// the two blocks, ghost layers take the neighbour's values.
__device__ __forceinline__ void exchange_point(const GView &B, const GView &T, const InnerDev &f,
                                               const int n[3], bool ghosts_only) {
  long long p, t;
  const bool shared = exchange_pair(B, T, f, n, p, t);
  const long long np = B.np, tnp = T.np;
  // Loads are grouped ahead of the stores (the two blocks' arrays may alias
  // as far as the compiler knows, so it keeps every store before any later
  // load: field by field, each would cost a memory round trip).
  if (shared) {
    if (ghosts_only) return;
    // the shared layer: both sides of a group of fields, then the averages
    auto average = [&](gptr<double> bb, gptr<double> tt, auto kc) {
      constexpr int K = decltype(kc)::value;
      double x[K > 0 ? K : 1], y[K > 0 ? K : 1];
#pragma unroll
      for (int l = 0; l < K; ++l) x[l] = tt[l * tnp + t], y[l] = bb[l * np + p];
#pragma unroll
      for (int l = 0; l < K; ++l) {
        const double a = 0.5 * (x[l] + y[l]);
        bb[l * np + p] = a;
        tt[l * tnp + t] = a;
      }
    };
    average(B.bv, T.bv, std::integral_constant<int, 6>{});
    average(B.cv, T.cv, std::integral_constant<int, 5 + NS>{});
    if constexpr (NS > 0)
      if (!B.mixed) average(B.yk, T.yk, std::integral_constant<int, NS>{});
  } else {
    // a ghost point: the neighbour's values, all read before any store
    double bvt[6], cvt[5 + NS], ykt[NSA];
#pragma unroll
    for (int l = 0; l < 6; ++l) bvt[l] = T.bv[l * tnp + t];
#pragma unroll
    for (int l = 0; l < 5 + NS; ++l) cvt[l] = T.cv[l * tnp + t];
    if (!B.mixed) {
#pragma unroll
      for (int l = 0; l < NS; ++l) ykt[l] = T.yk[l * tnp + t];
    }
#pragma unroll
    for (int l = 0; l < 6; ++l) B.bv[l * np + p] = bvt[l];
#pragma unroll
    for (int l = 0; l < 5 + NS; ++l) B.cv[l * np + p] = cvt[l];
    if (!B.mixed) {
#pragma unroll
      for (int l = 0; l < NS; ++l) B.yk[l * np + p] = ykt[l];
    }
  }
}

// One launch runs a set of ghost-fill ops that touch disjoint data (one
// level of the op schedule, or a single op): workgroup -> op by the prefix
// off[], then one point of the op per thread.
__global__ void __launch_bounds__(kTpb) face_ops_kernel(const BlockView *__restrict__ views,
                                                        const FaceOp *__restrict__ ops, const int *__restrict__ off,
                                                        int nops, const SpeciesDev *__restrict__ spg, SchemeDev S,
                                                        const InflowDev *__restrict__ inflow) {
  const SpeciesPtrT<double> sp = const_table<double>(spg);
  const int w = blockIdx.x + off[0];
  const int s = find_seg(off, nops, w);
  const FaceOp &op = ops[s];
  const long long n = (long long)(w - off[s]) * kTpb + threadIdx.x;
  if (n >= op.npts) return;
  const int e0 = op.ext[0], e1 = op.ext[1];
  const int nn[3] = {(int)(n % e0), (int)((n / e0) % e1), (int)(n / ((long long)e0 * e1))};
  const GView B = gview(views[op.blk]);
  const int i = op.r.rs[0] + nn[0], j = op.r.rs[1] + nn[1], k = op.r.rs[2] + nn[2];
  switch (op.kind) {
    case CFX_BC_OUTFLOW: bc_outflow_point(B, op.r, i, j, k); break;
    case CFX_BC_INFLOW: bc_inflow_point(B, op.r, i, j, k, inflow + op.cond); break;
    case CFX_BC_WALL: bc_wall_point(B, op.r, i, j, k, sp, S, op.wl); break;
    case CFX_BC_SYMMETRY: bc_symmetry_point(B, op.r, i, j, k, sp, S); break;
    case kOpExchange: {
      const GView T = gview(views[op.tgt]);
      exchange_point(B, T, op.f, nn, op.ghosts_only != 0);
      break;
    }
    default: break;
  }
}

// The same for a level that only copies and averages (outflow conditions,
// exchanges): blockIdx.y takes one of the arrays bv, cv, yk, whose fields do not
// depend on each other.  A third of the chain per thread, and of the registers
// that hold a point's fields: the middles of 27 blocks of 20..90 points 424 -> 339
// us FP64, of 64 blocks of 12..44 mixed 125 -> 96, the edges of one block 13 -> 8.
__global__ void __launch_bounds__(kTpb) copy_ops_kernel(const BlockView *__restrict__ views,
                                                        const FaceOp *__restrict__ ops, const int *__restrict__ off,
                                                        int nops) {
  const int w = blockIdx.x + off[0];
  const int s = find_seg(off, nops, w);
  const FaceOp &op = ops[s];
  const long long n = (long long)(w - off[s]) * kTpb + threadIdx.x;
  if (n >= op.npts) return;
  const int e0 = op.ext[0], e1 = op.ext[1];
  const int nn[3] = {(int)(n % e0), (int)((n / e0) % e1), (int)(n / ((long long)e0 * e1))};
  const GView B = gview(views[op.blk]);
  const long long np = B.np;
  auto by_array = [&](auto f) {
    if (blockIdx.y == 0) f(B.bv, std::integral_constant<int, 6>{}, 0);
    else if (blockIdx.y == 1) f(B.cv, std::integral_constant<int, 5 + NS>{}, 1);
    else if constexpr (NS > 0) f(B.yk, std::integral_constant<int, NS>{}, 2);
  };
  if (op.kind == CFX_BC_OUTFLOW) {
    const long long p = pidx(B, op.r.rs[0] + nn[0], op.r.rs[1] + nn[1], op.r.rs[2] + nn[2]);
    const long long stride[3] = {1, B.sy, B.sz}, step = op.r.direction * stride[op.r.face];
    by_array([&](gptr<double> a, auto kc, int) {
      constexpr int K = decltype(kc)::value;
      double x[K];
#pragma unroll
      for (int l = 0; l < K; ++l) x[l] = a[l * np + p];
#pragma unroll
      for (int g = 1; g <= kNgg; ++g)
#pragma unroll
        for (int l = 0; l < K; ++l) a[l * np + p + g * step] = x[l];
    });
    return;
  }
  const GView T = gview(views[op.tgt]);
  const long long tnp = T.np;
  long long p, t;
  const bool shared = exchange_pair(B, T, op.f, nn, p, t);
  if (shared && op.ghosts_only) return;
  by_array([&](gptr<double> a, auto kc, int which) {
    constexpr int K = decltype(kc)::value;
    const gptr<double> b = which == 0 ? T.bv : (which == 1 ? T.cv : T.yk);
    double x[K];
#pragma unroll
    for (int l = 0; l < K; ++l) x[l] = b[l * tnp + t];
    if (shared) {  // both sides take the average
      double y[K];
#pragma unroll
      for (int l = 0; l < K; ++l) y[l] = a[l * np + p];
#pragma unroll
      for (int l = 0; l < K; ++l) b[l * tnp + t] = x[l] = 0.5 * (x[l] + y[l]);
    }
#pragma unroll
    for (int l = 0; l < K; ++l) a[l * np + p] = x[l];
  });
}

int launch_update(const Batch &b, const SpeciesDev *sp, const SchemeDev &S, int mixed, int stage, const double *dt,
                  int *flags, unsigned long long *nf, hipStream_t st) {
  if (b.total <= 0) return 0;
  if (mixed)
    update_kernel<true><<<b.total, kTpb, 0, st>>>(b.views, b.off, b.nb, sp, S, stage, dt, flags, nf);
  else
    update_kernel<false><<<b.total, kTpb, 0, st>>>(b.views, b.off, b.nb, sp, S, stage, dt, flags, nf);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------- LU-SGS ---
// Matrix-free LU-SGS (Yoon & Jameson, AIAA J. 26 (1988) 1025-1026), the
// implicit treatment the reference declares without a body (LUSGS,
// TemporalScheme.cuh:19-21).  Per interior cell:
//   D = J/dt + sum_d (omega r_d + 2 v_d),  a_d = omega r_d / 2 + v_d,
//   r_d = J (|V.grad xi_d| + c |grad xi_d|),  v_d = max(gamma, 4/3) mu/(rho Pr) J |grad xi_d|^2;
//   forward  D dQ*_i = R_i + sum_d [ dG_d(i-e_d)/2 + a_d(i-e_d) dQ*_(i-e_d) ]
//   backward dQ_i = dQ*_i + sum_d [ a_d(i+e_d) dQ_(i+e_d) - dG_d(i+e_d)/2 ] / D_i
// dG_d(n) = G_d(Q_n + dQ_n) - G_d(Q_n): the inviscid flux of cell n through
// S_d = J grad xi_d, the pressure change at the cell's frozen gamma; dQ = 0
// outside the block.  dq holds R on entry and dQ on exit (in place: a cell
// reads only final neighbour values).

// lus: D over the interior, then a_d for d = 0, 1, 2
__global__ void __launch_bounds__(kTpb) lusgs_coef_kernel(const BlockView *__restrict__ views,
                                                          const int *__restrict__ off, int nb, SchemeDev S) {
  const PointWork pw = point_work(off, nb);
  const GView B = gview(views[pw.blk]);
  const long long np = B.np, ni = B.ni;
  const long long q = pw.base + threadIdx.x;
  if (q >= ni) return;
  const long long p = interior_pidx(B, q);
  const double J = B.jac[p], rho = B.bv[p];
  const double u = B.bv[np + p], v = B.bv[2 * np + p], w = B.bv[3 * np + p];
  const double gam = B.props[p], c = B.props[np + p], mu = B.props[2 * np + p];
  const double vc = fmax(gam, 4.0 / 3.0) * mu / rho / S.pr;
  double diag = J / B.dt_local[q];
  for (int d = 0; d < S.dim; ++d) {
    const double gx = B.metric[(3 * d) * np + p], gy = B.metric[(3 * d + 1) * np + p],
                 gz = B.metric[(3 * d + 2) * np + p];
    const double g2 = gx * gx + gy * gy + gz * gz;
    const double r = J * (fabs(u * gx + v * gy + w * gz) + c * sqrt(g2));
    const double vd = vc * J * g2;
    diag += S.omega * r + 2 * vd;
    B.lus[(1 + d) * ni + q] = 0.5 * S.omega * r + vd;
  }
  B.lus[q] = diag;
}

// The sweeps.  A workgroup owns a patch of kLuP x kLuP columns along i and
// marches through them.  In its first wavefront lane (vg, c) updates group vg
// of the variables of column c = jl + kLuP kl, at step s the cell
// i = s - jl - kl, whose upstream neighbours are the same column's last cell
// and the cells that the columns jl - 1 and kl - 1 updated in the step before.
// Group 0 is (rho, rho V, E), the others are a third of the species each.
// Having updated its cell, a lane forms the terms that the downstream
// neighbours along each direction d add (dG_d / 2 + a_d dQ, in the forward
// sweep): the one along i stays in its registers, the others move by DPP row
// shifts (the 16 columns of a group are a DPP row), and those of the patch's
// last columns go to the patches after it through memory.  The second wavefront
// moves the cells between memory and LDS, kLuG steps at a time.
//
// Patches hand over terms while they run.  The places of the terms hold kLuNone
// until they are written, so a lane that needs one loads it (two steps ahead)
// and loads it again until it is there; every value is one 64-bit atomic store
// and load of agent scope and says by itself whether it is valid.  No wait can
// last: a workgroup takes its patch from a ticket counter whose order holds
// every patch behind the two that it waits for, so these are done or running.
// (A wait beyond kLuWait, which none of this allows, is given up with an error
// flag, and raises an abort word that ends the sweep's other waits: ticket[1].)
//
// The backward sweep is the forward one in mirrored indices, with the other
// sign of dG.
//
// What bounds it is the chain of dependent steps, mx + my + mz of them at 0.7
// us, and the hand-overs, 3 us each beyond the steps.  The form before it ran
// tiles of 4 x 8 x 8 cells, one launch per tile hyperplane, with two barriers per
// step and the neighbours' terms formed by the consumer: 96x80x64 cells with 9
// species took 80 launches of 39 us per solve, now two of 0.36 ms.  Measured on
// the way: one wavefront that also moves the cells 1.1 us per step; hand-over
// records by cell instead of by step (scattered stores) 0.47 ms per sweep;
// chunks of 4 steps, with three workgroups per CU, 0.42 (the workgroups of a CU
// meet on one SIMD), with one 0.35, but 7% slower than 8 on larger blocks.
constexpr int kLuCols = kLuP * kLuP, kLuG = 8;
constexpr int kLuHeld = kLuCols * kLuG / 64;  // cells of a chunk per lane of the second wavefront
static_assert(kLuCols == 16, "the columns of a variable group are one DPP row");
constexpr unsigned long long kLuNone = 0x7FF4DEADBEEF5AA5ull;  // a signalling NaN: no result of arithmetic is one
constexpr long long kLuWait = 1000000000ll;                    // of the 100 MHz clock: 10 s
constexpr int kLuFlag = 2;                                     // in the context's error flags

// v of the lane N before this one in its row of 16, or in the row's first N lanes
// `first`
template <int N>
__device__ __forceinline__ double row_up(double first, double v) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(first), __double2loint(v), 0x110 | N, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(first), __double2hiint(v), 0x110 | N, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// the first row's v in every row (the odd rows swapped with the even ones of a
// copy, then the halves of the wavefront)
__device__ __forceinline__ double first_row(double v) {
  auto word = [](unsigned x) {
    const unsigned y = __builtin_amdgcn_permlane16_swap(x, x, false, false)[0];
    return __builtin_amdgcn_permlane32_swap(y, y, false, false)[0];
  };
  return __hiloint2double((int)word((unsigned)__double2hiint(v)), (int)word((unsigned)__double2loint(v)));
}

// every place of a hand-over empty, the ticket counter and the abort word back to 0
__global__ void __launch_bounds__(kTpb) lusgs_reset_kernel(const BlockView *__restrict__ views,
                                                           const int *__restrict__ off, int nb, int *ticket) {
  const PointWork pw = point_work(off, nb);
  const GView B = gview(views[pw.blk]);
  const long long q = pw.base + threadIdx.x;
  if (blockIdx.x == 0 && threadIdx.x == 0) ticket[0] = ticket[1] = 0;
  if (q >= B.ni) return;
  const int m[3] = {B.mx, B.my, B.mz};
  const long long n = lu_hand_over(m, NS);
  gptr<unsigned long long> f = (gptr<unsigned long long>)B.luf;
  for (long long x = q; x < n; x += B.ni) f[x] = kLuNone;
}

template <bool FWD>
__global__ void __launch_bounds__(128, 1) lusgs_sweep_kernel(const BlockView *__restrict__ views,
                                                            const LuPatch *__restrict__ order, int n_patch,
                                                            int *ticket, SchemeDev S, int *flags) {
  // variables of a lane (group 0 has 5); places of a cell's variables, group by group
  constexpr int NV = 5 + NS, N3 = lu_third(NS), NSL = N3 > 5 ? N3 : 5, NP = lu_places(NS);
  static_assert(N3 <= 5, "the groups after the first hold at most its 5 variables");
  // a staged cell: dQ (R or dQ* until it is updated), state (the energy's place
  // holds E + p), S_d = J grad xi_d (3 x 3), a_d, U_d / 2 (its sign as in the
  // sweep's terms), 1/D, gamma - 1, kinetic energy
  constexpr int XC = NP, XS = 2 * NP, XA = XS + 9, XU = XA + 3, XI = XU + 3, XG = XI + 1, XK = XG + 1, RS = (XK + 1) | 1;
  constexpr double SG = FWD ? 0.5 : -0.5;
  constexpr int CHUNK = kLuG * kLuCols * RS;
  __shared__ double rec[2 * CHUNK];
  __shared__ int mine;
  const int lane = threadIdx.x & 63;
  const bool mover = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 1;
  if (threadIdx.x == 0) mine = atomicAdd(ticket, 1);
  __syncthreads();
  const int tk = __builtin_amdgcn_readfirstlane(mine);
  if (tk >= n_patch) return;  // uniform over the workgroup
  const LuPatch pt = order[tk];
  const GView B = gview(views[pt.blk]);
  const int mx = B.mx, my = B.my, mz = B.mz;
  const long long np = B.np, ni = B.ni;
  const bool dim3_ = S.dim == 3;

  const int c = lane & 15, vg = lane >> 4, jl = c % kLuP, kl = c / kLuP;
  const int jj = pt.J * kLuP + jl, kk = pt.K * kLuP + kl;
  const bool col = jj < my && kk < mz;
  const int h0 = vg == 0 ? 0 : 5 + (vg - 1) * N3;  // this lane's places
  const int nJ = (my + kLuP - 1) / kLuP, steps = lu_steps(mx, my, mz), n_chunk = (steps + kLuG - 1) / kLuG;
  constexpr int ST = lu_record(NS);
  const long long at = (long long)pt.K * nJ + pt.J;
  typedef unsigned long long u64;
  const gptr<u64> F = (gptr<u64>)B.luf;
  const gptr<u64> FK = F + lu_along_k(NS, mx, my, mz);
  const bool need_j = col && jl == 0 && jj > 0, need_k = col && kl == 0 && kk > 0;
  const bool give_j = col && jl == kLuP - 1 && jj + 1 < my, give_k = col && kl == kLuP - 1 && kk + 1 < mz;
  gptr<u64> in_j = F + lu_at(NS, steps, at - 1, kLuAhead, vg, kl);
  gptr<u64> in_k = FK + lu_at(NS, steps, at - nJ, kLuAhead, vg, jl);
  gptr<u64> out_j = F + lu_at(NS, steps, at, 0, vg, kl), out_k = FK + lu_at(NS, steps, at, 0, vg, jl);
  auto place = [](int q) { return lu_place(NS, q); };  // this lane's value q in a step's record

  if (mover) {
    // ---- the second wavefront moves the cells: lane e + kLuG (column % 8) holds
    // cell e of a chunk, of one column in each half.  While chunk n is worked on
    // it takes chunk n - 1 out of LDS, puts chunk n + 1 there and loads chunk n + 2.
    const int e = lane % kLuG;
    long long row[kLuHeld], prow[kLuHeld];
    int i00[kLuHeld];
    bool real[kLuHeld];
    double *own[kLuHeld];
#pragma unroll
    for (int h = 0; h < kLuHeld; ++h) {
      const int cr = lane / kLuG + 64 / kLuG * h, j0 = pt.J * kLuP + cr % kLuP, k0 = pt.K * kLuP + cr / kLuP;
      const int jc = min(j0, my - 1), kc = min(k0, mz - 1), j = FWD ? jc : my - 1 - jc, k = FWD ? kc : mz - 1 - kc;
      row[h] = ((long long)k * my + j) * mx;
      prow[h] = pidx(B, 0, j, k);
      i00[h] = e - cr % kLuP - cr / kLuP;
      real[h] = j0 == jc && k0 == kc;
      own[h] = rec + (e * kLuCols + cr) * RS;
    }
    auto cell = [&](int n, int h, int &i) {  // of chunk n, whether it is on the block
      const int im = n * kLuG + i00[h], ic = min(max(im, 0), mx - 1);
      i = FWD ? ic : mx - 1 - ic;
      return im == ic && real[h];
    };
    double xx[kLuHeld][2 * NV], mm[kLuHeld][16];
    auto load = [&](int n) {
#pragma unroll
      for (int h = 0; h < kLuHeld; ++h) {
        int i;
        cell(n, h, i);
        const long long q = row[h] + i, p = prow[h] + i;
        double *x = xx[h], *m = mm[h];
#pragma unroll
        for (int l = 0; l < NV; ++l) x[l] = B.dq[l * ni + q], x[NV + l] = B.cv[l * np + p];
#pragma unroll
        for (int v = 0; v < 9; ++v) m[v] = B.metric[v * np + p];
#pragma unroll
        for (int v = 0; v < 4; ++v) m[9 + v] = B.lus[v * ni + q];
        m[13] = B.jac[p];
        m[14] = B.bv[4 * np + p];
        m[15] = B.props[p];
      }
    };
    auto stage = [&](int n) {
#pragma unroll
      for (int h = 0; h < kLuHeld; ++h) {
        int i;
        const bool in = cell(n, h, i);
        double *r = own[h] + (n & 1) * CHUNK;
        const double *x = xx[h], *m = mm[h], *q0 = x + NV;
        const double J = in ? m[13] : 0.0;  // cells off the block: no terms
        const double r0 = frcp<double>(q0[0]);
#pragma unroll
        for (int l = 0; l < NP; ++l) {
          r[l] = l < NV && in ? x[l < NV ? l : 0] : 0.0;
          r[XC + l] = l == 4 ? q0[4] + m[14] : (l < NV ? q0[l < NV ? l : 0] : 0.0);
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const double Sx = J * m[3 * d], Sy = J * m[3 * d + 1], Sz = J * m[3 * d + 2];
          r[XS + 3 * d] = Sx, r[XS + 3 * d + 1] = Sy, r[XS + 3 * d + 2] = Sz;
          r[XU + d] = SG * ((Sx * q0[1] + Sy * q0[2] + Sz * q0[3]) * r0);
          r[XA + d] = in ? m[10 + d] : 0.0;
        }
        r[XI] = frcp<double>(m[9]);
        r[XG] = m[15] - 1;
        r[XK] = (0.5 * (q0[1] * q0[1] + q0[2] * q0[2] + q0[3] * q0[3])) * r0;
      }
    };
    auto take = [&](int n) {
#pragma unroll
      for (int h = 0; h < kLuHeld; ++h) {
        int i;
        if (!cell(n, h, i)) continue;
        const double *r = own[h] + (n & 1) * CHUNK;
#pragma unroll
        for (int l = 0; l < NV; ++l) B.dq[l * ni + row[h] + i] = r[l];
      }
    };
    load(0);
    stage(0);
    if (n_chunk > 1) load(1);
    for (int n = 0; n < n_chunk; ++n) {
      __syncthreads();
      if (n > 0) take(n - 1);
      if (n + 1 < n_chunk) stage(n + 1);
      if (n + 2 < n_chunk) load(n + 2);
    }
    __syncthreads();
    take(n_chunk - 1);
    return;
  }

  struct Cell {
    double R[NSL], q0[NSL], S[9], a[3], U[3], rD, gm, ke;
  };
  auto read = [&](const double *chunk, int t, Cell &x) {
    const double *r = chunk + (t * kLuCols + c) * RS;
#pragma unroll
    for (int q = 0; q < NSL; ++q) {
      const int v = q < N3 ? h0 + q : q;
      x.R[q] = r[v], x.q0[q] = r[XC + v];
    }
#pragma unroll
    for (int v = 0; v < 9; ++v) x.S[v] = r[XS + v];
#pragma unroll
    for (int v = 0; v < 3; ++v) x.a[v] = r[XA + v], x.U[v] = r[XU + v];
    x.rD = r[XI], x.gm = r[XG], x.ke = r[XK];
  };

  // ---- terms from the patches before this one and to those after it; a place
  // past a lane's N3 is one of group 0
  // and a lane that needs no term keeps the zeros
  u64 ij[2][NSL] = {}, ik[2][NSL] = {};
  auto fetch = [&](bool now, gptr<u64> from, u64 *in) {
    if (now) {
#pragma unroll
      for (int q = 0; q < N3; ++q)
        in[q] = __hip_atomic_load((u64 *)(from + place(q)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (vg == 0) {
#pragma unroll
        for (int q = N3; q < NSL; ++q)
          in[q] = __hip_atomic_load((u64 *)(from + place(q)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  };
  auto give = [&](bool on, gptr<u64> to, const double *T) {
    if (on) {
#pragma unroll
      for (int q = 0; q < N3; ++q)
        __hip_atomic_store((u64 *)(to + place(q)), (u64)__double_as_longlong(T[q]), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      if (vg == 0) {
#pragma unroll
        for (int q = N3; q < NSL; ++q)
          __hip_atomic_store((u64 *)(to + place(q)), (u64)__double_as_longlong(T[q]), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  };
  auto missing = [&](const u64 *x, const u64 *y) {  // by the high words
    unsigned m = ~0u;
#pragma unroll
    for (int q = 0; q < NSL; ++q)
      m = min(min(m, (unsigned)(x[q] >> 32) ^ (unsigned)(kLuNone >> 32)), (unsigned)(y[q] >> 32) ^ (unsigned)(kLuNone >> 32));
    return m == 0;
  };

  double T0[NSL], T1[NSL], T2[NSL];
#pragma unroll
  for (int q = 0; q < NSL; ++q) T0[q] = T1[q] = T2[q] = 0.0;
  auto now = [&](bool need, int s) { return need && lu_active(mx, jl, kl, s); };
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    fetch(now(need_j, s), in_j + s * ST, ij[s]);
    fetch(now(need_k, s), in_k + s * ST, ik[s]);
  }
  for (int n = 0; n < n_chunk; ++n) {
    __syncthreads();
    double *const chunk = rec + (n & 1) * CHUNK;
    Cell cell[2];
    read(chunk, 0, cell[0]);
#pragma unroll 2
    for (int t = 0; t < kLuG; ++t) {
      const int s = n * kLuG + t;
      const bool act = col && lu_active(mx, jl, kl, s);
      const Cell &x = cell[t & 1];
      read(chunk, min(t + 1, kLuG - 1), cell[(t + 1) & 1]);
      u64 *aj = ij[t & 1], *ak = ik[t & 1];
      lu_wait([&] { return __any(missing(aj, ak)) != 0; },
              [&] {  // (a patch that waits for its first terms leaves the memory to the others)
                if (s < kLuP) __builtin_amdgcn_s_sleep(16);
                if (missing(aj, ak)) {
                  fetch(now(need_j, s), in_j, aj);
                  fetch(now(need_k, s), in_k, ak);
                }
              },
              [] { return (long long)wall_clock64(); }, kLuWait,
              [&] {
                atomicOr(flags, kLuFlag);
                __hip_atomic_store(ticket + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              },
              [&] { return __hip_atomic_load(ticket + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0; });
      double dn[NSL];
#pragma unroll
      for (int q = 0; q < NSL; ++q) {
        const double uj = row_up<1>(0.0, T1[q]), uk = row_up<kLuP>(__longlong_as_double((long long)ak[q]), T2[q]);
        const double acc = (FWD ? x.R[q] + T0[q] : T0[q]) + (jl == 0 ? __longlong_as_double((long long)aj[q]) : uj) + uk;
        dn[q] = FWD ? acc * x.rD : x.R[q] + acc * x.rD;
      }
      in_j += ST, in_k += ST;
      fetch(now(need_j, s + 2), in_j + ST, aj);
      fetch(now(need_k, s + 2), in_k + ST, ak);
      double *r = chunk + (t * kLuCols + c) * RS + h0;
#pragma unroll
      for (int q = 0; q < N3; ++q) r[q] = dn[q];
      if (vg == 0) {
#pragma unroll
        for (int q = N3; q < NSL; ++q) r[q] = dn[q];
      }
      // velocities and pressure change of the new state: group 0's, for all groups
      const double m0 = x.q0[0] + dn[0], m1 = x.q0[1] + dn[1], m2 = x.q0[2] + dn[2], m3 = x.q0[3] + dn[3];
      const double r1 = frcp<double>(m0);
      double U1[3];
#pragma unroll
      for (int d = 0; d < 3; ++d)
        U1[d] = first_row((x.S[3 * d] * m1 + x.S[3 * d + 1] * m2 + x.S[3 * d + 2] * m3) * r1);
      const double dp = x.gm * (dn[4] - ((0.5 * (m1 * m1 + m2 * m2 + m3 * m3)) * r1 - x.ke));
      const double hp = vg == 0 ? SG * dp : 0.0;
      // +-dG_d / 2 + a_d dQ with dG = dQ U1 + Q (U1 - U) (+ p terms)
      auto terms = [&](int d, double *T) {
        const double h1 = x.a[d] + SG * U1[d], h2 = SG * U1[d] - x.U[d];
#pragma unroll
        for (int q = 0; q < NSL; ++q) {
          T[q] = dn[q] * h1 + x.q0[q] * h2;
          if (q >= 1 && q <= 3) T[q] += x.S[3 * d + q - 1] * hp;
          if (q == 4) T[q] += U1[d] * hp;
        }
      };
      terms(1, T1);
      give(act && give_j, out_j, T1);
      if (dim3_) {
        terms(2, T2);
        give(act && give_k, out_k, T2);
      }
      terms(0, T0);
      out_j += ST, out_k += ST;
    }
  }
  __syncthreads();  // the last chunk is done
}

int launch_lusgs_coef(const Batch &b, const SchemeDev &S, hipStream_t st) {
  if (b.total <= 0) return 0;
  lusgs_coef_kernel<<<b.total, kTpb, 0, st>>>(b.views, b.off, b.nb, S);
  return (int)hipGetLastError();
}

int launch_lusgs_reset(const Batch &b, int *ticket, hipStream_t st) {
  if (b.total <= 0) return 0;
  lusgs_reset_kernel<<<b.total, kTpb, 0, st>>>(b.views, b.off, b.nb, ticket);
  return (int)hipGetLastError();
}

int launch_lusgs_sweep(const BlockView *views, const LuPatch *order, int n, int *ticket, const SchemeDev &S, int fwd,
                       int *flags, hipStream_t st) {
  if (n <= 0) return 0;
  if (fwd)
    lusgs_sweep_kernel<true><<<n, 128, 0, st>>>(views, order, n, ticket, S, flags);
  else
    lusgs_sweep_kernel<false><<<n, 128, 0, st>>>(views, order, n, ticket, S, flags);
  return (int)hipGetLastError();
}

int launch_cv_from_bv(const Batch &b, const SpeciesDev *sp, const SchemeDev &S, hipStream_t st) {
  if (b.total <= 0) return 0;
  cv_from_bv_kernel<<<b.total, kTpb, 0, st>>>(b.views, b.off, b.nb, sp, S);
  return (int)hipGetLastError();
}

int launch_face_ops(const BlockView *views, const FaceOp *ops, const int *off, int nops, int total,
                    const SpeciesDev *sp, const SchemeDev &S, const InflowDev *inflow, hipStream_t st) {
  if (total <= 0) return 0;
  face_ops_kernel<<<total, kTpb, 0, st>>>(views, ops, off, nops, sp, S, inflow);
  return (int)hipGetLastError();
}

int launch_copy_ops(const BlockView *views, const FaceOp *ops, const int *off, int nops, int total, int mixed,
                    hipStream_t st) {
  if (total <= 0) return 0;
  copy_ops_kernel<<<dim3(total, NS > 0 && !mixed ? 3 : 2, 1), kTpb, 0, st>>>(views, ops, off, nops);
  return (int)hipGetLastError();
}

// ------------------------------------------------- surrogate training set ---
// Counter-based uniform in [0, 1): SplitMix64 finaliser of (seed, sample, k);
// each sample owns 4096 counters (a sample draws at most 2 + ns (3*32 + 1)).
__device__ __forceinline__ double rng_uniform(unsigned long long seed, long long s, unsigned k) {
  unsigned long long z = seed + 0x9E3779B97F4A7C15ull * ((unsigned long long)s * 4096ull + k + 1ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

// Gamma(a, 1) by Marsaglia & Tsang (2000), "A simple method for generating
// gamma variables", with the boost G(a) = G(a+1) U^(1/a) for a < 1; normals
// by Box-Muller.  Bounded: after 32 rejections the mode is returned.
__device__ __forceinline__ double rng_gamma(unsigned long long seed, long long s, unsigned &k, double a) {
  const double aa = a < 1.0 ? a + 1.0 : a;
  const double d = aa - 1.0 / 3.0, c = 1.0 / sqrt(9.0 * d);
  double g = d;
  for (int it = 0; it < 32; ++it) {
    const double u1 = rng_uniform(seed, s, k++), u2 = rng_uniform(seed, s, k++);
    const double z = sqrt(-2.0 * log(1.0 - u1)) * cos(6.283185307179586 * u2);
    const double v1 = 1.0 + c * z;
    if (v1 <= 0.0) continue;
    const double v = v1 * v1 * v1;
    const double u = rng_uniform(seed, s, k++);
    if (log(1.0 - u) < 0.5 * z * z + d - d * v + d * log(v)) {
      g = d * v;
      break;
    }
  }
  if (a < 1.0) g *= pow(1.0 - rng_uniform(seed, s, k++), 1.0 / a);
  return g;
}

// Sample s: T ~ U[t_lo, t_hi], log p ~ U[lp_lo, lp_hi], Y ~ Dirichlet(alpha);
// inputs x = (T, log p, Y) and targets y = log(mu, kappa, rho*D_l) of the
// FP64 transport routine.
__global__ void __launch_bounds__(256) mlp_samples_kernel(const SpeciesDev *__restrict__ spg, SchemeDev S,
                                                          long long n, unsigned long long seed, double t_lo,
                                                          double t_hi, double lp_lo, double lp_hi, double alpha,
                                                          double *__restrict__ x, double *__restrict__ y) {
  const SpeciesPtrT<double> sp = const_table<double>(spg);
  const long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  unsigned k = 0;
  const double t = t_lo + (t_hi - t_lo) * rng_uniform(seed, s, k++);
  const double lp = lp_lo + (lp_hi - lp_lo) * rng_uniform(seed, s, k++);
  double Y[NSA], sum = 0.0;
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    Y[l] = rng_gamma(seed, s, k, alpha);
    sum += Y[l];
  }
  const double inv = sum > 0.0 ? 1.0 / sum : 0.0;
#pragma unroll
  for (int l = 0; l < NS; ++l) Y[l] = sum > 0.0 ? Y[l] * inv : 1.0 / NS;
  double cp[NSA], winv, gc[2], out[2 + NSA];
  mixture_gamma_c<double>(sp, nullptr, t, Y, cp, winv, gc);
  wilke_point<double>(sp, S, t, Y, cp, winv, out);
  double *xr = x + s * (NS + 2), *yr = y + s * (NS + 2);
  xr[0] = t;
  xr[1] = lp;
#pragma unroll
  for (int l = 0; l < NS; ++l) xr[2 + l] = Y[l];
#pragma unroll
  for (int o = 0; o < NS + 2; ++o) yr[o] = log(out[o]);
}

int launch_mlp_samples(const SpeciesDev *sp, const SchemeDev &S, long long n, unsigned long long seed,
                       const double lim[4], double alpha, double *x, double *y, hipStream_t st) {
  if constexpr (NS == 0) {
    return CFX_E_UNSUPPORTED;
  } else {
    if (n <= 0) return 0;
    mlp_samples_kernel<<<(int)((n + 255) / 256), 256, 0, st>>>(sp, S, n, seed, lim[0], lim[1], lim[2], lim[3],
                                                                alpha, x, y);
    return (int)hipGetLastError();
  }
}

struct Register64 {
  Register64() {
    KernelSet64 &k = g_kernels64[NS];
    k.mlp_samples = launch_mlp_samples;
    k.props = launch_props<double>;
    k.cv_from_bv = launch_cv_from_bv;
    k.update = launch_update;
    k.face_ops = launch_face_ops;
    k.copy_ops = launch_copy_ops;
    k.lusgs_coef = launch_lusgs_coef;
    k.lusgs_reset = launch_lusgs_reset;
    k.lusgs_sweep = launch_lusgs_sweep;
    register_rhs<double>(k);
    k.present = 1;
  }
} register64;

#else  // CFX_PREC == 32

// ----------------------------------------------- properties, MLP transport ---
// The mixed-precision properties with mu, kappa and rho*D from the surrogate.
// Each wavefront evaluates its 64 points as four 16-point MFMA tiles (inputs
// and outputs pass through a per-wavefront LDS buffer between the
// point-per-lane and the tile layouts).  Points outside the training envelope
// take the Wilke routine; one chunk-wavefront in check_every of each
// workgroup also evaluates Wilke at all its points and keeps Wilke where the
// surrogate is off by more than check_tol.  The work runs in three phases so
// that each holds only its own registers: (1) FP32 primitives, Y, gamma, c
// and the network inputs, with every output but the transport coefficients
// stored at once; (2) the network; (3) the coefficients, with the Wilke
// fallback recomputing its inputs from the FP64 state.
// counters: [0] points outside, [1] points checked, [2] checks failed.

// Orders the LDS accesses of one wavefront (its lanes exchange values through
// its own slice of LDS, so no workgroup barrier is needed).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Phase 1 from the FP32 primitives b32 (rho, u, v, w, p, T) and Y of padded
// point p (byte offset o4 in the FP32 arrays): the network inputs go to
// xl[lane], and with store set gamma, c and the FP32 copies are written.
// Returns whether the point lies outside the training envelope.
__device__ __forceinline__ bool mlp_phase1(const GView &B, SpeciesPtrT<float> sp, const MlpDev *__restrict__ mlp,
                                           const float *b32, const float *Y, float (*xl)[kMlpIO + 1], bool store,
                                           unsigned o4) {
  const int lane = threadIdx.x & 63;
  const long long np = B.np;
  float cp[NSA], winv, gc[2], x[kMlpIO];
  mixture_gamma_c<float>(sp, nullptr, b32[5], Y, cp, winv, gc);
  float ymax = 0.0f;  // largest Y_l / W_l: the largest mole fraction times winv
#pragma unroll
  for (int l = 0; l < NS; ++l) ymax = fmaxf(ymax, Y[l] * sp->inv_mw[l]);
  const bool outside = mlp_inputs<NS>(mlp, b32[5], flog<float>(b32[4]), Y, x, ymax * frcp<float>(winv));
#pragma unroll
  for (int f = 0; f < kMlpIO; ++f) xl[lane][f] = x[f];
  if (store) {
    *atg<float>(B.props32, o4) = gc[0];
    *atg<float>(B.props32 + np, o4) = gc[1];
#pragma unroll
    for (int v = 0; v < 6; ++v) *atg<float>(B.bv32 + v * np, o4) = b32[v];
#pragma unroll
    for (int l = 0; l < NS; ++l) *atg<float>(B.yk32 + l * np, o4) = Y[l];
  }
  return outside;
}

// Phases 2 and 3 for the wavefront: the network on xl with the operands
// staged in LDS, the coefficients, the Wilke fallback (its inputs reloaded
// from the FP64 state at byte offset o8; at every point when check is set),
// the counters over the lanes with store set, and their stores.
__device__ __forceinline__ void mlp_phase23(const GView &B, SpeciesPtrT<float> sp, const SchemeDev &S,
                                            const MlpDev *__restrict__ mlp, lds_ptr<const bf16x8> ops,
                                            lds_ptr<const f32x4> bias, unsigned long long *__restrict__ counters,
                                            float (*xl)[kMlpIO + 1], bool outside, bool store, unsigned o8,
                                            unsigned o4, bool check) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  wave_sync();
  {
    bf16x8 xo[4];
    f32x4 yv[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int j = 0; j < 4; ++j) xo[tt][j] = (__bf16)xl[16 * tt + c][4 * g + j], xo[tt][4 + j] = (__bf16)0.0f;
    wave_sync();
    mlp_infer_tiles<4>(ops, bias, xo, yv);
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int r = 0; r < 4; ++r) xl[16 * tt + c][4 * g + r] = yv[tt][r];
  }
  wave_sync();
  // fresh copies of the uniform bases, so that the field addresses of the
  // first phase need not stay live (in SGPRs) through the network
  gptr<const double> cvb = B.cv, bvb = B.bv;
  gptr<float> prb = B.props32;
  long long npl = B.np;
  asm volatile("" : "+s"(cvb), "+s"(bvb), "+s"(prb), "+s"(npl));
  float tr[2 + NSA];
#pragma unroll
  for (int o = 0; o < NS + 2; ++o) tr[o] = __expf(xl[lane][o] * mlp->t_std[o] + mlp->t_mean[o]);
  bool fail = false;
  if (check || outside) {
    float Y[NSA], cp[NSA], winv, gc[2], w[2 + NSA];
    const float t = float(ldg<double>(bvb + 5 * npl, o8));
    const double ir = 1.0 / ldg<double>(cvb, o8);
#pragma unroll
    for (int l = 0; l < NS; ++l) Y[l] = float(ldg<double>(cvb + (5 + l) * npl, o8) * ir);
    mixture_gamma_c<float>(sp, nullptr, t, Y, cp, winv, gc);
    wilke_point<float>(sp, S, t, Y, cp, winv, w);
    if (check) {
#pragma unroll
      for (int o = 0; o < NS + 2; ++o) fail = fail || !(fabsf(tr[o] - w[o]) <= mlp->check_tol * fabsf(w[o]));
    }
    if (outside || fail) {
#pragma unroll
      for (int o = 0; o < NS + 2; ++o) tr[o] = w[o];
    }
  }
  const unsigned long long n_out = __ballot(store && outside), n_chk = __ballot(store && check),
                           n_fail = __ballot(store && fail);
  if (lane == 0) {
    if (n_out) atomicAdd(&counters[0], (unsigned long long)__popcll(n_out));
    if (n_chk) atomicAdd(&counters[1], (unsigned long long)__popcll(n_chk));
    if (n_fail) atomicAdd(&counters[2], (unsigned long long)__popcll(n_fail));
  }
  if (!store) return;
#pragma unroll
  for (int o = 0; o < NS + 2; ++o) *atg<float>(prb + (2 + o) * npl, o4) = tr[o];
}

// Surrogate properties over the padded range.  A persistent grid: workgroup
// b walks the kTpb-point chunks b, b + gridDim.x, ... of the batch, and loads
// the FP64 inputs of its next chunk before the network runs on the current
// one, so that those loads overlap the arithmetic.  The inference operands
// are staged in LDS once per workgroup: the network then issues no vector
// memory instruction whose wait would also wait for the prefetch.
constexpr int kMlpInfBlocks = kB4;  // forward A operands (the first kB4 blocks)
constexpr int kMlpIn = 7 + NS;      // rho, u, v, w, p, T, rho and rho*Y_l of one point

__device__ __forceinline__ void mlp_fetch(const BlockView *__restrict__ views, const int *__restrict__ off, int nb,
                                          int w, double *in) {
  const int gw = w + off[0];
  const int blk = find_seg(off, nb, gw);
  const GView B = gview(views[blk]);
  const long long np = B.np;
  const long long p0 = (long long)(gw - off[blk]) * kTpb + threadIdx.x;
  const unsigned o8 = unsigned(p0 < np ? p0 : np - 1) * 8u;
#pragma unroll
  for (int v = 0; v < 6; ++v) in[v] = ldg<double>(B.bv + v * np, o8);
  in[6] = ldg<double>(B.cv, o8);
#pragma unroll
  for (int l = 0; l < NS; ++l) in[7 + l] = ldg<double>(B.cv + (5 + l) * np, o8);
}

__global__ void __launch_bounds__(kTpb) props_mlp_kernel(const BlockView *__restrict__ views,
                                                         const int *__restrict__ off, int nb, int total,
                                                         const SpeciesDev *__restrict__ spg, SchemeDev S,
                                                         const MlpDev *__restrict__ mlp,
                                                         const bf16x8 *__restrict__ ops,
                                                         const float *__restrict__ bias,
                                                         unsigned long long *__restrict__ counters) {
  __shared__ float buf[kTpb / 64][64][kMlpIO + 1];
  __shared__ bf16x8 ops_l[kMlpInfBlocks * 64];
  __shared__ f32x4 bias_l[4 * kMlpH / 4];
  for (int e = threadIdx.x; e < kMlpInfBlocks * 64; e += kTpb) ops_l[e] = ops[e];
  if (threadIdx.x < kMlpH) bias_l[threadIdx.x] = reinterpret_cast<const f32x4 *>(bias)[threadIdx.x];
  __syncthreads();
  const lds_ptr<const bf16x8> lops = (lds_ptr<const bf16x8>)ops_l;
  const lds_ptr<const f32x4> lbias = (lds_ptr<const f32x4>)bias_l;
  const SpeciesPtrT<float> sp = const_table<float>(spg);
  float(*xl)[kMlpIO + 1] = buf[threadIdx.x >> 6];
  double in[kMlpIn];
  int w = blockIdx.x;
  mlp_fetch(views, off, nb, w, in);
  // the sampled check takes every check_every-th chunk-wavefront of each
  // workgroup, phase-shifted by the workgroup, so every workgroup carries
  // the same share of Wilke evaluations
  int ck = blockIdx.x + (threadIdx.x >> 6);
  for (; w < total; w += gridDim.x, ck += kTpb / 64) {
    const int gw = w + off[0];
    const int blk = find_seg(off, nb, gw);
    const GView B = gview(views[blk]);
    const long long np = B.np;
    const long long p0 = (long long)(gw - off[blk]) * kTpb + threadIdx.x;
    const bool valid = p0 < np;
    const long long p = valid ? p0 : np - 1;  // every lane takes part in the MFMA tiles
    // field arrays are addressed by a wave-uniform base and a 32-bit byte offset
    const unsigned o8 = unsigned(p) * 8u, o4 = unsigned(p) * 4u;
    float b32[6], Y[NSA];
#pragma unroll
    for (int v = 0; v < 6; ++v) b32[v] = float(in[v]);
    const double ir = 1.0 / in[6];
#pragma unroll
    for (int l = 0; l < NS; ++l) Y[l] = float(in[7 + l] * ir);
    wave_sync();  // the previous chunk's reads of xl come first
    const bool outside = mlp_phase1(B, sp, mlp, b32, Y, xl, valid, o4);
    if (w + (int)gridDim.x < total) mlp_fetch(views, off, nb, w + gridDim.x, in);
    mlp_phase23(B, sp, S, mlp, lops, lbias, counters, xl, outside, valid, o8, o4, ck % mlp->check_every == 0);
  }
}

int launch_props_mlp(const Batch &b, const SpeciesDev *sp, const SchemeDev &S, const MlpDev *mlp, const void *ops,
                     const float *bias, unsigned long long *counters, hipStream_t st) {
  if constexpr (NS == 0 || NS > kMlpMaxSp) {
    return CFX_E_UNSUPPORTED;
  } else {
    if (b.total <= 0) return 0;
    // persistent grid: the resident workgroups of the current device (cached
    // per device; concurrent first calls compute the same value)
    constexpr int kMaxDev = 64;
    static std::atomic<int> resident[kMaxDev] = {};
    int dev = 0;
    (void)hipGetDevice(&dev);
    int r = dev >= 0 && dev < kMaxDev ? resident[dev].load(std::memory_order_relaxed) : 0;
    if (!r) {
      int n_cu = 0, per_cu = 0;
      if (hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) n_cu = 256;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, props_mlp_kernel, kTpb, 0) != hipSuccess)
        per_cu = 1;
      r = std::max(1, n_cu * std::max(1, per_cu));
      if (dev >= 0 && dev < kMaxDev) resident[dev].store(r, std::memory_order_relaxed);
    }
    const int grid = std::min(b.total, r);
    props_mlp_kernel<<<grid, kTpb, 0, st>>>(b.views, b.off, b.nb, b.total, sp, S, mlp, (const bf16x8 *)ops, bias,
                                           counters);
    return (int)hipGetLastError();
  }
}

struct Register32 {
  Register32() {
    KernelSet32 &k = g_kernels32[NS];
    k.props_mlp = launch_props_mlp;
    k.props = launch_props<float>;
    register_rhs<float>(k);
    k.present = 1;
  }
} register32;

#endif

}  // namespace

}  // namespace cfx
