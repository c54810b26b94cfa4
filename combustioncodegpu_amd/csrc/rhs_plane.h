// rhs_plane.h — the RHS of a 2-D block in one launch (3-D: rhs_march.h).
//
// A workgroup owns TX x TY cells of the plane k = 0.  Every primitive variable
// (rho, u, v, w, p, T, Y) of the tile and two halo cells around it goes to LDS
// once; then one face per thread: the first four wavefronts hold the x faces
// ((TX + 1) x TY), the other four the y faces (TX x (TY + 1)), so that
// everything that depends on the direction is uniform in a wavefront.  MUSCL
// and AUSM+ (InviscidScheme.cu:24-108 via Reconstruction.cu:12-89) and the
// viscous flux (ViscousScheme.cu:11-342) go to the thread's LDS slot, and the
// cell differences of both directions are written as dq, once.
//
// PLANAR: the ghost planes k = -1, 1 hold the plane's own values, so that the
// differences along k are zero and are left out.  Otherwise they come from
// memory.
//
// It replaces one launch per direction that staged the variables of three
// planes in batches: 1021x509 air, FP64, minmod: 76 us per evaluation ->
// 31.5 (PLANAR), 48.7 (with the differences along k).  Bound by the latency of
// a workgroup's one round of loads and by the vector ALU; its compulsory
// traffic (176 B per cell) takes 19 us.
//
// Tiles: 16 x 15 cells fill the 512 threads with 255 + 256 faces and stage
// 1.58 points per cell; 32 x 7 cells (variant 1) 231 + 256 and 1.77.
#pragma once

#include "device_physics.h"

namespace cfx {

template <int NS, int TX, int TY, typename R>
struct PlaneShape {
  static constexpr int NT = 512, NV = 5 + NS, NVS = 6 + NS;  // threads; fluxes; staged variables (with T)
  static constexpr int W0 = TX + 4, PL = W0 * (TY + 4);
  static constexpr int FB = NVS * PL;                            // flux slots, one per thread and variable
  static constexpr int MIX = (FB + NV * NT + 3) / 4 * 4, TOTAL = MIX + 24 * NS;  // mixture coefficients (16-byte reads)
  static_assert((TX + 1) * TY <= 256 && TX * (TY + 1) <= 256 && PL <= NT, "one face and one staged point per thread");
  static_assert(TOTAL * sizeof(R) <= 163840, "the plane and the fluxes fit in LDS");
};

template <int NS, int TX, int TY, int WPE, typename R, bool PLANAR>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
    rhs_plane_kernel(const BlockView *__restrict__ views, const int *__restrict__ off, int nb, int padded,
                     const SpeciesDev *__restrict__ spg, SchemeDev S) {
  using P = PlaneShape<NS, TX, TY, R>;
  using Fd = Fields<R>;
  constexpr int NV = P::NV, NVS = P::NVS, W0 = P::W0, PL = P::PL, NT = P::NT;
  __shared__ __attribute__((aligned(16))) R sm[P::TOTAL];
  const SpeciesPtrT<R> sp = const_table<R>(spg);
  const int total = off[nb] - off[0];
  // workgroups are dealt to the 8 XCDs round-robin: each works through a
  // contiguous run of tiles and keeps their halos in its own L2
  const int lid = ((int)blockIdx.x & 7) * (padded >> 3) + ((int)blockIdx.x >> 3);
  if (lid >= total) return;  // uniform per workgroup
  const int wgi = __builtin_amdgcn_readfirstlane(lid + off[0]);
  const int blk = __builtin_amdgcn_readfirstlane(find_seg(off, nb, wgi));
  const GView B = gview(views[blk]);
  const gptr<const R> __restrict__ BV_ = Fd::bv(B);
  const gptr<const R> __restrict__ YK_ = Fd::yk(B);
  const gptr<const R> __restrict__ PR_ = Fd::props(B);
  const gptr<const R> __restrict__ MT_ = Fd::metric(B);
  const gptr<const R> __restrict__ JC_ = Fd::jac(B);
  const int mx = B.mx, my = B.my;
  const long long np = B.np;
  const int ntx = (mx + TX - 1) / TX, q0 = wgi - off[blk];
  const int x0 = q0 % ntx * TX, y0 = q0 / ntx * TY;
  const int tid = threadIdx.x;
  const unsigned syb = (unsigned)B.sy * sizeof(R), szb = (unsigned)B.sz * sizeof(R), zb = (unsigned)kNgg * szb;

  // ---- this thread's face: the left point is (x0 + fi, y0 + fj)
  const bool isx = __builtin_amdgcn_readfirstlane(tid >> 6) < 4;  // uniform per wavefront
  const int f = tid & 255;
  const int fi = isx ? f % (TX + 1) - 1 : f % TX, fj = isx ? f / (TX + 1) : f / TX - 1;
  const int gx = x0 + fi, gy = y0 + fj;
  const bool ok = f < (isx ? (TX + 1) * TY : TX * (TY + 1)) && gx < mx && gy < my;
  // threads without a face work on the tile's first cell (in bounds, not used)
  const int el = ok ? (fj + 2) * W0 + fi + 2 : 2 * W0 + 2;
  const unsigned pl_b = ((unsigned)((ok ? gy : y0) + kNgg) * (unsigned)B.sy + (unsigned)((ok ? gx : x0) + kNgg)) *
                            (unsigned)sizeof(R) + zb;
  const unsigned dr = isx ? (unsigned)sizeof(R) : syb, pr_b = pl_b + dr;
  const bool q5 = (S.quirks & CFX_Q_METRIC_AVG) != 0 && isx;
  const unsigned pq_b = q5 ? pl_b : pr_b;  // right point of a metric the quirk does not average
  const bool viscous = S.viscous == 2;

  // ---- the plane to LDS; the face-point data behind it
  R m[9][2], fj_[2], rV[4], rD[NS > 0 ? NS : 1][2];
  {
    const int e = tid < PL ? tid : 0;
    const unsigned so = ((unsigned)(min(y0 - 2 + e / W0, my + 1) + kNgg) * (unsigned)B.sy +
                         (unsigned)(min(x0 - 2 + e % W0, mx + 1) + kNgg)) * (unsigned)sizeof(R) + zb;
    R G[NVS];
#pragma unroll
    for (int v = 0; v < NVS; ++v) G[v] = ldg<R>(v < 6 ? BV_ + v * np : YK_ + (v - 6) * np, so);
    fj_[0] = ldg<R>(JC_, pl_b), fj_[1] = ldg<R>(JC_, pr_b);
    const int ra = isx ? 0 : 3;  // rows of the metric: a along the face axis, b the other one in the plane, c along k
#pragma unroll
    for (int c = 0; c < 3; ++c) m[c][0] = ldg<R>(MT_ + (ra + c) * np, pl_b), m[c][1] = ldg<R>(MT_ + (ra + c) * np, pr_b);
    if (viscous) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const gptr<const R> b = MT_ + (3 - ra + c) * np;
        m[3 + c][0] = ldg<R>(b, pl_b), m[3 + c][1] = ldg<R>(b, pq_b);
        if constexpr (!PLANAR)
          m[6 + c][0] = ldg<R>(MT_ + (6 + c) * np, pl_b), m[6 + c][1] = ldg<R>(MT_ + (6 + c) * np, pq_b);
      }
#pragma unroll
      for (int v = 0; v < 2; ++v)
        rV[2 * v] = ldg<R>(PR_ + (2 + v) * np, pl_b), rV[2 * v + 1] = ldg<R>(PR_ + (2 + v) * np, pr_b);
    }
    if constexpr (NS > 0) {
      for (int n = tid; n < 24 * NS; n += NT) sm[P::MIX + n] = sp->mix[n / (8 * NS)][n / 8 % NS].v[n % 8];
    }
    if (tid < PL) {
#pragma unroll
      for (int v = 0; v < NVS; ++v) sm[v * PL + tid] = G[v];
    }
  }
  const ThermoLds<NS, R> th{sp, sm + P::MIX};
  __syncthreads();

  // ---- the face flux into this thread's slot
  if (ok) {
    const int da = isx ? 1 : W0, db = isx ? W0 : 1, fb = P::FB + tid;
    const R jl = fj_[0], jr = fj_[1];
    R k[3], mA[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      k[c] = R(0.5) * (jl * m[c][0] + jr * m[c][1]);
      mA[c] = R(0.5) * (m[c][0] + (q5 && c != 0 ? m[c][0] : m[c][1]));
    }
    {
      R pl[NV], pr[NV], F[NV];
      auto states = [&](auto mode) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          const R *s = sm + (v < 5 ? v : v + 1) * PL + el;  // T sits between p and Y
          const R q[1][4] = {{s[-da], s[0], s[da], s[2 * da]}};
          muscl_n<decltype(mode)::value, 1, R>(q, pl + v, pr + v);
        }
      };
      if (S.reconstruction != 2) states(std::integral_constant<int, 2>{});
      else if (S.limiter == 1) states(std::integral_constant<int, 1>{});
      else states(std::integral_constant<int, 0>{});
      ausm_from_states<NS, R>(sp, th, S, pl, pr, k[0], k[1], k[2], F);
#pragma unroll
      for (int v = 0; v < NV; ++v) sm[fb + v * NT] = F[v];
    }
    if (viscous) {
#pragma unroll
      for (int s = 0; s < NS; ++s)
        rD[s][0] = ldg<R>(PR_ + (4 + s) * np, pl_b), rD[s][1] = ldg<R>(PR_ + (4 + s) * np, pr_b);
      // four times the difference along b (and k), twice the average: the
      // factors are in mB, mC and where the average is used
      R mB[3], mC[3] = {0, 0, 0};
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        mB[c] = R(0.125) * (m[3 + c][0] + m[3 + c][1]);
        if constexpr (!PLANAR) mC[c] = R(0.125) * (m[6 + c][0] + m[6 + c][1]);
      }
      // variable n: 0..3 are u, v, w, T, then the mass fractions
      auto steps = [&](int n, R g[3], R &av) {
        const R *s = sm + (n < 3 ? n + 1 : n + 2) * PL + el;
        g[0] = s[da] - s[0];
        g[1] = (s[db] - s[-db]) + (s[da + db] - s[da - db]);
        av = s[0] + s[da];
        if constexpr (!PLANAR) {
          const gptr<const R> b = n < 4 ? BV_ + (n < 3 ? n + 1 : 5) * np : YK_ + (n - 4) * np;
          g[2] = (ldg<R>(b, pl_b + szb) - ldg<R>(b, pl_b - szb)) + (ldg<R>(b, pr_b + szb) - ldg<R>(b, pr_b - szb));
        }
      };
      auto grad = [&](int n, R d[3], R &av) {
        R g[3];
        steps(n, g, av);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          d[c] = g[0] * mA[c] + g[1] * mB[c];
          if constexpr (!PLANAR) d[c] += g[2] * mC[c];
        }
      };
      // the gradient along the face-area vector: all that T and Y_l need
      R ka = k[0] * mA[0] + k[1] * mA[1] + k[2] * mA[2];
      R kb = k[0] * mB[0] + k[1] * mB[1] + k[2] * mB[2];
      R kc = k[0] * mC[0] + k[1] * mC[1] + k[2] * mC[2];
      auto along = [&](int n, R &av) {
        R g[3];
        steps(n, g, av);
        R p = g[0] * ka + g[1] * kb;
        if constexpr (!PLANAR) p += g[2] * kc;
        return p;
      };
      R du[3], dv[3], dw[3], ua, va, wa, Ta;
      grad(0, du, ua);
      grad(1, dv, va);
      grad(2, dw, wa);
      const R dT = along(3, Ta);
      const R vis = R(0.5) * (rV[0] + rV[1]), cond = R(0.5) * (rV[2] + rV[3]);
      const R third = R(1.0 / 3.0);
      const R txx = vis * (R(4) * du[0] - R(2) * dv[1] - R(2) * dw[2]) * third;
      const R tyy = vis * (R(4) * dv[1] - R(2) * du[0] - R(2) * dw[2]) * third;
      const R tzz = vis * (R(4) * dw[2] - R(2) * du[0] - R(2) * dv[1]) * third;
      const R txy = vis * (du[1] + dv[0]);
      const R txz = vis * (du[2] + dw[0]);
      const R tyz = vis * (dv[2] + dw[1]);
      Ta *= R(0.5);
      const R G1 = k[0] * txx + k[1] * txy + k[2] * txz;
      const R G2 = k[0] * txy + k[1] * tyy + k[2] * tyz;
      const R G3 = k[0] * txz + k[1] * tyz + k[2] * tzz;
      R G4 = R(0.5) * (ua * G1 + va * G2 + wa * G3) + cond * dT;
      sm[fb + 1 * NT] -= G1;
      sm[fb + 2 * NT] -= G2;
      sm[fb + 3 * NT] -= G3;
      if constexpr (NS > 0) {
        // uc = sum_l rho D_l (k . grad Y_l): the correction velocity along k
        R dp[NS], yb[NS], uc = 0;
        ka *= R(0.5), kb *= R(0.5), kc *= R(0.5);  // the average of rho*D
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          dp[s] = (rD[s][0] + rD[s][1]) * along(4 + s, yb[s]);
          uc += dp[s];
        }
        G4 += carried_enthalpy<NS, R>(th, Ta, dp);
#pragma unroll
        for (int s = 0; s < NS; ++s) sm[fb + (5 + s) * NT] -= dp[s] - yb[s] * (R(0.5) * uc);
      }
      sm[fb + 4 * NT] -= G4;
    }
  }
  __syncthreads();

  // ---- the cell differences of both directions, half of the variables per
  // half of the workgroup
  const int c = tid & 255, ci = c % TX, cj = c / TX;
  if (c < TX * TY && x0 + ci < mx && y0 + cj < my) {
    const gptr<R> DQ = Fd::dq(B);
    const unsigned qb = (unsigned)((y0 + cj) * mx + x0 + ci) * (unsigned)sizeof(R);
#pragma unroll
    for (int h = 0; h < (NV + 1) / 2; ++h) {
      const int v = 2 * h + (tid >> 8);
      if (v >= NV) continue;
      const R *fx = sm + P::FB + v * NT + cj * (TX + 1) + ci, *fy = sm + P::FB + v * NT + 256 + c;
      *atg<R>(DQ + v * B.ni, qb) = -(fx[1] - fx[0]) - (fy[TX] - fy[0]);
    }
  }
}

}  // namespace cfx
