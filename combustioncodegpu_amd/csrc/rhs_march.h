// rhs_march.h — the RHS of all three face directions in one launch.
//
// A workgroup owns a column of TX x TY cells and marches through a chunk of
// k planes.  Three planes of every primitive variable (rho, u, v, w, p, T, Y)
// with two halo cells around the tile are held in LDS; the plane after next
// is on its way into the registers of the last wavefront, which only moves
// data, while a plane is worked on.  At step k the planes k-1, k, k+1 are
// resident and the workgroup forms
//   the x and y faces of plane k,
//   the z faces between the planes k-1 and k (the MUSCL point k-2 comes from
//   a column buffer: each z thread keeps its own value of the plane that is
//   about to be overwritten),
// one face per thread (InviscidScheme.cu:24-108 via Reconstruction.cu:12-89,
// ViscousScheme.cu:11-342).  Then the dq of plane k-1 is complete (its upper z
// flux was the missing part) and is written once; the in-plane differences of
// plane k and its lower z flux wait in LDS for the next step.
//
// Every thread runs the same instructions whatever the direction of its
// face: the LDS and memory strides along the face axes a (normal) and b, c
// (tangential, in increasing axis order) are per-thread values.  The kernel
// is therefore a third of the size of three specialised ones (it stays in
// the instruction cache) and wavefronts may hold faces of two directions.
//
// Why this and not one launch per direction (the form it replaces): there
// every variable was staged five times per cell and direction pass, the
// metric, transport and dq arrays were read or rewritten by every pass, and
// the passes waited for their staged batches (VALU busy 45% of a SIMD's
// cycles).  256x128x128 cells, 9 species, per evaluation: FP64 2.44 -> 1.12
// ms, mixed 1.15 -> 0.58 ms; 11.1 -> 2.0 GB through HBM in FP64.
//
// What bounds it now is the vector ALU: about 1350 instructions per face, and
// in FP64 seven wavefronts of faces on four SIMDs (the planes and fluxes of
// 9 species fill the LDS, so a larger tile does not fit).
#pragma once

#include "device_physics.h"

namespace cfx {

template <int NS, int TX, int TY, int NT, typename R>
struct MarchShape {
  static constexpr int NV = 5 + NS, NVS = 6 + NS;  // fluxes; staged variables (with T)
  static constexpr int W0 = TX + 4, W1 = TY + 4, PL = W0 * W1;
  static constexpr int NFZ = TX * TY, NFX = (TX + 1) * TY, NFY = TX * (TY + 1), NF = NFZ + NFX + NFY;
  static constexpr int PLP = (PL + 63) / 64 * 64;      // threads that stage one plane of one variable
  static constexpr int GRP = NT / PLP;                 // ... and how many variables go side by side
  static constexpr int KVG = (NVS + GRP - 1) / GRP;    // variables per thread
  static constexpr int SLOT = NVS * PL;                // one resident plane
  static constexpr int COL = 3 * SLOT, FB = COL + NV * NFZ, ACC = FB + NV * NF;
  static constexpr int MIX = (ACC + NV * NFZ + 3) / 4 * 4, TOTAL = MIX + 24 * NS;  // mixture coefficients (16-byte reads)
  static_assert(NFZ % 64 == 0, "a wavefront of the dq pass works on one variable");
  static_assert(NF <= NT - 64 && PLP <= NT, "one face per thread, the last wavefront moves the data");
  static_assert(MIX % 4 == 0 && TOTAL * sizeof(R) <= 163840, "the planes and fluxes fit in LDS");
};

// BIG: a block's nine metric fields pass 4 GiB, and the offset of a metric row
// needs 64 bits.
template <int NS, int TX, int TY, int NT, int WPE, typename R, bool BIG>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
    rhs_march_kernel(const BlockView *__restrict__ views, const int *__restrict__ off, int nb, int padded, int chunk,
                     const SpeciesDev *__restrict__ spg, SchemeDev S) {
  using P = MarchShape<NS, TX, TY, NT, R>;
  using Fd = Fields<R>;
  constexpr int NV = P::NV, NVS = P::NVS, W0 = P::W0, PL = P::PL, NFZ = P::NFZ, NFX = P::NFX, NF = P::NF;
  constexpr int KVG = P::KVG, SLOT = P::SLOT;
  __shared__ __attribute__((aligned(16))) R sm[P::TOTAL];
  const SpeciesPtrT<R> sp = const_table<R>(spg);
  const int total = off[nb] - off[0];
  // workgroups are dealt to the 8 XCDs round-robin: each works through a
  // contiguous run of columns and keeps their halos in its own L2
  const int lid = ((int)blockIdx.x & 7) * (padded >> 3) + ((int)blockIdx.x >> 3);
  if (lid >= total) return;  // uniform per workgroup
  const int wgi = __builtin_amdgcn_readfirstlane(lid + off[0]);
  const int blk = __builtin_amdgcn_readfirstlane(find_seg(off, nb, wgi));
  const GView B = gview(views[blk]);
  const gptr<const R> __restrict__ BV0 = Fd::bv(B);
  const gptr<const R> __restrict__ YK0 = Fd::yk(B);
  const gptr<const R> __restrict__ PR0 = Fd::props(B);
  const gptr<const R> __restrict__ MT0 = Fd::metric(B);
  const gptr<const R> __restrict__ JC0 = Fd::jac(B);
  const gptr<R> __restrict__ DQ0 = Fd::dq(B);
  const int mx = B.mx, my = B.my, mz = B.mz;
  const int ntx = (mx + TX - 1) / TX, nty = (my + TY - 1) / TY;
  const int nch = mz <= chunk ? 1 : (mz + chunk - 1) / chunk, len = (mz + nch - 1) / nch;
  const int q0 = wgi - off[blk];
  const int x0 = (q0 % ntx) * TX, y0 = (q0 / ntx) % nty * TY;
  const int k0 = q0 / (ntx * nty) * len, k1 = min(k0 + len, mz);
  if (k0 >= k1) return;  // uniform per workgroup
  const int tid = threadIdx.x;
  const unsigned syb = (unsigned)B.sy * sizeof(R), szb = (unsigned)B.sz * sizeof(R);

  // the mixture coefficients of all ranges
  if constexpr (NS > 0) {
    for (int n = tid; n < 24 * NS; n += NT) sm[P::MIX + n] = sp->mix[n / (8 * NS)][n / 8 % NS].v[n % 8];
  }
  const ThermoLds<NS, R> th{sp, sm + P::MIX};

  // ---- staging: thread tid holds point e of KVG variables of its group
  const int gid = __builtin_amdgcn_readfirstlane(tid / P::PLP);
  const int e = tid - gid * P::PLP;
  const bool stager = gid < P::GRP && e < PL;
  const int ec = e < PL ? e : 0;
  unsigned so = ((unsigned)(min(y0 - 2 + ec / W0, my + 1) + kNgg) * (unsigned)B.sy +
                 (unsigned)(min(x0 - 2 + ec % W0, mx + 1) + kNgg)) * (unsigned)sizeof(R) +
                (unsigned)(k0 - 1 + kNgg) * szb;
  // variable of place q: the last group repeats variable NVS-1 where it has none left
  auto fetch = [&](gptr<const R> bv, gptr<const R> yk, long long n, R *G, unsigned o) {
#pragma unroll
    for (int q = 0; q < KVG; ++q) {
      auto base = [&](int g) {
        const int v = g * KVG + q < NVS ? g * KVG + q : NVS - 1;
        return (unsigned long long)(v < 6 ? bv + v * n : yk + (v - 6) * n);
      };
      unsigned long long b = base(0);
#pragma unroll
      for (int g = 1; g < P::GRP; ++g) b = gid == g ? base(g) : b;
      G[q] = ldg<R>((gptr<const R>)b, o);
    }
  };
  const int gv = gid * KVG * PL + ec;
  auto put = [&](const R *G, int slot) {
#pragma unroll
    for (int q = 0; q < KVG; ++q) {
      // (GRP - 1) * KVG + q is the last group's variable of this place
      const int back = (P::GRP - 1) * KVG + q < NVS || gid < P::GRP - 1 ? 0 : ((P::GRP - 1) * KVG + q - (NVS - 1)) * PL;
      sm[slot + gv + q * PL - back] = G[q];
    }
  };
  // LDS writes of the workgroup are visible after it; loads stay in flight
  auto barrier = [] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // The fluxes of step k out of their slots (all wavefronts but the last, each
  // with its share of the variables and 64-cell groups): dq of plane k-1 gets
  // its upper z flux and is written; the in-plane differences of plane k and
  // its lower z flux are put together for the next step.
  auto take = [&](int k) {
    gptr<R> dq = DQ0;
    long long ni = B.ni;
    asm volatile("" : "+s"(dq), "+s"(ni));
    constexpr int GR = NFZ / 64, ITEMS = NV * GR, IT = (ITEMS + NT / 64 - 2) / (NT / 64 - 1);
    const int w0 = __builtin_amdgcn_readfirstlane(tid >> 6) * IT;
    R f[IT][6];
#pragma unroll
    for (int q = 0; q < IT; ++q) {
      const int i = min(w0 + q, ITEMS - 1), v = i / GR, c = i % GR * 64 + (tid & 63);
      const R *fz = sm + P::FB + v * NF + c, *fx = fz + NFZ + c / TX, *fy = fz + NFZ + NFX;
      f[q][0] = *fz, f[q][1] = fx[1], f[q][2] = fx[0], f[q][3] = fy[TX], f[q][4] = fy[0];
      f[q][5] = sm[P::ACC + v * NFZ + c];
    }
#pragma unroll
    for (int q = 0; q < IT; ++q) {
      const int i = w0 + q, v = i / GR, c = i % GR * 64 + (tid & 63), ci = c % TX, cj = c / TX;
      if (i >= ITEMS) continue;  // uniform per wavefront
      if (k > k0 && x0 + ci < mx && y0 + cj < my)
        *atg<R>(dq + v * ni, (unsigned)(((k - 1) * my + y0 + cj) * mx + x0 + ci) * (unsigned)sizeof(R)) = f[q][5] - f[q][0];
      sm[P::ACC + v * NFZ + c] = f[q][0] - (f[q][1] - f[q][2]) - (f[q][3] - f[q][4]);
    }
  };

  // ---- this thread's face: the left point is (x0 + fi, y0 + fj) of plane k
  // (x, y faces) or k-1 (z faces)
  const bool isz = tid < NFZ, isx = !isz && tid < NFZ + NFX, isy = !isz && !isx;
  int fi = 0, fj = 0;
  if (isz) {
    fi = tid % TX, fj = tid / TX;
  } else if (isx) {
    fi = (tid - NFZ) % (TX + 1) - 1, fj = (tid - NFZ) / (TX + 1);
  } else if (tid < NF) {
    fi = (tid - NFZ - NFX) % TX, fj = (tid - NFZ - NFX) / TX - 1;
  }
  const int gx = x0 + fi, gy = y0 + fj;
  const bool ok = gx + (isx ? 1 : 0) <= mx - (isx ? 0 : 1) && gy + (isy ? 1 : 0) <= my - (isy ? 0 : 1);
  const int el0 = (fj + 2) * W0 + fi + 2;
  const int da = isz ? 0 : (isx ? 1 : W0);
  const int db = isx ? W0 : 1;
  // byte offsets of the face's points in the field arrays; threads whose face
  // lies off the block work on the block's first point (in bounds, not used)
  unsigned pl_b = ((unsigned)((ok ? gy : 0) + kNgg) * (unsigned)B.sy + (unsigned)((ok ? gx : 0) + kNgg)) *
                      (unsigned)sizeof(R) + (unsigned)(k0 - (isz ? 1 : 0) + kNgg) * szb;
  const unsigned dr = isz ? szb : (isx ? (unsigned)sizeof(R) : syb);
  const bool q5 = (S.quirks & CFX_Q_METRIC_AVG) != 0 && !isy;
  const unsigned dr5 = q5 ? 0u : dr;                // right point of a metric the quirk does not average
  const unsigned drb0 = q5 && isx ? 0u : dr;        // ... of xi_x on its tangential row
  const unsigned drD = (NS > 0 && isz && (S.quirks & CFX_Q_HV_RHOD_J)) ? syb : dr;
  // rows of the metric along a, b, c
  using Row = std::conditional_t<BIG, unsigned long long, unsigned>;
  const Row row = (Row)(3 * B.np) * (Row)sizeof(R);
  const Row ra = isx ? 0 : (isz ? 2 * row : row);
  const Row rb = isx ? row : 0;
  const Row rc = isz ? row : 2 * row;
  auto ldm = [](gptr<const R> base, Row o) { return *(gptr<const R>)((gptr<const char>)base + o); };
  const bool viscous = S.viscous == 2;

  // ---- planes k0-1, k0, k0+1 into slots 0, 1, 2; k0-2 into the column buffer
  {
    R G0[KVG], G1[KVG], G2[KVG];
    if (stager) {
      fetch(BV0, YK0, B.np, G0, so);
      fetch(BV0, YK0, B.np, G1, so + szb);
      fetch(BV0, YK0, B.np, G2, so + 2 * szb);
    }
    if (isz) {
      R c[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) c[v] = ldg<R>(v < 5 ? BV0 + v * B.np : YK0 + (v - 5) * B.np, pl_b - szb);
#pragma unroll
      for (int v = 0; v < NV; ++v) sm[P::COL + v * NFZ + tid] = c[v];
    }
    if (stager) {
      put(G0, 0);
      put(G1, SLOT);
      put(G2, 2 * SLOT);
    }
  }
  barrier();

  // Each step has two barriers: the planes have been read and the fluxes are
  // in their slots; the next plane is in place and the slots are free.
  int s0 = 0, s1 = SLOT, s2 = 2 * SLOT;  // slots of the planes k-1, k, k+1
  if (__builtin_amdgcn_readfirstlane(tid >> 6) == NT / 64 - 1) {
    // ---- the last wavefront moves the data
    const int lane = tid & 63;
    constexpr int NC = (PL + 63) / 64;  // loads of one variable
    unsigned go[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int q = min(c * 64 + lane, PL - 1);
      go[c] = ((unsigned)(min(y0 - 2 + q / W0, my + 1) + kNgg) * (unsigned)B.sy +
               (unsigned)(min(x0 - 2 + q % W0, mx + 1) + kNgg)) * (unsigned)sizeof(R) +
              (unsigned)(k0 + 2 + kNgg) * szb;
    }
    for (int k = k0; k <= k1; ++k) {
      const bool more = k < k1;
      R G[NVS][NC];
      if (more) {  // plane k+2
        gptr<const R> bv = BV0, yk = YK0;
        long long n = B.np;
        asm volatile("" : "+s"(bv), "+s"(yk), "+s"(n));
#pragma unroll
        for (int v = 0; v < NVS; ++v)
#pragma unroll
          for (int c = 0; c < NC; ++c) G[v][c] = ldg<R>(v < 6 ? bv + v * n : yk + (v - 6) * n, go[c]);
#pragma unroll
        for (int c = 0; c < NC; ++c) go[c] += szb;
      }
      barrier();  // the planes are read, the fluxes are in their slots
      if (more) {
#pragma unroll
        for (int v = 0; v < NVS; ++v)
#pragma unroll
          for (int c = 0; c + 1 < NC; ++c) sm[s0 + v * PL + c * 64 + lane] = G[v][c];
        if ((NC - 1) * 64 + lane < PL) {
#pragma unroll
          for (int v = 0; v < NVS; ++v) sm[s0 + v * PL + (NC - 1) * 64 + lane] = G[v][NC - 1];
        }
      }
      const int t = s0;
      s0 = s1, s1 = s2, s2 = t;
      barrier();  // plane k+2 is in place, the slots are free
    }
    return;
  }
  for (int k = k0; k <= k1; ++k) {
    // fresh copies of the uniform bases: their per-variable sums are formed
    // where they are used instead of staying in scalar registers over the loop
    gptr<const R> PR_ = PR0, MT_ = MT0, JC_ = JC0;
    long long np = B.np;
    asm volatile("" : "+s"(PR_), "+s"(MT_), "+s"(JC_), "+s"(np));
    const bool more = k < k1;
    const bool active = isz || (more && tid < NF);
    R k1_ = 0, k2_ = 0, k3_ = 0, mA[3] = {0, 0, 0};
    const unsigned pr_b = pl_b + dr;
    R fj_[2], fm[3][2];
    if (active) {
      fj_[0] = ldg<R>(JC_, pl_b), fj_[1] = ldg<R>(JC_, pr_b);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        fm[c][0] = ldm(MT_ + c * np, pl_b + ra);
        fm[c][1] = ldm(MT_ + c * np, pr_b + ra);
      }
    }
    if (active) {
      // a wavefront further ahead in its step yields to one behind it on the
      // same SIMD, so that both reach the barrier together
      __builtin_amdgcn_s_setprio(3);
      // opaque copies, so that no address is kept in registers over the loop
      int el = el0, fb = P::FB + tid;
      asm volatile("" : "+v"(el), "+v"(fb));
      const int iL = (isz ? s0 : s1) + el, iR = s1 + el + da;
      const int i3 = isz ? s2 + el : iR + da;
      const int i0 = isz ? P::COL + tid : iL - da;
      // the face-point data of the viscous flux; issued ahead of AUSM+ where
      // the registers hold it (256 of them at 2 waves per SIMD; at 128 it spills)
      constexpr bool EARLY = WPE <= 2;
      R rB[3][2], rC[3][2], rV[4];
      auto face_point = [&] {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          rB[c][0] = ldm(MT_ + c * np, pl_b + rb), rB[c][1] = ldm(MT_ + c * np, pl_b + (c == 0 ? drb0 : dr5) + rb);
          rC[c][0] = ldm(MT_ + c * np, pl_b + rc), rC[c][1] = ldm(MT_ + c * np, pl_b + dr5 + rc);
        }
        rV[0] = ldg<R>(PR_ + 2 * np, pl_b), rV[1] = ldg<R>(PR_ + 2 * np, pr_b);
        rV[2] = ldg<R>(PR_ + 3 * np, pl_b), rV[3] = ldg<R>(PR_ + 3 * np, pr_b);
      };
      // ---- inviscid: MUSCL and AUSM+, flux into this thread's slot
      {
        R pl[NV], pr[NV];
        // variables two by two, the next pair's LDS reads issued before the
        // current pair is limited (all at once would not fit the registers);
        // a z thread's left value goes to its column buffer
        auto states = [&](auto mode) {
          constexpr int NP2 = (NV + 1) / 2;
          R st[2][2][4];
          int ci0 = i0;
          const int d0 = isz ? NFZ : PL;
          auto read2 = [&](int n) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              const int v = 2 * n + q;
              if (v >= NV) continue;
              const int o = (v < 5 ? v : v + 1) * PL;
              R *t = st[n & 1][q];
              t[0] = sm[ci0], t[1] = sm[iL + o], t[2] = sm[iR + o], t[3] = sm[i3 + o];
              ci0 += d0;
              if (v == 4 && !isz) ci0 += PL;  // T sits between p and Y
            }
          };
          read2(0);
#pragma unroll
          for (int n = 0; n < NP2; ++n) {
            if (n + 1 < NP2) read2(n + 1);
            __builtin_amdgcn_sched_barrier(0);
            constexpr int M = decltype(mode)::value;
            const R(*t)[4] = st[n & 1];
            if (2 * n + 1 < NV) {
              muscl_n<M, 2, R>(t, pl + 2 * n, pr + 2 * n);
              asm volatile("" : "+v"(pl[2 * n]), "+v"(pr[2 * n]), "+v"(pl[2 * n + 1]), "+v"(pr[2 * n + 1]));
            } else {
              muscl_n<M, 1, R>(t, pl + 2 * n, pr + 2 * n);
              asm volatile("" : "+v"(pl[2 * n]), "+v"(pr[2 * n]));
            }
            if (isz) {  // uniform per wavefront
              sm[i0 + 2 * n * NFZ] = t[0][1];
              if (2 * n + 1 < NV) sm[i0 + (2 * n + 1) * NFZ] = t[1][1];
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        };
        if (S.reconstruction != 2) states(std::integral_constant<int, 2>{});
        else if (S.limiter == 1) states(std::integral_constant<int, 1>{});
        else states(std::integral_constant<int, 0>{});
        const R jl = fj_[0], jr = fj_[1];
        k1_ = R(0.5) * (jl * fm[0][0] + jr * fm[0][1]);
        k2_ = R(0.5) * (jl * fm[1][0] + jr * fm[1][1]);
        k3_ = R(0.5) * (jl * fm[2][0] + jr * fm[2][1]);
        mA[0] = R(0.5) * (fm[0][0] + (q5 && isz ? fm[0][0] : fm[0][1]));
        mA[1] = R(0.5) * (fm[1][0] + (q5 ? fm[1][0] : fm[1][1]));
        mA[2] = R(0.5) * (fm[2][0] + (q5 ? fm[2][0] : fm[2][1]));
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" : "+v"(k1_), "+v"(k2_), "+v"(k3_), "+v"(mA[0]), "+v"(mA[1]), "+v"(mA[2]));
        if constexpr (EARLY)
          if (viscous) face_point();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(2);
        R F[NV];
        ausm_from_states<NS, R>(sp, th, S, pl, pr, k1_, k2_, k3_, F);
#pragma unroll
        for (int v = 0; v < NV; ++v) sm[fb + v * NF] = F[v];
      }
      // ---- viscous: subtracted from the slot as it is formed
      __builtin_amdgcn_s_setprio(1);
      if (viscous) {
        if constexpr (!EARLY) face_point();
        __builtin_amdgcn_sched_barrier(0);
        const int iLbm = iL - db, iLbp = iL + db, iRbm = iR - db, iRbp = iR + db;
        const int iLcm = isz ? iL - W0 : s0 + el, iLcp = isz ? iL + W0 : s2 + el;
        const int iRcm = isz ? iR - W0 : s0 + el + da, iRcp = isz ? iR + W0 : s2 + el + da;
        // the ten LDS reads of a variable go out one variable ahead
        R st[2][10];
        auto read10 = [&](auto nc) {
          constexpr int n = decltype(nc)::value;
          if constexpr (n < 4 + NS) {
            constexpr int o = (n < 3 ? n + 1 : n + 2) * PL;
            R *t = st[n & 1];
            t[0] = sm[iL + o], t[1] = sm[iR + o];
            t[2] = sm[iLbp + o], t[3] = sm[iLbm + o], t[4] = sm[iRbp + o], t[5] = sm[iRbm + o];
            t[6] = sm[iLcp + o], t[7] = sm[iLcm + o], t[8] = sm[iRcp + o], t[9] = sm[iRcm + o];
          }
        };
        auto steps = [&](auto nc, R g[3], R &av) {
          constexpr int n = decltype(nc)::value;
          read10(std::integral_constant<int, n + 1>{});
          __builtin_amdgcn_sched_barrier(0);
          const R *t = st[n & 1];
          // four times the tangential differences, twice the average: the
          // factors are in mB, mC, kb, kc and where the average is used
          g[0] = t[1] - t[0];
          g[1] = (t[2] - t[3]) + (t[4] - t[5]);
          g[2] = (t[6] - t[7]) + (t[8] - t[9]);
          av = t[0] + t[1];
        };
        // gradient (u, v, w) and face average of variable n
        R mB[3], mC[3];
        auto grad = [&](auto nc, R d[3], R &av) {
          R g[3];
          steps(nc, g, av);
#pragma unroll
          for (int c = 0; c < 3; ++c) d[c] = g[0] * mA[c] + g[1] * mB[c] + g[2] * mC[c];
          asm volatile("" : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(av));
        };
        // the gradient along the face-area vector (T, Y_l: nothing else of it
        // enters their fluxes), with k.(row a, b, c of the metric) formed once
        R ka, kb, kc;
        auto along = [&](auto nc, R &proj, R &av) {
          R g[3];
          steps(nc, g, av);
          proj = g[0] * ka + g[1] * kb + g[2] * kc;
          asm volatile("" : "+v"(proj), "+v"(av));
        };
        R du[3], dv[3], dw[3], dT, ua, va, wa, Ta;
        read10(std::integral_constant<int, 0>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          mB[c] = R(0.125) * (rB[c][0] + rB[c][1]);
          mC[c] = R(0.125) * (rC[c][0] + rC[c][1]);
        }
        R vis = R(0.5) * (rV[0] + rV[1]), cond = R(0.5) * (rV[2] + rV[3]);
        asm volatile("" : "+v"(mB[0]), "+v"(mB[1]), "+v"(mB[2]), "+v"(mC[0]), "+v"(mC[1]), "+v"(mC[2]), "+v"(vis), "+v"(cond));
        grad(std::integral_constant<int, 0>{}, du, ua);
        grad(std::integral_constant<int, 1>{}, dv, va);
        __builtin_amdgcn_sched_barrier(0);
        const unsigned pD_b = pl_b + drD;
        R rD[NS > 0 ? NS : 1][2];
#pragma unroll
        for (int s = 0; s < NS; ++s)
          rD[s][0] = ldg<R>(PR_ + (4 + s) * np, pl_b), rD[s][1] = ldg<R>(PR_ + (4 + s) * np, pD_b);
        __builtin_amdgcn_sched_barrier(0);
        grad(std::integral_constant<int, 2>{}, dw, wa);
        ka = k1_ * mA[0] + k2_ * mA[1] + k3_ * mA[2];
        kb = k1_ * mB[0] + k2_ * mB[1] + k3_ * mB[2];
        kc = k1_ * mC[0] + k2_ * mC[1] + k3_ * mC[2];
        along(std::integral_constant<int, 3>{}, dT, Ta);
        const R third = R(1.0 / 3.0);
        const R txx = vis * (R(4) * du[0] - R(2) * dv[1] - R(2) * dw[2]) * third;
        const R tyy = vis * (R(4) * dv[1] - R(2) * du[0] - R(2) * dw[2]) * third;
        const R tzz = vis * (R(4) * dw[2] - R(2) * du[0] - R(2) * dv[1]) * third;
        const R txy = vis * (du[1] + dv[0]);
        const R txz = vis * (du[2] + dw[0]);
        const R tyz = vis * (dv[2] + dw[1]);
        Ta *= R(0.5);
        const R G1 = k1_ * txx + k2_ * txy + k3_ * txz;
        const R G2 = k1_ * txy + k2_ * tyy + k3_ * tyz;
        const R G3 = k1_ * txz + k2_ * tyz + k3_ * tzz;
        R G4 = R(0.5) * (ua * G1 + va * G2 + wa * G3) + cond * dT;
        sm[fb + 1 * NF] -= G1;
        sm[fb + 2 * NF] -= G2;
        sm[fb + 3 * NF] -= G3;
        if constexpr (NS > 0) {
          __builtin_amdgcn_s_setprio(0);
          // uc = sum_l rho D_l (k . grad Y_l): the correction velocity along k
          R dp[NS], yb[NS], uc = 0;
          ka *= R(0.5), kb *= R(0.5), kc *= R(0.5);  // the average of rho*D
          static_for<NS>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            R proj;
            along(std::integral_constant<int, 4 + s>{}, proj, yb[s]);
            dp[s] = (rD[s][0] + rD[s][1]) * proj;
            uc += dp[s];
            asm volatile("" : "+v"(dp[s]), "+v"(uc));
            __builtin_amdgcn_sched_barrier(0);
          });
          G4 += carried_enthalpy<NS, R>(th, Ta, dp);
#pragma unroll
          for (int s = 0; s < NS; ++s) sm[fb + (5 + s) * NF] -= dp[s] - yb[s] * (R(0.5) * uc);
        }
        sm[fb + 4 * NF] -= G4;
      }
    }
    __builtin_amdgcn_s_setprio(0);
    barrier();  // the planes are read, the fluxes are in their slots
    take(k);
    const int t = s0;
    s0 = s1, s1 = s2, s2 = t;
    pl_b += szb;
    barrier();  // plane k+2 is in place, the slots are free
  }
}

}  // namespace cfx
