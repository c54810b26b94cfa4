// cfx_api.cpp — the C ABI of include/cfx.h: context, device memory, the
// reference's Driver step loop (Driver.cu:113-192) over the HIP kernels.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <limits>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/cfx.h"
#include "context.h"
#include "kernels.h"
#include "mesh.h"

using namespace cfx;

namespace {

constexpr double kRuH = 8314.462618;

// Host NASA-7 evaluation, identical to species_h_cp (device_physics.h).
void host_h_cp(const SpeciesT<double> &s, int l, double t, double &h, double &cp) {
  const int r = t >= s.t_mid[l] ? 1 : 0;
  const double *c = s.cpc[r][l], *e = s.hc[r][l];
  const double cpp = c[0] + t * (c[1] + t * (c[2] + t * (c[3] + t * c[4])));
  const double hp = t * (e[0] + t * (e[1] + t * (e[2] + t * (e[3] + t * e[4])))) + e[5];
  if (t < s.t_low[l]) {
    cp = s.cp_tlow[l];
    h = s.h_tlow[l] + s.cp_tlow[l] * (t - s.t_low[l]);
  } else {
    cp = cpp;
    h = hp;
  }
}

template <typename A, typename B>
void round_table(const A &a, B &b) {
  b.ns = a.ns;
  using T = std::remove_reference_t<decltype(b.mw[0])>;
  auto cp1 = [](const auto &src, auto &dst) {
    const double *x = reinterpret_cast<const double *>(&src);
    T *y = reinterpret_cast<T *>(&dst);
    for (size_t i = 0; i < sizeof(src) / sizeof(double); ++i) y[i] = (T)x[i];
  };
  cp1(a.mw, b.mw); cp1(a.inv_mw, b.inv_mw); cp1(a.r_sp, b.r_sp); cp1(a.t_low, b.t_low); cp1(a.t_mid, b.t_mid);
  cp1(a.cpc, b.cpc); cp1(a.hc, b.hc); cp1(a.h_tlow, b.h_tlow); cp1(a.cp_tlow, b.cp_tlow); cp1(a.lj_inv, b.lj_inv);
  cp1(a.om145, b.om145); cp1(a.vis_coeff, b.vis_coeff); cp1(a.cond_add, b.cond_add); cp1(a.wj4, b.wj4);
  cp1(a.sqw8, b.sqw8);
}

// the per-species thermo records from the arrays (same values, regrouped)
template <typename T>
void fill_thermo(SpeciesT<T> &s) {
  for (int l = 0; l < s.ns; ++l) {
    T *v = s.th[l].v;
    for (int g = 0; g < 2; ++g) {
      for (int k = 0; k < 5; ++k) v[kThCp + 5 * g + k] = s.cpc[g][l][k];
      for (int k = 0; k < 6; ++k) v[kThH + 6 * g + k] = s.hc[g][l][k];
    }
    for (int g = 0; g < 2; ++g)
      for (int k = 0; k < 6; ++k) s.mix[g][l].v[k] = s.hc[g][l][k];
    s.mix[2][l].v[0] = s.cp_tlow[l];
    s.mix[2][l].v[5] = (T)((double)s.h_tlow[l] - (double)s.cp_tlow[l] * (double)s.t_low[l]);
    v[kThTmid] = s.t_mid[l];
    v[kThTlow] = s.t_low[l];
    v[kThHtlow] = s.h_tlow[l];
    v[kThCptlow] = s.cp_tlow[l];
  }
  T tmid_min = std::numeric_limits<T>::max(), tmid_max = std::numeric_limits<T>::lowest();
  T tlow_max = std::numeric_limits<T>::lowest();
  for (int l = 0; l < s.ns; ++l) {
    tmid_min = std::min(tmid_min, s.t_mid[l]);
    tmid_max = std::max(tmid_max, s.t_mid[l]);
    tlow_max = std::max(tlow_max, s.t_low[l]);
  }
  s.hi_from = std::max(tmid_max, tlow_max);
  s.lo_from = tlow_max;
  s.lo_to = tmid_min;
}

int build_species(const cfx_species *sp, SpeciesDev &tables, std::string &err) {
  std::memset(&tables, 0, sizeof(tables));
  SpeciesT<double> &s = tables.d;
  s.ns = sp ? sp->n_spec : 0;
  if (s.ns < 0 || s.ns > kMaxSp) {
    err = "n_spec out of range";
    return CFX_E_ARG;
  }
  for (int l = 0; l < s.ns; ++l) {
    const double W = sp->mw[l];
    if (!(W > 0) || !(sp->eps_k[l] > 0) || !(sp->sigma[l] > 0)) {
      err = "species " + std::to_string(l) + ": non-positive mw / eps_k / sigma";
      return CFX_E_ARG;
    }
    const double rs = kRuH / W;
    s.mw[l] = W;
    s.inv_mw[l] = 1.0 / W;
    s.r_sp[l] = rs;
    s.t_low[l] = sp->t_low[l];
    s.t_mid[l] = sp->t_mid[l];
    for (int r = 0; r < 2; ++r) {
      const double *a = (r == 0 ? sp->coeff_lo : sp->coeff_hi) + 7 * l;
      for (int k = 0; k < 5; ++k) {
        s.cpc[r][l][k] = a[k] * rs;
        s.hc[r][l][k] = a[k] / (k + 1) * rs;
      }
      s.hc[r][l][5] = a[5] * rs;
    }
    // enthalpy and cp at t_low with the low set (Thermo.cu:30-37)
    const double tt = sp->t_low[l];
    const double *c = s.cpc[0][l], *e = s.hc[0][l];
    s.cp_tlow[l] = c[0] + tt * (c[1] + tt * (c[2] + tt * (c[3] + tt * c[4])));
    s.h_tlow[l] = tt * (e[0] + tt * (e[1] + tt * (e[2] + tt * (e[3] + tt * e[4])))) + e[5];
    s.lj_inv[l] = 1.0 / sp->eps_k[l];
    s.om145[l] = std::pow(s.lj_inv[l], -0.145);
    s.vis_coeff[l] = 2.6693e-6 * std::sqrt(W) / (sp->sigma[l] * sp->sigma[l]);  // ChemData.cpp:249-250
    s.cond_add[l] = 1.25 * rs;
  }
  for (int m = 0; m < s.ns; ++m)
    for (int n = 0; n < s.ns; ++n) {
      s.wj4[m][n] = std::pow(s.mw[n] / s.mw[m], 0.25);
      s.sqw8[m][n] = 1.0 / std::sqrt(8 * (1 + s.mw[m] / s.mw[n]));
    }
  round_table(tables.d, tables.f);
  fill_thermo(tables.d);
  fill_thermo(tables.f);
  return 0;
}

// Inflow::Inflow state (BoundCond.cu:13-105): (mach|velocity, p, T|rho).
int build_inflow(const cfx_inflow &in, const SpeciesT<double> &s, const SchemeDev &S, InflowDev &out,
                 std::string &err) {
  std::memset(&out, 0, sizeof(out));
  const int ns = s.ns;
  double mw = kRuH / S.r_air;
  if (ns > 0) {
    if (!in.yk) {
      err = "inflow without mass fractions on a multispecies case";
      return CFX_E_ARG;
    }
    double w = 0;
    for (int l = 0; l < ns; ++l) {
      out.y[l] = in.yk[l];
      w += in.yk[l] / s.mw[l];
    }
    mw = 1 / w;
  }
  double T = in.temperature, mach = in.mach, vel = in.velocity, rho = in.density;
  const double p = in.pressure;
  if (T < 0) T = p * mw / (rho * kRuH);
  double gamma = S.gamma_air;
  if (ns > 0) {
    double cp = 0, cv = 0;
    for (int l = 0; l < ns; ++l) {
      double h, c;
      host_h_cp(s, l, T, h, c);
      cp += out.y[l] * c;
      cv += out.y[l] * (c - s.r_sp[l]);
    }
    gamma = cp / cv;
  }
  const double c = std::sqrt(gamma * kRuH / mw * T);
  if (mach < 0) mach = vel / c;
  else vel = mach * c;
  if (rho < 0) rho = p * mw / (kRuH * T);
  out.st[0] = rho;
  out.st[1] = in.u * vel;
  out.st[2] = in.v * vel;
  out.st[3] = in.w * vel;
  out.st[4] = p;
  out.st[5] = T;
  // total energy (Thermo.cu:66-86)
  double e = 0.5 * rho * (out.st[1] * out.st[1] + out.st[2] * out.st[2] + out.st[3] * out.st[3]);
  if (ns > 0) {
    for (int l = 0; l < ns; ++l) {
      double h, cp;
      host_h_cp(s, l, T, h, cp);
      e += h * (rho * out.y[l]);
    }
    e -= p;
  } else {
    e += p / (S.gamma_air - 1);
  }
  out.st[6] = e;
  return 0;
}


// ---------------------------------------------------------------- tables ---
int upload_table(cfx_ctx *ctx, Table &t, const std::vector<int> &counts) {
  t.host.assign(counts.size() + 1, 0);
  for (size_t b = 0; b < counts.size(); ++b) t.host[b + 1] = t.host[b] + counts[b];
  int rc = 0;
  t.dev = ctx->dalloc<int>(t.host.size(), rc);
  if (rc) return rc;
  return (int)hipMemcpy(t.dev, t.host.data(), sizeof(int) * t.host.size(), hipMemcpyHostToDevice);
}

int chunks(long long n, int per) { return (int)((n + per - 1) / per); }

int build_tables(cfx_ctx *ctx) {
  const int nb = (int)ctx->hb.size();
  std::vector<int> pad(nb), in1(nb), dtc(nb), last(nb), res(nb);
  for (int b = 0; b < nb; ++b) {
    const HostBlock &H = ctx->hb[b];
    pad[b] = chunks(H.np, kTpb);
    in1[b] = chunks(H.ni, kTpb);
    res[b] = chunks(H.ni, kTpb * kResIter);
  }
  int rc;
  // small contexts spread the points over the chip instead (128x64 points: time
  // step 10.5 -> 4.4 us, snapshot 7.1 -> 4.6); the time step ends in an atomic
  // per workgroup, and takes few of them (1021x509 points: 2031 workgroups 29 us,
  // 508 16 us)
  long long all = 0;
  for (const HostBlock &H : ctx->hb) all += H.ni;
  ctx->dt_iter = (int)std::min<long long>(kDtIter, 1 + all / (kTpb * 512));
  ctx->last_iter = (int)std::min<long long>(kLastIter, 1 + all / (kTpb * 2048));
  for (int b = 0; b < nb; ++b) {
    dtc[b] = chunks(ctx->hb[b].ni, kTpb * ctx->dt_iter);
    last[b] = chunks(ctx->hb[b].ni, kTpb * ctx->last_iter);
  }
  if ((rc = upload_table(ctx, ctx->t_pad, pad)) || (rc = upload_table(ctx, ctx->t_int, in1)) ||
      (rc = upload_table(ctx, ctx->t_dt, dtc)) || (rc = upload_table(ctx, ctx->t_last, last)) ||
      (rc = upload_table(ctx, ctx->t_res, res)))
    return rc;
  if (ctx->dim != 2) return 0;
  std::vector<int> count(nb);
  for (int b = 0; b < nb; ++b) count[b] = chunks((long long)(ctx->hb[b].mx + 2 * kNgg) * (ctx->hb[b].my + 2 * kNgg), kTpb);
  if ((rc = upload_table(ctx, ctx->t_plane, count))) return rc;
  for (int v = 0; v < kNVar2; ++v) {
    for (int b = 0; b < nb; ++b) {
      const int m[3] = {ctx->hb[b].mx, ctx->hb[b].my, ctx->hb[b].mz};
      count[b] = plane_groups(m, kTiles2[v]);
    }
    if ((rc = upload_table(ctx, ctx->t_rhs[v], count))) return rc;
  }
  return 0;
}

// The order in which the sweeps of LU-SGS take the patches: by J + K, so that
// the two patches a patch waits for stand before it.
int plan_sweeps(cfx_ctx *ctx) {
  if (!ctx->lusgs) return 0;
  std::vector<LuPatch> all;
  std::vector<int> my, mz;
  for (const HostBlock &H : ctx->hb) my.push_back(H.my), mz.push_back(H.mz);
  lu_plan(my, mz, all, ctx->lu_off);
  int rc = 0;
  ctx->lu_order = ctx->dalloc<LuPatch>(all.size(), rc);
  ctx->lu_ticket = ctx->dalloc<int>(2, rc);
  if (rc) return rc;
  return (int)hipMemcpy(ctx->lu_order, all.data(), sizeof(LuPatch) * all.size(), hipMemcpyHostToDevice);
}

// The marching RHS of a 3-D context: the planes per workgroup of every variant
// and its workgroup prefix.
int plan_march(cfx_ctx *ctx) {
  if (ctx->dim != 3) return 0;
  const MarchTile t = ctx->mixed ? kMarch32 : kMarch64;
  const OccFn occ = ctx->mixed ? g_kernels32[ctx->ns].march_occ : g_kernels64[ctx->ns].march_occ;
  const double word = ctx->mixed ? 4 : 8;
  const size_t nb = ctx->hb.size();
  std::vector<int> groups(nb);
  int top = 0;
  for (const HostBlock &H : ctx->hb) {
    ctx->march_big = ctx->march_big || 9.0 * word * (double)H.np >= 4294967296.0;
    top = std::max(top, H.mz);
  }
  auto split = [&](int chunk) {
    for (size_t b = 0; b < nb; ++b) {
      const int m[3] = {ctx->hb[b].mx, ctx->hb[b].my, ctx->hb[b].mz};
      groups[b] = march_groups(m, t, chunk);
    }
  };
  // Variant 0: a chunk of n planes costs about n + kFill planes' time (the
  // first planes' loads, the last z faces; 256x128x128 with 9 species in
  // chunks of 8 and of 128 or 64 planes: 1.2 in FP64, 1.4 in FP32).  The
  // workgroups go to the 8 XCDs in contiguous runs of equal count; a launch
  // lasts as long as its fullest XCD: whole rounds of one block, an average
  // load and half of the longest chunk of many (27 blocks of 33..90 points:
  // planned without the runs 6.98 ms per step in FP64, with them 6.24).
  constexpr double kFill = 1.3;
  const double slots = std::max(1.0, (double)std::max(1, occ()) * ctx->n_cu / 8);
  double best = 1e300;
  int planned = top;
  for (int parts = 1; parts <= top; ++parts) {
    const int chunk = chunks(top, parts);
    if (parts > 1 && chunk == chunks(top, parts - 1)) continue;
    split(chunk);
    long long total = 0;
    for (size_t b = 0; b < nb; ++b) total += groups[b];
    const long long run = (total + 7) / 8;
    double est = 0;
    size_t b = 0;
    long long left = groups[0];
    for (int x = 0; x < 8; ++x) {
      double work = 0, longest = 0, n = 0;
      for (long long room = run; room > 0 && b < nb;) {
        const long long k = std::min(room, left);
        const double len = chunks(ctx->hb[b].mz, chunks(ctx->hb[b].mz, chunk)) + kFill;
        work += (double)k * len;
        n += (double)k;
        longest = std::max(longest, len);
        room -= k;
        left -= k;
        if (left == 0 && ++b < nb) left = groups[b];
      }
      est = std::max(est, nb == 1 ? std::ceil(n / slots) * longest : std::max(longest, work / slots + 0.5 * longest));
    }
    if (est < best) best = est, planned = chunk;
  }
  for (int v = 0; v < kNVar3; ++v) {
    ctx->march_chunk[v] = v == 0 ? planned : kMarchChunk[v];
    split(ctx->march_chunk[v]);
    if (int rc = upload_table(ctx, ctx->t_march[v], groups)) return rc;
  }
  return 0;
}

// ------------------------------------------------------- ghost-fill ops ---
// Boxes of points an op reads or writes, per block (unpadded indices, ghosts
// negative or beyond the extent).
struct Touch {
  int blk, lo[3], hi[3];
  bool write;
};

Touch box_of(int blk, const int a[3], const int b[3], bool write) {
  Touch t{blk, {0, 0, 0}, {0, 0, 0}, write};
  for (int q = 0; q < 3; ++q) {
    t.lo[q] = std::min(a[q], b[q]);
    t.hi[q] = std::max(a[q], b[q]);
  }
  return t;
}

std::vector<Touch> touches(const FaceOp &op) {
  std::vector<Touch> out;
  if (op.kind == kOpExchange) {
    const InnerDev &f = op.f;
    out.push_back(box_of(op.blk, f.rs, f.re, true));
    int lo[3], hi[3], flo[3], fhi[3];
    const int face_layer = f.direction > 0 ? f.rs[f.face] : f.re[f.face];
    const int nface = (face_layer - f.rs[f.face]) * f.loop_dir[f.face];
    for (int q = 0; q < 3; ++q) {
      const int s = f.src_tar[q];
      const int step = f.target_loop_dir[q] * f.loop_dir[s];
      lo[q] = f.ts[q];
      hi[q] = f.ts[q] + step * (f.n_point[s] - 1);
      flo[q] = lo[q];
      fhi[q] = hi[q];
      if (s == f.face) flo[q] = fhi[q] = f.ts[q] + step * nface;
    }
    out.push_back(box_of(op.tgt, lo, hi, false));
    out.push_back(box_of(op.tgt, flo, fhi, true));
    return out;
  }
  const FaceRange &r = op.r;
  const int a = r.face, s = r.direction;
  int lo[3], hi[3];
  for (int q = 0; q < 3; ++q) lo[q] = r.rs[q], hi[q] = r.re[q];
  auto layer = [&](int from, int to, bool write) {
    int l2[3] = {lo[0], lo[1], lo[2]}, h2[3] = {hi[0], hi[1], hi[2]};
    l2[a] = r.rs[a] + s * from;
    h2[a] = r.rs[a] + s * to;
    out.push_back(box_of(op.blk, l2, h2, write));
  };
  switch (op.kind) {
    case CFX_BC_OUTFLOW: layer(0, 0, false); layer(1, kNgg, true); break;
    case CFX_BC_INFLOW: layer(1, kNgg, true); break;
    default: layer(-kNgg, -1, false); layer(0, 0, true); layer(1, kNgg, true); break;  // wall, symmetry
  }
  return out;
}

bool conflict(const std::vector<Touch> &x, const std::vector<Touch> &y) {
  for (const Touch &a : x)
    for (const Touch &b : y) {
      if (a.blk != b.blk || !(a.write || b.write)) continue;
      bool meet = true;
      for (int q = 0; q < 3; ++q) meet = meet && a.lo[q] <= b.hi[q] && b.lo[q] <= a.hi[q];
      if (meet) return true;
    }
  return false;
}

// Levels for ops[first..last): an op goes one level after the latest earlier
// op it conflicts with, so every conflicting pair keeps the application
// order and the result equals the one-op-at-a-time loop.  levelize=false
// gives each op its own level (that loop itself).
int build_schedule(cfx_ctx *ctx, const std::vector<FaceOp> &all, Schedule &sc, int first, int last, bool levelize,
                   const std::vector<int> *group = nullptr) {
  const int n = last - first;
  std::vector<int> level(n, 0);
  if (!levelize && group) {  // one level per group of pieces of one op (disjoint boxes)
    for (int i = 0; i < n; ++i) level[i] = (*group)[first + i] - (*group)[first];
  } else if (levelize) {
    std::vector<std::vector<Touch>> tc(n);
    for (int i = 0; i < n; ++i) tc[i] = touches(all[first + i]);
    for (int j = 0; j < n; ++j)
      for (int i = 0; i < j; ++i)
        if (level[i] + 1 > level[j] && conflict(tc[i], tc[j])) level[j] = level[i] + 1;
  } else {
    for (int i = 0; i < n; ++i) level[i] = i;
  }
  const int nlev = n ? *std::max_element(level.begin(), level.end()) + 1 : 0;
  std::vector<FaceOp> ordered;
  sc.lvl.assign(1, 0);
  sc.copies.clear();
  for (int L = 0; L < nlev; ++L) {
    for (int i = 0; i < n; ++i)
      if (level[i] == L) ordered.push_back(all[first + i]);
    bool copies = true;
    for (int i = sc.lvl.back(); i < (int)ordered.size(); ++i)
      copies = copies && (ordered[i].kind == CFX_BC_OUTFLOW || ordered[i].kind == kOpExchange);
    sc.copies.push_back(copies ? 1 : 0);
    sc.lvl.push_back((int)ordered.size());
  }
  sc.off_host.assign(ordered.size() + 1, 0);
  for (size_t i = 0; i < ordered.size(); ++i) sc.off_host[i + 1] = sc.off_host[i] + chunks(ordered[i].npts, kTpb);
  int rc = 0;
  sc.ops = ctx->dalloc<FaceOp>(ordered.size(), rc);
  sc.off = ctx->dalloc<int>(sc.off_host.size(), rc);
  if (rc) return rc;
  if (!ordered.empty())
    if ((rc = (int)hipMemcpy(sc.ops, ordered.data(), sizeof(FaceOp) * ordered.size(), hipMemcpyHostToDevice)))
      return rc;
  return (int)hipMemcpy(sc.off, sc.off_host.data(), sizeof(int) * sc.off_host.size(), hipMemcpyHostToDevice);
}

// An outflow op whose range is the whole face (the face's points and the
// ngg layers around them tangentially) copies the face layer into the ghost
// layers behind it.  Its interior rows (tangential indices inside the block)
// read only points the update kernel has just written; when no op before it
// in the application order touches those rows (box conflict as for the
// levels), applying them inside the update kernel, right after the point's
// own stores, gives the same values in the same order.  The op is then
// replaced in the step's list by its ring of edge rows.  Sets the blocks'
// fuse flags (uploaded with the views).
void fold_outflow(cfx_ctx *ctx) {
  ctx->ops_step.clear();
  ctx->ops_step_src.clear();
  ctx->n_fused = 0;
  for (auto &V : ctx->views) {
    for (int f = 0; f < 6; ++f) V.fuse[f] = 0;
    V.fuse_any = 0;
  }
  const int n = (int)ctx->ops.size();
  std::vector<std::vector<Touch>> before;
  for (int i = 0; i < n; ++i) {
    const FaceOp &op = ctx->ops[i];
    bool fold = false;
    FaceOp inner = op;
    if (op.kind == CFX_BC_OUTFLOW) {
      const HostBlock &H = ctx->hb[op.blk];
      const int m[3] = {H.mx, H.my, H.mz};
      const int a = op.r.face;
      fold = op.r.rs[a] == op.r.re[a] && op.r.rs[a] == (op.r.direction < 0 ? 0 : m[a] - 1);
      for (int t = 0; t < 3 && fold; ++t) {
        if (t == a) continue;
        fold = op.r.rs[t] == -kNgg && op.r.re[t] == m[t] - 1 + kNgg;
        inner.r.rs[t] = 0;
        inner.r.re[t] = m[t] - 1;
      }
      if (fold) {
        const std::vector<Touch> ti = touches(inner);
        for (const auto &tb : before) fold = fold && !conflict(tb, ti);
      }
      if (fold) {
        // the ring: rows with a tangential index outside the block
        const int t1 = a == 0 ? 1 : 0, t2 = a == 2 ? 1 : 2;
        auto add = [&](int lo1, int hi1, int lo2, int hi2) {
          if (lo1 > hi1 || lo2 > hi2) return;
          FaceOp r = op;
          r.r.rs[t1] = lo1, r.r.re[t1] = hi1, r.r.rs[t2] = lo2, r.r.re[t2] = hi2;
          for (int q = 0; q < 3; ++q) r.ext[q] = r.r.re[q] - r.r.rs[q] + 1;
          r.npts = (long long)r.ext[0] * r.ext[1] * r.ext[2];
          ctx->ops_step.push_back(r);
          ctx->ops_step_src.push_back(i);
        };
        add(-kNgg, -1, -kNgg, m[t2] - 1 + kNgg);
        add(m[t1], m[t1] - 1 + kNgg, -kNgg, m[t2] - 1 + kNgg);
        add(0, m[t1] - 1, -kNgg, -1);
        add(0, m[t1] - 1, m[t2], m[t2] - 1 + kNgg);
        BlockView &V = ctx->views[op.blk];
        V.fuse[2 * a + (op.r.direction < 0 ? 0 : 1)] = 1;
        V.fuse_any = 1;
        ++ctx->n_fused;
      }
    }
    if (!fold) {
      ctx->ops_step.push_back(op);
      ctx->ops_step_src.push_back(i);
    }
    before.push_back(touches(op));
  }
}

// ------------------------------------------------------- split exchange ---
// The exchange ops in two launches.  In the middle of a face (more than
// kStrip points from its edges, ghosts included) only the two ops of the face
// meet: the first averages the shared layer and fills the ghost layers of its
// block, the second would average two equal values and fills the other
// block's ghost layers from interior layers nobody writes.  So all middles
// run in one launch, the second op without the shared layer.  Near the edges
// the ops of several faces meet, always on copies of one grid point: there
// the point ops are grouped into components of linked points, and a thread
// runs a component's ops in their order.  Every point sees the same
// operations in the same order as in the one-op-at-a-time loop.
//
// The level schedule it replaces needs one launch per level of whole faces:
// 51 launches for the 64-block lattice, 18.5 us each at 27 points per axis.
// A step of 64 blocks of 12..44 points per axis, mixed: 6.1 -> 4.7 ms; of 27
// blocks of 20..90 points, FP64: 17.8 -> 15.5 ms (9 species).
constexpr int kStrip = 5;  // the ngg ghosts and the layers 0..ngg of the face across the edge

// the part of an exchange op whose loop index along axis q runs over [n0[q], n0[q] + n[q])
FaceOp sub_exchange(const FaceOp &op, const int n0[3], const int n[3]) {
  FaceOp s = op;
  int d[3];
  for (int q = 0; q < 3; ++q) d[q] = op.f.loop_dir[q] * n0[q];
  for (int q = 0; q < 3; ++q) {
    s.f.rs[q] = op.f.rs[q] + d[q];
    s.f.re[q] = s.f.rs[q] + op.f.loop_dir[q] * (n[q] - 1);
    s.f.ts[q] = op.f.ts[q] + op.f.target_loop_dir[q] * d[op.f.src_tar[q]];
    s.f.n_point[q] = s.ext[q] = n[q];
  }
  s.npts = (long long)n[0] * n[1] * n[2];
  return s;
}

// point n of an exchange op in its block and in the target
void exchange_map(const InnerDev &f, const int n[3], int p[3], int t[3]) {
  int d[3];
  for (int q = 0; q < 3; ++q) {
    d[q] = f.loop_dir[q] * n[q];
    p[q] = f.rs[q] + d[q];
  }
  for (int q = 0; q < 3; ++q) t[q] = f.ts[q] + f.target_loop_dir[q] * d[f.src_tar[q]];
}

// loop index of the shared layer along the face axis
int shared_layer(const InnerDev &f) {
  return ((f.direction > 0 ? f.rs[f.face] : f.re[f.face]) - f.rs[f.face]) * f.loop_dir[f.face];
}

// whether two exchange ops are the two sides of one face
bool mirrored(const FaceOp &a, const FaceOp &b) {
  if (a.blk == a.tgt || a.blk != b.tgt || a.tgt != b.blk) return false;
  const int fa = a.f.face, fb = b.f.face;
  if (a.f.src_tar[fb] != fa || b.f.src_tar[fa] != fb) return false;
  // the corners of a's shared layer map to b's shared layer and back
  for (int c = 0; c < 4; ++c) {
    int n[3], p[3], t[3], m[3], p2[3], t2[3];
    for (int q = 0, k = 0; q < 3; ++q) n[q] = q == fa ? shared_layer(a.f) : ((c >> k++) & 1 ? a.f.n_point[q] - 1 : 0);
    exchange_map(a.f, n, p, t);
    for (int q = 0; q < 3; ++q) {
      m[q] = (t[q] - b.f.rs[q]) * b.f.loop_dir[q];
      if (m[q] < 0 || m[q] >= b.f.n_point[q]) return false;
    }
    if (m[fb] != shared_layer(b.f)) return false;
    exchange_map(b.f, m, p2, t2);
    for (int q = 0; q < 3; ++q)
      if (t2[q] != p[q]) return false;
  }
  for (int q = 0; q < 3; ++q)
    if (q != fa) {
      int axis_b = 0;
      while (a.f.src_tar[axis_b] != q) ++axis_b;
      if (a.f.n_point[q] != b.f.n_point[axis_b]) return false;
    }
  return true;
}

// The split of ops[first..): middles (one level) and the rest of every op.
// False where the mesh does not allow it.
bool split_ops(const std::vector<FaceOp> &ops, int first, int dim, std::vector<FaceOp> &mid,
               std::vector<std::vector<FaceOp>> &rest) {
  const int n = (int)ops.size();
  std::vector<int> partner(n, -1);
  for (int j = first; j < n; ++j) {
    for (int i = first; i < j && partner[j] < 0; ++i)
      if (partner[i] < 0 && mirrored(ops[i], ops[j])) partner[i] = j, partner[j] = i;
  }
  for (int i = first; i < n; ++i) {
    if (partner[i] < 0) return false;
    const FaceOp &op = ops[i];
    // loop-index cuts per axis: {begin, end} of the middle
    int lo[3], hi[3];
    bool empty = false;
    for (int q = 0; q < 3; ++q) {
      const bool cut = q != op.f.face && !(dim == 2 && q == 2);
      lo[q] = cut ? kStrip : 0;
      hi[q] = op.f.n_point[q] - lo[q];
      empty = empty || hi[q] <= lo[q];
    }
    rest.emplace_back();
    if (empty) {
      rest.back().push_back(op);
      continue;
    }
    const int len[3] = {hi[0] - lo[0], hi[1] - lo[1], hi[2] - lo[2]};
    mid.push_back(sub_exchange(op, lo, len));
    mid.back().ghosts_only = partner[i] < i;
    // the frame around it, axis by axis
    int a[3] = {0, 0, 0}, b[3] = {op.f.n_point[0], op.f.n_point[1], op.f.n_point[2]};
    for (int q = 0; q < 3; ++q) {
      if (lo[q] == 0) continue;
      for (int side = 0; side < 2; ++side) {
        int n0[3] = {a[0], a[1], a[2]}, m[3] = {b[0] - a[0], b[1] - a[1], b[2] - a[2]};
        n0[q] = side ? hi[q] : 0;
        m[q] = kStrip;
        rest.back().push_back(sub_exchange(op, n0, m));
      }
      a[q] = lo[q];
      b[q] = hi[q];
    }
  }
  // a middle meets nothing but its partner (and that as described above)
  std::vector<std::vector<Touch>> tm, tr;
  for (const FaceOp &m : mid) tm.push_back(touches(m));
  for (const auto &r : rest)
    for (const FaceOp &p : r) tr.push_back(touches(p));
  std::vector<std::vector<std::pair<int, int>>> by_blk;  // (0 middle / 1 rest, index) per block
  auto add = [&](int kind, int idx, const std::vector<Touch> &t) {
    for (const Touch &x : t) {
      if ((int)by_blk.size() <= x.blk) by_blk.resize(x.blk + 1);
      if (by_blk[x.blk].empty() || by_blk[x.blk].back() != std::make_pair(kind, idx)) by_blk[x.blk].push_back({kind, idx});
    }
  };
  for (size_t i = 0; i < tm.size(); ++i) add(0, (int)i, tm[i]);
  for (size_t i = 0; i < tr.size(); ++i) add(1, (int)i, tr[i]);
  for (const auto &v : by_blk)
    for (const auto &x : v) {
      if (x.first != 0) continue;
      for (const auto &y : v) {
        if (y.first == 0 && (y.second >= x.second || mirrored(mid[y.second], mid[x.second]))) continue;
        if (conflict(tm[x.second], y.first ? tr[y.second] : tm[y.second])) return false;
      }
    }
  return true;
}

// The strips as components of linked points; false if one holds too many.
bool build_strips(const cfx_ctx *ctx, const std::vector<std::vector<FaceOp>> &rest, std::vector<ExSlot> &slots,
                  std::vector<ExOp> &ops, std::vector<int> &slot_off, std::vector<int> &op_off, int end[3]) {
  struct PointOp {
    int a, b;  // point ids: written (and averaged) / read
    bool average;
  };
  std::vector<PointOp> pops;
  std::vector<ExSlot> pts;
  std::vector<int> parent;
  // open-addressing table of (block, padded index) -> id
  size_t n_est = 0;
  for (const auto &r : rest)
    for (const FaceOp &p : r) n_est += 2 * (size_t)p.npts;
  size_t cap = 64;
  while (cap < 2 * n_est) cap *= 2;
  std::vector<int> table(cap, -1);
  pops.reserve(n_est / 2);
  pts.reserve(n_est);
  parent.reserve(n_est);
  auto id_of = [&](int blk, unsigned p) {
    // runs of 16 points share a cache line of the table
    const unsigned long long h = ((unsigned long long)blk << 32 | p >> 4) * 0x9E3779B97F4A7C15ull;
    for (size_t k = ((size_t)(h >> 24) << 4 | (p & 15)) & (cap - 1);; k = (k + 1) & (cap - 1)) {
      if (table[k] < 0) {
        table[k] = (int)pts.size();
        pts.push_back(ExSlot{blk, p});
        parent.push_back(table[k]);
        return table[k];
      }
      if (pts[table[k]].blk == blk && pts[table[k]].p == p) return table[k];
    }
  };
  auto root = [&](int x) {
    while (parent[x] != x) x = parent[x] = parent[parent[x]];
    return x;
  };
  for (const auto &r : rest) {
    // the pieces of one op are disjoint: their order does not matter
    for (const FaceOp &p : r) {
      const HostBlock &B = ctx->hb[p.blk], &T = ctx->hb[p.tgt];
      const int face_layer = p.f.direction > 0 ? p.f.rs[p.f.face] : p.f.re[p.f.face];
      int n[3], i[3], t[3];
      for (n[2] = 0; n[2] < p.ext[2]; ++n[2])
        for (n[1] = 0; n[1] < p.ext[1]; ++n[1])
          for (n[0] = 0; n[0] < p.ext[0]; ++n[0]) {
            exchange_map(p.f, n, i, t);
            const int a = id_of(p.blk, (unsigned)B.pidx(i[0], i[1], i[2]));
            const int b = id_of(p.tgt, (unsigned)T.pidx(t[0], t[1], t[2]));
            pops.push_back(PointOp{a, b, i[p.f.face] == face_layer});
            const int ra = root(a), rb = root(b);
            if (ra != rb) parent[std::max(ra, rb)] = std::min(ra, rb);
          }
    }
  }
  // components in order of their first point
  const int np = (int)pts.size();
  std::vector<int> comp(np, -1), local(np, 0);
  slot_off.assign(1, 0);
  std::vector<int> count;
  for (int x = 0; x < np; ++x) {
    const int r = root(x);
    if (comp[r] < 0) {
      comp[r] = (int)count.size();
      count.push_back(0);
    }
    comp[x] = comp[r];
    local[x] = count[comp[x]]++;
    if (local[x] >= kMaxSlots) return false;
  }
  // ... then by their slots, as many as fit each form of the kernel
  const int nc = (int)count.size();
  std::vector<int> rank(nc);
  for (int q = 0, r = 0; q < 3; ++q) {
    for (int c = 0; c < nc; ++c) {
      if (count[c] > kStripSlots[q] || (q > 0 && count[c] <= kStripSlots[q - 1])) continue;
      rank[c] = r++;
      slot_off.push_back(slot_off.back() + count[c]);
    }
    end[q] = r;
  }
  for (int x = 0; x < np; ++x) comp[x] = rank[comp[x]];
  slots.resize(np);
  for (int x = 0; x < np; ++x) slots[slot_off[comp[x]] + local[x]] = pts[x];
  op_off.assign(nc + 1, 0);
  for (const PointOp &o : pops) ++op_off[comp[o.a] + 1];
  for (int c = 0; c < nc; ++c) op_off[c + 1] += op_off[c];
  std::vector<int> at(op_off.begin(), op_off.end() - 1);
  ops.resize(pops.size());
  for (const PointOp &o : pops) {
    const int c = comp[o.a];
    ops[at[c]++] = ExOp{(unsigned char)local[o.a], (unsigned char)local[o.b], (unsigned char)(o.average ? 1 : 0), 0};
    slots[slot_off[c] + local[o.a]].p |= kSlotWritten;
    if (o.average) slots[slot_off[c] + local[o.b]].p |= kSlotWritten;
  }
  return true;
}

template <class T>
int upload(cfx_ctx *ctx, const std::vector<T> &v, const T *&dev) {
  int rc = 0;
  T *d = ctx->dalloc<T>(v.size(), rc);
  if (rc) return rc;
  dev = d;
  return v.empty() ? 0 : (int)hipMemcpy(d, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice);
}

// Sets up the split exchange of the context, if its mesh allows it.
int split_exchange(cfx_ctx *ctx) {
  ctx->ex_split = false;
  if (ctx->n_bc_ops == (int)ctx->ops.size()) return 0;
  std::vector<FaceOp> mid;
  std::vector<std::vector<FaceOp>> rest;
  std::vector<ExSlot> slots;
  std::vector<ExOp> ops;
  std::vector<int> slot_off, op_off;
  if (!split_ops(ctx->ops, ctx->n_bc_ops, ctx->dim, mid, rest)) return 0;
  if (!build_strips(ctx, rest, slots, ops, slot_off, op_off, ctx->strips.end)) return 0;
  int rc;
  std::vector<int> one(mid.size(), 0);
  if ((rc = build_schedule(ctx, mid, ctx->sched_mid, 0, (int)mid.size(), false, &one)) ||
      (rc = upload(ctx, slots, ctx->strips.slots)) || (rc = upload(ctx, ops, ctx->strips.ops)) ||
      (rc = upload(ctx, slot_off, ctx->strips.slot_off)) || (rc = upload(ctx, op_off, ctx->strips.op_off)))
    return rc;
  ctx->ex_split = true;
  return 0;
}

// BC ops in the application order (BoundCond.cu:251-313), then the inner-face
// exchanges block by block, face by face (Driver.cu:194-217).
int build_ops(cfx_ctx *ctx) {
  ctx->ops.clear();
  for (const BcOp &b : ctx->bc_order) {
    const HostBlock &H = ctx->hb[b.blk];
    FaceOp op{};
    op.kind = b.type;
    op.blk = b.blk;
    op.tgt = b.blk;
    op.cond = H.bc_cond[b.face];
    op.r = H.bc_range[b.face];
    if (b.type == CFX_BC_WALL) {
      op.wl = ctx->walls[op.cond];
      for (int q = 0; q < 3; ++q) {
        if (q == op.r.face) continue;
        op.r.rs[q] += kNgg;
        op.r.re[q] -= kNgg;
      }
      if (op.r.rs[0] > op.r.re[0] || op.r.rs[1] > op.r.re[1] || op.r.rs[2] > op.r.re[2]) continue;
    }
    for (int q = 0; q < 3; ++q) op.ext[q] = op.r.re[q] - op.r.rs[q] + 1;
    op.npts = (long long)op.ext[0] * op.ext[1] * op.ext[2];
    ctx->ops.push_back(op);
  }
  ctx->n_bc_ops = (int)ctx->ops.size();
  for (size_t b = 0; b < ctx->hb.size(); ++b)
    for (const InnerDev &f : ctx->hb[b].inner) {
      FaceOp op{};
      op.kind = kOpExchange;
      op.blk = (int)b;
      op.tgt = f.target_block;
      op.f = f;
      for (int q = 0; q < 3; ++q) op.ext[q] = f.n_point[q];
      op.npts = (long long)op.ext[0] * op.ext[1] * op.ext[2];
      ctx->ops.push_back(op);
    }
  const int n = (int)ctx->ops.size(), nbc = ctx->n_bc_ops;
  int rc;
  if ((rc = build_schedule(ctx, ctx->ops, ctx->sched_seq, 0, n, false)) ||
      (rc = build_schedule(ctx, ctx->ops, ctx->sched_bc, 0, nbc, true)) ||
      (rc = build_schedule(ctx, ctx->ops, ctx->sched_ex, nbc, n, true)) ||
      (rc = build_schedule(ctx, ctx->ops, ctx->sched_all, 0, n, true)))
    return rc;
  // the step's ghost fill, with the outflow faces folded into the update
  fold_outflow(ctx);
  const int ns = (int)ctx->ops_step.size();
  if ((rc = build_schedule(ctx, ctx->ops_step, ctx->sched_seq_step, 0, ns, false, &ctx->ops_step_src)) ||
      (rc = build_schedule(ctx, ctx->ops_step, ctx->sched_all_step, 0, ns, true)))
    return rc;
  ctx->plane_only = ctx->dim == 2;
  for (const FaceOp &op : ctx->ops) {
    const HostBlock &H = ctx->hb[op.blk];
    const int a = op.kind == kOpExchange ? op.f.face : op.r.face;
    const int end[3] = {H.mx - 1, H.my - 1, H.mz - 1};
    bool edge = a != 2;
    if (op.kind == kOpExchange) edge = edge && op.f.src_tar[2] == 2;
    else edge = edge && op.r.rs[a] == op.r.re[a] && (op.r.rs[a] == 0 || op.r.rs[a] == end[a]);
    ctx->plane_only = ctx->plane_only && edge;
  }
  int nbc_step = 0;  // fold_outflow keeps the order: boundary conditions first
  while (nbc_step < ns && ctx->ops_step[nbc_step].kind != kOpExchange) ++nbc_step;
  if ((rc = split_exchange(ctx)) ||
      (rc = build_schedule(ctx, ctx->ops_step, ctx->sched_bc_step, 0, nbc_step, true)))
    return rc;
  return (int)hipMemcpy(ctx->views_dev, ctx->views.data(), sizeof(BlockView) * ctx->views.size(),
                        hipMemcpyHostToDevice);
}

// levels [l0, l1) of a schedule, one launch each
int run_levels(cfx_ctx *ctx, const Schedule &sc, int l0, int l1) {
  const KernelSet64 &k = g_kernels64[ctx->ns];
  for (int L = l0; L < l1; ++L) {
    const int a = sc.lvl[L], b = sc.lvl[L + 1];
    const int total = sc.off_host[b] - sc.off_host[a];
    CFX_TRY(ctx->timed_launch(K_BC, [&] {
      if (sc.copies[L])
        return k.copy_ops(ctx->views_dev, sc.ops + a, sc.off + a, b - a, total, ctx->mixed ? 1 : 0, ctx->stream);
      return k.face_ops(ctx->views_dev, sc.ops + a, sc.off + a, b - a, total, ctx->sp_dev, ctx->S, ctx->inflow_dev,
                        ctx->stream);
    }));
  }
  return 0;
}

// ------------------------------------------------------------ step parts ---
// 2-D: both face directions; the variant of direction 1 counts
int rhs_plane(cfx_ctx *ctx, int blk, bool planar) {
  const int v = ctx->rhs_var[1];
  const PlaneFn fn = ctx->mixed ? g_kernels32[ctx->ns].plane[v] : g_kernels64[ctx->ns].plane[v];
  const Batch b = blk < 0 ? ctx->all(ctx->t_rhs[v]) : ctx->one(ctx->t_rhs[v], blk);
  return ctx->timed_launch(K_RHS, [&] { return fn(b, planar ? 1 : 0, ctx->sp_dev, ctx->S, ctx->stream); });
}

// 3-D: all face directions; the march runs along k, so the variant of that direction counts
int rhs_march(cfx_ctx *ctx, int blk) {
  const int v = ctx->rhs_var[2];
  const MarchFn fn = ctx->mixed ? g_kernels32[ctx->ns].march : g_kernels64[ctx->ns].march;
  const Batch b = blk < 0 ? ctx->all(ctx->t_march[v]) : ctx->one(ctx->t_march[v], blk);
  return ctx->timed_launch(K_RHS, [&] {
    return fn(b, ctx->march_chunk[v], ctx->march_big ? 1 : 0, ctx->sp_dev, ctx->S, ctx->stream);
  });
}

// blk < 0: every block; planar: see rhs_plane
int do_rhs(cfx_ctx *ctx, int blk, bool planar = false) {
  auto run = [&](int b) { return ctx->dim == 3 ? rhs_march(ctx, b) : rhs_plane(ctx, b, planar); };
  if (blk >= 0 || ctx->batched) {
    CFX_TRY(run(blk));
    return 0;
  }
  for (int b = 0; b < (int)ctx->views.size(); ++b) CFX_TRY(run(b));
  return 0;
}

// runs f(batch) over all blocks at once, or block by block
template <class F>
int per_batch(cfx_ctx *ctx, const Table &t, F &&f) {
  if (ctx->batched) return f(ctx->all(t));
  for (size_t b = 0; b < ctx->views.size(); ++b)
    if (int rc = f(ctx->one(t, (int)b))) return rc;
  return 0;
}

// reset: whether the reduction's target needs it (not after do_store_last with reset)
int do_dt(cfx_ctx *ctx, int global, int store_local, bool reset = true) {
  auto *bits = reinterpret_cast<unsigned long long *>(ctx->d_dt);
  if (global && reset) CFX_TRY(ctx->timed_launch(K_DT, [&] { return launch_dt_reset(bits, ctx->stream); }));
  CFX_TRY(per_batch(ctx, ctx->t_dt, [&](const Batch &b) {
    return ctx->timed_launch(K_DT, [&] {
      return launch_dt(b, ctx->S, ctx->ns, ctx->dt_iter, store_local, global ? bits : ctx->d_minscratch, ctx->stream);
    });
  }));
  return 0;
}

int do_update(cfx_ctx *ctx, int stage) {
  const KernelSet64 &k = g_kernels64[ctx->ns];
  CFX_TRY(per_batch(ctx, ctx->t_int, [&](const Batch &b) {
    return ctx->timed_launch(K_UPDATE, [&] {
      return k.update(b, ctx->sp_dev, ctx->S, ctx->mixed ? 1 : 0, stage, ctx->d_dt, ctx->d_flags, ctx->d_newton,
                      ctx->stream);
    });
  }));
  return 0;
}

// LU-SGS solve (the implicit treatment of Driver.cu:156): coefficients, then
// the forward and the backward sweep; dq <- dQ
int do_lusgs(cfx_ctx *ctx) {
  const KernelSet64 &k = g_kernels64[ctx->ns];
  CFX_TRY(per_batch(ctx, ctx->t_int, [&](const Batch &b) {
    return ctx->timed_launch(K_UPDATE, [&] { return k.lusgs_coef(b, ctx->S, ctx->stream); });
  }));
  // blk < 0: every block in one launch
  auto sweep = [&](int blk, int fwd) {
    const Batch pts = blk < 0 ? ctx->all(ctx->t_int) : ctx->one(ctx->t_int, blk);
    const int first = blk < 0 ? 0 : ctx->lu_off[blk], n = (blk < 0 ? ctx->lu_off[0] : ctx->lu_off[blk + 1]) - first;
    const BlockView *views = blk < 0 ? ctx->views_dev : ctx->views_dev + blk;
    CFX_TRY(ctx->timed_launch(K_UPDATE, [&] { return k.lusgs_reset(pts, ctx->lu_ticket, ctx->stream); }));
    CFX_TRY(ctx->timed_launch(K_UPDATE, [&] {
      return k.lusgs_sweep(views, ctx->lu_order + first, n, ctx->lu_ticket, ctx->S, fwd, ctx->d_flags, ctx->stream);
    }));
    return 0;
  };
  for (int fwd = 1; fwd >= 0; --fwd) {
    if (ctx->batched) {
      if (int rc = sweep(-1, fwd)) return rc;
      continue;
    }
    for (int b = 0; b < (int)ctx->views.size(); ++b)
      if (int rc = sweep(b, fwd)) return rc;
  }
  return 0;
}

int do_bc(cfx_ctx *ctx) {
  if (ctx->batched) return run_levels(ctx, ctx->sched_bc, 0, ctx->sched_bc.levels());
  return run_levels(ctx, ctx->sched_seq, 0, ctx->n_bc_ops);
}

int exchange_split(cfx_ctx *ctx) {
  if (int rc = run_levels(ctx, ctx->sched_mid, 0, ctx->sched_mid.levels())) return rc;
  CFX_TRY(ctx->timed_launch(K_BC, [&] {
    return launch_exchange_strips(ctx->views_dev, ctx->strips, ctx->ns, ctx->mixed ? 1 : 0, ctx->stream);
  }));
  return 0;
}

int do_exchange(cfx_ctx *ctx) {
  if (ctx->batched && ctx->ex_split) return exchange_split(ctx);
  if (ctx->batched) return run_levels(ctx, ctx->sched_ex, 0, ctx->sched_ex.levels());
  return run_levels(ctx, ctx->sched_seq, ctx->n_bc_ops, ctx->sched_seq.levels());
}

// boundary conditions followed by the inner-face exchange; after_update:
// the step's schedule, whose folded outflow rows the update kernel has filled
int do_ghosts(cfx_ctx *ctx, bool after_update) {
  if (ctx->batched && ctx->ex_split) {
    const Schedule &bc = after_update ? ctx->sched_bc_step : ctx->sched_bc;
    if (int rc = run_levels(ctx, bc, 0, bc.levels())) return rc;
    return exchange_split(ctx);
  }
  const Schedule &all = after_update ? ctx->sched_all_step : ctx->sched_all;
  const Schedule &seq = after_update ? ctx->sched_seq_step : ctx->sched_seq;
  if (ctx->batched) return run_levels(ctx, all, 0, all.levels());
  return run_levels(ctx, seq, 0, seq.levels());
}

int do_elim(cfx_ctx *ctx) {
  if (ctx->dim != 2) return 0;
  for (auto &B : ctx->views)
    CFX_TRY(ctx->timed_launch(K_OTHER, [&] { return launch_eliminate_k(B, ctx->ns, ctx->stream); }));
  return 0;
}

// mode: kProps... (the 2-D ones not with the surrogate)
int do_props(cfx_ctx *ctx, int mode = kPropsPadded) {
  if (ctx->transport == CFX_TRANSPORT_MLP) {
    if (!ctx->mlp_ready) return ctx->fail(CFX_E_SURROGATE, "surrogate transport selected but not trained or loaded");
    auto fn = g_kernels32[ctx->ns].props_mlp;
    CFX_TRY(per_batch(ctx, ctx->t_pad, [&](const Batch &b) {
      return ctx->timed_launch(K_PROPS, [&] {
        return fn(b, ctx->sp_dev, ctx->S, ctx->mlp_dev, ctx->mlp_ops_inf, ctx->mlp_bias_inf, ctx->mlp_counters,
                  ctx->stream);
      });
    }));
    return 0;
  }
  auto fn = ctx->mixed ? g_kernels32[ctx->ns].props : g_kernels64[ctx->ns].props;
  CFX_TRY(per_batch(ctx, mode == kPropsPadded ? ctx->t_pad : ctx->t_plane, [&](const Batch &b) {
    return ctx->timed_launch(K_PROPS, [&] { return fn(b, mode, ctx->sp_dev, ctx->S, ctx->stream); });
  }));
  return 0;
}

// reset_dt: also resets the target of the global time step's reduction
int do_store_last(cfx_ctx *ctx, bool reset_dt = false) {
  auto *bits = reset_dt ? reinterpret_cast<unsigned long long *>(ctx->d_dt) : nullptr;
  CFX_TRY(per_batch(ctx, ctx->t_last, [&](const Batch &b) {
    return ctx->timed_launch(K_OTHER, [&] { return launch_store_last(b, ctx->last_iter, bits, ctx->stream); });
  }));
  return 0;
}

// Driver::steady_simulation loop body (Driver.cu:135-190): with rk_stages 1
// the reference's explicit Euler with local dt; with 3 the SSP-RK3 stages
// with the global CFL dt taken at stage 0.
// 2-D RK3: the ghost planes along k are read by the RHS, whose differences
// along k vanish where they are copies of the plane, and near the faces by the
// ghost fills, which cover their tangential rows too.  The stages within the
// step therefore work on the plane alone (RHS without k differences, copies of
// the ring near the faces, properties of the plane); the full copies and the
// properties of all planes are made once, for the state the step leaves.  The
// properties kernel makes the copies: 1021x509 air, copies and properties
// together 68 us per stage -> 11 us within a step, 34 us at its end.  (The
// surrogate counts the points it falls back on, over all planes, and keeps the
// full stages.)
bool works_on_plane(const cfx_ctx *ctx) { return ctx->plane_only && ctx->transport != CFX_TRANSPORT_MLP; }
// whether a step has stages after the first that do
bool stages_on_plane(const cfx_ctx *ctx) { return ctx->rk == 3 && works_on_plane(ctx); }

int do_step(cfx_ctx *ctx) {
  int rc;
  if ((rc = do_store_last(ctx, ctx->rk == 3))) return rc;
  const int stages = ctx->rk == 3 ? 3 : 1;
  const bool planar = works_on_plane(ctx);
  for (int s = 0; s < stages; ++s) {
    const bool last = s == stages - 1;
    if ((rc = do_rhs(ctx, -1, planar && s > 0))) return rc;
    if (ctx->rk == 3) {
      if (s == 0 && (rc = do_dt(ctx, 1, 0, /*reset=*/false))) return rc;
    } else {
      if ((rc = do_dt(ctx, 0, 1))) return rc;
    }
    if (ctx->lusgs && (rc = do_lusgs(ctx))) return rc;
    if ((rc = do_update(ctx, s))) return rc;
    if ((rc = do_ghosts(ctx, true))) return rc;
    if (!planar && (rc = do_elim(ctx))) return rc;
    if ((rc = do_props(ctx, !planar ? kPropsPadded : (last ? kPropsPlanes : kPropsRing)))) return rc;
  }
  return 0;
}

// One step captured as a graph (kernel nodes only: the dt reset is a kernel,
// nothing is copied or set by the runtime inside the step).
int ensure_graph(cfx_ctx *ctx) {
  if (ctx->graph_exec) return 0;
  CFX_TRY((int)hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
  const int rc = do_step(ctx);
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(ctx->stream, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return ctx->fail((int)e, "hipStreamEndCapture");
  ctx->graph = g;
  CFX_TRY((int)hipGraphInstantiate(&ctx->graph_exec, g, nullptr, nullptr, 0));
  return 0;
}

int run_steps(cfx_ctx *ctx, int n_steps) {
  if (ctx->use_graph && !ctx->profiling) {
    if (n_steps > 0) CFX_TRY(ensure_graph(ctx));
    for (int s = 0; s < n_steps; ++s) CFX_TRY((int)hipGraphLaunch(ctx->graph_exec, ctx->stream));
    return 0;
  }
  for (int s = 0; s < n_steps; ++s)
    if (int rc = do_step(ctx)) return rc;
  return 0;
}

}  // namespace

extern "C" {

namespace cfx {
namespace {

// The (ngg+1)-layer coordinate arrays of every block built on the device
// (Mesh::init_ghost_grid, Mesh.cpp:718-922): interior vertices uploaded and
// scattered, mirror extrapolation per block, the inter-block copies in the
// reference's block and face order, then edges and corners per block; the
// arrays stay resident (CFX_COORD, the metric fallback).  A block whose inner
// face names the block itself would read points the same copy writes, so
// such meshes keep the host path (ctx->coords empty, hb[].xyz filled).
int device_ghost_grid(cfx_ctx *ctx, const cfx_block *blocks, int n_block) {
  const int nb = n_block;
  ctx->coords.assign(nb, nullptr);
  int rc = 0;
  long long max_ni = 0;
  for (int b = 0; b < nb; ++b) {
    const HostBlock &H = ctx->hb[b];
    ctx->coords[b] = ctx->dalloc<double>(3 * (size_t)H.gx * H.gy * H.gz, rc);
    max_ni = std::max(max_ni, H.ni);
  }
  if (rc) return ctx->fail(rc, "hipMalloc coordinates");
  double *raw = nullptr;
  rc = (int)hipMalloc(&raw, sizeof(double) * 3 * (size_t)max_ni);
  for (int b = 0; b < nb && !rc; ++b) {
    const HostBlock &H = ctx->hb[b];
    const size_t ni = (size_t)H.ni;
    const double *src[3] = {blocks[b].x, blocks[b].y, blocks[b].z};
    for (int c = 0; c < 3 && !rc; ++c) rc = (int)hipMemcpy(raw + c * ni, src[c], sizeof(double) * ni, hipMemcpyHostToDevice);
    if (!rc) rc = launch_coord_scatter(raw, H.mx, H.my, H.mz, ctx->coords[b], nullptr);
    if (!rc) rc = launch_ghost_extrapolate(ctx->coords[b], H.mx, H.my, H.mz, ctx->dim, nullptr);
    if (!rc) rc = (int)hipDeviceSynchronize();  // raw is reused by the next block
  }
  (void)hipFree(raw);
  if (rc) return ctx->fail(rc, "device ghost grid");
  for (const GhostCopy &g : inner_ghost_copies(ctx->hb, blocks, ctx->dim)) {
    const HostBlock &D = ctx->hb[g.blk], &S = ctx->hb[g.src];
    if ((rc = launch_ghost_inner(g, ctx->coords[g.blk], D.mx, D.my, D.mz, ctx->coords[g.src], S.mx, S.my, S.mz,
                                 nullptr)))
      return ctx->fail(rc, "device inner ghost grid");
  }
  for (int b = 0; b < nb; ++b) {
    const HostBlock &H = ctx->hb[b];
    if ((rc = launch_ghost_corners(ctx->coords[b], H.mx, H.my, H.mz, nullptr))) return ctx->fail(rc, "device corners");
  }
  rc = (int)hipDeviceSynchronize();
  return rc ? ctx->fail(rc, "device ghost grid") : 0;
}

// The host copy of block b's coordinates (downloaded from the device arrays
// when the ghost grid was built there).
int host_coords(cfx_ctx *ctx, int b) {
  HostBlock &H = ctx->hb[b];
  if (!H.xyz[0].empty() || ctx->coords.empty()) return 0;
  const size_t ng = (size_t)H.gx * H.gy * H.gz;
  for (int c = 0; c < 3; ++c) {
    H.xyz[c].resize(ng);
    if (int rc = (int)hipMemcpy(H.xyz[c].data(), ctx->coords[b] + c * ng, sizeof(double) * ng, hipMemcpyDeviceToHost))
      return ctx->fail(rc, "coordinate download");
  }
  return 0;
}

// Metrics of one block computed on the device from its ghost-grid
// coordinates; a block with a non-positive Jacobian anywhere is recomputed on
// the host with the reference's fallback rules and uploaded.
int device_metrics(cfx_ctx *ctx, int b, const BlockView &V) {
  HostBlock &H = ctx->hb[b];
  const size_t ng = (size_t)H.gx * H.gy * H.gz, np = (size_t)H.np;
  const bool resident = !ctx->coords.empty();
  double *xyz = resident ? ctx->coords[b] : nullptr;
  int *bad = nullptr;
  int rc = resident ? 0 : (int)hipMalloc(&xyz, sizeof(double) * 3 * ng);
  if (!rc) rc = (int)hipMalloc(&bad, sizeof(int));
  for (int c = 0; c < 3 && !rc && !resident; ++c)
    rc = (int)hipMemcpy(xyz + c * ng, H.xyz[c].data(), sizeof(double) * ng, hipMemcpyHostToDevice);
  if (!rc) rc = (int)hipMemset(bad, 0, sizeof(int));
  if (!rc) rc = launch_metrics(xyz, H.mx, H.my, H.mz, V.metric, V.jac, V.mixed ? V.metric32 : nullptr,
                               V.mixed ? V.jac32 : nullptr, bad, nullptr);
  int n_bad = 0;
  if (!rc) rc = (int)hipMemcpy(&n_bad, bad, sizeof(int), hipMemcpyDeviceToHost);
  if (!resident) (void)hipFree(xyz);
  (void)hipFree(bad);
  if (rc) return ctx->fail(rc, "device metrics");
  if (n_bad == 0) return 0;
  if ((rc = host_coords(ctx, b))) return rc;
  if ((rc = compute_metrics(H, ctx->err))) return rc;
  rc = (int)hipMemcpy(V.metric, H.metric.data(), sizeof(double) * 9 * np, hipMemcpyHostToDevice);
  if (!rc) rc = (int)hipMemcpy(V.jac, H.jac.data(), sizeof(double) * np, hipMemcpyHostToDevice);
  if (!rc && V.mixed) {
    std::vector<float> m32(9 * np), j32(np);
    for (size_t i = 0; i < 9 * np; ++i) m32[i] = (float)H.metric[i];
    for (size_t i = 0; i < np; ++i) j32[i] = (float)H.jac[i];
    rc = (int)hipMemcpy(V.metric32, m32.data(), sizeof(float) * 9 * np, hipMemcpyHostToDevice);
    if (!rc) rc = (int)hipMemcpy(V.jac32, j32.data(), sizeof(float) * np, hipMemcpyHostToDevice);
  }
  std::vector<double>().swap(H.metric);
  std::vector<double>().swap(H.jac);
  if (resident)
    for (int c = 0; c < 3; ++c) std::vector<double>().swap(H.xyz[c]);
  return rc ? ctx->fail(rc, "metric upload") : 0;
}

}  // namespace
}  // namespace cfx

int cfx_version(void) { return CFX_ABI_VERSION; }

int cfx_ghost_grid(const cfx_block *blocks, int n_block, double *const *xyz) {
  if (!blocks || n_block <= 0 || !xyz) return CFX_E_ARG;
  std::vector<HostBlock> hb;
  int dim = 0;
  std::string err;
  if (int rc = build_mesh(blocks, n_block, hb, dim, err, /*metrics=*/false)) return rc;
  for (int b = 0; b < n_block; ++b) {
    const HostBlock &B = hb[b];
    if (!xyz[b]) return CFX_E_ARG;
    for (int c = 0; c < 3; ++c)
      for (int k = -kNgg; k < B.mz + kNgg; ++k)
        for (int j = -kNgg; j < B.my + kNgg; ++j)
          for (int i = -kNgg; i < B.mx + kNgg; ++i)
            xyz[b][c * B.np + B.pidx(i, j, k)] = B.xyz[c][B.gidx(i, j, k)];
  }
  return 0;
}

int cfx_inflow_state(const cfx_params *params, const cfx_species *species, int index, double bv[6], double *yk) {
  if (!params || !bv || index < 0 || index >= params->n_inflow || !params->inflow) return CFX_E_ARG;
  SpeciesDev tables;
  std::string err;
  if (int rc = build_species(species, tables, err)) return rc;
  SchemeDev S{};
  S.gamma_air = params->gamma_air > 0 ? params->gamma_air : 1.4;
  S.r_air = params->r_air > 0 ? params->r_air : kRuH / kMwAir;
  InflowDev d;
  if (int rc = build_inflow(params->inflow[index], tables.d, S, d, err)) return rc;
  for (int v = 0; v < 6; ++v) bv[v] = d.st[v];
  if (yk)
    for (int l = 0; l < tables.d.ns; ++l) yk[l] = d.y[l];
  return 0;
}

int cfx_create(const cfx_params *params, const cfx_species *species, const cfx_block *blocks, int n_block,
               cfx_ctx **out) {
  if (!params || !blocks || n_block <= 0 || !out) return CFX_E_ARG;
  *out = nullptr;
  auto *ctx = new cfx_ctx;
  auto bail = [&](int rc) {
    cfx_destroy(ctx);
    return rc;
  };
  int rc = build_species(species, ctx->sp_host, ctx->err);
  if (rc) return bail(rc);
  ctx->ns = ctx->sp_host.d.ns;
  ctx->nv = 5 + ctx->ns;
  if (!g_kernels64[ctx->ns].present) {
    ctx->err = "no kernels built for " + std::to_string(ctx->ns) + " species";
    return bail(CFX_E_UNSUPPORTED);
  }
  if (params->inviscid_scheme != 3 && params->inviscid_scheme != 0) return bail(CFX_E_UNSUPPORTED);
  if ((params->precision != CFX_FP64 && params->precision != CFX_MIXED) ||
      (params->transport != CFX_TRANSPORT_WILKE && params->transport != CFX_TRANSPORT_MLP))
    return bail(CFX_E_UNSUPPORTED);
  ctx->mixed = params->precision == CFX_MIXED;
  if (params->transport == CFX_TRANSPORT_MLP &&
      (!ctx->mixed || ctx->ns < 1 || ctx->ns > kMlpMaxSp || !g_kernels32[ctx->ns].props_mlp)) {
    ctx->err = "surrogate transport needs the mixed-precision path and 1..14 species";
    return bail(CFX_E_UNSUPPORTED);
  }
  ctx->transport = params->transport;
  if (ctx->mixed && !g_kernels32[ctx->ns].present) {
    ctx->err = "no FP32 kernels built for " + std::to_string(ctx->ns) + " species";
    return bail(CFX_E_UNSUPPORTED);
  }
  bool self_face = false;  // an inner face that names its own block keeps the host ghost grid
  for (int b = 0; b < n_block; ++b)
    for (int f = 0; f < blocks[b].n_inner; ++f) self_face |= blocks[b].inner[f].target_block == b + 1;
  rc = build_mesh(blocks, n_block, ctx->hb, ctx->dim, ctx->err, /*metrics=*/false, /*ghosts=*/self_face);
  if (rc) return bail(rc);
  SchemeDev &S = ctx->S;
  S.reconstruction = params->reconstruction;
  S.limiter = params->limiter;
  S.viscous = params->viscous_order;
  S.quirks = params->quirks;
  S.rk = params->rk_stages == 3 ? 3 : 1;
  S.dim = ctx->dim;
  S.cfl = params->cfl;
  S.pr = params->prandtl;
  S.sc = params->schmidt;
  S.gamma_air = params->gamma_air > 0 ? params->gamma_air : 1.4;
  S.r_air = params->r_air > 0 ? params->r_air : kRuH / kMwAir;
  S.inv_sc = 1.0 / S.sc;
  S.inv_pr = 1.0 / S.pr;
  S.lusgs = params->lusgs ? 1 : 0;
  S.omega = params->lusgs_omega > 0 ? params->lusgs_omega : 1.0;
  ctx->rk = S.rk;
  ctx->lusgs = S.lusgs != 0;
  if (ctx->lusgs && (S.rk != 1 || ctx->mixed)) {
    ctx->err = "the LU-SGS step needs rk_stages 1 (local time step) and FP64";
    return bail(CFX_E_UNSUPPORTED);
  }
  for (int i = 0; i < params->n_inflow; ++i) {
    InflowDev d;
    rc = build_inflow(params->inflow[i], ctx->sp_host.d, S, d, ctx->err);
    if (rc) return bail(rc);
    ctx->inflow_host.push_back(d);
  }
  for (int i = 0; i < params->n_wall; ++i)
    ctx->walls.push_back(WallDev{params->wall[i].adiabatic, params->wall[i].temperature});
  // boundary application order (BoundCond.cu:251-313): outflow, inflow,
  // symmetry, wall; within a type by condition record, block, face
  const int order[4] = {CFX_BC_OUTFLOW, CFX_BC_INFLOW, CFX_BC_SYMMETRY, CFX_BC_WALL};
  for (int type : order) {
    const bool by_cond = type == CFX_BC_INFLOW || type == CFX_BC_WALL;
    const int ncond = type == CFX_BC_INFLOW ? (int)ctx->inflow_host.size()
                                            : (type == CFX_BC_WALL ? (int)ctx->walls.size() : 1);
    for (int cond = 0; cond < ncond; ++cond)
      for (int b = 0; b < n_block; ++b)
        for (size_t f = 0; f < ctx->hb[b].bc_type.size(); ++f)
          if (ctx->hb[b].bc_type[f] == type && (!by_cond || ctx->hb[b].bc_cond[f] == cond))
            ctx->bc_order.push_back(BcOp{type, b, (int)f});
  }
  for (int b = 0; b < n_block; ++b)
    for (size_t f = 0; f < ctx->hb[b].bc_type.size(); ++f) {
      const int t = ctx->hb[b].bc_type[f], c = ctx->hb[b].bc_cond[f];
      if ((t == CFX_BC_INFLOW && (c < 0 || c >= (int)ctx->inflow_host.size())) ||
          (t == CFX_BC_WALL && (c < 0 || c >= (int)ctx->walls.size()))) {
        ctx->err = "boundary condition record out of range";
        return bail(CFX_E_ARG);
      }
    }
  hipError_t e = hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking);
  if (e != hipSuccess) return bail(ctx->fail((int)e, "hipStreamCreate"));
  rc = 0;
  ctx->sp_dev = ctx->dalloc<SpeciesDev>(1, rc);
  ctx->inflow_dev = ctx->dalloc<InflowDev>(std::max<size_t>(1, ctx->inflow_host.size()), rc);
  ctx->d_dt = ctx->dalloc<double>(1, rc);
  ctx->d_res = ctx->dalloc<double>(4, rc);
  ctx->d_flags = ctx->dalloc<int>(1, rc);
  ctx->d_newton = ctx->dalloc<unsigned long long>(1, rc);
  ctx->d_minscratch = ctx->dalloc<unsigned long long>(1, rc);
  if (rc) return bail(ctx->fail(rc, "hipMalloc"));
  rc = (int)hipMemcpy(ctx->sp_dev, &ctx->sp_host, sizeof(SpeciesDev), hipMemcpyHostToDevice);
  if (!rc && !ctx->inflow_host.empty())
    rc = (int)hipMemcpy(ctx->inflow_dev, ctx->inflow_host.data(), sizeof(InflowDev) * ctx->inflow_host.size(),
                        hipMemcpyHostToDevice);
  if (!rc) rc = (int)hipMemset(ctx->d_flags, 0, sizeof(int));
  if (!rc) rc = (int)hipMemset(ctx->d_newton, 0, sizeof(unsigned long long));
  const double dt0 = 0.0;
  if (!rc) rc = (int)hipMemcpy(ctx->d_dt, &dt0, sizeof(double), hipMemcpyHostToDevice);
  if (rc) return bail(ctx->fail(rc, "context upload"));
  for (int b = 0; b < n_block; ++b)
    if (ctx->hb[b].np >= (1LL << 29)) {  // the RHS kernels address a block with 32-bit byte offsets
      ctx->err = "block " + std::to_string(b) + " exceeds 2^29 padded points";
      return bail(CFX_E_UNSUPPORTED);
    }
  for (int b = 0; b < n_block; ++b) {
    const HostBlock &H = ctx->hb[b];
    BlockView V{};
    V.mx = H.mx;
    V.my = H.my;
    V.mz = H.mz;
    V.px = H.px;
    V.py = H.py;
    V.pz = H.pz;
    V.np = H.np;
    V.ni = H.ni;
    V.sy = H.px;
    V.sz = (long long)H.px * H.py;
    const size_t np = (size_t)H.np, ni = (size_t)H.ni;
    V.cv = ctx->dalloc<double>(ctx->nv * np, rc);
    V.bv = ctx->dalloc<double>(6 * np, rc);
    V.yk = ctx->dalloc<double>(ctx->ns * np, rc);
    V.props = ctx->dalloc<double>((4 + ctx->ns) * np, rc);
    V.metric = ctx->dalloc<double>(9 * np, rc);
    V.jac = ctx->dalloc<double>(np, rc);
    V.dq = ctx->dalloc<double>(ctx->nv * ni, rc);
    V.qn = ctx->dalloc<double>(ctx->nv * ni, rc);
    V.dt_local = ctx->dalloc<double>(ni, rc);
    V.bv_last = ctx->dalloc<double>(4 * ni, rc);
    if (ctx->lusgs) {
      V.lus = ctx->dalloc<double>(4 * ni, rc);
      // the implicit step has no stage base: its array takes the hand-over,
      // unless the block is so thin that the patches' edges need more
      const int m[3] = {H.mx, H.my, H.mz};
      const size_t n = (size_t)lu_hand_over(m, ctx->ns);
      V.luf = n <= ctx->nv * ni ? V.qn : ctx->dalloc<double>(n, rc);
    }
    if (rc) return bail(ctx->fail(rc, "hipMalloc block arrays"));
    V.mixed = ctx->mixed ? 1 : 0;
    if (ctx->mixed) {
      V.bv32 = ctx->dalloc<float>(6 * np, rc);
      V.yk32 = ctx->dalloc<float>(ctx->ns * np, rc);
      V.props32 = ctx->dalloc<float>((4 + ctx->ns) * np, rc);
      V.metric32 = ctx->dalloc<float>(9 * np, rc);
      V.jac32 = ctx->dalloc<float>(np, rc);
      V.dq32 = ctx->dalloc<float>(ctx->nv * ni, rc);
      if (rc) return bail(ctx->fail(rc, "hipMalloc FP32 arrays"));
      rc = (int)hipMemset(V.props32, 0, sizeof(float) * (4 + ctx->ns) * np);
      if (!rc) rc = (int)hipMemset(V.dq32, 0, sizeof(float) * ctx->nv * ni);
    }
    if (!rc) rc = (int)hipMemset(V.props, 0, sizeof(double) * (4 + ctx->ns) * np);
    if (!rc) rc = (int)hipMemset(V.dq, 0, sizeof(double) * ctx->nv * ni);
    if (rc) return bail(ctx->fail(rc, "block array clear"));
    ctx->views.push_back(V);
    ctx->n_grid_total += H.ni;
  }
  if (!self_face && (rc = device_ghost_grid(ctx, blocks, n_block))) return bail(rc);
  for (int b = 0; b < n_block; ++b)
    if ((rc = device_metrics(ctx, b, ctx->views[b]))) return bail(rc);
  ctx->views_dev = ctx->dalloc<BlockView>(ctx->views.size(), rc);
  if (rc) return bail(ctx->fail(rc, "hipMalloc block table"));
  if ((rc = (int)hipMemcpy(ctx->views_dev, ctx->views.data(), sizeof(BlockView) * ctx->views.size(),
                           hipMemcpyHostToDevice)))
    return bail(ctx->fail(rc, "block table upload"));
  if ((rc = build_tables(ctx))) return bail(ctx->fail(rc, "work tables"));
  if ((rc = build_ops(ctx))) return bail(ctx->fail(rc, "ghost-fill schedule"));
  ctx->n_partial = ctx->t_res.host.back();
  ctx->d_partial = ctx->dalloc<double>(4 * (size_t)ctx->n_partial, rc);
  if (rc) return bail(ctx->fail(rc, "hipMalloc partials"));
  {
    int dev = 0, ncu = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && ncu > 0)
      ctx->n_cu = ncu;
  }
  if ((rc = plan_march(ctx))) return bail(ctx->fail(rc, "march table"));
  if ((rc = plan_sweeps(ctx))) return bail(ctx->fail(rc, "sweep order"));
  e = hipDeviceSynchronize();
  if (e != hipSuccess) return bail(ctx->fail((int)e, "device setup"));
  *out = ctx;
  return 0;
}

void cfx_destroy(cfx_ctx *ctx) {
  if (!ctx) return;
  if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
  ctx->drop_graph();
  for (auto &t : ctx->timed) {
    (void)hipEventDestroy(t.a);
    (void)hipEventDestroy(t.b);
  }
  for (auto e : ctx->event_pool) (void)hipEventDestroy(e);
  for (void *p : ctx->allocs) (void)hipFree(p);
  if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
  delete ctx;
}

const char *cfx_last_error(const cfx_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

static int check_blk(cfx_ctx *ctx, int blk) {
  if (!ctx) return CFX_E_ARG;
  if (blk < 0 || blk >= (int)ctx->views.size()) return ctx->fail(CFX_E_ARG, "block index out of range");
  return 0;
}

int cfx_upload_primitive(cfx_ctx *ctx, int blk, const double *bv, const double *yk) {
  if (int rc = check_blk(ctx, blk)) return rc;
  if (!bv || (ctx->ns > 0 && !yk)) return ctx->fail(CFX_E_ARG, "null field");
  BlockView &V = ctx->views[blk];
  (void)hipStreamSynchronize(ctx->stream);
  CFX_TRY((int)hipMemcpy(V.bv, bv, sizeof(double) * 6 * V.np, hipMemcpyHostToDevice));
  if (ctx->ns > 0) CFX_TRY((int)hipMemcpy(V.yk, yk, sizeof(double) * ctx->ns * V.np, hipMemcpyHostToDevice));
  return 0;
}

int cfx_upload_state(cfx_ctx *ctx, int blk, const double *cv, const double *bv, const double *yk) {
  if (int rc = cfx_upload_primitive(ctx, blk, bv, yk)) return rc;
  if (!cv) return ctx->fail(CFX_E_ARG, "null cv");
  BlockView &V = ctx->views[blk];
  CFX_TRY((int)hipMemcpy(V.cv, cv, sizeof(double) * ctx->nv * V.np, hipMemcpyHostToDevice));
  return 0;
}

int cfx_download(cfx_ctx *ctx, int blk, int what, double *dst) {
  if (int rc = check_blk(ctx, blk)) return rc;
  if (!dst) return ctx->fail(CFX_E_ARG, "null destination");
  BlockView &V = ctx->views[blk];
  CFX_TRY((int)hipStreamSynchronize(ctx->stream));
  const size_t np = (size_t)V.np, ni = (size_t)V.ni;
  const double *src = nullptr;
  size_t n = 0;
  if (V.mixed && (what == CFX_PROPS || what == CFX_DQ)) {  // FP32 arrays, returned as double
    const float *s32 = what == CFX_PROPS ? V.props32 : V.dq32;
    const size_t n32 = what == CFX_PROPS ? (4 + ctx->ns) * np : ctx->nv * ni;
    std::vector<float> tmp(n32);
    CFX_TRY(ctx->to_host.to_host(tmp.data(), s32, sizeof(float) * n32, ctx->stream));
    for (size_t i = 0; i < n32; ++i) dst[i] = tmp[i];
    return 0;
  }
  if (V.mixed && what == CFX_YK) {  // the mixed path keeps Y only as rho*Y / rho
    std::vector<double> cv(ctx->nv * np);
    CFX_TRY(ctx->to_host.to_host(cv.data(), V.cv, sizeof(double) * cv.size(), ctx->stream));
    for (size_t p = 0; p < np; ++p) {
      const double ir = 1.0 / cv[p];
      for (int l = 0; l < ctx->ns; ++l) dst[l * np + p] = cv[(5 + l) * np + p] * ir;
    }
    return 0;
  }
  switch (what) {
    case CFX_CV: src = V.cv, n = ctx->nv * np; break;
    case CFX_BV: src = V.bv, n = 6 * np; break;
    case CFX_YK: src = V.yk, n = ctx->ns * np; break;
    case CFX_PROPS: src = V.props, n = (4 + ctx->ns) * np; break;
    case CFX_DQ: src = V.dq, n = ctx->nv * ni; break;
    case CFX_DTLOCAL: src = V.dt_local, n = ni; break;
    case CFX_METRIC:
      CFX_TRY(ctx->to_host.to_host(dst, V.metric, sizeof(double) * 9 * np, ctx->stream));
      CFX_TRY((int)hipMemcpy(dst + 9 * np, V.jac, sizeof(double) * np, hipMemcpyDeviceToHost));
      return 0;
    case CFX_COORD: {
      CFX_TRY(host_coords(ctx, blk));
      const HostBlock &B = ctx->hb[blk];
      for (int c = 0; c < 3; ++c)
        for (int k = -kNgg; k < B.mz + kNgg; ++k)
          for (int j = -kNgg; j < B.my + kNgg; ++j)
            for (int i = -kNgg; i < B.mx + kNgg; ++i) dst[c * np + B.pidx(i, j, k)] = B.xyz[c][B.gidx(i, j, k)];
      return 0;
    }
    default: return ctx->fail(CFX_E_ARG, "unknown download selector");
  }
  if (n) CFX_TRY(ctx->to_host.to_host(dst, src, sizeof(double) * n, ctx->stream));
  return 0;
}

int cfx_init_conservative(cfx_ctx *ctx) {
  if (!ctx) return CFX_E_ARG;
  const KernelSet64 &k = g_kernels64[ctx->ns];
  CFX_TRY(per_batch(ctx, ctx->t_pad, [&](const Batch &b) { return k.cv_from_bv(b, ctx->sp_dev, ctx->S, ctx->stream); }));
  if (int rc = do_ghosts(ctx, false)) return rc;
  if (int rc = do_props(ctx)) return rc;
  return 0;
}

int cfx_store_last_step(cfx_ctx *ctx) { return ctx ? do_store_last(ctx) : CFX_E_ARG; }

int cfx_rhs(cfx_ctx *ctx, int blk) {
  if (!ctx) return CFX_E_ARG;
  if (blk >= (int)ctx->views.size()) return ctx->fail(CFX_E_ARG, "block index out of range");
  return do_rhs(ctx, blk);
}

int cfx_time_step(cfx_ctx *ctx, int global, double *dt_out) {
  if (!ctx) return CFX_E_ARG;
  if (int rc = do_dt(ctx, global ? 1 : 0, 1)) return rc;
  if (dt_out) return cfx_get_dt(ctx, dt_out);
  return 0;
}

int cfx_update(cfx_ctx *ctx, int stage) {
  if (!ctx) return CFX_E_ARG;
  if (stage < 0 || stage > 2 || (ctx->rk == 1 && stage != 0)) return ctx->fail(CFX_E_ARG, "bad stage");
  return do_update(ctx, stage);
}

int cfx_lusgs(cfx_ctx *ctx) {
  if (!ctx) return CFX_E_ARG;
  if (!ctx->lusgs) return ctx->fail(CFX_E_ARG, "cfx_lusgs needs cfx_params.lusgs = 1");
  return do_lusgs(ctx);
}

int cfx_apply_bc(cfx_ctx *ctx) { return ctx ? do_bc(ctx) : CFX_E_ARG; }
int cfx_exchange(cfx_ctx *ctx) { return ctx ? do_exchange(ctx) : CFX_E_ARG; }
int cfx_eliminate_k_gradient(cfx_ctx *ctx) { return ctx ? do_elim(ctx) : CFX_E_ARG; }
int cfx_update_properties(cfx_ctx *ctx) { return ctx ? do_props(ctx) : CFX_E_ARG; }

int cfx_residual(cfx_ctx *ctx, double res[4]) {
  if (!ctx || !res) return CFX_E_ARG;
  CFX_TRY(per_batch(ctx, ctx->t_res, [&](const Batch &b) { return launch_residual_partial(b, ctx->d_partial, ctx->stream); }));
  CFX_TRY(launch_residual_final(ctx->d_partial, ctx->n_partial, ctx->d_res, ctx->stream));
  double h[4];
  CFX_TRY((int)hipMemcpyAsync(h, ctx->d_res, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
  CFX_TRY((int)hipStreamSynchronize(ctx->stream));
  for (int l = 0; l < 4; ++l) res[l] = std::sqrt(h[l] / (double)ctx->n_grid_total);
  return 0;
}

int cfx_step(cfx_ctx *ctx, int n_steps) {
  if (!ctx || n_steps < 0) return CFX_E_ARG;
  return run_steps(ctx, n_steps);
}

int cfx_get_dt(cfx_ctx *ctx, double *dt) {
  if (!ctx || !dt) return CFX_E_ARG;
  CFX_TRY((int)hipMemcpyAsync(dt, ctx->d_dt, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  CFX_TRY((int)hipStreamSynchronize(ctx->stream));
  return 0;
}

int cfx_set_dt(cfx_ctx *ctx, double dt) {
  if (!ctx) return CFX_E_ARG;
  CFX_TRY((int)hipStreamSynchronize(ctx->stream));
  CFX_TRY((int)hipMemcpy(ctx->d_dt, &dt, sizeof(double), hipMemcpyHostToDevice));
  return 0;
}

int cfx_check(cfx_ctx *ctx, long long *n_newton_fail) {
  if (!ctx) return CFX_E_ARG;
  CFX_TRY((int)hipStreamSynchronize(ctx->stream));
  int flags = 0;
  unsigned long long nf = 0;
  CFX_TRY((int)hipMemcpy(&flags, ctx->d_flags, sizeof(int), hipMemcpyDeviceToHost));
  CFX_TRY((int)hipMemcpy(&nf, ctx->d_newton, sizeof(nf), hipMemcpyDeviceToHost));
  if (n_newton_fail) *n_newton_fail = (long long)nf;
  if (flags & 2) return ctx->fail((int)hipErrorLaunchTimeOut, "an LU-SGS sweep gave up waiting for a patch");
  if (flags) return ctx->fail(CFX_E_NONFINITE, "non-finite or non-positive rho/T/p in the update");
  if (nf) return ctx->fail(CFX_E_NEWTON, std::to_string(nf) + " Newton temperature inversions did not converge");
  return 0;
}

int cfx_sync(cfx_ctx *ctx) {
  if (!ctx) return CFX_E_ARG;
  CFX_TRY((int)hipStreamSynchronize(ctx->stream));
  return 0;
}

int cfx_time_steps(cfx_ctx *ctx, int n_steps, double *ms_total) {
  if (!ctx || n_steps < 0) return CFX_E_ARG;
  hipEvent_t a, b;
  (void)hipEventCreate(&a);
  (void)hipEventCreate(&b);
  (void)hipEventRecord(a, ctx->stream);
  int rc = cfx_step(ctx, n_steps);
  (void)hipEventRecord(b, ctx->stream);
  (void)hipEventSynchronize(b);
  float ms = 0;
  (void)hipEventElapsedTime(&ms, a, b);
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  if (ms_total) *ms_total = ms;
  if (rc) return rc;
  if (ctx->profiling) {
    for (auto &t : ctx->timed) {
      float m = 0;
      (void)hipEventElapsedTime(&m, t.a, t.b);
      ctx->class_ms[t.cls] += m;
      ctx->class_n[t.cls] += 1;
      ctx->event_pool.push_back(t.a);
      ctx->event_pool.push_back(t.b);
    }
    ctx->timed.clear();
  }
  return 0;
}

int cfx_set_rhs_variant(cfx_ctx *ctx, int variant) {
  if (!ctx) return CFX_E_ARG;
  if (variant < 0 || variant >= rhs_variants(ctx->dim)) return ctx->fail(CFX_E_ARG, "rhs variant out of range");
  CFX_TRY((int)hipStreamSynchronize(ctx->stream));
  for (int d = 0; d < 3; ++d) ctx->rhs_var[d] = variant, ctx->rhs_persist[d] = 0;
  ctx->drop_graph();
  return 0;
}

int cfx_rhs_variants(cfx_ctx *ctx) { return ctx ? rhs_variants(ctx->dim) : CFX_E_ARG; }

int cfx_set_rhs_tiles(cfx_ctx *ctx, const int variant[3], const int persist[3]) {
  if (!ctx || !variant || !persist) return CFX_E_ARG;
  for (int d = 0; d < ctx->dim; ++d)
    if (variant[d] < 0 || variant[d] >= rhs_variants(ctx->dim) || persist[d] < 0 || persist[d] > 64)
      return ctx->fail(CFX_E_ARG, "rhs tile choice out of range");
  CFX_TRY((int)hipStreamSynchronize(ctx->stream));
  for (int d = 0; d < ctx->dim; ++d) ctx->rhs_var[d] = variant[d], ctx->rhs_persist[d] = persist[d];
  ctx->drop_graph();
  return 0;
}

int cfx_get_rhs_tiles(cfx_ctx *ctx, int variant[3], int persist[3]) {
  if (!ctx || !variant || !persist) return CFX_E_ARG;
  for (int d = 0; d < 3; ++d) variant[d] = ctx->rhs_var[d], persist[d] = ctx->rhs_persist[d];
  return 0;
}

// Times every variant on this context's blocks (reps launches each, after one
// warm-up launch) and keeps the fastest: in 2-D every tile shape, in 3-D every
// chunk length of the march; the choice is the last direction's.  What is timed is
// what a step runs: where the later stages of RK3 work on the plane alone (see
// do_step), one RHS with the differences along k and two without.  dq holds no
// result afterwards; the next RHS rewrites it.
int cfx_autotune(cfx_ctx *ctx, int reps, double *best_ms) {
  if (!ctx || reps <= 0) return CFX_E_ARG;
  const bool prof = ctx->profiling;
  ctx->profiling = false;
  hipEvent_t a, b;
  (void)hipEventCreate(&a);
  (void)hipEventCreate(&b);
  int rc = 0;
  if (best_ms)
    for (int d = 0; d < ctx->dim; ++d) best_ms[d] = 0;
  const int d = ctx->dim - 1, n = stages_on_plane(ctx) ? 3 : 1;
  double best = 1e30;
  int bv = 0;
  auto evaluate = [&] {
    for (int s = 0; s < n; ++s)
      if (int e = do_rhs(ctx, -1, /*planar=*/s > 0)) return e;
    return 0;
  };
  for (int v = 0; v < rhs_variants(ctx->dim) && !rc; ++v) {
    ctx->rhs_var[d] = v;
    if ((rc = evaluate())) break;
    (void)hipEventRecord(a, ctx->stream);
    for (int r = 0; r < reps && !rc; ++r) rc = evaluate();
    (void)hipEventRecord(b, ctx->stream);
    (void)hipEventSynchronize(b);
    float ms = 0;
    (void)hipEventElapsedTime(&ms, a, b);
    const double each = ms / ((double)reps * n);
    if (each < best) best = each, bv = v;
  }
  ctx->rhs_var[d] = bv;
  if (best_ms) best_ms[d] = best;
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  ctx->profiling = prof;
  ctx->drop_graph();
  if (rc) return ctx->fail(rc, "autotune launch");
  return (int)hipStreamSynchronize(ctx->stream);
}

int cfx_set_execution(cfx_ctx *ctx, int batched, int graph) {
  if (!ctx) return CFX_E_ARG;
  CFX_TRY((int)hipStreamSynchronize(ctx->stream));
  ctx->batched = batched != 0;
  ctx->use_graph = graph != 0;
  ctx->drop_graph();
  return 0;
}

int cfx_schedule_info(cfx_ctx *ctx, int *n_ops, int *n_levels) {
  if (!ctx) return CFX_E_ARG;
  if (n_ops) *n_ops = (int)ctx->ops_step.size();
  if (n_levels)
    *n_levels = ctx->ex_split ? ctx->sched_bc_step.levels() + ctx->sched_mid.levels() + 1 : ctx->sched_all_step.levels();
  return 0;
}

int cfx_kernel_times(cfx_ctx *ctx, int cls, double *ms, long long *launches) {
  if (!ctx || cls < 0 || cls >= K_NCLASS) return CFX_E_ARG;
  if (ms) *ms = ctx->class_ms[cls];
  if (launches) *launches = ctx->class_n[cls];
  return 0;
}

int cfx_set_profiling(cfx_ctx *ctx, int on) {
  if (!ctx) return CFX_E_ARG;
  ctx->profiling = on != 0;
  for (int c = 0; c < K_NCLASS; ++c) ctx->class_ms[c] = 0, ctx->class_n[c] = 0;
  return 0;
}

}  // extern "C"
