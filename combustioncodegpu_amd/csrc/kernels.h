// kernels.h — host launchers of the step kernels.  Every kernel works on a
// batch of blocks: a device table of BlockViews and a prefix table off[] of
// workgroups per block, so one launch covers any subset of the blocks (a
// single block is a batch of one).  The species-count templated launchers
// are compiled once per supported species count and precision
// (kernels_ns.hip) and register themselves in g_kernels64 / g_kernels32.
// All launchers return 0 or a hipError_t / CFX_E_* code and are asynchronous
// on the given stream.
#pragma once

#include <hip/hip_runtime.h>

#include "cfx_types.h"

namespace cfx {

// ------------------------------------------------------------ work units ---
constexpr int kTpb = 256;        // threads per workgroup of the point kernels
constexpr int kDtIter = 8;       // most points per thread of the time-step reduction
constexpr int kLastIter = 4;     // most points per thread of the last-step snapshot
constexpr int kResIter = 8;      // points per thread of the residual partials

// A batch of blocks: views[0..nb) with workgroup prefix off[0..nb] (device
// pointers, off[0] need not be 0) and total = off[nb] - off[0] workgroups.
struct Batch {
  const BlockView *views;
  const int *off;
  int nb;
  int total;
};

// --------------------------------------------------------- RHS tile shapes ---
// 3-D: one launch marches along k (rhs_march.h); a workgroup of nt threads
// owns tx x ty cells.  A variant is the number of planes a workgroup marches
// through: variant 0 as planned for the context's blocks, the others at most
// kMarchChunk[v].
struct MarchTile {
  int tx, ty, nt, wpe;
};
// 16 x 8 cells have 408 faces, 7 wavefronts, and with the one that moves data
// fill 2 waves per SIMD; the FP64 planes and fluxes of 9 species then take
// 158 KB of LDS, FP32 half of it, so that two workgroups share a CU.
constexpr MarchTile kMarch64 = {16, 8, 512, 2}, kMarch32 = {16, 8, 512, 4};
constexpr int kNVar3 = 6;
constexpr int kMarchChunk[kNVar3] = {0, 8, 16, 32, 64, 1 << 30};
// workgroups of a block of m[3] points marched in chunks of at most `chunk` planes
inline int march_groups(const int m[3], const MarchTile &t, int chunk) {
  const int parts = m[2] <= chunk ? 1 : (m[2] + chunk - 1) / chunk;
  return (m[0] + t.tx - 1) / t.tx * ((m[1] + t.ty - 1) / t.ty) * parts;
}
// big: a block's nine metric fields pass 4 GiB
using MarchFn = int (*)(const Batch &b, int chunk, int big, const SpeciesDev *sp, const SchemeDev &S, hipStream_t st);
using OccFn = int (*)();  // resident workgroups per CU of the kernel

// 2-D: one launch over tiles of tx x ty cells (rhs_plane.h); variant v is
// shape v.
struct PlaneTile {
  int tx, ty;
};
constexpr int kNVar2 = 2;
constexpr PlaneTile kTiles2[kNVar2] = {{16, 15}, {32, 7}};
inline int plane_groups(const int m[3], const PlaneTile &t) {
  return (m[0] + t.tx - 1) / t.tx * ((m[1] + t.ty - 1) / t.ty);
}
// planar: the ghost planes along k equal the plane, and are not read
using PlaneFn = int (*)(const Batch &b, int planar, const SpeciesDev *sp, const SchemeDev &S, hipStream_t st);

// Properties over the padded range; or of the plane k = 0 alone with the copies
// of the ring near the faces to the ghost planes along k; or of all planes, with
// the copies of the whole plane.
constexpr int kPropsPadded = 0, kPropsRing = 1, kPropsPlanes = 2;

inline int rhs_variants(int dim) { return dim == 3 ? kNVar3 : kNVar2; }

struct KernelSet64 {
  int present;
  // mode: kPropsPadded, or (2-D, a batch of the blocks' planes) kPropsRing, kPropsPlanes
  int (*props)(const Batch &b, int mode, const SpeciesDev *sp, const SchemeDev &S, hipStream_t st);
  int (*cv_from_bv)(const Batch &b, const SpeciesDev *sp, const SchemeDev &S, hipStream_t st);
  int (*update)(const Batch &b, const SpeciesDev *sp, const SchemeDev &S, int mixed, int stage, const double *dt,
                int *flags, unsigned long long *newton_fail, hipStream_t st);
  // ops[0..nops) with workgroup prefix off[0..nops], total workgroups
  int (*face_ops)(const BlockView *views, const FaceOp *ops, const int *off, int nops, int total,
                  const SpeciesDev *sp, const SchemeDev &S, const InflowDev *inflow, hipStream_t st);
  // the same for ops that only copy and average (outflow, exchange)
  int (*copy_ops)(const BlockView *views, const FaceOp *ops, const int *off, int nops, int total, int mixed,
                  hipStream_t st);
  PlaneFn plane[kNVar2];
  MarchFn march;
  OccFn march_occ;
  // surrogate training set: n samples of (T, log p, Y) and log(mu, kappa,
  // rho*D) from the FP64 transport; lim = t_lo, t_hi, log p_lo, log p_hi
  int (*mlp_samples)(const SpeciesDev *sp, const SchemeDev &S, long long n, unsigned long long seed,
                     const double lim[4], double alpha, double *x, double *y, hipStream_t st);
  // LU-SGS: the diagonal and neighbour coefficients over the interior (point
  // batch); what a sweep expects of its hand-over and of ticket[0..1], its ticket
  // counter and abort word (point batch); and the forward (fwd = 1) or backward
  // sweep of n patches
  int (*lusgs_coef)(const Batch &b, const SchemeDev &S, hipStream_t st);
  int (*lusgs_reset)(const Batch &b, int *ticket, hipStream_t st);
  int (*lusgs_sweep)(const BlockView *views, const LuPatch *order, int n, int *ticket, const SchemeDev &S, int fwd,
                     int *flags, hipStream_t st);
};

struct MlpDev;
struct KernelSet32 {
  int present;
  int (*props)(const Batch &b, int mode, const SpeciesDev *sp, const SchemeDev &S, hipStream_t st);
  // properties with the surrogate transport (mixed precision)
  int (*props_mlp)(const Batch &b, const SpeciesDev *sp, const SchemeDev &S, const MlpDev *mlp, const void *ops,
                   const float *bias, unsigned long long *counters, hipStream_t st);
  PlaneFn plane[kNVar2];
  MarchFn march;
  OccFn march_occ;
};

extern KernelSet64 g_kernels64[kMaxSp + 1];
extern KernelSet32 g_kernels32[kMaxSp + 1];

// ------------------------------------------------ species-independent ones ---
int launch_dt_reset(unsigned long long *dt_bits, hipStream_t st);
// iter: points per thread (as in the batch's prefix)
int launch_dt(const Batch &b, const SchemeDev &S, int ns, int iter, int store_local, unsigned long long *dt_bits,
              hipStream_t st);
// reset (may be null): also resets the target of the reduction to follow
int launch_store_last(const Batch &b, int iter, unsigned long long *reset, hipStream_t st);
// metrics and Jacobian of one block from its coordinates over ngg+1 ghost
// layers (3 planes of (mx+2ngg+2)(my+2ngg+2)(mz+2ngg+2)); FP32 copies when
// metric32 is non-null; *bad counts points with a non-positive Jacobian
int launch_metrics(const double *xyz, int mx, int my, int mz, double *metric, double *jac, float *metric32,
                   float *jac32, int *bad, hipStream_t st);
// The ghost grid of Mesh::init_ghost_grid on the device, over the (ngg+1)-
// layer coordinate array of a block (3 planes of (mx+2ngg+2)(my+2ngg+2)(mz+2ngg+2)):
// raw (3 x mx*my*mz, i fastest) scattered into it; the mirror extrapolation
// (and the 2-D z layers); one inter-block copy; the edges and corners.
struct GhostCopy;
int launch_coord_scatter(const double *raw, int mx, int my, int mz, double *xyz, hipStream_t st);
int launch_ghost_extrapolate(double *xyz, int mx, int my, int mz, int dim, hipStream_t st);
int launch_ghost_inner(const GhostCopy &g, double *dst, int dmx, int dmy, int dmz, const double *src, int smx,
                       int smy, int smz, hipStream_t st);
int launch_ghost_corners(double *xyz, int mx, int my, int mz, hipStream_t st);
// partial sums of workgroup w go to partial[4 * (w)] with w counted from 0 of
// the full prefix, so a per-block launch and a batched one fill the same slots
int launch_residual_partial(const Batch &b, double *partial, hipStream_t st);
int launch_residual_final(const double *partial, int n, double *out, hipStream_t st);
// every component of the strips, one lane per component, the fields over the wavefronts
int launch_exchange_strips(const BlockView *views, const ExStrips &x, int ns, int mixed, hipStream_t st);
int launch_eliminate_k(const BlockView &B, int ns, hipStream_t st);

}  // namespace cfx
