// mlp_kernels.hip — training and inference kernels of the transport
// surrogate that do not depend on the species count (the network sizes are
// run-time: nin = nout = n_spec + 2 <= 16).  See mlp.h for the layout.
#include <hip/hip_runtime.h>

#include "mlp.h"
#include "mlp_kernels.h"

namespace cfx {

namespace {

constexpr int kTS = 40;  // LDS row stride (bf16) of the 32-point transposes

__device__ __forceinline__ bf16x8 x_operand(const float *__restrict__ xs, long long s, int g) {
  // slots j < 4 carry features 4g..4g+3, slots j >= 4 features 16+ (zero)
  const f32x4 v = *reinterpret_cast<const f32x4 *>(xs + s * kMlpIO + 4 * g);
  bf16x8 r;
  r[0] = (__bf16)v[0]; r[1] = (__bf16)v[1]; r[2] = (__bf16)v[2]; r[3] = (__bf16)v[3];
  r[4] = (__bf16)0.0f; r[5] = (__bf16)0.0f; r[6] = (__bf16)0.0f; r[7] = (__bf16)0.0f;
  return r;
}

__device__ __forceinline__ bf16x8 lds_operand(const __bf16 (*t)[kTS], int row, int g) {
  bf16x8 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    r[j] = t[row][4 * g + j];
    r[4 + j] = t[row][16 + 4 * g + j];
  }
  return r;
}

__device__ __forceinline__ long long sample_of(long long k, long long offset, long long mult, long long n) {
  return (long long)(((unsigned long long)(k + offset) * (unsigned long long)mult) % (unsigned long long)n);
}

// One workgroup = 32 samples, two 16-point tiles: forward, loss, backward; the
// weight and bias gradients of the 32 samples go to partial[w * P + i].
// loss = scale * sum over samples and outputs of (y - t)^2.
//
// Bound by the chain of dependent layers: a batch of 4096 samples is 128
// workgroups, and a layer is two MFMAs and the SiLU (or its derivative) of its
// results.  Wavefront (t, mb) therefore computes the 16 outputs of M-block mb of
// tile t in every layer, all its operands on their way from the start, and the
// activations pass to the next layer through LDS; the products of the weight
// gradients are shared out over all eight.  One wavefront per 32 samples, which
// did all of it in turn, took 18.8 us per batch, this form 8.0.  The values
// are the same bit for bit (each product and sum has the same operands and
// order).
constexpr int kTrainTpb = 512;
__global__ void __launch_bounds__(kTrainTpb) mlp_train_kernel(const float *__restrict__ xs,
                                                              const float *__restrict__ ts, long long n_train,
                                                              long long first, long long offset, long long mult,
                                                              const bf16x8 *__restrict__ ops,
                                                              const float *__restrict__ bias, MlpShape shp,
                                                              float scale, float *__restrict__ partial,
                                                              float *__restrict__ loss_out) {
  __shared__ __bf16 tD[208][kTS];  // dZ rows: layer 1 [0,64), 2 [64,128), 3 [128,192), output [192,208)
  __shared__ __bf16 tH[208][kTS];  // H rows: inputs [0,16), H1 [16,80), H2 [80,144), H3 [144,208)
  __shared__ bf16x4 pass[2][2][4][64];  // activations on their way to the next layer: [turn][tile][M-block][lane]
  __shared__ f32x4 dy1[64];             // y - t of tile 1, for the loss
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t = wv >> 2, mb = wv & 3;
  const int w = blockIdx.x;
  const int P = shp.count();
  const long long s = sample_of(first + 32LL * w + 16 * t + c, offset, mult, n_train);
  const bf16x8 x = x_operand(xs, s, g);
  const f32x4 tg = *reinterpret_cast<const f32x4 *>(ts + s * kMlpIO + 4 * g);
  const bf16x8 f1 = load_op(ops, kF1 + mb, lane), b4 = load_op(ops, kB4 + mb, lane);
  bf16x8 f2[2], f3[2], f4[2], b3[2], b2[2];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    f2[kb] = load_op(ops, kF2 + 2 * mb + kb, lane);
    f3[kb] = load_op(ops, kF3 + 2 * mb + kb, lane);
    f4[kb] = load_op(ops, kF4 + kb, lane);
    b3[kb] = load_op(ops, kB3 + 2 * mb + kb, lane);
    b2[kb] = load_op(ops, kB2 + 2 * mb + kb, lane);
  }
  const f32x4 bz1 = load_bias(bias, 0, mb, lane), bz2 = load_bias(bias, 1, mb, lane), bz3 = load_bias(bias, 2, mb, lane),
              by = load_bias(bias, 3, 0, lane);
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  const int col = 16 * t + c, row = 16 * mb + 4 * g;
  // four rows of the M-block to a transpose and, as B operand of the next
  // product, to the wavefronts of the tile
  int turn = 0;
  auto share = [&](const f32x4 v, __bf16(*tr)[kTS], bf16x8 *op) {
    bf16x4 h;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      h[r] = (__bf16)v[r];
      tr[row + r][col] = h[r];
    }
    pass[turn][t][mb][lane] = h;
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
      op[kb] = __builtin_shufflevector(pass[turn][t][2 * kb][lane], pass[turn][t][2 * kb + 1][lane], 0, 1, 2, 3, 4, 5, 6, 7);
    turn ^= 1;
  };
  // ---- forward
  bf16x8 op[2];
  const f32x4 z1 = mfma_bf16(f1, x, bz1);
  share(silu4(z1), tH + 16, op);
  const f32x4 z2 = mfma_bf16(f2[1], op[1], mfma_bf16(f2[0], op[0], bz2));
  share(silu4(z2), tH + 80, op);
  const f32x4 z3 = mfma_bf16(f3[1], op[1], mfma_bf16(f3[0], op[0], bz3));
  share(silu4(z3), tH + 144, op);
  const f32x4 y = mfma_bf16(f4[1], op[1], mfma_bf16(f4[0], op[0], by));
  f32x4 d, dy;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    d[r] = (4 * g + r < shp.nout) ? y[r] - tg[r] : 0.0f;
    dy[r] = 2.0f * scale * d[r];
  }
  bf16x8 dyop;
#pragma unroll
  for (int r = 0; r < 4; ++r) dyop[r] = (__bf16)dy[r], dyop[4 + r] = (__bf16)0.0f;
  if (mb == 0) {
    if (t == 1) dy1[lane] = d;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      tH[4 * g + r][col] = x[r];
      tD[192 + 4 * g + r][col] = dyop[r];
    }
  }
  // ---- backward: dH_{l-1} = W_l^T dZ_l
  auto through = [&](const f32x4 dh, const f32x4 z) {
    f32x4 dz;
#pragma unroll
    for (int r = 0; r < 4; ++r) dz[r] = dh[r] * mlp_dsilu(z[r]);
    return dz;
  };
  share(through(mfma_bf16(b4, dyop, zero), z3), tD + 128, op);
  share(through(mfma_bf16(b3[1], op[1], mfma_bf16(b3[0], op[0], zero)), z2), tD + 64, op);
  const f32x4 dz1 = through(mfma_bf16(b2[1], op[1], mfma_bf16(b2[0], op[0], zero)), z1);
#pragma unroll
  for (int r = 0; r < 4; ++r) tD[row + r][col] = (__bf16)dz1[r];
  __syncthreads();
  // ---- weight gradients dW = sum over the 32 points of dZ H^T; bias gradients
  float *__restrict__ out = partial + (long long)w * P;
  auto product = [&](int drow, int hrow, int m, int nb, int n_out, int n_in, int woff) {
    const f32x4 v = mfma_bf16(lds_operand(tD, drow + 16 * m + c, g), lds_operand(tH, hrow + 16 * nb + c, g), zero);
    const int in = 16 * nb + c;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int o = 16 * m + 4 * g + r;
      if (o < n_out && in < n_in) out[woff + o * n_in + in] = v[r];
    }
  };
  auto bias_sum = [&](int drow, int m, int n_out, int boff) {  // of the bf16 dZ of a row over the 32 points
    const int o = 16 * m + c;
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) sum += (float)tD[drow + o][4 * g + j] + (float)tD[drow + o][16 + 4 * g + j];
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (g == 0 && o < n_out) out[boff + o] = sum;
  };
  // wavefront (t, mb): columns 2t, 2t + 1 of row block mb of layers 2 and 3, and
  // one product of the first or the last layer
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    product(64, 16, mb, 2 * t + q, kMlpH, kMlpH, shp.w2());
    product(128, 80, mb, 2 * t + q, kMlpH, kMlpH, shp.w3());
  }
  if (t == 0) {
    product(0, 0, mb, 0, kMlpH, shp.nin, shp.w1());
    bias_sum(0, mb, kMlpH, shp.b1());
    bias_sum(64, mb, kMlpH, shp.b2());
  } else {
    product(192, 144, 0, mb, shp.nout, kMlpH, shp.w4());
    bias_sum(128, mb, kMlpH, shp.b3());
    if (mb == 0) bias_sum(192, 0, shp.nout, shp.b4());
  }
  if (wv == 0) {
    float lsum = 0.0f;
    const f32x4 d1 = dy1[lane];
#pragma unroll
    for (int r = 0; r < 4; ++r) lsum += d[r] * d[r];
#pragma unroll
    for (int r = 0; r < 4; ++r) lsum += d1[r] * d1[r];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o, 64);
    if (lane == 0) loss_out[w] = lsum * scale;
  }
}

// Place in the packed operands (element index) of weight (row, k) of an A
// operand with M rows and K columns, of whose blocks `blk` is the first and
// `nk` go side by side along K.
__device__ __forceinline__ int op_index(int blk, int nk, int row, int k) {
  const int kk = k & 31, g = (kk & 15) >> 2, j = (kk & 3) + (kk >= 16 ? 4 : 0);
  return ((blk + (row >> 4) * nk + (k >> 5)) * 64 + g * 16 + (row & 15)) * 8 + j;
}

// Sum of the per-workgroup gradients and an Adam step on the FP32 master
// parameters, and (ops not null) the new value's places in the training
// operands that mlp_pack_kernel lays out: the padding there stays as it is.  A
// workgroup takes 64 parameters; its four wavefronts sum quarters of the
// partials (each in increasing order, loads coalesced over the parameters) and
// the quarter sums are added in order, so the result is deterministic.
// Bound by the latency of the partials (5 MB from the caches), so 32 loads are
// in flight per lane: 3.5 us (9.8 with the loads in turn, and 3.8 for the
// operands in a launch of their own).
__global__ void __launch_bounds__(256) mlp_adam_kernel(float *__restrict__ params, float *__restrict__ m,
                                                       float *__restrict__ v, const float *__restrict__ partial,
                                                       int n_partial, int P, float lr, float b1, float b2,
                                                       float eps, float c1, float c2, float *__restrict__ grad_out,
                                                       MlpShape shp, __bf16 *__restrict__ ops,
                                                       float *__restrict__ bias) {
  __shared__ float quarter[4][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + lane;
  const int w0 = (int)((long long)n_partial * wv / 4), w1 = (int)((long long)n_partial * (wv + 1) / 4);
  float part = 0.0f;
  if (i < P) {
    int w = w0;
    for (; w + 32 <= w1; w += 32) {
      float v32[32];
#pragma unroll
      for (int q = 0; q < 32; ++q) v32[q] = partial[(long long)(w + q) * P + i];
#pragma unroll
      for (int q = 0; q < 32; ++q) part += v32[q];
    }
    for (; w < w1; ++w) part += partial[(long long)w * P + i];
  }
  quarter[wv][lane] = part;
  __syncthreads();
  if (wv != 0 || i >= P) return;
  const float gsum = ((quarter[0][lane] + quarter[1][lane]) + quarter[2][lane]) + quarter[3][lane];
  if (grad_out) grad_out[i] = gsum;
  if (lr <= 0.0f) return;
  const float mi = b1 * m[i] + (1.0f - b1) * gsum;
  const float vi = b2 * v[i] + (1.0f - b2) * gsum * gsum;
  m[i] = mi;
  v[i] = vi;
  const float p = params[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  params[i] = p;
  if (!ops) return;
  const __bf16 h = (__bf16)p;
  if (i < shp.b1()) {
    ops[op_index(kF1, 1, i / shp.nin, i % shp.nin)] = h;
  } else if (i < shp.w2()) {
    bias[i - shp.b1()] = p;
  } else if (i < shp.w4()) {  // layers 2 and 3: the weights and their transposes, or the bias
    const bool l3 = i >= shp.w3();
    const int e = i - (l3 ? shp.w3() : shp.w2()), r = e / kMlpH, k = e % kMlpH;
    if (r < kMlpH) {
      ops[op_index(l3 ? kF3 : kF2, 2, r, k)] = h;
      ops[op_index(l3 ? kB3 : kB2, 2, k, r)] = h;
    } else {
      bias[(l3 ? 2 : 1) * kMlpH + k] = p;
    }
  } else if (i < shp.b4()) {
    const int e = i - shp.w4(), r = e / kMlpH, k = e % kMlpH;
    ops[op_index(kF4, 2, r, k)] = h;
    ops[op_index(kB4, 1, k, r)] = h;
  } else {
    bias[3 * kMlpH + i - shp.b4()] = p;
  }
}

// BF16 A operands of the forward and backward products, and the biases
// padded to 64 per layer, from the FP32 master parameters.  fold: the
// inference operands, with -log2(e) on the layer-1 weights and the layer 1-3
// biases and -ln(2) on the output weights (float products, then BF16).
constexpr float kFold = -1.4426950408889634f, kUnfold = -0.69314718055994531f;

__global__ void __launch_bounds__(256) mlp_pack_kernel(const float *__restrict__ p, MlpShape shp,
                                                       __bf16 *__restrict__ ops, float *__restrict__ bias,
                                                       int fold) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < 4 * kMlpH) {
    const int layer = e / kMlpH, row = e % kMlpH;
    float b = 0.0f;
    if (layer == 0) b = p[shp.b1() + row];
    else if (layer == 1) b = p[shp.b2() + row];
    else if (layer == 2) b = p[shp.b3() + row];
    else if (row < shp.nout) b = p[shp.b4() + row];
    bias[e] = fold && layer < 3 ? b * kFold : b;
  }
  if (e >= kNBlocks * kOpBlock) return;
  const int blk = e / kOpBlock, lane = (e % kOpBlock) / 8, j = e % 8;
  const int g = lane >> 4, c = lane & 15, k = mlp_kperm(g, j);
  float val = 0.0f;
  if (blk < kF2) {  // W1, M-block blk
    const int row = 16 * blk + c;
    if (k < shp.nin) val = p[shp.w1() + row * shp.nin + k];
    if (fold) val *= kFold;
  } else if (blk < kF4) {  // W2 / W3
    const int q = blk < kF3 ? blk - kF2 : blk - kF3, mb = q / 2, kb = q % 2;
    const int w = blk < kF3 ? shp.w2() : shp.w3();
    val = p[w + (16 * mb + c) * kMlpH + 32 * kb + k];
  } else if (blk < kB4) {  // W4, K-block
    const int kb = blk - kF4;
    if (c < shp.nout) val = p[shp.w4() + c * kMlpH + 32 * kb + k];
    if (fold) val *= kUnfold;
  } else if (blk < kB3) {  // W4^T: rows = hidden units, k = outputs
    const int mb = blk - kB4;
    if (k < shp.nout) val = p[shp.w4() + k * kMlpH + 16 * mb + c];
  } else {  // W3^T / W2^T
    const int q = blk < kB2 ? blk - kB3 : blk - kB2, mb = q / 2, kb = q % 2;
    const int w = blk < kB2 ? shp.w3() : shp.w2();
    val = p[w + (32 * kb + k) * kMlpH + 16 * mb + c];
  }
  ops[e] = (__bf16)val;
}

// Normalised predictions of normalised inputs (validation), on the folded
// inference operands: n a multiple of 16 is not required; the last tile
// repeats a valid sample.
__global__ void __launch_bounds__(64) mlp_predict_kernel(const float *__restrict__ xs, long long n,
                                                         const bf16x8 *__restrict__ ops,
                                                         const float *__restrict__ bias, int nout,
                                                         float *__restrict__ ys) {
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  const long long s = (long long)blockIdx.x * 16 + c;
  const long long sv = s < n ? s : n - 1;
  const f32x4 y = mlp_infer_tile(ops, bias, x_operand(xs, sv, g));
  if (s < n)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * g + r < nout) ys[s * kMlpIO + 4 * g + r] = y[r];
}

// Per-workgroup sums of the features, their squares and (inputs) the
// cross products, for normalisation and the envelope (double).
__global__ void __launch_bounds__(256) mlp_moments_kernel(const double *__restrict__ x, long long n, int nf,
                                                          int cross, double *__restrict__ out) {
  // out per workgroup: nf sums, nf squares, nf*nf cross (if cross)
  __shared__ double red[256];
  const int nval = 2 * nf + (cross ? nf * nf : 0);
  const long long per = (n + gridDim.x - 1) / gridDim.x;
  const long long s0 = (long long)blockIdx.x * per, s1 = s0 + per < n ? s0 + per : n;
  for (int q = 0; q < nval; ++q) {
    double acc = 0.0;
    for (long long s = s0 + threadIdx.x; s < s1; s += blockDim.x) {
      const double *r = x + s * nf;
      if (q < nf) acc += r[q];
      else if (q < 2 * nf) acc += r[q - nf] * r[q - nf];
      else acc += r[(q - 2 * nf) / nf] * r[(q - 2 * nf) % nf];
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
      if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
      __syncthreads();
    }
    if (threadIdx.x == 0) out[(long long)blockIdx.x * nval + q] = red[0];
    __syncthreads();
  }
}

// x_norm = (x - mean) * inv_std into rows of 16 floats (zero padded).
__global__ void __launch_bounds__(256) mlp_normalize_kernel(const double *__restrict__ x, long long n, int nf,
                                                            const float *__restrict__ mean,
                                                            const float *__restrict__ inv_std,
                                                            float *__restrict__ xs) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n * kMlpIO) return;
  const long long s = e / kMlpIO;
  const int f = (int)(e % kMlpIO);
  xs[e] = f < nf ? (float)((x[s * nf + f] - (double)mean[f]) * (double)inv_std[f]) : 0.0f;
}

// Squared Mahalanobis distances of the training inputs (host loop before: 16 ms
// for 490,000 samples of 11 inputs while the GPU waited).  Every product and
// sum rounds by itself, as in the host's dist2, so that the quantile taken of
// them is the same value.
__global__ void __launch_bounds__(256) mlp_dist2_kernel(const float *__restrict__ xs, long long n, MlpAxes ax,
                                                        double *__restrict__ d2) {
#pragma clang fp contract(off)
  const long long s = (long long)blockIdx.x * 256 + threadIdx.x;
  if (s >= n) return;
  double x[kMlpIO];
#pragma unroll
  for (int i = 0; i < kMlpIO; ++i) x[i] = (double)xs[s * kMlpIO + i];
  double sum = 0.0;
  for (int k = 0; k < ax.n; ++k) {
    double a = 0.0;
#pragma unroll
    for (int i = 0; i < kMlpIO; ++i)
      if (i < ax.n) a += (double)ax.axis[k][i] * x[i];
    sum += (double)ax.inv_var[k] * a * a;
  }
  d2[s] = sum;
}

}  // namespace

int launch_mlp_dist2(const float *xs, long long n, const MlpAxes &ax, double *d2, hipStream_t st) {
  if (n <= 0) return 0;
  mlp_dist2_kernel<<<(int)((n + 255) / 256), 256, 0, st>>>(xs, n, ax, d2);
  return (int)hipGetLastError();
}

int launch_mlp_train(const float *xs, const float *ts, long long n_train, long long first, long long offset,
                     long long mult, int waves, const void *ops, const float *bias, const MlpShape &shp,
                     float scale, float *partial, float *loss, hipStream_t st) {
  mlp_train_kernel<<<waves, kTrainTpb, 0, st>>>(xs, ts, n_train, first, offset, mult, (const bf16x8 *)ops, bias, shp,
                                         scale, partial, loss);
  return (int)hipGetLastError();
}

int launch_mlp_adam(float *params, float *m, float *v, const float *partial, int n_partial, int P, float lr,
                    float b1, float b2, float eps, float c1, float c2, float *grad_out, const MlpShape &shp, void *ops,
                    float *bias, hipStream_t st) {
  mlp_adam_kernel<<<(P + 63) / 64, 256, 0, st>>>(params, m, v, partial, n_partial, P, lr, b1, b2, eps, c1, c2,
                                                 grad_out, shp, (__bf16 *)ops, bias);
  return (int)hipGetLastError();
}

int launch_mlp_pack(const float *params, const MlpShape &shp, void *ops, float *bias, int fold, hipStream_t st) {
  mlp_pack_kernel<<<(kNBlocks * kOpBlock + 255) / 256, 256, 0, st>>>(params, shp, (__bf16 *)ops, bias, fold);
  return (int)hipGetLastError();
}

int launch_mlp_predict(const float *xs, long long n, const void *ops, const float *bias, int nout, float *ys,
                       hipStream_t st) {
  if (n <= 0) return 0;
  mlp_predict_kernel<<<(int)((n + 15) / 16), 64, 0, st>>>(xs, n, (const bf16x8 *)ops, bias, nout, ys);
  return (int)hipGetLastError();
}

int launch_mlp_moments(const double *x, long long n, int nf, int cross, int groups, double *out, hipStream_t st) {
  mlp_moments_kernel<<<groups, 256, 0, st>>>(x, n, nf, cross, out);
  return (int)hipGetLastError();
}

int launch_mlp_normalize(const double *x, long long n, int nf, const float *mean, const float *inv_std, float *xs,
                         hipStream_t st) {
  const long long e = n * kMlpIO;
  mlp_normalize_kernel<<<(int)((e + 255) / 256), 256, 0, st>>>(x, n, nf, mean, inv_std, xs);
  return (int)hipGetLastError();
}

}  // namespace cfx
