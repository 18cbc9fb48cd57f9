// wx_surrogate.hip -- training and evaluation kernels of the cooling
// surrogate (the network of wx_mlp.h), and the exact coolingh update on a
// list of states that produces its training pairs.
//
//   k_sur_pack     FP32 parameters -> bf16 operand copies
//   k_sur_altab    al(T, x_HII) = ALOSS/n^2 table from the exact loss function
//   k_sur_feat     raw surrogate features of a list of states
//   k_sur_infer    forward pass of a batch (standardised in and out)
//   k_sur_packt    transposed bf16 copies for the backward pass
//   k_sur_grad     forward + backward of a batch, mean squared error; every
//                  workgroup keeps its gradient in registers and writes it
//                  once to a row of its own
//   k_sur_sum      the sum of the rows: the gradient, or (training) one
//                  bias-corrected Adam step of the FP32 parameters and their
//                  bf16 copies
//   k_cool_pairs   src/coolingh.f90:171-259 on (n, T, y0, dt) states
#include <hip/hip_runtime.h>

#include "wx_mlp.h"

namespace wx {

__global__ __launch_bounds__(256) void k_sur_pack(SurDev *__restrict__ M) {
  const float *th = M->theta;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < 64 * 64; t += gridDim.x * blockDim.x) {
    M->w2[t] = f2bf(th[SUR_W2 + t]);
    M->w3[t] = f2bf(th[SUR_W3 + t]);
    if (t < 64 * 16) {
      const int o = t / 16, i = t % 16;
      M->w1[t] = i < 4 ? f2bf(th[SUR_W1 + o * 4 + i]) : (uint16_t)0;
      const int o4 = t / 64, i4 = t % 64;
      M->w4[t] = o4 < 2 ? f2bf(th[SUR_W4 + o4 * 64 + i4]) : (uint16_t)0;
    }
  }
}

__global__ __launch_bounds__(256) void k_sur_altab(SurDev *__restrict__ M) {
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < SUR_NT * SUR_NX; t += gridDim.x * blockDim.x) {
    const int it = t / SUR_NX, ix = t % SUR_NX;
    const double T = pow(10.0, (double)SUR_TLO + (double)SUR_DT * it);
    const double rr = pow(10.0, -4.0 + 8.0 * (double)ix / (double)(SUR_NX - 1));
    const double x = dmin(dmax((rr * (1.0 + 1e-4) - 1e-4) / (1.0 + rr), 0.0), 1.0);
    const double y = 1.0 - x;
    // aloss(x1 = old neutral fraction, den, dh0 = new neutral density, T) at
    // n = 1 and an unchanged fraction
    M->altab[t] = (float)log10(dmax(aloss(y, 1.0, y, T), 1e-300));
  }
}

__global__ __launch_bounds__(256) void k_sur_feat(const SurDev *__restrict__ M, const double *__restrict__ in,
                                                  int64_t n, float *__restrict__ f, float *__restrict__ cedt) {
  for (int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; s < n; s += (int64_t)gridDim.x * blockDim.x) {
    float ff[4], ce;
    const bool inh = sur_features(M, in[4 * s], in[4 * s + 1], in[4 * s + 2], in[4 * s + 3], ff, ce);
    (void)inh;
#pragma unroll
    for (int k = 0; k < 4; ++k) f[4 * s + k] = ff[k];
    cedt[s] = ce;
  }
}

// Standardised inputs x[n][4] -> standardised outputs y[n][2]; a wave takes
// G groups of 16 samples at a time.
template <int G>
__global__ __launch_bounds__(256) void k_sur_infer(const SurDev *__restrict__ M, const float *__restrict__ x,
                                                   int64_t n, float *__restrict__ y) {
  const int l = threadIdx.x & 63, r = l & 15, q = l >> 4;
  const int64_t nset = (n + 16 * G - 1) / (16 * G);
  for (int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); b < nset; b += (int64_t)gridDim.x * 4) {
    bf16x4 xb[G];
    f32x4 yt[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int64_t s = 16 * (G * b + g) + r;
      xb[g] = bf16x4{0, 0, 0, 0};
      if (q == 0 && s < n) xb[g] = pack4(x[4 * s], x[4 * s + 1], x[4 * s + 2], x[4 * s + 3]);
    }
    mlp_fwd16<G>(M, xb, yt);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int64_t s = 16 * (G * b + g) + r;
      if (q == 0 && s < n) {
        y[2 * s] = yt[g][0];
        y[2 * s + 1] = yt[g][1];
      }
    }
  }
}

__global__ __launch_bounds__(256) void k_sur_packt(const SurDev *__restrict__ M, SurTrain *__restrict__ W) {
  const float *th = M->theta;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < 64 * 64; t += gridDim.x * blockDim.x) {
    const int o = t / 64, i = t % 64;
    W->w2t[i * 64 + o] = f2bf(th[SUR_W2 + t]);
    W->w3t[i * 64 + o] = f2bf(th[SUR_W3 + t]);
    if (t < 64 * 16) W->w4t[t] = t % 16 < 2 ? f2bf(th[SUR_W4 + (t % 16) * 64 + t / 16]) : (uint16_t)0;
  }
}

// Sum over the 16 lanes of a row, valid in the row's last lane.
__device__ __forceinline__ float row_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xf, 0xf, true));   // row_shr:1
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x112, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x114, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x118, 0xf, 0xf, true));
  return v;
}

// What a workgroup of k_sur_grad shares: the activations that enter each
// layer and the deltas that leave it, [feature][sample] of its 64 samples in
// bf16, rows of 68 so that the 16 rows of an operand fall on different banks.
constexpr int kSurPitch = 68;
struct SurGradLds {
  uint16_t x[16 * kSurPitch], a[3][64 * kSurPitch];
  uint16_t d4[16 * kSurPitch], d[3][64 * kSurPitch];
  float db[4][3][64], db4[4][2], loss[4];
};

// Gradient of the mean over a batch of sum_j w_j (y_j - t_j)^2.  Sample k of
// the batch (0 <= k < nb <= nd) is data row (off + k) mod nd.  A workgroup
// takes 64 samples at a time: each wave runs 16 of them forward and back in
// registers (a layer's D tile is the next product's B operand in both
// directions) and leaves the activations and deltas in LDS; then the waves
// share the weight gradients dW = d a^T by output rows, 64 samples deep,
// accumulated in registers over the workgroup's batches of 64.  Bias
// gradients are FP32 sums of the unrounded deltas.
// The batch of 16 384 is one pass of 256 workgroups.  With the weight
// gradients added to LDS by atomics (16 samples per product) and from there
// to memory by atomics of all workgroups on the same 8 770 words it took
// 89 us, 103 us a training step with the clearing, Adam and packing launches;
// with a row per workgroup 19 us, and 24 us a step with the sum, Adam and
// packing in one launch.  What is left is one wave per SIMD running a chain of
// products, exponentials and LDS stores.
__global__ __launch_bounds__(256, 1) void k_sur_grad(const SurDev *__restrict__ M, const SurTrain *__restrict__ W,
                                                     const float *__restrict__ x, const float *__restrict__ t,
                                                     int64_t off, int64_t nb, int64_t nd, float w0, float w1,
                                                     float *__restrict__ part, float *__restrict__ lpart) {
  __shared__ __align__(16) SurGradLds S;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, r = l & 15, q = l >> 4;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // operands: the weights and their transposes
  bf16x4 W1[4], W2[4][4], W3[4][4], W4[4], T2[4][4], T3[4][4], T4[4];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    W1[mt] = ld4(M->w1 + (16 * mt + r) * 16 + 4 * q);
    W4[mt] = ld4(M->w4 + r * 64 + 16 * mt + 4 * q);
    T4[mt] = ld4(W->w4t + (16 * mt + r) * 16 + 4 * q);
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      const int at = (16 * mt + r) * 64 + 16 * kt + 4 * q;
      W2[mt][kt] = ld4(M->w2 + at);
      W3[mt][kt] = ld4(M->w3 + at);
      T2[mt][kt] = ld4(W->w2t + at);
      T3[mt][kt] = ld4(W->w3t + at);
    }
  }
  f32x4 bias[3][4];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    bias[0][mt] = *reinterpret_cast<const f32x4 *>(M->theta + SUR_B1 + 16 * mt + 4 * q);
    bias[1][mt] = *reinterpret_cast<const f32x4 *>(M->theta + SUR_B2 + 16 * mt + 4 * q);
    bias[2][mt] = *reinterpret_cast<const f32x4 *>(M->theta + SUR_B3 + 16 * mt + 4 * q);
  }
  const float b40 = M->theta[SUR_B4], b41 = M->theta[SUR_B4 + 1];
  f32x4 g1 = zero, g4 = zero, g2[4] = {zero, zero, zero, zero}, g3[4] = {zero, zero, zero, zero};
  f32x4 db[3][4] = {{zero, zero, zero, zero}, {zero, zero, zero, zero}, {zero, zero, zero, zero}};
  float db40 = 0.f, db41 = 0.f, lsum = 0.f;
  const float inv = 1.f / (float)nb;
  const int col = 16 * w + r;   // this lane's sample of the 64
  for (int64_t base = (int64_t)blockIdx.x * 64; base < nb; base += (int64_t)gridDim.x * 64) {
    const int64_t k = base + col;
    const bool valid = k < nb;
    const int64_t kk = off + (valid ? k : 0);
    const int64_t s = kk < nd ? kk : kk - nd;
    bf16x4 xb = {0, 0, 0, 0};
    float t0 = 0.f, t1 = 0.f;
    if (q == 0 && valid) {
      xb = pack4(x[4 * s], x[4 * s + 1], x[4 * s + 2], x[4 * s + 3]);
      t0 = t[2 * s];
      t1 = t[2 * s + 1];
    }
    // a 64x64 product: the four output tiles side by side, so that each matrix
    // instruction's successor does not wait for it
    auto product = [&](const bf16x4(*A)[4], const bf16x4 *B, f32x4 *out) __attribute__((always_inline)) {
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) out[mt] = zero;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) out[mt] = mfma16(A[mt][kt], B[kt], out[mt]);
    };
    f32x4 acc[4];
    // forward; z and the sigmoid kept for the backward pass
    f32x4 z[3][4], sg[3][4];
    bf16x4 a[4], an[4];
    auto activate = [&](int L, int mt, f32x4 acc) __attribute__((always_inline)) {
      f32x4 h;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        z[L][mt][e] = acc[e] + bias[L][mt][e];
        sg[L][mt][e] = sigm(z[L][mt][e]);
        h[e] = z[L][mt][e] * sg[L][mt][e];
      }
      an[mt] = pack4(h[0], h[1], h[2], h[3]);
#pragma unroll
      for (int e = 0; e < 4; ++e) S.a[L][(16 * mt + 4 * q + e) * kSurPitch + col] = (uint16_t)an[mt][e];
    };
#pragma unroll
    for (int e = 0; e < 4; ++e) S.x[(4 * q + e) * kSurPitch + col] = (uint16_t)xb[e];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) activate(0, mt, mfma16(W1[mt], xb, zero));
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) a[mt] = an[mt];
    product(W2, a, acc);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) activate(1, mt, acc[mt]);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) a[mt] = an[mt];
    product(W3, a, acc);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) activate(2, mt, acc[mt]);
    f32x4 y = zero;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) y = mfma16(W4[kt], an[kt], y);
    // output deltas: rows 0, 1 of the tile (lanes q == 0)
    f32x4 d4 = zero;
    if (q == 0 && valid) {
      const float e0 = y[0] + b40 - t0, e1 = y[1] + b41 - t1;
      d4[0] = 2.f * w0 * e0 * inv;
      d4[1] = 2.f * w1 * e1 * inv;
      lsum += (w0 * e0 * e0 + w1 * e1 * e1) * inv;
      db40 += d4[0];
      db41 += d4[1];
    }
    const bf16x4 b4 = pack4(d4[0], d4[1], d4[2], d4[3]);
#pragma unroll
    for (int e = 0; e < 4; ++e) S.d4[(4 * q + e) * kSurPitch + col] = (uint16_t)b4[e];
    // back through the layers: da = W^T d, d = da * silu'(z)
    bf16x4 bd[4];
    auto delta = [&](int L, int mt, f32x4 da, bf16x4 *out) __attribute__((always_inline)) {
      f32x4 d;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float sv = sg[L][mt][e];
        d[e] = da[e] * (sv * (1.f + z[L][mt][e] * (1.f - sv)));
        db[L][mt][e] += d[e];
      }
      out[mt] = pack4(d[0], d[1], d[2], d[3]);
#pragma unroll
      for (int e = 0; e < 4; ++e) S.d[L][(16 * mt + 4 * q + e) * kSurPitch + col] = (uint16_t)out[mt][e];
    };
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) delta(2, mt, mfma16(T4[mt], b4, zero), bd);
    bf16x4 be[4];
    product(T3, bd, acc);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) delta(1, mt, acc[mt], be);
    product(T2, be, acc);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) delta(0, mt, acc[mt], bd);
    __syncthreads();
    // dW[o][k] = sum over the samples of d[o][n] a[k][n]: wave w takes output
    // rows 16 w .. 16 w + 15 (of layer 4, whose rows are one tile, inputs
    // 16 w .. 16 w + 15)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int n = 16 * ks + 4 * q;
      const bf16x4 d3 = ld4(S.d[2] + (16 * w + r) * kSurPitch + n), d2 = ld4(S.d[1] + (16 * w + r) * kSurPitch + n);
      g1 = mfma16(ld4(S.d[0] + (16 * w + r) * kSurPitch + n), ld4(S.x + r * kSurPitch + n), g1);
      g4 = mfma16(ld4(S.d4 + r * kSurPitch + n), ld4(S.a[2] + (16 * w + r) * kSurPitch + n), g4);
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        g3[nt] = mfma16(d3, ld4(S.a[1] + (16 * nt + r) * kSurPitch + n), g3[nt]);
        g2[nt] = mfma16(d2, ld4(S.a[0] + (16 * nt + r) * kSurPitch + n), g2[nt]);
      }
    }
    __syncthreads();   // the next 64 samples reuse the tiles
  }
  float *P = part + (size_t)blockIdx.x * SUR_ROW;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int o = 16 * w + 4 * q + e;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      P[SUR_W2 + o * 64 + 16 * nt + r] = g2[nt][e];
      P[SUR_W3 + o * 64 + 16 * nt + r] = g3[nt][e];
    }
    if (r < 4) P[SUR_W1 + o * 4 + r] = g1[e];
    if (q == 0 && e < 2) P[SUR_W4 + e * 64 + 16 * w + r] = g4[e];
  }
#pragma unroll
  for (int L = 0; L < 3; ++L)
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = row_sum(db[L][mt][e]);
        if (r == 15) S.db[w][L][16 * mt + 4 * q + e] = v;
      }
  const float v0 = row_sum(db40), v1 = row_sum(db41), v2 = row_sum(lsum);
  if (l == 15) {
    S.db4[w][0] = v0;
    S.db4[w][1] = v1;
    S.loss[w] = v2;
  }
  __syncthreads();
  if (tid < 192) {
    const int L = tid / 64, f = tid % 64;
    P[(L == 0 ? SUR_B1 : L == 1 ? SUR_B2 : SUR_B3) + f] = ((S.db[0][L][f] + S.db[1][L][f]) + S.db[2][L][f]) + S.db[3][L][f];
  } else if (tid < 194) {
    const int e = tid - 192;
    P[SUR_B4 + e] = ((S.db4[0][e] + S.db4[1][e]) + S.db4[2][e]) + S.db4[3][e];
  } else if (tid == 194) {
    lpart[blockIdx.x] = ((S.loss[0] + S.loss[1]) + S.loss[2]) + S.loss[3];
  }
}

// Sums the rows of k_sur_grad, 32 parameters per workgroup, 8 threads each;
// ADAM: the step, and the new parameters' bf16 copies; else the sums to grad.
// loss: the sum of the rows' losses.
template <bool ADAM>
__global__ __launch_bounds__(256) void k_sur_sum(SurDev *__restrict__ M, SurTrain *__restrict__ W,
                                                 const float *__restrict__ part, const float *__restrict__ lpart,
                                                 int nrow, float *__restrict__ grad, float *__restrict__ m,
                                                 float *__restrict__ v, int step, float lr, float *__restrict__ loss) {
  __shared__ float red[8][32];
  const int c = threadIdx.x & 31, sl = threadIdx.x >> 5;
  const int i = blockIdx.x * 32 + c;
  float g = 0.f;
  if (i < SUR_NPARAM)
#pragma unroll 8
    for (int k = sl; k < nrow; k += 8) g += part[(size_t)k * SUR_ROW + i];
  red[sl][c] = g;
  __syncthreads();
  if (blockIdx.x == 0 && threadIdx.x >= 64 && threadIdx.x < 128) {
    float s = 0.f;
    for (int k = threadIdx.x - 64; k < nrow; k += 64) s += lpart[k];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (threadIdx.x == 64) *loss = s;
  }
  if (sl != 0 || i >= SUR_NPARAM) return;
  float gi = red[0][c];
#pragma unroll
  for (int k = 1; k < 8; ++k) gi += red[k][c];
  if constexpr (!ADAM) {
    grad[i] = gi;
    return;
  }
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float th = M->theta[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  M->theta[i] = th;
  const uint16_t h = f2bf(th);
  if (i >= SUR_W1 && i < SUR_B1) {
    M->w1[(i - SUR_W1) / 4 * 16 + (i - SUR_W1) % 4] = h;
  } else if (i >= SUR_W2 && i < SUR_B2) {
    const int k = i - SUR_W2;
    M->w2[k] = h;
    W->w2t[k % 64 * 64 + k / 64] = h;
  } else if (i >= SUR_W3 && i < SUR_B3) {
    const int k = i - SUR_W3;
    M->w3[k] = h;
    W->w3t[k % 64 * 64 + k / 64] = h;
  } else if (i >= SUR_W4 && i < SUR_B4) {
    const int k = i - SUR_W4;
    M->w4[k] = h;
    W->w4t[k % 64 * 16 + k / 64] = h;
  }
}

// Exact coolingh update of (n, T, y0, dt[s]) states at rest: the conserved
// state is built so that uprim recovers T (src/uprim.f90:37-41), atomic runs,
// and (T1, y1) are read back the same way.
__global__ __launch_bounds__(256) void k_cool_pairs(const wx_params *__restrict__ p, const double *__restrict__ in,
                                                    int64_t n, double *__restrict__ out) {
  for (int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; s < n; s += (int64_t)gridDim.x * blockDim.x) {
    const double nn = in[4 * s], T = in[4 * s + 1], y0 = in[4 * s + 2], dts = in[4 * s + 3];
    double uu[5] = {nn, 0., 0., p->cv * (2. * nn - y0 * nn) * T / p->Tempsc, y0 * nn};
    atomic_h<5>(p, dts, uu);
    out[2 * s] = uu[3] / p->cv * p->Tempsc / (2. * uu[0] - uu[4]);
    out[2 * s + 1] = uu[4] / uu[0];
  }
}

static inline int hip_ok() { return hipGetLastError() == hipSuccess ? WX_OK : WX_EHIP; }

static inline int grid_for(int64_t n, int per) {
  int64_t g = (n + per - 1) / per;
  if (g < 1) g = 1;
  if (g > 4096) g = 4096;
  return (int)g;
}

int launch_sur_pack(SurDev *M, hipStream_t stream) {
  hipLaunchKernelGGL(k_sur_pack, dim3(16), dim3(256), 0, stream, M);
  return hip_ok();
}

int launch_sur_altab(const wx_params *P, SurDev *M, hipStream_t stream) {
  (void)P;
  hipLaunchKernelGGL(k_sur_altab, dim3(grid_for(SUR_NT * SUR_NX, 256)), dim3(256), 0, stream, M);
  return hip_ok();
}

int launch_sur_feat(const SurDev *M, const double *in, int64_t n, float *f, float *cedt, hipStream_t stream) {
  if (n <= 0) return WX_OK;
  hipLaunchKernelGGL(k_sur_feat, dim3(grid_for(n, 256)), dim3(256), 0, stream, M, in, n, f, cedt);
  return hip_ok();
}

// Up to one group of 16 samples for each of the card's 1 024 SIMDs, a wave takes
// one: it lasts as long as its chain of four layers, which more groups lengthen.
// Above, four share each weight operand's load.  us per wx_sur_infer_noalloc
// with one / two / four groups a wave: 1 000 samples 11.5 / 12.5 / 14.4, 16 384
// 11.6 / 12.6 / 14.6, 24 576 16.0 / 12.7 / 14.7, 65 536 24.8 / 17.0 / 14.6,
// 262 144 77 / 44 / 35, 2 000 005 146 / 168 / 154.
constexpr int64_t kInferOne = 16384;

int launch_sur_infer(const SurDev *M, const float *x, int64_t n, float *y, hipStream_t stream) {
  if (n <= 0) return WX_OK;
  if (n <= kInferOne) hipLaunchKernelGGL(k_sur_infer<1>, dim3(grid_for(n, 64)), dim3(256), 0, stream, M, x, n, y);
  else hipLaunchKernelGGL(k_sur_infer<4>, dim3(grid_for(n, 256)), dim3(256), 0, stream, M, x, n, y);
  return hip_ok();
}

int launch_sur_packt(const SurDev *M, SurTrain *W, hipStream_t stream) {
  hipLaunchKernelGGL(k_sur_packt, dim3(16), dim3(256), 0, stream, M, W);
  return hip_ok();
}

int launch_sur_grad(const SurDev *M, const SurTrain *W, const float *x, const float *t, int64_t off, int64_t nb,
                    int64_t nd, float w0, float w1, float *part, float *lpart, hipStream_t stream) {
  if (nb <= 0 || nb > nd || off < 0 || off >= nd) return WX_EARG;
  hipLaunchKernelGGL(k_sur_grad, dim3(sur_rows(nb)), dim3(256), 0, stream, M, W, x, t, off, nb, nd, w0, w1, part, lpart);
  return hip_ok();
}

int launch_sur_sum(SurDev *M, const float *part, const float *lpart, int nrow, float *grad, float *loss,
                   hipStream_t stream) {
  hipLaunchKernelGGL((k_sur_sum<false>), dim3((SUR_NPARAM + 31) / 32), dim3(256), 0, stream, M, nullptr, part, lpart, nrow,
                     grad, nullptr, nullptr, 0, 0.f, loss);
  return hip_ok();
}

int launch_sur_adam(SurDev *M, SurTrain *W, const float *part, const float *lpart, int nrow, float *m, float *v,
                    int step, float lr, float *loss, hipStream_t stream) {
  hipLaunchKernelGGL((k_sur_sum<true>), dim3((SUR_NPARAM + 31) / 32), dim3(256), 0, stream, M, W, part, lpart, nrow,
                     nullptr, m, v, step, lr, loss);
  return hip_ok();
}

int launch_cool_pairs(const wx_params *P, const double *in, int64_t n, double *out, hipStream_t stream) {
  if (n <= 0) return WX_OK;
  hipLaunchKernelGGL(k_cool_pairs, dim3(grid_for(n, 256)), dim3(256), 0, stream, P, in, n, out);
  return hip_ok();
}

}  // namespace wx
