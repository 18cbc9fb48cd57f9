// wx_mlp.h -- device code of the cooling surrogate shared by the training
// kernels (wx_surrogate.hip) and the fused cooling pass (wx_kernels.hip).
//
// Matrix-core layout (v_mfma_f32_16x16x16_bf16, one wave64):
//   A (16x16, M x K): lane l holds A[l % 16][4*(l/16) + e], e = 0..3
//   B (16x16, K x N): lane l holds B[4*(l/16) + e][l % 16]
//   D (16x16, M x N): lane l holds D[4*(l/16) + e][l % 16]
// The network is evaluated transposed, Z = W * A_prev with samples as the
// N dimension: a layer's D tile t (output features 16t .. 16t+15) is then,
// lane for lane, the B operand of K-step t of the next layer, so the
// activations never leave registers.
#pragma once
#include <hip/hip_runtime.h>

#include "wx_physics.h"
#include "wx_surrogate.h"

namespace wx {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// To bf16, round to nearest even (v_cvt_pk_bf16_f32: two values an instruction).
typedef __bf16 bf16x2h __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t f2bf_pk(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2h));
}
__device__ __forceinline__ uint16_t f2bf(float f) { return (uint16_t)f2bf_pk(f, f); }

__device__ __forceinline__ bf16x4 pack4(float a, float b, float c, float d) {
  const uint2 v = make_uint2(f2bf_pk(a, b), f2bf_pk(c, d));
  return __builtin_bit_cast(bf16x4, v);
}

__device__ __forceinline__ bf16x4 ld4(const uint16_t *p) {   // 4 consecutive bf16 (8-byte aligned)
  return __builtin_bit_cast(bf16x4, *reinterpret_cast<const uint2 *>(p));
}

__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}


// SiLU with the hardware exp2 and reciprocal (1 ulp each).
__device__ __forceinline__ float sigm(float z) { return __builtin_amdgcn_rcpf(1.f + __expf(-z)); }
__device__ __forceinline__ float silu(float z) { return z * sigm(z); }

// Forward pass of G groups of 16 samples by one wave.  x[g]: B operand of
// layer 1 (lanes 0-15 carry their sample's 4 standardised features, lanes
// 16-63 zeros).  y[g]: the D tile of layer 4 (rows 0, 1 = standardised outputs
// of sample l in lanes l < 16).  Each weight operand is loaded once, from
// cache, and used by all groups.  With the weights staged in LDS by every
// workgroup of the fill, read again for every group and kept at 47 KB of LDS
// and two waves per SIMD, and with whole waves running the exact routine for
// one cell outside, the fill took 139 us on 1 870 blocks; it takes 68.  A group
// costs 48 exponentials and reciprocals per lane, about 2 300 SIMD cycles: 35
// of the 68 us.
template <int G>
__device__ __forceinline__ void mlp_fwd16(const SurDev *__restrict__ M, const bf16x4 *x, f32x4 *y) {
  const int l = threadIdx.x & 63;
  const int r = l & 15, q = l >> 4;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  bf16x4 a[G][4], an[G][4];
  auto activate = [&](const f32x4 &acc, const f32x4 &b) __attribute__((always_inline)) {
    const f32x4 z = acc + b;
    return pack4(silu(z[0]), silu(z[1]), silu(z[2]), silu(z[3]));
  };
  auto bias = [&](int off, int mt) __attribute__((always_inline)) {
    return *reinterpret_cast<const f32x4 *>(M->theta + off + 16 * mt + 4 * q);
  };
  // layer 1: K = 4 features padded to 16
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    const bf16x4 w = ld4(M->w1 + (16 * mt + r) * 16 + 4 * q);
    const f32x4 b = bias(SUR_B1, mt);
#pragma unroll
    for (int g = 0; g < G; ++g) a[g][mt] = activate(mfma16(w, x[g], zero), b);
  }
  // layers 2 and 3: 64 -> 64
  auto hidden = [&](const uint16_t *__restrict__ w, int off, bf16x4(*in)[4], bf16x4(*out)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const f32x4 b = bias(off, mt);
      f32x4 acc[G];
#pragma unroll
      for (int g = 0; g < G; ++g) acc[g] = zero;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) {
        const bf16x4 wk = ld4(w + (16 * mt + r) * 64 + 16 * kt + 4 * q);
#pragma unroll
        for (int g = 0; g < G; ++g) acc[g] = mfma16(wk, in[g][kt], acc[g]);
      }
#pragma unroll
      for (int g = 0; g < G; ++g) out[g][mt] = activate(acc[g], b);
    }
  };
  hidden(M->w2, SUR_B2, a, an);
  hidden(M->w3, SUR_B3, an, a);
  // layer 4: 64 -> 2 (rows padded to 16)
#pragma unroll
  for (int g = 0; g < G; ++g) y[g] = zero;
#pragma unroll
  for (int kt = 0; kt < 4; ++kt) {
    const bf16x4 wk = ld4(M->w4 + r * 64 + 16 * kt + 4 * q);
#pragma unroll
    for (int g = 0; g < G; ++g) y[g] = mfma16(wk, a[g][kt], y[g]);
  }
  if (q == 0) {
    const float b0 = M->theta[SUR_B4], b1 = M->theta[SUR_B4 + 1];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      y[g][0] += b0;
      y[g][1] += b1;
    }
  }
}

// al = ALOSS / n^2 at (T, x_HII) from the table (bilinear in log10 T and
// u = log10((x + 1e-4) / (1 - x + 1e-4)) on log10 al).
__device__ __forceinline__ float sur_al(const SurDev *__restrict__ M, float lt, float x) {
  float ft = (lt - SUR_TLO) / SUR_DT;
  ft = fminf(fmaxf(ft, 0.f), (float)(SUR_NT - 1) - 1e-3f);
  const float xc = fminf(fmaxf(x, 0.f), 1.f);
  float fx = (log10f((xc + 1e-4f) / (1.f - xc + 1e-4f)) + 4.f) * 0.125f * (float)(SUR_NX - 1);
  fx = fmaxf(fx, 0.f);
  fx = fminf(fx, (float)(SUR_NX - 1) - 1e-3f);
  const int it = (int)ft, ix = (int)fx;
  const float wt = ft - (float)it, wx = fx - (float)ix;
  const float *t = M->altab + it * SUR_NX + ix;
  return exp10f((1.f - wt) * ((1.f - wx) * t[0] + wx * t[1]) + wt * ((1.f - wx) * t[SUR_NX] + wx * t[SUR_NX + 1]));
}

// Raw features of one cell (n, T, y0 = n_HI/n, dt in seconds); returns
// ce*dt of the tabulated relaxation and whether the cell is in the hull.
__device__ __forceinline__ bool sur_features(const SurDev *__restrict__ M, double n, double T, double y0, double dts,
                                             float f[4], float &cedt) {
  const float lt = log10f((float)T);
  const float x = (float)(1.0 - y0);
  const float al = sur_al(M, lt, x);
  const double boltzm = 1.3807e-16;
  cedt = (float)((2. * n * (double)al) / (3. * boltzm * T) * dts);
  f[0] = log10f((float)n);
  f[1] = lt;
  f[2] = x;
  f[3] = log10f(fmaxf(cedt, 1e-30f));
  bool in = true;
#pragma unroll
  for (int k = 0; k < 4; ++k) in = in && f[k] >= M->lo[k] && f[k] <= M->hi[k];
  return in;
}

}  // namespace wx
