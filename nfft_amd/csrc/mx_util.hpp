// Pieces shared by the matrix-core B and B^T kernels (mx.hpp, spread_mx2d.hpp):
// 16 x 16 x 4 products, window rows in LDS, moves within and across 16-lane
// rows.
#pragma once

#include "engine.hpp"
#include "window.hpp"

namespace nfft_hip {

template <typename R> struct MxTypes;
template <> struct MxTypes<float> {
  using v4 = float __attribute__((ext_vector_type(4)));
};
template <> struct MxTypes<double> {
  using v4 = double __attribute__((ext_vector_type(4)));
};
template <typename R> using mx4 = typename MxTypes<R>::v4;

// c + a b for a 16 x 4 operand a (lane l holds row l & 15, column l >> 4), a
// 4 x 16 operand b (lane l: row l >> 4, column l & 15) and a 16 x 16 result
// (lane l, element r: column l & 15 and row mx_row<R>(l, r)).
__device__ __forceinline__ mx4<float> mx_mul(float a, float b, mx4<float> c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ mx4<double> mx_mul(double a, double b, mx4<double> c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
template <typename R> __device__ __forceinline__ int mx_row(int q, int r) {
  return sizeof(R) == 4 ? 4 * q + r : q + 4 * r;
}

// DPP move within 16-lane rows: lane I of the row
template <int CTRL> __device__ __forceinline__ float mx_dpp(float x) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int CTRL> __device__ __forceinline__ double mx_dpp(double x) {
  const long long u = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(u & 0xffffffffLL), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
template <int I, typename R> __device__ __forceinline__ R mx_bcast(R x) {
  return mx_dpp<0x150 + I>(x);
}
// sum over the four lanes of a column (l & 15), in every lane
__device__ __forceinline__ float mx_col_sum(float x) {
  const int v = __float_as_int(x);
  auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  x = __int_as_float(a[0]) + __int_as_float(a[1]);
  const int w = __float_as_int(x);
  auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  return __int_as_float(b[0]) + __int_as_float(b[1]);
}
__device__ __forceinline__ double mx_col_sum(double x) {
  x += __shfl_xor(x, 32, 64);
  return x + __shfl_xor(x, 16, 64);
}

// Window rows of a chunk of nodes in LDS: row (t, node) holds the node's
// dimension-t window over the positions, kMxPitch elements apart (rows of 16
// or more positions; 20 spreads the 4 x 16 operand reads over the banks).
constexpr int kMxPitch = 20;
// coefficients per polynomial in the LDS table of plans whose dimensions
// differ in sigma
template <typename R> constexpr int kMxCoef = (poly_deg_v<R> + 4) / 4 * 4;

// One window row of PITCH positions: taps at shift .. shift + W - 1, zeros at
// the others.  Tap pairs (w, W-1-w) come from one polynomial's even
// and odd parts at tt = frac - 1/2; pc(w) gives tap w's coefficients.
template <typename R, int W, int PITCH = kMxPitch, typename Coef>
__device__ __forceinline__ void mx_window_row(R *row, int shift, R tt, Coef pc) {
  constexpr int PD = poly_deg_v<R>;
  constexpr int KE = PD - (PD % 2);      // highest even power
  constexpr int KO = PD - 1 + (PD % 2);  // highest odd power
  constexpr int V = 16 / sizeof(R);
  using vec = R __attribute__((ext_vector_type(V)));
#pragma unroll
  for (int z = 0; z < PITCH; z += V) *reinterpret_cast<vec *>(row + z) = vec(0);
  const R t2 = tt * tt;
  R *at = row + shift;
#pragma unroll
  for (int w = 0; w < W / 2; w++) {
    const R *c = pc(w);
    R e = c[KE];
#pragma unroll
    for (int k = KE - 2; k >= 0; k -= 2) e = fma(e, t2, c[k]);
    R o = c[KO];
#pragma unroll
    for (int k = KO - 2; k >= 1; k -= 2) o = fma(o, t2, c[k]);
    at[w] = fma(tt, o, e);
    at[W - 1 - w] = fma(-tt, o, e);
  }
}

// copies the window polynomials of D dimensions (lower half of the taps) to
// LDS, kMxCoef apart
template <typename R, int D, int W>
__device__ __forceinline__ void mx_load_poly(R *spoly, const R *poly, int tid, int nthr) {
  constexpr int C = poly_deg_v<R> + 1, H = W / 2;
  for (int i = tid; i < D * H * C; i += nthr) {
    const int k = i % C, w = (i / C) % H, t = i / (C * H);
    spoly[(t * H + w) * kMxCoef<R> + k] = poly[(t * W + w) * C + k];
  }
}

// v[r] = 0 in place, for a branch of the node loop: a plain assignment made the
// compiler copy all accumulators at the loop's head
template <typename V> __device__ __forceinline__ void mx_clear(V &v, int r) {
  auto x = v[r];
  if constexpr (sizeof(x) == 4) asm("v_mov_b32 %0, 0" : "+v"(x));
  else asm("v_mov_b64 %0, 0" : "+v"(x));
  v[r] = x;
}

// a[i] = p1 times lane i of every 16-lane row of p0
template <typename R, int H, int I = 0>
__device__ __forceinline__ void mx_weights(R (&a)[H], R p0, R p1) {
  a[I] = mx_bcast<I>(p0) * p1;
  if constexpr (I + 1 < H) mx_weights<R, H, I + 1>(a, p0, p1);
}

}  // namespace nfft_hip
