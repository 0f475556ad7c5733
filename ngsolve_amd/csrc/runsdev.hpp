// Device side of the runs layout's products, shared by the single (spmv.hip)
// and the batched (batch.hip) kernels: a group of lanes per run, the run's
// row sums in registers.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "csr.hpp"

namespace ngsamd {

// column slots per lane and pass, whose loads are all in flight together:
// about 50 registers of loads whatever R, fewer slots where several vectors'
// sums take the registers
constexpr int RunUnroll(int R, int KC = 1) {
  const int one = R == 1 ? 8 : R == 2 ? 6 : R <= 4 ? 4 : R <= 6 ? 3 : 2;
  const int fit = (130 - 2 * R * KC) / (3 + 2 * KC + 2 * R);
  return KC == 1 || fit > one ? one : fit < 1 ? 1 : fit;
}

// Calls f(R, U) as compile-time constants for a task of run length R whose
// runs hold up to m slots per lane: U = min(m, RunUnroll(R, KC)), so that no
// pass loads slots that no lane has (KC = 8: R <= 3 only).
template <int KC, int R, int U, class F>
__device__ __forceinline__ void ForRunSlots(int m, F&& f) {
  if constexpr (U < RunUnroll(R, KC)) {
    if (m <= U) f(std::integral_constant<int, R>{}, std::integral_constant<int, U>{});
    else ForRunSlots<KC, R, U + 1>(m, f);
  } else {
    f(std::integral_constant<int, R>{}, std::integral_constant<int, U>{});
  }
}
template <int KC, int R = 1, class F>
__device__ __forceinline__ void ForRunShape(int r, int m, F&& f) {
  if constexpr (R < (KC == 8 ? 3 : kMaxRun)) {
    if (r == R) ForRunSlots<KC, R, 1>(m, f);
    else ForRunShape<KC, R + 1>(r, m, f);
  } else {
    ForRunSlots<KC, R, 1>(m, f);
  }
}

template <int CTRL>
__device__ __forceinline__ double DppMove(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// Sum over the lane's group of 2^lg lanes, in every lane of it (lg uniform,
// 3 to 6): lanes i and i ^ 1, then i ^ 2 (quad permutations), then the other
// quad of 8, the other 8 of 16 (mirrors), then by shuffles.
__device__ __forceinline__ double GroupSum(double v, int lg) {
  v += DppMove<0xB1>(v);
  v += DppMove<0x4E>(v);
  v += DppMove<0x141>(v);
  if (lg > 3) v += DppMove<0x140>(v);
  if (lg > 4) v += __shfl_xor(v, 16, 64);
  if (lg > 5) v += __shfl_xor(v, 32, 64);
  return v;
}

// two adjacent doubles in one 16-byte load, aligned like a double
typedef double double2u __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ void LoadPair(const double* p, double& a, double& b) {
  const double2u t = *reinterpret_cast<const double2u*>(p);
  a = t.x;
  b = t.y;
}

// R adjacent floats in 16-, 8- and 4-byte loads, aligned like a float
typedef float float2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
template <int R>
__device__ __forceinline__ void LoadFloats(const float* p, double* v) {
  constexpr int n4 = R / 4 * 4, n2 = n4 + (R % 4) / 2 * 2;
#pragma unroll
  for (int q = 0; q < n4; q += 4) {
    const float4u t = *reinterpret_cast<const float4u*>(p + q);
    v[q] = t.x, v[q + 1] = t.y, v[q + 2] = t.z, v[q + 3] = t.w;
  }
  if constexpr (n2 > n4) {
    const float2u t = *reinterpret_cast<const float2u*>(p + n4);
    v[n4] = t.x, v[n4 + 1] = t.y;
  }
  if constexpr (R > n2) v[n2] = p[n2];
}

// acc[q][j] = this lane's share of row q of its run (first column c0, first
// value v0, L slots) times component j0 + j of the K-vector x (a pointer), or
// times x(column) (KC = 1)
template <int R, int KC, int U, class X, class M>
__device__ __forceinline__ void RunPartials(const int* __restrict__ rcols, const M* __restrict__ rvals,
                                            const X& x, int K, int j0, int c0, int v0, int L, int l,
                                            int G, double (&acc)[R][KC]) {
#pragma unroll
  for (int q = 0; q < R; q++)
#pragma unroll
    for (int j = 0; j < KC; j++) acc[q][j] = 0.0;
  for (int k0 = l; k0 < L; k0 += U * G) {
    // unconditional loads from clamped slots, so that all are in flight at once
    int c[U];
    double v[U][R], xv[U][KC];
#pragma unroll
    for (int i = 0; i < U; i++) c[i] = rcols[c0 + min(k0 + i * G, L - 1)];
#pragma unroll
    for (int i = 0; i < U; i++) {
      const M* vp = rvals + (v0 + min(k0 + i * G, L - 1) * R);
      if constexpr (sizeof(M) == 8) {
#pragma unroll
        for (int q = 0; q + 1 < R; q += 2) LoadPair(vp + q, v[i][q], v[i][q + 1]);
        if constexpr (R % 2 == 1) v[i][R - 1] = vp[R - 1];
      } else {
        LoadFloats<R>(vp, v[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < U; i++) {
      if constexpr (std::is_class<X>::value) {
        xv[i][0] = x(c[i]);
      } else {
        const double* xp = x + ((int64_t)c[i] * K + j0);
        if constexpr (KC == 1) xv[i][0] = xp[0];
#pragma unroll
        for (int j = 0; j + 1 < KC; j += 2) LoadPair(xp + j, xv[i][j], xv[i][j + 1]);
      }
    }
#pragma unroll
    for (int i = 0; i < U; i++) {
      const bool ok = k0 + i * G < L;
#pragma unroll
      for (int q = 0; q < R; q++)
#pragma unroll
        for (int j = 0; j < KC; j++) {
          const double t = __builtin_fma(v[i][q], xv[i][j], acc[q][j]);
          acc[q][j] = ok ? t : acc[q][j];
        }
    }
  }
}

// Lanes per run of R rows and L columns (log2): the fewest, from 8 (16 for
// runs of 4 and more rows and 9 and more columns), whose first pass covers the
// run.  us per apply with at least 8 / 16 lanes: 128^2 p=5 (runs of 4 and 6
// rows) 27.2 / 21.7; runs of up to 3 rows 32^3 p=4 327 / 340, 64^2 p=3 4.4 /
// 4.8.
inline int RunGroupLog2(int R, int L) {
  int lg = L <= 8 || R < 4 ? 3 : 4;
  while (lg < 6 && L > RunUnroll(R) << lg) lg++;
  return lg;
}

}  // namespace ngsamd
