// Device helpers shared by the matrix-free kernels (matfree.hip, mfpatch.hip):
// MFMA wrappers and their operand types, the metric product, copies into LDS.
#pragma once
#include <hip/hip_runtime.h>

namespace ngsamd {

typedef double double4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double4v Mfma(double a, double b, double4v c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4v Mfma(float a, float b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <class T> struct Acc4;
template <> struct Acc4<double> { typedef double4v type; };
template <> struct Acc4<float> { typedef float4v type; };

// Row of the 16x16 result held in accumulator element r of a lane in lane
// group grp = lane/16 (the column is lane%16).  Measured on gfx950:
// v_mfma_f32_16x16x4f32 holds rows 4*grp+r, v_mfma_f64_16x16x4f64 holds
// rows grp+4*r.
template <class T>
__device__ __forceinline__ constexpr int AccRow(int grp, int r) {
  return sizeof(T) == 8 ? grp + 4 * r : 4 * grp + r;
}

template <class V>
__device__ __forceinline__ void AtomicAddV(V* p, V v) {
  atomicAdd(p, v);
}

// Metric G (symmetric, packed) times vector: 2D (xx,yy,xy), 3D (xx,yy,zz,xy,xz,yz).
template <int DIM, class T>
__device__ __forceinline__ void ApplyMetric(const T* g, const T* u, T* v) {
  if constexpr (DIM == 2) {
    v[0] = g[0] * u[0] + g[2] * u[1];
    v[1] = g[2] * u[0] + g[1] * u[1];
  } else {
    v[0] = g[0] * u[0] + g[3] * u[1] + g[4] * u[2];
    v[1] = g[3] * u[0] + g[1] * u[1] + g[5] * u[2];
    v[2] = g[4] * u[0] + g[5] * u[1] + g[2] * u[2];
  }
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
template <class H> struct Vec8;
template <> struct Vec8<__bf16> { typedef bf16x8 type; };
template <> struct Vec8<_Float16> { typedef half8 type; };
__device__ __forceinline__ float4v Mfma16(bf16x8 a, bf16x8 b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4v Mfma16(half8 a, half8 b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Copy n 16-byte words of a class's matrices from global memory into LDS.
// Each thread issues 4 loads before its first LDS write (from clamped
// indices, so no load sits behind a branch): a plain load-then-store loop
// waits for every load in turn.
template <int BLOCK>
__device__ __forceinline__ void CopyToLds(void* dst, const void* src, int n) {
  constexpr int U = 4;
  const uint4* s = reinterpret_cast<const uint4*>(src);
  uint4* d = reinterpret_cast<uint4*>(dst);
  for (int base = 0; base < n; base += BLOCK * U) {
    uint4 v[U];
#pragma unroll
    for (int j = 0; j < U; j++) v[j] = s[min(base + j * BLOCK + (int)threadIdx.x, n - 1)];
#pragma unroll
    for (int j = 0; j < U; j++) {
      const int i = base + j * BLOCK + (int)threadIdx.x;
      if (i < n) d[i] = v[j];
    }
  }
}

}  // namespace ngsamd
