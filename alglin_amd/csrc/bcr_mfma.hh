// Matrix-core helpers of the pair kernels and the several-column sweeps.
#pragma once
#include <hip/hip_runtime.h>

namespace bcr {

template <typename T>
using V2 = T __attribute__((ext_vector_type(2)));
template <typename T>
using V4 = T __attribute__((ext_vector_type(4)));
template <typename T>
using V16 = T __attribute__((ext_vector_type(16)));

// one 16 x 16 x 4 product-accumulate: FP32 or FP64 matrix cores (the same
// operand and accumulator layouts)
__device__ __forceinline__ V4<float> mfma1(float a, float b, V4<float> c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ V4<double> mfma1(double a, double b, V4<double> c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// The 16 x 16 x 4 products take A (16 x 4) as A[m][k] in lane m + 16 k and B
// (4 x 16) as B[k][n] in lane n + 16 k, in both precisions; the 16 x 16
// result comes back as four values per lane, lane n + 16 g holding in its
// value i row 4 g + i (FP32) or row g + 4 i (FP64) of column n.  kro gives
// that row; every k sum below runs in the same order (the i-th product of a
// 16-wide block takes k = kro(g, i) in lane group g), so a 16-row block in
// the result layout is the next product's B operand as it stands.
template <typename T>
__device__ __forceinline__ constexpr int kro(int g, int i) {
  return sizeof(T) == 4 ? 4 * g + i : g + 4 * i;
}
// rows kro(g, 0..3) of a 16-row block (LDS): one 16-byte read for FP32,
// four strided reads for FP64
template <typename T>
__device__ __forceinline__ V4<T> ld4(const T* blk, int g) {
  if constexpr (sizeof(T) == 4) {
    return *reinterpret_cast<const V4<T>*>(blk + 4 * g);
  } else {
    return V4<T>{blk[g], blk[g + 4], blk[g + 8], blk[g + 12]};
  }
}

template <typename T>
__device__ __forceinline__ V4<T> mfma4(V4<T> a, V4<T> b, V4<T> c) {
  c = mfma1(a.x, b.x, c);
  c = mfma1(a.y, b.y, c);
  c = mfma1(a.z, b.z, c);
  c = mfma1(a.w, b.w, c);
  return c;
}

}  // namespace bcr
