// The two MFMA shapes the kernels use (gfx950): 16 x 16 output blocks,
// k = 4 per instruction, float64 and float32.
//
// Operand layouts (measured on gfx950): for k-step inputs A (16 x 4) and
// B (4 x 16), lane m + 16 k holds A[m][k] and lane n + 16 k holds B[k][n];
// accumulator slot r of lane l holds row (l / 16) + 4 r (float64) or
// 4 (l / 16) + r (float32) of column l % 16.
#pragma once

#include <hip/hip_runtime.h>

namespace qsv {

template <typename T>
struct Mfma;
template <>
struct Mfma<double> {
  typedef double acc __attribute__((ext_vector_type(4)));
  __device__ static acc op(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma<float> {
  typedef float acc __attribute__((ext_vector_type(4)));
  __device__ static acc op(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// A 4 x 4 transpose over the lane groups g = lane / 16: r[c] of group g becomes
// r[g] of group c.
__device__ __forceinline__ void group_transpose(uint32_t (&r)[4]) {
  // odd groups of the first with even groups of the second, then upper halves of
  // the first with lower halves of the second
  const auto a = __builtin_amdgcn_permlane16_swap(r[0], r[1], false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(r[2], r[3], false, false);
  const auto e = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
  const auto o = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
  r[0] = e[0];
  r[1] = o[0];
  r[2] = e[1];
  r[3] = o[1];
}

// pb[s] = row[4 s + kk], lane group kk = lane / 16 of four with the same row: four
// loads of four entries a lane (group g: k-steps 4 i + g) and a transpose over
// the groups, for sixteen loads of which each touches sixteen cache lines (a
// block of k_apply64d: 2.3 us more).
template <typename T>
__device__ __forceinline__ void row_operand(const T* row, int kk, T (&pb)[16]) {
  typedef T t4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  t4 v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const t4*>(row + 16 * i + 4 * kk);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if constexpr (sizeof(T) == 4) {
        lo[c] = __float_as_uint(v[i][c]);
      } else {
        lo[c] = uint32_t(__double2loint(v[i][c]));
        hi[c] = uint32_t(__double2hiint(v[i][c]));
      }
    }
    group_transpose(lo);
    if constexpr (sizeof(T) == 8) group_transpose(hi);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if constexpr (sizeof(T) == 4)
        pb[4 * i + c] = __uint_as_float(lo[c]);
      else
        pb[4 * i + c] = __hiloint2double(int(hi[c]), int(lo[c]));
    }
  }
}

}  // namespace qsv
