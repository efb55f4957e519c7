// Shared helpers of libf3d: error reporting, launch checks, wave reductions.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "../../include/f3d.h"

namespace f3d {

// Thread-local last error message, read back through f3d_last_error().
void set_error(const char* fmt, ...);

#define F3D_REQUIRE(cond, code, ...)     \
  do {                                   \
    if (!(cond)) {                       \
      ::f3d::set_error(__VA_ARGS__);     \
      return (code);                     \
    }                                    \
  } while (0)

#define F3D_HIP_CHECK(expr)                                                   \
  do {                                                                        \
    hipError_t e_ = (expr);                                                   \
    if (e_ != hipSuccess) {                                                   \
      ::f3d::set_error("%s failed: %s", #expr, hipGetErrorString(e_));        \
      return F3D_EHIP;                                                        \
    }                                                                         \
  } while (0)

// Launch a kernel and report a launch failure as F3D_EHIP.
#define F3D_LAUNCH(kernel, grid, block, lds, stream, ...)                     \
  do {                                                                        \
    hipLaunchKernelGGL(kernel, grid, block, lds, stream, __VA_ARGS__);        \
    hipError_t e_ = hipGetLastError();                                        \
    if (e_ != hipSuccess) {                                                   \
      ::f3d::set_error("launch of %s failed: %s", #kernel,                    \
                       hipGetErrorString(e_));                                \
      return F3D_EHIP;                                                        \
    }                                                                         \
  } while (0)

// Compute units of the current device (256 where it cannot be asked).
int num_cus();

inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }
inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

constexpr double kPi = 3.14159265358979323846;

// Workgroup barrier that orders LDS only: global loads and stores stay in
// flight (a __syncthreads waits for them).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ---- wave64 reductions (device) -----------------------------------------
// Lane l meets lane l ^ O, for O = 32, 16, 8, 4, 2, 1: exchanges of register
// halves and rows, and row rotations (after the step over 8, lanes 8 apart
// agree, so that a rotation by 4 reaches lane l ^ 4).  No step goes through
// LDS, whose shuffles cost a wave's start several microseconds when all eight
// waves of a SIMD reduce at once; the pairs and their order are those of a
// butterfly of shuffles, so sums are the same to the bit.
template <int O>
__device__ __forceinline__ void wave_meet(int v, int& x, int& y) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  if constexpr (O == 32 || O == 16) {
    const u2 s = O == 32 ? __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false)
                         : __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    x = (int)s[0];
    y = (int)s[1];
  } else {
    constexpr int ctrl = O == 8 ? 0x128 : O == 4 ? 0x124 : O == 2 ? 0x4e : 0xb1;
    x = v;
    y = __builtin_amdgcn_mov_dpp(v, ctrl, 0xf, 0xf, false);
  }
}
template <int O>
__device__ __forceinline__ void wave_meet(double v, double& x, double& y) {
  const unsigned long long u = __double_as_longlong(v);
  int xl, yl, xh, yh;
  wave_meet<O>((int)(unsigned)u, xl, yl);
  wave_meet<O>((int)(u >> 32), xh, yh);
  x = __longlong_as_double(((unsigned long long)(unsigned)xh << 32) | (unsigned)xl);
  y = __longlong_as_double(((unsigned long long)(unsigned)yh << 32) | (unsigned)yl);
}
template <int O = 32, typename T, typename Op>
__device__ __forceinline__ T wave_fold(T v, Op op) {
  T x, y;
  wave_meet<O>(v, x, y);
  v = op(x, y);
  if constexpr (O > 1) v = wave_fold<O / 2>(v, op);
  return v;
}
__device__ __forceinline__ int wave_min_i32(int v) {
  return wave_fold(v, [](int a, int b) { return min(a, b); });
}
__device__ __forceinline__ int wave_max_i32(int v) {
  return wave_fold(v, [](int a, int b) { return max(a, b); });
}
__device__ __forceinline__ double wave_sum_f64(double v) {
  return wave_fold(v, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ double wave_min_f64(double v) {
  return wave_fold(v, [](double a, double b) { return fmin(a, b); });
}
__device__ __forceinline__ double wave_max_f64(double v) {
  return wave_fold(v, [](double a, double b) { return fmax(a, b); });
}

}  // namespace f3d
