// Values of other lanes without LDS: broadcasts within the 16-lane rows of a wave.
#pragma once
#include <hip/hip_runtime.h>
#include <utility>

namespace kad {

// The value of lane N of every 16-lane row to all its lanes (DPP row_newbcast).  Every lane
// must be active.
template <int N>
__device__ __forceinline__ double lane16(double v) {
  return __longlong_as_double(__builtin_amdgcn_update_dpp(0LL, __double_as_longlong(v), 0x150 + N, 0xF, 0xF, true));
}
template <int N>
__device__ __forceinline__ float lane16(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + N, 0xF, 0xF, true));
}

// f(integral_constant 0), f(1), ..., f(N - 1): a loop whose index is a constant expression.
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>()), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>());
}

}  // namespace kad
