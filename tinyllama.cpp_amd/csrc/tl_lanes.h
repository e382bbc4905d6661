// tl_lanes.h — exchanges and reductions between the lanes of a wave in vector instructions. __shfl_xor goes through the LDS unit
// (ds_bpermute), about 60 ns a step; a reduction over a wave is six of them one after another, which a launch of 4 to 6 us that is a
// chain of such steps notices: the residual norms of a one-token step, a row sum and, for half of them, a router's choice of 4 of 16,
// 5.40 -> 4.79 us on average.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

template <int CTRL>
__device__ __forceinline__ unsigned tl_dpp(unsigned x) {
  return (unsigned)__builtin_amdgcn_update_dpp((int)x, (int)x, CTRL, 0xf, 0xf, false);
}
// x of lane (this one ^ O): what __shfl_xor(x, O) returns where both lanes are active
template <int O>
__device__ __forceinline__ unsigned tl_xor_bits(unsigned x) {
  static_assert(O == 1 || O == 2 || O == 4 || O == 8 || O == 16 || O == 32, "");
  if constexpr (O == 1) return tl_dpp<0xB1>(x);                   // quad_perm [1,0,3,2]
  else if constexpr (O == 2) return tl_dpp<0x4E>(x);              // quad_perm [2,3,0,1]
  else if constexpr (O == 4) return tl_dpp<0x1B>(tl_dpp<0x141>(x));  // lane ^ 7 (row_half_mirror), then ^ 3 (quad_perm [3,2,1,0])
  else if constexpr (O == 8) return tl_dpp<0x128>(x);             // row_ror:8
  else {
    // both operands x: the results hold the lower and the upper partner's x
    const auto r = O == 16 ? __builtin_amdgcn_permlane16_swap(x, x, false, false) : __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return threadIdx.x & O ? r[0] : r[1];
  }
}
template <int O>
__device__ __forceinline__ float tl_xor(float x) {
  return __uint_as_float(tl_xor_bits<O>(__float_as_uint(x)));
}
template <int O>
__device__ __forceinline__ int tl_xor(int x) {
  return (int)tl_xor_bits<O>((unsigned)x);
}
template <int O>
__device__ __forceinline__ double tl_xor(double x) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  const unsigned lo = tl_xor_bits<O>((unsigned)b), hi = tl_xor_bits<O>((unsigned)(b >> 32));
  return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}
// f(distance) for the distances FROM (32: over a wave, 16: a half, 8: a row of 16) down to 1
template <int FROM, class F>
__device__ __forceinline__ void tl_butterfly(F f) {
  if constexpr (FROM >= 32) f(std::integral_constant<int, 32>{});
  if constexpr (FROM >= 16) f(std::integral_constant<int, 16>{});
  if constexpr (FROM >= 8) f(std::integral_constant<int, 8>{});
  if constexpr (FROM >= 4) f(std::integral_constant<int, 4>{});
  if constexpr (FROM >= 2) f(std::integral_constant<int, 2>{});
  f(std::integral_constant<int, 1>{});
}
// the order of __shfl_xor by 32, 16, .. 1: the same bits
template <class T>
__device__ __forceinline__ T tl_wave_sum(T s) {
  tl_butterfly<32>([&](auto o) __attribute__((always_inline)) { s += tl_xor<decltype(o)::value>(s); });
  return s;
}
template <int FROM = 32>
__device__ __forceinline__ float tl_wave_max(float m) {
  tl_butterfly<FROM>([&](auto o) __attribute__((always_inline)) { m = fmaxf(m, tl_xor<decltype(o)::value>(m)); });
  return m;
}
// the largest value of a wave (FROM 32; 8: of each row of 16) and its index, the lower index among equals, as seen from each lane
template <int FROM>
__device__ __forceinline__ void tl_lanes_best(float& v, int& i) {
  tl_butterfly<FROM>([&](auto o) __attribute__((always_inline)) {
    const float ov = tl_xor<decltype(o)::value>(v);
    const int oi = tl_xor<decltype(o)::value>(i);
    if (ov > v || (ov == v && oi < i)) {
      v = ov;
      i = oi;
    }
  });
}
__device__ __forceinline__ void tl_wave_best(float& v, int& i) { tl_lanes_best<32>(v, i); }
