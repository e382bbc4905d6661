// tl_hsplit.h — an activation's two f16 parts, its power of two and its block's sum, as the f16 GEMM (tl_hgemm.hip) reads them: written by
// the norm, SwiGLU and split launches and by the attention kernels that finish whole super-blocks.
#pragma once
#include <hip/hip_runtime.h>

#include "tl_lanes.h"

// eight columns i0.. of token t (all lanes of a half wave on one super-block): both parts, the power of two, the block sum
__device__ __forceinline__ void tl_hsplit8(const float* v, _Float16* __restrict__ planes, size_t ps, int t, int K, int i0, int tpad) {
  float top = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) top = fmaxf(top, fabsf(v[e]));
  top = tl_wave_max<16>(top);
  if (i0 >= K) return;  // (whole quads of threads: K is a multiple of 32)
  // top * 2^k in [512, 1024); k of zeros and of sub-normals keeps 2^k and 2^-k normal
  int ex = (int)((__builtin_bit_cast(unsigned, top) >> 23) & 255u) - 127;
  ex = top == 0.f ? 0 : ex < -117 ? -117 : ex;
  const float scale = __builtin_bit_cast(float, (unsigned)(127 + 9 - ex) << 23);
  _Float16* bs = planes + 2 * ps;
  float* inv = reinterpret_cast<float*>(bs + ps / 16);
  const int sb = i0 >> 8;
  if ((i0 & 255) == 0) inv[(size_t)sb * tpad + t] = __builtin_bit_cast(float, (unsigned)(127 - 9 + ex) << 23);
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = v[e] * scale;
  float s = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));  // (scaled: below 2^15 whatever the row holds)
  s += tl_xor<1>(s);
  s += tl_xor<2>(s);
  if ((i0 & 31) == 0 && (K & 255) == 0) {  // sum of the 32-column block, at the place of its minimum in the operand
    const int j = (i0 >> 5) & 7, at = j < 4 ? 2 * j : 2 * (j - 4) + 1;
    _Float16* o = bs + ((size_t)sb * tpad + t) * 16 + at;
    const _Float16 h = (_Float16)s;
    o[0] = h;
    o[8] = (_Float16)(s - (float)h);
  }
  constexpr int ORDER[8] = {0, 2, 1, 3, 4, 6, 5, 7};
  typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
  f16x8 hi, lo;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    hi[e] = (_Float16)x[ORDER[e]];
    lo[e] = (_Float16)(x[ORDER[e]] - (float)hi[e]);
  }
  *reinterpret_cast<f16x8*>(planes + (size_t)t * K + i0) = hi;
  *reinterpret_cast<f16x8*>(planes + ps + (size_t)t * K + i0) = lo;
}
