// tl_parts.h — the sum over the slices of a K-split GEMM where its consumer takes it. Every slice's load is in flight before the first
// addition: with the slice count known only at run time the loads go out in groups, each of which the compiler waits for, and in a launch
// of a few workgroups (a step of 8 sequences, a prompt of 23 tokens) those round trips are what it takes.
#pragma once
#include <hip/hip_runtime.h>

#include "tl_internal.h"

typedef float tl_f32x4 __attribute__((ext_vector_type(4)));

template <int S, int M, int N>
__device__ __forceinline__ void tl_parts_of(const GemmParts (&g)[M], size_t o, tl_f32x4 (&sum)[M][N]) {
  tl_f32x4 p[S][M][N];
#pragma unroll
  for (int z = 0; z < S; ++z)
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int n = 0; n < N; ++n) p[z][m][n] = *reinterpret_cast<const tl_f32x4*>(g[m].part + (size_t)z * g[m].n + o + 4 * n);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int n = 0; n < N; ++n) {
      sum[m][n] = p[0][m][n];
#pragma unroll
      for (int z = 1; z < S; ++z) sum[m][n] += p[z][m][n];
    }
}
// 4 N numbers at o (16 bytes) of M products that have the same number of slices, 1 and more, each added up in slice order
template <int M, int N>
__device__ __forceinline__ void tl_parts_sum(const GemmParts (&g)[M], size_t o, tl_f32x4 (&sum)[M][N]) {
  switch (g[0].S) {
    case 1: tl_parts_of<1>(g, o, sum); return;
    case 2: tl_parts_of<2>(g, o, sum); return;
    case 3: tl_parts_of<3>(g, o, sum); return;
    case 4: tl_parts_of<4>(g, o, sum); return;
    case 5: tl_parts_of<5>(g, o, sum); return;
    case 6: tl_parts_of<6>(g, o, sum); return;
    case 7: tl_parts_of<7>(g, o, sum); return;
    default: break;
  }
  tl_parts_of<8>(g, o, sum);
  for (int z = 8; z < g[0].S; ++z)
    for (int m = 0; m < M; ++m)
      for (int n = 0; n < N; ++n) sum[m][n] += *reinterpret_cast<const tl_f32x4*>(g[m].part + (size_t)z * g[m].n + o + 4 * n);
}
