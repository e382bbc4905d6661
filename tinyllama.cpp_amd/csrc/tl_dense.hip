// tl_dense.hip — products with bf16 weight matrices [rows][cols] (row-major, y = W x), FP32 activations and accumulation.
//
//   GEMV (one token): a wave per output row, 16 B of weights per lane per step, widened exactly to FP32: FP32 arithmetic
//   throughout, bound by the bytes of the matrix.
//   GEMM (a chunk of tokens) on the matrix cores: v_mfma_f32_32x32x16_bf16 with the WEIGHTS as the A operand (M = output
//   features) and the tokens as B (N = tokens), so that a lane ends up holding 4 x 4 consecutive features of ONE token and
//   stores them as 16-byte pieces of that token's output row. The FP32 activations are split while they are staged into
//   LDS: terms = 1 keeps their bf16 rounding, terms = 3 keeps hi + mid + lo (3 x 8 mantissa bits = all 24 of an FP32
//   value); the weights are bf16 to begin with, so three MFMAs per product reproduce the FP32 product exactly and only the
//   order of the FP32 accumulation differs from a scalar loop.
//   A workgroup of 4 waves owns a 64 x 64 or (enough rows and tokens) a 128 x 128 feature x token tile and walks 64 or 32
//   columns a step. What bounds it is the way of the operands: a few workgroups a CU wait for the loads of a step, many of them
//   for the 64 bytes a cycle that a CU's cache hands out (the activations are FP32 and every tile reads them). So two steps are
//   in flight while a third is multiplied out of LDS, which needs loads without a branch around them: one kernel for wide
//   loads, one for odd shapes. One step in flight behind a branch, products of eight columns: 2048 x 2048 times 64 / 512 / 1999
//   tokens 30 / 39 / 63 us, now 17 / 19 / 47; 8192 x 2048 times 1999 148 -> 113 (594 TFLOP/s; among a prompt's other launches 182 -> 140).
//   Large products of one term do without the conversion in every tile: the items are rounded to a bf16 plane once, and both sides go
//   from memory to LDS without registers in between (dense_plane_kernel: 10304 x 2048 times 1999 tokens 174 -> 114 us with the
//   conversion of 8, that is 740 and 800 TFLOP/s; staged through registers from the same plane 133). What bounds it now: barriers
//   and fragment reads between the products of a step, and at these sizes the last of 2.5 rounds of tiles.
//   Items may be gathered (x_rows), scattered (y_rows) and grouped (group_off: blockIdx.z = matrix of the group; tiles beyond a
//   group's items leave at once), which is what the experts of a mixture need: the plan lives on the device, the grid is sized for
//   the worst case.
#include <math.h>
#include <stdlib.h>

#include <atomic>

#include "tl_bf16.h"
#include "tl_lds.h"
#include "tl_stack.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;

// The epilogue of a wave: WM x WN products of 32 x 32, features from f0 on, items from i0 on (items below hi are stored). 32 items at a
// time go through the wave's part of LDS (dense_store_floats, left by everybody before), out of which a short loop takes four features
// a lane, 128 WM consecutive bytes of a row at a time. Out of the registers, whose numbers are fixed at compile time, the activations'
// code stood there once per accumulator, and a launch's only pass through it waited for instructions: with xIELU behind it,
// 4096 x 2048 times 1998 tokens took 82 us, 10304 x 2048 with tanh on some features 159, now 51 and 120. The same bits.
constexpr int dense_store_floats(int wm) { return 32 * (32 * wm + 4); }
template <int WM, int WN>
__device__ __forceinline__ void dense_store(const DenseArgs& a, const f32x16 (&acc)[WM][WN], float* Y, int f0, int i0, int hi, int lane, float* st) {
  constexpr int LD = 32 * WM + 4, Q = 8 * WM;  // (padded: 16 items' pieces meet no bank twice)
  const bool v4 = (a.ldy & 3) == 0 && ((size_t)Y & 15) == 0;
  const int act_to = a.act_to > 0 ? a.act_to : a.rows;
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    // C layout: lane holds token (lane & 31) of a 32 x 32 product, features (e / 4) * 8 + (lane >> 5) * 4 + (e & 3)
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int gq = 0; gq < 4; ++gq)
        *reinterpret_cast<f32x4*>(st + (lane & 31) * LD + i * 32 + gq * 8 + (lane >> 5) * 4) =
            f32x4{acc[i][j][gq * 4], acc[i][j][gq * 4 + 1], acc[i][j][gq * 4 + 2], acc[i][j][gq * 4 + 3]};
    __builtin_amdgcn_wave_barrier();  // (a wave's LDS operations run in order)
#pragma unroll 1
    for (int p = lane; p < 32 * Q; p += 64) {
      const int tok = p / Q, it = i0 + j * 32 + tok, f = f0 + p % Q * 4;
      if (it >= hi || f >= a.rows) continue;
      f32x4 v = *reinterpret_cast<const f32x4*>(st + tok * LD + p % Q * 4);
      float* yr = Y + (size_t)(a.y_rows ? a.y_rows[it] : it) * a.ldy;
      if (a.glu) {  // (gate, up) pairs: features f, f + 1 -> unit f / 2; f + 2, f + 3 -> the next one
#pragma unroll
        for (int e = 0; e < 2; ++e)
          if (f + 2 * e + 1 < a.rows) yr[(f >> 1) + e] = tl_glu_apply(a.glu_kind, v[2 * e], v[2 * e + 1], a.glu_limit, a.glu_alpha, a.glu_up_add);
        continue;
      }
      if (a.bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (f + e < a.rows) v[e] += a.bias[f + e];
      }
      if (a.softcap > 0.0f) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = a.softcap * tanhf(v[e] / a.softcap);
      }
      if (a.act && f + 4 > a.act_from && f < act_to) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (f + e >= a.act_from && f + e < act_to) v[e] = tl_act_apply(a.act, v[e], a.act_p, a.act_q);
      }
      if (v4 && f + 4 <= a.rows) {
        *reinterpret_cast<f32x4*>(yr + f) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (f + e < a.rows) yr[f + e] = v[e];
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// A workgroup of 4 waves (2 x 2) owns a (64 WM)-feature x (64 WN)-token tile; a wave WM x WN products of 32 x 32.
// FIRST: the first 32 items are multiplied with two terms (terms == 1 otherwise): the second terms of those rows have a place of their
// own in LDS, and the waves that own the 32 items add their products. (All three terms doubled those waves' products and cost 6 % of a
// prompt of 2048 tokens at width 4096, since a launch of one round ends with its slowest workgroup; the second one alone costs 2 %.)
template <int TERMS, int WM, int WN, bool VEC, bool FIRST>
__global__ __launch_bounds__(256) void dense_gemm_kernel(const DenseArgs a) {
  constexpr int BM = 64 * WM, BN = 64 * WN;
  constexpr int BK = TERMS == 1 && WM == 1 ? 64 : 32;  // columns of a step
  constexpr int LDK = BK + 8;                          // padded row of a tile in LDS: sixteen rows' 16-byte reads meet no bank twice
  constexpr int NB = TERMS == 1 ? 2 : 1;               // steps in LDS (three terms in two would leave one workgroup a CU)
  constexpr int KP = BK / 8, RP = 256 / KP;            // 16-byte pieces of a row, rows that the workgroup stages at a time
  constexpr int PW = BM / RP, PX = BN / RP;            // pieces a thread stages
  constexpr int TILES = NB * (BM + TERMS * BN) * LDK * 2;
  static_assert(TILES >= 4 * dense_store_floats(WM) * 4, "");
  __shared__ __attribute__((aligned(16))) unsigned char tiles[TILES];  // (the waves' outputs at the end)
  auto& Ws = *reinterpret_cast<unsigned short(*)[NB][BM][LDK]>(tiles);
  auto& Xs = *reinterpret_cast<unsigned short(*)[NB][TERMS][BN][LDK]>(tiles + NB * BM * LDK * 2);
  __shared__ __attribute__((aligned(16))) unsigned short Xe[NB][FIRST ? 32 : 1][LDK];
  __shared__ int xrow[BN];
  const int tid = threadIdx.x, g = blockIdx.z;
  int lo = 0, hi = a.T;
  if (a.group_off) {
    lo = a.group_off[g];
    hi = a.group_off[g + 1];
  }
  const int t0 = lo + blockIdx.y * BN;
  if (t0 >= hi) return;
  const int f0 = blockIdx.x * BM;
  const unsigned short* W = a.w + (size_t)g * a.rows * a.cols;
  const float* X = a.x + (size_t)g * a.x_gstride;  // (one product per head: the group picks its columns)
  float* Y = a.y + (size_t)g * a.y_gstride;
  for (int i = tid; i < BN; i += 256) {
    const int it = t0 + i;
    int r = -1;
    if (it < hi) r = a.x_rows ? a.x_rows[it] / a.x_div : it;
    xrow[i] = r;
  }
  __syncthreads();
  const int wave = tid >> 6, lane = tid & 63, wm = wave & 1, wn = wave >> 1;
  const bool lead = FIRST && blockIdx.y == 0;
  const int lr = tid / KP, lk = (tid % KP) * 8;  // this thread stages 8 consecutive k of rows lr + RP i of both tiles
  const int K = a.cols;
  const unsigned short* wp[PW];
  const float* xp[PX];
#pragma unroll
  for (int i = 0; i < PW; ++i) {  // (rows and items beyond the last: the first one's values, never stored)
    const int frow = f0 + lr + RP * i;
    wp[i] = W + (size_t)(frow < a.rows ? frow : 0) * K;
  }
#pragma unroll
  for (int j = 0; j < PX; ++j) {
    const int xr = xrow[lr + RP * j];
    xp[j] = X + (size_t)(xr >= 0 ? xr : 0) * a.ldx;
  }
  struct Step {
    u32x4 w[PW];
    f32x4 x[PX][2];
  };
  // a step's pieces; columns beyond K as zeros (a step beyond the last reads the first column's pieces)
  auto fetch = [&](Step& r, int k0) __attribute__((always_inline)) {
    const int k = k0 + lk;
    if (VEC) {
      const bool in = k < K;
      const int kc = in ? k : 0;
#pragma unroll
      for (int i = 0; i < PW; ++i) r.w[i] = *reinterpret_cast<const u32x4*>(wp[i] + kc);
#pragma unroll
      for (int j = 0; j < PX; ++j) {
        r.x[j][0] = *reinterpret_cast<const f32x4*>(xp[j] + kc);
        r.x[j][1] = *reinterpret_cast<const f32x4*>(xp[j] + kc + 4);
      }
    } else {
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        unsigned short wv[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) wv[e] = k + e < K ? wp[i][k + e] : (unsigned short)0;
#pragma unroll
        for (int e = 0; e < 4; ++e) r.w[i][e] = wv[2 * e] | ((unsigned)wv[2 * e + 1] << 16);
      }
#pragma unroll
      for (int j = 0; j < PX; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) r.x[j][e >> 2][e & 3] = k + e < K ? xp[j][k + e] : 0.0f;
    }
  };
  f32x16 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  auto stage = [&](Step& r, int buf, int k0) __attribute__((always_inline)) {
    const bool in = !VEC || k0 + lk < K;  // (VEC: a piece is inside or outside as a whole)
#pragma unroll
    for (int i = 0; i < PW; ++i) *reinterpret_cast<u32x4*>(&Ws[buf][lr + RP * i][lk]) = in ? r.w[i] : u32x4{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < PX; ++j) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = in ? r.x[j][e >> 2][e & 3] : 0.0f;
#pragma unroll
      for (int t = 0; t < TERMS + (FIRST ? 1 : 0); ++t) {
        if (t == TERMS && !(lead && lr + RP * j < 32)) break;
        bf16x8 p;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          p[e] = (__bf16)x[e];
          if (t + 1 < TERMS + (FIRST ? 1 : 0)) x[e] -= (float)p[e];  // exact: the remainder of an FP32 value after its leading 8 bits
        }
        *reinterpret_cast<bf16x8*>(t < TERMS ? &Xs[buf][t < TERMS ? t : 0][lr + RP * j][lk] : &Xe[buf][FIRST ? (lr + RP * j) & 31 : 0][lk]) = p;
      }
    }
  };
  auto multiply = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      const int kk = ks * 16 + (lane >> 5) * 8;
      bf16x8 af[WM];
#pragma unroll
      for (int i = 0; i < WM; ++i) af[i] = *reinterpret_cast<const bf16x8*>(&Ws[buf][(wm * WM + i) * 32 + (lane & 31)][kk]);
#pragma unroll
      for (int t = TERMS - 1; t >= 0; --t) {  // small terms first
#pragma unroll
        for (int j = 0; j < WN; ++j) {
          const bf16x8 bfr = *reinterpret_cast<const bf16x8*>(&Xs[buf][t][(wn * WN + j) * 32 + (lane & 31)][kk]);
#pragma unroll
          for (int i = 0; i < WM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bfr, acc[i][j], 0, 0, 0);
        }
      }
    }
    if (FIRST && lead && wn == 0) {  // (a loop of its own: the one above keeps its schedule)
#pragma unroll
      for (int ks = 0; ks < BK / 16; ++ks) {
        const int kk = ks * 16 + (lane >> 5) * 8;
        const bf16x8 bfr = *reinterpret_cast<const bf16x8*>(&Xe[buf][FIRST ? lane & 31 : 0][kk]);
#pragma unroll
        for (int i = 0; i < WM; ++i)
          acc[i][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              *reinterpret_cast<const bf16x8*>(&Ws[buf][(wm * WM + i) * 32 + (lane & 31)][kk]), bfr, acc[i][0], 0, 0, 0);
      }
    }
  };
  // DEPTH steps' loads in flight: the one behind the step in LDS has arrived or is about to, the DEPTH-th after it is asked for
  // now (four instead of two gain nothing)
  constexpr int DEPTH = 2;
  Step r[DEPTH];
#pragma unroll
  for (int u = 0; u < DEPTH; ++u) fetch(r[u], u * BK);
  stage(r[0], 0, 0);
  __syncthreads();
  const int steps = (K + BK - 1) / BK;  // (rounded up to DEPTH: steps beyond the last multiply zeros)
  for (int st = 0; st < steps; st += DEPTH) {
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      const int k0 = (st + u) * BK, buf = u & (NB - 1);
      fetch(r[u], k0 + DEPTH * BK);
      __builtin_amdgcn_sched_barrier(0);
      multiply(buf);
      __builtin_amdgcn_sched_barrier(0);
      if (NB == 1) __syncthreads();
      stage(r[(u + 1) % DEPTH], buf ^ (NB - 1), k0 + BK);  // (NB == 2: its last readers are in front of the barrier of the step before)
      __syncthreads();
    }
  }
  dense_store<WM, WN>(a, acc, Y, f0 + wm * WM * 32, t0 + wn * WN * 32, hi, lane, reinterpret_cast<float*>(tiles) + wave * dense_store_floats(WM));
}

template <int N>
__device__ __forceinline__ void dma_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// One matrix, one term, items whose bf16 values lie in a plane [items][cols] already (dense_rows_kernel), whole steps of 64 columns.
// NWM x NWN waves, 32 WM features x 32 WN items each. Workgroups walk panels of eight item tiles, a contiguous range of tiles per XCD
// (as in the f16 GEMM of quantized matrices). Both sides go from memory to LDS directly, NS - 1 steps ahead;
// the loop has no other loads, so that waiting for all but the last NS - 2 steps' pieces is waiting for the step in hand.
// FIRST: the first 32 items' second terms join after every `join` products of 16 columns, where the tile of the kernel above that this
// launch would have taken has them: the same bits.
template <int NWM, int NWN, int WM, int WN, int NS, bool FIRST>
__global__ __launch_bounds__(64 * NWM * NWN, 2) void dense_plane_kernel(const DenseArgs a, int mtiles, int ntiles, int join) {
  constexpr int NW = NWM * NWN, BM = 32 * WM * NWM, BN = 32 * WN * NWN, ROWS = BM + BN + (FIRST ? 32 : 0), STAGE = ROWS * 128;
  constexpr int IW = BM / 8 / NW, IX = BN / 8 / NW;  // pieces of 8 rows x 64 columns that a wave fetches
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "");
  extern __shared__ __attribute__((aligned(16))) unsigned char dlds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave % NWM, wn = wave / NWM;
  constexpr int PANEL = 8;
  const int total = mtiles * ntiles, per8 = total >> 3, rem8 = total & 7, xcd = blockIdx.x & 7, at = blockIdx.x >> 3;
  const int v = xcd * per8 + (xcd < rem8 ? xcd : rem8) + at;
  const int panel = v / (PANEL * mtiles), in_panel = v - panel * PANEL * mtiles;
  const int width = ntiles - PANEL * panel < PANEL ? ntiles - PANEL * panel : PANEL;
  const int t0 = (PANEL * panel + in_panel % width) * BN, f0 = in_panel / width * BM;
  const int K = a.cols, hi = a.T;
  const bool lead = FIRST && t0 == 0;
  // row r of a stage lies at 128 r, its 16-byte piece q at q ^ (r / 2 & 7): the 16 rows of a fragment read cover the 64 banks once
  const int lr = lane >> 3;
  unsigned wo[IW], xo[IX], eo = 0;
#pragma unroll
  for (int i = 0; i < IW; ++i) {  // (rows and items beyond the last: the first one's values, never stored)
    const int row = (wave * IW + i) * 8 + lr, r = f0 + row;
    wo[i] = ((unsigned)(r < a.rows ? r : 0) * (unsigned)K + (((lane & 7) ^ ((row >> 1) & 7)) << 3)) * 2u;
  }
#pragma unroll
  for (int j = 0; j < IX; ++j) {
    const int row = (wave * IX + j) * 8 + lr, r = t0 + row;
    xo[j] = ((unsigned)(r < hi ? r : 0) * (unsigned)K + (((lane & 7) ^ ((row >> 1) & 7)) << 3)) * 2u;
  }
  if (FIRST) {
    const int row = (wave & 3) * 8 + lr;
    eo = ((unsigned)(row < a.T ? row : 0) * (unsigned)K + (((lane & 7) ^ ((row >> 1) & 7)) << 3)) * 2u;
  }
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)dlds;
  const int steps = K / 64;
  auto fetch = [&](int st, int slot) __attribute__((always_inline)) {  // (a step beyond the last: the last one again, never read)
    const size_t k = (size_t)(st < steps ? st : steps - 1) * 128;
    const unsigned b = lds0 + slot * STAGE;
    const char* wb = reinterpret_cast<const char*>(a.w) + k;
    const char* xb = reinterpret_cast<const char*>(a.plane) + k;
#pragma unroll
    for (int i = 0; i < IW; ++i) tl_lds_load16(b + (wave * IW + i) * 1024, wo[i], wb);
#pragma unroll
    for (int j = 0; j < IX; ++j) tl_lds_load16(b + BM * 128 + (wave * IX + j) * 1024, xo[j], xb);
    if (FIRST && lead) tl_lds_load16(b + (BM + BN) * 128 + (wave & 3) * 1024, eo, xb + (size_t)a.T * K * 2);
  };
  f32x16 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  const int fr = lane & 31, sw = (fr >> 1) & 7;
  auto second = [&](const unsigned char* b, int from, int to) __attribute__((always_inline)) {
    for (int ks = from; ks < to; ++ks) {
      const int q = ((2 * ks + (lane >> 5)) ^ sw) << 4;
      const bf16x8 x = *reinterpret_cast<const bf16x8*>(b + (BM + BN + fr) * 128 + q);
#pragma unroll
      for (int i = 0; i < WM; ++i)
        acc[i][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(b + ((wm * WM + i) * 32 + fr) * 128 + q), x, acc[i][0], 0, 0, 0);
    }
  };
#pragma unroll
  for (int st = 0; st < NS - 1; ++st) fetch(st, st);
  int slot = 0;
  for (int st = 0; st < steps; ++st) {
    if (FIRST && lead) dma_wait<(IW + IX + 1) * (NS - 2)>();
    else dma_wait<(IW + IX) * (NS - 2)>();
    __syncthreads();  // the step has arrived for all waves, and all have left the slot of the step before
    fetch(st + NS - 1, slot == 0 ? NS - 1 : slot - 1);
    const unsigned char* b = dlds + slot * STAGE;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int q = ((2 * ks + (lane >> 5)) ^ sw) << 4;
      bf16x8 af[WM], bf[WN];
#pragma unroll
      for (int i = 0; i < WM; ++i) af[i] = *reinterpret_cast<const bf16x8*>(b + ((wm * WM + i) * 32 + fr) * 128 + q);
#pragma unroll
      for (int j = 0; j < WN; ++j) bf[j] = *reinterpret_cast<const bf16x8*>(b + (BM + (wn * WN + j) * 32 + fr) * 128 + q);
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int i = 0; i < WM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
      if (FIRST && lead && wn == 0 && (ks & 1)) {  // (behind the products that the kernel above has in a step)
        if (join == 2) second(b, ks - 1, ks + 1);
        else if (ks == 3) second(b, 0, 4);
      }
    }
    slot = slot == NS - 1 ? 0 : slot + 1;
  }
  static_assert(NS * STAGE >= NW * dense_store_floats(WM) * 4, "");
  dma_wait<0>();
  __syncthreads();  // (the stages have been read and no piece is on its way)
  dense_store<WM, WN>(a, acc, a.y, f0 + wm * WM * 32, t0 + wn * WN * 32, hi, lane, reinterpret_cast<float*>(dlds) + wave * dense_store_floats(WM));
}

// x[T][ldx] -> bf16 [T][cols], and behind it the second terms of the first `second` rows; eight columns a thread
__global__ __launch_bounds__(256) void dense_rows_kernel(const float* __restrict__ x, int ldx, int T, int cols, int second,
                                                         unsigned short* __restrict__ plane) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i >= (long long)T * cols) return;
  const int t = (int)(i / cols), c = (int)(i - (long long)t * cols);
  const f32x4 a = *reinterpret_cast<const f32x4*>(x + (size_t)t * ldx + c), b = *reinterpret_cast<const f32x4*>(x + (size_t)t * ldx + c + 4);
  bf16x8 hi, lo;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float f = e < 4 ? a[e] : b[e - 4];
    hi[e] = (__bf16)f;
    lo[e] = (__bf16)(f - (float)hi[e]);
  }
  *reinterpret_cast<bf16x8*>(plane + i) = hi;
  if (t < second) *reinterpret_cast<bf16x8*>(plane + (size_t)T * cols + i) = lo;
}

// RW rows per wave, 4 waves per workgroup: 2 x RW sixteen-byte weight loads in flight per lane (tl_bf16.h)
template <int RW>
__global__ __launch_bounds__(256) void dense_gemv_kernel(const unsigned short* __restrict__ W, int rows, int cols,
                                                         const float* __restrict__ x, float* __restrict__ y, int vec,
                                                         float softcap, const GemvActArgs act, int x_stride, int y_stride) {
  const int lane = threadIdx.x & 63;
  const int row0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * RW;
  if (row0 >= rows) return;
  // blockIdx.y: the head of a one-product-per-head launch (its matrix, its columns of x, its piece of y)
  W += (size_t)blockIdx.y * rows * cols;
  x += (size_t)blockIdx.y * x_stride;
  y += (size_t)blockIdx.y * y_stride;
  float out[RW];
  tl_wave_dot_rows<RW>(W + (size_t)row0 * cols, (size_t)cols, rows - row0, x, cols, vec != 0, lane, out);
  if (lane == 0) {
#pragma unroll
    for (int r = 0; r < RW; ++r)
      if (row0 + r < rows) {
        if (act.bias) out[r] += act.bias[row0 + r];
        float v = softcap > 0.0f ? softcap * tanhf(out[r] / softcap) : out[r];
        if (act.act && row0 + r >= act.act_from && (act.act_to <= 0 || row0 + r < act.act_to)) v = tl_act_apply(act.act, v, act.act_p, act.act_q);
        y[row0 + r] = v;
      }
  }
}

// One token: x_out = x + y / rms(y) * (1 + norm_w) in every workgroup (one of them writes it), out = W x_out, columns 512 NP. A row a wave
// (more where a launch has more rows than waves), its NP 16-byte pieces asked for with the vectors. A residual norm of its own is a launch of
// one workgroup that the product waits for: 3072 x 2048 4.9 + 4.4 us, here 4.8. A token of six layers, us, with launches of their own / carried:
// 512 columns 201 / 193, 1024 216 / 203, 1536 249 / 241, 2048 268 / 255, 2560 317 / 302, 3072 328 / 319, 3584 388 / 372, 4096 413 / 394, 4608 495 /
// 468, 5120 533 / 502. Ten pieces are 124 of the 128 registers that a thread of sixteen waves has, eleven spill: wider rows keep the two
// launches, and so do rows that end inside a piece (the kernel has no tail).
constexpr int RESID_PIECES = 10;
template <int NP>
__global__ __launch_bounds__(1024) void dense_gemv_resid_kernel(const unsigned short* __restrict__ W, const float* __restrict__ x, const float* __restrict__ y,
                                                                const float* __restrict__ nw, float* __restrict__ x_out, float* __restrict__ out,
                                                                int rows, float eps, int nthr, int grid) {
  constexpr int COLS = 512 * NP, Q = COLS / 4;
  __shared__ __attribute__((aligned(16))) float xs[COLS];  // four values each: even pieces, then odd ones (a lane reads two neighbours)
  __shared__ float red[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = nthr >> 6;
  f32x4 xv[2], yv[2], nv[2];  // (two pieces a thread are enough: the launcher)
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int q = tid + k * nthr < Q ? tid + k * nthr : Q - 1;
    yv[k] = reinterpret_cast<const f32x4*>(y)[q];
    xv[k] = reinterpret_cast<const f32x4*>(x)[q];
    nv[k] = reinterpret_cast<const f32x4*>(nw)[q];
  }
  int r = blockIdx.x * nwaves + wave;
  uint4 w[NP];
  auto load = [&]() __attribute__((always_inline)) {
    const unsigned short* wr = W + (size_t)(r < rows ? r : rows - 1) * COLS + lane * 8;
#pragma unroll
    for (int p = 0; p < NP; ++p) w[p] = tl_ldw(wr + 512 * p);
  };
  load();
  float ss = 0.0f;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const float s = (yv[k][0] * yv[k][0] + yv[k][1] * yv[k][1]) + (yv[k][2] * yv[k][2] + yv[k][3] * yv[k][3]);
    ss += tid + k * nthr < Q ? s : 0.0f;
  }
  ss = tl_wave_sum(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  const float part = red[lane & 15];
  const float inv = 1.0f / sqrtf(tl_row16_sum((lane & 15) < nwaves ? part : 0.0f) / (float)COLS + eps);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int q = tid + k * nthr;
    if (q < Q) {
      const f32x4 v = xv[k] + yv[k] * inv * (1.0f + nv[k]);
      reinterpret_cast<f32x4*>(xs)[(q >> 1) + (q & 1) * (Q / 2)] = v;
      if (blockIdx.x == 0) reinterpret_cast<f32x4*>(x_out)[q] = v;
    }
  }
  __syncthreads();
  for (;;) {
    float acc = 0.0f;
#pragma unroll
    for (int p = 0; p < NP; ++p)
      acc = tl_dot8(w[p], reinterpret_cast<const float4*>(xs)[lane + 64 * p], reinterpret_cast<const float4*>(xs)[Q / 2 + lane + 64 * p], acc);
    acc = tl_wave_sum(acc);
    if (lane == 0 && r < rows) out[r] = acc;
    r += grid * nwaves;
    if (r >= rows) break;
    load();
  }
}

template <int NWM, int NWN, int WM, int WN, int NS, bool FIRST>
int dense_plane_go(const DenseArgs& a, int join, hipStream_t s) {
  constexpr int BM = 32 * WM * NWM, BN = 32 * WN * NWN, LDS = NS * 128 * (BM + BN + (FIRST ? 32 : 0));
  static TlDeviceOnce lds_raised;
  auto kernel = dense_plane_kernel<NWM, NWN, WM, WN, NS, FIRST>;
  TL_TRY(tl_raise_lds_limit(kernel, LDS, lds_raised));
  const int mt = (a.rows + BM - 1) / BM, nt = (a.T + BN - 1) / BN;
  kernel<<<mt * nt, 64 * NWM * NWN, LDS, s>>>(a, mt, nt, join);
  TL_HIP(hipGetLastError());
  return 0;
}

int dense_plane_run(const DenseArgs& a, int waves, bool big, hipStream_t s) {
  const bool first = a.exact_items > 0;  // (the kernels multiply the second terms of 32 items whatever their number)
  const int join = big ? 2 : 4;
  const long long pieces = (long long)a.T * a.cols / 8;
  dense_rows_kernel<<<dim3((unsigned)((pieces + 255) / 256)), 256, 0, s>>>(a.x, a.ldx, a.T, a.cols, first ? 32 : 0, a.plane);
  TL_HIP(hipGetLastError());
  if (waves == 8) return first ? dense_plane_go<4, 2, 1, 2, 4, true>(a, join, s) : dense_plane_go<4, 2, 1, 2, 4, false>(a, join, s);
  return first ? dense_plane_go<2, 2, 2, 2, 2, true>(a, join, s) : dense_plane_go<2, 2, 2, 2, 2, false>(a, join, s);
}
// whole steps, the items and 32 second terms inside the plane, 32-bit byte offsets in it and in the matrix
bool dense_plane_fits(const DenseArgs& a) {
  return a.cols % 64 == 0 && (size_t)a.rows * a.cols < ((size_t)1 << 31) && ((size_t)a.T + 32) * a.cols < ((size_t)1 << 31) &&
         ((size_t)a.T + 32) * a.cols <= a.plane_room;
}
long long dense_big_tiles(int rows, long long items) { return ((rows + 127) / 128) * ((items + 127) / 128); }
// The plane kernel takes the launches whose 128 x 128 tiles occupy half of the CUs or more and are long enough to pay for the
// conversion (rows x columns x items, without / with it, conversion included: 10304 x 2048 x 1999 174 / 114 us, x 512 56 / 36,
// x 200 36 / 25; 4096 x 2048 x 1999 66 / 45, x 1024 46 / 30; 2048 x 4096 x 1999 80 / 51, x 1024 47 / 43; 4096 x 1024 x 1024 26 / 20;
// many rows and a tile of items that is half full 32000 x 2048 x 64 26.5 / 26.1, 65536 x 1024 x 64 29.7 / 27.1, 128256 x 4096 x 100
// 290 / 240; on the line 4096 x 2048 x 512 26.3 / 25.8 and 2048 x 2048 x 1024 26.4 / 26.5; below 1024 x 1024 x 1999 16 / 18,
// 2048 x 4096 x 512 33 / 39).
bool dense_plane_pays(const DenseArgs& a, int cus) {
  const long long tiles = dense_big_tiles(a.rows, a.T);
  return dense_plane_fits(a) && 2 * tiles >= cus && tiles * a.cols > 1024ll * cus;
}

}  // namespace

int tl_launch_dense_gemm(const DenseArgs& a, hipStream_t s) {
  TL_REQUIRE(a.w && a.x && a.y && a.rows > 0 && a.cols > 0 && a.T > 0, "dense gemm: bad arguments");
  TL_REQUIRE(a.terms == 1 || a.terms == 3, "dense gemm: terms must be 1 or 3 (got %d)", a.terms);
  TL_REQUIRE(!a.x_rows || a.x_div >= 1, "dense gemm: x_div must be >= 1");
  TL_REQUIRE(a.exact_items <= 0 || (a.exact_items <= 32 && !a.group_off && a.groups <= 1 && !a.x_rows),
             "dense gemm: %d first items with two terms (at most 32, one matrix)", a.exact_items);
  TL_REQUIRE(!a.glu || (a.rows & 1) == 0, "dense gemm: gated pairs need an even number of rows (got %d)", a.rows);
  const int groups = a.groups > 0 ? a.groups : 1;
  TL_REQUIRE(groups == 1 || a.group_off || (a.x_gstride >= 0 && a.y_gstride > 0 && !a.x_rows && !a.y_rows),
             "dense gemm: groups without group_off or per-head column strides");
  TL_REQUIRE(!a.act || !a.glu, "dense gemm: an activation and a gated unit in one epilogue");
  TL_REQUIRE(!a.bias || (!a.glu && groups == 1), "dense gemm: a bias with a gated unit or several matrices");
  // 128 x 128 tiles when there is enough of both sides to fill them (grouped launches: tokens per group on average)
  const long long per_group = a.group_off ? (long long)a.T / groups : a.T;
  // Measured: a dense launch needs a 128 x 128 tile a CU (192 tiles, 6144 rows, 4096 columns, 512 tokens: 78 us against 75 in
  // small ones with one term, 153 against 126 with three). Where its small tiles are four a CU, one round, large ones need long
  // rows too, so that a tile's way in and out is short beside its products: 256 tiles, large / small, 512 columns 22.1 / 16.4 us
  // with one term and 32.2 / 23.7 with three, 1024 29.3 / 25.9 and 48.4 / 41.7, 2048 43.7 / 42.1 and 82.9 / 77.5, 4096 74 / 78 and
  // 148 / 149, 14336 224 / 345 and 483 / 511. Beyond, small tiles start a second round: 264 tiles of 2048 columns 56 / 63 and
  // 87 / 91, 384 of 1024 32 / 36 and 53 / 59, 448 of 4096 107 / 154 and 200 / 265. Either tile gives the same bits (but
  // for exact_items, whose second terms join after each step's products). The experts'
  // grouped launches, whose small tiles are mostly half-empty, gain from large ones with one term (221 -> 193 us) and lose with
  // three (356 -> 413 us).
  const long long small_tiles = ((a.rows + 63) / 64) * ((per_group + 63) / 64) * groups;
  const long long big_tiles = dense_big_tiles(a.rows, per_group) * groups;
  const char* force = getenv("TL_DENSE_TILE");  // 64 / 128: tests and A/B runs pick the tile themselves
  const bool big = force ? atoi(force) == 128
                         : a.rows >= 256 && (a.group_off ? a.terms == 1 && per_group >= 96
                                                         : big_tiles >= tl_num_cus() && (small_tiles > 4 * tl_num_cus() || a.cols >= 4096));
  const bool first = a.exact_items > 0 && a.terms == 1;
  // wide loads: every matrix, row and piece of eight columns at 16 bytes
  const bool vec = (a.cols & 7) == 0 && (a.ldx & 3) == 0 && ((size_t)a.x & 15) == 0 && ((size_t)a.w & 15) == 0 && (a.x_gstride & 3) == 0;
  // the plane kernel: one tile a CU: eight waves and three steps ahead; more: two workgroups of four waves, which fill each other's
  // waits (256 tiles 30.3 / 32.5 us, 324 tiles 44.8 / 36.4). TL_DENSE_TILE=64, 128: the kernel above.
  if (a.plane && a.terms == 1 && groups == 1 && !a.group_off && !a.x_rows && vec && !force && dense_plane_pays(a, tl_num_cus()))
    return dense_plane_run(a, big_tiles <= tl_num_cus() ? 8 : 4, big, s);
  const int BM = big ? 128 : 64, BN = big ? 128 : 64;
  dim3 grid((a.rows + BM - 1) / BM, (a.T + BN - 1) / BN, groups);
  TL_REQUIRE(grid.y <= 65535 && grid.z <= 65535, "dense gemm: launch too large");
#define DENSE(T, W, F) (vec ? dense_gemm_kernel<T, W, W, true, F><<<grid, 256, 0, s>>>(a) : dense_gemm_kernel<T, W, W, false, F><<<grid, 256, 0, s>>>(a))
  if (big) {
    if (first) DENSE(1, 2, true);
    else if (a.terms == 1) DENSE(1, 2, false);
    else DENSE(3, 2, false);
  } else {
    if (first) DENSE(1, 1, true);
    else if (a.terms == 1) DENSE(1, 1, false);
    else DENSE(3, 1, false);
  }
#undef DENSE
  TL_HIP(hipGetLastError());
  return 0;
}

static int launch_gemv(const uint16_t* w, int groups, int rows, int cols, const float* x, int x_stride, float* y, int y_stride,
                       float softcap, const GemvActArgs& act, hipStream_t s) {
  TL_REQUIRE(w && x && y && rows > 0 && cols > 0 && groups > 0 && groups <= 65535, "dense gemv: bad arguments");
  // 16-byte loads need every head's matrix and columns aligned as the first one's
  const int vec = (cols & 7) == 0 && ((size_t)x & 15) == 0 && ((size_t)w & 15) == 0 &&
                  (groups == 1 || ((x_stride & 3) == 0 && (((size_t)rows * cols) & 7) == 0));
  // rows per wave: as many as still leave every CU a few workgroups
  const int cus = tl_num_cus();
  const long long all = (long long)rows * groups;
  if (all >= 16 * 4 * cus) dense_gemv_kernel<4><<<dim3((rows + 15) / 16, groups), 256, 0, s>>>(w, rows, cols, x, y, vec, softcap, act, x_stride, y_stride);
  else if (all >= 8 * 4 * cus) dense_gemv_kernel<2><<<dim3((rows + 7) / 8, groups), 256, 0, s>>>(w, rows, cols, x, y, vec, softcap, act, x_stride, y_stride);
  else dense_gemv_kernel<1><<<dim3((rows + 3) / 4, groups), 256, 0, s>>>(w, rows, cols, x, y, vec, softcap, act, x_stride, y_stride);
  TL_HIP(hipGetLastError());
  return 0;
}

int tl_launch_dense_gemv(const uint16_t* w, int rows, int cols, const float* x, float* y, hipStream_t s, float softcap) {
  return launch_gemv(w, 1, rows, cols, x, 0, y, 0, softcap, GemvActArgs{}, s);
}

int tl_launch_dense_gemv_act(const uint16_t* w, int rows, int cols, const float* x, float* y, const GemvActArgs& act, hipStream_t s) {
  return launch_gemv(w, 1, rows, cols, x, 0, y, 0, 0.0f, act, s);
}

int tl_launch_dense_gemv_heads(const uint16_t* w, int groups, int rows, int cols, const float* x, int x_stride, float* y,
                               int y_stride, hipStream_t s) {
  return launch_gemv(w, groups, rows, cols, x, x_stride, y, y_stride, 0.0f, GemvActArgs{}, s);
}

namespace {
std::atomic<long long> g_resid_products{0};  // tl_debug_resid_products
template <int NP = RESID_PIECES>
void gemv_resid_go(const uint16_t* w, int rows, int cols, const float* x, const float* y, const float* norm_w, float eps, float* x_out, float* out, int grid,
                   int waves, hipStream_t s) {
  if (cols == 512 * NP) dense_gemv_resid_kernel<NP><<<grid, 64 * waves, 0, s>>>(w, x, y, norm_w, x_out, out, rows, eps, 64 * waves, grid);
  else if constexpr (NP > 1) gemv_resid_go<NP - 1>(w, rows, cols, x, y, norm_w, eps, x_out, out, grid, waves, s);
}
}  // namespace
bool tl_dense_gemv_resid_fits(const uint16_t* w, int rows, int cols) {
  return rows > 0 && cols > 0 && cols % 512 == 0 && cols <= 512 * RESID_PIECES && ((size_t)w & 15) == 0;
}
int tl_launch_dense_gemv_resid(const uint16_t* w, int rows, int cols, const float* x, const float* y, const float* norm_w, float eps, float* x_out,
                               float* out, hipStream_t s) {
  TL_REQUIRE(w && x && y && norm_w && x_out && out && x_out != x && tl_dense_gemv_resid_fits(w, rows, cols) &&
                 (((size_t)x | (size_t)y | (size_t)norm_w | (size_t)x_out) & 15) == 0, "dense gemv: bad arguments of a product behind a residual norm");
  // a row a wave and a workgroup a CU where that is at most sixteen waves; at least two pieces of the vectors a thread
  const int cus = tl_num_cus(), least = cols / 512 > 4 ? cols / 512 : 4;
  int waves = (rows + cus - 1) / cus;
  waves = waves < least ? least : waves > 16 ? 16 : waves;
  int grid = (rows + waves - 1) / waves;
  if (grid > cus) grid = cus;
  gemv_resid_go(w, rows, cols, x, y, norm_w, eps, x_out, out, grid, waves, s);
  TL_HIP(hipGetLastError());
  g_resid_products.fetch_add(1, std::memory_order_relaxed);
  return 0;
}
extern "C" int tl_debug_resid_products(long long* count_out) {
  TL_REQUIRE(count_out, "tl_debug_resid_products: null argument");
  *count_out = g_resid_products.load(std::memory_order_relaxed);
  return 0;
}

extern "C" int tl_dense_matmul(const void* w_bf16_dev, int rows, int cols, const float* x_dev, float* y_dev, int num_tokens,
                               int terms, void* stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (terms == 0) {
    TL_REQUIRE(num_tokens == 1, "tl_dense_matmul: terms 0 (FP32 GEMV) takes one token, not %d", num_tokens);
    return tl_launch_dense_gemv(static_cast<const uint16_t*>(w_bf16_dev), rows, cols, x_dev, y_dev, s);
  }
  DenseArgs a = {};
  a.w = static_cast<const uint16_t*>(w_bf16_dev);
  a.rows = rows;
  a.cols = cols;
  a.x = x_dev;
  a.ldx = cols;
  a.y = y_dev;
  a.ldy = rows;
  a.T = num_tokens;
  a.terms = terms;
  return tl_launch_dense_gemm(a, s);
}

extern "C" int tl_dense_matmul_act(const void* w_bf16_dev, int rows, int cols, const float* x_dev, float* y_dev, int num_tokens,
                                   int terms, int act, float act_p, float act_q, int act_from, void* stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  TL_REQUIRE(act >= TL_ACT_NONE && act <= TL_ACT_GELU, "tl_dense_matmul_act: activation kind %d", act);
  if (terms == 0) {
    TL_REQUIRE(num_tokens == 1, "tl_dense_matmul_act: terms 0 (FP32 GEMV) takes one token, not %d", num_tokens);
    return tl_launch_dense_gemv_act(static_cast<const uint16_t*>(w_bf16_dev), rows, cols, x_dev, y_dev,
                                    GemvActArgs{act, act_from, act_p, act_q, 0, nullptr}, s);
  }
  DenseArgs a = {};
  a.w = static_cast<const uint16_t*>(w_bf16_dev);
  a.rows = rows;
  a.cols = cols;
  a.x = x_dev;
  a.ldx = cols;
  a.y = y_dev;
  a.ldy = rows;
  a.T = num_tokens;
  a.terms = terms;
  a.act = act;
  a.act_from = act_from;
  a.act_p = act_p;
  a.act_q = act_q;
  return tl_launch_dense_gemm(a, s);
}

extern "C" int tl_dense_matmul_bias(const void* w_bf16_dev, int rows, int cols, const float* x_dev, float* y_dev, int num_tokens,
                                    int terms, const float* bias_dev, int act, float act_p, float act_q, int act_from, int act_to,
                                    void* stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  TL_REQUIRE(act >= TL_ACT_NONE && act <= TL_ACT_SIGMOID_POWER, "tl_dense_matmul_bias: activation kind %d", act);
  if (terms == 0) {
    TL_REQUIRE(num_tokens == 1, "tl_dense_matmul_bias: terms 0 (FP32 GEMV) takes one token, not %d", num_tokens);
    return tl_launch_dense_gemv_act(static_cast<const uint16_t*>(w_bf16_dev), rows, cols, x_dev, y_dev,
                                    GemvActArgs{act, act_from, act_p, act_q, act_to, bias_dev}, s);
  }
  DenseArgs a = {};
  a.w = static_cast<const uint16_t*>(w_bf16_dev);
  a.rows = rows;
  a.cols = cols;
  a.x = x_dev;
  a.ldx = cols;
  a.y = y_dev;
  a.ldy = rows;
  a.T = num_tokens;
  a.terms = terms;
  a.bias = bias_dev;
  a.act = act;
  a.act_from = act_from;
  a.act_to = act_to;
  a.act_p = act_p;
  a.act_q = act_q;
  return tl_launch_dense_gemm(a, s);
}

extern "C" int tl_dense_matmul_heads(const void* w_bf16_dev, int groups, int rows, int cols, const float* x_dev, int ldx,
                                     int x_stride, float* y_dev, int ldy, int y_stride, int num_tokens, int terms, void* stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (terms == 0) {
    TL_REQUIRE(num_tokens == 1, "tl_dense_matmul_heads: terms 0 (FP32 GEMV) takes one token, not %d", num_tokens);
    return tl_launch_dense_gemv_heads(static_cast<const uint16_t*>(w_bf16_dev), groups, rows, cols, x_dev, x_stride, y_dev,
                                      y_stride, s);
  }
  DenseArgs a = {};
  a.w = static_cast<const uint16_t*>(w_bf16_dev);
  a.rows = rows;
  a.cols = cols;
  a.x = x_dev;
  a.ldx = ldx;
  a.y = y_dev;
  a.ldy = ldy;
  a.T = num_tokens;
  a.terms = terms;
  a.groups = groups;
  a.x_gstride = x_stride;
  a.y_gstride = y_stride;
  return tl_launch_dense_gemm(a, s);
}

extern "C" int tl_debug_dense_plane(const void* w_bf16_dev, int rows, int cols, const float* x_dev, int ldx, float* y_dev, int num_tokens,
                                    int exact_items, int waves, void* plane_dev, void* stream) {
  DenseArgs a = {};
  a.w = static_cast<const uint16_t*>(w_bf16_dev);
  a.rows = rows;
  a.cols = cols;
  a.x = x_dev;
  a.ldx = ldx;
  a.y = y_dev;
  a.ldy = rows;
  a.T = num_tokens;
  a.terms = 1;
  a.exact_items = exact_items;
  a.plane_room = ((size_t)num_tokens + 32) * cols;
  TL_REQUIRE(a.w && x_dev && y_dev && rows > 0 && cols > 0 && num_tokens > 0 && ldx >= cols && ldx % 4 == 0 &&
                 exact_items >= 0 && exact_items <= 32 && (waves == 4 || waves == 8) && dense_plane_fits(a) &&
                 (((size_t)w_bf16_dev | (size_t)x_dev | (size_t)plane_dev) & 15) == 0,
             "tl_debug_dense_plane: bad argument");
  if (!plane_dev) return tl_launch_dense_gemm(a, static_cast<hipStream_t>(stream));
  a.plane = static_cast<uint16_t*>(plane_dev);
  const char* tile = getenv("TL_DENSE_TILE");
  return dense_plane_run(a, waves, tile && atoi(tile) == 128, static_cast<hipStream_t>(stream));
}

extern "C" int tl_debug_dense_plane_taken(int rows, int cols, int num_tokens, long long room, int cus) {
  DenseArgs a = {};
  a.rows = rows;
  a.cols = cols;
  a.T = num_tokens;
  a.plane_room = (size_t)room;
  return dense_plane_pays(a, cus);
}
