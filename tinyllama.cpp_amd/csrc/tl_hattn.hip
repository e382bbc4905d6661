// Causal prefill attention over one FP32 cache, its products in f16 matrix instructions at the 32-bit grade (gfx950).
// Reference behaviour: cpu_attention.cpp:254-325 (causal softmax attention with 1 / (sum + 1e-9)), gpu_kernels.cu attention.
//
// The FP32 matrix instructions do 64 multiply-adds a cycle and SIMD, the f16 ones 512: a product of two-part numbers
// (x 2^k = hi + lo, 22 bits, lo lo left out) costs three of the latter and still leaves a factor of five. The FP32 kernel
// (tl_prefill.hip) was bound by its matrix cores: 3989 tokens of 24 heads of 128 in chunks of 512, 28 layers, took it 44 ms;
// the three kernels here take 16 ms of such chunks (of which the conversion 2.2, the sums 1.9; the whole prompt 136 -> 105 ms)
// and 12 of chunks of 2048 (0.7 and 1.0).
//   1. kv_planes_kernel cuts the cache rows of every kv head into 32-key tiles of two-part f16 in the order in which the
//      lanes of a matrix instruction take them (K: eight columns of one key; V: eight keys of one column, the keys in the
//      order in which the accumulator of K Q^T holds them, so that the probabilities never change lanes). One power of two
//      per tile brings its largest finite value to 2^14: a value is held to 2^-23 of itself and 2^-39 of its tile's largest.
//      Against float64 the output's error is 5e-8 of its weights times its values' size, the FP32 matrix kernel's 7e-8 (both sides
//      lose what the order of the sums gives); a row of a tile that is 2^20 times the others' size brings it to 1e-7, 2^24 to
//      1.3e-6. The sums of a tile and of the small products are kept apart, and the weights' 2^12 stands outside the
//      exponential: 8B prompts' logits 2.65e-6 -> 2.21e-6 off float64, for 1.7 % of the kernel's time (0 to 7 % over 70 shapes: 8 heads of
//      128 over 64, 64 tokens, 12.0 -> 12.9 us; two blocks of 32 columns in turn gain nothing back).
//   2. hattn_kernel: four waves, 128 rows (query, head of the kv head's group), tiles through a double-buffered LDS window
//      that all four waves read: one wave's operands straight from memory would need 85 bytes a cycle and CU. Two workgroups
//      a CU, so that one's softmax runs under the other's products. A row tile's keys are cut into up to 16 pieces.
//   3. hattn_combine_kernel sums the pieces of a row tile that has more than one, in order.
#include <math.h>

#include <atomic>

#include "tl_internal.h"
#include "tl_lanes.h"
#include "tl_lds.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));

namespace {

constexpr int HA_ROWS = 128, HA_MAX_SPLIT = 16, HA_MAX_SLOTS = 2048;
constexpr float LOG2E = 1.44269504088896340736f;
constexpr float HA_P_UNIT = 4096.f;  // probabilities are held times 2^12: their second part stays normal down to 2^-15
constexpr int HA_P_SPARE = 8;      // ... and to 2^-29 of a row's largest at worst: what they may give up for a tile of small values

__device__ __forceinline__ int acc_row(int e, int h) { return (e & 3) + 8 * (e >> 2) + 4 * h; }

// exponent k with max 2^k in [2^14, 2^15); values beyond what one factor can bring there are left smaller or larger
__device__ __forceinline__ int scale_exp(float max_abs) {
  const int k = 14 - (int)((__float_as_uint(max_abs) >> 23) & 255u) + 127;
  return k < -113 ? -113 : k > 60 ? 60 : k;
}
__device__ __forceinline__ float pow2i(int k) { return __uint_as_float((unsigned)(k + 127) << 23); }  // |k| <= 126
__device__ __forceinline__ void two_parts(const float (&x)[8], float f, half8& hi, half8& lo) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float v = x[i] * f;
    const _Float16 a = (_Float16)v;
    hi[i] = a;
    lo[i] = fabsf(v) < INFINITY ? (_Float16)(v - (float)a) : (_Float16)0.0f;
  }
}

struct HPlanesArgs {
  const float *kc, *vc;  // key rows kld floats apart, a head's part khs apart; value rows vld apart
  int kld, khs, vld, lo, len, nkv, tile0, tiles;  // rows lo .. len - 1; tiles tile0 .. tile0 + tiles - 1 (others' rows: zeros)
  _Float16* planes;      // [nkv][tiles][(KD + VD) * 64]: K then V fragments
  int* exps;             // [nkv][tiles][2]
};
template <int KD, int VD>
__global__ __launch_bounds__(256) void kv_planes_kernel(const HPlanesArgs a) {
  constexpr int PK = (KD + 63) / 64, PV = (VD + 63) / 64;  // fragments of each operand per thread
  __shared__ float red[8];
  const int tile = blockIdx.x, kvh = blockIdx.y, tid = threadIdx.x, p0 = (a.tile0 + tile) * 32;
  const float *kp = a.kc + (size_t)kvh * a.khs, *vp = a.vc + (size_t)kvh * VD;
  float k[PK][8], v[PV][8], mk = 0.f, mv = 0.f;
#pragma unroll
  for (int t = 0; t < PK; ++t) {
    const int f = tid + 256 * t, lane = f & 63, r = lane & 31, h = lane >> 5, g = f >> 6;
    f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = x;
    if (f < 4 * KD && p0 + r >= a.lo && p0 + r < a.len) {
      const float* src = kp + (size_t)(p0 + r) * a.kld + 16 * g + 8 * h;
      x = *reinterpret_cast<const f32x4*>(src);
      y = *reinterpret_cast<const f32x4*>(src + 4);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) k[t][i] = i < 4 ? x[i & 3] : y[i & 3];
  }
#pragma unroll
  for (int t = 0; t < PV; ++t) {
    const int f = tid + 256 * t, lane = f & 63, r = lane & 31, h = lane >> 5, g = f >> 6;
    const int j = g / (VD / 32), d = 32 * (g % (VD / 32)) + r;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int key = p0 + acc_row(8 * j + i, h);
      v[t][i] = f < 4 * VD && key >= a.lo && key < a.len ? vp[(size_t)key * a.vld + d] : 0.f;
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {  // (an infinity or a NaN spoils its own key only)
#pragma unroll
    for (int t = 0; t < PK; ++t)
      if (fabsf(k[t][i]) < INFINITY) mk = fmaxf(mk, fabsf(k[t][i]));
#pragma unroll
    for (int t = 0; t < PV; ++t)
      if (fabsf(v[t][i]) < INFINITY) mv = fmaxf(mv, fabsf(v[t][i]));
  }
  mk = tl_wave_max(mk);
  mv = tl_wave_max(mv);
  if ((tid & 63) == 0) {
    red[tid >> 6] = mk;
    red[4 + (tid >> 6)] = mv;
  }
  __syncthreads();
  const int ek = scale_exp(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
  const int ev = scale_exp(fmaxf(fmaxf(red[4], red[5]), fmaxf(red[6], red[7])));
  const size_t at = (size_t)kvh * a.tiles + tile;
  if (tid == 0) {
    a.exps[2 * at] = ek;
    a.exps[2 * at + 1] = ev;
  }
  _Float16* out = a.planes + at * ((KD + VD) * 64);
  const float fk = pow2i(ek), fv = pow2i(ev);
  half8 hi, lo;
#pragma unroll
  for (int t = 0; t < PK; ++t) {
    const int f = tid + 256 * t, lane = f & 63, g = f >> 6;
    if (f >= 4 * KD) break;
    two_parts(k[t], fk, hi, lo);
    *reinterpret_cast<half8*>(out + ((size_t)(2 * g) * 64 + lane) * 8) = hi;
    *reinterpret_cast<half8*>(out + ((size_t)(2 * g + 1) * 64 + lane) * 8) = lo;
  }
#pragma unroll
  for (int t = 0; t < PV; ++t) {
    const int f = tid + 256 * t, lane = f & 63, g = f >> 6;
    if (f >= 4 * VD) break;
    two_parts(v[t], fv, hi, lo);
    *reinterpret_cast<half8*>(out + KD * 64 + ((size_t)(2 * g) * 64 + lane) * 8) = hi;
    *reinterpret_cast<half8*>(out + KD * 64 + ((size_t)(2 * g + 1) * 64 + lane) * 8) = lo;
  }
}

// maximum of the two halves' lanes r and r + 32
__device__ __forceinline__ float half_max(float v) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
}

struct HAttnArgs {
  TlHattn x;
  const _Float16* planes;
  const int* exps;
  float* part;             // [slot][HA_ROWS][VD]
  float2* ml;              // [slot][HA_ROWS] (maximum in bits, sum)
  int group, tile0, tiles, splits, piece;
  float scale;             // times log2(e)
};
// first position that position i sees
__host__ __device__ __forceinline__ int first_key(const TlHattn& x, int i) {
  int lo = x.window > 0 && i - x.window + 1 > 0 ? i - x.window + 1 : 0;
  if (x.chunk > 0 && i - i % x.chunk > lo) lo = i - i % x.chunk;
  return lo;
}
// key tiles [lo, hi) of row tile rt (rows rt * 128 ..: row = query * group + head of the group)
struct TileRange {
  int lo, hi;
};
__host__ __device__ __forceinline__ TileRange row_tiles(const TlHattn& x, int group, int rt) {
  const int last = (rt * HA_ROWS + HA_ROWS - 1) / group;
  return {first_key(x, x.start_pos + rt * HA_ROWS / group) / 32, (x.start_pos + (last < x.T ? last : x.T - 1)) / 32 + 1};
}

// factor on a row's sum of values, whose weights are relative to 2^m and add up to l
__device__ __forceinline__ float finish(const TlHattn& x, int t, int head, float m, float l) {
  float f = 1.0f;
  if (x.sink) {  // one more key without a value
    const float sv = (x.sink_val ? x.sink_val[head] : 0.0f) * LOG2E, M = fmaxf(m, sv);
    f = __builtin_amdgcn_exp2f(m - M);
    l = l * f + __builtin_amdgcn_exp2f(sv - M);
  }
  f /= l + x.eps;
  return x.gate ? f / (1.0f + expf(-x.gate[(size_t)t * x.gate_ld + head])) : f;
}

template <int KD, int VD>
__global__ __launch_bounds__(256, 2) void hattn_kernel(const HAttnArgs a) {
  constexpr int DS = KD / 16, DB = VD / 32, TILE = (KD + VD) * 64, NLD = TILE / 8 / 256;
  __shared__ __attribute__((aligned(16))) _Float16 win[2][TILE];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5, wave = tid >> 6;
  // workgroup L runs on XCD L mod 8: with a multiple of eight kv heads every L2 holds the planes of its own ones; the row
  // tiles with the most keys first
  const int nkv = a.x.kv_heads;
  const int kvh = blockIdx.x % nkv, slot = blockIdx.x / nkv, split = slot % a.splits;
  const int rows = a.x.T * a.group, nrt = (rows + HA_ROWS - 1) / HA_ROWS, rt = nrt - 1 - slot / a.splits;
  const TileRange range = row_tiles(a.x, a.group, rt);
  const int nt = range.hi - range.lo, ns = (nt + a.piece - 1) / a.piece;
  if (split >= ns) return;
  const int t0 = range.lo + (int)((long long)nt * split / ns), t1 = range.lo + (int)((long long)nt * (split + 1) / ns);
  const int row = rt * HA_ROWS + wave * 32 + r;
  const int rq = (row < rows ? row : rows - 1) / a.group, head = kvh * a.group + (row < rows ? row : rows - 1) - rq * a.group;
  const int qpos = a.x.start_pos + rq, qlo = first_key(a.x, qpos);
  const int row0 = __builtin_amdgcn_readfirstlane(rt * HA_ROWS + wave * 32);
  const int wave_last = a.x.start_pos + min(row0 + 31, rows - 1) / a.group, wave_first = a.x.start_pos + min(row0, rows - 1) / a.group;
  const int lo_first = first_key(a.x, wave_first), lo_last = first_key(a.x, wave_last);
  const u32x4* src = reinterpret_cast<const u32x4*>(a.planes + ((long long)kvh * a.tiles - a.tile0) * TILE);
  const int2* ex = reinterpret_cast<const int2*>(a.exps) + ((long long)kvh * a.tiles - a.tile0);
  // a tile goes straight into the window (32 registers fewer than through them, which is what keeps heads of 128 from spilling)
  const int first = __builtin_amdgcn_readfirstlane(wave * 64);
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) _Float16*)&win[0][0];
  int2 stage_ex;
  auto load = [&](int t, int buf) __attribute__((always_inline)) {
    stage_ex = ex[t];
#pragma unroll
    for (int i = 0; i < NLD; ++i)
      tl_lds_load16(lds0 + (unsigned)(buf * TILE * 2 + (i * 256 + first) * 16), lane * 16, src + (size_t)t * (TILE / 8) + i * 256 + first);
  };
  auto arrived = [] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };  // of this wave's pieces; the barrier behind it: of all
  load(t0, 0);
  const float* qp = a.x.q + (size_t)rq * a.x.ldq + (size_t)head * a.x.qhs + 8 * h;
  half8 qh[DS], ql[DS];
  float cq;
  {
    float x[DS][8], mx = 0.f;
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      const f32x4 u = *reinterpret_cast<const f32x4*>(qp + 16 * s);
      const f32x4 w = *reinterpret_cast<const f32x4*>(qp + 16 * s + 4);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        x[s][i] = i < 4 ? u[i & 3] : w[i & 3];
        if (fabsf(x[s][i]) < INFINITY) mx = fmaxf(mx, fabsf(x[s][i]));
      }
    }
    mx = fmaxf(mx, tl_xor<32>(mx));
    const int k = scale_exp(mx);
    const float f = pow2i(k);
#pragma unroll
    for (int s = 0; s < DS; ++s) two_parts(x[s], f, qh[s], ql[s]);
    cq = a.scale * pow2i(-k);
  }
  f32x16 o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[b][e] = 0.f;
  float mrun = -INFINITY, lrun = 0.f;
  // o is held times 2^krun. A tile of larger values (a smaller exponent) has o follow at once, one of smaller values when its
  // probabilities would lose more than HA_P_SPARE bits: a tile with one huge row does not coarsen the tiles behind it. low: the
  // smallest exponent so far, o is below 2^(27 + krun - low) times the weights' sum, hence krun <= low + 60
  int krun = 60, low = 60;
  arrived();
  int ek = __builtin_amdgcn_readfirstlane(stage_ex.x), ev = __builtin_amdgcn_readfirstlane(stage_ex.y);
  __syncthreads();
  for (int t = t0; t < t1; ++t) {
    const int buf = (t - t0) & 1, p0 = t * 32;
    if (t + 1 < t1) load(t + 1, buf ^ 1);  // (last read a tile ago, in front of the barrier below)
    __builtin_amdgcn_sched_barrier(0);
    if (p0 <= wave_last && p0 + 31 >= lo_first) {
      const half8* kf = reinterpret_cast<const half8*>(&win[buf][0]) + lane;
      const half8* vf = reinterpret_cast<const half8*>(&win[buf][KD * 64]) + lane;
      f32x16 s, small;  // (the small products apart: the sums round once, not three times, per 16 columns)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = small[e] = 0.f;
#pragma unroll
      for (int d = 0; d < DS; ++d) {
        const half8 kl = kf[(2 * d + 1) * 64], kh = kf[(2 * d) * 64];
        small = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl, qh[d], small, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, qh[d], s, 0, 0, 0);
        small = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, ql[d], small, 0, 0, 0);
      }
      // operands two products ahead of their use
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int d = 0; d < DS - 2; ++d) {
        __builtin_amdgcn_sched_group_barrier(0x8, 3, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x8, 6, 0);
      __builtin_amdgcn_sched_barrier(0);
      half8 vl[2], vh[2];  // the first V operands arrive under the softmax
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        vl[j] = vf[(2 * j * DB + 1) * 64];
        vh[j] = vf[(2 * j * DB) * 64];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] += small[e];
      const float c = cq * pow2i(-ek);
      if (p0 + 31 > wave_first || p0 < lo_last) {  // some query of the wave does not see all of the tile
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int p = p0 + acc_row(e, h);
          s[e] = p <= qpos && p >= qlo ? s[e] : -INFINITY;
        }
      }
      float tmax = fmaxf(s[0], s[1]);
#pragma unroll
      for (int e = 2; e < 16; ++e) tmax = fmaxf(tmax, s[e]);
      tmax = half_max(tmax) * c;  // (c > 0)
      const float mnew = fmaxf(mrun, tmax), mref = mnew == -INFINITY ? 0.f : mnew;
      float corr = __builtin_amdgcn_exp2f(mrun - mref);
      mrun = mnew;
      // (the weights' 2^12 comes behind the exponential: inside it, 12 - mref would cost the largest weights' arguments twelve bits)
      float psum = 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], c, -mref));
        psum += s[e];
      }
      lrun = lrun * corr + psum;
      if (ev != krun) {  // (uniform)
        int over = ev - krun;
        if (over < 0 || over > HA_P_SPARE) {  // o takes the tile's unit, as far as its size allows
          const int to = ev < low + 60 ? ev : low + 60, by = to - krun, part = by < -126 ? -126 : by;
          corr *= pow2i(part) * pow2i(by - part);
          krun = to;
          over = ev - to;
        }
        if (over > 0) {  // the probabilities take o's
          const float f = pow2i(over < 126 ? -over : -126);
#pragma unroll
          for (int e = 0; e < 16; ++e) s[e] *= f;
        }
        low = ev < low ? ev : low;
      }
      half8 ph[2], pl[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          ph[j][i] = (_Float16)(s[8 * j + i] * HA_P_UNIT);
          pl[j][i] = (_Float16)__builtin_fmaf(s[8 * j + i], HA_P_UNIT, -(float)ph[j][i]);
        }
      __builtin_amdgcn_sched_barrier(0);
      // a tile's products meet in a sum of their own, small ones first: o, over all tiles, rounds once a tile
#pragma unroll
      for (int b = 0; b < DB; ++b) {
        f32x16 u;
#pragma unroll
        for (int e = 0; e < 16; ++e) u[e] = 0.f;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int n = 2 * b + j;
          u = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl[n & 1], ph[j], u, 0, 0, 0);
          u = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh[n & 1], pl[j], u, 0, 0, 0);
          u = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh[n & 1], ph[j], u, 0, 0, 0);
          if (n + 2 < 2 * DB) {
            vl[n & 1] = vf[(2 * (((n + 2) & 1) * DB + (n + 2) / 2) + 1) * 64];
            vh[n & 1] = vf[(2 * (((n + 2) & 1) * DB + (n + 2) / 2)) * 64];
          }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) o[b][e] = __builtin_fmaf(o[b][e], corr, u[e]);
      }
#pragma unroll
      for (int n = 0; n < 2 * DB - 2; ++n) {
        __builtin_amdgcn_sched_group_barrier(0x8, 3, 1);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
      }
      __builtin_amdgcn_sched_group_barrier(0x8, 6, 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    arrived();
    ek = __builtin_amdgcn_readfirstlane(stage_ex.x);
    ev = __builtin_amdgcn_readfirstlane(stage_ex.y);
    __syncthreads();
  }
  float l = lrun + tl_xor<32>(lrun);
  const float unit = 1.0f / HA_P_UNIT * pow2i(-krun);
  float* dst;
  float f = unit;
  if (ns == 1) {
    if (row >= rows) return;
    f = unit * finish(a.x, rq, head, mrun, l);
    dst = a.x.out + ((size_t)rq * nkv * a.group + head) * VD;
  } else {
    const size_t at = (size_t)blockIdx.x * HA_ROWS + wave * 32 + r;
    if (h == 0) a.ml[at] = make_float2(mrun, l);
    dst = a.part + at * VD;
  }
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
      const f32x4 v = {o[b][e] * f, o[b][e + 1] * f, o[b][e + 2] * f, o[b][e + 3] * f};
      *reinterpret_cast<f32x4*>(dst + 32 * b + acc_row(e, h)) = v;
    }
}

// rows of the row tiles with several pieces: VD / 4 threads a row
template <int VD>
__global__ __launch_bounds__(256) void hattn_combine_kernel(const HAttnArgs a) {
  constexpr int TR = VD / 4, RPB = 256 / TR;  // threads a row, rows a workgroup
  const int kvh = blockIdx.y, row = blockIdx.x * RPB + threadIdx.x / TR, c = threadIdx.x % TR;
  const int rows = a.x.T * a.group, nkv = a.x.kv_heads;
  if (row >= rows) return;
  const int rt = row / HA_ROWS, nrt = (rows + HA_ROWS - 1) / HA_ROWS;
  const TileRange range = row_tiles(a.x, a.group, rt);
  const int ns = (range.hi - range.lo + a.piece - 1) / a.piece;
  if (ns == 1) return;  // (written by the piece itself)
  const size_t at = ((size_t)(nrt - 1 - rt) * a.splits * nkv + kvh) * HA_ROWS + row % HA_ROWS;
  const size_t step = (size_t)nkv * HA_ROWS;
  float2 ml[HA_MAX_SPLIT];
  f32x4 v[HA_MAX_SPLIT];
#pragma unroll
  for (int s = 0; s < HA_MAX_SPLIT; ++s) {
    const size_t p = at + (s < ns ? s : 0) * step;
    ml[s] = a.ml[p];
    if (s >= ns) ml[s].x = -INFINITY;
    if (s < ns) v[s] = *reinterpret_cast<const f32x4*>(a.part + p * VD + 4 * c);
  }
  float M = ml[0].x;
#pragma unroll
  for (int s = 1; s < HA_MAX_SPLIT; ++s) M = fmaxf(M, ml[s].x);
  const float mref = M == -INFINITY ? 0.f : M;
  float L = 0.f;
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < HA_MAX_SPLIT; ++s)
    if (s < ns) {
      const float w = __builtin_amdgcn_exp2f(ml[s].x - mref);
      L += w * ml[s].y;
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[i] += w * v[s][i];
    }
  const int rq = row / a.group, head = kvh * a.group + row - rq * a.group;
  const float f = finish(a.x, rq, head, M, L);
#pragma unroll
  for (int i = 0; i < 4; ++i) sum[i] *= f;
  *reinterpret_cast<f32x4*>(a.x.out + ((size_t)rq * nkv * a.group + head) * VD + 4 * c) = sum;
}

size_t plane_bytes(int tiles, int nkv, int kd, int vd) { return (size_t)tiles * nkv * (kd + vd) * 64 * sizeof(_Float16); }
size_t exps_bytes(int tiles, int nkv) { return ((size_t)tiles * nkv * 2 * sizeof(int) + 255) & ~(size_t)255; }

// Number of pieces: the least rounds of 2 workgroups a CU times tiles a piece, plus what a piece costs beside its tiles
// (first tile, queries, output: about eight tiles of 2 us) and the pieces' way through memory.
int plan_splits(const TlHattn& x, int group, int* piece_out) {
  const int nrt = (x.T * group + HA_ROWS - 1) / HA_ROWS;
  const int slots = 2 * tl_num_cus();
  int most = 1;
  for (int rt = 0; rt < nrt; ++rt) {
    const TileRange g = row_tiles(x, group, rt);
    if (g.hi - g.lo > most) most = g.hi - g.lo;
  }
  int best = 1, best_piece = most;
  double best_cost = 1e30;
  for (int S = 1; S <= HA_MAX_SPLIT && S <= most; ++S) {
    if (S > 1 && (long long)nrt * S * x.kv_heads > HA_MAX_SLOTS) break;
    const int piece = (most + S - 1) / S;
    long long items = 0;
    for (int rt = 0; rt < nrt; ++rt) {
      const TileRange g = row_tiles(x, group, rt);
      items += (g.hi - g.lo + piece - 1) / piece;
    }
    const double rounds = (double)((items * x.kv_heads + slots - 1) / slots);
    const double cost = rounds * (piece + 8) + (S > 1 ? 2.0 + (double)items * x.kv_heads / slots * 2.0 : 0.0);
    if (cost < best_cost) best_cost = cost, best = S, best_piece = piece;
  }
  *piece_out = best_piece;
  return best;
}

template <int KD, int VD>
void launch(const HPlanesArgs& p, const HAttnArgs& a, hipStream_t s) {
  const int rows = a.x.T * a.group, nrt = (rows + HA_ROWS - 1) / HA_ROWS, per = 256 / (VD / 4);
  kv_planes_kernel<KD, VD><<<dim3(p.tiles, p.nkv), 256, 0, s>>>(p);
  hattn_kernel<KD, VD><<<dim3(nrt * a.splits * a.x.kv_heads), 256, 0, s>>>(a);
  if (a.splits > 1) hattn_combine_kernel<VD><<<dim3((rows + per - 1) / per, a.x.kv_heads), 256, 0, s>>>(a);
}

}  // namespace

// head sizes that are whole matrix instructions, and rows and heads at 16 bytes: wide loads of queries and keys. The kernel takes
// its maximum and its masks before the factor on the scores, so the factor has to be positive, and large enough to stay above
// zero beside the powers of two of a query and a key tile of (almost) zeros, 2^-60 each; any other one is the FP32 kernels'
bool tl_hattn_supported(const TlHattn& x) {
  if (!(x.scale >= 0x1p-16f && x.scale <= 0x1p16f)) return false;
  const bool sizes = x.vdim == 64 ? x.dim == 64 || x.dim == 96 || x.dim == 128 : x.vdim == 128 && x.dim == 128;
  return sizes && x.kv_heads > 0 && x.kv_heads <= 65535 && x.heads > 0 && x.heads % x.kv_heads == 0 &&
         ((x.ldq | x.qhs | x.kld | x.khs) & 3) == 0 && (((size_t)x.q | (size_t)x.kc | (size_t)x.out) & 15) == 0;
}

// for launches over at most max_keys positions (those that T tokens see), any T
size_t tl_hattn_bytes(int max_keys, int kv_heads, int dim, int vdim) {
  const int tiles = max_keys / 32 + 2;  // (a range of keys starts and ends inside a tile)
  return plane_bytes(tiles, kv_heads, dim, vdim) + exps_bytes(tiles, kv_heads) +
         (size_t)HA_MAX_SLOTS * HA_ROWS * (sizeof(float) * vdim + sizeof(float2));
}

// ws: tl_hattn_bytes of at least the positions that the tokens see
static std::atomic<long long> g_hattn_launches{0};
int tl_launch_hattn(const TlHattn& x, void* ws, size_t ws_bytes, hipStream_t s) {
  if (x.T == 0) return 0;
  TL_REQUIRE(tl_hattn_supported(x) && x.T > 0 && x.start_pos >= 0, "tl_launch_hattn: unsupported shapes");
  const int len = x.start_pos + x.T, lo = first_key(x, x.start_pos), tile0 = lo / 32, tiles = (len + 31) / 32 - tile0;
  TL_REQUIRE(ws && ws_bytes >= tl_hattn_bytes(len - lo, x.kv_heads, x.dim, x.vdim), "tl_launch_hattn: workspace too small");
  unsigned char* w = static_cast<unsigned char*>(ws);
  HPlanesArgs p = {x.kc, x.vc, x.kld, x.khs, x.vld, lo, len, x.kv_heads, tile0, tiles, reinterpret_cast<_Float16*>(w), nullptr};
  w += plane_bytes(tiles, x.kv_heads, x.dim, x.vdim);
  p.exps = reinterpret_cast<int*>(w);
  w += exps_bytes(tiles, x.kv_heads);
  HAttnArgs a = {};
  a.x = x;
  a.planes = p.planes;
  a.exps = p.exps;
  a.part = reinterpret_cast<float*>(w);
  a.ml = reinterpret_cast<float2*>(w + (size_t)HA_MAX_SLOTS * HA_ROWS * sizeof(float) * x.vdim);
  a.group = x.heads / x.kv_heads;
  a.tile0 = tile0;
  a.tiles = tiles;
  a.scale = x.scale * LOG2E;
  a.splits = plan_splits(x, a.group, &a.piece);
  TL_REQUIRE(((long long)x.T * a.group / HA_ROWS + 1) * a.splits * x.kv_heads <= 0x7fffffff, "tl_launch_hattn: launch too large");
  if (x.vdim == 128) launch<128, 128>(p, a, s);
  else if (x.dim == 128) launch<128, 64>(p, a, s);
  else if (x.dim == 96) launch<96, 64>(p, a, s);
  else launch<64, 64>(p, a, s);
  TL_HIP(hipGetLastError());
  g_hattn_launches.fetch_add(1, std::memory_order_relaxed);
  return 0;
}

// Diagnostic hook (tlhip_debug.h): calls of the function above so far in this process
extern "C" int tl_debug_half_attention_launches(long long* count_out) {
  TL_REQUIRE(count_out, "tl_debug_half_attention_launches: null argument");
  *count_out = g_hattn_launches.load();
  return 0;
}
// Measurement and test hook: the kernels above as an operator (tlhip_debug.h)
extern "C" int tl_debug_half_attention(const float* q_dev, const float* k_cache_dev, const float* v_cache_dev, float* out_dev, int num_tokens,
                                       int start_pos, int heads, int kv_heads, int dim, int vdim, int window, float scale, void* stream) {
  TL_REQUIRE(q_dev && k_cache_dev && v_cache_dev && out_dev && num_tokens > 0 && start_pos >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0,
             "tl_debug_half_attention: bad argument");
  TlHattn x = {};
  x.q = q_dev;
  x.kc = k_cache_dev;
  x.vc = v_cache_dev;
  x.out = out_dev;
  x.ldq = heads * dim;
  x.kld = kv_heads * dim;
  x.vld = kv_heads * vdim;
  x.qhs = x.khs = x.dim = dim;
  x.vdim = vdim;
  x.T = num_tokens;
  x.start_pos = start_pos;
  x.heads = heads;
  x.kv_heads = kv_heads;
  x.scale = scale;
  x.window = window;
  TL_REQUIRE(tl_hattn_supported(x), "tl_debug_half_attention: not shapes of the two-part f16 kernel");
  const size_t bytes = tl_hattn_bytes(start_pos + num_tokens, kv_heads, dim, vdim);
  void* ws = nullptr;
  TL_TRY(tl_scratch(TL_SCRATCH_ATTN, bytes, &ws));
  return tl_launch_hattn(x, ws, bytes, static_cast<hipStream_t>(stream));
}
