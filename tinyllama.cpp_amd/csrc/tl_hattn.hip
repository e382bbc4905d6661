// Causal prefill attention over one FP32 cache, its products in f16 matrix instructions at the 32-bit grade (gfx950).
// Reference behaviour: cpu_attention.cpp:254-325 (causal softmax attention with 1 / (sum + 1e-9)), gpu_kernels.cu attention.
//
// The FP32 matrix instructions do 64 multiply-adds a cycle and SIMD, the f16 ones 512: a product of two-part numbers
// (x 2^k = hi + lo, 22 bits, lo lo left out) costs three of the latter and still leaves a factor of five. The FP32 kernel
// (tl_prefill.hip) was bound by its matrix cores: 3989 tokens of 24 heads of 128 in chunks of 512, 28 layers, took it 44 ms;
// the three kernels here take 16 ms (of which the conversion 2.2, the sums 1.9), and the whole prompt 136 -> 105 ms. Now the
// matrix cores are half busy (a 32 x 32 tile pair of 2 us holds 1.5 us of products at the clock they leave).
//   1. kv_planes_kernel cuts the cache rows of every kv head into 32-key tiles of two-part f16 in the order in which the
//      lanes of a matrix instruction take them (K: eight columns of one key; V: eight keys of one column, the keys in the
//      order in which the accumulator of K Q^T holds them, so that the probabilities never change lanes). One power of two
//      per tile brings its largest finite value to 2^14: products of the tile's rows keep 22 bits over 2^18 of range.
//   2. hattn_kernel: four waves, 128 rows (query, head of the kv head's group), tiles through a double-buffered LDS window
//      that all four waves read: one wave's operands straight from memory would need 85 bytes a cycle and CU. Two workgroups
//      a CU, so that one's softmax runs under the other's products. A row tile's keys are cut into up to 16 pieces.
//   3. hattn_combine_kernel sums the pieces of a row tile that has more than one, in order.
#include <math.h>

#include "tl_internal.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));

namespace {

constexpr int HA_ROWS = 128, HA_MAX_SPLIT = 16, HA_MAX_SLOTS = 2048;
constexpr float HA_P_BITS = 12.f;  // probabilities are held times 2^12: their second part stays normal down to 2^-15

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

// tile (blockIdx.x) of kv head (blockIdx.y): K then V fragments, 64 HD halves each, and the two exponents
template <int HD>
__global__ __launch_bounds__(256) void kv_planes_kernel(const float* __restrict__ kc, const float* __restrict__ vc, int len, int nkv,
                                                        _Float16* __restrict__ planes, int* __restrict__ exps, int tiles) {
  constexpr int PT = HD / 64;  // fragments of each operand per thread
  __shared__ float red[8];
  const int tile = blockIdx.x, kvh = blockIdx.y, tid = threadIdx.x, p0 = tile * 32;
  const size_t row = (size_t)nkv * HD;
  const float *kp = kc + (size_t)kvh * HD, *vp = vc + (size_t)kvh * HD;
  float k[PT][8], v[PT][8], mk = 0.f, mv = 0.f;
#pragma unroll
  for (int t = 0; t < PT; ++t) {
    const int f = tid + 256 * t, lane = f & 63, r = lane & 31, h = lane >> 5, g = f >> 6;
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
    if (p0 + r < len) {
      const float* src = kp + (size_t)(p0 + r) * row + 16 * g + 8 * h;
      a = *reinterpret_cast<const f32x4*>(src);
      b = *reinterpret_cast<const f32x4*>(src + 4);
    }
    const int j = g / (HD / 32), d = 32 * (g % (HD / 32)) + r;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      k[t][i] = i < 4 ? a[i & 3] : b[i & 3];
      const int key = p0 + acc_row(8 * j + i, h);
      v[t][i] = key < len ? vp[(size_t)key * row + d] : 0.f;
    }
  }
#pragma unroll
  for (int t = 0; t < PT; ++t)
#pragma unroll
    for (int i = 0; i < 8; ++i) {  // (an infinity or a NaN spoils its own key only)
      if (fabsf(k[t][i]) < INFINITY) mk = fmaxf(mk, fabsf(k[t][i]));
      if (fabsf(v[t][i]) < INFINITY) mv = fmaxf(mv, fabsf(v[t][i]));
    }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    mk = fmaxf(mk, __shfl_xor(mk, o));
    mv = fmaxf(mv, __shfl_xor(mv, o));
  }
  if ((tid & 63) == 0) {
    red[tid >> 6] = mk;
    red[4 + (tid >> 6)] = mv;
  }
  __syncthreads();
  const int ek = scale_exp(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
  const int ev = scale_exp(fmaxf(fmaxf(red[4], red[5]), fmaxf(red[6], red[7])));
  if (tid == 0) {
    exps[2 * ((size_t)kvh * tiles + tile)] = ek;
    exps[2 * ((size_t)kvh * tiles + tile) + 1] = ev;
  }
  _Float16* out = planes + ((size_t)kvh * tiles + tile) * (HD * 128);
  const float fk = pow2i(ek), fv = pow2i(ev);
#pragma unroll
  for (int t = 0; t < PT; ++t) {
    const int f = tid + 256 * t, lane = f & 63, g = f >> 6;
    half8 hi, lo;
    two_parts(k[t], fk, hi, lo);
    *reinterpret_cast<half8*>(out + ((size_t)(2 * g) * 64 + lane) * 8) = hi;
    *reinterpret_cast<half8*>(out + ((size_t)(2 * g + 1) * 64 + lane) * 8) = lo;
    two_parts(v[t], fv, hi, lo);
    *reinterpret_cast<half8*>(out + HD * 64 + ((size_t)(2 * g) * 64 + lane) * 8) = hi;
    *reinterpret_cast<half8*>(out + HD * 64 + ((size_t)(2 * g + 1) * 64 + lane) * 8) = lo;
  }
}

// maximum of the two halves' lanes r and r + 32
__device__ __forceinline__ float half_max(float v) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
}

struct HAttnArgs {
  const float* q;          // [T][nh][HD]
  const _Float16* planes;  // [nkv][tiles][HD * 128]
  const int* exps;         // [nkv][tiles][2]
  float* out;              // [T][nh][HD]
  float* part;             // [slot][HA_ROWS][HD]
  float2* ml;              // [slot][HA_ROWS] (maximum in bits, sum)
  int T, start_pos, nkv, group, tiles, splits, piece;
  float scale;             // times log2(e)
};
// key tiles of row tile rt (rows rt * 128 ..: row = query * group + head of the group)
__host__ __device__ __forceinline__ int row_tiles(int T, int start_pos, int group, int rt) {
  const int last = (rt * HA_ROWS + HA_ROWS - 1) / group;
  return (start_pos + (last < T ? last : T - 1)) / 32 + 1;
}

template <int HD>
__global__ __launch_bounds__(256, 2) void hattn_kernel(const HAttnArgs a) {
  constexpr int DS = HD / 16, DB = HD / 32, TILE = HD * 128, NLD = TILE / 8 / 256;
  __shared__ __attribute__((aligned(16))) _Float16 win[2][TILE];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5, wave = tid >> 6;
  // workgroup L runs on XCD L mod 8: with a multiple of eight kv heads every L2 holds the planes of its own ones; the row
  // tiles with the most keys first
  const int kvh = blockIdx.x % a.nkv, slot = blockIdx.x / a.nkv, split = slot % a.splits;
  const int nrt = (a.T * a.group + HA_ROWS - 1) / HA_ROWS, rt = nrt - 1 - slot / a.splits;
  const int nt = row_tiles(a.T, a.start_pos, a.group, rt), ns = (nt + a.piece - 1) / a.piece;
  if (split >= ns) return;
  const int t0 = (int)((long long)nt * split / ns), t1 = (int)((long long)nt * (split + 1) / ns);
  const int row = rt * HA_ROWS + wave * 32 + r, rows = a.T * a.group;
  const int rq = (row < rows ? row : rows - 1) / a.group, rg = (row < rows ? row : rows - 1) - rq * a.group;
  const int qpos = a.start_pos + rq;
  const int row0 = __builtin_amdgcn_readfirstlane(rt * HA_ROWS + wave * 32);
  const int wave_last = a.start_pos + min(row0 + 31, rows - 1) / a.group, wave_first = a.start_pos + min(row0, rows - 1) / a.group;
  const u32x4* src = reinterpret_cast<const u32x4*>(a.planes + (size_t)kvh * a.tiles * TILE);
  const int2* ex = reinterpret_cast<const int2*>(a.exps) + (size_t)kvh * a.tiles;
  u32x4 stage[NLD];
  int2 stage_ex;
  auto load = [&](int t) __attribute__((always_inline)) {
    stage_ex = ex[t];
#pragma unroll
    for (int i = 0; i < NLD; ++i) stage[i] = src[(size_t)t * (TILE / 8) + i * 256 + tid];
  };
  auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NLD; ++i) *reinterpret_cast<u32x4*>(&win[buf][(i * 256 + tid) * 8]) = stage[i];
  };
  load(t0);
  const size_t q_at = ((size_t)rq * a.nkv * a.group + (size_t)kvh * a.group + rg) * HD;
  half8 qh[DS], ql[DS];
  float cq;
  {
    float x[DS][8], mx = 0.f;
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      const f32x4 u = *reinterpret_cast<const f32x4*>(a.q + q_at + 16 * s + 8 * h);
      const f32x4 w = *reinterpret_cast<const f32x4*>(a.q + q_at + 16 * s + 8 * h + 4);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        x[s][i] = i < 4 ? u[i & 3] : w[i & 3];
        if (fabsf(x[s][i]) < INFINITY) mx = fmaxf(mx, fabsf(x[s][i]));
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32));
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
  int krun = 60;  // smallest exponent of the V tiles so far: o is held times 2^krun
  store(0);
  int ek = __builtin_amdgcn_readfirstlane(stage_ex.x), ev = __builtin_amdgcn_readfirstlane(stage_ex.y);
  __syncthreads();
  for (int t = t0; t < t1; ++t) {
    const int buf = (t - t0) & 1, p0 = t * 32;
    load(t + 1 < t1 ? t + 1 : t);  // (the last one is not stored for anybody)
    __builtin_amdgcn_sched_barrier(0);
    if (p0 <= wave_last) {
      const half8* kf = reinterpret_cast<const half8*>(&win[buf][0]) + lane;
      const half8* vf = reinterpret_cast<const half8*>(&win[buf][HD * 64]) + lane;
      f32x16 s;
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = 0.f;
#pragma unroll
      for (int d = 0; d < DS; ++d) {
        const half8 kl = kf[(2 * d + 1) * 64], kh = kf[(2 * d) * 64];
        s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl, qh[d], s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, ql[d], s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, qh[d], s, 0, 0, 0);
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
      for (int b = 0; b < 2; ++b) {
        vl[b] = vf[(2 * b + 1) * 64];
        vh[b] = vf[(2 * b) * 64];
      }
      __builtin_amdgcn_sched_barrier(0);
      const float c = cq * pow2i(-ek);
      if (p0 + 31 > wave_first) {  // some query of the wave does not see all of the tile
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = p0 + acc_row(e, h) <= qpos ? s[e] : -INFINITY;
      }
      float tmax = fmaxf(s[0], s[1]);
#pragma unroll
      for (int e = 2; e < 16; ++e) tmax = fmaxf(tmax, s[e]);
      tmax = half_max(tmax) * c;  // (c > 0)
      const float mnew = fmaxf(mrun, tmax), mref = mnew == -INFINITY ? 0.f : mnew;
      float corr = __builtin_amdgcn_exp2f(mrun - mref);
      mrun = mnew;
      const float bias = HA_P_BITS - mref;
      float psum = 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], c, bias));
        psum += s[e];
      }
      lrun = lrun * corr + psum;
      if (ev != krun) {  // (uniform) the smaller exponent rules: o takes the tile's unit, or the probabilities take o's
        const int down = ev - krun;
        if (down < 0) {
          corr *= pow2i(down < -126 ? -126 : down);
          krun = ev;
        } else {
          const float f = pow2i(-down < -126 ? -126 : -down);
#pragma unroll
          for (int e = 0; e < 16; ++e) s[e] *= f;
        }
      }
      if (__any(corr != 1.f)) {
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[b][e] *= corr;
      }
      half8 ph[2], pl[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          ph[j][i] = (_Float16)s[8 * j + i];
          pl[j][i] = (_Float16)__builtin_fmaf((float)ph[j][i], -1.0f, s[8 * j + i]);
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < 2 * DB; ++n) {
        const int j = n / DB, b = n % DB;
        o[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl[n & 1], ph[j], o[b], 0, 0, 0);
        o[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh[n & 1], pl[j], o[b], 0, 0, 0);
        o[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh[n & 1], ph[j], o[b], 0, 0, 0);
        if (n + 2 < 2 * DB) {
          vl[n & 1] = vf[(2 * (n + 2) + 1) * 64];
          vh[n & 1] = vf[(2 * (n + 2)) * 64];
        }
      }
#pragma unroll
      for (int n = 0; n < 2 * DB - 2; ++n) {
        __builtin_amdgcn_sched_group_barrier(0x8, 3, 1);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
      }
      __builtin_amdgcn_sched_group_barrier(0x8, 6, 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    store(buf ^ 1);  // (last read a tile ago, in front of the barrier below)
    ek = __builtin_amdgcn_readfirstlane(stage_ex.x);
    ev = __builtin_amdgcn_readfirstlane(stage_ex.y);
    __syncthreads();
  }
  float l = lrun + __shfl_xor(lrun, 32);
  l *= pow2i(-(int)HA_P_BITS);
  const float unit = pow2i(-(int)HA_P_BITS) * pow2i(-krun);
  float* dst;
  float f = unit;
  if (ns == 1) {
    if (row >= rows) return;
    f = unit * (1.0f / (l + 1e-9f));
    dst = a.out + q_at;
  } else {
    const size_t at = (size_t)blockIdx.x * HA_ROWS + wave * 32 + r;
    if (h == 0) a.ml[at] = make_float2(mrun, l);
    dst = a.part + at * HD;
  }
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
      const f32x4 v = {o[b][e] * f, o[b][e + 1] * f, o[b][e + 2] * f, o[b][e + 3] * f};
      *reinterpret_cast<f32x4*>(dst + 32 * b + acc_row(e, h)) = v;
    }
}

// rows of the row tiles with several pieces: HD / 4 threads a row
template <int HD>
__global__ __launch_bounds__(256) void hattn_combine_kernel(const HAttnArgs a) {
  constexpr int TR = HD / 4, RPB = 256 / TR;  // threads a row, rows a workgroup
  const int kvh = blockIdx.y, row = blockIdx.x * RPB + threadIdx.x / TR, c = threadIdx.x % TR;
  if (row >= a.T * a.group) return;
  const int rt = row / HA_ROWS, nrt = (a.T * a.group + HA_ROWS - 1) / HA_ROWS;
  const int nt = row_tiles(a.T, a.start_pos, a.group, rt), ns = (nt + a.piece - 1) / a.piece;
  if (ns == 1) return;  // (written by the piece itself)
  const size_t at = ((size_t)(nrt - 1 - rt) * a.splits * a.nkv + kvh) * HA_ROWS + row % HA_ROWS;
  const size_t step = (size_t)a.nkv * HA_ROWS;
  float2 ml[HA_MAX_SPLIT];
  f32x4 v[HA_MAX_SPLIT];
#pragma unroll
  for (int s = 0; s < HA_MAX_SPLIT; ++s) {
    const size_t p = at + (s < ns ? s : 0) * step;
    ml[s] = a.ml[p];
    if (s >= ns) ml[s].x = -INFINITY;
    if (s < ns) v[s] = *reinterpret_cast<const f32x4*>(a.part + p * HD + 4 * c);
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
  const float inv = 1.0f / (L + 1e-9f);
  const int rq = row / a.group, rg = row - rq * a.group;
#pragma unroll
  for (int i = 0; i < 4; ++i) sum[i] *= inv;
  *reinterpret_cast<f32x4*>(a.out + ((size_t)rq * a.nkv * a.group + (size_t)kvh * a.group + rg) * HD + 4 * c) = sum;
}

size_t plane_bytes(int tiles, int nkv, int hd) { return (size_t)tiles * nkv * hd * 128 * sizeof(_Float16); }
size_t exps_bytes(int tiles, int nkv) { return ((size_t)tiles * nkv * 2 * sizeof(int) + 255) & ~(size_t)255; }

// Number of pieces: the least rounds of 2 workgroups a CU times tiles a piece, plus what a piece costs beside its tiles
// (first tile, queries, output: about eight tiles of 2 us) and the pieces' way through memory.
int plan_splits(int T, int start_pos, int nkv, int group, int* piece_out) {
  const int nrt = (T * group + HA_ROWS - 1) / HA_ROWS, most = row_tiles(T, start_pos, group, nrt - 1);
  const int slots = 2 * tl_num_cus();
  int best = 1, best_piece = most;
  double best_cost = 1e30;
  for (int S = 1; S <= HA_MAX_SPLIT && S <= most; ++S) {
    if (S > 1 && (long long)nrt * S * nkv > HA_MAX_SLOTS) break;
    const int piece = (most + S - 1) / S;
    long long items = 0;
    for (int rt = 0; rt < nrt; ++rt) items += (row_tiles(T, start_pos, group, rt) + piece - 1) / piece;
    const double rounds = (double)((items * nkv + slots - 1) / slots);
    const double cost = rounds * (piece + 8) + (S > 1 ? 2.0 + (double)items * nkv / slots * 2.0 : 0.0);
    if (cost < best_cost) best_cost = cost, best = S, best_piece = piece;
  }
  *piece_out = best_piece;
  return best;
}

}  // namespace

bool tl_hattn_supported(int nh, int nkv, int hd) { return (hd == 64 || hd == 128) && nkv > 0 && nh > 0 && nh % nkv == 0; }

size_t tl_hattn_bytes(int max_len, int nkv, int hd) {
  const int tiles = (max_len + 31) / 32;
  return plane_bytes(tiles, nkv, hd) + exps_bytes(tiles, nkv) + (size_t)HA_MAX_SLOTS * HA_ROWS * (sizeof(float) * hd + sizeof(float2));
}

// q [T][nh][hd] (rotated), caches [.][nkv][hd] already holding positions 0 .. start_pos + T - 1, out [T][nh][hd];
// ws: tl_hattn_bytes of at least start_pos + T positions
int tl_launch_hattn(const float* q, const float* kc, const float* vc, float* out, int T, int start_pos, int nh, int nkv, int hd,
                    float scale, void* ws, size_t ws_bytes, hipStream_t s) {
  TL_REQUIRE(tl_hattn_supported(nh, nkv, hd), "tl_launch_hattn: unsupported head shape");
  if (T == 0) return 0;
  const int len = start_pos + T, tiles = (len + 31) / 32;
  TL_REQUIRE(ws && ws_bytes >= tl_hattn_bytes(len, nkv, hd), "tl_launch_hattn: workspace too small");
  HAttnArgs a = {};
  unsigned char* w = static_cast<unsigned char*>(ws);
  _Float16* planes = reinterpret_cast<_Float16*>(w);
  w += plane_bytes(tiles, nkv, hd);
  int* exps = reinterpret_cast<int*>(w);
  w += exps_bytes(tiles, nkv);
  a.q = q;
  a.planes = planes;
  a.exps = exps;
  a.out = out;
  a.part = reinterpret_cast<float*>(w);
  a.ml = reinterpret_cast<float2*>(w + (size_t)HA_MAX_SLOTS * HA_ROWS * sizeof(float) * hd);
  a.T = T;
  a.start_pos = start_pos;
  a.nkv = nkv;
  a.group = nh / nkv;
  a.tiles = tiles;
  a.scale = scale * 1.44269504088896340736f;
  a.splits = plan_splits(T, start_pos, nkv, a.group, &a.piece);
  const int rows = T * a.group, nrt = (rows + HA_ROWS - 1) / HA_ROWS, per = 256 / (hd / 4);
  TL_REQUIRE((long long)nrt * a.splits * nkv <= 0x7fffffff && nkv <= 65535, "tl_launch_hattn: launch too large");
  const dim3 grid(nrt * a.splits * nkv), cgrid((rows + per - 1) / per, nkv);
  if (hd == 128) {
    kv_planes_kernel<128><<<dim3(tiles, nkv), 256, 0, s>>>(kc, vc, len, nkv, planes, exps, tiles);
    hattn_kernel<128><<<grid, 256, 0, s>>>(a);
    if (a.splits > 1) hattn_combine_kernel<128><<<cgrid, 256, 0, s>>>(a);
  } else {
    kv_planes_kernel<64><<<dim3(tiles, nkv), 256, 0, s>>>(kc, vc, len, nkv, planes, exps, tiles);
    hattn_kernel<64><<<grid, 256, 0, s>>>(a);
    if (a.splits > 1) hattn_combine_kernel<64><<<cgrid, 256, 0, s>>>(a);
  }
  TL_HIP(hipGetLastError());
  return 0;
}
