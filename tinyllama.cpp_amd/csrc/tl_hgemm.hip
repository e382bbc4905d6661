// tl_hgemm.hip — batched GEMM over the quantized plane layout with f16 matrix instructions:
//   Y[T][rows] (+ resid) = X[T][cols] . W[rows][cols]^T      for the batched paths (prompts, multi-sequence steps)
//
// The same product as tl_gemm.hip's kernels (smart_gemm_batch_cuda, model.cpp:2141-2249; numerics target
// matmul_f32_f32_batch_cpu, utils.cpp:730-782) at the same 32-bit grade, with fewer matrix instructions and fewer vector
// instructions per weight:
//   - an activation is held as two f16 parts of x * 2^k, k chosen per token and super-block (256 columns) so that the
//     largest value there lies in [2^9, 2^10): x = hi + lo to 22 bits and sign, and to 2^-35 of that largest value where lo
//     is sub-normal. Two matrix instructions per weight operand instead of the three that bf16 parts need;
//   - what a weight operand holds is exact in f16, which has 11 bits: Q4_K's sub-block scale times the nibble (<= 945), the
//     bytes of Q8, and of Q6_K the product scale * q (13 bits) as a rounded part plus its remainder. A running sum
//     therefore spans a whole 256-column super-block (Q8_0: a 32-column block) before a vector FMA applies the
//     super-block's factor to it: 16 FMAs per 33 matrix instructions (Q4_K) where integer operands need 16 per 3;
//   - Q4_K's minima: sum_j m_j * (sum of x over sub-block j) is one more K = 16 matrix instruction per super-block, with
//     the eight sub-block sums' two f16 parts side by side along K and the same eight m_j against either half.
// hgemm_kernel (tiles of up to 128 rows, Q8_K 256): weights go from HBM straight into registers (a super-block ahead), are unpacked
// there and never touch LDS; the activation tile is staged through LDS, up to 32 tokens a super-block ahead with one barrier
// per super-block, 64 tokens in a ring of three 64-column steps. hgemm_lds_body (256 and 512 rows): activations and
// weights are both copied from memory to LDS as they lie there, with a barrier per 64-column step, and unpacked behind it.
//
// The order of the columns inside an operand is free as long as both sides agree. Lane half h of a Q4_K / Q6_K step takes
// the 32-weight chunk 2 s + h (one 16-byte load), of a Q8 step 16 of the 32 bytes of a chunk; the eight columns of an
// operand are in the order [0 2 1 3 4 6 5 7], which is what masking a dword into 16-bit halves gives without moving a
// byte, and which the activation planes are written in.
#include <atomic>
#include <type_traits>

#include "tl_internal.h"
#include "tl_hsplit.h"
#include "tl_lanes.h"
#include "tl_lds.h"
#include "tl_parts.h"

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

namespace {

// ---- activation planes: [2][ps] f16 (hi, lo), then per super-block the block sums [cols / 256][tpad][hi 8 | lo 8] f16,
//      then 2^-k [cols / 256][tpad] (tpad: padded tokens)
struct HAct {
  const _Float16* x;
  size_t ps;
  const _Float16* bs;
  const float* inv;
  int tpad;
};
inline HAct hact(const void* planes, size_t ps, int T) {
  const _Float16* x = static_cast<const _Float16*>(planes);
  const _Float16* bs = x + 2 * ps;
  return HAct{x, ps, bs, reinterpret_cast<const float*>(bs + ps / 16), (int)tl_gemm_padded_tokens(T)};
}

__device__ __forceinline__ float h2f(unsigned h) { return (float)__builtin_bit_cast(_Float16, (unsigned short)h); }
__device__ __forceinline__ float h2f_scale(unsigned h) {  // |d| for finite negatives (quantization.cpp:85-87)
  const float d = h2f(h);
  return (d < 0.0f && d > -INFINITY) ? -d : d;
}
__device__ __forceinline__ f16x2 as_h2(unsigned u) { return __builtin_bit_cast(f16x2, u); }
__device__ __forceinline__ f16x2 h2(float v) { return f16x2{(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ f16x8 join(f16x2 a, f16x2 b, f16x2 c, f16x2 d) {
  return f16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// A matrix instruction covers TK tokens x TK weight rows: 32 x 32 x 16 columns, or 16 x 16 x 32 for 16 tokens and fewer. The
// 64 / TK = NG lane groups hold eight columns each.
template <int TK>
struct Tile {
  typedef f32x16 Acc;
  static constexpr int E = 16;
  static __device__ __forceinline__ Acc mfma(f16x8 a, f16x8 b, Acc c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int quad(int q, int g) { return 8 * q + 4 * g; }  // token of element 4 q
};
template <>
struct Tile<16> {
  typedef f32x4 Acc;
  static constexpr int E = 4;
  static __device__ __forceinline__ Acc mfma(f16x8 a, f16x8 b, Acc c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int quad(int, int g) { return 4 * g; }
};

// what one lane holds of a step (NG 32-weight chunks of one row, four operands), and of a super-block
template <int TYPE>
struct WStep {
  u32x4 q;       // Q4_K / Q6_K: chunk NG u + group; Q8: the lane's eight bytes of operands 0 and 1
  u32x4 q1;      // Q8: of operands 2 and 3
  u32x2 hi;      // Q6_K: high bits of the chunk
  unsigned d[2]; // Q8_0: d of the step's chunks
};
template <int TYPE>
struct WHead {
  u32x4 h;     // Q4_K: super-block header; Q6_K: the 16 sub-block scales
  unsigned d;  // Q6_K / Q8_K: d
};
// step u of super-block sb; steps past the end of a Q8_0 row (not a whole number of super-blocks) read its last chunks
template <int TYPE, int TK>
__device__ __forceinline__ void load_step(WStep<TYPE>& g, const QW& w, unsigned R, int sb, int u, int fg) {
  constexpr int NG = 64 / TK;
  const unsigned K = (unsigned)w.cols;
  if (TYPE == TL_Q4_K || TYPE == TL_Q6_K) {
    const unsigned c = sb * 8 + NG * u + fg;
    g.q = *reinterpret_cast<const u32x4*>(w.p0 + (size_t)(R * (K >> 1) + c * 16));
    if (TYPE == TL_Q6_K) g.hi = *reinterpret_cast<const u32x2*>(w.p1 + (size_t)(R * (K >> 2) + c * 8));
  } else {
    const unsigned last = (K >> 6) - 1;  // (pairs of chunks: K is a multiple of 64)
    const unsigned s = (TK == 32 ? sb * 4 + u : sb * 4 + 2 * u), s0 = s < last ? s : last, s1 = s + 1 < last ? s + 1 : last;
    if (TK == 32) {
      g.q = *reinterpret_cast<const u32x4*>(w.p0 + (size_t)(R * K + s0 * 64 + fg * 16));
      g.q1 = *reinterpret_cast<const u32x4*>(w.p0 + (size_t)(R * K + s0 * 64 + fg * 16 + 32));
    } else {
      const u32x2 a = *reinterpret_cast<const u32x2*>(w.p0 + (size_t)(R * K + s0 * 64 + fg * 8));
      const u32x2 b = *reinterpret_cast<const u32x2*>(w.p0 + (size_t)(R * K + s0 * 64 + fg * 8 + 32));
      const u32x2 c = *reinterpret_cast<const u32x2*>(w.p0 + (size_t)(R * K + s1 * 64 + fg * 8));
      const u32x2 d = *reinterpret_cast<const u32x2*>(w.p0 + (size_t)(R * K + s1 * 64 + fg * 8 + 32));
      g.q = u32x4{a[0], a[1], b[0], b[1]};
      g.q1 = u32x4{c[0], c[1], d[0], d[1]};
    }
    if (TYPE == TL_Q8_0) {
      g.d[0] = *reinterpret_cast<const unsigned*>(w.p1 + (size_t)((R * (K >> 5) + 2 * s0) * 2));
      if (TK == 16) g.d[1] = *reinterpret_cast<const unsigned*>(w.p1 + (size_t)((R * (K >> 5) + 2 * s1) * 2));
    }
  }
}
template <int TYPE>
__device__ __forceinline__ void load_head(WHead<TYPE>& g, const QW& w, unsigned R, int sb) {
  const unsigned K = (unsigned)w.cols;
  if (TYPE == TL_Q4_K) g.h = *reinterpret_cast<const u32x4*>(w.p1 + (size_t)(R * (K >> 4) + sb * 16));
  if (TYPE == TL_Q6_K) {
    g.h = *reinterpret_cast<const u32x4*>(w.p2 + (size_t)(R * (K >> 4) + sb * 16));
    g.d = *reinterpret_cast<const uint16_t*>(w.p3 + (size_t)((R * (K >> 8) + sb) * 2));
  }
  if (TYPE == TL_Q8_K) g.d = *reinterpret_cast<const uint16_t*>(w.p1 + (size_t)((R * (K >> 8) + sb) * 2));
}

// the eight weights of operand w (0..3) of step u (0..3 inside the super-block), in operand order
constexpr unsigned MAGIC = 0x64006400u;  // f16 1024: a small integer or-ed into the mantissa is 1024 + itself
// (v & mask) | MAGIC in one instruction: v_and_or_b32 takes no literals, so both constants have to sit in registers
__device__ __forceinline__ unsigned pick(unsigned v, unsigned mask) {
  unsigned r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(mask), "v"(MAGIC));
  return r;
}
struct Scale4 {
  f16x2 c, cn, c16, cn16;  // sc, -1024 sc, sc / 16, -64 sc
};
__device__ __forceinline__ Scale4 q4_scale(unsigned h1, unsigned h3, int c) {  // h1, h3 already shifted to the lane group's chunk
  const unsigned sc = ((h1 >> (4 * c)) & 15u) | (((h3 >> (2 * c)) & 3u) << 4);
  Scale4 r;
  r.c = as_h2(sc | (sc << 16) | MAGIC) - h2(1024.f);
  r.cn = r.c * h2(-1024.f);
  r.c16 = r.c * h2(0.0625f);
  r.cn16 = r.c * h2(-64.f);
  return r;
}
__device__ __forceinline__ f16x8 q4_operand(unsigned u, const Scale4& s) {
  const unsigned v = u >> 8;
  // (1024 + q) sc - 1024 sc and (1024 + 16 q) sc / 16 - 64 sc: one rounding each, of a value that needs none
  return join(__builtin_elementwise_fma(as_h2(pick(u, 0x000F000Fu)), s.c, s.cn),
              __builtin_elementwise_fma(as_h2(pick(v, 0x000F000Fu)), s.c, s.cn),
              __builtin_elementwise_fma(as_h2(pick(u, 0x00F000F0u)), s.c16, s.cn16),
              __builtin_elementwise_fma(as_h2(pick(v, 0x00F000F0u)), s.c16, s.cn16));
}
// the minima m_0..m_7 of a super-block in the order [0 4 1 5 2 6 3 7] (the block sums' order)
__device__ __forceinline__ f16x8 q4_minima(unsigned m_lo, unsigned hi) {
  const unsigned hh = ((hi >> 16) & 0xFFu) | ((hi >> 8) & 0x00FF0000u);
  f16x2 r[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) r[p] = as_h2(((m_lo >> (4 * p)) & 0x000F000Fu) | (((hh >> (2 * p)) & 0x00030003u) << 4) | MAGIC) - h2(1024.f);
  return join(r[0], r[1], r[2], r[3]);
}
__device__ __forceinline__ void q6_operand(unsigned u, unsigned hv, int odd, f16x2 sc, f16x8& hi, f16x8& lo) {
  f16x2 a[4], b[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {  // pairs (0 2) (1 3) (4 6) (5 7): byte shift 8 (p & 1), part p >> 1
    // low nibbles to bits 0..3, high bits to bits 4..5 of the 16-bit halves
    const int at = 8 * (p & 1) + 2 * (2 * odd + (p >> 1)) - 4;
    const unsigned h = pick(at < 0 ? hv << -at : hv >> at, 0x00300030u);
    unsigned l = u >> (8 * (p & 1) + 4 * (p >> 1));
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(l) : "v"(l), "s"(0x000F000Fu), "v"(h));
    const f16x2 q = as_h2(l) - h2(1056.f);
    a[p] = q * sc;                                      // 13 bits rounded to 11
    b[p] = __builtin_elementwise_fma(q, sc, -a[p]);     // the remainder, exact
  }
  hi = join(a[0], a[1], a[2], a[3]);
  lo = join(b[0], b[1], b[2], b[3]);
}
__device__ __forceinline__ f16x8 q8_operand(unsigned a, unsigned b) {
  const unsigned x = a ^ 0x80808080u, y = b ^ 0x80808080u;
  const f16x2 off = h2(1152.f);
  return join(as_h2(pick(x, 0x00FF00FFu)) - off, as_h2(pick(x >> 8, 0x00FF00FFu)) - off,
              as_h2(pick(y, 0x00FF00FFu)) - off, as_h2(pick(y >> 8, 0x00FF00FFu)) - off);
}

// v / d of 31-bit v by one multiplication: m = floor(2^(31 + l) / d) + 1 with l = ceil(log2 d) fits 32 bits, and v m / 2^(31 + l) exceeds v / d
// by less than 1 / d
struct Div {
  unsigned m, l;
  static Div by(unsigned d) {
    unsigned l = 0;
    while ((1ull << l) < d) ++l;
    return Div{(unsigned)((1ull << (31 + l)) / d + 1), l};
  }
  __device__ __forceinline__ int of(int v) const { return (int)(__umulhi(2u * (unsigned)v, m) >> l); }
};
// A launch: up to three matrices over the same activations (q | k | v, gate | up), whose row tiles follow each other, and the grid's
// division into slices, panels and tiles. What every workgroup would otherwise work out for itself is worked out here: in a launch of few
// tokens the instructions in front of the first load are a part of its time (eight tokens in Q4_K: 313 and six waits for arguments, each
// asked for when the one before had come; now 161 and three. 0.4 us of 7: steps of 8 sequences over 28 layers of 3072 1.86 -> 1.80 ms)
struct HSegs {
  int T, K, nsb, per;                          // tokens, columns, super-blocks of a row and of a slice
  int per8, rem8, slice_tiles, panel_tiles;    // workgroups of an XCD (and how many XCDs have one more), of a slice, of a panel
  Div by_slice, by_panel, by_width, by_last;   // ... and divisions by the tiles of a slice and of a panel, and by the token tiles of a panel and of the last one
  int panel, width_last, last_panel, mt_end[2];
  const float* resid;
  HAct act;
  QW w[3];
  float* y[3];
};

// Which tile a workgroup computes.
// consecutive workgroups go to the 8 XCDs in turn: each XCD walks a contiguous range, panels of `panel` token tiles one after another
// and inside a panel token tiles fastest. The workgroups that read the same weights thereby share an L2, and the 32 or 64 that an
// XCD runs at a time read 8 token tiles' activations and 4 or 8 row tiles' weights; with all token tiles side by side, 2048 tokens
// (32 tiles, 32 MB of activations a round) fetched three times as much through the fabric, which costs time and clock: 28672 x 4096
// in Q4_K times 2048 tokens 986 -> 967 us in waves of 64 rows and 1200 -> 1116 in shape 4, 16384 x 3072 in Q6_K 682 -> 648.
struct Place {
  int slice, nt, mt, seg;
};
__device__ __forceinline__ Place place_of(const HSegs& g, int block) {
  const int xcd = block & 7, at = block >> 3;
  const int v = xcd * g.per8 + (xcd < g.rem8 ? xcd : g.rem8) + at;
  Place p;
  p.slice = g.by_slice.of(v);
  const int in_slice = v - p.slice * g.slice_tiles, pi = g.by_panel.of(in_slice), in_panel = in_slice - pi * g.panel_tiles;
  const bool last = pi == g.last_panel;
  int wl = g.width_last, wp = g.panel;
  Div dl = g.by_last, dp = g.by_width;
  asm("" : "+s"(wl), "+s"(wp), "+s"(dl.m), "+s"(dl.l), "+s"(dp.m), "+s"(dp.l));  // (loads of both, not one whose address is chosen first)
  const int width = last ? wl : wp;
  p.mt = Div{last ? dl.m : dp.m, last ? dl.l : dp.l}.of(in_panel);
  p.nt = g.panel * pi + in_panel - p.mt * width;
  p.seg = (p.mt >= g.mt_end[0]) + (p.mt >= g.mt_end[1]);
  p.mt -= p.seg == 0 ? 0 : p.seg == 1 ? g.mt_end[0] : g.mt_end[1];
  return p;
}

// STACK: the upper half of the wave has the small sums of the lower half's tokens. The whole, in both halves (Q6_K: tl holds the
// remainders' products, small in either half)
template <int TYPE>
__device__ __forceinline__ float stacked_sum(float t, float tl, int fg) {
  float small = fg >= 2 ? t : 0.f;
  if (TYPE == TL_Q6_K) small += tl;
  const float big = fg >= 2 ? 0.f : t, other = tl_xor<32>(small);
  return big + (TYPE == TL_Q6_K ? small + other : other);
}
// acc += a super-block's sums times the rows' factors and the tokens' powers of two. bs: its block sums [token][hi 8 | lo 8], then 2^-k
// (APART: sums of the hi part's products t and of the small ones tl)
template <int TYPE, int TK, int NI, int MI, bool STACK>
__device__ __forceinline__ void add_superblock(typename Tile<TK>::Acc (&acc)[NI][MI], const typename Tile<TK>::Acc (&t)[NI][MI],
                                               const typename Tile<TK>::Acc (&tl)[NI][MI], const typename Tile<TK>::Acc (&c8)[NI][MI],
                                               const WHead<TYPE> (&H)[MI], const _Float16* ab, const _Float16* invs, int fr, int fg) {
  typedef Tile<TK> TL;
  typedef typename TL::Acc Acc;
  constexpr bool APART = TK == 16 || MI == 1;
  const Acc zero = {};
  float d[MI], dm[MI];
  f16x8 mn[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    d[i] = TYPE == TL_Q4_K ? h2f(H[i].h[0] & 0xFFFFu) : TYPE == TL_Q6_K ? h2f(H[i].d) : TYPE == TL_Q8_K ? h2f_scale(H[i].d) : 1.f;
    if (TYPE == TL_Q4_K) {
      mn[i] = q4_minima(H[i].h[2], H[i].h[3]);
      dm[i] = -h2f(H[i].h[0] >> 16);
    }
  }
#pragma unroll
  for (int n = 0; n < NI; ++n) {
    f16x8 bs;
    if (TYPE == TL_Q4_K) {
      bs = *reinterpret_cast<const f16x8*>(ab + (TK * n + (STACK ? fr & 7 : fr)) * 16 + (fg & 1) * 8);
      if (TK == 16 && fg >= 2) bs = f16x8{};  // (the instruction's columns 16..31: nothing)
    }
    const float* inv = reinterpret_cast<const float*>(invs) + TK * n;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      Acc s;
      if (TYPE == TL_Q4_K) s = TL::mfma(bs, mn[i], zero);
#pragma unroll
      for (int q = 0; q < TL::E / 4; ++q) {
        const f32x4 iv = *reinterpret_cast<const f32x4*>(inv + TL::quad(q, STACK ? fg & 1 : fg));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float x;
          if (TYPE == TL_Q8_0) x = c8[n][i][4 * q + e];
          else if (STACK) x = d[i] * stacked_sum<TYPE>(t[n][i][4 * q + e], tl[n][i][4 * q + e], fg);
          else x = d[i] * (APART ? t[n][i][4 * q + e] + tl[n][i][4 * q + e] : t[n][i][4 * q + e]);
          if (TYPE == TL_Q8_0 && STACK) x += tl_xor<32>(x);
          if (TYPE == TL_Q4_K) x = fmaf(dm[i], s[4 * q + e], x);
          acc[n][i][4 * q + e] = fmaf(iv[e], x, acc[n][i][4 * q + e]);
        }
      }
    }
  }
}
template <int TK, int NI, int MI, bool STACK>
__device__ __forceinline__ void store_tile(float* __restrict__ y, const float* __restrict__ resid, const typename Tile<TK>::Acc (&acc)[NI][MI],
                                           int n0, int m0, int T, int M, int fr, int fg) {
#pragma unroll
  for (int n = 0; n < NI; ++n)
#pragma unroll
    for (int q = 0; q < Tile<TK>::E / 4; ++q) {
      const int t0 = n0 + TK * n + Tile<TK>::quad(q, fg);
      if (STACK && fg >= 2) continue;
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int r = m0 + TK * i + fr;
        if (r >= M) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (t0 + e < T) {
            const size_t o = (size_t)(t0 + e) * M + r;
            const float val = acc[n][i][4 * q + e];
            y[o] = resid ? resid[o] + val : val;
          }
        }
      }
    }
}

// Workgroup: NW waves of TK MI rows each x TK NI tokens (STACK, for up to 8 tokens: x 8, whose hi parts are rows 0..7 of the instruction's
// operand and whose lo parts are rows 8..15: half the matrix instructions, half the activations' way through LDS; 64 rows of Q4_K x 256
// columns, four workgroups on a CU, 0.80 -> 0.67 us). LDS: two buffers of a super-block's activation tile, [4 x 64
// columns][2 parts][tokens][64] f16, the 16-byte pieces of a token's 128 bytes at piece ^ (row / 2 & 7), row = part x tokens + token: the 16
// consecutive rows of a fragment read and the 2 x 8 pieces of a staging write cover the 64 banks once; behind them the
// super-block's block sums and powers of two.
template <int TYPE, int TK, int NI, int MI, int NW, bool STACK>
__device__ __forceinline__ void hgemm_body(const HSegs& segs, int block) {
  typedef Tile<TK> TL;
  typedef typename TL::Acc Acc;
  constexpr int NG = 64 / TK, US = 8 / NG;                        // lane groups, steps of a super-block
  constexpr int BN = STACK ? 8 : TK * NI, NT = 64 * NW, STEP = 2 * BN * 64;  // STEP: halfs of 64 columns
  constexpr int XP = 16 * BN, XR = (BN > 32 ? XP : 4 * XP) / NT;  // 16-byte pieces of 64 columns; per thread of a fetch (RINGED: 64 columns)
  constexpr int PARTS = STACK ? 1 : 2;                            // fragments of an operand
  constexpr int AUXH = 18 * BN;                                   // halfs of a super-block's block sums and 2^-k (float)
  constexpr int BUF = 4 * STEP + AUXH;                            // !RINGED: halfs of a buffer
  constexpr bool CHUNKED = TYPE == TL_Q4_K || TYPE == TL_Q6_K;
  constexpr bool RINGED = BN > 32;                                // the tile goes through a ring of three 64-column steps
  extern __shared__ __attribute__((aligned(16))) _Float16 hlds[];
  const Place pl = place_of(segs, block);
  QW w = segs.w[pl.seg];
  const HAct act = segs.act;
  const int nt = pl.nt, mt = pl.mt, T = segs.T;
  const int M = w.rows, K = segs.K;
  w.cols = K;  // (known before the matrix is)
  const int sb0 = pl.slice * segs.per, nsb = segs.nsb - sb0 < segs.per ? segs.nsb - sb0 : segs.per;
  const int slast = (K >> 6) - 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fr = lane & (TK - 1), fg = lane / TK;
  const int n0 = nt * BN, m0 = mt * (TK * MI * NW) + wave * (TK * MI);
  unsigned R[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int r = m0 + TK * i + fr;
    R[i] = (unsigned)(r < M ? r : M - 1);
  }
  // staging: this thread's pieces of 64 columns (padding tokens repeat the last one: lines that are read anyway)
  unsigned xg[XR];
  int xl[XR];
#pragma unroll
  for (int r = 0; r < XR; ++r) {
    const int id = (tid + r * NT) % XP, q = id & 7, row = id >> 3, tok = row % BN, part = row / BN;
    xg[r] = (unsigned)((size_t)part * act.ps + (size_t)(n0 + tok < T ? n0 + tok : T - 1) * K + q * 8);
    xl[r] = (tid + r * NT) / XP * STEP + row * 64 + ((q ^ ((row >> 1) & 7)) << 3);
  }
  auto load_x = [&](int r, int sb, int c) {  // 64-column piece c (and on) of super-block sb
    const int s = sb * 4 + c + (tid + r * NT) / XP;
    return *reinterpret_cast<const f16x8*>(act.x + (size_t)(xg[r] + (unsigned)((s < slast ? s : slast) * 64)));
  };
  // 16-byte pieces of a super-block's block sums (2 BN) and powers of two (BN / 4); spare threads copy a piece again
  constexpr int AUX = 2 * BN + BN / 4;
  const int ap = tid % AUX;
  const unsigned char* const abase = reinterpret_cast<const unsigned char*>(act.bs);  // (the powers of two lie ps / 8 bytes behind)
  const unsigned ashift = ap < 2 * BN ? 5u : 2u;
  const unsigned ag = ((unsigned)n0 << ashift) + (unsigned)ap * 16u + (ap < 2 * BN ? 0u : (unsigned)(act.ps >> 3) - 32u * BN);
  const unsigned astride = (unsigned)act.tpad << ashift;
  // fragment reads: where the lane's eight columns of operand k lie in a step's part of the tile
  int xo[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int col = CHUNKED ? 32 * fg + 8 * k : TK == 32 ? 32 * (k >> 1) + 16 * fg + 8 * (k & 1) : 32 * k + 8 * fg;
    xo[k] = (col >> 6) * STEP + fr * 64 + ((((col & 63) >> 3) ^ ((fr >> 1) & 7)) << 3);
  }

  constexpr bool APART = TK == 16 || MI == 1;
  constexpr int WD = US == 4 && NI * MI == 4 ? 2 : US;  // steps the weight loads run ahead: a super-block
  WStep<TYPE> W[MI][WD];
  WHead<TYPE> H[MI], Hn[MI];
  // (in the order in which the first super-block waits for them: the counted waits of the loop depend on it)
#pragma unroll
  for (int i = 0; i < MI; ++i) load_head<TYPE>(H[i], w, R[i], sb0);
  {
    const u32x4 aux = *reinterpret_cast<const u32x4*>(abase + (ag + (unsigned)sb0 * astride));
    constexpr int FIRST = RINGED ? 2 : 1;
    f16x8 xr[FIRST][XR];
#pragma unroll
    for (int c = 0; c < FIRST; ++c)
#pragma unroll
      for (int r = 0; r < XR; ++r) xr[c][r] = load_x(r, sb0, c);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < WD; ++u)
#pragma unroll
      for (int i = 0; i < MI; ++i) load_step<TYPE, TK>(W[i][u], w, R[i], sb0, u, fg);
    __builtin_amdgcn_sched_barrier(0);
    *reinterpret_cast<u32x4*>(hlds + (RINGED ? 3 : 4) * STEP + ap * 8) = aux;
#pragma unroll
    for (int c = 0; c < FIRST; ++c)
#pragma unroll
      for (int r = 0; r < XR; ++r) *reinterpret_cast<f16x8*>(hlds + c * STEP + xl[r]) = xr[c][r];
  }
  int slot = 0;  // RINGED: where the step in hand lies
  const Acc zero = {};
  Acc acc[NI][MI];
#pragma unroll
  for (int n = 0; n < NI; ++n)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[n][i] = zero;
  __syncthreads();

  auto superblock = [&](int b, auto next_c) __attribute__((always_inline)) {
    constexpr bool NEXT = decltype(next_c)::value;  // another super-block follows: fetch it on the way
    const int sb = sb0 + b, cur = b & 1;
    const _Float16* xb = hlds + cur * BUF;
    _Float16* xn = hlds + (cur ^ 1) * BUF;
    const _Float16* ab = RINGED ? hlds + 3 * STEP + cur * AUXH : xb + 4 * STEP;
    _Float16* an = RINGED ? hlds + 3 * STEP + (cur ^ 1) * AUXH : xn + 4 * STEP;
    u32x4 aux;
    if (NEXT) {
      aux = *reinterpret_cast<const u32x4*>(abase + (ag + (unsigned)(sb + 1) * astride));
#pragma unroll
      for (int i = 0; i < MI; ++i) load_head<TYPE>(Hn[i], w, R[i], sb + 1);
    }
    // sums of the hi part's products and of the small ones (lo part; Q6_K's remainders): apart where registers are not
    // short, so that only the former's 16 additions round at the sum's own size, and as two chains. Q8_0: of a 32-column
    // block, c8 adds up the blocks
    Acc t[NI][MI], tl[NI][MI], c8[NI][MI];
    f16x8 xr[XR];
    unsigned h1[MI], h3[MI];
    if (TYPE == TL_Q4_K) {
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        h1[i] = H[i].h[1] >> (4 * fg);
        h3[i] = H[i].h[3] >> (2 * fg);
      }
    }
    // fragment reads run RD operands ahead of their matrix instructions. The compiler's scheduler would sink every load to
    // its use (measured: all of a super-block's loads behind its last matrix instruction); the barriers keep them here
    constexpr int RD = NI == 1 ? 3 : MI == 1 ? 2 : 1, RING = RD + 1, NF = 4 * US * NI;
    f16x8 fa[RING][2];
    auto read_frags = [&](int f, int u) __attribute__((always_inline)) {  // in step u: operand f / NI, token fragment f % NI
      const int kk = f / NI, n = f % NI;
      const _Float16* base = !RINGED ? xb + (kk >> 2) * (NG / 2) * STEP
                                     : hlds + ((kk >> 2) == u ? slot : slot == 2 ? 0 : slot + 1) * STEP;
#pragma unroll
      for (int p = 0; p < PARTS; ++p) fa[f % RING][p] = *reinterpret_cast<const f16x8*>(base + (p * BN + TK * n) * 64 + xo[kk & 3]);
    };
#pragma unroll
    for (int f = 0; f < RD; ++f) read_frags(f, 0);
#pragma unroll
    for (int u = 0; u < US; ++u) {
      if (RINGED && (NEXT || u + 2 < US)) {  // two steps on
#pragma unroll
        for (int r = 0; r < XR; ++r) xr[r] = load_x(r, sb, u + 2);
      } else if (NEXT && u == 0) {
#pragma unroll
        for (int r = 0; r < XR; ++r) xr[r] = load_x(r, sb + 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      Scale4 sc[MI];
      f16x2 s6[MI][2];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        if (TYPE == TL_Q4_K) sc[i] = q4_scale(h1[i], h3[i], NG * u);
        if (TYPE == TL_Q6_K) {
          const unsigned hs = NG == 2 ? H[i].h[u] : (fg & 2) ? H[i].h[(2 * u + 1) & 3] : H[i].h[(2 * u) & 3];
          const unsigned sw = hs >> (16 * (fg & 1));
          const _Float16 a = (_Float16)(short)(signed char)(sw & 0xFFu), c = (_Float16)(short)(signed char)((sw >> 8) & 0xFFu);
          s6[i][0] = f16x2{a, a};
          s6[i][1] = f16x2{c, c};
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int kk = 4 * u + k;
        f16x8 bh[MI], bl[MI];
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          const WStep<TYPE>& g = W[i][u % WD];
          if (TYPE == TL_Q4_K) bh[i] = q4_operand(g.q[k], sc[i]);
          else if (TYPE == TL_Q6_K) q6_operand(g.q[k], g.hi[k >> 1], k & 1, s6[i][k >> 1], bh[i], bl[i]);
          else bh[i] = k < 2 ? q8_operand(g.q[2 * (k & 1)], g.q[2 * (k & 1) + 1]) : q8_operand(g.q1[2 * (k & 1)], g.q1[2 * (k & 1) + 1]);
        }
        // Q8_0: a 32-column block is two operands (TK 32) or one (TK 16)
        const bool fresh = TYPE == TL_Q8_0 ? TK == 16 || (k & 1) == 0 : kk == 0;
#pragma unroll
        for (int n = 0; n < NI; ++n) {
          const int f = kk * NI + n;
          __builtin_amdgcn_sched_barrier(0);
          if (f + RD < NF) read_frags(f + RD, u);
          __builtin_amdgcn_sched_barrier(0);
          const f16x8 a0 = fa[f % RING][0], a1 = fa[f % RING][PARTS - 1];
          if (!STACK) {
#pragma unroll
            for (int i = 0; i < MI; ++i) {
              Acc& c = APART ? tl[n][i] : t[n][i];
              c = TL::mfma(a1, bh[i], fresh ? zero : c);
            }
          }
#pragma unroll
          for (int i = 0; i < MI; ++i) t[n][i] = TL::mfma(a0, bh[i], APART && fresh ? zero : t[n][i]);
          if (TYPE == TL_Q6_K) {
#pragma unroll
            for (int i = 0; i < MI; ++i) {
              Acc& c = APART ? tl[n][i] : t[n][i];
              c = TL::mfma(a0, bl[i], STACK && fresh ? zero : c);
            }
          }
        }
        if (TYPE == TL_Q8_0 && (TK == 16 || (k & 1))) {
          const int blk = TK == 16 ? 4 * u + k : 2 * u + (k >> 1), pair = TK == 16 ? k >> 1 : 0;  // block of the super-block
          const unsigned live = sb * 4 + (blk >> 1) <= slast ? 0xFFFFu : 0u;  // (the row may end inside the super-block)
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            const float d = h2f_scale((W[i][u % WD].d[pair] >> (16 * (blk & 1))) & live);
#pragma unroll
            for (int n = 0; n < NI; ++n) {
#pragma unroll
              for (int e = 0; e < TL::E; ++e) {
                const float c = STACK ? t[n][i][e] : APART ? t[n][i][e] + tl[n][i][e] : t[n][i][e];
                c8[n][i][e] = blk == 0 ? d * c : fmaf(d, c, c8[n][i][e]);
              }
              asm volatile("" : "+v"(c8[n][i]));  // here, not behind the loop (eight blocks' sums would stay live)
            }
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (NEXT || u + WD < US) {
#pragma unroll
        for (int i = 0; i < MI; ++i) load_step<TYPE, TK>(W[i][u % WD], w, R[i], sb + (u + WD) / US, (u + WD) % US, fg);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (RINGED) {
        if (NEXT || u + 2 < US) {  // into the slot that everybody left at the last barrier
#pragma unroll
          for (int r = 0; r < XR; ++r) *reinterpret_cast<f16x8*>(hlds + (slot == 0 ? 2 : slot - 1) * STEP + xl[r]) = xr[r];
        }
        slot = slot == 2 ? 0 : slot + 1;
        if (u < US - 1) __syncthreads();
      } else if (NEXT && u == US - 1) {
#pragma unroll
        for (int r = 0; r < XR; ++r) *reinterpret_cast<f16x8*>(xn + xl[r]) = xr[r];
      }
    }
    add_superblock<TYPE, TK, NI, MI, STACK>(acc, t, tl, c8, H, ab, ab + 16 * BN, fr, fg);
    if (NEXT) {
#pragma unroll
      for (int i = 0; i < MI; ++i) H[i] = Hn[i];
      *reinterpret_cast<u32x4*>(an + ap * 8) = aux;
      __syncthreads();
    }
  };
  for (int b = 0; b + 1 < nsb; ++b) superblock(b, std::true_type{});
  superblock(nsb - 1, std::false_type{});

  float* const y = segs.y[pl.seg] + (size_t)pl.slice * (size_t)T * (size_t)M;  // (slices beyond the first only where there are several)
  store_tile<TK, NI, MI, STACK>(y, segs.resid, acc, n0, m0, T, M, fr, fg);
}

// The same product in workgroups of eight waves and 64 tokens, one on a CU, rows in whole super-blocks: activations and weights go from
// memory to LDS directly (tl_lds_load16), the weights as they lie in memory, so that neither needs registers on the way. In the kernel
// above every step's LDS stores wait for loads asked for one step before, and with them, since loads are counted in order, for the
// weights asked for just before those; here whatever a step asks for has a step and a half to arrive. It also issues an eighth fewer
// vector instructions. The same operands in the same order: the same bits. 28672 x 4096 in Q4_K, us at 128 / 512 / 2048 tokens: 256
// rows 78 / 312 / 1057 -> 74 / 299 / 1006, waves of 64 rows 87 / 290 / 962 -> - / 266 / 892; 16384 x 3072 in Q6_K 72 / 179 / 634 -> 67
// / 160 / 604; 28672 x 4096 in Q8_0 104 / 389 / 1361 -> 97 / 375 / 1272. What bounds it (counters of single launches): the clock falls as
// the matrix cores fill, 28672 x 4096 in Q4_K at 128 / 512 / 2048 tokens 2.2 / 1.9 / 1.6 GHz with the cores busy in 39 / 50 / 60 % of the
// cycles, 16384 x 3072 in Q6_K at 2048 1.7 GHz and 53 %; the two waves of a SIMD wait in 26 to 29 % of theirs for data and barriers and in
// 33 to 42 % for their turn to issue. In Q8_0 (16 additions and FMAs a block) the cores are busy in 30 %, at 2.0 GHz.
// LDS, in bytes: activations of four 64-column steps [part][64 tokens][64] f16; two halves of a super-block of the rows' nibbles (bytes),
// behind them Q6_K's high bits; the rows' heads of two super-blocks (16 bytes and, Q6_K and Q8_K, the dword that d lies in); block sums and
// powers of two of two super-blocks. 16-byte pieces of a row are exchanged so that the 16 rows of a fragment read cover the 64 banks once.
template <int TYPE, int MI, int NW>
struct LdsMap {
  static constexpr int BM = 32 * MI * NW, XSLOT = 64 * 256;
  static constexpr int QROW = TYPE == TL_Q4_K || TYPE == TL_Q6_K ? 64 : 128, HROW = TYPE == TL_Q6_K ? 32 : 0;  // bytes of half a super-block
  static constexpr bool H16 = TYPE != TL_Q8_K, D4 = TYPE == TL_Q6_K || TYPE == TL_Q8_K;
  static constexpr int W = 4 * XSLOT, WSLOT = BM * (QROW + HROW);
  static constexpr int H = W + 2 * WSLOT, HSLOT = BM * ((H16 ? 16 : 0) + (D4 ? 4 : 0));
  static constexpr int A = H + 2 * HSLOT, ASLOT = 64 * 32 + 1024;
  static constexpr int BYTES = A + 2 * ASLOT;
};
template <int TYPE, int MI, int NW>
__device__ __forceinline__ void hgemm_lds_body(const HSegs& segs, int block) {
  typedef LdsMap<TYPE, MI, NW> L;
  typedef Tile<32> TL;
  typedef f32x16 Acc;
  constexpr int NI = 2, US = 4, BN = 64, BM = L::BM;
  constexpr bool CHUNKED = TYPE == TL_Q4_K || TYPE == TL_Q6_K, APART = MI == 1;
  static_assert(NW == 8 && (MI == 1 || MI == 2), "");
  extern __shared__ __attribute__((aligned(16))) _Float16 hlds[];
  unsigned char* const lds = reinterpret_cast<unsigned char*>(hlds);
  const Place pl = place_of(segs, block);
  const QW w = segs.w[pl.seg];
  const HAct act = segs.act;
  const int M = w.rows, K = segs.K, T = segs.T;
  const int nsb_all = segs.nsb;
  const int sb0 = __builtin_amdgcn_readfirstlane(pl.slice * segs.per), nsb = nsb_all - sb0 < segs.per ? nsb_all - sb0 : segs.per;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, fg = lane >> 5;
  const int n0 = pl.nt * BN, tile0 = pl.mt * BM, m0 = tile0 + wave * 32 * MI;
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)lds;
  auto row_at = [&](int r) { return (unsigned)(r < M ? r : M - 1); };  // (rows beyond the last: its values, never stored)
  // what this lane fetches: 16-byte pieces of the activations, of the wave's rows, of 64 rows' heads (MI 1: two waves fetch the same)
  constexpr int XI = 16 / NW, QI = MI * L::QROW / 32, HI = L::HROW ? MI : 0;
  unsigned xoff[XI], qoff[QI], hoff[HI ? HI : 1];
  const int xpart = wave >= NW / 2;  // (a wave's pieces are of one part)
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int tok = ((wave * XI + i) * 8 + (lane >> 3)) & (BN - 1);
    const int t = n0 + tok < T ? n0 + tok : T - 1;
    xoff[i] = ((unsigned)t * (unsigned)K + (((lane & 7) ^ ((tok >> 1) & 7)) << 3)) * 2u;
  }
  const char* xbase = tl_uniform(reinterpret_cast<const char*>(act.x + (xpart ? act.ps : 0)));
#pragma unroll
  for (int i = 0; i < QI; ++i) {
    const int row = L::QROW == 64 ? i * 16 + (lane >> 2) : i * 8 + (lane >> 3);
    const int piece = L::QROW == 64 ? (lane & 3) ^ ((row >> 2) & 3) : (lane & 7) ^ ((row >> 1) & 7);
    qoff[i] = row_at(m0 + row) * (unsigned)(CHUNKED ? K >> 1 : K) + (piece << 4);
  }
#pragma unroll
  for (int i = 0; i < HI; ++i) {
    const int row = i * 32 + (lane >> 1);
    hoff[i] = row_at(m0 + row) * (unsigned)(K >> 2) + (((lane & 1) ^ ((row >> 3) & 1)) << 4);
  }
  const int head64 = MI == 1 ? wave >> 1 : wave;
  const unsigned hrow = row_at(tile0 + head64 * 64 + lane), headoff = hrow * (unsigned)(K >> 4), drow = hrow * (unsigned)nsb_all;
  const unsigned char *q_base = tl_uniform(w.p0), *hi_base = tl_uniform(w.p1);
  const unsigned char* head_base = tl_uniform(TYPE == TL_Q6_K ? w.p2 : w.p1);
  const unsigned char* d_base = tl_uniform(TYPE == TL_Q6_K ? w.p3 : w.p1);
  const int apiece = wave % 3;  // two of block sums, one of powers of two
  const char* abase = tl_uniform(apiece < 2 ? reinterpret_cast<const char*>(act.bs + (size_t)n0 * 16) + apiece * 1024 : reinterpret_cast<const char*>(act.inv + n0));
  const unsigned astride = __builtin_amdgcn_readfirstlane((unsigned)act.tpad * (apiece < 2 ? 32 : 4));
  const unsigned aoff = (apiece < 2 ? lane : lane & 15) * 16;

  auto fetch_x = [&](int sb, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XI; ++i) tl_lds_load16(lds0 + c * L::XSLOT + (wave * XI + i) * 1024, xoff[i], xbase + (size_t)(sb * 4 + c) * 128);
  };
  auto fetch_w = [&](int sb, int h) __attribute__((always_inline)) {
    const unsigned b = lds0 + L::W + h * L::WSLOT;
#pragma unroll
    for (int i = 0; i < QI; ++i) tl_lds_load16(b + wave * (32 * MI * L::QROW) + i * 1024, qoff[i], q_base + (size_t)(2 * sb + h) * L::QROW);
#pragma unroll
    for (int i = 0; i < HI; ++i) tl_lds_load16(b + BM * L::QROW + (wave * MI + i) * 1024, hoff[i], hi_base + (size_t)(2 * sb + h) * L::HROW);
  };
  auto fetch_head = [&](int sb, int par) __attribute__((always_inline)) {
    const unsigned b = lds0 + L::H + par * L::HSLOT;
    if (L::H16) tl_lds_load16(b + head64 * 1024, headoff, head_base + (size_t)sb * 16);
    // (the aligned dword around a 2-byte d: a plane is a whole number of 256 bytes)
    if (L::D4) tl_lds_load4(b + (L::H16 ? BM * 16 : 0) + head64 * 256, ((drow + sb) & ~1u) * 2u, d_base);
  };
  auto fetch_aux = [&](int sb, int par) __attribute__((always_inline)) {
    tl_lds_load16(lds0 + L::A + par * L::ASLOT + apiece * 1024, aoff, abase + (size_t)sb * astride);
  };
  constexpr int WLOADS = QI + HI, HLOADS = (L::H16 ? 1 : 0) + (L::D4 ? 1 : 0);
  // what this lane reads: its eight columns of operand k in a step's activations, its weights of odd and even steps
  int xo[4], qo[2][2], ho[2];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int piece = CHUNKED ? 4 * fg + k : 4 * (k >> 1) + 2 * fg + (k & 1);
    xo[k] = (fr * 128 + ((piece ^ ((fr >> 1) & 7)) << 4)) / 2;
  }
#pragma unroll
  for (int o = 0; o < 2; ++o) {
    if (L::QROW == 64) {
      qo[o][0] = fr * 64 + (((2 * o + fg) ^ ((fr >> 2) & 3)) << 4);
      qo[o][1] = 0;
    } else {
#pragma unroll
      for (int k = 0; k < 2; ++k) qo[o][k] = fr * 128 + (((4 * o + 2 * k + fg) ^ ((fr >> 1) & 7)) << 4);
    }
    ho[o] = fr * 32 + ((o ^ ((fr >> 3) & 1)) << 4) + fg * 8;
  }
  auto read_w = [&](WStep<TYPE>(&g)[MI], int u) __attribute__((always_inline)) {
    const unsigned char* b = lds + L::W + (u >> 1) * L::WSLOT;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const unsigned char* r = b + (wave * MI + i) * (32 * L::QROW);
      g[i].q = *reinterpret_cast<const u32x4*>(r + qo[u & 1][0]);
      if (L::QROW == 128) g[i].q1 = *reinterpret_cast<const u32x4*>(r + qo[u & 1][1]);
      if (L::HROW) g[i].hi = *reinterpret_cast<const u32x2*>(b + BM * L::QROW + (wave * MI + i) * 1024 + ho[u & 1]);
    }
  };
  auto read_head = [&](WHead<TYPE>(&g)[MI], int sb, int par) __attribute__((always_inline)) {
    const unsigned char* b = lds + L::H + par * L::HSLOT;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int row = (wave * MI + i) * 32 + fr;
      if (L::H16) g[i].h = *reinterpret_cast<const u32x4*>(b + row * 16);
      if (L::D4) {
        const unsigned two = *reinterpret_cast<const unsigned*>(b + (L::H16 ? BM * 16 : 0) + row * 4);
        g[i].d = (two >> (16 * ((row_at(tile0 + row) * (unsigned)nsb_all + sb) & 1))) & 0xFFFFu;
      }
    }
  };

  const Acc zero = {};
  Acc acc[NI][MI];
#pragma unroll
  for (int n = 0; n < NI; ++n)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[n][i] = zero;
  WStep<TYPE> W[2][MI];
  WHead<TYPE> H[MI], Hn[MI];
  fetch_head(sb0, 0);
  fetch_w(sb0, 0);
  fetch_x(sb0, 0);
  fetch_x(sb0, 1);
  fetch_aux(sb0, 0);
  fetch_w(sb0, 1);
  fetch_x(sb0, 2);
  tl_lds_barrier<0>();
  read_head(H, sb0, 0);
  read_w(W[0], 0);

  auto superblock = [&](int b, auto next_c) __attribute__((always_inline)) {
    constexpr bool NEXT = decltype(next_c)::value;  // another super-block follows: fetch it on the way
    const int sb = __builtin_amdgcn_readfirstlane(sb0 + b), cur = __builtin_amdgcn_readfirstlane(b & 1);  // (scalar: bases of loads)
    const _Float16* ab = hlds + (L::A + cur * L::ASLOT) / 2;
    Acc t[NI][MI], tl[NI][MI], c8[NI][MI];  // (as above)
    unsigned h1[MI], h3[MI];
    if (TYPE == TL_Q4_K) {
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        h1[i] = H[i].h[1] >> (4 * fg);
        h3[i] = H[i].h[3] >> (2 * fg);
      }
    }
    constexpr int RD = MI == 1 ? 2 : 1, RING = RD + 1, NF = 4 * US * NI;
    f16x8 fa[RING][2];
    auto read_frags = [&](int f) __attribute__((always_inline)) {  // operand f / NI of the super-block, token fragment f % NI
      const int kk = f / NI, n = f % NI;
#pragma unroll
      for (int p = 0; p < 2; ++p)
        fa[f % RING][p] = *reinterpret_cast<const f16x8*>(hlds + ((kk >> 2) * L::XSLOT + (p * BN + 32 * n) * 128) / 2 + xo[kk & 3]);
    };
#pragma unroll
    for (int f = 0; f < RD; ++f) read_frags(f);
#pragma unroll
    for (int u = 0; u < US; ++u) {
      // Step u of the super-block lies in slot u and is read up to its barrier, the next step from its own start on. What a step asks for is
      // there at the barrier of the step after: activations three steps ahead, into the slot of the step before; the next
      // super-block's weights as soon as both steps of a half have been read into registers (a step ahead); heads and block sums
      // where the other super-block's are long read
      if (u == 0) fetch_x(sb, 3);
      else if (NEXT) fetch_x(sb + 1, u - 1);
      if (NEXT && u == 1) {
        fetch_w(sb + 1, 0);
        fetch_head(sb + 1, cur ^ 1);
      }
      if (NEXT && u == 2) fetch_aux(sb + 1, cur ^ 1);
      if (NEXT && u == 3) fetch_w(sb + 1, 1);
      if (NEXT || u < US - 1) read_w(W[(u + 1) & 1], (u + 1) & 3);
      if (NEXT && u == 3) read_head(Hn, sb + 1, cur ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      Scale4 sc[MI];
      f16x2 s6[MI][2];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        if (TYPE == TL_Q4_K) sc[i] = q4_scale(h1[i], h3[i], 2 * u);
        if (TYPE == TL_Q6_K) {
          const unsigned sw = H[i].h[u] >> (16 * fg);
          const _Float16 a = (_Float16)(short)(signed char)(sw & 0xFFu), c = (_Float16)(short)(signed char)((sw >> 8) & 0xFFu);
          s6[i][0] = f16x2{a, a};
          s6[i][1] = f16x2{c, c};
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int kk = 4 * u + k;
        f16x8 bh[MI], bl[MI];
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          const WStep<TYPE>& g = W[u & 1][i];
          if (TYPE == TL_Q4_K) bh[i] = q4_operand(g.q[k], sc[i]);
          else if (TYPE == TL_Q6_K) q6_operand(g.q[k], g.hi[k >> 1], k & 1, s6[i][k >> 1], bh[i], bl[i]);
          else bh[i] = k < 2 ? q8_operand(g.q[2 * (k & 1)], g.q[2 * (k & 1) + 1]) : q8_operand(g.q1[2 * (k & 1)], g.q1[2 * (k & 1) + 1]);
        }
        const bool fresh = TYPE == TL_Q8_0 ? (k & 1) == 0 : kk == 0;
#pragma unroll
        for (int n = 0; n < NI; ++n) {
          const int f = kk * NI + n;
          __builtin_amdgcn_sched_barrier(0);
          if (f + RD < NF) read_frags(f + RD);
          __builtin_amdgcn_sched_barrier(0);
          const f16x8 a0 = fa[f % RING][0], a1 = fa[f % RING][1];
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            Acc& c = APART ? tl[n][i] : t[n][i];
            c = TL::mfma(a1, bh[i], fresh ? zero : c);
          }
#pragma unroll
          for (int i = 0; i < MI; ++i) t[n][i] = TL::mfma(a0, bh[i], APART && fresh ? zero : t[n][i]);
          if (TYPE == TL_Q6_K) {
#pragma unroll
            for (int i = 0; i < MI; ++i) {
              Acc& c = APART ? tl[n][i] : t[n][i];
              c = TL::mfma(a0, bl[i], c);
            }
          }
        }
        if (TYPE == TL_Q8_0 && (k & 1)) {
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            const float d = h2f_scale((H[i].h[u] >> (16 * (k >> 1))) & 0xFFFFu);
#pragma unroll
            for (int n = 0; n < NI; ++n) {
#pragma unroll
              for (int e = 0; e < 16; ++e) {
                const float c = APART ? t[n][i][e] + tl[n][i][e] : t[n][i][e];
                c8[n][i][e] = kk == 1 ? d * c : fmaf(d, c, c8[n][i][e]);
              }
              asm volatile("" : "+v"(c8[n][i]));
            }
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (NEXT) {
        if (u == 0) tl_lds_barrier<XI>();
        if (u == 1) tl_lds_barrier<XI + WLOADS + HLOADS>();
        if (u == 2) tl_lds_barrier<XI + 1>();
        if (u == 3) tl_lds_barrier<XI + WLOADS>();
      } else {
        if (u == 0) tl_lds_barrier<XI>();
        if (u == 1) tl_lds_barrier<0>();
      }
    }
    add_superblock<TYPE, 32, NI, MI, false>(acc, t, tl, c8, H, ab, ab + 16 * BN, fr, fg);
    if (NEXT) {
#pragma unroll
      for (int i = 0; i < MI; ++i) H[i] = Hn[i];
    }
  };
  for (int b = 0; b + 1 < nsb; ++b) superblock(b, std::true_type{});
  superblock(nsb - 1, std::false_type{});
  float* const y = segs.y[pl.seg] + (size_t)pl.slice * (size_t)T * (size_t)M;
  store_tile<32, NI, MI, false>(y, segs.resid, acc, n0, m0, T, M, fr, fg);
}

// ---- producer of the activation planes ----------------------------------------------------------------------------------
// MODE 0: x; 1: rmsnorm_batch(x, aux = weight, eps) (utils.cpp:613-646); 2: swiglu(x, aux) (cpu_batch_processor.cpp:252-256).
// a / b: pending K-split sums (see tl_launch_split); RMSNORM with a pending projection writes the new residual row to xout.
// 8 columns per thread, so a super-block is half a wave. RMSNORM: one workgroup per token, NIT pieces of 8 columns per
// thread; else grid.y covers the row.
// (S <= 8; the loads of all slices are in flight together, four at a time: one after another they are S round trips to L2)
__device__ __forceinline__ f32x4 hparts4(const GemmParts& g, size_t o) {
  auto ld = [&](int z) { return *reinterpret_cast<const f32x4*>(g.part + (size_t)z * g.n + o); };
  f32x4 acc = ld(0);
  int z = 1;
  for (; z + 4 <= g.S; z += 4) {
    const f32x4 a = ld(z), b = ld(z + 1), c = ld(z + 2), d = ld(z + 3);
    acc = acc + a + b + c + d;
  }
  if (z + 2 <= g.S) {
    const f32x4 a = ld(z), b = ld(z + 1);
    acc = acc + a + b;
    z += 2;
  }
  if (z < g.S) acc += ld(z);
  return acc;
}
constexpr int HNORM_THREADS = 512, HMAX_COLS = 8 * 8 * HNORM_THREADS;
// WIDE (a piece a thread; launches whose workgroups are all on the chip at once, so that registers cost nothing): the row, the weights and
// all slices in one round trip. In whole calls: 8 rows of 3072, 2 to 8 slices, 5.06 -> 4.03 us on average, 128 of 4096 7.47 -> 6.53; gate and
// up of 8 x 8192 (hsplit_kernel) 4.50 -> 3.65.
template <int NIT, bool WIDE>
__global__ __launch_bounds__(HNORM_THREADS) void hsplit_norm_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                    _Float16* __restrict__ planes, size_t ps, int K, float eps,
                                                                    GemmParts a, float* __restrict__ xout, int tpad) {
  __shared__ float red[HNORM_THREADS / 64];
  const int t = blockIdx.x, tid = threadIdx.x;
  const size_t row = (size_t)t * K;
  float v[NIT][8];
  float ssq = 0.f;
  f32x4 wv[2];
  if constexpr (WIDE) {
    const int i0 = tid * 8;
    const bool in = i0 < K;
    const size_t o = row + (in ? i0 : 0);
    f32x4 p[2], q[1][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      p[h] = *reinterpret_cast<const f32x4*>(x + o + 4 * h);
      wv[h] = *reinterpret_cast<const f32x4*>(w + (in ? i0 : 0) + 4 * h);
    }
    const GemmParts g[1] = {a};
    if (a.S) tl_parts_sum(g, o, q);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (a.S) {
        p[h] += q[0][h];
        if (in) *reinterpret_cast<f32x4*>(xout + o + 4 * h) = p[h];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[0][4 * h + e] = in ? p[h][e] : 0.f;
        ssq = fmaf(v[0][4 * h + e], v[0][4 * h + e], ssq);
      }
    }
  }
#pragma unroll
  for (int it = 0; it < (WIDE ? 0 : NIT); ++it) {
    const int i0 = (it * HNORM_THREADS + tid) * 8;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 p = {0.f, 0.f, 0.f, 0.f};
      if (i0 < K) {
        const size_t o = row + i0 + 4 * h;
        p = *reinterpret_cast<const f32x4*>(x + o);
        if (a.S) {
          p += hparts4(a, o);
          *reinterpret_cast<f32x4*>(xout + o) = p;
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[it][4 * h + e] = p[e];
        ssq = fmaf(p[e], p[e], ssq);
      }
    }
  }
  ssq = tl_wave_sum(ssq);
  if ((tid & 63) == 0) red[tid >> 6] = ssq;
  __syncthreads();
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < HNORM_THREADS / 64; ++i) sum += red[i];
  const float nf = 1.0f / sqrtf(sum / (float)K + eps);
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int i0 = (it * HNORM_THREADS + tid) * 8;
    if (i0 < K) {
      if (!WIDE) {
        wv[0] = *reinterpret_cast<const f32x4*>(w + i0);
        wv[1] = *reinterpret_cast<const f32x4*>(w + i0 + 4);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) v[it][e] = v[it][e] * nf * wv[e >> 2][e & 3];
    }
    tl_hsplit8(v[it], planes, ps, t, K, i0, tpad);
  }
}
template <int MODE, bool WIDE>
__global__ __launch_bounds__(256) void hsplit_kernel(const float* __restrict__ x, const float* __restrict__ aux,
                                                     _Float16* __restrict__ planes, size_t ps, int K, GemmParts a, GemmParts b,
                                                     int tpad) {
  const int t = blockIdx.x, i0 = (blockIdx.y * 256 + threadIdx.x) * 8;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (WIDE && i0 < K) {  // (both products in the same number of slices)
    const GemmParts g[2] = {a, b};
    f32x4 p[2][2];
    tl_parts_sum(g, (size_t)t * K + i0, p);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (p[0][e >> 2][e & 3] / (1.0f + expf(-p[0][e >> 2][e & 3]))) * p[1][e >> 2][e & 3];
  } else if (i0 < K) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const size_t o = (size_t)t * K + i0 + 4 * h;
      f32x4 p = MODE == 2 && a.S ? hparts4(a, o) : *reinterpret_cast<const f32x4*>(x + o);
      if (MODE == 2) {
        const f32x4 up = b.S ? hparts4(b, o) : *reinterpret_cast<const f32x4*>(aux + o);
#pragma unroll
        for (int e = 0; e < 4; ++e) p[e] = (p[e] / (1.0f + expf(-p[e]))) * up[e];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * h + e] = p[e];
    }
  }
  tl_hsplit8(v, planes, ps, t, K, i0, tpad);
}

// The shapes of a workgroup. Up to 8 tokens: both parts of a token's activations in the 16 rows of one matrix instruction (stack), 64 or
// 128 rows of weights a workgroup; up to 16: the same with an instruction for either part. Up to 32: 64 rows in 16-row waves
// (8) or 128 in 32-row waves (1), both two workgroups on a CU, whose LDS two super-blocks of 32 tokens fill. Up to 64: these, or the 64-token tiles of long chunks. More: 64-token tiles, each operand
// unpacked once for two token fragments, in workgroups of 256 rows (2), of 512 in waves of 64 (3; Q4_K: for others registers or LDS are
// short) and of 128, two on a CU (4). Which of them is taken is a matter of filling the chip, so the plan below weighs them.
// (8 layers of the 8B shape in ms, this kernel / the bf16 kernels it replaced: 8 sequences 0.86 / 1.56, 32: 1.05 / 1.62,
// 64: 1.52 / 2.03, 128: 2.2 / 2.7; a prompt of 512: 5.3 / 7.0.)
struct HShape {
  int tk, ni, mi, nw, wpe, percu;
  bool lds, stack;  // lds: hgemm_lds_body
};
constexpr int HGEMM_SHAPES = 9;
constexpr HShape hgemm_shape(int type, int shape) {
  constexpr HShape all[HGEMM_SHAPES] = {
      {16, 1, 1, 4, 4, 4, false, false}, {32, 1, 1, 4, 2, 2, false, false}, {32, 2, 1, 8, 2, 1, true, false},
      {32, 2, 2, 8, 2, 1, true, false},  {32, 2, 1, 4, 2, 2, false, false}, {16, 1, 1, 4, 4, 4, false, true},
      {16, 1, 1, 8, 4, 2, false, true},  {16, 1, 1, 8, 4, 2, false, false}, {16, 2, 1, 4, 3, 2, false, false}};
  if (shape == 3 && type != TL_Q4_K) return {32, 2, 2, 4, 2, 2, false, false};  // (Q8_K)
  return all[shape];
}
constexpr int hgemm_tokens(const HShape& q) { return q.stack ? 8 : q.tk * q.ni; }
template <int TYPE, int V>
constexpr size_t hgemm_lds_bytes() {
  constexpr HShape q = hgemm_shape(TYPE, V);
  constexpr int BN = hgemm_tokens(q);
  constexpr size_t lds = q.lds ? (size_t)LdsMap<TYPE, q.mi, q.nw>::BYTES
                               : (size_t)(BN > 32 ? 3 * 2 * 64 + 2 * 18 : 2 * (4 * 2 * 64 + 18)) * BN * sizeof(_Float16);
  static_assert(q.percu * lds <= 160 * 1024, "hgemm_price counts on `percu` workgroups on a CU");
  return lds;
}
template <int TYPE, int V>
__device__ __forceinline__ void hgemm_any(const HSegs& g, int block) {
  constexpr HShape q = hgemm_shape(TYPE, V);
  if constexpr (q.lds) hgemm_lds_body<TYPE, q.mi, q.nw>(g, block);
  else hgemm_body<TYPE, q.tk, q.ni, q.mi, q.nw, q.stack>(g, block);
}
template <int TYPE, int V>
__global__ __launch_bounds__(64 * hgemm_shape(TYPE, V).nw, hgemm_shape(TYPE, V).wpe) void hgemm_kernel(const HSegs g) {
  hgemm_any<TYPE, V>(g, blockIdx.x);
}
// Matrices of two formats over the same activations (Q4_K files hold v as Q6_K in some layers, q and k as Q4_K): the longer workgroups
// first, and the others fill up what they leave of the chip. A launch of v's 1024 x 3072 alone is 48 workgroups and 6 us for 8 tokens. Steps of
// 8 sequences, 3B, half of whose layers hold v so, 1.79 -> 1.74 ms; 128 sequences, 8B, 7.5 -> 7.3; whole prompts of 9 to 1900 tokens, 1.1B, 3B
// and 8B, 0 to 4 % less.
struct HPair {
  HSegs q6, q4;
  int first;  // workgroups of q6
};
template <int V6, int V4>
__global__ __launch_bounds__(64 * hgemm_shape(TL_Q4_K, V4).nw, hgemm_shape(TL_Q4_K, V4).wpe) void hgemm_pair_kernel(const HPair p) {
  if ((int)blockIdx.x < p.first) hgemm_any<TL_Q6_K, V6>(p.q6, blockIdx.x);
  else hgemm_any<TL_Q4_K, V4>(p.q4, blockIdx.x - p.first);
}
// Up to 64 tokens a launch takes, in us with weights that no cache holds, its start and end (a quarter of that again for every further
// round over the chip) and, of the CU with the most workgroups, all their super-blocks one after another: co-resident ones share the issue
// slots and the CU's way to memory, so none of them is free. Fitted to 2048 .. 28672 rows of 2048 .. 14336 columns times 8, 16, 24, 32 and
// 48 tokens in 1 to 8 slices (rms 5 to 10 % a shape); the choice by it is within 1 % of the best of all on average (11 % at worst), and
// against one shape and rounds over the chip a launch got 10 to 12 % shorter at 8 tokens, 8 to 10 at 16, 9 to 11 at 32, 11 to 14 at 48
// (Q4_K, 8 tokens: 16384 x 3072 12.5 -> 11.0 us, 4096 x 14336 14.6 -> 12.6; 48 tokens: 28672 x 4096 51.5 -> 39.4).
struct HFew {
  float start, superblock[4];  // Q4_K, Q6_K, Q8_0, Q8_K
};
constexpr HFew HGEMM_FEW[HGEMM_SHAPES] = {
    {4.0f, {0.80f, 1.15f, 1.54f, 1.26f}}, {5.7f, {1.43f, 2.20f, 2.46f, 1.72f}}, {9.0f, {3.18f, 4.65f, 4.58f, 3.09f}},
    {},                                   {7.2f, {2.40f, 3.28f, 3.56f, 2.68f}}, {4.0f, {0.67f, 1.01f, 1.41f, 1.09f}},
    {4.5f, {0.98f, 1.66f, 2.66f, 2.00f}}, {4.8f, {1.09f, 1.79f, 2.76f, 2.08f}}, {4.9f, {1.10f, 1.49f, 1.75f, 1.41f}}};
// Beyond: us of a super-block of a workgroup on a full chip. Shape 3 is priced so that, over the projections of the 1B, 3B and 8B shapes
// and 65 to 2048 tokens, it is taken as often as where it ran in pairs of 256 rows (at its own 7.4 it would be taken in a sixth more of
// them, and its single chain of sums rounds more: 2.1e-7 against 1.7e-7 at 2048 columns)
constexpr float HGEMM_US[] = {0.f, 0.f, 4.25f, 7.8f, 5.0f}, HGEMM_US_3_Q8_K = 9.0f;
constexpr float HGEMM_US_Q6_K[] = {0.f, 0.f, 6.3f, 0.f, 6.85f}, HGEMM_US_Q8_0[] = {0.f, 0.f, 5.5f, 0.f, 6.0f};
constexpr float HGEMM_ENDS = 0.6f;  // start and end of a workgroup of these two, in its super-blocks
// partial sums: of a slice, and of a number of it (Q6_K and Q8_0 beyond 64 tokens: 1.4e-6)
constexpr float HGEMM_SLICE_US = 0.3f, HGEMM_SUM_US = 2e-6f;
// Price of a launch over T tokens of n workgroups of `per` super-blocks, and of S slices' partial sums of `outputs` numbers.
// Q4_K and Q8_K beyond 64 tokens: rounds over the chip x (super-blocks + start and end) + the partial sums written and read once at about
// 4 TB/s. Q6_K (a third product, longer unpacking) and Q8_0 (16 additions and FMAs a block): the
// time of the fullest CU, whose last workgroup takes 0.6 of a pair's time where two share it, and 0.16 of the way to what an even
// share would take (clocks rise where CUs run dry). Over the projections of the 1B, 3B and 8B shapes and 100 to 2048 tokens that
// picks within 0.7 % (Q6_K), 1 % (Q8_0) and 2 % (Q4_K) of the best shape and slices on average and 11, 11 and 20 % at worst.
float hgemm_price(int cus, int type, int shape, int T, long n, int per, int S, float outputs) {
  const HShape q = hgemm_shape(type, shape);
  const long most = (n + cus - 1) / cus, rounds = (most + q.percu - 1) / q.percu;
  const float sums = S > 1 ? (float)S * (HGEMM_SLICE_US + outputs * HGEMM_SUM_US) : 0.f;
  if (T <= 64) {
    const HFew& f = HGEMM_FEW[shape];
    return f.start * (0.75f + 0.25f * (float)rounds) + (float)(most * per) * f.superblock[type == TL_Q4_K ? 0 : type == TL_Q6_K ? 1 : type == TL_Q8_0 ? 2 : 3] + sums;
  }
  if (type == TL_Q6_K || type == TL_Q8_0) {
    const float us = (type == TL_Q6_K ? HGEMM_US_Q6_K : HGEMM_US_Q8_0)[shape], alone = q.percu == 2 ? 0.6f : 1.f;
    const float fullest = q.percu == 2 ? (float)(most / 2) + (most & 1 ? alone : 0.f) : (float)most;
    const float even = (float)n / (float)cus / (float)q.percu;
    return (0.84f * fullest + 0.16f * (even > alone ? even : alone)) * ((float)per + HGEMM_ENDS) * us + (S > 1 ? (float)S * (HGEMM_SLICE_US + outputs * 1.4e-6f) : 0.f);
  }
  return (float)rounds * (float)(per + 1) * (shape == 3 && !q.lds ? HGEMM_US_3_Q8_K : HGEMM_US[shape]) + sums;
}
// the shape and the K slices of the least price, which is added to *sum
HgemmPlan hgemm_plan(const QW* w, int n, int T, float* sum = nullptr) {
  const int nsb = (w[0].cols + 255) / 256, type = w[0].type, cus = tl_num_cus();  // (the call asks the runtime: once a plan)
  const unsigned few = T <= 8 ? 1u << 5 | 1u << 6 : T <= 16 ? 1u << 0 | 1u << 7 : 1u << 1 | 1u << 8, many = 1u << 2 | 1u << 4;
  const unsigned shapes = T <= 32 ? few : T <= 64 ? few | many : many | 1u << 3;  // (shape 3 sums in one chain: not for few tokens)
  HgemmPlan best = {};
  float least = -1.f;
  for (int v = 0; v < HGEMM_SHAPES; ++v) {
    if (!(shapes >> v & 1)) continue;
    if (v == 3 && (type == TL_Q6_K || type == TL_Q8_0)) continue;  // (spills)
    if (v == 2 && w[0].cols % 256) continue;                       // (rows that end inside a super-block)
    const HShape q = hgemm_shape(type, v);
    const int bm = q.tk * q.mi * q.nw, bn = hgemm_tokens(q), ntiles = (T + bn - 1) / bn;
    long tiles = 0, rows = 0;
    for (int i = 0; i < n; ++i) {
      tiles += (long)((w[i].rows + bm - 1) / bm) * ntiles;
      rows += w[i].rows;
    }
    for (int S = 1; S <= 8 && S <= nsb; ++S) {
      const int per = (nsb + S - 1) / S;
      if ((nsb + per - 1) / per != S) continue;  // (no empty slice)
      const float price = hgemm_price(cus, type, v, T, tiles * S, per, S, (float)T * (float)rows);
      if (least < 0.f || price < least) {
        least = price;
        best = {v, S};
      }
    }
  }
  if (sum) *sum += least;
  return best;
}

// Price of one launch over both (HPair), as hgemm_price for its workgroups: their super-blocks one after another on the CU that has most of
// them, the longer workgroups dealt first. A launch takes no less than an even share of all super-blocks and its partial sums: where that is
// more than `most_price` it is the answer (a plan weighs some 36 pairs of slices a shape, in front of a prompt's first launches: a host's time
// for a plan of 4096 columns with 8 / 64 / 2000 tokens 1.5 / 2.4 / 2.5 us without, 1.5 / 1.8 / 1.2 with; of 8192 2.5 / 4.6 / 6.6 and 1.7 / 2.3 / 1.5)
float hgemm_pair_price(int cus, int v6, int v4, int T, long n6, int per6, int S6, long n4, int per4, int S4, float outputs6, float outputs4,
                       float most_price) {
  const bool few = v4 != 2 && v4 != 3;
  const HFew& f = HGEMM_FEW[v4];
  const float t6 = few || T <= 64 ? (float)per6 * f.superblock[1] : ((float)per6 + HGEMM_ENDS) * HGEMM_US_Q6_K[v6];
  const float t4 = few || T <= 64 ? (float)per4 * f.superblock[0] : (float)(per4 + 1) * HGEMM_US[v4];
  const int S = S6 > S4 ? S6 : S4;
  const float sums = (S > 1 ? HGEMM_SLICE_US * (float)S : 0.f) + HGEMM_SUM_US * ((S6 > 1 ? (float)S6 * outputs6 : 0.f) + (S4 > 1 ? (float)S4 * outputs4 : 0.f));
  const float even = 0.999f * ((float)n6 * t6 + (float)n4 * t4) / (float)cus + sums + (few || T <= 64 ? f.start : 0.f);  // (0.999: roundings of the loads below)
  if (even > most_price) return even;
  // the CUs' loads: `more` of them at `high`, the others at `low`
  const bool six = t6 >= t4;
  const float tb = six ? t6 : t4, ts = six ? t4 : t6;
  const long nb = six ? n6 : n4;
  long ns = six ? n4 : n6, more = nb % cus;
  float low = (float)(nb / cus) * tb, high = more ? low + tb : low;
  if (!more) more = cus;
  float top = high;
  while (ns > 0) {  // a shorter one for each of the CUs with the least
    const long least = low < high ? cus - more : more;
    float& at = low < high ? low : high;
    if (ns < least || more == cus) {
      const long rounds = more == cus ? (ns + cus - 1) / cus : 1;
      at += (float)rounds * ts;
      ns = 0;
    } else {
      at += ts;
      ns -= least;
    }
    top = at > top ? at : top;
  }
  if (!few && T > 64) return top + sums;
  const long most = (n6 + n4 + cus - 1) / cus, percu = hgemm_shape(TL_Q4_K, v4).percu, rounds = (most + percu - 1) / percu;
  return f.start * (0.75f + 0.25f * (float)rounds) + top + sums;
}

// tiles and constants of the launch's division into workgroups; returns their number
int hgemm_grid(HSegs& g, const QW* w, int n, const HShape& q, const HAct& act, float* const* out, const float* resid, int T, int S) {
  const int bm = q.tk * q.mi * q.nw, BN = hgemm_tokens(q);
  int mt = 0;
  g.T = T;
  g.K = w[0].cols;
  g.nsb = (w[0].cols + 255) / 256;
  g.resid = resid;
  g.act = act;
  for (int i = 0; i < 3; ++i) {
    const int k = i < n ? i : n - 1;  // (unused slots repeat the last matrix; their tile range is empty)
    g.w[i] = w[k];
    g.y[i] = out[k];
    if (i < n) mt += (w[i].rows + bm - 1) / bm;
    if (i < 2) g.mt_end[i] = mt;
  }
  // panels of eight token tiles and more, all alike: a panel of the one tile that is left over reads all weights again for it (28672 x
  // 4096 in Q4_K times 513 tokens, nine tiles, 274 us in one panel of shape 3 with 256 rows, 281 in eight and one)
  const int ntiles = (T + BN - 1) / BN, panels = ntiles < 16 ? 1 : ntiles / 8, panel = (ntiles + panels - 1) / panels;
  g.per = (g.nsb + S - 1) / S;
  g.per8 = mt * ntiles * S / 8;
  g.rem8 = mt * ntiles * S % 8;
  g.slice_tiles = mt * ntiles;
  g.panel = panel;
  g.panel_tiles = panel * mt;
  g.last_panel = (ntiles - 1) / panel;
  g.width_last = ntiles - g.last_panel * panel;
  g.by_slice = Div::by(g.slice_tiles);
  g.by_panel = Div::by(g.panel_tiles);
  g.by_width = Div::by(panel);
  g.by_last = Div::by(g.width_last);
  return mt * ntiles * S;
}
template <int TYPE, int V>
int hgemm_go(const HSegs& g, int blocks, hipStream_t s) {
  static TlDeviceOnce lds_raised;
  constexpr size_t lds = hgemm_lds_bytes<TYPE, V>();
  TL_TRY(tl_raise_lds_limit(hgemm_kernel<TYPE, V>, (int)lds, lds_raised));
  hgemm_kernel<TYPE, V><<<dim3((unsigned)blocks), dim3(64 * hgemm_shape(TYPE, V).nw), lds, s>>>(g);
  TL_HIP(hipGetLastError());
  return 0;
}
template <int TYPE>
int hgemm_typed(const QW* w, int n, const HgemmPlan& p, const HAct& act, float* const* out, const float* resid, int T, hipStream_t s) {
  HSegs g = {};
  const int shape = p.shape == 2 && w[0].cols % 256 ? 4 : p.shape;  // (rows that end inside a super-block: shape 4's kernel has the same sums)
  const int blocks = hgemm_grid(g, w, n, hgemm_shape(TYPE, shape), act, out, resid, T, p.S);
  if (shape == 0) return hgemm_go<TYPE, 0>(g, blocks, s);
  if (shape == 1) return hgemm_go<TYPE, 1>(g, blocks, s);
  if (shape == 2) return hgemm_go<TYPE, 2>(g, blocks, s);
  if constexpr (TYPE == TL_Q4_K || TYPE == TL_Q8_K)
    if (shape == 3) return hgemm_go<TYPE, 3>(g, blocks, s);
  if (shape == 5) return hgemm_go<TYPE, 5>(g, blocks, s);
  if (shape == 6) return hgemm_go<TYPE, 6>(g, blocks, s);
  if (shape == 7) return hgemm_go<TYPE, 7>(g, blocks, s);
  if (shape == 8) return hgemm_go<TYPE, 8>(g, blocks, s);
  return hgemm_go<TYPE, 4>(g, blocks, s);
}
std::atomic<long long> g_pair_launches[HGEMM_SHAPES];  // of either shape of Q4_K (tl_debug_half_pair_launches)
template <int V6, int V4>
int hgemm_pair_go(const HPair& g, int blocks, hipStream_t s) {
  static TlDeviceOnce lds_raised;
  constexpr size_t l6 = hgemm_lds_bytes<TL_Q6_K, V6>(), l4 = hgemm_lds_bytes<TL_Q4_K, V4>(), lds = l6 > l4 ? l6 : l4;
  static_assert(hgemm_shape(TL_Q6_K, V6).nw == hgemm_shape(TL_Q4_K, V4).nw && hgemm_shape(TL_Q6_K, V6).wpe == hgemm_shape(TL_Q4_K, V4).wpe, "");
  TL_TRY(tl_raise_lds_limit(hgemm_pair_kernel<V6, V4>, (int)lds, lds_raised));
  hgemm_pair_kernel<V6, V4><<<dim3((unsigned)blocks), dim3(64 * hgemm_shape(TL_Q4_K, V4).nw), lds, s>>>(g);
  TL_HIP(hipGetLastError());
  return 0;
}

}  // namespace

bool tl_hgemm_supported(const QW& w) {
  const bool k256 = w.type == TL_Q4_K || w.type == TL_Q6_K || w.type == TL_Q8_K;
  return (k256 || w.type == TL_Q8_0) && w.cols % (k256 ? 256 : 64) == 0 && w.cols <= HMAX_COLS && w.rows > 0 &&
         (size_t)w.rows * w.cols < ((size_t)1 << 32);  // (32-bit byte offsets)
}
HgemmPlan tl_hgemm_plan(const QW* w, int n, int T) { return hgemm_plan(w, n, T); }
bool tl_hgemm_pair_plan(const QW* w4, int n4, const QW& w6, int T, int most_slices, HgemmPlan* p4, HgemmPlan* p6) {
  if (w4[0].type != TL_Q4_K || w6.type != TL_Q6_K || w4[0].cols != w6.cols || n4 < 1 || n4 > 3) return false;
  for (int i = 0; i < n4; ++i)
    if (!tl_hgemm_supported(w4[i]) || w4[i].type != TL_Q4_K || w4[i].cols != w6.cols) return false;
  if (!tl_hgemm_supported(w6)) return false;
  const int nsb = w6.cols / 256, cus = tl_num_cus(), slices = most_slices < nsb ? most_slices : nsb;
  long rows4 = 0;
  for (int i = 0; i < n4; ++i) rows4 += w4[i].rows;
  const float out4 = (float)T * (float)rows4, out6 = (float)T * (float)w6.rows;
  const unsigned few = T <= 8 ? 1u << 5 | 1u << 6 : T <= 16 ? 1u << 0 | 1u << 7 : 1u << 1 | 1u << 8, many = 1u << 2;
  const unsigned shapes = T <= 32 ? few : T <= 64 ? few | many : many | 1u << 3;
  // (two launches: each at its own best. The prices of long chunks are right to a few per cent)
  float apart = 0.f;
  *p4 = hgemm_plan(w4, n4, T, &apart);
  *p6 = hgemm_plan(&w6, 1, T, &apart);
  float least = (T > 64 ? 0.96f : 1.f) * apart;
  bool joint = false;
  for (int v = 0; v < HGEMM_SHAPES; ++v) {
    if (!(shapes >> v & 1)) continue;
    const int v6 = v == 3 ? 2 : v;
    const HShape q4 = hgemm_shape(TL_Q4_K, v), q6 = hgemm_shape(TL_Q6_K, v6);
    const int ntiles = (T + hgemm_tokens(q4) - 1) / hgemm_tokens(q4), bm4 = q4.tk * q4.mi * q4.nw, bm6 = q6.tk * q6.mi * q6.nw;
    long t4 = 0;
    for (int i = 0; i < n4; ++i) t4 += (long)((w4[i].rows + bm4 - 1) / bm4) * ntiles;
    const long t6 = (long)((w6.rows + bm6 - 1) / bm6) * ntiles;
    for (int a = 1; a <= 8 && a <= slices; ++a) {
      const int per4 = (nsb + a - 1) / a;
      if ((nsb + per4 - 1) / per4 != a) continue;
      for (int b = 1; b <= 8 && b <= slices; ++b) {
        const int per6 = (nsb + b - 1) / b;
        if ((nsb + per6 - 1) / per6 != b) continue;
        const float price = hgemm_pair_price(cus, v6, v, T, t6 * b, per6, b, t4 * a, per4, a, out6, out4, least);
        if (price < least) {
          least = price;
          joint = true;
          *p4 = {v, a};
          *p6 = {v6, b};
        }
      }
    }
  }
  return joint;
}
int tl_launch_hgemm_pair(const QW* w4, int n4, const QW& w6, const void* planes, size_t ps, float* const* out4, float* out6, int T,
                         const HgemmPlan& p4, const HgemmPlan& p6, hipStream_t s) {
  const int nsb = w6.cols / 256;
  for (int i = 0; i < n4; ++i)
    TL_REQUIRE(tl_hgemm_supported(w4[i]) && w4[i].type == TL_Q4_K && w4[i].cols == w6.cols, "half-plane GEMM: matrix %d does not fit", i);
  TL_REQUIRE(n4 >= 1 && n4 <= 3 && T > 0 && tl_hgemm_supported(w6) && w6.type == TL_Q6_K && ps < ((size_t)1 << 31) &&
                 ps >= tl_gemm_padded_tokens(T) * (size_t)w6.cols, "half-plane GEMM: bad argument of a launch of two formats");
  for (const HgemmPlan& p : {p4, p6})
    TL_REQUIRE(p.S >= 1 && (p.S - 1) * ((nsb + p.S - 1) / p.S) < nsb && p.shape >= 0 && p.shape < HGEMM_SHAPES && p6.shape == (p4.shape == 3 ? 2 : p4.shape),
               "half-plane GEMM: shape %d, %d K slices of %d super-blocks", p.shape, p.S, nsb);
  g_pair_launches[p4.shape].fetch_add(1, std::memory_order_relaxed);
  const HAct act = hact(planes, ps, T);
  HPair g = {};
  g.first = hgemm_grid(g.q6, &w6, 1, hgemm_shape(TL_Q6_K, p6.shape), act, &out6, nullptr, T, p6.S);
  const int blocks = g.first + hgemm_grid(g.q4, w4, n4, hgemm_shape(TL_Q4_K, p4.shape), act, out4, nullptr, T, p4.S);
  switch (p4.shape) {
    case 0: return hgemm_pair_go<0, 0>(g, blocks, s);
    case 1: return hgemm_pair_go<1, 1>(g, blocks, s);
    case 2: return hgemm_pair_go<2, 2>(g, blocks, s);
    case 3: return hgemm_pair_go<2, 3>(g, blocks, s);
    case 5: return hgemm_pair_go<5, 5>(g, blocks, s);
    case 6: return hgemm_pair_go<6, 6>(g, blocks, s);
    case 7: return hgemm_pair_go<7, 7>(g, blocks, s);
    case 8: return hgemm_pair_go<8, 8>(g, blocks, s);
    default: break;
  }
  TL_REQUIRE(false, "half-plane GEMM: shape %d has no launch of two formats", p4.shape);
  return 0;
}
extern "C" int tl_debug_half_pair_launches(long long* counts_out) {
  TL_REQUIRE(counts_out, "tl_debug_half_pair_launches: null argument");
  for (int i = 0; i < HGEMM_SHAPES; ++i) counts_out[i] = g_pair_launches[i].load(std::memory_order_relaxed);
  return 0;
}
int tl_launch_hgemm(const QW* w, int n, const void* planes, size_t ps, float* const* out, const float* resid, int T, const HgemmPlan& p,
                    hipStream_t s) {
  for (int i = 0; i < n; ++i)
    TL_REQUIRE(tl_hgemm_supported(w[i]) && w[i].type == w[0].type && w[i].cols == w[0].cols, "half-plane GEMM: matrix %d does not fit", i);
  const int nsb = (w[0].cols + 255) / 256;
  TL_REQUIRE(p.S >= 1 && (p.S - 1) * ((nsb + p.S - 1) / p.S) < nsb && p.shape >= 0 && p.shape < HGEMM_SHAPES &&
                 !(p.shape == 3 && w[0].type != TL_Q4_K && w[0].type != TL_Q8_K),
             "half-plane GEMM: shape %d, %d K slices of %d super-blocks", p.shape, p.S, nsb);
  TL_REQUIRE(n >= 1 && n <= 3 && T > 0 && ps < ((size_t)1 << 31) && ps >= tl_gemm_padded_tokens(T) * (size_t)w[0].cols, "half-plane GEMM: bad argument");
  const HAct act = hact(planes, ps, T);
  switch (w[0].type) {
    case TL_Q4_K: return hgemm_typed<TL_Q4_K>(w, n, p, act, out, resid, T, s);
    case TL_Q6_K: return hgemm_typed<TL_Q6_K>(w, n, p, act, out, resid, T, s);
    case TL_Q8_0: return hgemm_typed<TL_Q8_0>(w, n, p, act, out, resid, T, s);
    default: return hgemm_typed<TL_Q8_K>(w, n, p, act, out, resid, T, s);
  }
}
int tl_launch_hsplit(int mode, const float* x, const float* aux, void* planes, size_t ps, int T, int K, float eps, hipStream_t s,
                     const GemmParts& a, const GemmParts& b, float* xout) {
  TL_REQUIRE(K > 0 && K % 32 == 0 && K <= HMAX_COLS && T > 0 && T <= 65535, "half-plane split: bad shape %d x %d", T, K);
  _Float16* pl = static_cast<_Float16*>(planes);
  const int tpad = (int)tl_gemm_padded_tokens(T);
  if (mode == 1) {
    const int nit = (K + 8 * HNORM_THREADS - 1) / (8 * HNORM_THREADS);
    if (nit <= 1 && T <= tl_num_cus()) hsplit_norm_kernel<1, true><<<T, HNORM_THREADS, 0, s>>>(x, aux, pl, ps, K, eps, a, xout, tpad);
    else if (nit <= 1) hsplit_norm_kernel<1, false><<<T, HNORM_THREADS, 0, s>>>(x, aux, pl, ps, K, eps, a, xout, tpad);
    else if (nit <= 2) hsplit_norm_kernel<2, false><<<T, HNORM_THREADS, 0, s>>>(x, aux, pl, ps, K, eps, a, xout, tpad);
    else hsplit_norm_kernel<8, false><<<T, HNORM_THREADS, 0, s>>>(x, aux, pl, ps, K, eps, a, xout, tpad);
  } else {
    const dim3 grid(T, (K + 2047) / 2048);
    if (mode == 2 && a.S && a.S == b.S && (long)grid.x * grid.y <= 3l * tl_num_cus()) hsplit_kernel<2, true><<<grid, 256, 0, s>>>(x, aux, pl, ps, K, a, b, tpad);
    else if (mode == 2) hsplit_kernel<2, false><<<grid, 256, 0, s>>>(x, aux, pl, ps, K, a, b, tpad);
    else hsplit_kernel<0, false><<<grid, 256, 0, s>>>(x, aux, pl, ps, K, a, b, tpad);
  }
  TL_HIP(hipGetLastError());
  return 0;
}
