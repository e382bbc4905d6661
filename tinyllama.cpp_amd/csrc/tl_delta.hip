// tl_delta.hip — the gated delta rule with a decay per key channel, as a mixer of a layer-list model: a recurrent state
// S [dim][vdim] per head instead of a cache of keys. Per token and head (q / k head = head / (heads / kv_heads)):
//
//     S <- diag(g) S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q        (the read-out sees the token's own write)
//
// with q, k from a short causal convolution over time + silu, made unit vectors per head (q also times dim^-1/2),
// beta = sigmoid(.), g = exp(-exp(A_log[head]) * softplus(a + dt_bias)) per head and key channel. Everything that enters the
// recurrence is FP32, and so is the state.
//
//   delta_pre    one workgroup per token and head: convolution (its last taps - 1 inputs of earlier calls come from a history
//                that is part of the sequence's state), silu, the unit norms, beta and the decay.
//   delta_scan   the recurrence. The columns of S (one per value channel) never mix: o_c = s_c . q, u_c = beta (v_c - s_c . k),
//                s_c <- g * s_c + k u_c. Sixteen lanes share a column (each holds dim / 16 of its key channels in registers),
//                four columns a wave, sixteen a workgroup, heads * vdim / 16 workgroups; the tokens are walked in order with
//                the next token's operands in flight. The three dot products a token needs -- (g s) . k, (g s) . q and k . q,
//                since o = (g s) . q + u (k . q) -- are reduced together over the sixteen lanes with row-local lane swaps, so a
//                token costs one reduction latency, not two. A decode step is the same kernel with one token.
//                With plain_write nothing is removed before the write: linear attention with a decay per key channel. gla_step is
//                its one-token form with everything between the two products around it (decay projection, head norm, gate).
//   gated norm   o / rms(o) * w * sigmoid(gate) per head, in front of the output projection.
//
// A second recurrence lives here beside it, the generalized delta rule: a decay w and a removal rate a per head and key
// channel, the unit key u = k / sqrt(sum k^2 + 1e-6),
//
//     S <- diag(w) S - (a u)(u^T S) + k v^T      (both terms read the old S);   o = S^T r
//
//   gdelta_pre   per token and head: w = exp(-decay_scale sigmoid(dw + w0)), u, a u = sigmoid(a + b_a) u, and the two
//                products that do not touch the state, r . (a u) and r . k.
//   gdelta_scan  the same column-per-16-lanes layout as delta_scan. With x = u . s and y = (w r) . s over the OLD column s,
//                o_c = y - (r . a u) x + (r . k) v_c and s <- w s - (a u) x + k v_c: the two sums over the state are reduced
//                together, so a token again costs one reduction latency.
//   gdelta_chunk_pre, gdelta_chunks   the same recurrence sixteen tokens at a time, as matrix products (below).
#include <math.h>

#include <type_traits>

#include "tl_bf16.h"
#include "tl_lds.h"
#include "tl_stack.h"

namespace {

__device__ __forceinline__ float sigmoidf_(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float softplusf_(float z) { return z > 20.0f ? z : log1pf(expf(z)); }

// grid (T, 2 * kv_heads + heads): a workgroup of 128 threads owns one head of one token -- a q head, a k head (convolution,
// silu, unit norm), or a v head (convolution, silu) together with that head's decay channels and beta. One token (the decode
// step) is thereby spread over as many workgroups as the layer has heads.
__global__ __launch_bounds__(128) void delta_pre_kernel(const DeltaPreArgs a) {
  __shared__ float red[2];
  const int t = blockIdx.x, unit = blockIdx.y, tid = threadIdx.x;
  const int qd = a.kv_heads * a.dim, vd = a.heads * a.vdim, C = 2 * qd + vd, H = a.taps - 1;
  const bool is_v = unit >= 2 * a.kv_heads;
  const int n = is_v ? a.vdim : a.dim;                                            // channels of this head
  const int c0 = is_v ? 2 * qd + (unit - 2 * a.kv_heads) * a.vdim : unit * a.dim;  // its first channel
  float* out = a.qkv + (size_t)t * C + c0;
  float ss = 0.0f;
  float y[4];  // n <= 512: four channels a thread
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int d = tid + 128 * r;
    y[r] = 0.0f;
    if (d >= n) continue;
    const int c = c0 + d;
    const unsigned short* w = a.conv + (size_t)c * a.taps;
    float acc = 0.0f;
    for (int j = 0; j < a.taps; ++j) {
      const int tt = t - H + j;  // token of this tap, relative to the call
      const float in = tt >= 0 ? a.p[(size_t)tt * a.ld + c] : a.hist[(size_t)(H + tt) * C + c];
      acc += tl_bf2f(w[j]) * in;
    }
    y[r] = acc * sigmoidf_(acc);
    ss += y[r] * y[r];
    if (a.T == 1 && H > 0) {  // one token: this thread is the only reader of its channel's history, so it may shift it now
      for (int j = 0; j + 1 < H; ++j) a.hist[(size_t)j * C + c] = a.hist[(size_t)(j + 1) * C + c];
      a.hist[(size_t)(H - 1) * C + c] = a.p[c];
    }
  }
  float inv = 1.0f;
  if (!is_v) {
    ss = tl_wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    inv = 1.0f / sqrtf(red[0] + red[1] + 1e-6f);
    if (unit < a.kv_heads) inv *= 1.0f / sqrtf((float)a.dim);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int d = tid + 128 * r;
    if (d < n) out[d] = y[r] * inv;
  }
  if (!is_v) return;
  const int h = unit - 2 * a.kv_heads, gd = a.heads * a.dim;
  if (tid == 0) a.beta[(size_t)t * a.heads + h] = sigmoidf_(a.p[(size_t)t * a.ld + C + h]);
  const float rate = expf(a.a_log[h]);
  if (a.a_per_head) {  // one decay for the whole head, spread over its key channels
    const float gh = expf(-rate * softplusf_(a.a[(size_t)t * a.a_ld + h] + a.dt_bias[h]));
    for (int d = tid; d < a.dim; d += 128) a.g[(size_t)t * gd + h * a.dim + d] = gh;
    return;
  }
  for (int d = tid; d < a.dim; d += 128) {
    const int c = h * a.dim + d;
    a.g[(size_t)t * gd + c] = expf(-rate * softplusf_(a.a[(size_t)t * gd + c] + a.dt_bias[c]));
  }
}

// after a call of several tokens: the history becomes the last taps - 1 inputs (a call shorter than that keeps the tail of
// the old history in front). A thread owns a channel and walks its rows in ascending order, so no row is read after it was
// overwritten.
__global__ __launch_bounds__(256) void conv_history_kernel(const DeltaPreArgs a) {
  const int qd = a.kv_heads * a.dim, C = 2 * qd + a.heads * a.vdim, H = a.taps - 1;
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= C) return;
  for (int i = 0; i < H; ++i) {
    const int src = a.T - H + i;  // token whose input lands in row i
    a.hist[(size_t)i * C + c] = src >= 0 ? a.p[(size_t)src * a.ld + c] : a.hist[(size_t)(i + a.T) * C + c];
  }
}

// E key channels per lane: dim <= 16 E. grid (vdim / 16 rounded up, heads), 256 threads.
// The operands of 16 (8 for the largest key size) tokens at a time (k, q, g of the head; v of the workgroup's 16 columns; beta) are staged in LDS by
// all threads together, the next stage's global loads in flight while the tokens of the stage in hand are walked: a token
// then waits for an LDS read, not for a round trip to memory.
// PLAIN (plain_write): s <- g s + k u does not wait for any sum over the state, and o = s . q afterwards is the only one
template <int E, bool PLAIN>
__global__ __launch_bounds__(256) void delta_scan_kernel(const DeltaScanArgs a) {
  constexpr int DELTA_TB = E == 16 ? 8 : 16;  // tokens per stage (48 KB of LDS at most)
  constexpr int DP = 16 * E;                 // padded key size
  constexpr int NL = (DELTA_TB * DP) / 256;  // k / q / g elements a thread stages = E
  __shared__ __attribute__((aligned(16))) float sk_[2][DELTA_TB][DP], sq_[2][DELTA_TB][DP], sg_[2][DELTA_TB][DP];
  __shared__ float sv_[2][DELTA_TB][16], sb_[2][DELTA_TB];
  const int tid = threadIdx.x, sub = tid & 15, cl = tid >> 4;
  const int col = blockIdx.x * 16 + cl, h = blockIdx.y;
  const int kvh = h / (a.heads / a.kv_heads);
  const bool live = col < a.vdim;           // lanes of a column beyond vdim compute on zeros and store nothing
  const int d0 = sub * E;
  const float oscale = a.q_scale != 0.0f ? a.q_scale : 1.0f;
  float* sp = a.state + ((size_t)h * a.vdim + (live ? col : 0)) * a.dim;
  float s[E];
#pragma unroll
  for (int e = 0; e < E; ++e) s[e] = (live && d0 + e < a.dim) ? sp[d0 + e] : 0.0f;
  const float* qp = a.q + (size_t)kvh * a.dim;
  const float* kp = a.k + (size_t)kvh * a.dim;
  const float* gp = a.g + (size_t)h * a.dim;
  const int gd = a.heads * a.dim;
  // staging registers: element i of this thread is (token i * 256 + tid) / DP, channel (i * 256 + tid) % DP of the stage
  float rk[NL], rq[NL], rg[NL], rv, rb;
  auto fetch = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int idx = i * 256 + tid, tt = idx / DP, d = idx % DP;
      const bool in = t0 + tt < a.T && d < a.dim;
      rk[i] = in ? kp[(size_t)(t0 + tt) * a.ldq + d] : 0.0f;
      rq[i] = in ? qp[(size_t)(t0 + tt) * a.ldq + d] : 0.0f;
      rg[i] = in ? gp[(size_t)(t0 + tt) * gd + d] : 0.0f;
    }
    const int tt = tid >> 4, c = blockIdx.x * 16 + (tid & 15);
    rv = (tt < DELTA_TB && t0 + tt < a.T && c < a.vdim) ? a.v[(size_t)(t0 + tt) * a.ldv + (size_t)h * a.vdim + c] : 0.0f;
    rb = (tid < DELTA_TB && t0 + tid < a.T) ? (a.beta ? a.beta[(size_t)(t0 + tid) * a.heads + h] : 1.0f) : 0.0f;
  };
  auto stash = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int idx = i * 256 + tid, tt = idx / DP, d = idx % DP;
      sk_[b][tt][d] = rk[i];
      sq_[b][tt][d] = rq[i];
      sg_[b][tt][d] = rg[i];
    }
    if ((tid >> 4) < DELTA_TB) sv_[b][tid >> 4][tid & 15] = rv;
    if (tid < DELTA_TB) sb_[b][tid] = rb;
  };
  fetch(0);
  stash(0);
  __syncthreads();
  int b = 0;
  for (int t0 = 0; t0 < a.T; t0 += DELTA_TB, b ^= 1) {
    const bool more = t0 + DELTA_TB < a.T;
    if (more) fetch(t0 + DELTA_TB);  // in flight under this stage's tokens
    const int nt = a.T - t0 < DELTA_TB ? a.T - t0 : DELTA_TB;
    for (int tt = 0; tt < nt; ++tt) {
      float kc[E], qc[E], gc[E];
#pragma unroll
      for (int e = 0; e < E; ++e) {
        kc[e] = sk_[b][tt][d0 + e];
        qc[e] = sq_[b][tt][d0 + e];
        gc[e] = sg_[b][tt][d0 + e];
      }
      const float vc = sv_[b][tt][cl], bc = sb_[b][tt];
      float sk = 0.0f, sq = 0.0f, kq = 0.0f;
      if (PLAIN) {
        const float u = bc * vc;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          s[e] = s[e] * gc[e] + kc[e] * u;
          sq += s[e] * qc[e];
        }
        sq = tl_row16_sum(sq);
        if (live && sub == 0) a.o[(size_t)(t0 + tt) * a.heads * a.vdim + (size_t)h * a.vdim + col] = sq * oscale;
        continue;
      }
#pragma unroll
      for (int e = 0; e < E; ++e) {
        s[e] *= gc[e];
        sk += s[e] * kc[e];
        sq += s[e] * qc[e];
        kq += kc[e] * qc[e];
      }
      sk = tl_row16_sum(sk);
      sq = tl_row16_sum(sq);
      kq = tl_row16_sum(kq);
      const float u = bc * (vc - sk);
#pragma unroll
      for (int e = 0; e < E; ++e) s[e] += kc[e] * u;
      if (live && sub == 0) a.o[(size_t)(t0 + tt) * a.heads * a.vdim + (size_t)h * a.vdim + col] = (sq + u * kq) * oscale;
    }
    if (more) stash(b ^ 1);  // the other buffer: its last readers passed the barrier at the end of the stage before
    __syncthreads();
  }
  if (live) {
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (d0 + e < a.dim) sp[d0 + e] = s[e];
  }
}

// grid (heads), 1024 threads: 64 columns of S at a time, sixteen lanes a column (E key channels each, dim <= 16 E). The state is
// asked for first, the decay of the head's key channels (eight lanes a channel) is formed under its round trip.
template <int E>
__global__ __launch_bounds__(1024) void gla_step_kernel(const GlaStepArgs a, int vec) {
  extern __shared__ __attribute__((aligned(16))) float sl[];  // k | q | alpha (16 E each) | v | o (vdim each) | a1
  __shared__ float red[16];
  constexpr int DP = 16 * E, P = E >= 16 ? 1 : 16 / E;  // column passes in flight together
  float *sk = sl, *sq = sl + DP, *sa = sl + 2 * DP, *sv = sl + 3 * DP, *so = sv + a.vdim, *s1 = so + a.vdim;
  const int tid = threadIdx.x, sub = tid & 15, cl = tid >> 4, h = blockIdx.x, d0 = sub * E;
  const int hd = a.heads * a.dim, vd = a.heads * a.vdim;
  float* S = a.state + (size_t)h * a.vdim * a.dim;
  float s[P][E];
  auto load = [&](int col, float* to) __attribute__((always_inline)) {
    const float* p = S + (size_t)(col < a.vdim ? col : 0) * a.dim + d0;
    if (vec && E >= 4) {
#pragma unroll
      for (int e = 0; e + 4 <= E; e += 4) {
        const float4 f = *reinterpret_cast<const float4*>(p + e);
        to[e] = f.x, to[e + (E > 1 ? 1 : 0)] = f.y, to[e + (E > 2 ? 2 : 0)] = f.z, to[e + (E > 3 ? 3 : 0)] = f.w;
      }
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) to[e] = d0 + e < a.dim ? p[e] : 0.0f;
    }
  };
#pragma unroll
  for (int i = 0; i < P; ++i) load(cl + 64 * i, s[i]);
  for (int i = tid; i < DP; i += 1024) {
    sk[i] = i < a.dim ? a.p[hd + h * a.dim + i] : 0.0f;
    sq[i] = i < a.dim ? a.p[h * a.dim + i] : 0.0f;
  }
  for (int i = tid; i < a.vdim; i += 1024) sv[i] = a.p[2 * hd + h * a.vdim + i];
  for (int i = tid; i < a.rank; i += 1024) s1[i] = a.p[2 * hd + 2 * vd + i];
  __syncthreads();
  for (int c0 = 0; c0 < DP; c0 += 128) {  // (every lane stays in the loop: the sum below crosses lanes)
    const int c = c0 + (tid >> 3);
    float z = 0.0f;
    if (c < a.dim) {
      const unsigned short* w = a.a2 + ((size_t)h * a.dim + c) * a.rank;
      for (int r = tid & 7; r < a.rank; r += 8) z += tl_bf2f(w[r]) * s1[r];
    }
    z += __shfl_xor(z, 1);
    z += __shfl_xor(z, 2);
    z += __shfl_xor(z, 4);
    if ((tid & 7) == 0 && c < DP) sa[c] = c < a.dim ? tl_act_apply(TL_ACT_SIGMOID_POWER, z + a.a2_b[h * a.dim + c], a.power, 0.0f) : 0.0f;
  }
  __syncthreads();
  float kc[E], qc[E], ac[E];
#pragma unroll
  for (int e = 0; e < E; ++e) kc[e] = sk[d0 + e], qc[e] = sq[d0 + e], ac[e] = sa[d0 + e];
  for (int b = 0; b < a.vdim; b += 64 * P) {
    if (b > 0) {
#pragma unroll
      for (int i = 0; i < P; ++i) load(b + cl + 64 * i, s[i]);
    }
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int col = b + cl + 64 * i;
      const bool live = col < a.vdim;
      const float v = live ? sv[col] : 0.0f;
      float o = 0.0f;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        s[i][e] = ac[e] * s[i][e] + kc[e] * v;
        o += s[i][e] * qc[e];
      }
      o = tl_row16_sum(o);
      if (!live) continue;
      if (sub == 0) so[col] = o * a.q_scale;
      float* p = S + (size_t)col * a.dim + d0;
      if (vec && E >= 4) {
#pragma unroll
        for (int e = 0; e + 4 <= E; e += 4)
          *reinterpret_cast<float4*>(p + e) = make_float4(s[i][e], s[i][e + (E > 1 ? 1 : 0)], s[i][e + (E > 2 ? 2 : 0)], s[i][e + (E > 3 ? 3 : 0)]);
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e)
          if (d0 + e < a.dim) p[e] = s[i][e];
      }
    }
  }
  __syncthreads();
  float ss = 0.0f;
  for (int c = tid; c < a.vdim; c += 1024) ss += so[c] * so[c];
  ss = tl_wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  ss = 0.0f;
#pragma unroll
  for (int w = 0; w < 16; ++w) ss += red[w];
  const float inv = 1.0f / sqrtf(ss / (float)a.vdim + a.eps);
  const float* gp = a.p + 2 * hd + vd + h * a.vdim;
  for (int c = tid; c < a.vdim; c += 1024) a.o[h * a.vdim + c] = so[c] * inv * a.norm[c] * (gp[c] * sigmoidf_(gp[c]));
}

// a wave per (token, head); gate rows gate_ld floats apart; weights of its own for every head or one vector for all
__global__ __launch_bounds__(256) void head_norm_kernel(const HeadNormArgs a) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= a.T * a.heads) return;
  const int t = i / a.heads, h = i - t * a.heads, vdim = a.vdim;
  float* x = a.o + (size_t)i * vdim;
  const float* sub = a.sub ? a.sub + (size_t)i * vdim : nullptr;
  const float* g = a.gate ? a.gate + (size_t)t * a.gate_ld + (size_t)h * vdim : nullptr;
  const float* wh = a.w ? a.w + (a.w_per_head ? (size_t)h * vdim : 0) : nullptr;
  const float scale = a.out_scale;
  float ss = 0.0f;
  for (int d = lane; d < vdim; d += 64) {
    const float v = sub ? x[d] - a.sub_coef * sub[d] : x[d];
    ss += v * v;
  }
  ss = tl_wave_sum(ss);
  const float inv = 1.0f / sqrtf(ss / (float)vdim + a.eps);
  for (int d = lane; d < vdim; d += 64) {
    float v = (sub ? x[d] - a.sub_coef * sub[d] : x[d]) * inv * scale;
    if (wh) v *= wh[d];
    if (g) v *= a.gate_act == 1 ? g[d] * sigmoidf_(g[d]) : sigmoidf_(g[d]);
    x[d] = v;
  }
}

// grid (column blocks of 256 over heads * dim, T)
__global__ __launch_bounds__(256) void linear_pre_kernel(const LinearPreArgs a) {
  const int t = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x, hd = a.heads * a.dim;
  if (c >= hd) return;
  const float* row = a.p + (size_t)t * a.ld;
  const float q = row[c], z = row[hd + c] + a.f_bias[c], low = a.lower[c];
  a.qk[(size_t)t * 2 * hd + c] = q * sigmoidf_(q);
  a.qk[(size_t)t * 2 * hd + hd + c] = (1.0f - low) * sigmoidf_(-z);  // 1 - f
  a.g[(size_t)t * hd + c] = low + (1.0f - low) * sigmoidf_(z);
}

// grid (T, heads): a workgroup of 128 threads owns one head of one token (dim <= 512: four channels a thread)
__global__ __launch_bounds__(128) void gdelta_pre_kernel(const GDeltaPreArgs a) {
  __shared__ float red[3][2];
  const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int hd = a.heads * a.dim;
  const float* row = a.p + (size_t)t * a.ld;
  const float* rp = row + (size_t)h * a.dim;
  const float* kp = row + hd + (size_t)h * a.dim;
  const float* ap = row + 4 * (size_t)hd + (size_t)h * a.dim;
  const size_t o0 = (size_t)t * hd + (size_t)h * a.dim;
  float kv[4], rv[4], av[4];
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int d = tid + 128 * j;
    kv[j] = rv[j] = av[j] = 0.0f;
    if (d >= a.dim) continue;
    kv[j] = kp[d];
    rv[j] = rp[d];
    av[j] = sigmoidf_(ap[d] + a.a_bias[h * a.dim + d]);
    ss += kv[j] * kv[j];
    a.w[o0 + d] = expf(-a.decay_scale * sigmoidf_(a.dw[o0 + d] + a.w0[h * a.dim + d]));
  }
  ss = tl_wave_sum(ss);
  if ((tid & 63) == 0) red[0][tid >> 6] = ss;
  __syncthreads();
  const float inv = 1.0f / sqrtf(red[0][0] + red[0][1] + 1e-6f);
  float s_rau = 0.0f, s_rk = 0.0f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int d = tid + 128 * j;
    if (d >= a.dim) continue;
    const float u = kv[j] * inv, au = av[j] * u;
    a.u[o0 + d] = u;
    a.au[o0 + d] = au;
    s_rau += rv[j] * au;
    s_rk += rv[j] * kv[j];
  }
  s_rau = tl_wave_sum(s_rau);
  s_rk = tl_wave_sum(s_rk);
  if ((tid & 63) == 0) {
    red[1][tid >> 6] = s_rau;
    red[2][tid >> 6] = s_rk;
  }
  __syncthreads();
  if (tid == 0) {
    a.rau[(size_t)t * a.heads + h] = red[1][0] + red[1][1];
    a.rk[(size_t)t * a.heads + h] = red[2][0] + red[2][1];
  }
}

// E key channels per lane: dim <= 16 E. grid (vdim / 16 rounded up, heads), 256 threads; staging as in delta_scan_kernel
// (five key-channel vectors per token here: r, k, w, u, a u).
template <int E>
__global__ __launch_bounds__(256) void gdelta_scan_kernel(const GDeltaScanArgs a) {
  constexpr int TB = E == 16 ? 4 : E == 8 ? 8 : 16;  // tokens per stage (40 KB of LDS at most)
  constexpr int DP = 16 * E;                           // padded key size
  constexpr int NL = (TB * DP) / 256;                  // elements of each vector a thread stages
  __shared__ __attribute__((aligned(16))) float sr_[2][TB][DP], sk_[2][TB][DP], sw_[2][TB][DP], su_[2][TB][DP], sa_[2][TB][DP];
  __shared__ float sv_[2][TB][16], sc_[2][TB][2];
  const int tid = threadIdx.x, sub = tid & 15, cl = tid >> 4;
  const int col = blockIdx.x * 16 + cl, h = blockIdx.y;
  const bool live = col < a.vdim;  // lanes of a column beyond vdim compute on zeros and store nothing
  const int d0 = sub * E;
  float* sp = a.state + ((size_t)h * a.vdim + (live ? col : 0)) * a.dim;
  float s[E];
#pragma unroll
  for (int e = 0; e < E; ++e) s[e] = (live && d0 + e < a.dim) ? sp[d0 + e] : 0.0f;
  const int hd = a.heads * a.dim;
  const float* rp = a.r + (size_t)h * a.dim;
  const float* kp = a.k + (size_t)h * a.dim;
  const size_t c0 = (size_t)h * a.dim;
  float rr[NL], rk[NL], rw[NL], ru[NL], ra[NL], rv, rc;
  auto fetch = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int idx = i * 256 + tid, tt = idx / DP, d = idx % DP;
      const bool in = t0 + tt < a.T && d < a.dim;
      const size_t g = (size_t)(t0 + tt) * hd + c0 + d;
      rr[i] = in ? rp[(size_t)(t0 + tt) * a.ld + d] : 0.0f;
      rk[i] = in ? kp[(size_t)(t0 + tt) * a.ld + d] : 0.0f;
      rw[i] = in ? a.w[g] : 0.0f;
      ru[i] = in ? a.u[g] : 0.0f;
      ra[i] = in ? a.au[g] : 0.0f;
    }
    const int tt = tid >> 4, c = blockIdx.x * 16 + (tid & 15);
    rv = (tt < TB && t0 + tt < a.T && c < a.vdim) ? a.v[(size_t)(t0 + tt) * a.ld + (size_t)h * a.vdim + c] : 0.0f;
    const int t2 = tid >> 1;  // threads 0 .. 2 TB - 1: (r . a u, r . k) of the stage's tokens
    rc = (t2 < TB && t0 + t2 < a.T) ? ((tid & 1) ? a.rk : a.rau)[(size_t)(t0 + t2) * a.heads + h] : 0.0f;
  };
  auto stash = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int idx = i * 256 + tid, tt = idx / DP, d = idx % DP;
      sr_[b][tt][d] = rr[i];
      sk_[b][tt][d] = rk[i];
      sw_[b][tt][d] = rw[i];
      su_[b][tt][d] = ru[i];
      sa_[b][tt][d] = ra[i];
    }
    if ((tid >> 4) < TB) sv_[b][tid >> 4][tid & 15] = rv;
    if ((tid >> 1) < TB) sc_[b][tid >> 1][tid & 1] = rc;
  };
  fetch(0);
  stash(0);
  __syncthreads();
  int b = 0;
  for (int t0 = 0; t0 < a.T; t0 += TB, b ^= 1) {
    const bool more = t0 + TB < a.T;
    if (more) fetch(t0 + TB);  // in flight under this stage's tokens
    const int nt = a.T - t0 < TB ? a.T - t0 : TB;
    for (int tt = 0; tt < nt; ++tt) {
      float rc_[E], kc[E], wc[E], uc[E], ac[E];
#pragma unroll
      for (int e = 0; e < E; ++e) {
        rc_[e] = sr_[b][tt][d0 + e];
        kc[e] = sk_[b][tt][d0 + e];
        wc[e] = sw_[b][tt][d0 + e];
        uc[e] = su_[b][tt][d0 + e];
        ac[e] = sa_[b][tt][d0 + e];
      }
      const float vc = sv_[b][tt][cl], rau = sc_[b][tt][0], rkk = sc_[b][tt][1];
      float x = 0.0f, y = 0.0f;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        x += uc[e] * s[e];
        s[e] *= wc[e];
        y += rc_[e] * s[e];
      }
      x = tl_row16_sum(x);
      y = tl_row16_sum(y);
#pragma unroll
      for (int e = 0; e < E; ++e) s[e] += kc[e] * vc - ac[e] * x;
      if (live && sub == 0) a.o[(size_t)(t0 + tt) * a.heads * a.vdim + (size_t)h * a.vdim + col] = y - rau * x + rkk * vc;
    }
    if (more) stash(b ^ 1);  // the other buffer: its last readers passed the barrier at the end of the stage before
    __syncthreads();
  }
  if (live) {
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (d0 + e < a.dim) sp[d0 + e] = s[e];
  }
}

// The same for key sizes of exactly 16 E and rows at 16 bytes. One wave a SIMD walks the tokens, so what a token costs is the number of
// its instructions: here five 16-byte LDS reads at constant offsets (a stage is unrolled), 5 E products and sums, and two row sums. (r w)
// is formed once in staging; the lane whose number is the token's keeps x and y, and a stage's outputs are finished and stored together.
// The new column is one rounding of w s + (k v - a u x). 32 heads of 64 times 1998 tokens 241 us. Models take it for few tokens and for
// decays that gdelta_chunks does not take.
template <int E>
__global__ __launch_bounds__(256) void gdelta_scan_wide_kernel(const GDeltaScanArgs a) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr int DP = 16 * E, TB = 1024 / DP;  // tokens per stage: a 16-byte piece of each vector per thread
  static_assert(TB <= 16, "a token of a stage per lane of a column");
  constexpr int RW = 0, K = 1, W = 2, U = 3, A = 4;
  __shared__ __attribute__((aligned(16))) float st[2][5][TB][DP];
  __shared__ float sv[2][TB][16], sc[2][TB][2];
  const int tid = threadIdx.x, sub = tid & 15, cl = tid >> 4, h = blockIdx.y;
  const int col = blockIdx.x * 16 + cl, d0 = sub * E;
  const bool live = col < a.vdim;  // lanes of a column beyond vdim compute on the first one's numbers and store nothing
  float* sp = a.state + ((size_t)h * a.vdim + (live ? col : 0)) * DP + d0;
  f32x4 s[E / 4];
#pragma unroll
  for (int e = 0; e < E / 4; ++e) s[e] = *reinterpret_cast<const f32x4*>(sp + 4 * e);
  const int hd = a.heads * DP, ft = tid / (DP / 4), fd = tid % (DP / 4) * 4;
  const float* rp = a.r + (size_t)h * DP + fd;
  const float* kp = a.k + (size_t)h * DP + fd;
  const size_t c0 = (size_t)h * DP + fd;
  const int vt = tid >> 4, vcol = blockIdx.x * 16 + sub;
  const float* vp = a.v + (size_t)h * a.vdim + (vcol < a.vdim ? vcol : 0);
  const float* cp = (tid & 1 ? a.rk : a.rau) + h;
  f32x4 g[5];
  float gv, gc;
  auto fetch = [&](int t0) __attribute__((always_inline)) {  // (tokens beyond the last: the last one's, never walked)
    const size_t t = t0 + ft < a.T ? t0 + ft : a.T - 1;
    g[RW] = *reinterpret_cast<const f32x4*>(rp + t * a.ld);
    g[K] = *reinterpret_cast<const f32x4*>(kp + t * a.ld);
    g[W] = *reinterpret_cast<const f32x4*>(a.w + t * hd + c0);
    g[U] = *reinterpret_cast<const f32x4*>(a.u + t * hd + c0);
    g[A] = *reinterpret_cast<const f32x4*>(a.au + t * hd + c0);
    gv = vp[(size_t)(t0 + vt < a.T ? t0 + vt : a.T - 1) * a.ld];
    gc = cp[(size_t)(t0 + (tid >> 1) < a.T ? t0 + (tid >> 1) : a.T - 1) * a.heads];
  };
  auto stash = [&](int b) __attribute__((always_inline)) {
    g[RW] *= g[W];
#pragma unroll
    for (int i = 0; i < 5; ++i) *reinterpret_cast<f32x4*>(&st[b][i][ft][fd]) = g[i];
    if (vt < TB) sv[b][vt][sub] = gv;
    if (tid < 2 * TB) sc[b][tid >> 1][tid & 1] = gc;
  };
  float xk = 0.0f, yk = 0.0f;
  auto token = [&](int b, int tt) __attribute__((always_inline)) {
    f32x4 q[5][E / 4];
#pragma unroll
    for (int i = 0; i < 5; ++i)
#pragma unroll
      for (int e = 0; e < E / 4; ++e) q[i][e] = *reinterpret_cast<const f32x4*>(&st[b][i][tt][d0 + 4 * e]);
    const float vc = sv[b][tt][cl];
    float x = 0.0f, y = 0.0f;
#pragma unroll
    for (int e = 0; e < E / 4; ++e) {
      x += fmaf(q[U][e][0], s[e][0], q[U][e][1] * s[e][1]) + fmaf(q[U][e][2], s[e][2], q[U][e][3] * s[e][3]);
      y += fmaf(q[RW][e][0], s[e][0], q[RW][e][1] * s[e][1]) + fmaf(q[RW][e][2], s[e][2], q[RW][e][3] * s[e][3]);
    }
    x = tl_row16_sum(x);
    y = tl_row16_sum(y);
#pragma unroll
    for (int e = 0; e < E / 4; ++e)
#pragma unroll
      for (int j = 0; j < 4; ++j) s[e][j] = fmaf(q[W][e][j], s[e][j], fmaf(-q[A][e][j], x, q[K][e][j] * vc));
    xk = sub == tt ? x : xk;
    yk = sub == tt ? y : yk;
  };
  float* op = a.o + (size_t)h * a.vdim + col;
  auto finish = [&](int b, int t0, int nt) __attribute__((always_inline)) {
    if (live && sub < nt) op[(size_t)(t0 + sub) * a.heads * a.vdim] = yk - sc[b][sub][0] * xk + sc[b][sub][1] * sv[b][sub][cl];
  };
  fetch(0);
  stash(0);
  __syncthreads();
  int b = 0, t0 = 0;
  for (; t0 + TB <= a.T; t0 += TB, b ^= 1) {
    const bool more = t0 + TB < a.T;
    if (more) fetch(t0 + TB);  // in flight under this stage's tokens
#pragma unroll
    for (int tt = 0; tt < TB; ++tt) token(b, tt);
    finish(b, t0, TB);
    if (more) stash(b ^ 1);  // the other buffer: its last readers passed the barrier at the end of the stage before
    __syncthreads();
  }
  if (t0 < a.T) {
    for (int tt = 0; tt < a.T - t0; ++tt) token(b, tt);
    finish(b, t0, a.T - t0);
  }
  if (live) {
#pragma unroll
    for (int e = 0; e < E / 4; ++e) *reinterpret_cast<f32x4*>(sp + 4 * e) = s[e];
  }
}

// ---- the generalized delta rule in chunks of 16 tokens ---------------------------------------------------------------------------------
// With W_t the product of a chunk's decays up to token t, the column after token t is W_t (s0 + sum_{j <= t} (k_j v_j - (a u)_j x_j) / W_j),
// so that the chunk's sixteen x = u_t . s_{t-1} solve (I + D) x = U s0 + B v and everything else is a product:
//     U_t = u_t W_{t-1},  R_t = r_t W_t,  K_j = k_j / W_j,  A_j = (a u)_j / W_j
//     B = U K^T, D = U A^T (j < t);  E = R K^T, F = R A^T (j <= t);  T = (I + D)^-1
//     z = U s0 + B v,  x = T z,  y = R s0 + E v - F x,  s <- W_16 (s0 + K^T v - A^T x)
// All but s0 and v is the same for a head's columns and does not wait for the state: gdelta_chunk_pre forms it for all chunks at once,
// gdelta_chunks walks the chunks. W shrinks by at most e a token here (tl_gdelta_chunks_take), so that 1 / W stays below e^16.
// A chunk with a number that is not finite or beyond 1e12 would spread it to the tokens before: it is marked and walked token by token.
constexpr int GC = 16;  // tokens of a chunk
constexpr float GC_LARGE = 1e12f;
// floats of a chunk of a head: U, R [D / 16][16 tokens][16 channels], (k times the decays behind it)^T, -(a u times those)^T [D][16], B, E, -F,
// T [16][16], W_16 [D], decays [16][D]. Where the chunk is marked, the last number of B's first row, 0 otherwise, is 1, the first four
// parts are u, r, k, a u [16][D] and the decays are there.
__host__ __device__ constexpr int gc_floats(int D) { return 5 * GC * D + 4 * GC * GC + D; }
__host__ __device__ constexpr int gc_mats(int D) { return 4 * GC * D; }
__host__ __device__ constexpr int gc_w(int D) { return gc_mats(D) + 4 * GC * GC; }
struct GDeltaChunkArgs {
  const float* p;
  int ld;
  const float *dw, *w0, *a_bias;
  float decay_scale;
  float *ws, *state, *o;
  int T, heads, nchunks;
};

typedef float gc4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ gc4 gc_mfma(float a, float b, gc4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// a b of 16 x 16 numbers: lane (m, g) holds a[m][4 g ..] and b[4 g ..][m] (the layout that products leave). Two sums of eight: with one sum
// over all of a chain's products the read-outs were 1.8 times as far from 64 bits as the token-by-token kernel's
__device__ __forceinline__ gc4 gc_mul16(gc4 a, gc4 b) {
  return gc_mfma(a[1], b[1], gc_mfma(a[0], b[0], gc4{})) + gc_mfma(a[3], b[3], gc_mfma(a[2], b[2], gc4{}));
}

// grid (chunks, heads): 16 lanes a token, E channels a lane
template <int E>
__global__ __launch_bounds__(256, 2) void gdelta_chunk_pre_kernel(const GDeltaChunkArgs a) {
  constexpr int D = 16 * E, LD = D + 4;
  __shared__ __attribute__((aligned(16))) float su[GC][LD], sr[GC][LD], sk[GC][LD], sa[GC][LD], sw[GC][LD];
  __shared__ __attribute__((aligned(16))) float mat[4][GC][GC + 4];  // B, D, E, F
  __shared__ float diag[2][GC];                                      // r . k, r . (a u)
  __shared__ int marked;
  const int tid = threadIdx.x, tt = tid >> 4, sub = tid & 15, h = blockIdx.y, t = blockIdx.x * GC + tt, hd = a.heads * D, d0 = sub * E;
  const bool in = t < a.T;
  const float* row = a.p + (size_t)(in ? t : a.T - 1) * a.ld + (size_t)h * D + d0;
  const float* dwp = a.dw + (size_t)(in ? t : a.T - 1) * hd + (size_t)h * D + d0;
  if (tid == 0) marked = 0;
  float r[E], k[E], u[E], au[E], w[E];
  float ss = 0.0f, top = 0.0f;
  bool bad = false;
#pragma unroll
  for (int e = 0; e < E; e += 4) {
    const gc4 rv = *reinterpret_cast<const gc4*>(row + e), kv = *reinterpret_cast<const gc4*>(row + hd + e);
    const gc4 vv = *reinterpret_cast<const gc4*>(row + 2 * (size_t)hd + e), av = *reinterpret_cast<const gc4*>(row + 4 * (size_t)hd + e);
    const gc4 dv = *reinterpret_cast<const gc4*>(dwp + e);
    const gc4 ab = *reinterpret_cast<const gc4*>(a.a_bias + h * D + d0 + e), wb = *reinterpret_cast<const gc4*>(a.w0 + h * D + d0 + e);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      r[e + c] = in ? rv[c] : 0.0f;
      k[e + c] = in ? kv[c] : 0.0f;
      au[e + c] = sigmoidf_(av[c] + ab[c]);
      w[e + c] = in ? expf(-a.decay_scale * sigmoidf_(dv[c] + wb[c])) : 1.0f;
      ss += k[e + c] * k[e + c];
      top = fmaxf(top, fmaxf(fmaxf(fabsf(rv[c]), fabsf(kv[c])), fabsf(vv[c])));  // (fmaxf drops a NaN: the sum below does not)
      bad |= !(rv[c] + kv[c] + vv[c] + au[e + c] + w[e + c] < INFINITY);
    }
  }
  bad |= !(top <= GC_LARGE);
  ss = tl_row16_sum(ss);
  const float inv = 1.0f / sqrtf(ss + 1e-6f);
  float rk = 0.0f, rau = 0.0f;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    u[e] = k[e] * inv;
    au[e] *= u[e];
    rk += r[e] * k[e];
    rau += r[e] * au[e];
  }
  rk = tl_row16_sum(rk);
  rau = tl_row16_sum(rau);
  if (sub == 0) {
    diag[0][tt] = rk;
    diag[1][tt] = rau;
  }
  __syncthreads();
  if (in && bad) marked = 1;
#pragma unroll
  for (int e = 0; e < E; e += 4) *reinterpret_cast<gc4*>(&sw[tt][d0 + e]) = gc4{w[e], w[e + 1], w[e + 2], w[e + 3]};
  __syncthreads();
  float* ws = a.ws + ((size_t)blockIdx.x * a.heads + h) * gc_floats(D);
  if (marked) {
#pragma unroll
    for (int e = 0; e < E; e += 4) {
      float* o = ws + tt * D + d0 + e;
      *reinterpret_cast<gc4*>(o) = gc4{u[e], u[e + 1], u[e + 2], u[e + 3]};
      *reinterpret_cast<gc4*>(o + GC * D) = gc4{r[e], r[e + 1], r[e + 2], r[e + 3]};
      *reinterpret_cast<gc4*>(o + 2 * GC * D) = gc4{k[e], k[e + 1], k[e + 2], k[e + 3]};
      *reinterpret_cast<gc4*>(o + 3 * GC * D) = gc4{au[e], au[e + 1], au[e + 2], au[e + 3]};
      *reinterpret_cast<gc4*>(o + gc_w(D) + D) = gc4{w[e], w[e + 1], w[e + 2], w[e + 3]};
    }
    if (tid == 0) ws[gc_mats(D) + GC - 1] = 1.0f;
    return;
  }
  // the channels' k and a u times the decays behind their token, from the last one back: as often rounded as in the recurrence
#pragma unroll
  for (int e = 0; e < E; e += 4) {
    *reinterpret_cast<gc4*>(&sk[tt][d0 + e]) = gc4{k[e], k[e + 1], k[e + 2], k[e + 3]};
    *reinterpret_cast<gc4*>(&sa[tt][d0 + e]) = gc4{au[e], au[e + 1], au[e + 2], au[e + 3]};
  }
  __syncthreads();
  if (tid < D) {
    float c[GC], kc[GC], ac[GC], back = 1.0f;
#pragma unroll
    for (int i = GC - 1; i >= 0; --i) {
      c[i] = sw[i][tid];
      kc[i] = sk[i][tid] * back;
      ac[i] = -(sa[i][tid] * back);
      back *= c[i];
    }
#pragma unroll
    for (int i = 0; i < GC; i += 4) {
      *reinterpret_cast<gc4*>(ws + 2 * GC * D + tid * GC + i) = gc4{kc[i], kc[i + 1], kc[i + 2], kc[i + 3]};
      *reinterpret_cast<gc4*>(ws + 3 * GC * D + tid * GC + i) = gc4{ac[i], ac[i + 1], ac[i + 2], ac[i + 3]};
    }
    ws[gc_w(D) + tid] = back;
#pragma unroll
    for (int i = 1; i < GC; ++i) c[i] *= c[i - 1];
#pragma unroll
    for (int i = 0; i < GC; ++i) sw[i][tid] = c[i];
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; e += 4) {
    const gc4 now = *reinterpret_cast<const gc4*>(&sw[tt][d0 + e]);
    gc4 before = gc4{1.0f, 1.0f, 1.0f, 1.0f};
    if (tt) before = *reinterpret_cast<const gc4*>(&sw[tt - 1][d0 + e]);
    gc4 U, R, K, A;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      U[c] = u[e + c] * before[c];
      R[c] = r[e + c] * now[c];
      K[c] = k[e + c] / now[c];
      A[c] = au[e + c] / now[c];
    }
    *reinterpret_cast<gc4*>(&su[tt][d0 + e]) = U;
    *reinterpret_cast<gc4*>(&sr[tt][d0 + e]) = R;
    *reinterpret_cast<gc4*>(&sk[tt][d0 + e]) = K;
    *reinterpret_cast<gc4*>(&sa[tt][d0 + e]) = A;
    const int at = (d0 + e) / 16 * 256 + tt * 16 + (d0 + e) % 16;
    *reinterpret_cast<gc4*>(ws + at) = U;
    *reinterpret_cast<gc4*>(ws + GC * D + at) = R;
  }
  __syncthreads();
  // a wave forms one of B, D, E, F
  const int wave = tid >> 6, lane = tid & 63, m = lane & 15, g = lane >> 4;
  {
    const float* left = wave < 2 ? &su[m][0] : &sr[m][0];
    const float* right = wave & 1 ? &sa[m][0] : &sk[m][0];
    gc4 c = {};
#pragma unroll
    for (int i = 0; i < D / 16; ++i) c += gc_mul16(*reinterpret_cast<const gc4*>(left + 16 * i + 4 * g), *reinterpret_cast<const gc4*>(right + 16 * i + 4 * g));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t1 = 4 * g + e;
      mat[wave][t1][m] = m < t1 ? c[e] : m == t1 && wave >= 2 ? diag[wave - 2][m] : 0.0f;
    }
  }
  __syncthreads();
  float* mw = ws + gc_mats(D);  // B, E, -F, T
  if (wave) {
    const gc4 c = *reinterpret_cast<const gc4*>(&mat[wave == 1 ? 0 : wave][m][4 * g]);
    *reinterpret_cast<gc4*>(mw + (wave - 1) * GC * GC + m * GC + 4 * g) = wave == 3 ? -c : c;
    return;
  }
  // T, column m a lane (every group of lanes all of it): T_t = e_t - sum_{j < t} D_tj T_j
  float c[GC];
#pragma unroll
  for (int i = 0; i < GC; ++i) {
    float x = i == m ? 1.0f : 0.0f;
#pragma unroll
    for (int j = 0; j < i; ++j) x = fmaf(-mat[1][i][j], c[j], x);
    c[i] = x;
    if (g == 0) mw[3 * GC * GC + i * GC + m] = x;
  }
}

// A workgroup owns 16 columns of a head, each of its first four waves 16 KT of their key channels, as products leave them: lane (m, g)
// column m, channels 4 g .. of each 16. What bounds it is the chain of a chunk: products with the wave's channels, a meeting of the
// waves for z, T z, the update: 23 products of 32 cycles and a barrier a wave. A fifth wave moves the operands straight into LDS two chunks
// ahead and adds up and stores y. The workgroups of a head run on one XCD and share the operands in its L2. 32 heads of 64 times 1998
// tokens: 117 us and 39 for gdelta_chunk_pre, where the walk token by token took 241 and 46; with operands loaded by the four waves
// themselves, into registers or LDS, 153 to 163.
// LDS, in floats: U, R, K, A of the channels, W_16, B, E, F, T and v of four chunks; z and y of two.
template <int KT>
struct GcMap {
  static constexpr int D = 64 * KT, PARTS = 4 * GC * D, W = PARTS, M = W + 64 * KT, V = M + 4 * GC * GC, SLOT = V + GC * GC;
  static constexpr int NS = KT == 1 ? 4 : 3;  // (three: the fifth wave asks for a chunk behind the barrier, not in front of it)
  static constexpr int Z = NS * SLOT, Y = Z + 2 * 4 * 256, FLOATS = Y + 2 * 4 * 256;
};
template <int KT>
__global__ __launch_bounds__(320, 2) void gdelta_chunks_kernel(const GDeltaChunkArgs a) {
  typedef GcMap<KT> L;
  constexpr int D = L::D, CB = D / 16;
  extern __shared__ __attribute__((aligned(16))) float gl[];
  const int total = a.heads * CB, per8 = total >> 3, rem8 = total & 7, xcd = blockIdx.x & 7;
  const int at = xcd * per8 + (xcd < rem8 ? xcd : rem8) + (blockIdx.x >> 3);
  const int h = at / CB, col0 = at % CB * 16;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, m = lane & 15, g = lane >> 4;
  const int hd = a.heads * D, tile = m * 16 + 4 * g;
  const float* vp = a.p + 2 * (size_t)hd + (size_t)h * D + col0;
  float* op = a.o + (size_t)h * D + col0;
  const float* base = tl_uniform(a.ws + (size_t)h * gc_floats(D));
  auto meet = []() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  auto is_marked = [&](const float* slot) { return __builtin_amdgcn_readfirstlane(__float_as_int(slot[L::M + GC - 1])) == 0x3f800000; };
  if (wave == 4) {
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) float*)gl;
    const float* vbase = tl_uniform(vp);
    constexpr int LOADS = 16 * KT + KT + 4 + 4;
    auto fetch = [&](int c) __attribute__((always_inline)) {  // (beyond the last: the last one again, not walked)
      const int cc = __builtin_amdgcn_readfirstlane(c < a.nchunks ? c : a.nchunks - 1);
      const float* ws = base + (size_t)cc * a.heads * gc_floats(D);
      const unsigned slot = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)c % L::NS * L::SLOT * 4);
#pragma unroll
      for (int j = 0; j < 16 * KT; ++j) tl_lds_load16(slot + j * 1024, lane * 16, ws + j * 256);
#pragma unroll
      for (int j = 0; j < KT; ++j) tl_lds_load4(slot + (L::W + 64 * j) * 4, lane * 4, ws + gc_w(D) + 64 * j);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        tl_lds_load16(slot + L::M * 4 + j * 1024, lane * 16, ws + gc_mats(D) + j * 256);
        const int t = cc * GC + 4 * j + g;
        tl_lds_load4(slot + (L::V + j * 64) * 4, ((unsigned)(t < a.T ? t : a.T - 1) * (unsigned)a.ld + m) * 4u, vbase);
      }
    };
    // y of a chunk, out of the four waves' parts: four numbers a lane
    auto store_y = [&](int c) __attribute__((always_inline)) {
      const float* p = gl + L::Y + (c & 1) * 1024 + lane * 4;
      auto part = [&](int w) { return *reinterpret_cast<const gc4*>(p + 256 * w); };
      const gc4 y = (part(0) + part(1)) + (part(2) + part(3));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = c * GC + 4 * g + e;
        if (t < a.T) op[(size_t)t * hd + m] = y[e];
      }
    };
    fetch(0);
    fetch(1);
    tl_lds_barrier<0>();
    bool pending = false;
    for (int c = 0; c < a.nchunks; ++c) {
      const bool marked = is_marked(gl + (unsigned)c % L::NS * L::SLOT);
      if (marked) {
        meet();
        if (pending) store_y(c - 1);
        fetch(c + 2);
        for (int i = 0; i < 4 * GC; ++i) meet();
        tl_lds_barrier<0>();
      } else if (L::NS == 4) {  // (stores are counted, too: those of the chunk before are older)
        fetch(c + 2);
        tl_lds_barrier<LOADS>();
        if (pending) store_y(c - 1);
      } else {
        tl_lds_barrier<0>();
        fetch(c + 2);
        if (pending) store_y(c - 1);
      }
      pending = !marked;
    }
    meet();
    if (pending) store_y(a.nchunks - 1);
    return;
  }
  float* sp = a.state + ((size_t)h * D + col0 + m) * D + wave * 16 * KT + 4 * g;
  gc4 s[KT];
#pragma unroll
  for (int i = 0; i < KT; ++i) s[i] = *reinterpret_cast<const gc4*>(sp + 16 * i);
  // a marked chunk, token by token in the recurrence's own order, four meetings a token; z's place carries the two sums
  auto walk = [&](int c) {
    const float* ws = base + (size_t)c * a.heads * gc_floats(D);
    float* zz = gl + L::Z;
    for (int tt = 0; tt < GC; ++tt) {
      const bool in = c * GC + tt < a.T;
      const float v = in ? vp[(size_t)(c * GC + tt) * a.ld + m] : 0.0f;
      float x = 0.0f, y = 0.0f;
      for (int i = 0; i < KT; ++i) {
        const gc4 u = *reinterpret_cast<const gc4*>(ws + tt * D + (wave * KT + i) * 16 + 4 * g);
        x += (u[0] * s[i][0] + u[1] * s[i][1]) + (u[2] * s[i][2] + u[3] * s[i][3]);
      }
      x += __shfl_xor(x, 16);
      x += __shfl_xor(x, 32);
      meet();
      zz[wave * 64 + lane] = x;
      meet();
      x = (zz[lane] + zz[64 + lane]) + (zz[128 + lane] + zz[192 + lane]);
      for (int i = 0; i < KT; ++i) {
        const float* q = ws + tt * D + (wave * KT + i) * 16 + 4 * g;
        const gc4 r = *reinterpret_cast<const gc4*>(q + GC * D), k = *reinterpret_cast<const gc4*>(q + 2 * GC * D);
        const gc4 n = *reinterpret_cast<const gc4*>(q + 3 * GC * D), w = *reinterpret_cast<const gc4*>(q + gc_w(D) + D);
        for (int e = 0; e < 4; ++e) {
          s[i][e] = in ? fmaf(w[e], s[i][e], fmaf(-n[e], x, k[e] * v)) : s[i][e];
          y += r[e] * s[i][e];
        }
      }
      y += __shfl_xor(y, 16);
      y += __shfl_xor(y, 32);
      meet();
      zz[wave * 64 + lane] = y;
      meet();
      y = (zz[lane] + zz[64 + lane]) + (zz[128 + lane] + zz[192 + lane]);
      if (in && wave == 0 && g == 0) op[(size_t)(c * GC + tt) * hd + m] = y;
    }
  };
  // what a chunk's first products take, read a chunk ahead
  struct Lead {
    gc4 u[KT], r[KT], k[KT], v;
    float vw, b, e;
    bool marked;
  };
  auto lead = [&](Lead& q, int c) __attribute__((always_inline)) {
    const float* slot = gl + (unsigned)c % L::NS * L::SLOT;
    const float* own = slot + wave * KT * 256 + tile;
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      q.u[i] = *reinterpret_cast<const gc4*>(own + i * 256);
      q.r[i] = *reinterpret_cast<const gc4*>(own + GC * D + i * 256);
      q.k[i] = *reinterpret_cast<const gc4*>(own + 2 * GC * D + i * 256);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) q.v[e] = slot[L::V + (4 * g + e) * GC + m];
    q.vw = slot[L::V + (4 * g + wave) * GC + m];  // (a wave adds one of the four products with v to z and y, and of those with x to y)
    q.b = slot[L::M + tile + wave];
    q.e = slot[L::M + GC * GC + tile + wave];
    q.marked = is_marked(slot);
  };
  meet();
  Lead q;
  lead(q, 0);
  for (int c = 0; c < a.nchunks; ++c) {
    if (q.marked) {
      meet();
      walk(c);
      meet();
      lead(q, c + 1);
      continue;
    }
    const float* slot = gl + (unsigned)c % L::NS * L::SLOT;
    float* zb = gl + L::Z + (c & 1) * 1024 + lane * 4;
    if (c == a.nchunks - 1) {  // tokens beyond the last
#pragma unroll
      for (int e = 0; e < 4; ++e) q.v[e] = c * GC + 4 * g + e < a.T ? q.v[e] : 0.0f;
      q.vw = c * GC + 4 * g + wave < a.T ? q.vw : 0.0f;
    }
    gc4 z = gc_mfma(q.b, q.vw, gc4{});
#pragma unroll
    for (int i = 0; i < KT; ++i) z += gc_mul16(q.u[i], s[i]);
    *reinterpret_cast<gc4*>(zb + wave * 256) = z;
    gc4 tm = *reinterpret_cast<const gc4*>(slot + L::M + 3 * GC * GC + tile), y = gc_mfma(q.e, q.vw, gc4{}), kv[KT], n[KT], w[KT];
    const float f = slot[L::M + 2 * GC * GC + tile + wave];
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      n[i] = *reinterpret_cast<const gc4*>(slot + 3 * GC * D + (wave * KT + i) * 256 + tile);
      w[i] = *reinterpret_cast<const gc4*>(slot + L::W + (wave * KT + i) * 16 + 4 * g);
      y += gc_mul16(q.r[i], s[i]);
      kv[i] = gc_mul16(q.k[i], q.v);
    }
    meet();
    const gc4 zs = (*reinterpret_cast<const gc4*>(zb) + *reinterpret_cast<const gc4*>(zb + 256)) +
                   (*reinterpret_cast<const gc4*>(zb + 512) + *reinterpret_cast<const gc4*>(zb + 768));
    lead(q, c + 1);
    const gc4 x = gc_mul16(tm, zs);
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const gc4 d = kv[i] + gc_mul16(n[i], x);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[i][e] = fmaf(w[i][e], s[i][e], d[e]);
    }
    const float xw = wave < 2 ? (wave ? x[1] : x[0]) : wave == 2 ? x[2] : x[3];
    *reinterpret_cast<gc4*>(gl + L::Y + (c & 1) * 1024 + wave * 256 + lane * 4) = y + gc_mfma(f, xw, gc4{});
  }
  meet();
#pragma unroll
  for (int i = 0; i < KT; ++i) *reinterpret_cast<gc4*>(sp + 16 * i) = s[i];
}
template <int KT>
int gdelta_chunks_go(const GDeltaChunkArgs& a, hipStream_t s) {
  constexpr int lds = GcMap<KT>::FLOATS * 4;
  static_assert(lds <= 160 * 1024, "");
  static TlDeviceOnce lds_raised;
  TL_TRY(tl_raise_lds_limit(gdelta_chunks_kernel<KT>, lds, lds_raised));
  gdelta_chunk_pre_kernel<4 * KT><<<dim3(a.nchunks, a.heads), 256, 0, s>>>(a);
  gdelta_chunks_kernel<KT><<<a.heads * 4 * KT, 320, lds, s>>>(a);
  TL_HIP(hipGetLastError());
  return 0;
}

}  // namespace

bool tl_gdelta_chunks_take(int dim, float decay_scale) { return (dim == 64 || dim == 128) && fabsf(decay_scale) <= 1.0f; }
size_t tl_gdelta_chunk_floats(int T, int heads, int dim) { return (size_t)((T + GC - 1) / GC) * heads * gc_floats(dim); }
int tl_launch_gdelta_chunks(const GDeltaPreArgs& in, float* ws, float* state, float* o, hipStream_t s) {
  TL_REQUIRE(in.p && in.dw && in.w0 && in.a_bias && ws && state && o && in.T > 0, "gdelta_chunks: bad arguments");
  TL_REQUIRE(in.heads > 0 && in.heads <= 65535 && tl_gdelta_chunks_take(in.dim, in.decay_scale), "gdelta_chunks: %d heads of size %d, decay %g",
             in.heads, in.dim, in.decay_scale);
  TL_REQUIRE(in.ld >= 5 * in.heads * in.dim && in.ld % 4 == 0 && (size_t)in.T * in.ld < (1u << 30) &&
                 (((size_t)in.p | (size_t)in.dw | (size_t)in.w0 | (size_t)in.a_bias | (size_t)ws | (size_t)state) & 15) == 0,
             "gdelta_chunks: rows of %d floats or addresses off 16 bytes", in.ld);
  const GDeltaChunkArgs a = {in.p, in.ld, in.dw, in.w0, in.a_bias, in.decay_scale, ws, state, o, in.T, in.heads, (in.T + GC - 1) / GC};
  return in.dim == 64 ? gdelta_chunks_go<1>(a, s) : gdelta_chunks_go<2>(a, s);
}

int tl_launch_delta_pre(const DeltaPreArgs& a, hipStream_t s) {
  TL_REQUIRE(a.p && a.a && a.conv && a.a_log && a.dt_bias && a.qkv && a.beta && a.g && a.T > 0, "delta_pre: bad arguments");
  TL_REQUIRE(a.heads > 0 && a.kv_heads > 0 && a.heads % a.kv_heads == 0 && a.dim > 0 && a.vdim > 0,
             "delta_pre: %d heads over %d query/key heads, sizes %d / %d", a.heads, a.kv_heads, a.dim, a.vdim);
  TL_REQUIRE(a.taps >= 1 && (a.taps == 1 || a.hist), "delta_pre: %d taps", a.taps);
  const int C = 2 * a.kv_heads * a.dim + a.heads * a.vdim;
  TL_REQUIRE(a.ld >= C + a.heads, "delta_pre: row stride %d below %d", a.ld, C + a.heads);
  TL_REQUIRE(!a.a_per_head || a.a_ld >= a.heads, "delta_pre: a decay per head with row stride %d", a.a_ld);
  TL_REQUIRE(a.dim <= 512 && a.vdim <= 512, "delta_pre: head sizes %d / %d above 512", a.dim, a.vdim);
  TL_REQUIRE(2 * a.kv_heads + a.heads <= 65535, "delta_pre: too many heads");
  delta_pre_kernel<<<dim3(a.T, 2 * a.kv_heads + a.heads), 128, 0, s>>>(a);
  if (a.T > 1 && a.taps > 1) conv_history_kernel<<<(C + 255) / 256, 256, 0, s>>>(a);
  TL_HIP(hipGetLastError());
  return 0;
}

int tl_launch_delta_scan(const DeltaScanArgs& a, hipStream_t s) {
  TL_REQUIRE(a.q && a.k && a.v && (a.beta || a.plain_write) && a.g && a.state && a.o && a.T > 0, "delta_scan: bad arguments");
  TL_REQUIRE(a.heads > 0 && a.kv_heads > 0 && a.heads % a.kv_heads == 0 && a.dim > 0 && a.vdim > 0 && a.heads <= 65535,
             "delta_scan: %d heads over %d query/key heads, sizes %d / %d", a.heads, a.kv_heads, a.dim, a.vdim);
  TL_REQUIRE(a.dim <= 256, "delta_scan: key size %d above 256", a.dim);
  const dim3 grid((a.vdim + 15) / 16, a.heads);
  const int e = (a.dim + 15) / 16;
  auto launch = [&](auto plain) {
    constexpr bool P = decltype(plain)::value;
    if (e <= 1) delta_scan_kernel<1, P><<<grid, 256, 0, s>>>(a);
    else if (e <= 2) delta_scan_kernel<2, P><<<grid, 256, 0, s>>>(a);
    else if (e <= 4) delta_scan_kernel<4, P><<<grid, 256, 0, s>>>(a);
    else if (e <= 8) delta_scan_kernel<8, P><<<grid, 256, 0, s>>>(a);
    else delta_scan_kernel<16, P><<<grid, 256, 0, s>>>(a);
  };
  if (a.plain_write) launch(std::true_type{});
  else launch(std::false_type{});
  TL_HIP(hipGetLastError());
  return 0;
}

bool tl_gla_step_fits(int dim, int vdim, int rank) { return dim <= 256 && vdim <= 2048 && rank <= 4096; }

int tl_launch_gla_step(const GlaStepArgs& a, hipStream_t s) {
  TL_REQUIRE(a.p && a.a2 && a.a2_b && a.norm && a.state && a.o && a.rank > 0 && a.heads > 0 && a.dim > 0 && a.vdim > 0, "gla_step: bad arguments");
  TL_REQUIRE(tl_gla_step_fits(a.dim, a.vdim, a.rank), "gla_step: sizes %d / %d, inner size %d", a.dim, a.vdim, a.rank);
  const int e = (a.dim + 15) / 16, ep = e <= 1 ? 1 : e <= 2 ? 2 : e <= 4 ? 4 : e <= 8 ? 8 : 16;
  const int vec = a.dim == 16 * ep && ((size_t)a.state & 15) == 0;
  const size_t lds = sizeof(float) * (3 * 16 * (size_t)ep + 2 * (size_t)a.vdim + a.rank);
  switch (ep) {
    case 1: gla_step_kernel<1><<<a.heads, 1024, lds, s>>>(a, vec); break;
    case 2: gla_step_kernel<2><<<a.heads, 1024, lds, s>>>(a, vec); break;
    case 4: gla_step_kernel<4><<<a.heads, 1024, lds, s>>>(a, vec); break;
    case 8: gla_step_kernel<8><<<a.heads, 1024, lds, s>>>(a, vec); break;
    default: gla_step_kernel<16><<<a.heads, 1024, lds, s>>>(a, vec); break;
  }
  TL_HIP(hipGetLastError());
  return 0;
}

int tl_launch_gated_head_norm_rows(float* o, const float* gate, int gate_ld, const float* w, int w_per_head, int T, int heads,
                                   int vdim, float eps, hipStream_t s) {
  TL_REQUIRE(o && gate && w, "gated_head_norm: bad arguments");
  HeadNormArgs a = {};
  a.o = o;
  a.gate = gate;
  a.gate_ld = gate_ld;
  a.w = w;
  a.w_per_head = w_per_head;
  a.out_scale = 1.0f;
  a.T = T;
  a.heads = heads;
  a.vdim = vdim;
  a.eps = eps;
  return tl_launch_head_norm(a, s);
}

int tl_launch_head_norm(const HeadNormArgs& a, hipStream_t s) {
  TL_REQUIRE(a.o && a.T > 0 && a.heads > 0 && a.vdim > 0 && (!a.gate || a.gate_ld >= a.heads * a.vdim), "head_norm: bad arguments");
  TL_REQUIRE(a.gate_act == 0 || a.gate_act == 1, "head_norm: gate activation %d", a.gate_act);
  const long long n = (long long)a.T * a.heads;
  TL_REQUIRE(n <= 0x7fffffffLL, "head_norm: too many heads");
  head_norm_kernel<<<(unsigned)((n + 3) / 4), 256, 0, s>>>(a);
  TL_HIP(hipGetLastError());
  return 0;
}

int tl_launch_linear_pre(const LinearPreArgs& a, hipStream_t s) {
  TL_REQUIRE(a.p && a.lower && a.f_bias && a.qk && a.g && a.T > 0 && a.T <= 65535 && a.heads > 0 && a.dim > 0,
             "linear_pre: bad arguments");
  TL_REQUIRE(a.ld >= 2 * a.heads * a.dim, "linear_pre: row stride %d below %d", a.ld, 2 * a.heads * a.dim);
  linear_pre_kernel<<<dim3((a.heads * a.dim + 255) / 256, a.T), 256, 0, s>>>(a);
  TL_HIP(hipGetLastError());
  return 0;
}

int tl_launch_gated_head_norm(float* o, const float* gate, const float* w, int T, int heads, int vdim, float eps, hipStream_t s) {
  return tl_launch_gated_head_norm_rows(o, gate, heads * vdim, w, 0, T, heads, vdim, eps, s);
}

int tl_launch_gdelta_pre(const GDeltaPreArgs& a, hipStream_t s) {
  TL_REQUIRE(a.p && a.dw && a.w0 && a.a_bias && a.w && a.u && a.au && a.rau && a.rk && a.T > 0, "gdelta_pre: bad arguments");
  TL_REQUIRE(a.heads > 0 && a.heads <= 65535 && a.dim > 0 && a.dim <= 512, "gdelta_pre: %d heads of size %d", a.heads, a.dim);
  TL_REQUIRE(a.ld >= 5 * a.heads * a.dim, "gdelta_pre: row stride %d below %d", a.ld, 5 * a.heads * a.dim);
  gdelta_pre_kernel<<<dim3(a.T, a.heads), 128, 0, s>>>(a);
  TL_HIP(hipGetLastError());
  return 0;
}

int tl_launch_gdelta_scan(const GDeltaScanArgs& a, hipStream_t s) {
  TL_REQUIRE(a.r && a.k && a.v && a.w && a.u && a.au && a.rau && a.rk && a.state && a.o && a.T > 0, "gdelta_scan: bad arguments");
  TL_REQUIRE(a.heads > 0 && a.heads <= 65535 && a.dim > 0 && a.vdim > 0, "gdelta_scan: %d heads, sizes %d / %d", a.heads, a.dim, a.vdim);
  TL_REQUIRE(a.dim <= 256, "gdelta_scan: key size %d above 256", a.dim);
  const dim3 grid((a.vdim + 15) / 16, a.heads);
  const int e = (a.dim + 15) / 16;
  const bool wide = (a.ld & 3) == 0 && (((size_t)a.r | (size_t)a.k | (size_t)a.w | (size_t)a.u | (size_t)a.au | (size_t)a.state) & 15) == 0;
  if (wide && a.dim == 64) gdelta_scan_wide_kernel<4><<<grid, 256, 0, s>>>(a);
  else if (wide && a.dim == 128) gdelta_scan_wide_kernel<8><<<grid, 256, 0, s>>>(a);
  else if (e <= 1) gdelta_scan_kernel<1><<<grid, 256, 0, s>>>(a);
  else if (e <= 2) gdelta_scan_kernel<2><<<grid, 256, 0, s>>>(a);
  else if (e <= 4) gdelta_scan_kernel<4><<<grid, 256, 0, s>>>(a);
  else if (e <= 8) gdelta_scan_kernel<8><<<grid, 256, 0, s>>>(a);
  else gdelta_scan_kernel<16><<<grid, 256, 0, s>>>(a);
  TL_HIP(hipGetLastError());
  return 0;
}

extern "C" int tl_debug_general_delta_chunks(const float* p_dev, int ld, const float* dw_dev, const float* w0_dev, const float* a_bias_dev,
                                             float decay_scale, float* state_dev, float* o_dev, float* ws_dev, long long ws_floats,
                                             int num_tokens, int heads, int dim, void* stream) {
  TL_REQUIRE(num_tokens > 0 && heads > 0 && heads <= 65535 && tl_gdelta_chunks_take(dim, decay_scale) &&
                 ws_floats >= (long long)tl_gdelta_chunk_floats(num_tokens, heads, dim),
             "tl_debug_general_delta_chunks: bad argument");
  GDeltaPreArgs p = {};
  p.p = p_dev;
  p.ld = ld;
  p.dw = dw_dev;
  p.w0 = w0_dev;
  p.a_bias = a_bias_dev;
  p.decay_scale = decay_scale;
  p.T = num_tokens;
  p.heads = heads;
  p.dim = dim;
  return tl_launch_gdelta_chunks(p, ws_dev, state_dev, o_dev, static_cast<hipStream_t>(stream));
}

extern "C" int tl_general_delta(const float* p_dev, int ld, const float* dw_dev, const float* w0_dev, const float* a_bias_dev,
                                float decay_scale, float* state_dev, float* o_dev, float* scratch_dev, int num_tokens, int heads,
                                int dim, void* stream) {
  TL_REQUIRE(scratch_dev && num_tokens > 0 && heads > 0 && dim > 0, "tl_general_delta: bad arguments");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t n = (size_t)num_tokens * heads * dim, m = (size_t)num_tokens * heads;
  GDeltaPreArgs p = {};
  p.p = p_dev;
  p.ld = ld;
  p.dw = dw_dev;
  p.w0 = w0_dev;
  p.a_bias = a_bias_dev;
  p.decay_scale = decay_scale;
  p.T = num_tokens;
  p.heads = heads;
  p.dim = dim;
  p.w = scratch_dev;
  p.u = scratch_dev + n;
  p.au = scratch_dev + 2 * n;
  p.rau = scratch_dev + 3 * n;
  p.rk = scratch_dev + 3 * n + m;
  TL_TRY(tl_launch_gdelta_pre(p, s));
  GDeltaScanArgs d = {};
  d.r = p_dev;
  d.k = p_dev + (size_t)heads * dim;
  d.v = p_dev + 2 * (size_t)heads * dim;
  d.ld = ld;
  d.w = p.w;
  d.u = p.u;
  d.au = p.au;
  d.rau = p.rau;
  d.rk = p.rk;
  d.state = state_dev;
  d.o = o_dev;
  d.T = num_tokens;
  d.heads = heads;
  d.dim = dim;
  d.vdim = dim;
  return tl_launch_gdelta_scan(d, s);
}

extern "C" int tl_delta_prepare(const float* p_dev, int ld, const float* a_dev, int num_tokens, int heads, int kv_heads, int dim,
                                int vdim, int taps, const void* conv_bf16_dev, float* history_dev, const float* a_log_dev,
                                const float* dt_bias_dev, float* qkv_dev, float* beta_dev, float* g_dev, void* stream) {
  DeltaPreArgs a = {};
  a.p = p_dev;
  a.ld = ld;
  a.a = a_dev;
  a.T = num_tokens;
  a.heads = heads;
  a.kv_heads = kv_heads;
  a.dim = dim;
  a.vdim = vdim;
  a.taps = taps;
  a.conv = static_cast<const uint16_t*>(conv_bf16_dev);
  a.hist = history_dev;
  a.a_log = a_log_dev;
  a.dt_bias = dt_bias_dev;
  a.qkv = qkv_dev;
  a.beta = beta_dev;
  a.g = g_dev;
  return tl_launch_delta_pre(a, static_cast<hipStream_t>(stream));
}

extern "C" int tl_gated_head_norm(float* o_dev, const float* gate_dev, const float* weight_dev, int num_tokens, int heads, int vdim,
                                  float eps, void* stream) {
  return tl_launch_gated_head_norm(o_dev, gate_dev, weight_dev, num_tokens, heads, vdim, eps, static_cast<hipStream_t>(stream));
}

extern "C" int tl_delta_rule(const float* q_dev, const float* k_dev, const float* v_dev, const float* beta_dev, const float* g_dev,
                             float* state_dev, float* o_dev, int num_tokens, int heads, int kv_heads, int dim, int vdim,
                             void* stream) {
  DeltaScanArgs a = {};
  a.q = q_dev;
  a.k = k_dev;
  a.ldq = kv_heads * dim;
  a.v = v_dev;
  a.ldv = heads * vdim;
  a.beta = beta_dev;
  a.g = g_dev;
  a.state = state_dev;
  a.o = o_dev;
  a.T = num_tokens;
  a.heads = heads;
  a.kv_heads = kv_heads;
  a.dim = dim;
  a.vdim = vdim;
  return tl_launch_delta_scan(a, static_cast<hipStream_t>(stream));
}

extern "C" int tl_head_norm(float* o_dev, const float* sub_dev, float sub_coef, const float* gate_dev, int gate_ld, int gate_act,
                            const float* weight_dev, int weight_per_head, float out_scale, int num_tokens, int heads, int vdim,
                            float eps, void* stream) {
  HeadNormArgs a = {};
  a.o = o_dev;
  a.sub = sub_dev;
  a.sub_coef = sub_coef;
  a.gate = gate_dev;
  a.gate_ld = gate_ld;
  a.gate_act = gate_act;
  a.w = weight_dev;
  a.w_per_head = weight_per_head;
  a.out_scale = out_scale;
  a.T = num_tokens;
  a.heads = heads;
  a.vdim = vdim;
  a.eps = eps;
  return tl_launch_head_norm(a, static_cast<hipStream_t>(stream));
}

extern "C" int tl_gated_linear_attention(const float* p_dev, int ld, const float* lower_dev, const float* f_bias_dev,
                                         float* state_dev, float* o_dev, float* scratch_dev, int num_tokens, int heads, int dim,
                                         int vdim, void* stream) {
  TL_REQUIRE(scratch_dev && num_tokens > 0 && heads > 0 && dim > 0 && vdim > 0, "tl_gated_linear_attention: bad arguments");
  TL_REQUIRE(ld >= 2 * heads * dim + heads * vdim, "tl_gated_linear_attention: row stride %d below q | f | v", ld);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t hd = (size_t)heads * dim;
  LinearPreArgs p = {};
  p.p = p_dev;
  p.ld = ld;
  p.T = num_tokens;
  p.heads = heads;
  p.dim = dim;
  p.lower = lower_dev;
  p.f_bias = f_bias_dev;
  p.qk = scratch_dev;
  p.g = scratch_dev + 2 * hd * num_tokens;
  TL_TRY(tl_launch_linear_pre(p, s));
  DeltaScanArgs d = {};
  d.q = p.qk;
  d.k = p.qk + hd;
  d.ldq = (int)(2 * hd);
  d.v = p_dev + 2 * hd;
  d.ldv = ld;
  d.g = p.g;
  d.state = state_dev;
  d.o = o_dev;
  d.T = num_tokens;
  d.heads = heads;
  d.kv_heads = heads;
  d.dim = dim;
  d.vdim = vdim;
  d.plain_write = 1;
  return tl_launch_delta_scan(d, s);
}

extern "C" int tl_channel_decay_attention(const float* p_dev, int ld, int q_off, int k_off, int v_off, const float* alpha_dev,
                                          float q_scale, float* state_dev, float* o_dev, int num_tokens, int heads, int dim, int vdim,
                                          void* stream) {
  TL_REQUIRE(p_dev && q_off >= 0 && k_off >= 0 && v_off >= 0 && q_off + heads * dim <= ld && k_off + heads * dim <= ld &&
                 v_off + heads * vdim <= ld,
             "tl_channel_decay_attention: columns outside rows of %d", ld);
  DeltaScanArgs d = {};
  d.q = p_dev + q_off;
  d.k = p_dev + k_off;
  d.ldq = ld;
  d.v = p_dev + v_off;
  d.ldv = ld;
  d.g = alpha_dev;
  d.state = state_dev;
  d.o = o_dev;
  d.T = num_tokens;
  d.heads = heads;
  d.kv_heads = heads;
  d.dim = dim;
  d.vdim = vdim;
  d.plain_write = 1;
  d.q_scale = q_scale;
  return tl_launch_delta_scan(d, static_cast<hipStream_t>(stream));
}

extern "C" int tl_channel_decay_step(const float* p_dev, const void* a2_bf16_dev, const float* a2_bias_dev, int rank, float power,
                                     float q_scale, const float* norm_dev, float eps, float* state_dev, float* o_dev, int heads, int dim,
                                     int vdim, void* stream) {
  GlaStepArgs a = {};
  a.p = p_dev;
  a.a2 = static_cast<const uint16_t*>(a2_bf16_dev);
  a.a2_b = a2_bias_dev;
  a.rank = rank;
  a.power = power;
  a.q_scale = q_scale;
  a.norm = norm_dev;
  a.eps = eps;
  a.state = state_dev;
  a.o = o_dev;
  a.heads = heads;
  a.dim = dim;
  a.vdim = vdim;
  return tl_launch_gla_step(a, static_cast<hipStream_t>(stream));
}
