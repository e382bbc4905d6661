// tl_sample.hip — temperature / top-k / top-p sampling on the device, the non-greedy half of
// sample_top_k_top_p_temperature (api.cpp:126-216) + apply_repetition_penalty (api.cpp:86-97).
//
// The reference copies vocab * 4 B to the host every token and sorts the whole vocabulary there (std::sort over
// 128 k pairs, ~10 ms: six decode steps' worth). Here the logits never leave HBM:
//   1. SK_SLICES workgroups apply the repetition penalty in place (once per occurrence) and take their slice's maximum,
//   2. the same ones sum exp((logit - max) / T) of their slices in FP64,
//   3. and round each probability to FP32 (api.cpp:143-175). The k-th largest of the slice maxima bounds the k-th largest
//      probability from below, so only entries at least as probable as that one can be selected: they go to a short list of
//      64-bit keys (prob bits << 32 | id), some 50 of them for k = 40,
//   4. one workgroup sorts the list in LDS (bitonic) — descending by probability, ties by HIGHER id, as
//      std::greater<std::pair<float,int>> orders them — or, where it is longer than 1024 (k > SK_SLICES, flat or underflowing
//      probabilities), selects the k largest keys of the whole vector with a radix select first; walks the FP32 cumulative
//      sum up to top_p, renormalises, draws with the inverse CDF in FP64 the way std::discrete_distribution does (normalised
//      partial sums, first entry whose partial sum exceeds u), writes the id and advances the step state.
// The whole of it in one workgroup, as it was, is bound by one CU's round trips and FP64 exponentials: 123 us for 32000
// logits at k = 40, more than a seventh of a 1.1B step; the four launches together take 27 us (16 sampled steps: 12.0 -> 10.5 ms).
// The uniform variate comes from a counter-based generator (splitmix64 of seed + step); the reference seeds a
// std::mt19937 from std::random_device, so its streams are not reproducible either: parity is on the candidate set
// and its probabilities (tests/test_sample_gpu.py), not on the random stream.
// Limit: effective top_k <= 1024 (top_k <= 0 or >= vocab means "no top-k" in the reference; that form stays on the
// host path, tl_session.cpp).
#include <math.h>

#include "tl_internal.h"
#include "tl_lanes.h"

namespace {

constexpr int SK_MAX = TL_SAMPLE_MAX_TOP_K;
constexpr int SK_THREADS = 1024;
typedef unsigned long long u64;

__device__ __forceinline__ u64 splitmix64(u64 x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

__device__ __forceinline__ u64 key_of(float p, int id) { return ((u64)__float_as_uint(p) << 32) | (unsigned)id; }

constexpr int SK_SLICES = 128, SK_SLICE_THREADS = 256;
struct SampleWs {  // behind the probabilities
  float smax[SK_SLICES];
  double ssum[SK_SLICES];
  unsigned count;
  u64 list[SK_MAX];
};
size_t ws_offset(int n) { return (sizeof(float) * (size_t)n + 15) & ~(size_t)15; }
__device__ __forceinline__ int slice_len(int n) { return (n + SK_SLICES - 1) / SK_SLICES; }

// the maximum over the slices, by every thread of a workgroup (sm: 1 + a word per wave)
template <int NT>
__device__ __forceinline__ float slices_max(const SampleWs* ws, float* sm) {
  float m = threadIdx.x < SK_SLICES ? ws->smax[threadIdx.x] : -INFINITY;
  m = tl_wave_max(m);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = m;
  __syncthreads();
  m = sm[0];
#pragma unroll
  for (int i = 1; i < NT / 64; ++i) m = fmaxf(m, sm[i]);
  return m;
}
__device__ __forceinline__ float prob_of(float logit, float mx, float inv_t, double total, int n) {
  const double e = exp((double)((logit - mx) * inv_t));
  return (float)(total > 0.0 ? e / total : 1.0 / n);
}

// 1. penalty of this slice's logits, its maximum
__global__ __launch_bounds__(SK_SLICE_THREADS) void sample_max_kernel(float* __restrict__ logits, int n, const int* __restrict__ state,
                                                                      int state_header, SampleWs* __restrict__ ws) {
  __shared__ float sm[SK_SLICE_THREADS / 64];
  const int len = slice_len(n), lo = blockIdx.x * len, hi = lo + len < n ? lo + len : n, tid = threadIdx.x;
  if (state) {
    const float penalty = __int_as_float(state[3]);
    if (penalty > 1.0f && tid < 64) {  // one of the last 64 ids per lane; the first lane that holds an id applies every occurrence
      const int n_hist = state[2], at = (n_hist > 64 ? n_hist - 64 : 0) + tid;
      const int id = at < n_hist ? state[state_header + at] : -1;
      int times = 0, first = 64;
      for (int j = 0; j < 64; ++j) {
        const int other = __builtin_amdgcn_readlane(id, j);
        if (other == id) {
          ++times;
          if (first == 64) first = j;
        }
      }
      if (first == tid && id >= lo && id < hi) {
        float l = logits[id];
        for (int j = 0; j < times; ++j) l = (l > 0.0f) ? l / penalty : l * penalty;
        logits[id] = l;
      }
    }
    __syncthreads();
  }
  float m = -INFINITY;
  for (int i = lo + tid; i < hi; i += SK_SLICE_THREADS) m = fmaxf(m, logits[i]);
  m = tl_wave_max(m);
  if ((tid & 63) == 0) sm[tid >> 6] = m;
  __syncthreads();
  if (tid == 0) {
    for (int i = 1; i < SK_SLICE_THREADS / 64; ++i) m = fmaxf(m, sm[i]);
    ws->smax[blockIdx.x] = m;
    if (blockIdx.x == 0) ws->count = 0;
  }
}
// 2. sum of this slice's exponentials
__global__ __launch_bounds__(SK_SLICE_THREADS) void sample_sum_kernel(const float* __restrict__ logits, int n,
                                                                      const TlSampleParams* __restrict__ sp, SampleWs* __restrict__ ws) {
  __shared__ float sm[SK_SLICE_THREADS / 64];
  __shared__ double sd[SK_SLICE_THREADS / 64];
  const float temperature = sp->temperature;
  if (temperature < 0.05f) return;  // greedy (uniform)
  const int len = slice_len(n), lo = blockIdx.x * len, hi = lo + len < n ? lo + len : n, tid = threadIdx.x;
  const float mx = slices_max<SK_SLICE_THREADS>(ws, sm), inv_t = 1.0f / temperature;
  double part = 0.0;
  for (int i = lo + tid; i < hi; i += SK_SLICE_THREADS) part += exp((double)((logits[i] - mx) * inv_t));
  part = tl_wave_sum(part);
  if ((tid & 63) == 0) sd[tid >> 6] = part;
  __syncthreads();
  if (tid == 0) {
    for (int i = 1; i < SK_SLICE_THREADS / 64; ++i) part += sd[i];
    ws->ssum[blockIdx.x] = part;
  }
}
__device__ __forceinline__ int effective_k(const TlSampleParams* sp, int n) {
  int k = sp->top_k;
  if (k <= 0 || k > n) k = n;
  return k > SK_MAX ? SK_MAX : k;  // (the host entry points reject more)
}
// 3. probabilities; the entries that can be among the k largest go to the list
__global__ __launch_bounds__(SK_SLICE_THREADS) void sample_list_kernel(const float* __restrict__ logits, int n, float* __restrict__ probs,
                                                                       const TlSampleParams* __restrict__ sp, SampleWs* __restrict__ ws) {
  __shared__ float sm[SK_SLICE_THREADS / 64], mxs[SK_SLICES], s_bound;
  __shared__ double sd[SK_SLICES];
  const float temperature = sp->temperature;
  if (temperature < 0.05f) return;  // greedy (uniform)
  const int len = slice_len(n), lo = blockIdx.x * len, hi = lo + len < n ? lo + len : n, tid = threadIdx.x;
  if (tid < SK_SLICES) {
    mxs[tid] = ws->smax[tid];
    sd[tid] = ws->ssum[tid];
  }
  const float mx = slices_max<SK_SLICE_THREADS>(ws, sm), inv_t = 1.0f / temperature;  // (its barrier covers mxs and sd)
  double total = 0.0;
#pragma unroll 8
  for (int i = 0; i < SK_SLICES; ++i) total += sd[i];
  // the k-th largest slice maximum: as many entries are at least as probable as it
  const int k = effective_k(sp, n);
  if (tid == 0) s_bound = -INFINITY;
  __syncthreads();
  if (tid < SK_SLICES && k <= SK_SLICES) {
    int rank = 0;
    const float own = mxs[tid];
#pragma unroll 8
    for (int i = 0; i < SK_SLICES; ++i) rank += mxs[i] > own || (mxs[i] == own && i < tid);
    if (rank == k - 1) s_bound = own;
  }
  __syncthreads();
  const float bound = prob_of(s_bound, mx, inv_t, total, n);
  for (int i = lo + tid; i < hi; i += SK_SLICE_THREADS) {
    const float p = prob_of(logits[i], mx, inv_t, total, n);
    probs[i] = p;
    if (!(p < bound) || k > SK_SLICES) {
      const unsigned at = atomicAdd(&ws->count, 1u);
      if (at < SK_MAX) ws->list[at] = key_of(p, i) + 1;
    }
  }
}

// 4. logits [n], probs [n] (from the list kernel). state: the engine's step state {token, pos, n_hist, penalty, history...}
// or NULL for the operator-level call.
__global__ __launch_bounds__(SK_THREADS) void sample_pick_kernel(const float* __restrict__ logits, int n,
                                                                 const float* __restrict__ probs, const SampleWs* __restrict__ ws,
                                                                 int* __restrict__ state, int state_header, int hist_cap,
                                                                 TlSampleParams* sp, int* __restrict__ out_id,
                                                                 int* __restrict__ cand_ids, float* __restrict__ cand_probs,
                                                                 int* __restrict__ n_cand) {
  __shared__ float sm[SK_THREADS / 64], pk[SK_MAX];
  __shared__ double pd[SK_MAX];
  __shared__ unsigned hist[256];
  __shared__ u64 keys[SK_MAX];
  __shared__ u64 s_prefix;
  __shared__ int s_remaining, s_done, s_count, s_pick, s_keep;
  __shared__ float s_kept;
  __shared__ double s_wsum;
  const int tid = threadIdx.x;
  const float temperature = sp->temperature, top_p = sp->top_p;
  if (temperature < 0.05f) {  // greedy: first maximum (api.cpp:134-136), in the first slice that holds it
    const float mx = slices_max<SK_THREADS>(ws, sm);
    if (tid == 0) s_pick = 0x7fffffff;
    __syncthreads();
    if (tid < SK_SLICES && ws->smax[tid] == mx) atomicMin(&s_pick, tid);
    __syncthreads();
    const int sl = s_pick, len = slice_len(n);
    __syncthreads();
    if (tid == 0) s_pick = 0x7fffffff;
    __syncthreads();
    if (sl < SK_SLICES)
      for (int i = sl * len + tid; i < n && i < (sl + 1) * len; i += SK_THREADS)
        if (logits[i] == mx) atomicMin(&s_pick, i);
    __syncthreads();
    if (tid == 0) {
      if (s_pick == 0x7fffffff) s_pick = 0;
      if (n_cand) *n_cand = 0;
    }
    __syncthreads();
  } else {
    const int k = effective_k(sp, n), listed = (int)ws->count;
    int nkeys = listed;
    if (listed <= SK_MAX) {
      if (tid < SK_MAX) keys[tid] = tid < listed ? ws->list[tid] : 0;  // 0 = empty slot (real keys are stored + 1)
      __syncthreads();
    } else {
      // radix select of the k largest keys (prob bits, id), most significant byte first
      if (tid == 0) {
        s_prefix = 0;
        s_remaining = k;
        s_done = 0;
      }
      __syncthreads();
      int nbytes = 0;  // bytes of the key fixed so far (from the top)
      for (int byte = 7; byte >= 0; --byte) {
        if (s_done) break;
        for (int b = tid; b < 256; b += SK_THREADS) hist[b] = 0;
        __syncthreads();
        const u64 prefix = s_prefix;
        const int sh = 8 * byte;
        for (int i = tid; i < n; i += SK_THREADS) {
          const u64 key = key_of(probs[i], i);
          if (byte == 7 || (key >> (sh + 8)) == (prefix >> (sh + 8))) atomicAdd(&hist[(unsigned)(key >> sh) & 255u], 1u);
        }
        __syncthreads();
        if (tid == 0) {
          int rem = s_remaining, b = 255;
          unsigned matching = 0;
          for (int q = 0; q < 256; ++q) matching += hist[q];
          if ((int)matching == rem) {  // everything that shares the prefix so far is selected
            s_done = 1;
          } else {
            while (b > 0 && (int)hist[b] < rem) rem -= hist[b--];
            s_prefix = prefix | ((u64)b << sh);
            s_remaining = rem;
          }
        }
        __syncthreads();
        if (!s_done) nbytes = 8 - byte;
      }
      if (tid == 0) s_count = 0;
      for (int i = tid; i < SK_MAX; i += SK_THREADS) keys[i] = 0;
      __syncthreads();
      const int sh = 64 - 8 * nbytes;  // bits below the fixed part
      const u64 prefix = s_prefix;
      for (int i = tid; i < n; i += SK_THREADS) {
        const u64 key = key_of(probs[i], i);
        // above the prefix on the fixed bytes: selected; equal: selected (either everything that matches was taken,
        // or all 8 bytes are fixed and the key is the k-th one itself)
        const bool sel = nbytes == 0 ? true : (key >> sh) >= (prefix >> sh);
        if (sel) {
          const int slot = atomicAdd(&s_count, 1);
          if (slot < SK_MAX) keys[slot] = key + 1;
        }
      }
      __syncthreads();
      nkeys = s_count < SK_MAX ? s_count : SK_MAX;
    }
    // bitonic sort of the first power of two >= nkeys slots, descending
    int slots = 2;
    while (slots < nkeys) slots <<= 1;
    for (int size = 2; size <= slots; size <<= 1)
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        const int j = tid ^ stride;
        if (tid < slots && j > tid) {
          const bool desc = (tid & size) == 0;
          const u64 a = keys[tid], b = keys[j];
          if (desc ? a < b : a > b) {
            keys[tid] = b;
            keys[j] = a;
          }
        }
        __syncthreads();
      }
    const int nsel = nkeys < k ? nkeys : k;
    if (tid < nsel) pk[tid] = __uint_as_float((unsigned)((keys[tid] - 1) >> 32));
    __syncthreads();
    // top-p cut, renormalisation, draw: the sums in order by one thread, as the reference does them; the quotients by all
    if (tid == 0) {
      float cum = 0.f;
      int keep = nsel;
      for (int i = 0; i < nsel; ++i) {
        cum += pk[i];
        if (cum >= top_p) {
          keep = i + 1;
          break;
        }
      }
      s_keep = keep;
      s_kept = cum;  // (the same additions in the same order)
    }
    __syncthreads();
    const int keep = s_keep;
    const float kept = s_kept;
    // std::discrete_distribution: weights normalised in FP64, pick the first index whose partial sum exceeds u
    const float fp = tid < keep ? (kept > 0.f ? pk[tid] / kept : 1.0f / (float)keep) : 0.f;
    __syncthreads();
    if (tid < keep) {
      pk[tid] = fp;
      if (cand_ids) cand_ids[tid] = (int)((keys[tid] - 1) & 0xffffffffu);
      if (cand_probs) cand_probs[tid] = fp;
    }
    __syncthreads();
    if (tid == 0) {
      double wsum = 0.0;
#pragma unroll 8
      for (int i = 0; i < keep; ++i) wsum += (double)pk[i];
      s_wsum = wsum;
    }
    __syncthreads();
    if (tid < keep) pd[tid] = (double)fp / s_wsum;
    __syncthreads();
    if (tid == 0) {
      double u;
      if (sp->use_fixed_u) {
        u = (double)sp->fixed_u;
      } else {
        const u64 r = splitmix64(sp->seed + 0xD1B54A32D192ED03ull * (u64)sp->counter);
        u = (double)(r >> 11) * (1.0 / 9007199254740992.0);
        sp->counter = sp->counter + 1;
      }
      double acc = 0.0;
      int chosen = keep - 1;
      for (int i = 0; i < keep - 1; ++i) {
        acc += pd[i];
        if (u < acc) {
          chosen = i;
          break;
        }
      }
      if (n_cand) *n_cand = keep;
      s_pick = keep > 0 ? (int)((keys[chosen] - 1) & 0xffffffffu) : 0;
    }
    __syncthreads();
  }
  if (tid == 0) {
    const int pick = s_pick;
    if (out_id) *out_id = pick;
    if (state) {  // advance the step state exactly as the greedy tail does
      const int n_hist = state[2];
      state[0] = pick;
      state[1] = state[1] + 1;
      if (n_hist < hist_cap) state[state_header + n_hist] = pick;
      state[2] = n_hist + 1;
    }
  }
}

}  // namespace

size_t tl_sample_scratch_bytes(int n) { return ws_offset(n) + sizeof(SampleWs); }
int tl_launch_sample_topk(float* logits, int n, float* probs_scratch, int* state, int state_header, int hist_cap,
                          TlSampleParams* params_dev, int* out_id, int* cand_ids, float* cand_probs, int* n_cand,
                          hipStream_t s) {
  SampleWs* ws = reinterpret_cast<SampleWs*>(reinterpret_cast<unsigned char*>(probs_scratch) + ws_offset(n));
  sample_max_kernel<<<SK_SLICES, SK_SLICE_THREADS, 0, s>>>(logits, n, state, state_header, ws);
  sample_sum_kernel<<<SK_SLICES, SK_SLICE_THREADS, 0, s>>>(logits, n, params_dev, ws);
  sample_list_kernel<<<SK_SLICES, SK_SLICE_THREADS, 0, s>>>(logits, n, probs_scratch, params_dev, ws);
  sample_pick_kernel<<<1, SK_THREADS, 0, s>>>(logits, n, probs_scratch, ws, state, state_header, hist_cap, params_dev, out_id, cand_ids,
                                              cand_probs, n_cand);
  TL_HIP(hipGetLastError());
  return 0;
}

// operator-level call: logits are NOT modified (no penalty); u in [0,1) is the caller's uniform variate
extern "C" int tl_sample_top_k_top_p(const float* logits_dev, int n, float temperature, int top_k, float top_p, float u,
                                     int* id_dev, int* cand_ids_dev, float* cand_probs_dev, int* n_cand_dev,
                                     void* stream) {
  TL_REQUIRE(logits_dev && id_dev && n > 0, "tl_sample_top_k_top_p: bad argument");
  TL_REQUIRE(u >= 0.0f && u < 1.0f, "tl_sample_top_k_top_p: u = %g outside [0,1)", (double)u);
  const int k = (top_k <= 0 || top_k > n) ? n : top_k;
  TL_REQUIRE(temperature < 0.05f || k <= SK_MAX,
             "tl_sample_top_k_top_p: effective top_k %d exceeds the device sampler's limit %d (use the host path)", k, SK_MAX);
  hipStream_t s = static_cast<hipStream_t>(stream);
  void *scratch_v = nullptr, *params_v = nullptr;  // per-device operator workspace (tl_scratch)
  TL_TRY(tl_scratch(TL_SCRATCH_SAMPLE_PROBS, tl_sample_scratch_bytes(n), &scratch_v));
  TL_TRY(tl_scratch(TL_SCRATCH_SAMPLE_PARAMS, sizeof(TlSampleParams), &params_v));
  float* scratch = static_cast<float*>(scratch_v);
  TlSampleParams* params = static_cast<TlSampleParams*>(params_v);
  TlSampleParams h = {};
  h.temperature = temperature;
  h.top_k = top_k;
  h.top_p = top_p;
  h.use_fixed_u = 1;
  h.fixed_u = u;
  TL_HIP(hipMemcpyAsync(params, &h, sizeof(h), hipMemcpyHostToDevice, s));
  TL_HIP(hipStreamSynchronize(s));  // h lives on this stack frame
  return tl_launch_sample_topk(const_cast<float*>(logits_dev), n, scratch, nullptr, 0, 0, params, id_dev, cand_ids_dev,
                               cand_probs_dev, n_cand_dev, s);
}
