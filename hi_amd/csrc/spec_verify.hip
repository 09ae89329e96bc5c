// Greedy speculative-decoding verification on the device (the acceptance
// of crates/hi-cuda/src/gpu.rs:10725-10762,
// speculative_greedy_next_tokens_paged_with_page_table, batched over
// requests; the rule of docs/deepseek-v4-spec-decode-plan.md:95-102).
//
// The reference copies the K + 1 verify rows of logits to the host, takes
// each row's argmax there (gpu.rs:6406-6435: best = 0, best_val = row[0],
// replaced by a later value only when strictly greater -- so a NaN at
// index 0 keeps index 0, other NaNs never win, ties keep the lower index),
// accepts draft[i] while it equals greedy[i], and emits
// greedy[0 ..= accepted] (the first mismatch's target token, or the bonus
// token after a fully accepted draft).  Here the rows are split over
// workgroups (one workgroup a row left most of the chip idle), which merge
// their maxima in the caller's out_greedy, and one workgroup per request then
// runs the acceptance.  Calls with different outputs share nothing, whatever
// streams, threads or graphs they run on, and only the emitted tokens and
// their count leave the device.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "hi_rocm.h"
#include "sampler_internal.h"
#include "wave_ops.h"

namespace hi_rocm {
namespace {

// Order key of a non-NaN float with -0 taken as +0 (the reference's '>'
// does not tell them apart).
__device__ __forceinline__ uint32_t order_key0(float x) {
  if (x == 0.0f) x = 0.0f;
  const uint32_t b = __float_as_uint(x);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// A value and index as one key: the larger value, then the lower index.
// Keys reduce by max, so a result does not depend on the reduction order.
__device__ __forceinline__ uint64_t verify_key(float v, uint32_t i) {
  return ((uint64_t)order_key0(v) << 32) | (uint64_t)(0xffffffffu - i);
}
__device__ __forceinline__ float verify_value(uint64_t key) {
  const uint32_t o = (uint32_t)(key >> 32);
  return __uint_as_float((o & 0x80000000u) ? o ^ 0x80000000u : ~o);
}
__device__ __forceinline__ uint64_t verify_wave_max(uint64_t best) {
  #pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(best >> 32), o, 64);
    const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)best, o, 64);
    const uint64_t w = ((uint64_t)hi << 32) | lo;
    best = w > best ? w : best;
  }
  return best;
}

// The key of the first maximum above -inf of the row x in [i0, i0 + n) (0:
// none), by a workgroup of T threads: range-checked 16-byte loads,
// kVerifyLoads a thread in flight, from a buffer of the part's own (ranges
// and offsets count bytes in 32 bits).  ahead() is called behind the first
// ones.
constexpr int kVerifyLoads = 8;
template <int T>
constexpr int kVerifySpan = T * 4 * kVerifyLoads;  // logits of a step
template <int T, typename AheadF>
__device__ __forceinline__ uint64_t verify_span_max(const float* x, int64_t i0, int n, uint64_t* red, AheadF ahead) {
  const int tid = threadIdx.x;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(x + i0), 0, n * 4, kBufferConfig);
  float bv = -__builtin_inff();
  uint32_t bi = 0xffffffffu;
  for (int b = 0; b < n; b += kVerifySpan<T>) {
    i32x4_t v[kVerifyLoads];
    #pragma unroll
    for (int j = 0; j < kVerifyLoads; ++j)
      v[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, (b + (j * T + tid) * 4) * 4, 0, 0);
    if (b == 0) ahead();
    #pragma unroll
    for (int j = 0; j < kVerifyLoads; ++j) {
      #pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = b + (j * T + tid) * 4 + q;
        const float f = __int_as_float(v[j][q]);
        const bool take = f > bv && i < n;  // (NaN never; a thread's indices rise)
        bv = take ? f : bv;
        bi = take ? (uint32_t)i : bi;
      }
    }
  }
  uint64_t best = verify_wave_max(bi == 0xffffffffu ? 0ull : verify_key(bv, (uint32_t)i0 + bi));
  if ((tid & 63) == 0) red[tid >> 6] = best;
  __syncthreads();
  best = red[0];
  #pragma unroll
  for (int w = 1; w < T / 64; ++w) best = red[w] > best ? red[w] : best;
  return best;
}

// Makes key's index the row's answer unless the answer comes before it (the
// larger value, then the lower index).  Whatever the caller's array holds at
// the start is no more than one more index to compare with: one of the row's
// stands for its own logit, any other (or a NaN's) gives way.  An index once
// taken only gives way to an earlier one, so the loop ends after at most one
// round per other part, and the result does not depend on their order.
// `cur`: the answer seen last.
__device__ __forceinline__ void verify_take(const float* x, int V, uint64_t key, uint32_t cur, float xc,
                                            uint32_t* answer) {
  const float bv = verify_value(key);
  const uint32_t bi = 0xffffffffu - (uint32_t)key;
  while (true) {
    if (xc > bv || (xc == bv && cur <= bi)) return;
    if (__hip_atomic_compare_exchange_strong(answer, &cur, bi, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT))
      return;
    xc = cur < (uint32_t)V ? x[cur] : -__builtin_inff();
  }
}

// Part blockIdx.x % n_parts (of `span` logits) of verify row blockIdx.x /
// n_parts.
template <int T>
__global__ void __launch_bounds__(T)
    verify_part_kernel(const float* logits, int V, int span, int n_parts, uint32_t* greedy) {
  __shared__ uint64_t red[T / 64];
  const uint32_t r = blockIdx.x / (uint32_t)n_parts;
  const int64_t i0 = (int64_t)(blockIdx.x % (uint32_t)n_parts) * span;
  const float* x = logits + (int64_t)r * V;
  uint32_t cur = 0u;
  if (threadIdx.x == 0) cur = __hip_atomic_load(greedy + r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  float xc = -__builtin_inff();
  const uint64_t best = verify_span_max<T>(x, i0, (int)min((int64_t)span, V - i0), red, [&]() {
    if (cur < (uint32_t)V && threadIdx.x == 0) xc = x[cur];
  });
  if (threadIdx.x == 0 && best != 0ull) verify_take(x, V, best, cur, xc, greedy + r);
}

constexpr int kAcceptThreads = 256;
// One workgroup per request: its rows' answers (index 0 with a NaN there, or
// when nothing is above -inf), the accepted prefix and the emitted tokens.
__global__ void __launch_bounds__(kAcceptThreads)
    verify_accept_kernel(const float* logits, int V, uint32_t* greedy, const uint32_t* draft, const int32_t* draft_len,
                         int K, uint32_t* out_tokens, int32_t* out_count) {
  __shared__ int accepted;
  const int b = blockIdx.x, tid = threadIdx.x;
  const int64_t r0 = (int64_t)b * (K + 1);
  const int k = draft_len ? min(max(draft_len[b], 0), K) : K;
  if (tid == 0) accepted = k;
  __syncthreads();
  for (int i = tid; i <= K; i += kAcceptThreads) {
    const float* x = logits + (r0 + i) * V;
    uint32_t g = greedy[r0 + i];
    const float x0 = x[0], xg = g < (uint32_t)V ? x[g] : -__builtin_inff();
    if (x0 != x0 || !(xg > -__builtin_inff())) greedy[r0 + i] = g = 0u;
    if (i < k && draft[(int64_t)b * K + i] != g) atomicMin(&accepted, i);
  }
  __syncthreads();
  const int n = accepted;
  for (int i = tid; i <= n; i += kAcceptThreads) out_tokens[r0 + i] = greedy[r0 + i];
  if (tid == 0) out_count[b] = n + 1;
}

// Parts of a row: steps of kVerifySpan logits, at most 64.  Rows of one step
// of 256 threads take such workgroups, longer ones steps of 1024: the parts
// of a row exchange through the memory behind the chip's L2s, about 5 ns an
// exchange on one cache line, so larger parts win from the first row that is
// split (40 rows of 151,936: 10.3 us, in parts of 256 threads 15.6, in one
// workgroup a row 12.7; 264 rows: 33, 42 and 40; 4096 rows of 4096: 14.4
// with 256 threads, 34 with 1024).  One workgroup of 1024 threads a row, with
// one load a thread in flight, took 62 us for the 40 rows.  A grid holds less
// than 2^32 work-items, so many rows take fewer parts.  (Inputs that change
// from call to call; answers that the array already holds exchange nothing.)
constexpr int kVerifyMaxParts = 64;

template <int T>
void launch_parts(const float* x, int64_t rows, int V, uint32_t* greedy, hipStream_t st) {
  constexpr int64_t kMaxGroups = (((int64_t)1 << 32) - 1) / T;
  const int64_t steps = ((int64_t)V + kVerifySpan<T> - 1) / kVerifySpan<T>;
  const int64_t most = std::min<int64_t>(kVerifyMaxParts, std::max<int64_t>(1, kMaxGroups / rows));
  // (2^28 logits are 2^30 bytes; with 64 parts a row's part is at most 2^25)
  const int span = (int)std::min<int64_t>(kVerifySpan<T> * ((steps + most - 1) / most), 1 << 28);
  const int n_parts = (int)((V + (int64_t)span - 1) / span);
  hipLaunchKernelGGL((verify_part_kernel<T>), dim3((unsigned)(rows * n_parts)), dim3(T), 0, st, x, V, span, n_parts,
                     greedy);
}

}  // namespace
}  // namespace hi_rocm

extern "C" int hi_rocm_spec_verify_greedy(const void* logits, int batch, int max_draft, int vocab,
                                          const void* draft_tokens, const void* draft_len, void* out_greedy,
                                          void* out_tokens, void* out_count, void* stream) {
  if (logits == nullptr || batch <= 0 || max_draft < 0 || vocab <= 0 || (max_draft > 0 && draft_tokens == nullptr) ||
      out_greedy == nullptr || out_tokens == nullptr || out_count == nullptr || stream == nullptr)
    return hi_rocm::api_fail(HI_ROCM_ERR_ARGS, "hi_rocm_spec_verify_greedy: invalid arguments");
  const int64_t rows = (int64_t)batch * (max_draft + 1);
  if (rows > INT32_MAX) return hi_rocm::api_fail(HI_ROCM_ERR_UNSUPPORTED, "hi_rocm_spec_verify_greedy: too many rows");
  hipStream_t st = (hipStream_t)stream;
  namespace hr = hi_rocm;
  const float* x = (const float*)logits;
  uint32_t* greedy = (uint32_t*)out_greedy;
  if (vocab <= hr::kVerifySpan<256>)
    hr::launch_parts<256>(x, rows, vocab, greedy, st);
  else
    hr::launch_parts<1024>(x, rows, vocab, greedy, st);
  hipLaunchKernelGGL(hr::verify_accept_kernel, dim3((unsigned)batch), dim3(hr::kAcceptThreads), 0, st, x, vocab, greedy,
                     (const uint32_t*)draft_tokens, (const int32_t*)draft_len, max_draft, (uint32_t*)out_tokens,
                     (int32_t*)out_count);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? HI_ROCM_OK : hr::api_hip_fail(e, "spec verify launch");
}
