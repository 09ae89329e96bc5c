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
// workgroups (one workgroup a row left most of the chip idle), and one
// workgroup per request then merges its rows' parts and runs the acceptance,
// so only the emitted tokens and their count leave the device.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>

#include "hi_rocm.h"
#include "sampler_internal.h"
#include "wave_ops.h"

namespace hi_rocm {
namespace {

constexpr int kVerifyThreads = 256;

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

// The key of the row's first maximum above -inf in [i0, i1) (0: none), by a
// workgroup of kVerifyThreads: range-checked 16-byte loads, kVerifyLoads a
// thread in flight.
constexpr int kVerifyLoads = 8;
constexpr int kVerifySpan = kVerifyThreads * 4 * kVerifyLoads;  // logits of a step
__device__ __forceinline__ uint64_t verify_span_max(const float* x, int V, int i0, int i1, uint64_t* red) {
  const int tid = threadIdx.x;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, V * 4, kBufferConfig);
  float bv = -__builtin_inff();
  uint32_t bi = 0xffffffffu;
  for (int b = i0; b < i1; b += kVerifySpan) {
    i32x4_t v[kVerifyLoads];
    #pragma unroll
    for (int j = 0; j < kVerifyLoads; ++j)
      v[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, (b + (j * kVerifyThreads + tid) * 4) * 4, 0, 0);
    #pragma unroll
    for (int j = 0; j < kVerifyLoads; ++j) {
      #pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = b + (j * kVerifyThreads + tid) * 4 + q;
        const float f = __int_as_float(v[j][q]);
        const bool take = f > bv && i < V;  // (NaN never; a thread's indices rise)
        bv = take ? f : bv;
        bi = take ? (uint32_t)i : bi;
      }
    }
  }
  uint64_t best = verify_wave_max(bi == 0xffffffffu ? 0ull : verify_key(bv, bi));
  if ((tid & 63) == 0) red[tid >> 6] = best;
  __syncthreads();
  best = red[0];
  #pragma unroll
  for (int w = 1; w < kVerifyThreads / 64; ++w) best = red[w] > best ? red[w] : best;
  return best;
}

// The row's answer from its key: index 0 with a NaN there, or when nothing
// is above -inf.
__device__ __forceinline__ uint32_t verify_index(uint64_t best, float x0) {
  return x0 != x0 || best == 0ull ? 0u : 0xffffffffu - (uint32_t)best;
}

// The key of part `blockIdx.x` (of `span` logits) of verify row blockIdx.y.
__global__ void __launch_bounds__(kVerifyThreads)
    verify_part_kernel(const float* logits, int V, int span, uint64_t* parts) {
  __shared__ uint64_t red[kVerifyThreads / 64];
  const int64_t r = blockIdx.y;
  const int i0 = (int)blockIdx.x * span;
  const uint64_t best = verify_span_max(logits + r * V, V, i0, min(i0 + span, V), red);
  if (threadIdx.x == 0) parts[r * gridDim.x + blockIdx.x] = best;
}

// greedy[r] by one workgroup a row, for a call that cannot have the parts'
// buffer.
__global__ void __launch_bounds__(kVerifyThreads) verify_argmax_kernel(const float* logits, int V, uint32_t* greedy) {
  __shared__ uint64_t red[kVerifyThreads / 64];
  const float* x = logits + (int64_t)blockIdx.x * V;
  const uint64_t best = verify_span_max(x, V, 0, V, red);
  if (threadIdx.x == 0) greedy[blockIdx.x] = verify_index(best, x[0]);
}

// One workgroup per request: its rows' greedy tokens from their parts (a
// wave a row, n_parts <= 64; null: greedy holds them already), the accepted
// prefix and the emitted tokens.
__global__ void __launch_bounds__(kVerifyThreads)
    verify_accept_kernel(const float* logits, int V, const uint64_t* parts, int n_parts, uint32_t* greedy,
                         const uint32_t* draft, const int32_t* draft_len, int K, uint32_t* out_tokens,
                         int32_t* out_count) {
  __shared__ int accepted;
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int64_t r0 = (int64_t)b * (K + 1);
  const int k = draft_len ? min(max(draft_len[b], 0), K) : K;
  if (tid == 0) accepted = k;
  if (parts) {
    for (int i = tid >> 6; i <= K; i += kVerifyThreads / 64) {
      const float x0 = logits[(r0 + i) * V];
      const uint64_t best = verify_wave_max(lane < n_parts ? parts[(r0 + i) * n_parts + lane] : 0ull);
      if (lane == 0) greedy[r0 + i] = verify_index(best, x0);
    }
  }
  __syncthreads();
  for (int i = tid; i < k; i += kVerifyThreads)
    if (draft[(int64_t)b * K + i] != greedy[r0 + i]) atomicMin(&accepted, i);
  __syncthreads();
  const int n = accepted;
  for (int i = tid; i <= n; i += kVerifyThreads) out_tokens[r0 + i] = greedy[r0 + i];
  if (tid == 0) out_count[b] = n + 1;
}

// Parts of a row: steps of kVerifySpan logits, at most 64 (a wave merges
// them).  One step a workgroup fills the chip from a few rows on (40 rows of
// 151,936: 760 workgroups, 61.7 -> 9.0 us).
constexpr int kVerifyMaxParts = 64;
std::mutex g_verify_mutex;  // both launches of a call on a stream's buffer, together

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
  const int steps = (vocab + hr::kVerifySpan - 1) / hr::kVerifySpan;
  const int span = hr::kVerifySpan * ((steps + hr::kVerifyMaxParts - 1) / hr::kVerifyMaxParts);
  const int n_parts = (vocab + span - 1) / span;
  const float* x = (const float*)logits;
  uint32_t* greedy = (uint32_t*)out_greedy;
  std::lock_guard<std::mutex> lock(hr::g_verify_mutex);
  // the stream's buffer for the parts; none while a capture would have to
  // allocate it, or beyond a grid's rows: then one workgroup a row
  void* ws = nullptr;
  if (rows <= 65535) {
    const int rc = hr::api_stream_buffer(hr::kWsVerify, (size_t)rows * n_parts * sizeof(uint64_t), 0, true, st, &ws);
    if (rc != HI_ROCM_OK) return rc;
  }
  if (ws)
    hipLaunchKernelGGL(hr::verify_part_kernel, dim3((unsigned)n_parts, (unsigned)rows), dim3(hr::kVerifyThreads), 0, st,
                       x, vocab, span, (uint64_t*)ws);
  else
    hipLaunchKernelGGL(hr::verify_argmax_kernel, dim3((unsigned)rows), dim3(hr::kVerifyThreads), 0, st, x, vocab, greedy);
  hipLaunchKernelGGL(hr::verify_accept_kernel, dim3((unsigned)batch), dim3(hr::kVerifyThreads), 0, st, x, vocab,
                     (const uint64_t*)ws, n_parts, greedy, (const uint32_t*)draft_tokens, (const int32_t*)draft_len,
                     max_draft, (uint32_t*)out_tokens, (int32_t*)out_count);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? HI_ROCM_OK : hr::api_hip_fail(e, "spec verify launch");
}
