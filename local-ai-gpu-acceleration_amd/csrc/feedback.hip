// Greedy token selection and the reference runner's RMSNorm/SiLU feedback
// family (decode_kernels.cu:122-289, 2993-3073).
//
// Feedback kernels: the reference recomputes sum(logits^2) in every thread
// (O(rows * cols)); here each 1024-thread workgroup reduces it once and then
// writes 1024 outputs, so the cost is O(rows * cols / 1024).
#include "argmax.cuh"
#include "common.h"
#include "internal.h"
#include "rtxllm/decode_kernels.h"

namespace rtxllm {
namespace {

constexpr int kFbThreads = 1024;

// 1 / sqrt(mean(logits^2) + eps) by one kFbThreads workgroup. Each workgroup of
// the launch reads all the logits, so the time is the latency of that read: four
// 16-byte loads a thread and step (values outside the 16-byte vectors one by
// one). The launch over 8192 logits and 4096 outputs 4.1 -> 2.7 us against 4-byte
// loads and a serial sum of the waves.
__device__ float inv_rms(const float* __restrict__ logits, std::uint32_t rows, float eps, float* sh) {
  const std::uint32_t tid = threadIdx.x;
  const std::uint32_t to16 =
      static_cast<std::uint32_t>((16u - (reinterpret_cast<std::uintptr_t>(logits) & 15u)) & 15u) / 4u;
  const std::uint32_t head = to16 < rows ? to16 : rows, nv = (rows - head) / 4u, tail0 = head + 4u * nv;
  const float4* const vec = reinterpret_cast<const float4*>(logits + head);
  const std::uint32_t edges = head + (rows - tail0);  // at most six values
  const float e = tid < edges ? logits[tid < head ? tid : tail0 + (tid - head)] : 0.0f;
  float s = e * e;
  for (std::uint32_t i0 = tid; i0 < nv; i0 += 4u * kFbThreads) {
    float4 v[4];
#pragma unroll
    for (std::uint32_t j = 0; j < 4u; ++j) {
      const std::uint32_t i = i0 + kFbThreads * j;
      v[j] = vec[i < nv ? i : nv - 1u];
    }
#pragma unroll
    for (std::uint32_t j = 0; j < 4u; ++j) {
      const float q = fmaf(v[j].w, v[j].w, fmaf(v[j].z, v[j].z, fmaf(v[j].y, v[j].y, v[j].x * v[j].x)));
      s += i0 + kFbThreads * j < nv ? q : 0.0f;
    }
  }
  s = wave_sum(s);
  if ((tid & 63u) == 0u) sh[tid >> 6] = s;
  __syncthreads();
  float total = sh[0];
#pragma unroll
  for (int i = 1; i < kFbThreads / 64; ++i) total += sh[i];
  return rsqrtf(total / static_cast<float>(rows) + eps);
}

__device__ __forceinline__ float silu(float v) {
  const float sig = 1.0f / (1.0f + expf(-v));
  return v * sig;
}

enum FbMode : int {
  kRmsnorm = 0,          // act = n
  kSiluRmsnorm = 1,      // act = silu(n)
  kWithSiluCache = 2,    // act = n, cache = silu(n)
  kGatedSilu = 3,        // act = cache[c % cache_cols] * n
  kSiluCache = 4,        // cache (+)= silu(n)
  kCache = 5,            // cache (+)= n
  kCacheGatedProduct = 6 // up (+)= n; act = gate * up
};

template <int MODE>
__global__ __launch_bounds__(kFbThreads) void feedback_kernel(const float* __restrict__ logits, const float* gate,
                                                              float* cache, float* act, std::uint32_t rows,
                                                              std::uint32_t cache_cols, std::uint32_t cols,
                                                              float eps, std::uint32_t accumulate) {
  __shared__ float sh[kFbThreads / 64];
  if (rows == 0u) return;
  if ((MODE == kGatedSilu || MODE == kCacheGatedProduct) && cache_cols == 0u) return;
  const std::uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  const float own = logits[c % rows];  // ahead of the sum
  const float inv = inv_rms(logits, rows, eps, sh);
  if (c >= cols) return;
  const float n = own * inv;
  if constexpr (MODE == kRmsnorm) {
    act[c] = n;
  } else if constexpr (MODE == kSiluRmsnorm) {
    act[c] = silu(n);
  } else if constexpr (MODE == kWithSiluCache) {
    act[c] = n;
    cache[c] = silu(n);
  } else if constexpr (MODE == kGatedSilu) {
    act[c] = gate[c % cache_cols] * n;
  } else if constexpr (MODE == kSiluCache) {
    const float v = silu(n);
    cache[c] = accumulate != 0u ? cache[c] + v : v;
  } else if constexpr (MODE == kCache) {
    cache[c] = accumulate != 0u ? cache[c] + n : n;
  } else {
    const float u = accumulate != 0u ? cache[c] + n : n;
    cache[c] = u;
    act[c] = gate[c] * u;
  }
}

template <int MODE>
hipError_t launch_feedback(const float* logits, const float* gate, float* cache, float* act, std::uint32_t rows,
                           std::uint32_t cache_cols, std::uint32_t cols, float eps, std::uint32_t accumulate,
                           hipStream_t stream) {
  // A zero-column launch is an invalid configuration, as the reference's
  // <<<ceil(cols / 256), 256>>> launch would report.
  if (cols == 0u) return hipErrorInvalidConfiguration;
  const dim3 grid((cols + kFbThreads - 1) / kFbThreads);
  hipLaunchKernelGGL(feedback_kernel<MODE>, grid, dim3(kFbThreads), 0, stream, logits, gate, cache, act, rows,
                     cache_cols, cols, eps, accumulate);
  return hipGetLastError();
}

// ---- argmax ---------------------------------------------------------------

// One workgroup per call (argmax.cuh: why, and the rules for ties and NaN).
__global__ __launch_bounds__(kArgmaxThreads) void argmax_token_kernel(const float* __restrict__ logits,
                                                                      std::uint32_t* token, std::uint32_t rows,
                                                                      int mode, std::uint32_t vocab,
                                                                      std::uint32_t offset) {
  const std::uint32_t before = (threadIdx.x == 0u && mode == 0) ? token[0] : 0u;  // read ahead of the scan
  const std::uint32_t bi = argmax_row(logits, rows);
  if (threadIdx.x == 0u) token[0] = mode == 0 ? (bi + before + 1u) % 32000u : (bi + offset) % vocab;
}

}  // namespace

hipError_t launch_argmax_token(const float* logits, std::uint32_t* token, std::uint32_t rows, int mode,
                               std::uint32_t vocab, std::uint32_t offset, hipStream_t stream) {
  hipLaunchKernelGGL(argmax_token_kernel, dim3(1), dim3(kArgmaxThreads), 0, stream, logits, token, rows, mode, vocab,
                     offset);
  return hipGetLastError();
}

}  // namespace rtxllm

using namespace rtxllm;

extern "C" hipError_t rtxllm_launch_rmsnorm_feedback(const float* logits, float* activation, std::uint32_t rows,
                                                     std::uint32_t cols, float epsilon, hipStream_t stream) {
  return launch_feedback<kRmsnorm>(logits, nullptr, nullptr, activation, rows, 0u, cols, epsilon, 0u, stream);
}

extern "C" hipError_t rtxllm_launch_silu_rmsnorm_feedback(const float* logits, float* activation,
                                                          std::uint32_t rows, std::uint32_t cols, float epsilon,
                                                          hipStream_t stream) {
  return launch_feedback<kSiluRmsnorm>(logits, nullptr, nullptr, activation, rows, 0u, cols, epsilon, 0u, stream);
}

extern "C" hipError_t rtxllm_launch_rmsnorm_feedback_with_silu_cache(const float* logits, float* activation,
                                                                     float* silu_cache, std::uint32_t rows,
                                                                     std::uint32_t cols, float epsilon,
                                                                     hipStream_t stream) {
  return launch_feedback<kWithSiluCache>(logits, nullptr, silu_cache, activation, rows, 0u, cols, epsilon, 0u,
                                         stream);
}

extern "C" hipError_t rtxllm_launch_gated_silu_rmsnorm_feedback(const float* logits, const float* silu_cache,
                                                                float* activation, std::uint32_t rows,
                                                                std::uint32_t cache_cols, std::uint32_t cols,
                                                                float epsilon, hipStream_t stream) {
  return launch_feedback<kGatedSilu>(logits, silu_cache, nullptr, activation, rows, cache_cols, cols, epsilon, 0u,
                                     stream);
}

extern "C" hipError_t rtxllm_launch_rmsnorm_silu_cache(const float* logits, float* silu_cache, std::uint32_t rows,
                                                       std::uint32_t cache_cols, float epsilon,
                                                       std::uint32_t accumulate, hipStream_t stream) {
  if (cache_cols == 0u) return hipErrorInvalidValue;
  return launch_feedback<kSiluCache>(logits, nullptr, silu_cache, nullptr, rows, cache_cols, cache_cols, epsilon,
                                     accumulate, stream);
}

extern "C" hipError_t rtxllm_launch_rmsnorm_cache(const float* logits, float* cache, std::uint32_t rows,
                                                  std::uint32_t cache_cols, float epsilon, std::uint32_t accumulate,
                                                  hipStream_t stream) {
  if (cache_cols == 0u) return hipErrorInvalidValue;
  return launch_feedback<kCache>(logits, nullptr, cache, nullptr, rows, cache_cols, cache_cols, epsilon,
                                 accumulate, stream);
}

extern "C" hipError_t rtxllm_launch_rmsnorm_cache_and_gated_product(const float* logits, const float* gate_cache,
                                                                    float* up_cache, float* activation,
                                                                    std::uint32_t rows, std::uint32_t cache_cols,
                                                                    std::uint32_t output_cols, float epsilon,
                                                                    std::uint32_t accumulate, hipStream_t stream) {
  if (cache_cols == 0u || output_cols == 0u) return hipErrorInvalidValue;
  return launch_feedback<kCacheGatedProduct>(logits, gate_cache, up_cache, activation, rows, cache_cols,
                                             output_cols, epsilon, accumulate, stream);
}

extern "C" hipError_t rtxllm_launch_output_token_sample(const float* logits, std::uint32_t* token,
                                                        std::uint32_t rows, std::uint32_t vocab_size,
                                                        std::uint32_t token_offset, hipStream_t stream) {
  if (logits == nullptr || token == nullptr || rows == 0u || vocab_size == 0u) return hipErrorInvalidValue;
  return launch_argmax_token(logits, token, rows, 1, vocab_size, token_offset, stream);
}
