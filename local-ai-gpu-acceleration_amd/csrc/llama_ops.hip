// Standalone C-ABI entry points for the Llama layer math that the decode runner
// otherwise fuses into its matvec epilogues: weighted RMSNorm, rotary embedding
// with a theta schedule, SiLU-gate multiply, the Q5_K embedding gather, GQA
// decode attention over a paged fp16 KV cache and greedy argmax. Each is one or
// two kernel launches on the caller's stream with caller-owned device memory
// (no allocation, no synchronisation: capture-safe).
//
// The reference runtime composes its per-stage math from separate launchers
// (rtxllm_launch_rmsnorm_feedback / output_token_sample etc.,
// runtime/kernels/decode/decode_kernels.h:38-101, 319-325, called per stage
// from launch_feedback, mixed_sequence_benchmark_runner/main.cpp:4073-4279);
// these entry points are the Llama-layer counterparts of that style. Formulas:
// weighted RMSNorm (x * inv_rms) * w with inv_rms = 1 / sqrt(mean(x^2) + eps)
// (main.cpp:1363-1382 plus the weight), rotary pairs (e c - o s, e s + o c)
// (decode_kernels.cu:327-343) at angle pos * theta^(-2i/d), silu(v) = v / (1 +
// exp(-v)) (main.cpp:1435-1503), Q5_K dequant (main.cpp:1231-1259), argmax with
// the lowest index among maxima (decode_kernels.cu:2993-3031).
#include "argmax.cuh"
#include "dequant.cuh"
#include "layer.h"
#include "layer_common.cuh"
#include "rtxllm/decode_kernels.h"

namespace rtxllm {
namespace {

constexpr std::uint32_t kOpThreads = 256;

__device__ float block_sum256(float v, float* sh) {
  v = wave_sum(v);
  const std::uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  if (lane == 0u) sh[wave] = v;
  __syncthreads();
  const float s = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return s;
}

// One workgroup of T threads per vector r of x [count][n], the vector held in
// registers: V 16-byte loads a thread (n <= 4 T V), so it is read once, and the
// weights are read ahead of the reduction. x, w and out 16-byte aligned, n % 4
// == 0; in place allowed (a thread writes what it alone read). Against the
// scalar two-pass kernel below (16 dependent loads, twice): one vector of 4096
// 7.1 -> 2.3 us, 256 of them 8.0 -> 3.3 us.
template <std::uint32_t T, std::uint32_t V>
__global__ __launch_bounds__(T) void rmsnorm_w_vec_kernel(const float* x, const float* __restrict__ w, std::uint32_t n,
                                                          float eps, float* out) {
  __shared__ float sh[T / 64u];
  const std::uint32_t n4 = n / 4u;
  const std::size_t base = static_cast<std::size_t>(blockIdx.x) * n4;
  float4 v[V], wv[V];
#pragma unroll
  for (std::uint32_t j = 0; j < V; ++j) {
    const std::uint32_t i = threadIdx.x + T * j, c = i < n4 ? i : n4 - 1u;  // past the end: read again, not summed
    v[j] = reinterpret_cast<const float4*>(x)[base + c];
    wv[j] = w != nullptr ? reinterpret_cast<const float4*>(w)[c] : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
  }
  float s = 0.0f;
#pragma unroll
  for (std::uint32_t j = 0; j < V; ++j) {
    const float t = fmaf(v[j].w, v[j].w, fmaf(v[j].z, v[j].z, fmaf(v[j].y, v[j].y, v[j].x * v[j].x)));
    s += threadIdx.x + T * j < n4 ? t : 0.0f;
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63u) == 0u) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  float total = sh[0];
#pragma unroll
  for (std::uint32_t k = 1; k < T / 64u; ++k) total += sh[k];
  const float inv = 1.0f / sqrtf(total / static_cast<float>(n) + eps);
#pragma unroll
  for (std::uint32_t j = 0; j < V; ++j) {
    const std::uint32_t i = threadIdx.x + T * j;
    if (i < n4)  // times 1 without a weight: exact
      reinterpret_cast<float4*>(out)[base + i] = make_float4(v[j].x * inv * wv[j].x, v[j].y * inv * wv[j].y,
                                                             v[j].z * inv * wv[j].z, v[j].w * inv * wv[j].w);
  }
}

// The rest: unaligned pointers, n % 4 != 0, vectors under 128 or over 16384 values.
__global__ __launch_bounds__(kOpThreads) void rmsnorm_w_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                               std::uint32_t n, float eps, float* __restrict__ out) {
  __shared__ float sh[kOpThreads / 64];
  const std::size_t base = static_cast<std::size_t>(blockIdx.x) * n;
  float s = 0.0f;
  for (std::uint32_t i = threadIdx.x; i < n; i += kOpThreads) {
    const float v = x[base + i];
    s = fmaf(v, v, s);
  }
  const float inv = 1.0f / sqrtf(block_sum256(s, sh) / static_cast<float>(n) + eps);
  for (std::uint32_t i = threadIdx.x; i < n; i += kOpThreads) {
    const float v = x[base + i] * inv;
    out[base + i] = w != nullptr ? v * w[i] : v;
  }
}

// (cos, sin) of pair i of a head at position pos: inv_freq = theta^(-2i/d) in
// double, rounded once, and the angle (float)pos * inv_freq in fp32, as the
// textbook rotary is evaluated; (cos, sin) of that fp32 angle in double, each
// rounded once.
__device__ __forceinline__ float2 rope_cos_sin(std::uint32_t i, std::uint32_t head_dim, double theta,
                                               std::uint32_t pos) {
  const float inv_freq = static_cast<float>(pow(theta, -2.0 * static_cast<double>(i) / static_cast<double>(head_dim)));
  const double angle = static_cast<double>(static_cast<float>(pos) * inv_freq);
  return make_float2(static_cast<float>(cos(angle)), static_cast<float>(sin(angle)));
}

// Workgroup (chunk of kOpThreads P pairs, vector r = blockIdx.y): the head_dim / 2
// angles of the vector once, into LDS, then P pairs a thread, whose loads were
// issued before. Against one double pow, cos and sin per pair of every head:
// 256 vectors of 32 heads of 128 8.0 -> 4.1 us (where it pays: rope_shared_pairs).
constexpr std::uint32_t kRopeMaxHalf = 1024;  // head_dim / 2 at most
template <std::uint32_t P>
__global__ __launch_bounds__(kOpThreads) void rope_theta_kernel(float* __restrict__ vec, std::uint32_t pairs,
                                                                std::uint32_t head_dim, double theta,
                                                                const std::uint32_t* __restrict__ pos) {
  __shared__ float2 cs[kRopeMaxHalf];
  const std::uint32_t r = blockIdx.y, half = head_dim / 2u, p0 = blockIdx.x * kOpThreads * P + threadIdx.x;
  float2* v = reinterpret_cast<float2*>(vec + static_cast<std::size_t>(r) * 2u * pairs);
  const std::uint32_t at = pos[r];
  float2 eo[P];
#pragma unroll
  for (std::uint32_t j = 0; j < P; ++j) {
    const std::uint32_t p = p0 + kOpThreads * j;
    eo[j] = v[p < pairs ? p : pairs - 1u];
  }
  for (std::uint32_t i = threadIdx.x; i < half; i += kOpThreads) cs[i] = rope_cos_sin(i, head_dim, theta, at);
  __syncthreads();
#pragma unroll
  for (std::uint32_t j = 0; j < P; ++j) {
    const std::uint32_t p = p0 + kOpThreads * j;
    if (p >= pairs) return;
    const float2 t = cs[p % half];
    v[p] = make_float2(eo[j].x * t.x - eo[j].y * t.y, eo[j].x * t.y + eo[j].y * t.x);
  }
}

// One thread per pair, its own angle.
__global__ __launch_bounds__(kOpThreads) void rope_theta_pair_kernel(float* __restrict__ vec, std::uint32_t pairs,
                                                                     std::uint32_t head_dim, double theta,
                                                                     const std::uint32_t* __restrict__ pos) {
  const std::uint32_t p = blockIdx.x * kOpThreads + threadIdx.x;
  if (p >= pairs) return;
  const std::uint32_t r = blockIdx.y;
  const float2 t = rope_cos_sin(p % (head_dim / 2u), head_dim, theta, pos[r]);
  float2* v = reinterpret_cast<float2*>(vec + static_cast<std::size_t>(r) * 2u * pairs) + p;
  const float2 eo = *v;
  *v = make_float2(eo.x * t.x - eo.y * t.y, eo.x * t.y + eo.y * t.x);
}

__global__ __launch_bounds__(kOpThreads) void silu_mul_kernel(const float* __restrict__ gate, const float* __restrict__ up,
                                                              std::size_t n, float* __restrict__ out) {
  const std::size_t i = static_cast<std::size_t>(blockIdx.x) * kOpThreads + threadIdx.x;
  if (i < n) out[i] = silu(gate[i]) * up[i];
}

// Four values a thread where the three pointers are 16-byte aligned; the last
// n % 4 values one each by the first threads past the vectors. 14336 values 4.6 ->
// 2.1 us against one value a thread; 256 x 14336 9.0 -> 8.0 us (44 MB: 5.5 TB/s;
// a 1 GiB copy reaches 5.15).
__global__ __launch_bounds__(kOpThreads) void silu_mul_vec_kernel(const float* gate, const float* up, std::size_t n,
                                                                  float* out) {
  const std::size_t i = static_cast<std::size_t>(blockIdx.x) * kOpThreads + threadIdx.x, n4 = n / 4u;
  if (i < n4) {
    const float4 g = reinterpret_cast<const float4*>(gate)[i], u = reinterpret_cast<const float4*>(up)[i];
    reinterpret_cast<float4*>(out)[i] =
        make_float4(silu(g.x) * u.x, silu(g.y) * u.y, silu(g.z) * u.z, silu(g.w) * u.w);
  } else if (i < n4 + (n & 3u)) {
    const std::size_t k = 4u * n4 + (i - n4);
    out[k] = silu(gate[k]) * up[k];
  }
}

// Workgroup (four blocks of the row, token t): a wave expands one block, four
// values a lane (dequant.cuh), and stores 16 bytes a lane at any 4-byte
// alignment of out. The time is two dependent reads (token, block); against
// a value a thread, each decoding the head, one row of 4096 4.7 -> 1.9 us, 256
// rows 5.1 -> 3.2 us.
__global__ __launch_bounds__(256) void embed_gather_q5k_kernel(const std::uint8_t* __restrict__ table,
                                                               std::uint32_t vocab, std::uint32_t cols,
                                                               const std::uint32_t* __restrict__ tokens,
                                                               float* __restrict__ out) {
  const std::uint32_t b = 4u * blockIdx.x + (threadIdx.x >> 6), t = blockIdx.y, bpr = cols / 256u;
  const std::uint32_t lane = threadIdx.x & 63u;
  if (b >= bpr) return;
  const std::uint32_t tok = tokens[t];
  const float nan = __builtin_nanf("");
  f32x4_any v = {nan, nan, nan, nan};  // no such row: a loud NaN row instead of a silent clamp
  if (tok < vocab) {
    const std::uint8_t* blk = table + (static_cast<std::size_t>(tok) * bpr + b) * 176u;
    const float4 x = run4_values<RTXLLM_FMT_Q5K>(run4_load<RTXLLM_FMT_Q5K>(blk, nullptr, lane), lane);
    v = f32x4_any{x.x, x.y, x.z, x.w};
  }
  *reinterpret_cast<f32x4_any*>(out + static_cast<std::size_t>(t) * cols + 256u * b + 4u * lane) = v;
}

// One workgroup per vector (argmax.cuh).
__global__ __launch_bounds__(kArgmaxThreads) void argmax_rows_kernel(const float* __restrict__ x, std::uint32_t n,
                                                                     std::uint32_t* __restrict__ index) {
  const std::uint32_t i = argmax_row(x + static_cast<std::size_t>(blockIdx.x) * n, n);
  if (threadIdx.x == 0u) index[blockIdx.x] = i;
}

// Pairs a thread of the shared-angle rotary kernel, or 0: one thread per pair. A
// few double evaluations more or less don't show in a launch of 3 us: sharing pays
// from where it saves one for every lane of the chip's 1024 SIMDs; short of that
// its LDS pass and barrier cost 1 to 10 % (us of own / shared angles, heads x head_dim, vectors: 32x128
// x256 8.0 / 4.1, x64 3.7 / 3.4, x32 3.0 / 3.1; 8x32 x64 3.0 / 3.3; 2x2048 x48
// 3.6 / 7.7). Heads of more than 512 values, whose threads evaluate several
// angles in turn, need half as much again (4x1024 x64 3.7 / 4.3, x128 5.1 /
// 4.5). Vectors of up to 128 pairs leave most of a workgroup's threads idle
// (1x256 x2048 5.2 / 6.6). Below 64 vectors one pair a thread spreads the loads
// over more workgroups (32x128 x48: one 3.1, four 3.4).
std::uint32_t rope_shared_pairs(std::uint32_t pairs, std::uint32_t half, std::uint32_t count) {
  if (half > kRopeMaxHalf || pairs <= 128u) return 0u;
  const std::uint32_t per = half > kOpThreads || count >= 64u ? 4u : 1u;
  const std::uint64_t chunks = (pairs + kOpThreads * per - 1u) / (kOpThreads * per);
  const std::uint64_t own = static_cast<std::uint64_t>(pairs) * count, shared = chunks * half * count;
  constexpr std::uint64_t kLanes = 1024u * 64u;
  return own > shared + (half > kOpThreads ? kLanes + kLanes / 2u : kLanes) ? per : 0u;
}

bool group_ok(std::uint32_t n_heads, std::uint32_t n_kv) {
  if (n_kv == 0u || n_heads == 0u || n_heads % n_kv != 0u) return false;
  const std::uint32_t g = n_heads / n_kv;
  return g == 1u || g == 2u || g == 4u || g == 8u;
}

std::size_t align256(std::size_t b) { return (b + 255u) & ~std::size_t{255}; }

}  // namespace
}  // namespace rtxllm

using namespace rtxllm;

extern "C" hipError_t rtxllm_rmsnorm_w(const float* x, const float* weight, uint32_t n, uint32_t count, float eps,
                                       float* out, hipStream_t stream) {
  if (x == nullptr || out == nullptr || n == 0u || count == 0u || count > 65535u * 1024u || !(eps >= 0.0f))
    return hipErrorInvalidValue;
  // (a launch holds fewer than 2^32 threads: more than 2^22 - 1 vectors wider than
  // 4096 stay with the 256-thread kernel)
  // (and vectors of less than half a wave's loads, which gain nothing: 16384 of 64
  // 6.6 us scalar, 7.0 vector)
  const bool vec = (n % 4u) == 0u && n >= 128u && n <= 16384u && (n <= 4096u || count < (1u << 22)) &&
                   ((reinterpret_cast<std::uintptr_t>(x) | reinterpret_cast<std::uintptr_t>(weight) |
                     reinterpret_cast<std::uintptr_t>(out)) % 16u) == 0u;
  // Four waves a vector up to 4096 values: 16 waves, one load each, take longer to
  // meet at the barrier also where one vector has the chip (one of 4096 2.35 us,
  // four waves 2.24; 64 of 4096 2.61 / 2.50; 512 of 2048 3.54 / 3.35).
  if (!vec)
    hipLaunchKernelGGL(rmsnorm_w_kernel, dim3(count), dim3(kOpThreads), 0, stream, x, weight, n, eps, out);
  else if (n <= 1024u)
    hipLaunchKernelGGL((rmsnorm_w_vec_kernel<256, 1>), dim3(count), dim3(256), 0, stream, x, weight, n, eps, out);
  else if (n <= 4096u)
    hipLaunchKernelGGL((rmsnorm_w_vec_kernel<256, 4>), dim3(count), dim3(256), 0, stream, x, weight, n, eps, out);
  else
    hipLaunchKernelGGL((rmsnorm_w_vec_kernel<1024, 4>), dim3(count), dim3(1024), 0, stream, x, weight, n, eps, out);
  return hipGetLastError();
}

extern "C" hipError_t rtxllm_rope_theta(float* vec, uint32_t n_heads, uint32_t head_dim, float theta,
                                        const uint32_t* pos, uint32_t count, hipStream_t stream) {
  if (vec == nullptr || pos == nullptr || n_heads == 0u || head_dim == 0u || (head_dim % 2u) != 0u || count == 0u ||
      count > 65535u || !(theta > 0.0f) || (reinterpret_cast<std::uintptr_t>(vec) % 8u) != 0u)
    return hipErrorInvalidValue;
  const std::uint64_t pairs = static_cast<std::uint64_t>(n_heads) * head_dim / 2u;
  if (pairs > 0xFFFFFFFFull / 2u) return hipErrorInvalidValue;
  const std::uint32_t np = static_cast<std::uint32_t>(pairs);
  const std::uint32_t shared = rope_shared_pairs(np, head_dim / 2u, count), per = shared > 0u ? shared : 1u;
  const dim3 grid((np + kOpThreads * per - 1u) / (kOpThreads * per), count);
  if (shared == 0u)
    hipLaunchKernelGGL(rope_theta_pair_kernel, grid, dim3(kOpThreads), 0, stream, vec, np, head_dim,
                       static_cast<double>(theta), pos);
  else if (shared == 1u)
    hipLaunchKernelGGL(rope_theta_kernel<1>, grid, dim3(kOpThreads), 0, stream, vec, np, head_dim,
                       static_cast<double>(theta), pos);
  else
    hipLaunchKernelGGL(rope_theta_kernel<4>, grid, dim3(kOpThreads), 0, stream, vec, np, head_dim,
                       static_cast<double>(theta), pos);
  return hipGetLastError();
}

extern "C" hipError_t rtxllm_silu_mul(const float* gate, const float* up, size_t n, float* out, hipStream_t stream) {
  if (gate == nullptr || up == nullptr || out == nullptr || n == 0u || n > (std::size_t{1} << 40))
    return hipErrorInvalidValue;
  const bool vec = ((reinterpret_cast<std::uintptr_t>(gate) | reinterpret_cast<std::uintptr_t>(up) |
                     reinterpret_cast<std::uintptr_t>(out)) % 16u) == 0u;
  const std::size_t items = vec ? n / 4u + (n & 3u) : n;
  const dim3 grid(static_cast<unsigned>((items + kOpThreads - 1u) / kOpThreads));
  if (vec)
    hipLaunchKernelGGL(silu_mul_vec_kernel, grid, dim3(kOpThreads), 0, stream, gate, up, n, out);
  else
    hipLaunchKernelGGL(silu_mul_kernel, grid, dim3(kOpThreads), 0, stream, gate, up, n, out);
  return hipGetLastError();
}

extern "C" hipError_t rtxllm_embed_gather_q5k(const uint8_t* table, uint32_t vocab, uint32_t cols,
                                              const uint32_t* tokens, uint32_t count, float* out,
                                              hipStream_t stream) {
  if (table == nullptr || tokens == nullptr || out == nullptr || vocab == 0u || cols == 0u || (cols % 256u) != 0u ||
      count == 0u || count > 65535u || (reinterpret_cast<std::uintptr_t>(table) % 4u) != 0u)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(embed_gather_q5k_kernel, dim3((cols / 256u + 3u) / 4u, count), dim3(256), 0, stream, table, vocab, cols,
                     tokens, out);
  return hipGetLastError();
}

extern "C" size_t rtxllm_attn_decode_workspace(uint32_t n_heads, uint32_t n_kv_heads, uint32_t capacity,
                                               uint32_t count) {
  if (!group_ok(n_heads, n_kv_heads) || capacity == 0u || count == 0u) return 0u;
  // the partials of every chunk
  return align256(4u * static_cast<std::size_t>(count) * attention_partials_floats(n_heads, n_kv_heads, capacity));
}

extern "C" hipError_t rtxllm_attn_decode_gqa_f16(const float* q, const uint16_t* k_cache, const uint16_t* v_cache,
                                                 const int32_t* block_table, uint32_t table_stride,
                                                 uint32_t n_heads, uint32_t n_kv_heads, uint32_t page_size,
                                                 uint32_t capacity, const uint32_t* pos, uint32_t count, float* out,
                                                 void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (q == nullptr || k_cache == nullptr || v_cache == nullptr || block_table == nullptr || pos == nullptr ||
      out == nullptr || workspace == nullptr || !group_ok(n_heads, n_kv_heads) || page_size == 0u ||
      capacity == 0u || capacity % page_size != 0u || count == 0u || count > 65535u ||
      (count > 1u && table_stride < capacity / page_size) ||
      (reinterpret_cast<std::uintptr_t>(k_cache) % 16u) != 0u || (reinterpret_cast<std::uintptr_t>(v_cache) % 16u) != 0u ||
      (reinterpret_cast<std::uintptr_t>(workspace) % 256u) != 0u)
    return hipErrorInvalidValue;
  const std::size_t need = rtxllm_attn_decode_workspace(n_heads, n_kv_heads, capacity, count);
  if (need == 0u || workspace_bytes < need) return hipErrorInvalidValue;
  auto* partials = static_cast<float*>(workspace);
  KvLayer kv{};
  kv.k = const_cast<std::uint16_t*>(k_cache);
  kv.v = const_cast<std::uint16_t*>(v_cache);
  kv.block_table = block_table;
  kv.page_size = page_size;
  kv.n_kv = n_kv_heads;
  kv.capacity = capacity;
  return launch_attention_batch(AttnQuery{nullptr, q}, kv, n_heads, pos, capacity, count, table_stride, partials, out,
                                nullptr, nullptr, stream);
}

extern "C" hipError_t rtxllm_argmax(const float* x, uint32_t n, uint32_t count, uint32_t* index,
                                    hipStream_t stream) {
  if (x == nullptr || index == nullptr || n == 0u || count == 0u || count > 65535u * 1024u)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(argmax_rows_kernel, dim3(count), dim3(kArgmaxThreads), 0, stream, x, n, index);
  return hipGetLastError();
}
