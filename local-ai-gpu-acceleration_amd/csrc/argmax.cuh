// Greedy argmax of one row by one workgroup, shared by the reference-named
// token kernels (feedback.hip) and rtxllm_argmax (llama_ops.hip).
#pragma once

#include <cfloat>

#include "common.h"

namespace rtxllm {

constexpr std::uint32_t kArgmaxThreads = 1024;

// Maximum (a) and, with it, minimum over the workgroup's 16 waves; every thread
// gets the result. The caller separates two uses of `sh` by a barrier.
template <class Op>
__device__ __forceinline__ std::uint32_t argmax_block_reduce(std::uint32_t v, std::uint32_t* sh, Op op) {
  v = lanes_reduce_exact(v, op);
  if ((threadIdx.x & 63u) == 0u) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  std::uint32_t r = sh[0];
#pragma unroll
  for (std::uint32_t w = 1; w < kArgmaxThreads / 64u; ++w) r = op(r, sh[w]);
  return r;
}

// Index of the largest of row[0, n): the lowest one among equal values; a NaN
// never wins and a row with nothing above -FLT_MAX gives 0 (the reference's
// scan from (-FLT_MAX, 0), decode_kernels.cu:2993-3031). Every thread of a
// kArgmaxThreads workgroup calls it and gets the index. n >= 1; row has any
// 4-byte alignment.
//
// One CU reads the whole row: the entry points have no scratch through which
// several could share it. So the time is the row's latency: a thread keeps two
// 16-byte loads in flight and only the maximum of each batch of eight values is
// compared, the index being found afterwards by reading the winning batch again.
// Against one 4-byte load and compare at a time: 8192 values 4.6 -> 2.8 us, 32768
// 8.4 -> 3.6, 128256 23.6 -> 6.0. Eight loads a thread are slower at every length
// (8193 values 4.6 us, two loads 2.8; 128256 7.6 / 6.0; 1000000 31.8 / 29.4).
__device__ __forceinline__ std::uint32_t argmax_row(const float* __restrict__ row, std::uint32_t n) {
  constexpr std::uint32_t U = 2;  // 16-byte loads of a batch
  __shared__ std::uint32_t sh[2][kArgmaxThreads / 64u];
  const std::uint32_t tid = threadIdx.x;
  // row = head (to the first 16-byte boundary), nv 16-byte vectors, tail
  const std::uint32_t to16 = static_cast<std::uint32_t>((16u - (reinterpret_cast<std::uintptr_t>(row) & 15u)) & 15u) / 4u;
  const std::uint32_t head = to16 < n ? to16 : n;
  const std::uint32_t nv = (n - head) / 4u, tail0 = head + 4u * nv;
  const float4* const vec = reinterpret_cast<const float4*>(row + head);
  float bv = -FLT_MAX;
  std::uint32_t bb = 0u;  // the batch that holds bv (of the thread's vectors)
  // vector j of batch b; past the end the row's last vector again (the same
  // value at its own index, so nothing has to be masked)
  auto at = [&](std::uint32_t b, std::uint32_t j) {
    const std::uint32_t i = (b * U + j) * kArgmaxThreads + tid;
    return i < nv ? i : nv - 1u;
  };
  const std::uint32_t batches = (nv + U * kArgmaxThreads - 1u) / (U * kArgmaxThreads);
  for (std::uint32_t b = 0; b < batches; ++b) {
    float4 v[U];
#pragma unroll
    for (std::uint32_t j = 0; j < U; ++j) v[j] = vec[at(b, j)];
    // fmaxf drops a NaN next to a number; of a batch of NaN nothing is > bv
    float m = fmaxf(fmaxf(v[0].x, v[0].y), fmaxf(v[0].z, v[0].w));
#pragma unroll
    for (std::uint32_t j = 1; j < U; ++j) m = fmaxf(m, fmaxf(fmaxf(v[j].x, v[j].y), fmaxf(v[j].z, v[j].w)));
    if (m > bv) bv = m, bb = b;
  }
  // the at most six values outside the vectors: one each for the first threads
  const std::uint32_t edges = head + (n - tail0);
  const std::uint32_t ei = tid < head ? tid : tail0 + (tid - head);
  const float ev = tid < edges ? row[ei] : -FLT_MAX;
  float mine = ev > bv ? ev : bv;
  mine += 0.0f;  // -0 -> +0: the ordered bits below then compare as the values do
  const std::uint32_t u = __float_as_uint(mine);
  const std::uint32_t key = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  const std::uint32_t best =
      argmax_block_reduce(key, sh[0], [](std::uint32_t a, std::uint32_t b) { return a > b ? a : b; });
  const float top = __uint_as_float((best & 0x80000000u) ? (best & 0x7FFFFFFFu) : ~best);
  std::uint32_t idx = 0xFFFFFFFFu;
  if (tid < edges && ev == top) idx = ei;
  if (bv == top && batches != 0u) {
#pragma unroll
    for (std::uint32_t j = 0; j < U; ++j) {
      const std::uint32_t i = at(bb, j);
      const float4 v = vec[i];
      const std::uint32_t k = v.x == top ? 0u : v.y == top ? 1u : v.z == top ? 2u : v.w == top ? 3u : 4u;
      const std::uint32_t c = head + 4u * i + k;
      if (k < 4u && c < idx) idx = c;
    }
  }
  idx = argmax_block_reduce(idx, sh[1], [](std::uint32_t a, std::uint32_t b) { return a < b ? a : b; });
  return top > -FLT_MAX ? idx : 0u;
}

}  // namespace rtxllm
