// Per-element dequant of the resident-pack layouts with the reference gate's
// expression order (runtime/apps/mixed_sequence_benchmark_runner/main.cpp:
// 1133-1259), compiled without FMA contraction: bit-exact with the CPU gate.
// Used by the dequant entry point, the Q5_K embedding gather and the decode step's
// embedding.
#pragma once

#include "mv.cuh"

namespace rtxllm {

#pragma clang fp contract(off)
// Value v of an IQ2_S or IQ3_S block (the unit layouts, whose bytes are gathered
// first; every other layout expands four values a lane, below).
template <int FMT>
__device__ __forceinline__ float dequant_value(const std::uint8_t* p, std::uint32_t v) {
  static_assert(FMT == RTXLLM_FMT_IQ2S || FMT == RTXLLM_FMT_IQ3S, "an IQ block");
  if constexpr (FMT == RTXLLM_FMT_IQ2S) {
    const std::uint32_t ib32 = v >> 5, grp = (v & 31u) >> 3, lane = v & 7u;
    const float d = f16_bits_to_f32(ld_u16(p));
    const std::uint32_t go = ib32 * 4u + grp;
    const std::uint32_t idx = p[2u + go] | ((static_cast<std::uint32_t>(p[66u + ib32]) << (8u - 2u * grp)) & 0x300u);
    const std::uint32_t grid = 2u * ((kIq2sGridDev[idx] >> (2u * lane)) & 3u) + 1u;
    const std::uint32_t sb = p[74u + ib32];
    const std::uint32_t nib = grp < 2u ? (sb & 15u) : (sb >> 4);
    const float scale = d * (0.5f + static_cast<float>(nib)) * 0.25f;
    const bool neg = (p[34u + go] >> lane) & 1u;
    return scale * static_cast<float>(grid) * (neg ? -1.0f : 1.0f);
  } else {
    const std::uint32_t ib32 = v >> 5, grp = (v & 31u) >> 3, lane = v & 7u, pair = lane >> 2, gl = lane & 3u;
    const float d = f16_bits_to_f32(ld_u16(p));
    const std::uint32_t sel = ib32 * 8u + grp * 2u + pair;
    const std::uint32_t hb = (p[66u + ib32] >> (2u * grp + pair)) & 1u;
    const std::uint32_t idx = p[2u + sel] | (hb << 8);
    const std::uint32_t grid = (kIq3sGridDev[idx] >> (8u * gl)) & 0xFFu;
    const std::uint32_t sb = p[106u + (ib32 >> 1)];
    const std::uint32_t nib = (ib32 & 1u) == 0u ? (sb & 15u) : (sb >> 4);
    const float scale = d * static_cast<float>(1u + 2u * nib);
    const bool neg = (p[74u + ib32 * 4u + grp] >> lane) & 1u;
    return scale * static_cast<float>(grid) * (neg ? -1.0f : 1.0f);
  }
}

// scale_min_k4 without its branch (a load would move into it, behind a wait).
__device__ __forceinline__ void scale_min_select(std::uint32_t j, std::uint32_t s0, std::uint32_t s1, std::uint32_t s2,
                                                 std::uint32_t& sc, std::uint32_t& m) {
  const std::uint32_t sh = 8u * (j & 3u), a = s0 >> sh, b = s1 >> sh, c = s2 >> sh;
  sc = j < 4u ? (a & 63u) : ((c & 15u) | ((a >> 2) & 0x30u));
  m = j < 4u ? (b & 63u) : (((c >> 4) & 15u) | ((b >> 2) & 0x30u));
}

// Values 4 l .. 4 l + 3 of a block (lane l of the wave that holds the block) in
// two steps, so that a wave can have several blocks' loads in flight: run4_load
// reads the fields, run4_values expands them with the reference's expressions in
// its order. The four values share the sub-block, its scale
// (and min) and, in the IQ formats, the codebook word, so those are read and
// decoded once; K-quant codes are one dword (blocks 4-byte aligned, or 2-byte in
// the IQ formats, which read theirs as bytes).
struct Run4 {
  std::uint32_t code;              // K: the four codes' dword; IQ: low index byte
  std::uint32_t h0, h1, h2, h3;    // K: head words (or the scale / min pair); IQ: d, qh, scales, signs
  std::uint32_t qh;                // Q5_K: high-bit dword
};
template <int FMT>
__device__ __forceinline__ Run4 run4_load(const std::uint8_t* p, const std::uint8_t* m, std::uint32_t l) {
  Run4 r{};
  if constexpr (FMT == RTXLLM_FMT_IQ2S || FMT == RTXLLM_FMT_IQ3S) {
    const std::uint32_t ib32 = l >> 3, grp = (l & 7u) >> 1;
    constexpr bool k2 = FMT == RTXLLM_FMT_IQ2S;
    r.h0 = ld_u16(p);
    r.code = p[2u + (k2 ? ib32 * 4u + grp : l)];  // IQ3_S: 8 ib32 + 2 grp + pair = l
    r.h1 = p[66u + ib32];
    r.h2 = p[k2 ? 74u + ib32 : 106u + (ib32 >> 1)];
    r.h3 = p[(k2 ? 34u : 74u) + ib32 * 4u + grp];
  } else {
    const std::uint32_t g = l >> 4, pair = l >> 3, lane0 = 4u * (l & 7u);
    constexpr bool kRaw = FMT == RTXLLM_FMT_Q4K_RAW || FMT == RTXLLM_FMT_Q4K_RAW_PREDECODED;
    const std::uint8_t* qs = p + (FMT == RTXLLM_FMT_Q5K ? 48u : kRaw ? 16u : 0u);
    r.code = ld_u32(qs + 32u * g + lane0);
    if constexpr (FMT == RTXLLM_FMT_Q5K) r.qh = ld_u32(p + 16u + lane0);
    if constexpr (FMT == RTXLLM_FMT_Q4K_SPLIT_PREDECODED || FMT == RTXLLM_FMT_Q4K_RAW_PREDECODED) {
      r.h0 = ld_u32(m + 8u * pair);
      r.h1 = ld_u32(m + 8u * pair + 4u);
    } else if constexpr (FMT == RTXLLM_FMT_Q4K_SPLIT_HALF) {
      r.h0 = ld_u32(m + 4u * pair);
    } else if constexpr (FMT == RTXLLM_FMT_Q4K_SPLIT_COMPACT) {
      r.h0 = ld_u32(m);
      r.h1 = m[4u + pair];
      r.h2 = m[12u + pair];
    } else {
      const std::uint8_t* h = (FMT == RTXLLM_FMT_Q4K_RAW || FMT == RTXLLM_FMT_Q5K) ? p : m;
      r.h0 = ld_u32(h), r.h1 = ld_u32(h + 4), r.h2 = ld_u32(h + 8), r.h3 = ld_u32(h + 12);
    }
  }
  return r;
}
template <int FMT>
__device__ __forceinline__ float4 run4_values(const Run4& r, std::uint32_t l) {
  if constexpr (FMT == RTXLLM_FMT_IQ2S) {
    const std::uint32_t grp = (l & 7u) >> 1, lane0 = 4u * (l & 1u);
    const std::uint32_t grid = kIq2sGridDev[r.code | ((r.h1 << (8u - 2u * grp)) & 0x300u)];
    const std::uint32_t nib = grp < 2u ? (r.h2 & 15u) : (r.h2 >> 4);
    const float scale = f16_bits_to_f32(r.h0) * (0.5f + static_cast<float>(nib)) * 0.25f;
    auto val = [&](std::uint32_t k) {
      const std::uint32_t lane = lane0 + k;
      return scale * static_cast<float>(2u * ((grid >> (2u * lane)) & 3u) + 1u) * (((r.h3 >> lane) & 1u) ? -1.0f : 1.0f);
    };
    return make_float4(val(0u), val(1u), val(2u), val(3u));
  } else if constexpr (FMT == RTXLLM_FMT_IQ3S) {
    const std::uint32_t ib32 = l >> 3, sub = l & 7u, pair = l & 1u;  // sub = 2 grp + pair
    const std::uint32_t grid = kIq3sGridDev[r.code | (((r.h1 >> sub) & 1u) << 8)];
    const std::uint32_t nib = (ib32 & 1u) == 0u ? (r.h2 & 15u) : (r.h2 >> 4);
    const float scale = f16_bits_to_f32(r.h0) * static_cast<float>(1u + 2u * nib);
    auto val = [&](std::uint32_t k) {
      return scale * static_cast<float>((grid >> (8u * k)) & 0xFFu) * (((r.h3 >> (4u * pair + k)) & 1u) ? -1.0f : 1.0f);
    };
    return make_float4(val(0u), val(1u), val(2u), val(3u));
  } else {
    const std::uint32_t high = (l >> 3) & 1u, pair = l >> 3;
    std::uint32_t codes = (r.code >> (4u * high)) & 0x0F0F0F0Fu;
    if constexpr (FMT == RTXLLM_FMT_Q5K) codes |= ((r.qh >> pair) & 0x01010101u) << 4;
    float s, mn;
    if constexpr (FMT == RTXLLM_FMT_Q4K_SPLIT_PREDECODED || FMT == RTXLLM_FMT_Q4K_RAW_PREDECODED) {
      s = __uint_as_float(r.h0), mn = __uint_as_float(r.h1);
    } else if constexpr (FMT == RTXLLM_FMT_Q4K_SPLIT_HALF) {
      s = f16_bits_to_f32(r.h0), mn = f16_bits_to_f32(r.h0 >> 16);
    } else {
      const float d = f16_bits_to_f32(r.h0), dmin = f16_bits_to_f32(r.h0 >> 16);
      std::uint32_t sc, m6;
      if constexpr (FMT == RTXLLM_FMT_Q4K_SPLIT_COMPACT)
        sc = r.h1, m6 = r.h2;
      else
        scale_min_select(pair, r.h1, r.h2, r.h3, sc, m6);
      s = d * static_cast<float>(sc), mn = dmin * static_cast<float>(m6);
    }
    auto val = [&](std::uint32_t k) { return s * static_cast<float>((codes >> (8u * k)) & 0xFFu) - mn; };
    return make_float4(val(0u), val(1u), val(2u), val(3u));
  }
}

// Values [16 t, 16 t + 16) of a Q5_K block (t in [0, 16)) from three aligned
// 16-byte loads: the head (d, dmin, scales), the 16 qh bytes and the 16 qs
// bytes the run uses (the run lies in one 32-value sub-block). Same values,
// bit for bit, as run4_values<Q5K> over the run. The block must be
// 16-byte aligned (176-byte blocks of a 16-byte aligned table are).
__device__ __forceinline__ void dequant_q5k_run16(const std::uint8_t* blk, std::uint32_t t, float out[16]) {
  const std::uint32_t v0 = 16u * t, g = v0 >> 6, high = (v0 & 63u) >= 32u ? 1u : 0u, lane0 = v0 & 31u;
  const uint4 head = *reinterpret_cast<const uint4*>(blk);
  const uint4 qh4 = *reinterpret_cast<const uint4*>(blk + 16u + lane0);
  const uint4 qs4 = *reinterpret_cast<const uint4*>(blk + 48u + 32u * g + lane0);
  const float d = f16_bits_to_f32(static_cast<std::uint16_t>(head.x & 0xFFFFu));
  const float dmin = f16_bits_to_f32(static_cast<std::uint16_t>(head.x >> 16));
  std::uint32_t sc, mn;
  scale_min_k4(static_cast<int>(2u * g + high), head.y, head.z, head.w, sc, mn);
  const std::uint32_t qh[4] = {qh4.x, qh4.y, qh4.z, qh4.w}, qs[4] = {qs4.x, qs4.y, qs4.z, qs4.w};
  const std::uint32_t hbit = 2u * g + high;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const std::uint32_t packed = (qs[j >> 2] >> (8 * (j & 3))) & 0xFFu;
    const std::uint32_t low = high ? (packed >> 4) : (packed & 15u);
    const std::uint32_t quant = low + (((((qh[j >> 2] >> (8 * (j & 3))) & 0xFFu) >> hbit) & 1u) ? 16u : 0u);
    out[j] = d * static_cast<float>(sc) * static_cast<float>(quant) - dmin * static_cast<float>(mn);
  }
}
#pragma clang fp contract(on)

}  // namespace rtxllm
