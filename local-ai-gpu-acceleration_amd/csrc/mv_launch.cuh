// Host-side launch of mv_kernel: geometry selection and the format switch,
// shared by the matvec entry points and the layer pipeline's fused matvecs.
#pragma once

#include "mv.cuh"

namespace rtxllm {

inline int num_cus() {
  static int cached = 0;
  if (cached == 0) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
      cached = n;
    else
      cached = 256;
  }
  return cached;
}

// Launch geometry of mv_kernel, from sweeps on MI355X at the 8B decode shapes:
//  * one unit (32 columns) per lane for rows of up to 16384 columns (two
//    beyond), ks = ceil(units / 64) waves per row;
//  * small matrices: nrg = 4 / ks row groups per workgroup (at least 1) and one
//    4-row tile per row group: many small workgroups, every tile in flight;
//  * large matrices (more row groups than the chip holds at once): a
//    persistent grid of exactly the workgroups that are resident together
//    (the kernel's occupancy, queried once per instantiation and block size),
//    nrg = 1 for the IQ formats; each row group double-buffers its tiles and
//    the workgroup copies its codebook once;
//  * epilogues with pairwise hand-over (max_waves > 8) on large matrices: as
//    many row groups per workgroup as max_waves allows, one workgroup per
//    resident slot;
//  * grouped epilogues (group_rows > 0): a group's tiles over as many row
//    groups as fit in 8 waves (nrg divides the group's tile count) and the rest
//    over consecutive rounds; one group per workgroup, or several in turn when
//    there are more groups than resident workgroups.
struct MvGeom {
  int upl;
  unsigned ks, nrg, grid;
};

// resident(block_threads) = workgroups of that size resident per CU (0: unknown).
// share > 0: the shared self-staging kernel with that many row groups a workgroup
// (mv_share_groups), the rest as the plain launches.
template <class Resident>
inline bool mv_geom(int fmt, std::uint32_t rows, std::uint32_t cols, int tile, std::uint32_t group_rows,
                    std::uint32_t max_waves, std::uint32_t share, Resident resident, MvGeom& g) {
  const std::uint32_t units = cols / 32u;
  g.upl = units > 512u ? 2 : 1;
  g.ks = (units + 64u * g.upl - 1u) / (64u * g.upl);
  if (g.ks > static_cast<unsigned>(kMaxKs)) return false;
  const std::uint32_t tiles = (rows + tile - 1) / tile;
  const std::uint32_t cus = static_cast<std::uint32_t>(num_cus());
  std::uint32_t grid;
  if (group_rows > 0u) {
    const std::uint32_t tg = group_rows / static_cast<std::uint32_t>(tile);
    g.nrg = 1u;
    while (2u * g.nrg <= tg && tg % (2u * g.nrg) == 0u && g.ks * 2u * g.nrg <= static_cast<unsigned>(kMaxKs))
      g.nrg *= 2u;
    grid = (tiles + tg - 1u) / tg;
  } else {
    g.nrg = g.ks >= 4u ? 1u : 4u / g.ks;
    if (share > 0u) g.nrg = share;
    grid = (tiles + g.nrg - 1) / g.nrg;
  }
  const std::uint32_t per_cu = static_cast<std::uint32_t>(resident(64u * g.ks * g.nrg));
  if (per_cu > 0u && grid > per_cu * cus) {
    const std::uint32_t nrg_wide = max_waves / g.ks;
    const std::uint32_t per_cu_wide =
        max_waves > static_cast<std::uint32_t>(kMaxKs) && nrg_wide > g.nrg
            ? static_cast<std::uint32_t>(resident(64u * g.ks * nrg_wide))
            : 0u;
    if (group_rows == 0u && per_cu_wide > 0u) {
      g.nrg = nrg_wide;
      grid = per_cu_wide * cus;
    } else if (group_rows == 0u && share == 0u && fmt_is_iq(fmt) && g.nrg > 1u) {
      g.nrg = 1u;
      const std::uint32_t per_cu1 = static_cast<std::uint32_t>(resident(64u * g.ks));
      grid = (per_cu1 > 0u ? per_cu1 : 1u) * cus;
    } else {
      grid = per_cu * cus;  // workgroups take several tiles / groups in turn
    }
  }
  g.grid = grid < 1u ? 1u : (grid > 1048576u ? 1048576u : grid);
  return true;
}

// Resident workgroups per CU of one mv_kernel instantiation at a block size
// (cached; 0 if the query fails).
template <int FMT, int UPL, int TILE, bool SELF, class Epi, bool SHARE = false>
inline int mv_resident(std::uint32_t block_threads) {
  constexpr std::uint32_t kW = EpiWaves<Epi>::value;
  static int cache[kW + 1] = {};
  const std::uint32_t w = block_threads / 64u;
  if (w == 0u || w > kW) return 0;
  if (cache[w] == 0) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &n, reinterpret_cast<const void*>(&mv_kernel<FMT, UPL, TILE, SELF, Epi, SHARE>),
            static_cast<int>(block_threads), 0) != hipSuccess || n <= 0)
      return 0;
    cache[w] = n;
  }
  return cache[w];
}

// Row groups per workgroup of the shared self-staging kernel (0: the kernel whose
// waves stage their own columns). Same results bit for bit, so the line is drawn
// by time alone, over 256 to 64000 rows and 256 to 8192 columns (fp32 x, cold
// weights, us of each without / with sharing). ks: waves a row; fill: whole
// 4-row tiles a CU. One row group a workgroup stages all of x as its wave would
// alone, and passes it through LDS (Q5_K 2000x2048 4.1 / 5.4), and three or six
// leave a last round of workgroups on part of the CUs (IQ3_S 3600x2560 with three
// 6.6 / 7.1, with four 5.6).
//  * IQ formats, a wave a row: four groups (IQ2_S 256x2048 4.9 / 3.8, 8192x2048 7.5
//    / 5.2; IQ3_S 3000x2048 5.1 / 4.7), eight from 16 tiles a CU on (IQ2_S 22000x768:
//    without 13.0, four 8.2, eight 7.8);
//  * two waves a row: four groups from two tiles a CU on (IQ2_S 14336x4096 14.6 /
//    10.8, IQ3_S 4096x4096 7.4 / 6.6); with fewer they leave CUs idle (IQ3_S
//    2000x4096 5.3 / 5.9);
//  * three or four: two groups, IQ2_S from two tiles a CU on (4096x8192 12.6 / 9.1),
//    in units with three waves up to nine (8192x5632 15.0 / 13.5, 14336x5632 18.4 /
//    19.0); IQ3_S with four waves from three tiles on (4096x8192 11.0 / 10.2,
//    3000x8192 9.3 / 9.8), with three between four and nine and not in units
//    (6000x5120 11.6 / 11.1, 3000x5120 7.9 / 8.3, 14336x6144 17.5 / 18.4, in units
//    7000x6144 12.8 / 16.2);
//  * K-quants only where one wave holds a row. Up to 1024 columns and below two
//    tiles a CU, two groups, or one where a workgroup each then fills no more than
//    the CUs and x is short (Q4_K 1000x512 3.5 / 3.1, 1000x1024 3.5 / 3.2). Else
//    Q5_K four (2000x2048 4.1 / 3.8, 14336x1024 8.1 / 7.4), Q4_K, up to 1024
//    columns, four from five tiles on (12000x1024 6.0 / 5.5) and none before
//    (3000x1024 3.5 / 3.7 with four, 4.4 with two);
//  * not from four rounds a row group on, where the staging is paid off anyway
//    and the row groups of a workgroup run in step (IQ3_S 64000x2560 29.3 / 31.3).
template <int FMT, bool SELF, class Epi>
inline std::uint32_t mv_share_groups(std::uint32_t rows, std::uint32_t cols) {
  if constexpr (!SELF || EpiGroupRows<Epi>::value > 0u) return 0u;
  const std::uint32_t ks = (cols / 32u + 63u) / 64u, cus = static_cast<std::uint32_t>(num_cus());
  const std::uint32_t tiles = (rows + Epi::kTile - 1u) / Epi::kTile, fill = tiles / cus;
  // 16 waves a CU resident: 16 / ks row groups
  if (cols > kSelfShareCols || static_cast<std::uint64_t>(tiles) * ks > 4ull * 16ull * cus) return 0u;
  if constexpr (!fmt_is_iq(FMT)) {
    if (ks > 1u || (FMT != RTXLLM_FMT_Q5K && cols > 1024u)) return 0u;
    if (cols <= 1024u && fill < 2u) return cols <= 512u && fill == 0u ? 1u : 2u;
    return FMT == RTXLLM_FMT_Q5K || fill >= 5u ? 4u : 0u;
  }
  if (ks == 1u) return fill < 16u ? 4u : 8u;
  if (ks == 2u) return fill < 2u ? 0u : 4u;
  if constexpr (FMT == RTXLLM_FMT_IQ3S || FMT == RTXLLM_FMT_IQ3S_UNITS) {
    if (ks == 4u) return fill < 3u ? 0u : 2u;
    return FMT == RTXLLM_FMT_IQ3S && fill >= 4u && fill < 9u ? 2u : 0u;
  }
  return fill >= 2u && (FMT != RTXLLM_FMT_IQ2S_UNITS || ks == 4u || fill < 9u) ? 2u : 0u;
}

template <int FMT, bool SELF, class Epi>
inline bool mv_geometry_fmt(std::uint32_t rows, std::uint32_t cols, MvGeom& g) {
  constexpr int kT = Epi::kTile;
  constexpr bool kCanShare = SELF && EpiGroupRows<Epi>::value == 0u;
  const std::uint32_t units = cols / 32u, share = mv_share_groups<FMT, SELF, Epi>(rows, cols);
  auto resident = [units, share](std::uint32_t threads) {
    if (kCanShare && share > 0u) return mv_resident<FMT, 1, kT, SELF, Epi, kCanShare>(threads);
    return units > 512u ? mv_resident<FMT, 2, kT, SELF, Epi>(threads) : mv_resident<FMT, 1, kT, SELF, Epi>(threads);
  };
  return mv_geom(FMT, rows, cols, kT, EpiGroupRows<Epi>::value, EpiWaves<Epi>::value, share, resident, g);
}

template <int FMT, bool SELF, class Epi>
inline hipError_t launch_mv_fmt(const QTensor& w, const XSrc& xs, std::uint32_t row_count, const Epi& epi,
                                hipStream_t stream) {
  constexpr int kT = Epi::kTile;
  // the kernel addresses each stream with 32-bit byte offsets
  const std::uint64_t blocks = static_cast<std::uint64_t>(row_count) * (w.cols / 256u);
  if (blocks * FmtBytes<FMT>::payload > 0xFFFFFFFFull || blocks * FmtBytes<FMT>::meta > 0xFFFFFFFFull)
    return hipErrorInvalidValue;
  MvGeom g;
  if (!mv_geometry_fmt<FMT, SELF, Epi>(row_count, w.cols, g)) return hipErrorInvalidValue;
  const dim3 grid(g.grid), block(64u * g.ks * g.nrg);
  if constexpr (SELF && EpiGroupRows<Epi>::value == 0u) {
    if (mv_share_groups<FMT, SELF, Epi>(row_count, w.cols) > 0u) {
      hipLaunchKernelGGL((mv_kernel<FMT, 1, kT, SELF, Epi, true>), grid, block, 0, stream, w, xs, row_count, g.ks, epi);
      return hipGetLastError();
    }
  }
  if (g.upl == 2) {
    hipLaunchKernelGGL((mv_kernel<FMT, 2, kT, SELF, Epi>), grid, block, 0, stream, w, xs, row_count, g.ks, epi);
  } else {
    hipLaunchKernelGGL((mv_kernel<FMT, 1, kT, SELF, Epi>), grid, block, 0, stream, w, xs, row_count, g.ks, epi);
  }
  return hipGetLastError();
}

// The geometry launch_mv<SELF, Epi> would use for this format and shape.
template <bool SELF, class Epi>
inline bool mv_geometry(int fmt, std::uint32_t rows, std::uint32_t cols, MvGeom& g) {
  switch (fmt) {
    case RTXLLM_FMT_Q4K_RAW: return mv_geometry_fmt<RTXLLM_FMT_Q4K_RAW, SELF, Epi>(rows, cols, g);
    case RTXLLM_FMT_Q4K_SPLIT_PREDECODED:
      return mv_geometry_fmt<RTXLLM_FMT_Q4K_SPLIT_PREDECODED, SELF, Epi>(rows, cols, g);
    case RTXLLM_FMT_Q4K_SPLIT_HALF: return mv_geometry_fmt<RTXLLM_FMT_Q4K_SPLIT_HALF, SELF, Epi>(rows, cols, g);
    case RTXLLM_FMT_Q4K_SPLIT_COMPACT:
      return mv_geometry_fmt<RTXLLM_FMT_Q4K_SPLIT_COMPACT, SELF, Epi>(rows, cols, g);
    case RTXLLM_FMT_Q4K_SPLIT_NATIVE: return mv_geometry_fmt<RTXLLM_FMT_Q4K_SPLIT_NATIVE, SELF, Epi>(rows, cols, g);
    case RTXLLM_FMT_Q5K: return mv_geometry_fmt<RTXLLM_FMT_Q5K, SELF, Epi>(rows, cols, g);
    case RTXLLM_FMT_IQ2S: return mv_geometry_fmt<RTXLLM_FMT_IQ2S, SELF, Epi>(rows, cols, g);
    case RTXLLM_FMT_IQ2S_UNITS: return mv_geometry_fmt<RTXLLM_FMT_IQ2S_UNITS, SELF, Epi>(rows, cols, g);
    case RTXLLM_FMT_IQ3S_UNITS: return mv_geometry_fmt<RTXLLM_FMT_IQ3S_UNITS, SELF, Epi>(rows, cols, g);
    case RTXLLM_FMT_IQ3S: return mv_geometry_fmt<RTXLLM_FMT_IQ3S, SELF, Epi>(rows, cols, g);
    case RTXLLM_FMT_Q4K_RAW_PREDECODED:
      return mv_geometry_fmt<RTXLLM_FMT_Q4K_RAW_PREDECODED, SELF, Epi>(rows, cols, g);
    default: return false;
  }
}

template <bool SELF, class Epi>
inline hipError_t launch_mv(int fmt, const QTensor& w, const XSrc& xs, std::uint32_t row_count, const Epi& epi,
                     hipStream_t stream) {
  switch (fmt) {
    case RTXLLM_FMT_Q4K_RAW: return launch_mv_fmt<RTXLLM_FMT_Q4K_RAW, SELF>(w, xs, row_count, epi, stream);
    case RTXLLM_FMT_Q4K_SPLIT_PREDECODED:
      return launch_mv_fmt<RTXLLM_FMT_Q4K_SPLIT_PREDECODED, SELF>(w, xs, row_count, epi, stream);
    case RTXLLM_FMT_Q4K_SPLIT_HALF:
      return launch_mv_fmt<RTXLLM_FMT_Q4K_SPLIT_HALF, SELF>(w, xs, row_count, epi, stream);
    case RTXLLM_FMT_Q4K_SPLIT_COMPACT:
      return launch_mv_fmt<RTXLLM_FMT_Q4K_SPLIT_COMPACT, SELF>(w, xs, row_count, epi, stream);
    case RTXLLM_FMT_Q4K_SPLIT_NATIVE:
      return launch_mv_fmt<RTXLLM_FMT_Q4K_SPLIT_NATIVE, SELF>(w, xs, row_count, epi, stream);
    case RTXLLM_FMT_Q5K: return launch_mv_fmt<RTXLLM_FMT_Q5K, SELF>(w, xs, row_count, epi, stream);
    case RTXLLM_FMT_IQ2S: return launch_mv_fmt<RTXLLM_FMT_IQ2S, SELF>(w, xs, row_count, epi, stream);
    case RTXLLM_FMT_IQ2S_UNITS: return launch_mv_fmt<RTXLLM_FMT_IQ2S_UNITS, SELF>(w, xs, row_count, epi, stream);
    case RTXLLM_FMT_IQ3S_UNITS: return launch_mv_fmt<RTXLLM_FMT_IQ3S_UNITS, SELF>(w, xs, row_count, epi, stream);
    case RTXLLM_FMT_IQ3S: return launch_mv_fmt<RTXLLM_FMT_IQ3S, SELF>(w, xs, row_count, epi, stream);
    case RTXLLM_FMT_Q4K_RAW_PREDECODED:
      return launch_mv_fmt<RTXLLM_FMT_Q4K_RAW_PREDECODED, SELF>(w, xs, row_count, epi, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace rtxllm
