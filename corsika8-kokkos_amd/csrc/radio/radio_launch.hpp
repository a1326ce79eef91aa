// Host-callable launchers for the radio kernels (defined in radio_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <stdexcept>

#include "c8mi/c8mi_types.h"
#include "radio_device.hpp"

namespace c8mi::radio {

// Threads per workgroup of the pooled projection, and the least a workgroup has:
// 256, 512 and 1024 are instantiated.
inline constexpr std::uint32_t kProjectionBlock = 256;
// Dynamic LDS a projection workgroup may request (gfx950: 160 KiB per CU).
inline constexpr std::size_t kMaxDynamicLdsBytes = 144 * 1024;
// Default window tile: its dynamic LDS and kProjectionStaticLdsBytes stay within
// this budget, so three workgroups of the exact kernels share a CU (160 KiB). A
// 4096-bin ZHS window in one 96 KiB tile (one workgroup per CU) measured 2x slower
// than two 2048-bin tiles; a 1024-bin CoREAS+ZHS window (48 KiB of bins) and a
// 2048-bin ZHS window keep one tile. The fused pooled kernel has 2 KiB more static
// LDS: with tiles of 1091 to 1124 bins two of its workgroups share a CU, which made
// no difference (twelve served showers with windows of 1080 and 1110 bins 341 and
// 340 ms, 2170 and 2230 353 and 353), where a second tile would evaluate every
// update twice.
inline constexpr std::size_t kPreferredWorkgroupLdsBytes = 53 * 1024;
// Upper bound of a projection kernel's static LDS beside the pair lists and
// budgets: the wave totals of the ZHS scan (16 x 8 B for 1024 threads) and counters.
inline constexpr std::size_t kProjectionStaticLdsBytes = 256;
// Pair lists of the fast CoREAS kernels, bytes per thread (512 per wave); budgets
// of the fast ZHS kernels, bytes per observer.
inline constexpr std::size_t kPairListBytesPerThread = 8;
inline constexpr std::size_t kBudgetBytesPerObserver = 128;
// Most observers of a group, and of a workgroup of so many threads: only one of
// 1024 takes several.
inline constexpr std::uint32_t kMaxGroup = 8;
inline constexpr std::uint32_t most_observers(std::uint32_t threads) { return threads == 1024 ? kMaxGroup : 1; }
// LDS of a CU; what a fast workgroup holds beside its window tiles, and the most
// its tiles may take.
inline constexpr std::size_t kCuLdsBytes = 160 * 1024;
inline constexpr std::size_t fast_static_lds(bool coreas, bool zhs, std::uint32_t threads) {
  return kProjectionStaticLdsBytes + (coreas ? kPairListBytesPerThread * threads : 0u) +
         (zhs ? kBudgetBytesPerObserver * most_observers(threads) : 0u);
}
inline constexpr std::size_t fast_dynamic_lds_limit(bool coreas, bool zhs, std::uint32_t threads) {
  return kCuLdsBytes - fast_static_lds(coreas, zhs, threads);
}
// Most tracks a workgroup takes (its tallies and lists use 32-bit words).
inline constexpr std::uint64_t kMaxChunkTracks = std::uint64_t{1} << 27;
// Tracks per workgroup the default chunking gives a batch large enough for
// eight such chunks, at least (a smaller batch is cut into eight chunks).
inline constexpr std::uint64_t kMinimumDefaultChunk = 32768;
// XCDs of the chip: the projection grid maps chunk c to XCD c % kXcdCount.
inline constexpr std::uint64_t kXcdCount = 8;
// Bins of the default tile for `per_bin` int64 words per bin (3 per algorithm);
// a ZHS tile holds one more word per component row (its difference array).
inline std::uint64_t default_tile_capacity(std::size_t per_bin, bool zhs) {
  std::size_t const extra = zhs ? 3u : 0u;
  std::uint64_t const most = (kMaxDynamicLdsBytes / sizeof(long long) - extra) / per_bin;
  std::uint64_t const preferred =
      ((kPreferredWorkgroupLdsBytes - kProjectionStaticLdsBytes) / sizeof(long long) - extra) / per_bin;
  return preferred < most ? preferred : most;
}

// Launch-shape knobs of a projection (set_tuning), 0 = automatic: tracks per
// workgroup, window tile limit in bins, target workgroups per launch and threads
// per workgroup.
struct LaunchTuning {
  std::uint64_t chunk_tracks = 0;
  std::uint32_t tile_bins_limit = 0;
  std::uint32_t target_workgroups = 0;
  std::uint32_t block_threads = 0;
  bool automatic() const noexcept {
    return chunk_tracks == 0 && tile_bins_limit == 0 && target_workgroups == 0 && block_threads == 0;
  }
};
// The knobs as a caller gives them; throws invalid_argument.
LaunchTuning make_tuning(std::uint64_t chunk_tracks, std::uint32_t tile_bins, std::uint32_t target_workgroups,
                         std::uint32_t block_threads);
// What an automatic knob stands for where the shape isn't estimated (the exact
// form, the fast one of both algorithms or with another knob given): about 8192 workgroups of 512
// threads, measured for 2^20 tracks on 160 antennas with 2048 bins.
inline constexpr std::uint32_t kDefaultWorkgroups = 8192, kDefaultThreads = 512;

// Fills the shape fields of `L` (tile_bins, bin_tiles, chunk_size, chunks, group,
// block_threads) for `count` tracks on `observers` observers whose longest window
// has `max_bins` bins; `fast`: the fast kernels (an estimate gives their shape, with
// groups of observers, for one algorithm while every knob is automatic). Throws
// length_error when the grid exceeds 2^32 workgroups.
void shape_projection(ProjectionLaunch& L, bool coreas, bool zhs, bool fast, std::uint32_t observers,
                      std::uint64_t max_bins, std::uint64_t count, LaunchTuning const& tuning);

// `count` tracks, or the first of its halves, quarters, ... for which `check` (a
// shape_projection of so many) does not throw length_error.
template <class Check>
std::uint64_t launchable(std::uint64_t count, Check const& check) {
  for (;; count = (count + 1) / 2) {
    try {
      check(count);
      return count;
    } catch (std::length_error const&) {
      if (count <= 1) throw;
    }
  }
}

// LDS bytes for one workgroup holding `tile_bins` bins of each enabled mode.
std::size_t projection_lds_bytes(bool coreas, bool zhs, std::uint32_t tile_bins);
// Workgroups launched for `launch` (chunks rounded up to whole XCD rounds).
std::uint32_t projection_grid(ProjectionLaunch const& launch);

// exact: the reference's FP64 operation order (bit-identical fixed-point
// sums); otherwise the fast FP64 form. Floating accumulation is always exact.
void launch_projection(ProjectionLaunch const& launch, bool coreas, bool zhs, bool fixed,
                       bool exact, hipStream_t stream);

// Pooled showers (launch.segments set): `grid` workgroups, an upper bound on
// the items (*launch.item_count); int64 fixed point.
void launch_pooled_projection(ProjectionLaunch const& launch, bool coreas, bool zhs, bool exact,
                              std::uint32_t grid, hipStream_t stream);

// The fast kernels (int64 fixed point), launch.group observers per workgroup.
void launch_fast(ProjectionLaunch const& launch, bool coreas, bool zhs, std::uint32_t block, std::uint32_t grid,
                 hipStream_t stream);

void launch_records_to_tracks(c8mi_lepton_transport_record const* records,
                              std::uint64_t count, double* tracks, std::uint64_t stride,
                              hipStream_t stream);

}  // namespace c8mi::radio
