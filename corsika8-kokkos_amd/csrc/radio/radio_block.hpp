// Workgroup-level pieces shared by the exact and the fast projection kernels:
// wave sums, the scan that turns a ZHS difference array into bins, the flush of
// a window tile and of the tallies.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "radio_device.hpp"

namespace c8mi::radio {

inline constexpr int kXcds = 8;

// Inclusive prefix sum over `count` entries of an LDS row, whole block: each
// thread sums a contiguous run, the run totals are scanned within each wave by
// shuffles and across waves by the first wave (wave_totals: one entry per wave).
template <class T>
__device__ __forceinline__ T wave_inclusive_sum(T x, std::uint32_t lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    T const y = __shfl_up(x, d, 64);
    if (static_cast<int>(lane) >= d) x += y;
  }
  return x;
}

template <class T>
__device__ __forceinline__ void block_inclusive_scan(T* row, std::uint32_t count, T* wave_totals) {
  std::uint32_t const tid = threadIdx.x;
  std::uint32_t const threads = blockDim.x;
  std::uint32_t const lane = tid & 63u, wave = tid >> 6;
  std::uint32_t const waves = (threads + 63u) >> 6;
  std::uint32_t const per = (count + threads - 1) / threads;
  std::uint32_t const begin = tid * per < count ? tid * per : count;
  std::uint32_t const end = begin + per < count ? begin + per : count;
  T running = 0;
  for (std::uint32_t i = begin; i < end; ++i) {
    running += row[i];
    row[i] = running;
  }
  T const inclusive = wave_inclusive_sum(running, lane);
  if (lane == 63u) wave_totals[wave] = inclusive;
  __syncthreads();
  if (wave == 0) {
    T const total = lane < waves ? wave_totals[lane] : T(0);
    T const before = wave_inclusive_sum(total, lane) - total;
    if (lane < waves) wave_totals[lane] = before;
  }
  __syncthreads();
  T const offset = wave_totals[wave] + (inclusive - running);
  for (std::uint32_t i = begin; i < end; ++i) row[i] += offset;
  __syncthreads();
}

template <class T>
__device__ __forceinline__ T wave_sum(T x) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) x += __shfl_xor(x, d, 64);
  return x;
}

// XCD-aware decode of a workgroup of an unpooled launch into (chunk, position
// in the chunk's observer groups and window tiles): workgroup b runs on XCD
// b % 8, which takes the chunks c with c % 8 == b % 8. False: no chunk.
__device__ __forceinline__ bool decode_chunk(ProjectionLaunch const& L, std::uint32_t per_chunk, std::uint32_t& within,
                                             std::uint64_t& begin, std::uint64_t& end) {
  std::uint32_t const sequence = blockIdx.x / kXcds;
  std::uint32_t const chunk = (sequence / per_chunk) * kXcds + blockIdx.x % kXcds;
  if (chunk >= L.chunks) return false;
  within = sequence % per_chunk;
  begin = static_cast<std::uint64_t>(chunk) * L.chunk_size;
  end = begin + L.chunk_size < L.track_count ? begin + L.chunk_size : L.track_count;
  return true;
}

// Pooled showers: the segment whose items hold blockIdx.x (binary search over
// item_begin). False: no item.
__device__ __forceinline__ bool decode_segment(ProjectionLaunch const& L, SegmentDev& seg, std::uint64_t& local) {
  unsigned long long const item = blockIdx.x;
  if (item >= *L.item_count) return false;
  std::uint32_t lo = 0, hi = *L.segment_count;  // segments[lo].item_begin <= item
  while (hi - lo > 1) {
    std::uint32_t const mid = (lo + hi) / 2;
    if (L.segments[mid].item_begin <= item) lo = mid;
    else hi = mid;
  }
  seg = L.segments[lo];
  local = item - seg.item_begin;
  return true;
}

// ---- sums in a tile cannot wrap ----
//
// Integer sums are exact modulo 2^64, and a bin's sum is bounded by the sum of its
// |increments|: a thread adds to the tile without further ado while the sum of its
// own stays below 2^51 (2^61 for 1024 threads). Past that limit
//  * a CoREAS sample is added with a look at the bin: one that has grown to 2^60 is
//    moved to the waveform. Bins stay below 2^60, the 2^61 above and what 1024
//    threads add before they look, 2^61;
//  * a short ZHS segment (its tile holds differences, so a bin shows in the sum over
//    them only) takes its share of 2^62 that a range of bins has in common; when
//    that is used up, it goes to the waveform bin by bin, as a longer one does.
// Additions to the waveform are checked. To compare a workgroup's sum of |increments|
// with 2^63 instead would refuse waveforms that fit, as most of that sum cancels, and
// the sooner the more observers and tracks a workgroup takes: 2^20 tracks of random
// charge on 160 antennas whose field peaks at 1% of 2^62 were refused, by 131072
// tracks of five observers a workgroup as by 32768 of one. They take (CoREAS + ZHS)
// 2.7 + 1.7 ms at a peak of 0.1% (1.9 + 1.6 within the limit), 3.0 + 2.3 at 1% and
// 7.7 + 15 at 10%.
inline constexpr double kThreadLimit = 2251799813685248.;      // 2^51
inline constexpr long long kBinLimit = 1LL << 60;
inline constexpr double kRangeLimit = 4611686018427387904.;    // 2^62
inline constexpr std::uint32_t kRanges = 16;  // of an observer's bins in a tile
using Budget = double;  // LDS, per range; zero at first

// The range of a tile's bin, for tiles of `bins`.
__device__ __forceinline__ std::uint32_t bin_range(std::uint32_t bin, std::uint32_t bins) {
  std::uint32_t const bits = bins > kRanges ? 32u - static_cast<std::uint32_t>(__builtin_clz(bins - 1)) - 4u : 0u;
  static_assert(kRanges == 16, "ranges are the upper four bits of a bin");
  return bin >> bits;
}

// Whether the tile takes a ZHS segment of bins [first, last] and `bound`.
__device__ __forceinline__ bool tile_takes(Budget* budgets, std::uint32_t first, std::uint32_t last, std::uint32_t bins,
                                           double bound) {
  std::uint32_t const range = bin_range(first, bins);
  return bound < kRangeLimit && bin_range(last, bins) == range && atomicAdd(budgets + range, bound) + bound < kRangeLimit;
}

// add_radio_fixed_point's rounding; false for a contribution that int64 cannot hold.
__device__ __forceinline__ bool round_increment(double scaled, long long& increment) {
  if (!(fabs(scaled) < 9223372036854775808.)) return false;  // 2^63
  increment = static_cast<long long>(rint(scaled));
  return true;
}

// checked_radio_atomic_add: 1 if the sum left the range of int64.
__device__ __forceinline__ unsigned long long checked_add(long long* address, long long value) {
  long long const previous = static_cast<long long>(
      atomicAdd(reinterpret_cast<unsigned long long*>(address), static_cast<unsigned long long>(value)));
  return (value > 0 && previous > 0x7fffffffffffffffLL - value) ||
                 (value < 0 && previous < (-0x7fffffffffffffffLL - 1) - value)
             ? 1
             : 0;
}

// A CoREAS increment below 2^51 to a tile's bin past the thread's limit; `wave` is the bin's waveform.
__device__ __forceinline__ unsigned long long add_watched(long long* bin, long long* wave, long long value) {
  auto* const cell = reinterpret_cast<unsigned long long*>(bin);
  long long const sum = static_cast<long long>(atomicAdd(cell, static_cast<unsigned long long>(value))) + value;
  if (sum < kBinLimit && sum > -kBinLimit) return 0;
  return checked_add(wave, static_cast<long long>(atomicExch(cell, 0ull)));
}

// An observer's waveform rows for contributions past its tile. Read from the
// kernel's argument where they are needed: the compiler would otherwise hold
// them in scalar registers through the pair loop.
struct Rows {
  long long* row;
  std::uint64_t stride;
};
template <bool Zhs>
__device__ __forceinline__ Rows waveform_rows(std::uint32_t observer) {
  auto const* launch = (__attribute__((address_space(4))) ProjectionLaunch const*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(launch));
  auto* const waves = static_cast<long long*>(Zhs ? launch->zhs_waves : launch->coreas_waves);
  ObserverDev const* const observers = Zhs ? launch->zhs_observers : launch->coreas_observers;
  return {waves + observers[observer].waveform_offset, Zhs ? launch->zhs_total_bins : launch->coreas_total_bins};
}

// Adds a tile's rows to the global waveforms (checked int64 atomics, as
// checked_radio_atomic_add, counting overflows; or FP64 atomics in floating mode).
template <bool Fixed, class Acc>
__device__ __forceinline__ unsigned long long flush_tile(Acc const* lds, std::uint32_t row, std::uint32_t bins,
                                                         void* global, std::uint64_t total_bins, std::uint64_t first) {
  Acc* const g = static_cast<Acc*>(global);
  unsigned long long overflows = 0;
  for (std::uint32_t c = 0; c < 3; ++c) {
    for (std::uint32_t b = threadIdx.x; b < bins; b += blockDim.x) {
      Acc const v = lds[c * row + b];
      if (v == 0) continue;
      std::uint64_t const at = c * total_bins + first + b;
      if constexpr (Fixed) {
        overflows += checked_add(g + at, v);
      } else {
        atomicAdd(g + at, v);
      }
    }
  }
  return overflows;
}

// Tallies of a workgroup: CoREAS and ZHS contributions, subtracks, valid
// tracks and overflows.
struct BlockTallies {
  unsigned long long counts[5];
};

__device__ __forceinline__ void clear_tallies(BlockTallies& block) {
  if (threadIdx.x < 5) block.counts[threadIdx.x] = 0;
}

// One LDS add per wave and tally.
template <bool Coreas, bool Zhs>
__device__ __forceinline__ void add_tallies(BlockTallies& block, unsigned long long const counts[5]) {
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    if ((k == 0 && !Coreas) || ((k == 1 || k == 2) && !Zhs)) continue;
    unsigned long long const sum = wave_sum(counts[k]);
    if (threadIdx.x % 64 == 0 && sum) atomicAdd(&block.counts[k], sum);
  }
}

__device__ __forceinline__ void publish_tallies(BlockTallies const& block, CountersDev* counters) {
  if (threadIdx.x != 0) return;
  if (block.counts[0]) atomicAdd(&counters->coreas_contributions, block.counts[0]);
  if (block.counts[1]) atomicAdd(&counters->zhs_contributions, block.counts[1]);
  if (block.counts[2]) atomicAdd(&counters->zhs_subtracks, block.counts[2]);
  if (block.counts[3]) atomicAdd(&counters->valid_tracks, block.counts[3]);
  if (block.counts[4]) atomicAdd(&counters->fixed_point_overflows, block.counts[4]);
}

}  // namespace c8mi::radio
