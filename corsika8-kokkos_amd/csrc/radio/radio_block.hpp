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
        long long const previous = static_cast<long long>(
            atomicAdd(reinterpret_cast<unsigned long long*>(g + at), static_cast<unsigned long long>(v)));
        if ((v > 0 && previous > 0x7fffffffffffffffLL - v) || (v < 0 && previous < (-0x7fffffffffffffffLL - 1) - v))
          ++overflows;
      } else {
        atomicAdd(g + at, v);
      }
    }
  }
  return overflows;
}

// Tallies of a workgroup: CoREAS and ZHS contributions, subtracks, valid
// tracks, overflows, and the sums of |increments| of CoREAS and ZHS.
struct BlockTallies {
  unsigned long long counts[5];
  double abs_sums[2];
};

__device__ __forceinline__ void clear_tallies(BlockTallies& block) {
  if (threadIdx.x < 5) block.counts[threadIdx.x] = 0;
  if (threadIdx.x < 2) block.abs_sums[threadIdx.x] = 0.;
}

// One LDS add per wave and tally.
template <bool Coreas, bool Zhs>
__device__ __forceinline__ void add_tallies(BlockTallies& block, unsigned long long const counts[5],
                                            double const abs_sums[2]) {
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    if ((k == 0 && !Coreas) || ((k == 1 || k == 2) && !Zhs)) continue;
    unsigned long long const sum = wave_sum(counts[k]);
    if (threadIdx.x % 64 == 0 && sum) atomicAdd(&block.counts[k], sum);
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if ((k == 0 && !Coreas) || (k == 1 && !Zhs)) continue;
    double const sum = wave_sum(abs_sums[k]);
    if (threadIdx.x % 64 == 0) atomicAdd(&block.abs_sums[k], sum);
  }
}

// Integer sums are exact modulo 2^64; every LDS partial is bounded by the sum of
// |increments|, so a workgroup whose bound reaches 2^63 may have lost its result
// and is reported as an overflow (conservatively).
__device__ __forceinline__ void publish_tallies(BlockTallies const& block, CountersDev* counters) {
  if (threadIdx.x != 0) return;
  constexpr double kLimit = 9223372036854775808.;  // 2^63
  unsigned long long overflow = block.counts[4];
  if (block.abs_sums[0] >= kLimit || block.abs_sums[1] >= kLimit) ++overflow;
  if (block.counts[0]) atomicAdd(&counters->coreas_contributions, block.counts[0]);
  if (block.counts[1]) atomicAdd(&counters->zhs_contributions, block.counts[1]);
  if (block.counts[2]) atomicAdd(&counters->zhs_subtracks, block.counts[2]);
  if (block.counts[3]) atomicAdd(&counters->valid_tracks, block.counts[3]);
  if (overflow) atomicAdd(&counters->fixed_point_overflows, overflow);
}

}  // namespace c8mi::radio
