// The fast FP64 form of one track-antenna update (CoREAS endpoints, ZHS segments)
// into int64 fixed-point window tiles in LDS.
//
// Bound: VALU issue. Every expression is written for the fewest FP64
// instructions that keep FP64 accuracy; the exact form (radio_kernels.hip) keeps
// the reference's operation order instead. Against that order:
//  * one Newton step of third order after the hardware reciprocal / reciprocal
//    square root (both good to 2^-24, so the step leaves ~2^-70) instead of two
//    of second order;
//  * e x (e x b) = e (e.b) - b with the e.b of the Doppler factor, three fused
//    multiply-adds instead of two cross products;
//  * the fixed-point scale rides on the amplitude, so a sample's components are
//    its increments; their range checks are one comparison of the thread's sum;
//  * the first, middle and last bins of a ZHS segment share their difference-array
//    entries (four per component instead of six).
// Arrival times stay at FP64 accuracy: a sample is a spike in one bin, and a delay
// error of 1e-15 s at 15 km already moves samples across bin edges.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "radio_block.hpp"
#include "radio_device.hpp"

namespace c8mi::radio::fast {

inline constexpr double kC = 299792458.;
inline constexpr double kInvC = 1. / 299792458.;
inline constexpr double kPi = 3.141592653589793238462643383279502884;
inline constexpr double kChargeEm = 1.6021766208e-19 * (1. / (4. * kPi * 8.8541878128e-12 * kC));
inline constexpr double kCoreasThreshold = 1.e-3;
inline constexpr double kShift = 6755399441055744.;            // 1.5 * 2^52
inline constexpr long long kShiftBits = 0x4338000000000000LL;  // its bit pattern

struct V3 {
  double x, y, z;
};
__device__ __forceinline__ double dot(V3 a, V3 b) { return fma(a.x, b.x, fma(a.y, b.y, a.z * b.z)); }

// 1 / b for finite normal b != 0 (0 and infinities give NaN).
__device__ __forceinline__ double reciprocal(double b) {
  double const r = __builtin_amdgcn_rcp(b);
  double const e = fma(-b, r, 1.);
  return fma(r, fma(e, e, e), r);
}

// 1 / sqrt(x) for x > 0.
__device__ __forceinline__ double reciprocal_sqrt(double x) {
  double const y = __builtin_amdgcn_rsq(x);
  double const e = fma(-(x * y), y, 1.);
  return fma(y, e * fma(0.375, e, 0.5), y);
}

// One observer and window tile. Workgroups hold the same observers in every
// wave, so the fields of a uniform view come from scalar loads.
struct View {
  V3 position;
  double start, end, rate, grid, two_pi_over_wavelength;
  double tile_begin, tile_end;  // bins of the tile, [begin, end)
  double destination_height, destination_index;
  double n_destination, integrated_destination;
  double scale;  // fixed-point scale of the algorithm
};

// A point of a track and what the propagation table says at it, shared by all
// observers of the workgroup (the two table gathers of a point cost more than
// the rest of its propagation: one L2 line per lane each).
struct Source {
  V3 at;
  double index, integrated;
  double height;  // table cell, or the height of a point off the table
};
enum SourceKind : std::uint32_t { kInside = 0, kAbove = 1, kAtZero = 2, kBelow = 3 };

template <bool Homogeneous>
__device__ __forceinline__ Source make_source(PropagationDev const& p, V3 at, std::uint32_t& kind) {
  Source s;
  s.at = at;
  kind = kInside;
  if constexpr (Homogeneous) {
    s.index = p.homogeneous_index;
    s.integrated = s.height = 0.;
    return s;
  }
  double const height = (at.z - p.minimum_height) * p.inverse_step;
  std::uint64_t const last = p.table_size - 1;
  if (height > 0. && height + 0.5 < static_cast<double>(last)) {
    // the table has fewer than 2^32 entries (checked on the host)
    std::uint32_t const cell = static_cast<std::uint32_t>(height + 0.5);
    s.index = p.refractivity[cell] + 1.;
    s.integrated = p.integrated[cell];
    s.height = static_cast<double>(cell);
  } else if (height + 0.5 >= static_cast<double>(last)) {
    kind = kAbove;
    s.index = p.refractivity[last] + p.slope_n_upper * fabs((at.z - p.maximum_height) * p.inverse_step) + 1.;
    s.integrated = p.integrated[last] + p.slope_i_upper * fabs(p.maximum_height - at.z);
    s.height = height;
  } else if (height == 0.) {
    kind = kAtZero;
    s.index = 1.;
    s.integrated = p.integrated[0];
    s.height = height;
  } else {
    kind = kBelow;
    s.index = p.refractivity[0] + p.slope_n_lower * fabs(height) + 1.;
    s.integrated = p.integrated[0] + p.slope_i_lower * fabs(height);
    s.height = fabs(height);
  }
  return s;
}

struct Track {
  V3 start, end, beta;
  double t0, t1, duration;
  double amplitude;  // charge x weight / (4 pi eps0 c)
};

// `base`: the batch's tracks from the workgroup's current position on, `lane`
// the thread's offset in it: the uniform pointer stays in scalar registers.
__device__ __forceinline__ bool load_track(double const* __restrict__ base, std::uint64_t stride,
                                           std::uint32_t lane, Track& t) {
  t.start = {base[lane], (base + stride)[lane], (base + 2 * stride)[lane]};
  t.end = {(base + 3 * stride)[lane], (base + 4 * stride)[lane], (base + 5 * stride)[lane]};
  t.t0 = (base + 6 * stride)[lane];
  t.t1 = (base + 7 * stride)[lane];
  t.amplitude = kChargeEm * (base + 8 * stride)[lane];
  t.duration = t.t1 - t.t0;
  V3 const d{t.end.x - t.start.x, t.end.y - t.start.y, t.end.z - t.start.z};
  if (!(t.duration > 0.) || !(dot(d, d) > 0.)) return false;
  double const c_duration = kC * t.duration;
  double r = __builtin_amdgcn_rcp(c_duration);
  double const e = fma(-c_duration, r, 1.);
  // an infinite product keeps the hardware result (0) instead of NaN
  r = isfinite(c_duration) ? fma(r, fma(e, e, e), r) : r;
  t.beta = {d.x * r, d.y * r, d.z * r};
  return true;
}
__device__ __forceinline__ V3 midpoint(Track const& t) {
  return {(t.start.x + t.end.x) * 0.5, (t.start.y + t.end.y) * 0.5, (t.start.z + t.end.z) * 0.5};
}

struct Path {
  double time, inv_distance;
  V3 emit;
};

// The reference's edge branches (RadioProjection.inl:170-238).
__device__ __forceinline__ double edge_mean_index(View const& o, Source const& s, std::uint32_t kind) {
  double const span = kind == kAbove ? s.height - o.destination_height : o.destination_height - s.height;
  return 1. + (s.integrated - o.integrated_destination) / span;
}

template <bool Homogeneous>
__device__ __forceinline__ Path propagate(PropagationDev const& p, View const& o, Source const& s,
                                          std::uint32_t kind) {
  Path r;
  V3 const d{o.position.x - s.at.x, o.position.y - s.at.y, o.position.z - s.at.z};
  double const r2 = dot(d, d);
  r.inv_distance = reciprocal_sqrt(r2);
  r.emit = {d.x * r.inv_distance, d.y * r.inv_distance, d.z * r.inv_distance};
  double const distance = r2 * r.inv_distance;
  if constexpr (Homogeneous) {
    r.time = s.index * distance * kInvC;  // the reference's order: see segment_arrival
    return r;
  }
  double const cells = s.height - o.destination_index;
  double const span = cells == 0. ? 1. : cells * p.step;
  double mean = fma(s.integrated - o.integrated_destination, reciprocal(span), 1.);
  if (kind != kInside) mean = edge_mean_index(o, s, kind);
  r.time = mean * (distance * kInvC);
  return r;
}

// Index at the observer as the reference's propagation gives it: 1 for sources
// at or below the table's lower end.
template <bool Homogeneous>
__device__ __forceinline__ double index_at_destination(PropagationDev const& p, View const& o, std::uint32_t kind) {
  if constexpr (Homogeneous) return p.homogeneous_index;
  return kind >= kAtZero ? 1. : o.n_destination;
}

// 1 - n b.e, with error-free products and sums where it cancels to zero.
__device__ __forceinline__ double cancelled_doppler(double index, V3 beta, V3 emit) {
  double const px = beta.x * emit.x, py = beta.y * emit.y, pz = beta.z * emit.z;
  double const ex = fma(beta.x, emit.x, -px);
  double const ey = fma(beta.y, emit.y, -py);
  double const ez = fma(beta.z, emit.z, -pz);
  double const xy = px + py;
  double const xyv = xy - px;
  double const xye = (px - (xy - xyv)) + (py - xyv);
  double const xyz = xy + pz;
  double const xyzv = xyz - xy;
  double const xyze = (xy - (xyz - xyzv)) + (pz - xyzv);
  double const low = ex + ey + ez + xye + xyze;
  double const product = index * xyz;
  double const perr = fma(index, xyz, -product) + index * low;
  return (1. - product) - perr;
}
__device__ __forceinline__ double doppler(double index, V3 beta, V3 emit, double beta_emit) {
  double const ordinary = fma(-index, beta_emit, 1.);
  if (ordinary != 0.) return ordinary;
  return cancelled_doppler(index, beta, emit);
}

// Per-thread tallies. The 32-bit counts cannot wrap: a workgroup takes at most
// 2^27 tracks (kMaxChunkTracks) of 8 observers (kMaxGroup), a thread 2^22 of the pairs.
struct Tally {
  std::uint32_t coreas = 0, single_subtracks = 0, valid = 0;
  unsigned long long zhs = 0, subtracks = 0, overflow = 0;
  double coreas_abs = 0., zhs_abs = 0.;  // sums of |increments|, for kThreadLimit
};

// What an observer's contributions past the thread's limit need.
struct Excess {
  std::uint32_t observer;
  Budget* budgets;  // ZHS: of the observer's ranges
};

// Round to nearest even below 2^51 (kThreadLimit): the same as rint.
__device__ __forceinline__ long long increment(double scaled) {
  return __double_as_longlong(scaled + kShift) - kShiftBits;
}
__device__ __forceinline__ void lds_add(long long* address, long long value) {
  atomicAdd(reinterpret_cast<unsigned long long*>(address), static_cast<unsigned long long>(value));
}

// One CoREAS sample: scaled components c at arrival `time` (no sample outside
// the window or the tile).
__device__ __forceinline__ void add_field(View const& o, long long* tile, std::uint32_t stride, double time,
                                          V3 c, Excess const& excess, Tally& tally) {
  if (!(time >= o.start && time <= o.end)) return;
  double const bin = floor(fma(time - o.start, o.rate, 0.5));
  if (!(bin >= o.tile_begin && bin < o.tile_end)) return;
  std::uint32_t const at = static_cast<std::uint32_t>(bin - o.tile_begin);
  double const magnitude = fabs(c.x) + fabs(c.y) + fabs(c.z);
  tally.coreas_abs += magnitude;
  if (__builtin_expect(tally.coreas_abs < kThreadLimit, 1)) {
    lds_add(tile + at, increment(c.x));
    lds_add(tile + stride + at, increment(c.y));
    lds_add(tile + 2 * stride + at, increment(c.z));
    ++tally.coreas;
    return;
  }
  Rows const waves = waveform_rows<false>(excess.observer);
  long long* const wave = waves.row + static_cast<std::uint64_t>(bin);
  double const cs[3] = {c.x, c.y, c.z};
  bool valid = true;
  unsigned long long overflows = 0;
  for (int k = 0; k < 3; ++k) {
    long long value = 0;
    if (!round_increment(cs[k], value)) valid = false;
    else if (magnitude < kThreadLimit) overflows += add_watched(tile + k * stride + at, wave + k * waves.stride, value);
    else overflows += checked_add(wave + k * waves.stride, value);
  }
  tally.overflow += overflows + (valid ? 0ull : 1ull);
  tally.coreas += valid ? 1u : 0u;
}

__device__ __forceinline__ double nearest_bin(double x) { return floor(x + 0.5); }

// separate_same_bin_endpoints (RadioProjection.inl:303-336).
__device__ __forceinline__ void separate_same_bin(double& start_time, double& end_time, View const& o,
                                                  bool signed_order) {
  double const s = start_time * o.rate;
  double const e = end_time * o.rate;
  if (nearest_bin(s) != nearest_bin(e)) return;
  double const sf = s - floor(s);
  double const ef = e - floor(e);
  bool const forward = !signed_order || end_time >= start_time;
  if (forward) {
    if (sf >= 0.5 && ef >= 0.5) start_time -= o.grid;
    else if (sf < 0.5 && ef < 0.5) end_time += o.grid;
    else if (ef >= 1. - sf) end_time += o.grid;
    else start_time -= o.grid;
  } else {
    if (sf >= 0.5 && ef >= 0.5) end_time -= o.grid;
    else if (sf < 0.5 && ef < 0.5) start_time += o.grid;
    else if (sf >= 1. - ef) start_time += o.grid;
    else end_time -= o.grid;
  }
}

__device__ __forceinline__ V3 scaled(V3 a, double s) { return {a.x * s, a.y * s, a.z * s}; }

// e x (e x b) s
__device__ __forceinline__ V3 transverse(V3 emit, V3 beta, double beta_emit, double s) {
  return {fma(emit.x, beta_emit, -beta.x) * s, fma(emit.y, beta_emit, -beta.y) * s,
          fma(emit.z, beta_emit, -beta.z) * s};
}

// The CoREAS update of a track whose endpoints see no small Doppler factor;
// returns true without adding anything where one does (`forward`: the start
// arrives before the end), for coreas_near.
template <bool Homogeneous>
__device__ __forceinline__ bool coreas_far(Track const& t, Source const& start, std::uint32_t start_kind,
                                           Source const& end, std::uint32_t end_kind, PropagationDev const& p,
                                           View const& o, long long* tile, std::uint32_t stride,
                                           Excess const& excess, Tally& tally, bool& forward) {
  Path const ps = propagate<Homogeneous>(p, o, start, start_kind);
  Path const pe = propagate<Homogeneous>(p, o, end, end_kind);
  double const bs = dot(t.beta, ps.emit), be = dot(t.beta, pe.emit);
  double const pre = doppler(start.index, t.beta, ps.emit, bs);
  double const post = doppler(end.index, t.beta, pe.emit, be);
  double start_receive = t.t0 + ps.time;
  double end_receive = t.t1 + pe.time;
  if (index_at_destination<Homogeneous>(p, o, start_kind) > 1. &&
      (fabs(pre) < kCoreasThreshold || fabs(post) < kCoreasThreshold)) {
    forward = start_receive < end_receive;
    return true;
  }
  double const q = t.amplitude * o.rate * o.scale;
  V3 fs = transverse(ps.emit, t.beta, bs, q * ps.inv_distance * reciprocal(pre));
  V3 fe = transverse(pe.emit, t.beta, be, -(q * pe.inv_distance * reciprocal(post)));
  if (pre < 1.e-9 || post < 1.e-9) {
    double const delta = end_receive - start_receive;
    if (fabs(delta) < o.grid) {
      double const shrink = fabs(delta * o.rate);
      fs = scaled(fs, shrink);
      fe = scaled(fe, shrink);
      separate_same_bin(start_receive, end_receive, o, false);
    }
  }
  add_field(o, tile, stride, start_receive, fs, excess, tally);
  add_field(o, tile, stride, end_receive, fe, excess, tally);
  return false;
}

// The CoREAS update near the Cherenkov angle: both samples from the midpoint.
template <bool Homogeneous>
__device__ __forceinline__ void coreas_near(Track const& t, PropagationDev const& p, View const& o,
                                            long long* tile, std::uint32_t stride, Excess const& excess,
                                            Tally& tally, bool forward) {
  std::uint32_t kind;
  Source const middle = make_source<Homogeneous>(p, midpoint(t), kind);
  Path const pm = propagate<Homogeneous>(p, o, middle, kind);
  double const middle_receive = (t.t0 + t.t1) * 0.5 + pm.time;
  double const bm = dot(t.beta, pm.emit);
  double const md = doppler(middle.index, t.beta, pm.emit, bm);
  V3 f = transverse(pm.emit, t.beta, bm, t.amplitude * o.rate * o.scale * pm.inv_distance * reciprocal(md));
  double const half = 0.5 * (t.duration * fabs(md));
  double start_receive = forward ? middle_receive - half : middle_receive + half;
  double end_receive = forward ? middle_receive + half : middle_receive - half;
  double const delta = end_receive - start_receive;
  if (fabs(delta) < o.grid) {
    f = scaled(f, fabs(delta * o.rate));
    separate_same_bin(start_receive, end_receive, o, true);
  }
  add_field(o, tile, stride, start_receive, f, excess, tally);
  add_field(o, tile, stride, end_receive, {-f.x, -f.y, -f.z}, excess, tally);
}

// One component row of a ZHS segment over bins l1 (first), l1 + 1 .. l2 - 1
// (middle) and l2 (last), relative to the tile of `bins` bins: the entries of
// the difference array, clipped to the tile (an entry before it acts from its
// first bin on, one behind it is dropped).
__device__ __forceinline__ void add_segment_row(long long* row, std::int32_t bins, std::int32_t l1,
                                                std::int32_t l2, long long first, long long middle,
                                                long long last) {
  auto add = [&](std::int32_t at, unsigned long long value) {  // modulo 2^64
    if (at < bins) lds_add(row + (at > 0 ? at : 0), static_cast<long long>(value));
  };
  auto const f = static_cast<unsigned long long>(first), m = static_cast<unsigned long long>(middle),
             l = static_cast<unsigned long long>(last);
  add(l1, f);
  if (l2 - l1 > 1) {
    add(l1 + 1, m - f);
    add(l2, l - m);
  } else {
    add(l1 + 1, l - f);
  }
  add(l2 + 1, 0ull - l);
}

// Arrival of a ZHS segment at the observer, in seconds and bins, in the
// reference's order: near the Cherenkov angle the difference of the two times is
// the rounding of each, divided by 1 - n e.b, and a mathematically equal form
// (midpoint -+ half the spread, or the duration in one bin) rounds differently:
// 1e-8 to 1e-7 of the field of an in-ice track list against 1e-9 to 9e-9.
struct Arrival {
  double d1, d2, x1, x2, b1, b2, den;
};
__device__ __forceinline__ Arrival segment_arrival(Path const& path, double index, double beta_emit,
                                                   double time1, double time2, View const& o) {
  Arrival a;
  double const slope = index * beta_emit;
  a.den = 1. - slope;
  double const middle = (time1 + time2) * 0.5;
  double const first = time1 + path.time - slope * (time1 - middle);
  double const second = time2 + path.time - slope * (time2 - middle);
  a.d1 = first > second ? second : first;
  a.d2 = first > second ? first : second;
  a.x1 = (a.d1 - o.start) * o.rate;
  a.x2 = (a.d2 - o.start) * o.rate;
  a.b1 = nearest_bin(a.x1);
  a.b2 = nearest_bin(a.x2);
  return a;
}

// A segment over one bin or two neighbouring ones, as the difference array's
// entries at the first bin and the two after it. u: e x (b x e) times the
// amplitude over the distance.
__device__ __forceinline__ void add_short_segment(V3 u, double duration, Arrival const& a, View const& o,
                                                  long long* tile, std::uint32_t stride, Excess const& excess,
                                                  Tally& tally) {
  bool const two = a.b1 != a.b2;
  double const k = reciprocal(fabs(a.den));
  std::int32_t const bins = static_cast<std::int32_t>(o.tile_end - o.tile_begin);
  std::int32_t const at = static_cast<std::int32_t>(a.b1 - o.tile_begin);  // -1 .. bins - 1
  bool const has_first = at >= 0, has_last = two && at + 1 < bins;
  // a part without its bin in this tile takes no part in the sums
  double const whole = fabs(a.den) > 1.e-15 ? fabs(a.d2 * o.rate - a.d1 * o.rate) * k : duration * o.rate;
  double const first = !has_first ? 0. : two ? (a.b1 + 0.5 - a.x1) * k : whole;
  double const last = has_last ? (a.x2 + 0.5 - a.b2) * k : 0.;
  double const bound = (fabs(u.x) + fabs(u.y) + fabs(u.z)) * (fabs(first) + fabs(last));
  std::uint32_t const base = at > 0 ? static_cast<std::uint32_t>(at) : 0u;
  std::uint32_t const n = (has_first ? 1u : 0u) + (has_last ? 1u : 0u);
  tally.zhs_abs += bound;
  double const us[3] = {u.x, u.y, u.z};
  if (__builtin_expect(tally.zhs_abs < kThreadLimit, 1)) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      long long* const row = tile + c * stride + base;
      long long const f = increment(us[c] * first), l = increment(us[c] * last);
      if (has_first) {
        lds_add(row, f);
        lds_add(row + 1, l - f);
        if (has_last) lds_add(row + 2, -l);
      } else {
        lds_add(row, l);
        lds_add(row + 1, -l);
      }
    }
    tally.zhs += n;
    return;
  }
  // the bins of the parts that are there (n of them, from `base` or the next on)
  std::uint32_t const from = has_first ? base : static_cast<std::uint32_t>(at + 1);
  bool const in_tile = n != 0 && tile_takes(excess.budgets, from, from + n - 1, static_cast<std::uint32_t>(bins), bound);
  Rows const waves = waveform_rows<true>(excess.observer);
  std::int64_t const bin = static_cast<std::int64_t>(o.tile_begin) + at;
  bool vf = true, vl = true;
  unsigned long long overflows = 0;
  for (int c = 0; c < 3; ++c) {
    long long* const row = tile + c * stride;
    long long* const wave = waves.row + c * waves.stride + bin;
    auto add = [&](bool has, int ahead, double value, bool& valid) {
      long long v = 0;
      if (!has) return;
      if (!round_increment(value, v)) {
        valid = false;
      } else if (in_tile) {
        lds_add(row + at + ahead, v);
        lds_add(row + at + ahead + 1, -v);
      } else {
        overflows += checked_add(wave + ahead, v);
      }
    };
    add(has_first, 0, us[c] * first, vf);
    add(has_last, 1, us[c] * last, vl);
  }
  unsigned long long const nf = has_first ? 1ull : 0ull, nl = has_last ? 1ull : 0ull;
  tally.zhs += (vf ? nf : 0ull) + (vl ? nl : 0ull);
  tally.overflow += overflows + (vf ? 0ull : nf) + (vl ? 0ull : nl);
}

// One ZHS segment of any length. `subdivided` keeps the reference's sign of the
// middle bins.
__device__ __forceinline__ void zhs_segment(Path const& path, double index, double beta_emit, double time1,
                                            double time2, Track const& t, View const& o,
                                            long long* tile, std::uint32_t stride, Excess const& excess, Tally& tally,
                                            bool subdivided) {
  Arrival const a = segment_arrival(path, index, beta_emit, time1, time2, o);
  if (!(a.b2 >= o.tile_begin && a.b1 < o.tile_end)) return;
  V3 const u = transverse(path.emit, t.beta, beta_emit, -(t.amplitude * path.inv_distance * o.scale));
  if (a.b2 - a.b1 <= 1.) {
    add_short_segment(u, time2 - time1, a, o, tile, stride, excess, tally);
    return;
  }
  std::int32_t const bins = static_cast<std::int32_t>(o.tile_end - o.tile_begin);
  // two bins either side of the tile tell everything the clipping needs
  std::int32_t const l1 = static_cast<std::int32_t>(fmax(a.b1 - o.tile_begin, -2.));
  std::int32_t const l2 = static_cast<std::int32_t>(fmin(a.b2 - o.tile_begin, static_cast<double>(bins) + 1.));
  V3 const edge = scaled(u, reciprocal(fabs(a.den)));
  bool const has_first = l1 >= 0, has_last = l2 < bins;
  std::int32_t const middle_bins = (l2 < bins ? l2 : bins) - (l1 + 1 > 0 ? l1 + 1 : 0);
  bool const has_middle = l2 - l1 > 1 && middle_bins > 0;
  // a part without bins in this tile takes no part in the sums
  double const first = has_first ? fabs(a.b1 + 0.5 - a.x1) : 0.;
  double const middle = has_middle ? (subdivided && a.den < 0. ? -1. : 1.) : 0.;
  double const last = has_last ? fabs(a.x2 + 0.5 - a.b2) : 0.;
  unsigned long long const nm = has_middle ? static_cast<unsigned long long>(middle_bins) : 0ull;
  unsigned long long const nf = has_first ? 1ull : 0ull, nl = has_last ? 1ull : 0ull;
  double const bound = (fabs(edge.x) + fabs(edge.y) + fabs(edge.z)) * (first + fabs(middle) + last);
  tally.zhs_abs += bound;
  double const es[3] = {edge.x, edge.y, edge.z};
  if (__builtin_expect(tally.zhs_abs < kThreadLimit, 1)) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
      add_segment_row(tile + c * stride, bins, l1, l2, increment(es[c] * first), increment(es[c] * middle),
                      increment(es[c] * last));
    tally.zhs += nf + nm + nl;
    return;
  }
  std::int32_t const from = l1 > 0 ? l1 : 0, to = l2 < bins ? l2 : bins - 1;
  Rows const waves = waveform_rows<true>(excess.observer);
  std::int64_t const begin = static_cast<std::int64_t>(o.tile_begin);
  bool vf = true, vm = true, vl = true;
  unsigned long long overflows = 0;
  for (int c = 0; c < 3; ++c) {
    long long f = 0, m = 0, l = 0;
    vf = round_increment(es[c] * first, f) && vf;
    vm = round_increment(es[c] * middle, m) && vm;
    vl = round_increment(es[c] * last, l) && vl;
    long long* const wave = waves.row + c * waves.stride + begin;
    for (std::int32_t b = from; b <= to; ++b) {
      long long const v = b == l1 ? f : b == l2 ? l : m;
      if (v != 0) overflows += checked_add(wave + b, v);
    }
  }
  tally.zhs += (vf ? nf : 0ull) + (vm ? nm : 0ull) + (vl ? nl : 0ull);
  tally.overflow += overflows + (vf ? 0ull : nf) + (vm ? 0ull : nm) + (vl ? 0ull : nl);
}

// The Fraunhofer measure of a track (RadioProjection.inl:482-529): above one it
// is subdivided. sin^2 L^2 = L^2 - (d.e)^2 with d = beta c duration.
__device__ __forceinline__ double fraunhofer(Path const& path, double beta_emit, double duration, double length2,
                                             View const& o) {
  double const along = beta_emit * (kC * duration);
  return fma(-along, along, length2) * path.inv_distance * o.two_pi_over_wavelength;
}

// The ZHS update of a track from its midpoint (`length2`: its squared length).
template <bool Homogeneous>
__device__ __forceinline__ void zhs_update(Track const& t, Source const& middle, std::uint32_t kind, double length2,
                                           PropagationDev const& p, std::uint32_t refinement, View const& o,
                                           long long* tile, std::uint32_t stride, Excess const& excess,
                                           Tally& tally, bool count_subtracks) {
  Path const mp = propagate<Homogeneous>(p, o, middle, kind);
  double const bm = dot(t.beta, mp.emit);
  double const measure = fraunhofer(mp, bm, t.duration, length2, o);
  if (!(measure > 1.) && refinement <= 1u) {
    if (count_subtracks) ++tally.single_subtracks;
    zhs_segment(mp, middle.index, bm, t.t0, t.t1, t, o, tile, stride, excess, tally, false);
    return;
  }
  double divisor = 1.;
  int nsub = 1;
  if (measure > 1.) {
    divisor = sqrt(measure) + 1.;
    nsub = static_cast<int>(ceil(divisor));
  }
  int const refine = static_cast<int>(refinement);
  if (count_subtracks) {
    tally.subtracks += static_cast<unsigned long long>(nsub);
    if (refine > 1) tally.subtracks += static_cast<unsigned long long>(nsub * (refine - 1));
  }
  int const segments = nsub * refine;
  double const parts = divisor * static_cast<double>(refine);
  V3 const step{(t.end.x - t.start.x) / parts, (t.end.y - t.start.y) / parts, (t.end.z - t.start.z) / parts};
  double const dt = t.duration / parts;
  V3 p1 = t.start;
  double time1 = t.t0;
  for (int i = 0; i < segments; ++i) {
    V3 const p2{p1.x + step.x, p1.y + step.y, p1.z + step.z};
    double const time2 = time1 + dt;
    std::uint32_t part_kind;
    Source const part =
        make_source<Homogeneous>(p, {(p1.x + p2.x) * 0.5, (p1.y + p2.y) * 0.5, (p1.z + p2.z) * 0.5}, part_kind);
    Path const path = propagate<Homogeneous>(p, o, part, part_kind);
    zhs_segment(path, part.index, dot(t.beta, path.emit), time1, time2, t, o, tile, stride, excess, tally, true);
    p1 = p2;
    time1 = time2;
  }
}

}  // namespace c8mi::radio::fast
