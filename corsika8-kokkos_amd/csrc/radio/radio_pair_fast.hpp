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
//    its increments; the three range checks are one comparison of their sum;
//  * a ZHS segment's arrival times are its midpoint's -+ (half duration)
//    |1 - n e.b|; in one bin the denominator cancels (no reciprocal);
//  * the first, middle and last bins of a ZHS segment share their difference-array
//    entries (four per component instead of six).
// Arrival times stay at FP64 accuracy: a sample is a spike in one bin, and a delay
// error of 1e-15 s at 15 km already moves samples across bin edges.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "radio_device.hpp"

namespace c8mi::radio::fast {

inline constexpr double kC = 299792458.;
inline constexpr double kInvC = 1. / 299792458.;
inline constexpr double kPi = 3.141592653589793238462643383279502884;
inline constexpr double kChargeEm = 1.6021766208e-19 * (1. / (4. * kPi * 8.8541878128e-12 * kC));
inline constexpr double kCoreasThreshold = 1.e-3;
inline constexpr double kIntLimit = 9223372036854775808.;      // 2^63
inline constexpr double kShiftLimit = 2251799813685248.;       // 2^51
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

// What a workgroup knows of its observer and window tile (uniform).
struct View {
  V3 position;
  double start, end, rate, grid, two_pi_over_wavelength;
  double tile_begin, tile_end;  // bins of the tile, [begin, end)
  double table_last;            // last propagation-table entry
  double destination_height, destination_index;
  double n_destination, integrated_destination;
  double coreas_scale, zhs_scale;
};

struct Track {
  V3 start, end, beta;
  double t0, t1, duration;
  double constant;  // charge x weight / (4 pi eps0 c)
};

// `base`: the batch's tracks from the workgroup's current position on, `lane`
// the thread's offset in it: the uniform pointer stays in scalar registers.
__device__ __forceinline__ bool load_track(double const* __restrict__ base, std::uint64_t stride,
                                           std::uint32_t lane, Track& t) {
  t.start = {base[lane], (base + stride)[lane], (base + 2 * stride)[lane]};
  t.end = {(base + 3 * stride)[lane], (base + 4 * stride)[lane], (base + 5 * stride)[lane]};
  t.t0 = (base + 6 * stride)[lane];
  t.t1 = (base + 7 * stride)[lane];
  t.constant = kChargeEm * (base + 8 * stride)[lane];
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

struct Path {
  double time, n_source, n_destination, inv_distance;
  V3 emit;
};

// Sources above, at or below the ends of the propagation table (the
// reference's edge branches; RadioProjection.inl:170-238).
__device__ __forceinline__ double edge_mean_index(PropagationDev const& p, View const& o, double source_z,
                                                  double source_height, double& n_source,
                                                  double& n_destination) {
  std::uint64_t const last = p.table_size - 1;
  double integrated, height;
  if (source_height + 0.5 >= o.table_last) {
    n_source = p.refractivity[last] + p.slope_n_upper * fabs((source_z - p.maximum_height) * p.inverse_step) + 1.;
    integrated = p.integrated[last] + p.slope_i_upper * fabs(p.maximum_height - source_z);
    height = source_height - o.destination_height;
  } else if (source_height == 0.) {
    n_source = 1.;
    n_destination = 1.;
    integrated = p.integrated[0];
    height = o.destination_height - source_height;
  } else {
    n_source = p.refractivity[0] + p.slope_n_lower * fabs(source_height) + 1.;
    integrated = p.integrated[0] + p.slope_i_lower * fabs(source_height);
    n_destination = 1.;
    height = o.destination_height - fabs(source_height);
  }
  return 1. + (integrated - o.integrated_destination) / height;
}

template <bool Homogeneous>
__device__ __forceinline__ Path propagate(PropagationDev const& p, View const& o, V3 source) {
  Path r;
  V3 const d{o.position.x - source.x, o.position.y - source.y, o.position.z - source.z};
  double const r2 = dot(d, d);
  r.inv_distance = reciprocal_sqrt(r2);
  r.emit = {d.x * r.inv_distance, d.y * r.inv_distance, d.z * r.inv_distance};
  double const flight = (r2 * r.inv_distance) * kInvC;
  if constexpr (Homogeneous) {
    r.n_source = r.n_destination = p.homogeneous_index;
    r.time = p.homogeneous_index * flight;
    return r;
  }
  double const height = (source.z - p.minimum_height) * p.inverse_step;
  double mean;
  r.n_destination = o.n_destination;
  if (height > 0. && height + 0.5 < o.table_last) {
    // the table has fewer than 2^32 entries (checked on the host)
    std::uint32_t const at = static_cast<std::uint32_t>(height + 0.5);
    r.n_source = p.refractivity[at] + 1.;
    double const difference = p.integrated[at] - o.integrated_destination;
    double const cells = static_cast<double>(at) - o.destination_index;
    double const span = cells == 0. ? 1. : cells * p.step;
    mean = fma(difference, reciprocal(span), 1.);
  } else {
    mean = edge_mean_index(p, o, source.z, height, r.n_source, r.n_destination);
  }
  r.time = mean * flight;
  return r;
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
// 2^30 tracks (kMaxChunkTracks), a thread 2^22 of them.
struct Tally {
  std::uint32_t coreas = 0, single_subtracks = 0, valid = 0;
  unsigned long long zhs = 0, subtracks = 0, overflow = 0;
  double coreas_abs = 0., zhs_abs = 0.;  // sums of |increments|: bound every LDS partial sum
};

__device__ __forceinline__ long long increment(double scaled) {
  return __double_as_longlong(scaled + kShift) - kShiftBits;
}
__device__ __forceinline__ void lds_add(long long* address, long long value) {
  atomicAdd(reinterpret_cast<unsigned long long*>(address), static_cast<unsigned long long>(value));
}

// A component beyond the shift form: rounded by rint below 2^63, else refused.
__device__ __forceinline__ bool checked_increment(double scaled, long long& inc, double& abs_sum) {
  double const magnitude = fabs(scaled);
  if (magnitude < kShiftLimit) {
    inc = increment(scaled);
  } else {
    if (!(magnitude < kIntLimit)) return false;
    inc = static_cast<long long>(rint(scaled));
  }
  abs_sum += magnitude;
  return true;
}

// One CoREAS sample: scaled components c at arrival `time` (no sample outside
// the window or the tile).
__device__ __forceinline__ void add_field(View const& o, long long* tile, std::uint32_t stride, double time,
                                          V3 c, Tally& tally) {
  if (!(time >= o.start && time <= o.end)) return;
  double const bin = floor(fma(time - o.start, o.rate, 0.5));
  if (!(bin >= o.tile_begin && bin < o.tile_end)) return;
  std::uint32_t const at = static_cast<std::uint32_t>(bin - o.tile_begin);
  double const magnitude = fabs(c.x) + fabs(c.y) + fabs(c.z);
  if (magnitude < kShiftLimit) {
    tally.coreas_abs += magnitude;
    lds_add(tile + at, increment(c.x));
    lds_add(tile + stride + at, increment(c.y));
    lds_add(tile + 2 * stride + at, increment(c.z));
    ++tally.coreas;
    return;
  }
  long long ix = 0, iy = 0, iz = 0;
  bool const vx = checked_increment(c.x, ix, tally.coreas_abs);
  bool const vy = checked_increment(c.y, iy, tally.coreas_abs);
  bool const vz = checked_increment(c.z, iz, tally.coreas_abs);
  if (vx) lds_add(tile + at, ix);
  if (vy) lds_add(tile + stride + at, iy);
  if (vz) lds_add(tile + 2 * stride + at, iz);
  bool const valid = vx && vy && vz;
  tally.overflow += valid ? 0ull : 1ull;
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
__device__ __forceinline__ bool coreas_far(Track const& t, PropagationDev const& p, View const& o,
                                           long long* tile, std::uint32_t stride, Tally& tally, bool& forward) {
  Path const ps = propagate<Homogeneous>(p, o, t.start);
  Path const pe = propagate<Homogeneous>(p, o, t.end);
  double const bs = dot(t.beta, ps.emit), be = dot(t.beta, pe.emit);
  double const pre = doppler(ps.n_source, t.beta, ps.emit, bs);
  double const post = doppler(pe.n_source, t.beta, pe.emit, be);
  double start_receive = t.t0 + ps.time;
  double end_receive = t.t1 + pe.time;
  if (ps.n_destination > 1. && (fabs(pre) < kCoreasThreshold || fabs(post) < kCoreasThreshold)) {
    forward = start_receive < end_receive;
    return true;
  }
  double const q = t.constant * o.rate * o.coreas_scale;
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
  add_field(o, tile, stride, start_receive, fs, tally);
  add_field(o, tile, stride, end_receive, fe, tally);
  return false;
}

// The CoREAS update near the Cherenkov angle: both samples from the midpoint.
template <bool Homogeneous>
__device__ __forceinline__ void coreas_near(Track const& t, PropagationDev const& p, View const& o,
                                            long long* tile, std::uint32_t stride, Tally& tally, bool forward) {
  V3 const midpoint{(t.start.x + t.end.x) * 0.5, (t.start.y + t.end.y) * 0.5, (t.start.z + t.end.z) * 0.5};
  Path const pm = propagate<Homogeneous>(p, o, midpoint);
  double const middle = (t.t0 + t.t1) * 0.5 + pm.time;
  double const bm = dot(t.beta, pm.emit);
  double const md = doppler(pm.n_source, t.beta, pm.emit, bm);
  V3 f = transverse(pm.emit, t.beta, bm, t.constant * o.rate * o.coreas_scale * pm.inv_distance * reciprocal(md));
  double const half = 0.5 * (t.duration * fabs(md));
  double start_receive = forward ? middle - half : middle + half;
  double end_receive = forward ? middle + half : middle - half;
  double const delta = end_receive - start_receive;
  if (fabs(delta) < o.grid) {
    f = scaled(f, fabs(delta * o.rate));
    separate_same_bin(start_receive, end_receive, o, true);
  }
  add_field(o, tile, stride, start_receive, f, tally);
  add_field(o, tile, stride, end_receive, {-f.x, -f.y, -f.z}, tally);
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

// One ZHS segment from its midpoint's path: half_duration either side of
// middle_time. `subdivided` keeps the reference's sign of the middle bins.
__device__ __forceinline__ void zhs_segment(Path const& path, double beta_emit, double middle_time,
                                            double half_duration, Track const& t, View const& o,
                                            long long* tile, std::uint32_t stride, Tally& tally,
                                            bool subdivided) {
  double const den = fma(-path.n_source, beta_emit, 1.);
  double const spread = half_duration * fabs(den);
  double const centre = middle_time + path.time;
  double const x1 = ((centre - spread) - o.start) * o.rate;
  double const x2 = ((centre + spread) - o.start) * o.rate;
  double const b1 = nearest_bin(x1), b2 = nearest_bin(x2);
  if (!(b2 >= o.tile_begin && b1 < o.tile_end)) return;
  double const base = t.constant * path.inv_distance * o.zhs_scale;
  // e x (b x e)
  V3 const u = transverse(path.emit, t.beta, beta_emit, -base);
  if (b1 == b2) {
    V3 const c = scaled(u, 2. * half_duration * o.rate);
    std::uint32_t const at = static_cast<std::uint32_t>(b2 - o.tile_begin);
    double const magnitude = fabs(c.x) + fabs(c.y) + fabs(c.z);
    if (magnitude < kShiftLimit) {
      tally.zhs_abs += magnitude;
      long long const ix = increment(c.x), iy = increment(c.y), iz = increment(c.z);
      lds_add(tile + at, ix);
      lds_add(tile + at + 1, -ix);
      lds_add(tile + stride + at, iy);
      lds_add(tile + stride + at + 1, -iy);
      lds_add(tile + 2 * stride + at, iz);
      lds_add(tile + 2 * stride + at + 1, -iz);
      ++tally.zhs;
      return;
    }
    double const cs[3] = {c.x, c.y, c.z};
    bool valid = true;
    for (int k = 0; k < 3; ++k) {
      long long inc = 0;
      if (checked_increment(cs[k], inc, tally.zhs_abs)) {
        lds_add(tile + k * stride + at, inc);
        lds_add(tile + k * stride + at + 1, -inc);
      } else {
        valid = false;
      }
    }
    tally.zhs += valid ? 1ull : 0ull;
    tally.overflow += valid ? 0ull : 1ull;
    return;
  }
  std::int32_t const bins = static_cast<std::int32_t>(o.tile_end - o.tile_begin);
  // two bins either side of the tile tell everything the clipping needs
  std::int32_t const l1 = static_cast<std::int32_t>(fmax(b1 - o.tile_begin, -2.));
  std::int32_t const l2 = static_cast<std::int32_t>(fmin(b2 - o.tile_begin, static_cast<double>(bins) + 1.));
  double const k = reciprocal(fabs(den));
  V3 const edge = scaled(u, k);
  double const first = fabs(b1 + 0.5 - x1), last = fabs(x2 + 0.5 - b2);
  double const sign = subdivided && den < 0. ? -1. : 1.;
  bool const has_first = l1 >= 0, has_last = l2 < bins;
  std::int32_t const middle_bins = (l2 < bins ? l2 : bins) - (l1 + 1 > 0 ? l1 + 1 : 0);
  bool const has_middle = l2 - l1 > 1 && middle_bins > 0;
  double const es[3] = {edge.x, edge.y, edge.z};
  bool vf = true, vm = true, vl = true;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    // a part without bins in this tile takes no part in the sums
    long long f = 0, m = 0, l = 0;
    if (has_first && !checked_increment(es[c] * first, f, tally.zhs_abs)) vf = false;
    if (has_middle && !checked_increment(es[c] * sign, m, tally.zhs_abs)) vm = false;
    if (has_last && !checked_increment(es[c] * last, l, tally.zhs_abs)) vl = false;
    add_segment_row(tile + c * stride, bins, l1, l2, f, m, l);
  }
  unsigned long long const nm = has_middle ? static_cast<unsigned long long>(middle_bins) : 0ull;
  unsigned long long const nf = has_first ? 1ull : 0ull, nl = has_last ? 1ull : 0ull;
  tally.zhs += (vf ? nf : 0ull) + (vm ? nm : 0ull) + (vl ? nl : 0ull);
  tally.overflow += (vf ? 0ull : nf) + (vm ? 0ull : nm) + (vl ? 0ull : nl);
}

template <bool Homogeneous>
__device__ __forceinline__ void zhs_update(Track const& t, PropagationDev const& p, std::uint32_t refinement,
                                           View const& o, long long* tile, std::uint32_t stride, Tally& tally,
                                           bool count_subtracks) {
  V3 const midpoint{(t.start.x + t.end.x) * 0.5, (t.start.y + t.end.y) * 0.5, (t.start.z + t.end.z) * 0.5};
  Path const mp = propagate<Homogeneous>(p, o, midpoint);
  V3 const d{t.end.x - t.start.x, t.end.y - t.start.y, t.end.z - t.start.z};
  // sin^2 L^2 from the direction of the displacement: L^2 - (d.e)^2
  double const along = dot(d, mp.emit);
  double const fraunhofer = fma(-along, along, dot(d, d)) * mp.inv_distance * o.two_pi_over_wavelength;
  if (!(fraunhofer > 1.) && refinement <= 1u) {
    if (count_subtracks) ++tally.single_subtracks;
    zhs_segment(mp, dot(t.beta, mp.emit), (t.t0 + t.t1) * 0.5, t.duration * 0.5, t, o, tile, stride, tally, false);
    return;
  }
  double divisor = 1.;
  int nsub = 1;
  if (fraunhofer > 1.) {
    divisor = sqrt(fraunhofer) + 1.;
    nsub = static_cast<int>(ceil(divisor));
  }
  int const refine = static_cast<int>(refinement);
  if (count_subtracks) {
    tally.subtracks += static_cast<unsigned long long>(nsub);
    if (refine > 1) tally.subtracks += static_cast<unsigned long long>(nsub * (refine - 1));
  }
  int const segments = nsub * refine;
  double const parts = divisor * static_cast<double>(refine);
  V3 const step{d.x / parts, d.y / parts, d.z / parts};
  double const dt = t.duration / parts;
  V3 p1 = t.start;
  double time1 = t.t0;
  for (int i = 0; i < segments; ++i) {
    V3 const p2{p1.x + step.x, p1.y + step.y, p1.z + step.z};
    double const time2 = time1 + dt;
    Path const path = propagate<Homogeneous>(p, o, {(p1.x + p2.x) * 0.5, (p1.y + p2.y) * 0.5, (p1.z + p2.z) * 0.5});
    zhs_segment(path, dot(t.beta, path.emit), (time1 + time2) * 0.5, (time2 - time1) * 0.5, t, o, tile, stride,
                tally, true);
    p1 = p2;
    time1 = time2;
  }
}

}  // namespace c8mi::radio::fast
