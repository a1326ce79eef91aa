// Qualifiers of the step path: every function one particle step calls is
// compiled for the device kernels and for the host's scalar stepper (the CPU
// steps of the handoff prefix), from the same source, so both sides run the
// same arithmetic.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#define C8MI_HD __host__ __device__ __forceinline__
#define C8MI_HD_NOINLINE __host__ __device__ __noinline__ inline

namespace c8mi::em {

// The classification functions of both sides (the device overloads live in
// std beside the host ones).
using std::isfinite;
using std::isinf;
using std::isnan;

// The long math functions of the step path, out of line on the device. Inlined
// at every use they were half the code of the step kernels (93000 instructions
// of the e+- move, 594 KB); a step runs most of its code once, so a front's time
// went into fetching it: 1861 instruction requests to L2 per wave of the move.
// Same library functions, same values; the host keeps its inline calls.
#if defined(__HIP_DEVICE_COMPILE__)
#define C8MI_MATH [[maybe_unused]] static __device__ __noinline__
C8MI_MATH double log(double x) { return ::log(x); }
C8MI_MATH double log1p(double x) { return ::log1p(x); }
C8MI_MATH double exp(double x) { return ::exp(x); }
C8MI_MATH double expm1(double x) { return ::expm1(x); }
C8MI_MATH double pow(double x, double y) { return ::pow(x, y); }
#undef C8MI_MATH
#endif

// Counter increment of the step path: one device atomic in a kernel; a plain
// add in the host stepper, whose accumulators belong to one thread.
C8MI_HD unsigned long long fetch_add(unsigned long long* address, unsigned long long value) {
#if defined(__HIP_DEVICE_COMPILE__)
  return atomicAdd(address, value);
#else
  unsigned long long const old = *address;
  *address = old + value;
  return old;
#endif
}

}  // namespace c8mi::em
