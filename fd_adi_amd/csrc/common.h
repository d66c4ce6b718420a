// Shared definitions for the fd_adi_amd HIP library (gfx950, FP64).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>

#include "../../include/fdadi.h"

namespace fdadi {

// Thread-local last-error message; fdadi_last_error() returns it.
void set_error(const std::string &msg);

// Every entry point returns an int status; these helpers keep it uniform.
#define FDADI_TRY_HIP(expr)                                                   \
  do {                                                                        \
    hipError_t _e = (expr);                                                   \
    if (_e != hipSuccess) {                                                   \
      fdadi::set_error(std::string(#expr) + ": " + hipGetErrorString(_e));    \
      return FDADI_ERR_HIP;                                                   \
    }                                                                         \
  } while (0)

#define FDADI_REQUIRE(cond, code, msg)                                        \
  do {                                                                        \
    if (!(cond)) {                                                            \
      fdadi::set_error(msg);                                                  \
      return code;                                                            \
    }                                                                         \
  } while (0)

// Check the launch that was just issued.
#define FDADI_CHECK_LAUNCH() FDADI_TRY_HIP(hipGetLastError())

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

// 1 / d by two Newton steps from the hardware estimate (relative error
// 2^-23, then 2^-46 and below 2^-90 before the last rounding): the IEEE
// division at half its instructions.  v_div_fixup supplies d's sign and the
// results for zeros, infinities, NaN and |d| <= 2^-1024 (whose reciprocals
// overflow).  For |d| within 2^-23 above that the estimate overflows and the
// reciprocal does not: recip_any holds the estimate to finite numbers, for
// pivots of any size (the line solver's); recip gives an infinity there, for
// those of I - theta dt A, whose diagonal starts from 1 (one instruction more
// per row made the spot sweeps 1% longer).
__device__ __forceinline__ double recip_from(double r, double d) {
  r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
  return __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
}
__device__ __forceinline__ double recip(double d) {
  return __builtin_amdgcn_div_fixup(recip_from(__builtin_amdgcn_rcp(d), d), d, 1.0);
}
__device__ __forceinline__ double recip_any(double d) {
  const double ad = __builtin_fabs(d);
  const double r = __builtin_fmin(__builtin_amdgcn_rcp(ad), 0x1.fffffffffffffp1023);
  return __builtin_amdgcn_div_fixup(recip_from(r, ad), d, 1.0);
}

inline unsigned grid_for(int64_t n, int block) {
  int64_t g = (n + block - 1) / block;
  if (g < 1) g = 1;
  return static_cast<unsigned>(g);
}

}  // namespace fdadi
