// Scalar f32 arithmetic of the matrix-core passes' epilogues.  Plain C++, so that a host program can
// check it against 64 bits.
#ifndef MSD_ARITH_H
#define MSD_ARITH_H

#include <math.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define MSD_ARITH __host__ __device__ inline
#else
#define MSD_ARITH inline
#endif

namespace msdc {

// SwiGLU of a gate/up pair (model.py:159).  The library exponential and an IEEE reciprocal: the hardware
// exponential of x log2(e) alone is off by up to |x| 2^-24 (its argument's rounding), against 2^-23 for any x.
MSD_ARITH float swiglu(float g, float u) { return (g * (1.f / (1.f + expf(-g)))) * u; }

// a / b, given rb = 1 / b rounded to nearest: a rb and one correction by its residual, which f32 holds
// exactly, so the quotient is the correctly rounded one unless it or the residual is subnormal (against ~10
// instructions per quotient for a divisor that is new each time).  The fixup gives the infinities,
// zeros and NaN of a division.
MSD_ARITH float quotient(float a, float b, float rb) {
  const float q = a * rb;
  const float r = fmaf(fmaf(-q, b, a), rb, q);
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_div_fixupf(r, b, a);
#else
  return isfinite(a) && isfinite(b) && isfinite(rb) ? r : a / b;
#endif
}

}  // namespace msdc

#undef MSD_ARITH
#endif  // MSD_ARITH_H
