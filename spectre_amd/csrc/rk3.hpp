// One substep of Rk3HesthavenSsp and its application to a kernel's results.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.hpp"

namespace sxd {

// Rk3HesthavenSsp::update_u (Time/TimeSteppers/Rk3HesthavenSsp.cpp:55-81) of one
// value.
__device__ __forceinline__ double rk3_value(int substep, double dt, double u0, double uk,
                                            double lk) {
  if (substep == 0) return u0 + dt * lk;
  if (substep == 1) return 0.25 * (3.0 * u0 + uk + dt * lk);
  return (1.0 / 3.0) * (u0 + 2.0 * uk + 2.0 * dt * lk);
}
__device__ __forceinline__ double rk3_step_size(const Rk3Update& up) {
  return up.dt_ptr != nullptr ? *up.dt_ptr : up.dt;
}

// v (the time derivative of the NC values uk of a point) to the substep's
// result; u0 of value c at at + c step.
template <int NC>
__device__ __forceinline__ void rk3_apply(double v[NC], const Rk3Update& up, const double* uk,
                                          int64_t at, int64_t step) {
  double u0[NC];
  const double dt = rk3_step_size(up);
#pragma unroll
  for (int c = 0; c < NC; ++c) u0[c] = up.substep == 0 ? uk[c] : up.u0[at + c * step];
#pragma unroll
  for (int c = 0; c < NC; ++c) v[c] = rk3_value(up.substep, dt, u0[c], uk[c], v[c]);
}

// The transposed substep of one value: a (A^T lam at lam = l) becomes lam_out,
// and mu is updated; after substep 0 nothing is left to store.  Applied by the
// adjoint kernels it saves a launch that reads and writes three fields: gradient
// of 5 ScalarWave steps on 512 x 6^3 465 -> 343 us, of 3 GH steps on 300 x 6^3
// 2386 -> 2308 us.
__device__ __forceinline__ double rk3_adjoint_value(int substep, double dt, double l, double a,
                                                    double* mu) {
  if (substep == 2) {
    *mu = (1.0 / 3.0) * l;
    return (2.0 / 3.0) * (l + dt * a);
  }
  if (substep == 1) {
    *mu = *mu + 0.75 * l;
    return 0.25 * (l + dt * a);
  }
  *mu = *mu + (l + dt * a);
  return 0.0;
}

}  // namespace sxd
