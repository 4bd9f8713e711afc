// The step-size control of the resident time loop, for the kernels that make
// the next step of a clock.
#ifndef ATMO_STEP_CONTROL_HPP
#define ATMO_STEP_CONTROL_HPP

#include <hip/hip_runtime.h>

namespace atmo {

// clock layout (M members): t[M] (start of the step in flight), dt[M], steps
// taken [M], status (1: non-finite wave speed), t_end, cfl
constexpr int kClockExtra = 3;

// what the control of member m reads, loaded while the partials are in flight
struct ClockIn {
  double t, dt, steps, t_end, cfl;
};

__device__ __forceinline__ ClockIn load_clock(const double* clock, const double* dt, int m, int M) {
  return {clock[m], dt[m], clock[2 * M + m], clock[3 * M + 1], clock[3 * M + 2]};
}

struct ClockOut {
  double t, dt, steps;
  bool failed;  // the wave speed is not a finite number
};

// the step just taken is added to t, then the next step size is
// dt = min(cfl * (2 / (n * max speed)), t_end - t) as atmo_max_dt and the host
// loop compute it (same operations in the same order), or 0 once t >= t_end
__device__ __forceinline__ ClockOut step_control(double max_speed, const ClockIn& c, int n) {
  ClockOut o{c.t + c.dt, 0.0, c.steps, false};
  if (o.t < c.t_end) {
    double mx = max_speed;
    if (!isfinite(mx)) {
      o.failed = true;
    } else {
      if (mx < 5e-324) mx = 5e-324;
      o.dt = fmin(c.cfl * (2.0 / (n * mx)), c.t_end - o.t);
      o.steps += 1.0;
    }
  }
  return o;
}

}  // namespace atmo

#endif
