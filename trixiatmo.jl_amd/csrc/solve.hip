// The time loop of the examples' solve(ode, CarpenterKennedy2N54(williamson_condition
// = false); callback = StepsizeCallback(cfl)) (e.g.
// examples/shallow_water/covariant/elixir_barotropic_instability.jl:79-80)
// kept on the device.  Every step begins with its control, a workgroup per
// member that reduces the elements' wave speeds and turns them into the step
// size (cut to end at t_end, as OrdinaryDiffEq's tstop handling does); the five
// fused stages read the step size from device memory, and the last of them
// writes the new state's speeds.  On small covariant meshes the control is part
// of the first stage instead.  Two steps are captured as one graph and
// replayed; the host reads the clock back only every `check_every` steps.  A
// member that has reached t_end takes steps of size 0, which leave its state
// unchanged, so the members of an ensemble each follow their own step sizes
// and finish together.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "handle.hpp"
#include "speed_max.hpp"
#include "step_control.hpp"

namespace atmo {

namespace {

__device__ __forceinline__ void store_step_control(double max_speed, const ClockIn& c, int m,
                                                   int M, int n, double* clock, double* dt) {
  const ClockOut o = step_control(max_speed, c, n);
  if (o.failed) clock[3 * M] = 1.0;  // every member that finds one stores the same value
  clock[2 * M + m] = o.steps;
  clock[m] = o.t;
  dt[m] = o.dt;
}

// maximum over partial[from .. to) of a workgroup of B lanes, on every lane of
// its first wave: eight independent loads in flight per lane, then their
// maximum (one load at a time waited for each: 33 us for 32,768 partials
// against 6)
template <int B>
__device__ __forceinline__ double block_max(const double* __restrict__ partial, int from, int to,
                                            double floor) {
  __shared__ double s[B / 64];
  const int t = threadIdx.x;
  double m = floor;
  for (int i0 = from + t; i0 < to; i0 += 8 * B) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = i0 + k * B < to ? partial[i0 + k * B] : floor;
#pragma unroll
    for (int k = 0; k < 8; ++k) m = speed_max(m, v[k]);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = speed_max(m, __shfl_xor(m, o, 64));
  if ((t & 63) == 0) s[t >> 6] = m;
  __syncthreads();
  for (int w = 0; w < B / 64; ++w) m = speed_max(m, s[w]);
  return m;
}

// the control of one member whose maximum speed is the maximum over per-element
// partials (written by the last stage of the step just taken).  One chain of
// latencies between two stages: the clock is loaded beside the partials, and
// the workgroup has as many lanes as one batch of block_max needs
template <int B>
__global__ __launch_bounds__(B) void step_control_reduce_kernel(const double* __restrict__ partial,
                                                                int n_items, int n, double* clock,
                                                                double* dt) {
  const ClockIn c = load_clock(clock, dt, 0, 1);
  const double m = block_max<B>(partial, 0, n_items, 0.0);
  if (threadIdx.x == 0) store_step_control(m, c, 0, 1, n, clock, dt);
}

// one workgroup per ensemble member: its maximum speed is the maximum over the
// per-element partials of its elements [member_first[m], member_first[m + 1])
__global__ __launch_bounds__(256) void step_control_members_reduce_kernel(
    const double* __restrict__ partial, const int* __restrict__ member_first, int M, int n,
    double* clock, double* dt) {
  const int m = blockIdx.x;
  const ClockIn c = load_clock(clock, dt, m, M);
  const double mx = block_max<256>(partial, member_first[m], member_first[m + 1], 0.0);
  if (threadIdx.x == 0) store_step_control(mx, c, m, M, n, clock, dt);
}

__global__ __launch_bounds__(1024) void reduce_max_kernel(const double* __restrict__ partial, int n,
                                                          double floor, double* result) {
  const double m = block_max<1024>(partial, 0, n, floor);
  if (threadIdx.x == 0) result[0] = m;
}

__global__ __launch_bounds__(256) void member_max_kernel(const double* __restrict__ partial,
                                                         const int* __restrict__ member_first,
                                                         double* result) {
  const int m = blockIdx.x;
  const double mx = block_max<256>(partial, member_first[m], member_first[m + 1], 5e-324);
  if (threadIdx.x == 0) result[m] = mx;
}

// one workgroup per row, the sum in a fixed order (one workgroup for all nine
// rows of 5,184 partials, 256 lanes and a load at a time: 40 us; this: 4)
__global__ __launch_bounds__(1024) void sum_rows_kernel(const double* __restrict__ partial, int n,
                                                        double* result) {
  __shared__ double s[1024 / 64];
  const int t = threadIdx.x;
  const double* p = partial + (size_t)blockIdx.x * n;
  double a = 0.0;
  for (int i0 = t; i0 < n; i0 += 8 * 1024) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = i0 + k * 1024 < n ? p[i0 + k * 1024] : 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k) a += v[k];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
  if ((t & 63) == 0) s[t >> 6] = a;
  __syncthreads();
  if (t != 0) return;
  a = s[0];
  for (int w = 1; w < 1024 / 64; ++w) a += s[w];
  result[blockIdx.x] = a;
}

}  // namespace

void launch_step_control_members_reduce(const double* partial, const int* member_first,
                                        int n_members, int n, double* clock, double* dt,
                                        hipStream_t s) {
  hipLaunchKernelGGL(step_control_members_reduce_kernel, dim3(n_members), dim3(256), 0, s, partial,
                     member_first, n_members, n, clock, dt);
}

namespace {
// a clock at time t before its first step; dt: the step sizes the stages read
__global__ void init_clock_kernel(double* clock, double* dt, int M, double t, double t_end,
                                  double cfl) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m < M) {
    clock[m] = t;
    clock[M + m] = 0.0;
    clock[2 * M + m] = 0.0;
    dt[m] = 0.0;
  }
  if (m == 0) {
    clock[3 * M] = 0.0;
    clock[3 * M + 1] = t_end;
    clock[3 * M + 2] = cfl;
  }
}

// t, the step sizes the stages read, the steps and the status
__global__ void read_clock_kernel(const double* __restrict__ clock, const double* __restrict__ dt,
                                  int M, double* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i <= 3 * M) out[i] = i >= M && i < 2 * M ? dt[i - M] : clock[i];
}

__global__ void fill_kernel(double* ptr, double value, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) ptr[i] = value;
}
}  // namespace

void launch_init_clock(double* clock, double* dt, int M, double t, double t_end, double cfl,
                       hipStream_t s) {
  hipLaunchKernelGGL(init_clock_kernel, dim3((M + 63) / 64), dim3(64), 0, s, clock, dt, M, t,
                     t_end, cfl);
}

void launch_read_clock(const double* clock, const double* dt, int M, double* out, hipStream_t s) {
  hipLaunchKernelGGL(read_clock_kernel, dim3((3 * M + 64) / 64), dim3(64), 0, s, clock, dt, M, out);
}

void launch_fill(double* ptr, double value, int n, hipStream_t s) {
  hipLaunchKernelGGL(fill_kernel, dim3((n + 63) / 64), dim3(64), 0, s, ptr, value, n);
}

void launch_reduce_max(const double* partial, int n, double floor, double* result, hipStream_t s) {
  hipLaunchKernelGGL(reduce_max_kernel, dim3(1), dim3(1024), 0, s, partial, n, floor, result);
}

void launch_member_max(const double* partial, const int* member_first, int n_members,
                       double* result, hipStream_t s) {
  hipLaunchKernelGGL(member_max_kernel, dim3(n_members), dim3(256), 0, s, partial, member_first,
                     result);
}

void launch_sum_rows(const double* partial, int n, int width, double* result, hipStream_t s) {
  hipLaunchKernelGGL(sum_rows_kernel, dim3(width), dim3(1024), 0, s, partial, n, result);
}

void launch_step_control_reduce(const double* partial, int n_items, int n, double* clock,
                                double* dt, hipStream_t s) {
  if (n_items <= 8 * 256)
    hipLaunchKernelGGL(step_control_reduce_kernel<256>, dim3(1), dim3(256), 0, s, partial, n_items,
                       n, clock, dt);
  else
    hipLaunchKernelGGL(step_control_reduce_kernel<1024>, dim3(1), dim3(1024), 0, s, partial,
                       n_items, n, clock, dt);
}

}  // namespace atmo

namespace {

using atmo::fail;
using atmo::kClockExtra;
using atmo::launch_init_clock;
using atmo::launch_read_clock;

int enqueue_resident_steps(atmo_handle* h, int n_steps, bool fused) {
  for (int s = 0; s < n_steps; ++s) {
    const int rc = h->eq == ATMO_EQ_COVARIANT_SWE_2D ? atmo::swe_enqueue_resident_step(h, fused ? s & 1 : -1)
                   : h->eq == ATMO_EQ_RAINY_EULER_2D ? atmo::rainy_enqueue_resident_step(h)
                                                     : atmo::e3_enqueue_resident_step(h);
    if (rc != ATMO_OK) return rc;
  }
  return ATMO_OK;
}

// two resident steps as one graph (the ping-pong state buffers return to
// their places after an even number of stages), kept for the next call with
// the same buffers and launch parameters (capturing and instantiating it takes
// about 60 us, which two steps on a small mesh take too)
int ensure_solve_graph(atmo_handle* h, bool fused) {
  std::vector<unsigned char> key;
  auto bytes = [&](const void* p, size_t n) {
    key.assign(static_cast<const unsigned char*>(p), static_cast<const unsigned char*>(p) + n);
  };
  if (h->eq == ATMO_EQ_COVARIANT_SWE_2D) bytes(&h->swe_base, sizeof(h->swe_base));
  if (h->eq == ATMO_EQ_RAINY_EULER_2D) bytes(&h->rainy_base, sizeof(h->rainy_base));
  if (h->solve_graph && h->solve_graph_u == h->d_u && h->solve_graph_epb == h->e3_epb &&
      h->solve_graph_key == key)
    return ATMO_OK;
  if (h->solve_graph) {
    HIP_TRY(h, hipGraphExecDestroy(h->solve_graph));
    h->solve_graph = nullptr;
  }
  hipGraph_t g = nullptr;
  HIP_TRY(h, hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
  const int rc = enqueue_resident_steps(h, 2, fused);
  const hipError_t ec = hipStreamEndCapture(h->stream, &g);
  if (rc != ATMO_OK) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  HIP_TRY(h, ec);
  const hipError_t ei = hipGraphInstantiate(&h->solve_graph, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  HIP_TRY(h, ei);
  h->solve_graph_u = h->d_u;
  h->solve_graph_epb = h->e3_epb;
  h->solve_graph_key = std::move(key);
  return ATMO_OK;
}

// the clock as it stands after everything enqueued, in h->h_clock: by a kernel
// that writes pinned host memory (a copy into pageable memory takes 12 us more)
int read_clock(atmo_handle* h, const double* d_dt, int M) {
  launch_read_clock(h->d_clock, d_dt, M, h->d_hclock, h->stream);
  HIP_TRY(h, hipGetLastError());
  HIP_TRY(h, hipStreamSynchronize(h->stream));
  return ATMO_OK;
}

}  // namespace

extern "C" {

int atmo_solve(atmo_handle* h, double t_end, double cfl, int32_t check_every, int64_t* steps,
               double* t_reached) {
  if (!h) return fail(nullptr, ATMO_ERR_INVALID, "null handle");
  if (!(cfl > 0) || !std::isfinite(cfl) || !std::isfinite(t_end) || check_every < 1)
    return fail(&h->err, ATMO_ERR_INVALID, "bad solve arguments");
  const bool swe = h->eq == ATMO_EQ_COVARIANT_SWE_2D;
  const int M = swe ? h->n_members : 1;
  const size_t clock_len = 3 * (size_t)M + kClockExtra;
  if (!h->d_clock) HIP_TRY(h, hipMalloc(&h->d_clock, sizeof(double) * 2 * clock_len));
  if (!h->d_hclock) {
    void* p = nullptr;
    if (!h->h_clock)
      HIP_TRY(h, hipHostMalloc(reinterpret_cast<void**>(&h->h_clock), sizeof(double) * clock_len,
                               hipHostMallocDefault));
    HIP_TRY(h, hipHostGetDevicePointer(&p, h->h_clock, 0));
    h->d_hclock = static_cast<double*>(p);
  }
  if (swe && !h->swe_tuned) {
    const int rc = atmo::swe_autotune(h, nullptr);
    if (rc != ATMO_OK) return rc;
  }
  if (h->eq == ATMO_EQ_EULER_ENERGY_GRAVITY_3D && !h->e3_tuned) {
    const int rc = atmo::e3_autotune(h, nullptr);
    if (rc != ATMO_OK) return rc;
  }
  // the control as part of the first stage (an even number of steps, which the
  // graph takes, ends on the clock it began with)
  const bool fused = swe && !h->timing && atmo::swe_fuses_control(h);
  // the step-size array the stages read: the shallow-water stage reads its
  // per-member array, the others the clock's
  double* d_dt = swe && !fused ? h->d_dt_member : h->d_clock + M;
  h->du_valid = false;
  launch_init_clock(h->d_clock, d_dt, M, h->time, t_end, cfl, h->stream);
  HIP_TRY(h, hipGetLastError());
  bool done = !(h->time < t_end);
  if (!done) {
    const int rc = h->eq == ATMO_EQ_EULER_ENERGY_GRAVITY_3D ? atmo::e3_resident_prologue(h)
                   : swe                                  ? atmo::swe_resident_prologue(h)
                                                          : atmo::rainy_resident_prologue(h);
    if (rc != ATMO_OK) return rc;
  }
  hipGraphExec_t graph = nullptr;
  if (!h->timing && !done) {
    const int rc = ensure_solve_graph(h, fused);
    if (rc != ATMO_OK) return rc;
    graph = h->solve_graph;
  }
  // the clock as last read (before the first step: where it starts)
  const double* back = h->h_clock;
  const double* dt_back = h->h_clock + M;
  if (done) {
    const int rc = read_clock(h, d_dt, M);
    if (rc != ATMO_OK) return rc;
  }
  int rc = ATMO_OK;
  // a first short chunk gives the step size the later chunks are sized by
  int64_t chunk = std::min<int64_t>(check_every, 2);
  while (!done) {
    if (graph) {
      for (int64_t s = 0; s < chunk; s += 2) {
        const hipError_t e = hipGraphLaunch(graph, h->stream);
        if (e != hipSuccess) {
          rc = fail(&h->err, ATMO_ERR_DEVICE, std::string("hipGraphLaunch: ") + hipGetErrorString(e));
          break;
        }
      }
    } else {
      rc = enqueue_resident_steps(h, (int)chunk, false);
    }
    if (rc != ATMO_OK) break;
    rc = read_clock(h, d_dt, M);
    if (rc != ATMO_OK) break;
    if (back[3 * M] != 0.0) {
      rc = fail(&h->err, ATMO_ERR_NONFINITE, "non-finite wave speed in state");
      break;
    }
    // members still running after the step in flight, and the steps they
    // still need at their last step size: the next chunk is sized to that
    done = true;
    double need = 0.0;
    for (int m = 0; m < M; ++m) {
      const double dtm = dt_back[m];
      const double tm = back[m] + dtm;
      if (tm < t_end) {
        done = false;
        need = std::max(need, dtm > 0 ? std::ceil((t_end - tm) / dtm) : (double)check_every);
      }
    }
    chunk = (int64_t)std::min<double>(std::max(need, 1.0), (double)check_every);
    if (graph) chunk += chunk & 1;
  }
  if (rc != ATMO_OK && rc != ATMO_ERR_NONFINITE) return rc;
  // each member's time is t + dt of its last step
  double t_min = 0.0;
  for (int m = 0; m < M; ++m) {
    const double tm = back[m] + dt_back[m];
    t_min = m == 0 ? tm : std::min(t_min, tm);
    if (steps) steps[m] = (int64_t)back[2 * M + m];
  }
  if (M == 0) t_min = h->time;
  h->time = t_min;
  if (t_reached) *t_reached = t_min;
  return rc;
}

}  // extern "C"
