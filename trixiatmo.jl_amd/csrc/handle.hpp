// Handle of libatmo_hip (internal): device buffers, stream and timers.
#ifndef ATMO_HANDLE_HPP
#define ATMO_HANDLE_HPP

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "../../include/atmo_hip.h"
#include "rainy_kernels.hpp"
#include "swe_kernels.hpp"

namespace atmo {

// the handles in use: the last one to go gives back the pinned transfer slots
struct HandleCount {
  HandleCount();
  ~HandleCount();
  HandleCount(const HandleCount&) = delete;
  HandleCount& operator=(const HandleCount&) = delete;
};

struct TimerPair {
  hipEvent_t a, b;
  int cls;
};

std::string& global_error();

inline int fail(std::string* slot, int code, const std::string& msg) {
  if (slot) *slot = msg;
  global_error() = msg;
  return code;
}

}  // namespace atmo

struct atmo_handle {
  atmo::HandleCount counted;
  int eq = ATMO_EQ_EULER_ENERGY_GRAVITY_3D;
  atmo_config cfg;
  int n = 0, n3 = 0, nv = 6;
  int64_t len = 0;  // doubles per state
  int device = 0;
  hipStream_t stream = nullptr;
  double *d_u = nullptr, *d_u2 = nullptr, *d_k = nullptr, *d_du = nullptr;
  double *d_uio = nullptr, *d_duio = nullptr;  // staging for atmo_rhs with host arrays
  double *d_cv = nullptr, *d_invJ = nullptr;
  float* d_cv32 = nullptr;  // FP32 geometry of the mixed-precision path
  bool bg_on = false;       // hydrostatic background split (mixed path)
  double *d_ubg = nullptr, *d_dubg = nullptr;
  float* d_B = nullptr;
  std::vector<double> dsplit, weights;
  int* d_nbr = nullptr;
  int* d_face_info = nullptr;
  double* d_partial = nullptr;
  // results of a reduction: pinned host memory that the last kernel writes
  // (device address d_result), read here after the stream is synchronised, so
  // no copy stands between them (launch to value 11.5 against 24 us with a
  // copy into pageable memory)
  double *h_result = nullptr, *d_result = nullptr;
  // covariant shallow water
  atmo_swe_config swe{};
  atmo::SweLaunch swe_base{};
  double *d_aux = nullptr, *d_xyz = nullptr, *d_dt_member = nullptr;
  double *d_geo = nullptr, *d_fxf = nullptr;  // stage-kernel geometry (compact, face transforms)
  float *d_geo32 = nullptr, *d_fxf32 = nullptr;  // the same in FP32 (ATMO_PREC_FP32_GEOMETRY)
  double* d_hs64 = nullptr;  // FP32 geometry with bottom topography: h_s kept in FP64
  int *d_member = nullptr, *d_member_first = nullptr;
  int n_members = 1;
  bool swe_tuned = false;                  // workgroup shape chosen by the autotuner
  hipGraphExec_t swe_graph = nullptr;      // two RK steps captured for replay
  int swe_graph_variant = -1;
  double* swe_graph_u = nullptr;           // state buffer the graph was captured with
  // rainy Euler
  atmo_rainy_config rainy{};
  atmo::RainyLaunch rainy_base{};
  double time = 0.0;                       // time of the resident state
  double* d_clock = nullptr;               // device clock of the resident time loop
  double *h_clock = nullptr, *d_hclock = nullptr;  // its copy in pinned host memory
  // two resident steps captured for replay, and the launch parameters (bytes of
  // swe_base or rainy_base) and state buffer they were captured with
  hipGraphExec_t solve_graph = nullptr;
  double* solve_graph_u = nullptr;
  int solve_graph_epb = 0;
  std::vector<unsigned char> solve_graph_key;
  // 3D atmo_step: two RK steps captured for replay, their step size read from d_step_dt
  hipGraphExec_t e3_graph = nullptr;
  double* e3_graph_u = nullptr;            // state buffer the graph was captured with
  int e3_graph_epb = 0;                    // and the stage shape
  int e3_epb = 1;                          // elements per workgroup of the 3D stage
  bool e3_tuned = false;
  double* d_step_dt = nullptr;
  // Newton statistics: per-wave slots [n_stat_slots][4], then the reduced [4]
  unsigned long long* d_stats = nullptr;
  int n_stat_slots = 0;
  atmo_mlp* mlp = nullptr;                 // seed of the saturation solve
  bool du_valid = false;
  bool timing = false;
  std::vector<atmo::TimerPair> timers;
  int64_t launches[2] = {0, 0};
  double total_ms[2] = {0, 0};
  std::string err;
};

#define HIP_TRY(h, expr)                                                         \
  do {                                                                           \
    hipError_t e__ = (expr);                                                     \
    if (e__ != hipSuccess)                                                       \
      return atmo::fail((h) ? &(h)->err : nullptr, ATMO_ERR_DEVICE,              \
                        std::string(#expr) + ": " + hipGetErrorString(e__));     \
  } while (0)

namespace atmo {
// copy from the device to caller memory on the handle's stream, complete on
// return (transfer.hip)
hipError_t copy_to_host(atmo_handle* h, void* dst, const void* src, size_t bytes);
// h_result / d_result of n doubles
bool alloc_result(atmo_handle* h, size_t n);
void timer_begin(atmo_handle* h, int cls, TimerPair* tp);
void timer_end(atmo_handle* h, TimerPair* tp);
// covariant shallow water paths of the generic entry points
int swe_rhs_device(atmo_handle* h, double* du, const double* u);
int swe_step(atmo_handle* h, const double* dt_members, double dt, int n_steps);
int swe_max_dt(atmo_handle* h, double cfl, double* dt_members);
int swe_integrals(atmo_handle* h, int fresh_rhs, double* out);
int swe_autotune(atmo_handle* h, double* ms_per_variant);
// 3D stage: one or two elements per workgroup (ms_per_variant[2] may be NULL)
int e3_autotune(atmo_handle* h, double* ms_per_variant);
// whether the 3D stage of this polydeg / precision has the two-element shape
bool e3_has_two_element_groups(int n, int precision);
// whether a mesh of n_elements runs the split form, which has one shape
bool e3_takes_split_form(int n, int precision, int n_elements);
// rainy Euler paths of the generic entry points
int rainy_rhs_device(atmo_handle* h, double* du, const double* u, double t);
int rainy_step(atmo_handle* h, double dt, int n_steps);
int rainy_max_dt(atmo_handle* h, double cfl, double* dt);
int rainy_integrals(atmo_handle* h, double* out);
void rainy_free(atmo_handle* h);
// the resident time loop: one step (maximum wave speed, step-size control,
// five stages reading the step size from d_clock) enqueued on the stream
int e3_enqueue_resident_step(atmo_handle* h);
// side: -1 with a control kernel of its own, else the clock (0 or 1) that the
// first stage reads while it writes the other
int swe_enqueue_resident_step(atmo_handle* h, int side);
// whether a resident step's first stage can take the control
bool swe_fuses_control(const atmo_handle* h);
int rainy_enqueue_resident_step(atmo_handle* h);
// ptr[0 .. n) = value, stream-ordered (a value for kernels that read it from memory)
void launch_fill(double* ptr, double value, int n, hipStream_t s);
// dt and the clock of one member from its elements' wave speeds
void launch_step_control_reduce(const double* partial, int n_items, int n, double* clock,
                                double* dt, hipStream_t s);
// result[0] = the maximum of floor and the n partials (NaN propagates)
void launch_reduce_max(const double* partial, int n, double floor, double* result, hipStream_t s);
// result[c] = the sum of row c of partial [width][n]
void launch_sum_rows(const double* partial, int n, int width, double* result, hipStream_t s);
// result[m] = the maximum of 5e-324 and member m's per-element partials
void launch_member_max(const double* partial, const int* member_first, int n_members,
                       double* result, hipStream_t s);
// set-up of a resident loop before its steps are enqueued (the first step's
// speeds where the stages provide the later ones)
int e3_resident_prologue(atmo_handle* h);
int swe_resident_prologue(atmo_handle* h);
int rainy_resident_prologue(atmo_handle* h);
// the same per ensemble member over its element range
void launch_step_control_members_reduce(const double* partial, const int* member_first,
                                        int n_members, int n, double* clock, double* dt,
                                        hipStream_t s);
}  // namespace atmo

#endif
