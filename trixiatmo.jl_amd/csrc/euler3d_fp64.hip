// FP64 instantiations of the fused stage kernel (compared with the oracle).
#include "euler3d_stage.hpp"

namespace atmo {
bool e3_launch_stage_fp64(const E3Launch& L, hipStream_t s) {
  return dispatch_stage<double, false>(L, s);
}

bool e3_has_two_element_groups(int n, int precision) {
  // the FP32-geometry form computes in FP64 (precision 3)
  const bool f64 = precision == 0 || precision == 3;
  switch (n) {
    case 4: return f64 ? has_two_element_groups<4, double>() : has_two_element_groups<4, float>();
    case 5: return f64 ? has_two_element_groups<5, double>() : has_two_element_groups<5, float>();
    default: return false;
  }
}

bool e3_takes_split_form(int n, int precision, int n_elements) {
  if (precision != 0 && precision != 3) return false;
  switch (n) {
    case 2: return n_elements <= split_max_elements<2>();
    case 3: return n_elements <= split_max_elements<3>();
    case 4: return n_elements <= split_max_elements<4>();
    case 5: return n_elements <= split_max_elements<5>();
    case 6: return n_elements <= split_max_elements<6>();
    case 7: return n_elements <= split_max_elements<7>();
    default: return false;
  }
}
}  // namespace atmo
