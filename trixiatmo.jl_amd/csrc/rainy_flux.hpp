// The entropy-conserving two-point flux of CompressibleRainyEulerEquations2D
// (flux_ec_rain, src/equations/compressible_rainy_euler_2d.jl:872-961) on
// per-node quantities formed once per node, and the equations' constants:
// shared by the stage kernels and by the tests' device probe.
#ifndef ATMO_RAINY_FLUX_HPP
#define ATMO_RAINY_FLUX_HPP

#include <hip/hip_runtime.h>

#include "euler3d_physics.hpp"

namespace atmo {
namespace rainy {

// CompressibleRainyEulerEquations2D() constants (:77-113)
constexpr double c_l = 4186, c_pd = 1004, c_vd = 717, c_pv = 1885, c_vv = 1424;
constexpr double R_d = c_pd - c_vd, R_v = c_pv - c_vv;
constexpr double ref_sp = 610.7, ref_T = 273.15, L_ref = 2500000;
constexpr double grav = 9.80616, N_0 = 8000000, v_0 = 130;
constexpr double kPi = 3.14159265358979323846;

// |v|^2 of one node, rounded the same way wherever it is formed
__device__ __forceinline__ double norm2(double v1, double v2) { return fma(v1, v1, v2 * v2); }

// the per-node quantities flux_ec_rain reads, formed once per node
struct ECNode {
  double rd, rv, rc, rr, v1, v2, it, vr;  // it = 1 / T, vr from rho_vapour + rho_cloud
  double lrd, lrv, lit;                   // log(rho_dry), log(rho_vapour), log(1 / T)
};

__device__ __forceinline__ void flux_ec_rain(const ECNode& l, const ECNode& r, double n1,
                                             double n2, double* f) {
#pragma clang fp contract(off)
  // every sum is symmetric in the two nodes, or changes both signs of a
  // quotient with them, and every fused multiply-add is written out: the flux
  // has the same bits in both orders
  const double v1a = 0.5 * (l.v1 + r.v1), v2a = 0.5 * (l.v2 + r.v2);
  const double K = 0.25 * (norm2(l.v1, l.v2) + norm2(r.v1, r.v2));
  const double vdn = fma(n1, v1a, n2 * v2a);
  const double vrn = 0.5 * n2 * (l.vr + r.vr);
  const double dry_s = l.rd + r.rd, vap_s = l.rv + r.rv;
  // logarithmic means from the node logarithms (the series branch where the
  // two values are close), no logarithm per pair
  double dry_log = 0.0, vap_log = 0.0;
  if (l.rd != 0.0 && r.rd != 0.0) dry_log = ln_mean_logs(l.rd, r.rd, l.lrd, r.lrd);
  if (l.rv != 0.0 && r.rv != 0.0) vap_log = ln_mean_logs(l.rv, r.rv, l.lrv, r.lrv);
  // the inverse logarithmic mean of 1 / T and 1 over its arithmetic mean from
  // one reciprocal of the sum
  const double d = r.it - l.it, s = l.it + r.it;
  const double r1 = rcp_refined(s);
  const double is = fma(fma(-s, r1, 1.0), r1, r1);
  double it_log;
  if (d * d < 1.0e-4 * (s * s)) {
    const double g = d * is, f2 = g * g;
    it_log = is * fma(f2, fma(f2, fma(f2, 2.0 / 7.0, 2.0 / 5.0), 2.0 / 3.0), 2.0);
  } else {
    it_log = div_nr(r.lit - l.lit, d);
  }
  const double p_int = is * fma(R_d, dry_s, R_v * vap_s);
  const double f_vap = vap_log * vdn;
  const double f_cld = 0.5 * (l.rc + r.rc) * vdn;
  const double f_dry = dry_log * vdn;
  const double f_rain = 0.5 * (l.rr + r.rr) * (vdn - vrn);
  const double f_moist = f_vap + f_cld;
  const double f_liq = f_cld + f_rain;
  const double f_rho = f_dry + f_moist + f_rain;
  const double f_m1 = fma(f_rho, v1a, p_int * n1);
  const double f_m2 = fma(f_rho, v2a, p_int * n2);
  f[0] = f_dry;
  f[1] = f_moist;
  f[2] = f_rain;
  f[3] = f_m1;
  f[4] = f_m2;
  f[5] = fma(it_log, fma(c_vd, f_dry, fma(c_vv, f_vap, c_l * f_liq)), -(K * f_rho)) +
         fma(L_ref, f_vap, fma(v1a, f_m1, v2a * f_m2));
}

}  // namespace rainy
}  // namespace atmo

#endif
