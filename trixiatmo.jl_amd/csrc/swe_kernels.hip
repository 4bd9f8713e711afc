// gfx950 kernels of the covariant shallow-water right-hand side
// (SplitCovariantShallowWaterEquations2D on the cubed sphere) and its RK stage.
//
// Layout: u [3, n, n, E] (h, h v^1, h v^2), aux [26, n, n, E] as Trixi's
// aux_node_vars (src/equations/equations.jl:178-250), node coordinates
// [3, n, n, E].  The stage kernel reads a compact structure-of-arrays copy of
// the 14 auxiliary rows it needs plus z / r (Trixi's node-major aux rows span
// 208 bytes, so reading a few of them fetches the whole row), and one 2 x 2
// basis map per face node instead of the 12 basis entries of both sides.
// A group of EPB elements has one lane per node (64, 128 or 256 lanes); the
// per-node fields the fluxes need (state, velocity v = hv / h, covariant
// velocity G v, J, G^-1, h_s, each formed once per node) are staged in LDS.
// Volume terms are gathered per node: sum_m Dsplit[own, m] (f#(own, m) +
// g(own, m) / 2) along both directions (the symmetric f# is evaluated for each
// ordering, the nonconservative g is non-symmetric anyway).  Every face node
// has a lane too: each element evaluates the interface flux of its own
// faces in its own contravariant basis with its own auxiliary variables,
// exactly as the reference does for each side
// (src/solvers/dgsem_p4est/dg_2d_manifold_in_3d_covariant.jl:301-432), lifts it
// with 1/w_end, and every node adds its face terms, applies -1/J and the
// geometric + Coriolis source, and stores du or applies the 2N RK update
// (per-element time step: ensemble members step with their own dt).
//
// Two forms of a group: the node lanes do all of it one after the other, or
// (SPLIT) three sets of waves share it: the node lanes take the volume terms
// of the first direction, a second set those of the second direction and a
// third set the face nodes, whose neighbour states are on their way from the
// start.  Both add the same sums in the same order, with every fused
// multiply-add written out (left to itself the compiler contracts each form
// its own way), so they give the same bits.
//
// What bounds it, and what each form is for (MI355X, microseconds per stage;
// in brackets the form before, whose volume loop took about twice the
// operations per pair, whose register reads waited for the stores before
// them and whose neighbour reads began after the volume terms): a small mesh
// is one chain of dependent operations per wave, so the split form, whose
// chain is shorter, wins (polydeg 3, 2,400 nodes: 3.9 split, 5.5 not [5.6];
// polydeg 4, 25,350 nodes: 4.7, 6.3 [7.4]); a full chip is bound by HBM, so
// the plain form, which needs fewer waves per node, wins (polydeg 3, 1.87 M
// nodes, 396 MB: 65.9 = 6.0 TB/s; split 71.7 [88.1]).  Between them (98,304
// nodes: 6.5 split, 6.9 plain [7.8]) the autotuner decides.
#include <hip/hip_runtime.h>

#include "euler3d_physics.hpp"
#include "handle.hpp"
#include "swe_kernels.hpp"
#include "speed_max.hpp"
#include "step_control.hpp"

namespace atmo {

namespace {

constexpr int NV = 3, NA = 26;

// quotients a / h and b / h from one refined reciprocal (each within one unit
// in the last place of the IEEE quotient, as div_nr)
__device__ __forceinline__ void div2(double a, double b, double h, double& qa, double& qb) {
  const double r = rcp_refined(h);
  qa = a * r;
  qb = b * r;
  qa = fma(fma(-h, qa, a), r, qa);
  qb = fma(fma(-h, qb, b), r, qb);
}

// J = sqrt(det G) and G^-1 = adj(G) / det G from the covariant metric tensor
// (metric_from_gcov with the shorter quotient and root of euler3d_physics.hpp);
// every kernel takes them from here, so each use gets the same bits
__device__ __forceinline__ void metric_of(double g11, double g12, double g22, double& J,
                                          double& c11, double& c12, double& c22) {
#pragma clang fp contract(off)
  const double det = fma(g11, g22, -(g12 * g12));
  const double inv = div_nr(1.0, det);
  J = sqrt_(det);
  c11 = g22 * inv;
  c12 = -g12 * inv;
  c22 = g11 * inv;
}

// CovariantShallowWaterEquations2D, the standard form (covariant_shallow_water.jl:166-187):
// contravariant flux in orientation o with the pressure term G^{io} g h^2 / 2
__device__ __forceinline__ void flux_standard(double g, double h, double hv1, double hv2,
                                              double J, double Gi_0o, double Gi_1o, double hvo,
                                              double vo, double* f) {
#pragma clang fp contract(off)
  const double grav = 0.5 * g * h * h;
  f[0] = J * hvo;
  f[1] = J * fma(hv1, vo, Gi_0o * grav);
  f[2] = J * fma(hv2, vo, Gi_1o * grav);
}

// what the node-local source reads of one node
struct SourceIn {
  double h, hv[2], v[2], vc[2];  // vc: covariant velocity G v
  double J, c11, c12, c22, sin_lat;
  double gam[6];  // Gamma^1_11, _12, _22, Gamma^2_11, _12, _22
};

// the Coriolis term 2 omega sin(lat) J (G^{k2} h v^1 - G^{k1} h v^2)
__device__ __forceinline__ double coriolis(double fJ, double ck1, double ck2, const double* hv) {
#pragma clang fp contract(off)
  return fJ * fma(ck2, hv[0], -(ck1 * hv[1]));
}

// source_terms_geometric_coriolis of the standard form (covariant_shallow_water.jl:215-238)
__device__ __forceinline__ void source_standard(double g, double omega, const SourceIn& a,
                                                double* s) {
#pragma clang fp contract(off)
  const double grav = 0.5 * g * a.h * a.h;
  // tau^{ij} = h v^i v^j + G^{ij} g h^2 / 2 (symmetric)
  const double t11 = fma(a.hv[0], a.v[0], grav * a.c11);
  const double t12 = fma(a.hv[0], a.v[1], grav * a.c12);
  const double t22 = fma(a.hv[1], a.v[1], grav * a.c22);
  const double fJ = 2 * omega * a.sin_lat * a.J;
  s[0] = 0.0;
  s[1] = -(fma(a.gam[0], t11, fma(2.0 * a.gam[1], t12, a.gam[2] * t22)) +
           coriolis(fJ, a.c11, a.c12, a.hv));
  s[2] = -(fma(a.gam[3], t11, fma(2.0 * a.gam[4], t12, a.gam[5] * t22)) +
           coriolis(fJ, a.c12, a.c22, a.hv));
}

// covariant_shallow_water_split.jl:273-302.  The reference's G_{ia} h v^a v^j
// is the covariant velocity times h v^j.
__device__ __forceinline__ void source_split(double omega, const SourceIn& a, double* s) {
#pragma clang fp contract(off)
  const double w11 = a.hv[0] * a.v[0], w12 = a.hv[0] * a.v[1], w22 = a.hv[1] * a.v[1];
  const double m00 = a.vc[0] * a.hv[0], m01 = a.vc[0] * a.hv[1];
  const double m10 = a.vc[1] * a.hv[0], m11 = a.vc[1] * a.hv[1];
  const double t1 = fma(a.gam[0], w11, fma(2.0 * a.gam[1], w12, a.gam[2] * w22));
  const double t2 = fma(a.gam[3], w11, fma(2.0 * a.gam[4], w12, a.gam[5] * w22));
  const double r1 = fma(a.gam[0], m00, a.gam[1] * m01) + fma(a.gam[3], m10, a.gam[4] * m11);
  const double r2 = fma(a.gam[1], m00, a.gam[2] * m01) + fma(a.gam[4], m10, a.gam[5] * m11);
  const double fJ = 2 * omega * a.sin_lat * a.J;
  s[0] = 0.0;
  s[1] = -fma(0.5, t1 - fma(a.c11, r1, a.c12 * r2), coriolis(fJ, a.c11, a.c12, a.hv));
  s[2] = -fma(0.5, t2 - fma(a.c12, r1, a.c22 * r2), coriolis(fJ, a.c12, a.c22, a.hv));
}

// Group of elements: WAVES waves of 64 lanes with one lane per node hold EPB =
// WAVES * 64 / n^2 elements (n^2 <= 64)
template <int N, int WAVES>
struct SweShape {
  static constexpr int N2 = N * N;
  static constexpr int LANES = 64 * WAVES;
  static constexpr int EPB = LANES / N2;
  static constexpr int NF = 4 * N;  // face nodes per element
  // passes of the face nodes over the group's lanes
  static constexpr int PASSES = (EPB * NF + LANES - 1) / LANES;
};

// per-node fields staged in LDS: h, hv^1, hv^2, v^1, v^2 (v = hv / h), J, the
// covariant velocity (G v)_1, (G v)_2, G^11, G^12, G^22, h_s
constexpr int kSweFields = 12;

// the stage's geometry rows and face maps in their storage type GT (double, or
// float under ATMO_PREC_FP32_GEOMETRY); a float operand widens to double in
// every expression it enters
template <typename GT>
__device__ __forceinline__ const GT* geo_rows(const SweLaunch& L) {
  if constexpr (sizeof(GT) == 4) return L.geo32; else return L.geo;
}
template <typename GT>
__device__ __forceinline__ const GT* face_maps(const SweLaunch& L) {
  if constexpr (sizeof(GT) == 4) return L.fxf32; else return L.fxf;
}

// a face node's inputs from memory: the neighbour's state and the map of its
// momentum into the own basis
template <typename GT>
struct FaceIn {
  double u[NV];
  GT M[4];
};

template <int N, int WAVES, typename GT>
__device__ __forceinline__ bool face_load(const SweLaunch& L, int e0, int fid, FaceIn<GT>& x) {
  using S = SweShape<N, WAVES>;
  const int fe = fid / S::NF;
  if (fid >= S::EPB * S::NF || e0 + fe >= L.n_elements) return false;
  const size_t fnode = (size_t)e0 * S::NF + fid;
  const GT* M = face_maps<GT>(L) + fnode * 4;
  const int link = L.nbr[fnode];
#pragma unroll
  for (int c = 0; c < 4; ++c) x.M[c] = M[c];
  const double* ur = L.u + (size_t)link * NV;
#pragma unroll
  for (int v = 0; v < NV; ++v) x.u[v] = ur[v];
  return true;
}

// surface flux plus half the nonconservative surface term of one face node,
// lifted by 1/w_end.  All of it is symmetric in the two states but for the
// dissipation: on a face whose outward normal points along -x_o both parts
// change sign and order, f*(own, nbr) for one side is
//   s (f#(own, nbr) + g / 2) - J lam (nbr - own) / 2,   s = +1 or -1.
// With one set of auxiliary variables on both sides the jump of h_s and the
// curvature part G^-1 G v - v of flux_nonconservative_ec vanish (:157-187),
// which leaves flux_nonconservative_surface_simplified (:229-250).
template <int N, typename GT>
__device__ __forceinline__ void face_flux(const SweLaunch& L, const double (*n)[N * N], int r,
                                          const FaceIn<GT>& x, double* fs) {
#pragma clang fp contract(off)
  const int f = r / N, k = r - f * N, o = f >> 1;
  const int i = f == 0 ? 0 : (f == 1 ? N - 1 : k);
  const int j = f == 2 ? 0 : (f == 3 ? N - 1 : k);
  const int q = i + N * j;
  const double sgn = (f & 1) ? 1.0 : -1.0;
  const double h = n[0][q], hv[2] = {n[1][q], n[2][q]}, v[2] = {n[3][q], n[4][q]};
  const double J = n[5][q], c1o = n[8 + o][q], c2o = n[9 + o][q], coo = n[8 + 2 * o][q];
  const double hvo = n[1 + o][q], vo = n[3 + o][q];
  // neighbour state in this element's contravariant basis (contravariant2global,
  // then global2contravariant: covariant_shallow_water.jl:140-153)
  const double ht = x.u[0];
  const double t1 = fma(x.M[0], x.u[1], x.M[1] * x.u[2]);
  const double t2 = fma(x.M[2], x.u[1], x.M[3] * x.u[2]);
  double vt1, vt2;
  div2(t1, t2, ht, vt1, vt2);
  const double to = o ? t2 : t1, vto = o ? vt2 : vt1;
  double F[NV];
  if (L.surface_flux == 3) {
    // flux_central of the standard form; no nonconservative term
    double fl[NV], fr[NV];
    flux_standard(L.gravity, h, hv[0], hv[1], J, c1o, c2o, hvo, vo, fl);
    flux_standard(L.gravity, ht, t1, t2, J, c1o, c2o, to, vto, fr);
#pragma unroll
    for (int c = 0; c < NV; ++c) F[c] = 0.5 * (fl[c] + fr[c]);
  } else {
    const double half_J = 0.5 * J;
    const double m = half_J * (hvo + to);
    F[0] = m;
    if (L.surface_flux == 1) {  // flux_central of the split flux (:66-80)
      F[1] = half_J * fma(hvo, v[0], to * vt1);
      F[2] = half_J * fma(hvo, v[1], to * vt2);
    } else {  // flux_ec (:100-122)
      F[1] = 0.5 * (v[0] + vt1) * m;
      F[2] = 0.5 * (v[1] + vt2) * m;
    }
    const double pr = half_J * (L.gravity * h * ht);
    F[1] = fma(pr, c1o, F[1]);
    F[2] = fma(pr, c2o, F[2]);
  }
#pragma unroll
  for (int c = 0; c < NV; ++c) F[c] *= sgn;
  if (L.surface_flux != 2) {  // DissipationLocalLaxFriedrichs, equations.jl:283-290
    const double gc = L.gravity * coo;
    const double lam = fmax(fabs(vo) + sqrt_(gc * h), fabs(vto) + sqrt_(gc * ht));
    const double d = -0.5 * J * lam;
    F[0] = fma(d, ht - h, F[0]);
    F[1] = fma(d, t1 - hv[0], F[1]);
    F[2] = fma(d, t2 - hv[1], F[2]);
  }
#pragma unroll
  for (int c = 0; c < NV; ++c) fs[c] = F[c] * L.inv_w;
}

// volume terms of node q along direction o: the sums over the partners in
// rotated order own + 1, ..., own + n - 1 (mod n), so every lane has a partner
// in each step.  Split form: with m = J hv^o of the two nodes, 4 times the term
// is (f#_h: 2 (m_l + m_r)), (v_l + v_r) (m_l + m_r) + m_l ((G^-1 (G v)_r) - v_r)
// + 2 g J h G^{.o} (h_r + h_s,r - h_s,l); the powers of two are applied to the
// sums, which rounds as applying them to each term.
template <int N, int UNROLL>
__device__ __forceinline__ void volume_terms(const SweLaunch& L, const double (*n)[N * N],
                                             const double* s_ds, int q, int o, double* sum) {
#pragma clang fp contract(off)
  const int ti = q % N, tj = q / N;
  const int own = o == 0 ? ti : tj, stride = o == 0 ? 1 : N;
  sum[0] = sum[1] = sum[2] = 0.0;
  if (L.volume_flux == 2) {
    // weak form (dg_2d_manifold_in_3d_covariant.jl:100-130): derivative_hat of
    // the standard flux, evaluated in place for every node of the line
    const int base = q - own * stride;
#pragma unroll
    for (int m = 0; m < N; ++m) {
      const int p = base + m * stride;
      double f[NV];
      flux_standard(L.gravity, n[0][p], n[1][p], n[2][p], n[5][p], n[8 + o][p], n[9 + o][p],
                    n[1 + o][p], n[3 + o][p], f);
      const double d = s_ds[own * N + m];
#pragma unroll
      for (int v = 0; v < NV; ++v) sum[v] = fma(d, f[v], sum[v]);
    }
    return;
  }
  const double hl = n[0][q], vl0 = n[3][q], vl1 = n[4][q], Jl = n[5][q], hsl = n[11][q];
  const double c11 = n[8][q], c12 = n[9][q], c22 = n[10][q];
  const double ml = Jl * n[1 + o][q];
  const double pf = 2.0 * L.gravity * Jl * hl;
  const double p0 = pf * (o == 0 ? c11 : c12), p1 = pf * (o == 0 ? c12 : c22);
  const bool ec = L.volume_flux == 0;
#pragma unroll UNROLL
  for (int j = 1; j < N; ++j) {
    const int step = own + j >= N ? j - N : j;
    const int p = q + step * stride;
    const double vr0 = n[3][p], vr1 = n[4][p], vc0 = n[6][p], vc1 = n[7][p];
    const double mr = n[5][p] * n[1 + o][p];
    const double ms = ml + mr;
    const double hh = n[0][p] + (n[11][p] - hsl);
    double a0, a1;
    if (ec) {  // flux_ec (:100-122)
      a0 = (vl0 + vr0) * ms;
      a1 = (vl1 + vr1) * ms;
    } else {  // flux_central of the split flux (:66-80)
      a0 = 2.0 * fma(ml, vl0, mr * vr0);
      a1 = 2.0 * fma(ml, vl1, mr * vr1);
    }
    // flux_nonconservative_ec (:157-187) of (own, partner)
    a0 += fma(ml, fma(c11, vc0, c12 * vc1) - vr0, p0 * hh);
    a1 += fma(ml, fma(c12, vc0, c22 * vc1) - vr1, p1 * hh);
    const double ds = s_ds[own * (N + 1) + step];
    sum[0] = fma(ds, ms, sum[0]);
    sum[1] = fma(ds, a0, sum[1]);
    sum[2] = fma(ds, a1, sum[2]);
  }
  sum[0] *= 0.5;
  sum[1] *= 0.25;
  sum[2] *= 0.25;
}

}  // namespace

// StepsizeCallback's scaled wave speeds at one node (stepsize_dg2d.jl:47-71):
// |v^i| + sqrt(G^ii h g); the max-speed reduction and the last stage of a
// resident step both call this one function, so their speeds agree bit for bit
__device__ __forceinline__ void swe_node_speeds(const double* u, double gcon11, double gcon22,
                                                double gravity, double l[2]) {
#pragma clang fp contract(off)
  double v1, v2;
  div2(u[1], u[2], u[0], v1, v2);
  l[0] = fabs(v1) + sqrt_(gcon11 * u[0] * gravity);
  l[1] = fabs(v2) + sqrt_(gcon22 * u[0] * gravity);
}

// SPEED: the RK stage also writes L.speed_partial (the last stage of a
// resident step); a variant of its own, so the other stages keep their
// register budget
// CONTROL: the first stage of a resident step forms its step size itself: the
// loads of its node waves go out with the node's own, the reduction follows
// the volume terms, while the face waves are still busy
template <int N, int WAVES, bool SPLIT, bool SPEED, bool CONTROL, typename GT>
__global__ __launch_bounds__((SPLIT ? 3 : 1) * 64 * WAVES)
__attribute__((amdgpu_waves_per_eu(N == 4 && !SPLIT ? 5 : 1)))
void swe_stage(SweLaunch L) {
#pragma clang fp contract(off)
  using S = SweShape<N, WAVES>;
  constexpr int N2 = S::N2, EPB = S::EPB, B = S::LANES;
  constexpr int UNROLL = SPLIT && N <= 5 ? N : 1;
  __shared__ double s_n[EPB][kSweFields][N2];
  __shared__ double s_sf[EPB][NV][S::NF];
  __shared__ double s_d1[SPLIT ? EPB : 1][NV][N2];  // the second direction's volume terms
  __shared__ double s_ds[N2];

  const int role = SPLIT ? __builtin_amdgcn_readfirstlane(threadIdx.x / B) : 0;
  const bool node_role = role == 0, dir1_role = !SPLIT || role == 1, face_role = !SPLIT || role == 2;
  const int t = threadIdx.x - role * B;
  const int e0 = blockIdx.x * EPB;
  const int es = t / N2, q = t - es * N2;
  const int ti = q % N, tj = q / N;
  const int e = e0 + es;
  const bool active = es < EPB && e < L.n_elements;
  const size_t g = (size_t)e * N2 + q;
  const long long NN = L.n_nodes;

  // the first pass's neighbour states are loaded before anything else is waited for
  FaceIn<GT> fin;
  bool has_face = false;
  if (face_role) has_face = face_load<N, WAVES, GT>(L, e0, t, fin);
  if (dir1_role && t < N2) s_ds[t] = L.volume_flux == 2 ? L.dhat[t] : L.dsplit[t];
  if (node_role && active) {
    const double* un = L.u + g * NV;
    const GT* gg = geo_rows<GT>(L) + g;
    const double h = un[0], hv1 = un[1], hv2 = un[2];
    const double G11 = gg[0], G12 = gg[NN], G22 = gg[2 * NN];
    double hs = 0.0;
    if (L.topography) {
      if constexpr (sizeof(GT) == 4) hs = L.hs64[g];
      else hs = gg[3 * NN];
    }
    double v1, v2, J, c11, c12, c22;
    div2(hv1, hv2, h, v1, v2);
    metric_of(G11, G12, G22, J, c11, c12, c22);
    // FP32 storage: J is the stored area element rounded once; it is the
    // same number on both sides of a face (G is not: it is expressed in each
    // element's own basis), so the two mass fluxes there agree
    if constexpr (sizeof(GT) == 4) J = gg[11 * NN];
    s_n[es][0][q] = h;
    s_n[es][1][q] = hv1;
    s_n[es][2][q] = hv2;
    s_n[es][3][q] = v1;
    s_n[es][4][q] = v2;
    s_n[es][5][q] = J;
    s_n[es][6][q] = fma(G11, v1, G12 * v2);
    s_n[es][7][q] = fma(G12, v1, G22 * v2);
    s_n[es][8][q] = c11;
    s_n[es][9][q] = c12;
    s_n[es][10][q] = c22;
    s_n[es][11][q] = hs;
  }
  // the node's remaining inputs: source geometry, register, step size
  SourceIn src;
  double kreg[NV], dt = L.rk_dt;
  auto load_rest = [&]() {
    if (L.source_terms) {
      const GT* gg = geo_rows<GT>(L) + g;
#pragma unroll
      for (int c = 0; c < 6; ++c) src.gam[c] = gg[(4 + c) * NN];
      src.sin_lat = gg[10 * NN];
    }
    if (L.mode != 0) {
#pragma unroll
      for (int v = 0; v < NV; ++v) kreg[v] = L.k[v * NN + g];
      if (!CONTROL && L.dt_member) dt = L.dt_member[L.member[e]];
    }
  };
  if (SPLIT && node_role && active) load_rest();
  double speeds[CONTROL ? 8 : 1];
  ClockIn clk{};
  if (CONTROL && node_role) {
    clk = load_clock(L.clock_in, L.clock_in + 1, 0, 1);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int i = (t & 63) + 64 * k;
      speeds[CONTROL ? k : 0] = i < L.n_elements ? L.control_partial[i] : 0.0;
    }
  }
  __syncthreads();

  double du[NV], d1[NV];
  if (node_role && active) volume_terms<N, UNROLL>(L, s_n[es], s_ds, q, 0, du);
  if (CONTROL && node_role) {  // each wave for itself
    double m = 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k) m = speed_max(m, speeds[CONTROL ? k : 0]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = speed_max(m, __shfl_xor(m, o, 64));
    const ClockOut next = step_control(m, clk, N);
    dt = next.dt;
    if (blockIdx.x == 0 && t == 0) {
      L.clock_out[0] = next.t;
      L.clock_out[1] = next.dt;
      L.clock_out[2] = next.steps;
      L.clock_out[3] = next.failed ? 1.0 : L.clock_in[3];
      L.clock_out[4] = clk.t_end;
      L.clock_out[5] = clk.cfl;
    }
  }
  if (dir1_role && active) {
    volume_terms<N, UNROLL>(L, s_n[es], s_ds, q, 1, d1);
    if constexpr (SPLIT) {
#pragma unroll
      for (int v = 0; v < NV; ++v) s_d1[es][v][q] = d1[v];
    }
  }
  if (!SPLIT && active) {
    load_rest();
#pragma unroll
    for (int v = 0; v < NV; ++v) du[v] += d1[v];
  }
  if (face_role) {
#pragma unroll
    for (int ps = 0; ps < S::PASSES; ++ps) {
      const int fid = t + ps * B;
      if (ps > 0) has_face = face_load<N, WAVES, GT>(L, e0, fid, fin);
      if (!has_face) continue;
      const int fe = fid / S::NF, r = fid - fe * S::NF;
      double fs[NV];
      face_flux<N, GT>(L, s_n[fe], r, fin, fs);
#pragma unroll
      for (int v = 0; v < NV; ++v) s_sf[fe][v][r] = fs[v];
    }
  }
  __syncthreads();
  if (node_role && active) {
    if constexpr (SPLIT) {
#pragma unroll
      for (int v = 0; v < NV; ++v) du[v] += s_d1[es][v][q];
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const bool on = f == 0 ? ti == 0 : f == 1 ? ti == N - 1 : f == 2 ? tj == 0 : tj == N - 1;
      if (!on) continue;
      const int k = f < 2 ? tj : ti;
#pragma unroll
      for (int v = 0; v < NV; ++v) du[v] += s_sf[es][v][f * N + k];
    }
    src.h = s_n[es][0][q];
    src.hv[0] = s_n[es][1][q];
    src.hv[1] = s_n[es][2][q];
    src.J = s_n[es][5][q];
    const double fac = div_nr(-1.0, src.J);
#pragma unroll
    for (int v = 0; v < NV; ++v) du[v] *= fac;
    if (L.source_terms) {
      src.v[0] = s_n[es][3][q];
      src.v[1] = s_n[es][4][q];
      src.vc[0] = s_n[es][6][q];
      src.vc[1] = s_n[es][7][q];
      src.c11 = s_n[es][8][q];
      src.c12 = s_n[es][9][q];
      src.c22 = s_n[es][10][q];
      double sv[NV];
      if (L.source_terms == 2) source_standard(L.gravity, L.rotation_rate, src, sv);
      else source_split(L.rotation_rate, src, sv);
#pragma unroll
      for (int v = 0; v < NV; ++v) du[v] += sv[v];
    }
    if (L.mode == 0) {
#pragma unroll
      for (int v = 0; v < NV; ++v) L.out[g * NV + v] = du[v];
    } else {
      const double uo[NV] = {src.h, src.hv[0], src.hv[1]};
      double un[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const double kn = fma(L.rk_a, kreg[v], dt * du[v]);
        L.k[v * NN + g] = kn;
        un[v] = fma(L.rk_b, kn, uo[v]);
      }
#pragma unroll
      for (int v = 0; v < NV; ++v) L.out[g * NV + v] = un[v];
      if constexpr (SPEED) {
        // the node's speeds go to its first two LDS fields, which only this
        // lane reads after the face phase and which it has read already
        double l[2];
        swe_node_speeds(un, s_n[es][8][q], s_n[es][10][q], L.gravity, l);
        s_n[es][0][q] = l[0];
        s_n[es][1][q] = l[1];
      }
    }
  }
  if constexpr (SPEED) {
    // per element: the maximum over its nodes of each speed (exact in any
    // order), one lane per line of nodes and then its first lane over the
    // lines, and the sum over the directions
    __syncthreads();
    if (node_role && active && tj == 0) {
      double m1 = s_n[es][0][ti], m2 = s_n[es][1][ti];
#pragma unroll
      for (int r = 1; r < N; ++r) {
        m1 = speed_max(m1, s_n[es][0][ti + N * r]);
        m2 = speed_max(m2, s_n[es][1][ti + N * r]);
      }
      s_n[es][2][ti] = m1;
      s_n[es][3][ti] = m2;
    }
    __syncthreads();
    if (node_role && active && q == 0) {
      double m1 = s_n[es][2][0], m2 = s_n[es][3][0];
#pragma unroll
      for (int r = 1; r < N; ++r) {
        m1 = speed_max(m1, s_n[es][2][r]);
        m2 = speed_max(m2, s_n[es][3][r]);
      }
      L.speed_partial[e] = m1 + m2;
    }
  }
}

// per-element maximum of the scaled wave speeds (stepsize_dg2d.jl:47-71)
// G^11 and G^22 are recomputed from the stage's G rows in their storage type,
// as the fused last stage does
template <int N, typename GT>
__global__ __launch_bounds__(64) void swe_max_speed(SweLaunch L, double* partial) {
  constexpr int N2 = N * N;
  const int e = blockIdx.x, t = threadIdx.x;
  __shared__ double s1[64], s2[64];
  double l1 = 0.0, l2 = 0.0;
  const GT* gr = geo_rows<GT>(L);
  for (int q = t; q < N2; q += 64) {
    const size_t g = (size_t)e * N2 + q;
    const double* u = L.u + g * NV;
    double J, c11, c12, c22, l[2];
    metric_of(gr[g], gr[L.n_nodes + g], gr[2 * L.n_nodes + g], J, c11, c12, c22);
    swe_node_speeds(u, c11, c22, L.gravity, l);
    l1 = speed_max(l1, l[0]);
    l2 = speed_max(l2, l[1]);
  }
  s1[t] = l1;
  s2[t] = l2;
  __syncthreads();
  for (int w = 32; w > 0; w >>= 1) {
    if (t < w) {
      s1[t] = speed_max(s1[t], s1[t + w]);
      s2[t] = speed_max(s2[t], s2[t + w]);
    }
    __syncthreads();
  }
  if (t == 0) partial[e] = s1[0] + s2[0];
}

namespace {

template <int N, int WAVES, bool SPLIT>
void launch_variant(const SweLaunch& L, hipStream_t s) {
  using S = SweShape<N, WAVES>;
  const dim3 grid((L.n_elements + S::EPB - 1) / S::EPB), block((SPLIT ? 3 : 1) * S::LANES);
  const bool speed = L.speed_partial && L.mode == 1;
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, s, L); };
  if constexpr (SPLIT) {
    if (L.control_partial) {
      if (L.geo32) go(swe_stage<N, WAVES, SPLIT, false, true, float>);
      else go(swe_stage<N, WAVES, SPLIT, false, true, double>);
      return;
    }
  }
  if (L.geo32) {
    if (speed) go(swe_stage<N, WAVES, SPLIT, true, false, float>);
    else go(swe_stage<N, WAVES, SPLIT, false, false, float>);
  } else if (speed) {
    go(swe_stage<N, WAVES, SPLIT, true, false, double>);
  } else {
    go(swe_stage<N, WAVES, SPLIT, false, false, double>);
  }
}

template <int N>
bool launch_n(const SweLaunch& L, int variant, hipStream_t s) {
  // variants: 0..2 = node lanes of 1, 2, 4 waves; 3..5 the same, split
  if constexpr (N * N > 64) {
    return false;
  } else {
    switch (variant) {
      case 0: launch_variant<N, 1, false>(L, s); return true;
      case 1: launch_variant<N, 2, false>(L, s); return true;
      case 2: launch_variant<N, 4, false>(L, s); return true;
      case 3: launch_variant<N, 1, true>(L, s); return true;
      case 4: launch_variant<N, 2, true>(L, s); return true;
      case 5: launch_variant<N, 4, true>(L, s); return true;
    }
    return false;
  }
}

}  // namespace

bool swe_launch_stage(const SweLaunch& L, hipStream_t s) {
  const int variant = L.variant;
  switch (L.n) {
    case 2: return launch_n<2>(L, variant, s);
    case 3: return launch_n<3>(L, variant, s);
    case 4: return launch_n<4>(L, variant, s);
    case 5: return launch_n<5>(L, variant, s);
    case 6: return launch_n<6>(L, variant, s);
    case 7: return launch_n<7>(L, variant, s);
    case 8: return launch_n<8>(L, variant, s);
  }
  return false;
}

bool swe_launch_member_max_speed(const SweLaunch& L, double* partial, const int* member_first,
                                 int n_members, double* out, hipStream_t s) {
#define ATMO_SWE_CASE(NN)                                                                       \
  case NN:                                                                                      \
    if (L.geo32)                                                                                \
      hipLaunchKernelGGL((swe_max_speed<NN, float>), dim3(L.n_elements), dim3(64), 0, s, L,     \
                         partial);                                                              \
    else                                                                                        \
      hipLaunchKernelGGL((swe_max_speed<NN, double>), dim3(L.n_elements), dim3(64), 0, s, L,    \
                         partial);                                                              \
    break;
  switch (L.n) {
    ATMO_SWE_CASE(2)
    ATMO_SWE_CASE(3)
    ATMO_SWE_CASE(4)
    ATMO_SWE_CASE(5)
    ATMO_SWE_CASE(6)
    ATMO_SWE_CASE(7)
    ATMO_SWE_CASE(8)
    default:
      return false;
  }
#undef ATMO_SWE_CASE
  launch_member_max(partial, member_first, n_members, out, s);
  return true;
}

}  // namespace atmo

namespace atmo {

namespace {
// the rows of one node's 26 auxiliary variables that the integrals read
struct AuxV {
  const double* a;
  __device__ __forceinline__ double J() const { return a[12]; }
  __device__ __forceinline__ double Gcov(int i, int j) const { return a[13 + i + j]; }
  __device__ __forceinline__ double hs() const { return a[19]; }
};
}  // namespace

// per element: mass, total energy (entropy) and int w(u).du with the exact
// area element (analysis_covariant.jl:53-105; covariant_shallow_water.jl:129-164)
template <int N>
__global__ __launch_bounds__(64) void swe_integrals_kernel(SweLaunch L, const double* du,
                                                           const double* w, double* partial) {
  constexpr int N2 = N * N;
  const int e = blockIdx.x, t = threadIdx.x;
  __shared__ double s[3][64];
  double a0 = 0, a1 = 0, a2 = 0;
  for (int q = t; q < N2; q += 64) {
    const size_t g = (size_t)e * N2 + q;
    const double* u = L.u + g * NV;
    const AuxV a{L.aux + g * NA};
    const double h = u[0], v1 = u[1] / h, v2 = u[2] / h;
    const double vc1 = a.Gcov(0, 0) * v1 + a.Gcov(0, 1) * v2;
    const double vc2 = a.Gcov(1, 0) * v1 + a.Gcov(1, 1) * v2;
    const double wJ = w[q % N] * w[q / N] * a.J();
    a0 += wJ * h;
    a1 += wJ * (0.5 * (h * (vc1 * v1 + vc2 * v2) + L.gravity * h * h) + L.gravity * h * a.hs());
    if (du) {
      const double w1 = L.gravity * (h + a.hs()) - 0.5 * (vc1 * v1 + vc2 * v2);
      a2 += wJ * (w1 * du[g * NV] + vc1 * du[g * NV + 1] + vc2 * du[g * NV + 2]);
    }
  }
  s[0][t] = a0;
  s[1][t] = a1;
  s[2][t] = a2;
  __syncthreads();
  for (int k = 32; k > 0; k >>= 1) {
    if (t < k)
      for (int c = 0; c < 3; ++c) s[c][t] += s[c][t + k];
    __syncthreads();
  }
  if (t < 3) partial[(size_t)t * gridDim.x + e] = s[t][0];
}

bool swe_launch_integrals(const SweLaunch& L, const double* du, const double* w, double* partial,
                          double* out, hipStream_t s) {
#define ATMO_SWE_CASE(NN)                                                                     \
  case NN:                                                                                    \
    hipLaunchKernelGGL(swe_integrals_kernel<NN>, dim3(L.n_elements), dim3(64), 0, s, L, du, w, \
                       partial);                                                              \
    break;
  switch (L.n) {
    ATMO_SWE_CASE(2)
    ATMO_SWE_CASE(3)
    ATMO_SWE_CASE(4)
    ATMO_SWE_CASE(5)
    ATMO_SWE_CASE(6)
    ATMO_SWE_CASE(7)
    ATMO_SWE_CASE(8)
    default:
      return false;
  }
#undef ATMO_SWE_CASE
  launch_sum_rows(partial, L.n_elements, 3, out, s);
  return true;
}

}  // namespace atmo
