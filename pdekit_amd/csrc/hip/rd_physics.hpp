// Point-wise physics of the cell loop, device side.
//
// Restates compute_properties / flux / the upwind matrix K+ = R max(L,0) L^-1
// of src/physics/scalar/RotationAdvection2D.hpp:201-336 (constant velocity),
// src/physics/scalar/Burgers2D.hpp:154-275, src/physics/euler/
// Euler2DCons.hpp:159-536 and Euler3DCons.hpp:159-450.
//
// For the Euler systems K+ is applied in the form
//   K+ = l0+ I + (lp+ - l0+) r_p l_p^T + (lm+ - l0+) r_m l_m^T,
// which follows from R L = I and the multiplicity of the convective
// eigenvalue u.n: only the two acoustic eigenvector pairs (r_p, l_p),
// (r_m, l_m) enter. Entries of r and l are those of the reference's R and
// L columns/rows for the eigenvalues |g| (u.n + a) and |g| (u.n - a).
#pragma once

#include <hip/hip_runtime.h>

namespace pdrd {

// PH_ROTATION2D: advection with the velocity (y, -x) of the point (the
// kernels pass it in the PhysParams of each point).
enum { PH_ADVECTION2D = 0, PH_BURGERS2D = 1, PH_EULER2D = 2, PH_EULER3D = 3, PH_ROTATION2D = 4 };
// SC_BPSI: the PSI / LDA blend, (1 - theta) LDA + theta PSI with the cell
// theta of PGB
enum { SC_LDA = 0, SC_N = 1, SC_B = 2, SC_PSI = 3, SC_BPSI = 4 };

template <int PH> struct PhysTraits;
template <> struct PhysTraits<PH_ADVECTION2D> { static constexpr int M = 1, DIM = 2; };
template <> struct PhysTraits<PH_ROTATION2D> { static constexpr int M = 1, DIM = 2; };
template <> struct PhysTraits<PH_BURGERS2D> { static constexpr int M = 1, DIM = 2; };
template <> struct PhysTraits<PH_EULER2D> { static constexpr int M = 4, DIM = 2; };
template <> struct PhysTraits<PH_EULER3D> { static constexpr int M = 5, DIM = 3; };

// Whether the P+1 flux element of a cell with ND nodes and NV vertices
// interpolates the scalar flux exactly (its divergence is then a . grad u).
template <int PH, int NV, int ND>
struct ScalarFlux
{
  static constexpr bool exact = PH == PH_ADVECTION2D || PH == PH_ROTATION2D || (PH == PH_BURGERS2D && ND == NV);
};

struct PhysParams
{
  double p0, p1;  // advection velocity (ax, ay) -- for PH_ROTATION2D the point's -- or (gamma, R)
};

// 1/x for |x| and 1/|x| in the normal range: the hardware reciprocal
// estimate y (relative error below 2^-22) with the error e = 1 - x y taken out
// to third order, y (1 + e + e^2): its truncation error e^3 is below 2^-66, so
// the result is the IEEE quotient but for 2 of 100 000 arguments, which round
// the other way, at a third of the instructions of the IEEE division sequence.
// x = 0 gives NaN. (A product n * recip(x) rounds twice: up to 1.5 ulp off the
// quotient n / x.)
__device__ __forceinline__ double recip(double x)
{
  const double y = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, y, 1.0);
  return fma(y, fma(e, e, e), y);
}

// n/x for x as in recip: the product with the reciprocal, its residual n - x q taken
// out once, which rounds as the IEEE quotient does (Markstein), at 7 dependent
// operations instead of 11.
__device__ __forceinline__ double quotient(double n, double x)
{
  const double r = recip(x);
  const double q = n * r;
  return fma(fma(-x, q, n), r, q);
}

// sqrt(x) and 1/sqrt(x) for x > 0 in the normal range, from one hardware
// reciprocal square root estimate y (relative error below 2^-22) with its
// error e = 1 - x y^2 (below 2^-21) taken out to third order, y (1 + e/2 +
// 3 e^2 / 8); the next term of the series, 5 e^3 / 16, is below 2^-64, so
// 1/sqrt(x) is within an ulp. Its product with x would be up to 1.7 ulp off the
// square root; the correction by half the residual x - s^2 takes that to 0.5.
// Replaces a square root and a division; x = 0 gives NaN for both.
__device__ __forceinline__ void sqrt_rsqrt(double x, double &s, double &rs)
{
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  rs = fma(y * e, fma(0.375, e, 0.5), y);
  const double g = x * rs;
  s = fma(fma(-g, g, x), 0.5 * rs, g);
}

// Thermodynamic state at a point (Euler); inv_a = 1 / a.
template <typename T, int D>
struct EulerState
{
  T rho, inv_rho, V[D], v2, P, H, a, inv_a;
  bool bad;
};

template <typename T, int D>
__device__ __forceinline__ EulerState<T, D> euler_state(const T *s, T gamma)
{
  EulerState<T, D> st;
  const T gm1 = gamma - T(1);
  st.rho = s[0];
  st.inv_rho = recip(st.rho);
  T v2 = T(0);
#pragma unroll
  for (int d = 0; d < D; ++d) {
    st.V[d] = s[1 + d] * st.inv_rho;
    v2 += st.V[d] * st.V[d];
  }
  st.v2 = v2;
  const T rhoE = s[D + 1];
  st.P = gm1 * (rhoE - T(0.5) * st.rho * st.v2);
  st.bad = !(st.P > T(0));
  const T RT = st.P * st.inv_rho;
  st.H = rhoE * st.inv_rho + RT;
  sqrt_rsqrt(gamma * RT, st.a, st.inv_a);
  return st;
}

// out += F(s) . b for the Euler fluxes at a state of momentum s[1..D] and a
// direction b (Euler fluxes contracted before they are formed: 3 D + 1
// operations instead of D (D + 1) for the fluxes and D (D + 2) for the product).
template <int D>
__device__ __forceinline__ void euler_flux_add(const double *s, const EulerState<double, D> &st, const double *b,
                                               double *out)
{
  double mb = 0.0;
#pragma unroll
  for (int d = 0; d < D; ++d) mb += s[1 + d] * b[d];
  out[0] += mb;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const double t = out[1 + d] + st.V[d] * mb;
    out[1 + d] = t + st.P * b[d];
  }
  out[D + 1] += st.H * mb;
}

// Physical flux F[d][k] at a state.
template <int PH, typename T>
__device__ __forceinline__ void point_flux(const T *s, const PhysParams &pp, T F[][PhysTraits<PH>::M], bool &bad)
{
  if constexpr (PH == PH_ADVECTION2D || PH == PH_ROTATION2D) {
    F[0][0] = T(pp.p0) * s[0];
    F[1][0] = T(pp.p1) * s[0];
  } else if constexpr (PH == PH_BURGERS2D) {
    F[0][0] = T(0.5) * s[0] * s[0];
    F[1][0] = s[0];
  } else {
    constexpr int D = PhysTraits<PH>::DIM;
    const EulerState<T, D> st = euler_state<T, D>(s, T(pp.p0));
    bad = bad || st.bad;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const T md = s[1 + d];
      F[d][0] = md;
#pragma unroll
      for (int k = 0; k < D; ++k) F[d][1 + k] = md * st.V[k] + ((k == d) ? st.P : T(0));
      F[d][D + 1] = md * st.H;
    }
  }
}

}  // namespace pdrd
