// pmw_common.h -- constants and pointwise device arithmetic shared by the
// PyMiniWeather HIP kernels (gfx950).
//
// Reconstruction, pressure, tendency and update keep the reference's
// floating-point operation order, and the library is compiled with
// -ffp-contract=off, so that they round like the NumPy code they replace. The
// expected differences from NumPy are fewer roundings in the fluxes' advective
// and viscous terms (flux_x_face), last-bit differences of the powers
// (pow_gamma of pmw_pow.h is correctly rounded in all but one of 3e6 cases,
// glibc's pow, which NumPy calls, in all but 8e-4) and of exp/cos in the
// initial conditions.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>

#include "pmw.h"
#include "pmw_pow.h"

namespace pmw {

// Device-global pointers. A pointer read from memory (a descriptor array)
// is generic to the compiler, which then emits flat_* accesses that also
// count against the LDS wait counter; typed in the global address space it
// emits global_* instead. Host code sees plain pointers (same layout).
#if defined(__HIP_DEVICE_COMPILE__)
#define PMW_GLOBAL __attribute__((address_space(1)))
#else
#define PMW_GLOBAL
#endif
using gdouble = PMW_GLOBAL double;
template <typename T>
__host__ __device__ inline PMW_GLOBAL T* gptr(T* p) {
  return (PMW_GLOBAL T*)p;
}

// A state element addressed from a block-uniform base (the start of a row
// or tile rows of one variable plane, kept in scalar registers) by a 32-bit
// byte offset per lane: one global access with a scalar base, instead of a
// 64-bit address computed per lane and access.
// The base goes through readfirstlane so that the compiler keeps it in
// scalar registers instead of folding the variable's plane offset into a
// per-lane 64-bit address.
__device__ __forceinline__ unsigned long long sgpr64(unsigned long long u) {
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
  return ((unsigned long long)hi << 32) | lo;
}
__device__ __forceinline__ double ld_off(const gdouble* base, unsigned boff) {
  const unsigned long long b = sgpr64((unsigned long long)base);
  return *(const gdouble*)((const PMW_GLOBAL char*)b + boff);
}
__device__ __forceinline__ void st_off(gdouble* base, unsigned boff, double v) {
  const unsigned long long b = sgpr64((unsigned long long)base);
  *(gdouble*)((PMW_GLOBAL char*)b + boff) = v;
}

// pyminiweather/data/constants.py:13-27 (rd is 287 in a float Enum -> 287.0)
constexpr double kHvBeta = 0.05;
constexpr double kP0 = 1.0e5;
constexpr double kC0 = 27.5629410929725921310572974482;
constexpr double kGamma = 1.40027894002789400278940027894;
constexpr double kGrav = 9.8;
constexpr double kCp = 1004.0;
constexpr double kCv = 717.0;
constexpr double kRd = 287.0;
constexpr double kPi = 3.14159265358979323846264338327;
constexpr double kTheta0 = 300.0;
constexpr double kExner0 = 1.0;

// Convolution weights in the order the direct correlation applies them
// (the stored kernels of data/fields.py:94-97, reversed).
constexpr double kW4a = -1.0 / 12;  // taps 0 and 3 of the 4th-order kernel
constexpr double kW4b = 7.0 / 12;   // taps 1 and 2
// 3rd-difference kernel [1,-3,3,-1] reversed: [-1, 3, -3, 1]

constexpr int kHs = 2;
constexpr int kNv = 4;

// Index helpers for a (4, nz+4, nx+4) state.
struct Grid {
  int nx, nz;
  int ld;          // nx + 4
  long long plane; // (nz + 4) * (nx + 4)
  __host__ __device__ Grid(int nx_, int nz_)
      : nx(nx_), nz(nz_), ld(nx_ + 4), plane((long long)(nz_ + 4) * (nx_ + 4)) {}
  __host__ __device__ long long at(int v, int prow, int pcol) const {
    return (long long)v * plane + (long long)prow * ld + pcol;
  }
};

// 1/b as y + yl, for quotients by b: y from v_rcp_f64 and one Newton step
// (relative error e below 2^-46), yl = e y the remainder, so that y + yl is
// 1/b to 2^-92, and a/b = RN(a y + RN(a yl)) is the correctly rounded
// quotient except with probability ~2^-38: 5 instructions, and 2 per
// quotient, instead of 10 for an IEEE reciprocal and 3. Unlike a division, a
// zero or infinite b gives NaN, and an infinite a gives an infinity or NaN with
// the sign of yl.
struct Recip {
  double y, yl;
};
__device__ __forceinline__ Recip recip(double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = fma(fma(-b, y, 1.0), y, y);
  return {y, fma(-b, y, 1.0) * y};
}
__device__ __forceinline__ double quot(double a, Recip r) { return fma(a, r.y, a * r.yl); }

// The remainder 1/d - id of a host reciprocal id = RN(1/d).
inline double recip_lo(double d, double id) { return std::fma(-d, id, 1.0) * id; }

// 4-tap reconstruction at one face: value and 3rd difference, accumulated
// left to right like scipy.signal.convolve's direct method.
__device__ __forceinline__ void recon4(double s0, double s1, double s2,
                                       double s3, double& val, double& d3) {
  val = ((s0 * kW4a + s1 * kW4b) + s2 * kW4b) + s3 * kW4a;
  d3 = ((s0 * -1.0 + s1 * 3.0) + s2 * -3.0) + s3 * 1.0;
}

// The power of a face: of any argument, or of 2^-6 <= x < 1024, where `rare` gets
// the lanes with other arguments (in scalar registers).
struct PowGamma {
  __device__ __forceinline__ double operator()(double x) const { return pow_gamma(x); }
};
struct PowGammaIn {
  unsigned long long& rare;
  __device__ __forceinline__ double operator()(double x) const {
    double s, l;
    unsigned k;
    pow_gamma_entry(x, s, l, k);
    rare |= __builtin_amdgcn_ballot_w64(k >= powt::kGamEntries);
    return s + l;
  }
};

// x-direction Euler flux with hyperviscosity (solve/interpolate.py:105-129).
// The pressure's argument rho * t, t = (rho*theta) / rho, keeps the
// reference's roundings (a last bit there is a last bit of a 1e5 Pa pressure).
// The advective terms take the reconstructed momentum m = rho u itself instead
// of rho * (m / rho), one product per term, and the products that are only
// added into a flux are not rounded before: fewer roundings than the
// reference's, which sit far below the pressure's last bit.
// power: PowGamma, or PowGammaIn where the caller looks at `rare` afterwards.
// CARRY: the mass flux of a face whose density is NaN or zero is NaN as rho * u
// would be, also where rho u itself is finite. The fused directions do without
// (0.5 to 1 % of a step): the other three fluxes of such a face are NaN, with them
// the momenta after the first stage, and the mass flux of the second.
template <bool CARRY, class Pow>
__device__ __forceinline__ void flux_x_face(const double val[4],
                                            const double d3[4], double hyr,
                                            double hyt, double hv,
                                            double F[4], Pow&& power) {
  const double rho = val[0] + hyr;
  const Recip r = recip(rho);
  const double u = quot(val[1], r);
  const double t = quot(val[3] + hyt, r);
  const double p = kC0 * power(rho * t);
  F[0] = fma(-hv, d3[0], CARRY ? fma(0.0, u, val[1]) : val[1]);
  F[1] = fma(-hv, d3[1], fma(val[1], u, p));
  F[2] = fma(-hv, d3[2], u * val[2]);
  F[3] = fma(-hv, d3[3], val[1] * t);
}

// z-direction flux (solve/interpolate.py:153-186); `wall` marks faces k = 0
// and k = nz, where w and the rho' 3rd difference are zeroed. CARRY as above; a
// wall's mass flux is rho * 0.
template <bool CARRY, class Pow>
__device__ __forceinline__ void flux_z_face(const double val[4], double d3[4],
                                            double hyr, double hyt,
                                            double hyp, double hv, bool wall,
                                            double G[4], Pow&& power) {
  const double rho = val[0] + hyr;
  const Recip r = recip(rho);
  const double m = wall ? 0.0 : val[2];  // rho w
  const double w = quot(m, r);
  const double t = quot(val[3] + hyt, r);
  const double p = kC0 * power(rho * t) - hyp;
  const double d0 = wall ? 0.0 : d3[0];
  G[0] = fma(-hv, d0, CARRY ? fma(0.0, wall ? rho : w, m) : m);
  G[1] = fma(-hv, d3[1], w * val[1]);
  G[2] = fma(-hv, d3[2], fma(m, w, p));
  G[3] = fma(-hv, d3[3], m * t);
}

// Tendency from two face fluxes (solve/interpolate.py:209-215, 239-245), with
// id + idl = 1/d to 2^-106 (recip_lo): the correctly rounded quotient.
__device__ __forceinline__ double tend_of(double f_lo, double f_hi, double id, double idl) {
  const double x = f_lo - f_hi;
  return fma(x, id, x * idl);
}

// Value the reference's set_bc_z leaves in z-halo row `prow` (0, 1, nz+2 or
// nz+3) of variable v, given the same column's value on the adjacent interior
// edge row (bcs.py:92-148). An IEEE division, so that an infinite momentum stays
// one (quot may make it NaN); only the wall's rows take it, and a step of every
// size from 100 x 50 to 8192 x 4096 takes as long with quot (+- 0.8 %).
__device__ __forceinline__ double wall_halo(int v, double edge_val,
                                            double hy_edge, double hy_halo) {
  if (v == 2) return 0.0;
  if (v == 1) return edge_val / hy_edge * hy_halo;
  return edge_val;
}

}  // namespace pmw

#define PMW_CHECK_LAUNCH()                         \
  do {                                             \
    hipError_t e_ = hipGetLastError();             \
    if (e_ != hipSuccess) return (int)e_;          \
  } while (0)
