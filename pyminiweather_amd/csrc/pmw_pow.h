// pmw_pow.h -- x^gamma for the pressure p = C0 (rho*theta)^gamma, and dp/dq.
//
// The kernels evaluate one power per face: pow_gamma in the fluxes, the
// background and the energy, pow_gamma_minus_one in the adjoint. Both take the
// fixed exponent into their tables (pmw_pow_tables.h, generated by
// gen_pow_tables.py). The powers of any exponent before them, pow_pos and its
// relatives, are what kernels used earlier; no kernel calls them any more, and
// the host tests hold them and, through them, the tables' generator.
//
// pow_pos evaluates x^y = exp(y ln x) for positive finite x with two small tables
// and double-double arithmetic where the rounding matters. The scheme is Tang's table-driven
// one (P. T. P. Tang, "Table-driven implementation of the logarithm function
// in IEEE floating-point arithmetic", ACM TOMS 16(4), 1990, and "... of the
// exponential function", ACM TOMS 15(2), 1989: reduce with a table entry,
// short polynomial, rebuild), with its table sizes and splits chosen here:
//
//   x = 2^e m, m in [1, 2); j = round(128 (m - 1)); c_j = 1/(1 + j/128) to 8
//   bits, so r = m c_j - 1 is exact in one fma and |r| < 0.0059:
//   ln x = e ln2 - ln c_j + log1p(r),  log1p(r) = r - r^2/2 + r^3 P(r)
//   z = y ln x  (double-double);  k = rint(256 z / ln2) = 256 n + i:
//   x^y = 2^n 2^(i/256) exp(s),  |s| <= ln2/512,  exp(s) = 1 + s + s^2 Q(s)
//
// -ln c_j, 2^(i/256), e ln2 and k ln2/256 are double-double; r^2 and s
// times the table value are exact Dekker products. The value before the
// final rounding is within 5e-22 relative of x^y (host maximum against
// 113-bit quadmath: 4.5e-22; the rounding of s^2 Q(s) dominates, which the
// 256-entry exp table keeps small), so the result is the correctly rounded
// one except when x^y lies that close to a rounding boundary (measured:
// ~1e-6 of arguments; glibc's pow, which NumPy calls, misses in 8e-4).
//
// pow_gamma evaluates the one power of the flux, x^gamma, without a logarithm
// or an exponential: the exponent is fixed, so (2^e / c_j)^gamma is a table and
// what is left is (1 + r)^gamma, |r| <= 2^-9, a short binomial series. About 40
// VALU instructions and one 16-byte load, against 131 and two dependent rounds of
// loads of pow_pos, at pow_pos's accuracy.
//
// pow_pos_near continues a power already evaluated at a nearby argument with
// the binomial series of (1 + e)^y and returns pow_pos's result bit for bit:
// where its own rounding could differ from pow_pos's, it evaluates pow_pos
// instead.
//
// Host and device share this code (the host build validates it); every fma
// is explicit and the library is compiled with -ffp-contract=off, so both
// evaluate the same roundings.
#pragma once

#include <math.h>
#include <string.h>

#include "pmw_pow_tables.h"

#ifndef __HIPCC__
#define PMW_HD inline
#else
#define PMW_HD __host__ __device__ __forceinline__
#endif

namespace pmw {

// TwoSum: s = RN(a + b), lo += the exact error (any magnitudes).
PMW_HD double two_sum(double a, double b, double& lo) {
  const double s = a + b;
  const double bb = s - a;
  lo = lo + ((a - (s - bb)) + (b - bb));
  return s;
}

// 1/x within an ulp or two for normal x (v_rcp_f64 and two Newton steps,
// enough from any start better than 2^-13) on the device; RN(1/x) on the
// host. The adjoint's quotients by rho are products with it; pow_pos_near stays
// equal to pow_pos with rx off by up to ~1e-14 relative (tests/test_pow_host.py;
// at 1e-13 it no longer is, through the e^2 terms evaluated from eh).
PMW_HD double rcp_approx(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
#else
  return 1.0 / x;
#endif
}

// The unrounded result of pow_pos at one argument, for continuing to nearby
// arguments with pow_pos_near: x^y = (h + l) with h + l within 5e-22
// relative of the exact power, x the argument and rx ~ 1/x (rcp_approx).
struct PowRef {
  double h, l, x, rx;
};

// x^y for 0 < y <= 1.5 (results of x in the physical range stay normal).
// Positive finite x take the scheme above; +-0, +-inf, other negative x and
// NaN give pow's results for such y (+0, +inf, NaN, NaN) through a final
// select, so no branch or call is compiled into the flux kernels.
PMW_HD double pow_pos_impl(double x, double y, PowRef* ref) {
  using namespace powt;
  const double inf = __builtin_inf();
  const bool fin = x > 0.0 && x < inf;
  const double sp = x == 0.0 ? 0.0 : (x == inf || x == -inf ? inf : __builtin_nan(""));
  int e;
  const double m = 2.0 * frexp(fin ? x : 1.0, &e);  // x = m 2^(e-1), m in [1, 2)
  // round(128 (m - 1)), 0..128: m * 128 and the difference are exact; the
  // mask states the range (a 32-bit table offset, no 64-bit index math)
  const unsigned j = (unsigned)(int)(m * 128.0 - 127.5) & 255u;
  const double r = fma(m, kLogC[j], -1.0);           // exact
  // log1p(r) = r - r^2/2 + r^3 (1/3 - r/4 + r^2/5 - ... + r^6/9). The
  // polynomial's own rounding reaches the result scaled by r^3 < 2.1e-7, so
  // its steps are a product and a sum each: two instructions, where an fma
  // with a constant addend costs three on gfx950 (the addend is copied into
  // the accumulator register first).
  const double r2 = r * r;
  const double r2l = fma(r, r, -r2);
  double q = 0x1.c71c71c71c71cp-4;                   // 1/9
  q = q * r + -0x1.0000000000000p-3;                 // -1/8
  q = q * r + 0x1.2492492492492p-3;                  // 1/7
  q = q * r + -0x1.5555555555555p-3;                 // -1/6
  q = q * r + 0x1.999999999999ap-3;                  // 1/5
  q = q * r + -0x1.0000000000000p-2;                 // -1/4
  q = q * r + 0x1.5555555555555p-2;                  // 1/3
  const double t3 = (r2 * r) * q;
  // ln x = (e-1) ln2 - ln c_j + (r - r^2/2) + t3, as hh + lo
  const double de = (double)(e - 1);
  double lo = kLogLo[j] + de * kLn2Lo;
  const double a = two_sum(de * kLn2Hi, kLogHi[j], lo);  // de * kLn2Hi is exact
  const double bh = r - 0.5 * r2;                    // Fast2Sum: |r| >= r^2/2
  lo = lo + (((r - bh) - 0.5 * r2) + (t3 - 0.5 * r2l));
  const double hh = two_sum(a, bh, lo);
  // z = y ln x
  const double zh = y * hh;
  const double zl = fma(y, hh, -zh) + y * lo;
  // z = k ln2/256 + s
  const double k = rint(zh * k256InvLn2);
  const int ki = (int)k;
  const int i = ki & 255;
  const int n = (ki - i) / 256;
  double sl = 0.0;
  const double sh = two_sum(fma(-k, kLn2_256Hi, zh), zl - k * kLn2_256Lo, sl);  // first exact
  // exp(s) - 1 = sh + [sh^2 (1/2 + sh/6 + ... + sh^4/720) + sl (1 + sh)]
  // (truncation sh^7/5040 < 2e-24; the polynomial's rounding is scaled by
  // sh^2 < 1.9e-6: products and sums)
  double u = 0x1.6c16c16c16c17p-10;                  // 1/720
  u = u * sh + 0x1.1111111111111p-7;                 // 1/120
  u = u * sh + 0x1.5555555555555p-5;                 // 1/24
  u = u * sh + 0x1.5555555555555p-3;                 // 1/6
  u = fma(u, sh, 0.5);                               // inline constant: one fma
  const double es = fma(sh * sh, u, fma(sl, sh, sl));
  // 2^(i/256) (1 + sh + es)
  const double th = kExpHi[i], tl = kExpLo[i];
  const double ph = th * sh;
  const double pl = fma(th, sh, -ph);
  const double s1 = th + ph;                         // Fast2Sum: th >= 1 > |ph|
  const double l1 = ((th - s1) + ph) + (pl + (tl + (th * es + tl * (sh + es))));
  const double res = ldexp(s1 + l1, n);
  if (ref) {
    // scaled by 2^n exactly while the result is a normal number; otherwise
    // (or for a non-positive / non-finite x) the reference is marked unusable
    const bool ok = fin && res >= 0x1p-1000 && res <= 0x1p+1000;
    ref->h = ok ? ldexp(s1, n) : 0.0;
    ref->l = ok ? ldexp(l1, n) : 0.0;
    ref->x = ok ? x : -1.0;
    ref->rx = ok ? rcp_approx(x) : 0.0;
  }
  return fin ? res : sp;
}

PMW_HD double pow_pos(double x, double y) { return pow_pos_impl(x, y, nullptr); }


// pow_pos(x, y) that also keeps the unrounded power for pow_pos_near.
PMW_HD double pow_pos_ref(double x, double y, PowRef& ref) {
  return pow_pos_impl(x, y, &ref);
}

// x^y continued from the reference power at a nearby argument x0 = ref.x:
// x^y = x0^y (1 + e)^y with e = (x - x0)/x0, |e| <= 2^-10. x - x0 is exact
// (Sterbenz), e is carried as eh + el (el from the exact fma residual), the
// binomial series (1 + e)^y - 1 = y e + c2 e^2 + ... + c7 e^7 (truncation
// below 1e-25) has its linear term in double-double, and the product with
// the reference's h + l is formed in double-double before the one rounding.
// The value before that rounding is within 6e-22 relative of x^y: the
// reference's own error plus ~1e-23 (host check against quadmath:
// tests/test_pow_host.py). About 45 instructions against pow_pos's ~130. Only for y = gamma (the
// series coefficients are gamma's).
// Returns the continuation's value before rounding, as s + lo
// (|lo| <~ ulp(s)). Requires x > 0 finite and |x - ref.x| <= 2^-10 ref.x.
PMW_HD void pow_pos_near_dd(double x, double y, const PowRef& ref, double& s, double& lo) {
  const double dx = x - ref.x;
  const double eh = dx * ref.rx;
  const double el = fma(-eh, ref.x, dx) * ref.rx;  // residual exact; (dx - eh x0) / x0
  // c_k = y (y-1) ... (y-k+1) / k!, k = 2..7, for y = gamma
  double q = -0x1.2cfc9a75b3dd8p-8;                 // c7
  q = q * eh + 0x1.ca0d127e7ec8ep-8;                // c6
  q = q * eh + -0x1.7dbd21dc9384dp-7;               // c5
  q = q * eh + 0x1.6f188e3a5d3e0p-6;                // c4
  q = q * eh + -0x1.caf32d76b8deap-5;               // c3
  q = q * eh + 0x1.1efa23f1c08bep-2;                // c2
  const double e2q = (eh * eh) * q;
  const double ph = y * eh;
  double tl = fma(y, eh, -ph) + y * el + e2q;
  const double th = ph + tl;                       // Fast2Sum: |ph| >> |tl|
  tl = tl - (th - ph);
  // (h + l)(1 + th + tl)
  const double mh = ref.h * th;
  const double ml = fma(ref.h, th, -mh) + (ref.h * tl + ref.l * th);
  s = ref.h + mh;                                  // Fast2Sum: |h| >> |mh|
  lo = ((ref.h - s) + mh) + (ml + ref.l);
}

// pow_pos(x, y) bit for bit, cheaper when x is near ref.x. Both pow_pos's
// and the continuation's values before their final rounding lie within
// 6e-22 relative of x^y (measured maxima 4.5e-22 and 5.5e-22 on the host
// against 113-bit quadmath, tests/test_pow_host.py). Where the
// continuation's value is farther than 2^-68 = 3.4e-21 relative (3x the sum
// of both bounds) from the midpoint between two doubles, both round to the
// same double; nearer a midpoint (about 4e-5 of arguments), at a power of
// two, or for arguments farther than 2^-10 from ref.x, pow_pos itself is
// evaluated. So the result never differs from pow_pos's.
// The continuation alone: returns true and sets r when its rounding is
// certain to equal pow_pos's (see pow_pos_near), false otherwise.
PMW_HD bool pow_pos_near_try(double x, double y, const PowRef& ref, double& r) {
  const double dx = x - ref.x;
  const bool close = x > 0.0 && x < __builtin_inf() && fabs(dx) <= 0x1p-10 * ref.x;
  double s, lo;
  pow_pos_near_dd(close ? x : ref.x, y, ref, s, lo);
  r = s + lo;
  const double d = (s - r) + lo;                   // value - r: |d| <= ulp(r)/2
  int e;
  const double m = frexp(r, &e);                   // r = m 2^e, m in [0.5, 1)
  const double hu = ldexp(1.0, e - 54);            // ulp(r) / 2
  return close && fabs(fabs(d) - hu) > r * 0x1p-68 && m != 0.5;
}

PMW_HD double pow_pos_near(double x, double y, const PowRef& ref) {
  double r;
  return pow_pos_near_try(x, y, ref, r) ? r : pow_pos(x, y);
}

// x^y to within a few 1e-15 relative (measured on the host for x in
// [1e-3, 1e5]) for positive finite x and 0 < y <= 1.5: the same reductions
// in plain double arithmetic, for a derivative that needs no last bit; about a
// third of pow_pos's instructions. Non-positive or non-finite x give NaN.
PMW_HD double pow_pos_fast(double x, double y) {
  using namespace powt;
  const bool fin = x > 0.0 && x < __builtin_inf();
  int e;
  const double m = 2.0 * frexp(fin ? x : 1.0, &e);  // table index always in range
  const unsigned j = (unsigned)(int)(m * 128.0 - 127.5) & 255u;
  const double r = fma(m, kLogC[j], -1.0);           // exact, |r| < 0.0059
  double q = -0x1.5555555555555p-3;                  // -1/6
  q = q * r + 0x1.999999999999ap-3;                  // 1/5
  q = q * r + -0x1.0000000000000p-2;                 // -1/4
  q = q * r + 0x1.5555555555555p-2;                  // 1/3
  q = fma(q, r, -0.5);                               // inline constant: one fma
  const double lnx = fma((double)(e - 1), 0x1.62e42fefa39efp-1, kLogHi[j]) + fma(r * r, q, r);
  const double z = y * lnx;
  const double k = rint(z * k64InvLn2);
  const int ki = (int)k;
  const int i = ki & 63;
  const double sh = fma(-k, kLn2_64Lo, fma(-k, kLn2_64Hi, z));
  double u = 0x1.6c16c16c16c17p-10;                  // 1/720
  u = u * sh + 0x1.1111111111111p-7;                 // 1/120
  u = u * sh + 0x1.5555555555555p-5;                 // 1/24
  u = u * sh + 0x1.5555555555555p-3;                 // 1/6
  u = fma(u, sh, 0.5);
  u = fma(u, sh, 1.0);
  const double res = ldexp(kExpHi[4 * i] * fma(u, sh, 1.0), (ki - i) / 64);  // 2^(i/64)
  return fin ? res : __builtin_nan("");
}

// a b + c for a constant c: one v_fma_f64 with c in scalar registers, where
// the compiler copies the constant into the accumulator and takes v_fmac (3
// VALU instructions).
PMW_HD double fma_c(double a, double b, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  double r;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
  return r;
#else
  return fma(a, b, c);
#endif
}

PMW_HD unsigned high_word(double x) {
  unsigned long long b;
  memcpy(&b, &x, 8);
  return (unsigned)(b >> 32);
}

// x's significand, as m in [1, 2) with x = 2^(e-1023) m for the biased
// exponent e (x positive and normal).
PMW_HD double significand(double x) {
  unsigned long long b;
  memcpy(&b, &x, 8);
  b = (b & 0x000fffffffffffffull) | 0x3ff0000000000000ull;
  double m;
  memcpy(&m, &b, 8);
  return m;
}

// x^gamma for gamma = kGamma's double (pmw_common.h), the exponent of the
// tables. x = 2^(e-1023) m; j = m's first 9 fraction bits; r = m c_j - 1,
// exact; x^gamma = (2^(e-1023) / c_j)^gamma (1 + r)^gamma. For 2^-6 <= x < 1024
// one 16-byte table entry holds c_j and the first factor as a double and a float;
// elsewhere the entry of the same significand there is scaled by a second,
// double-double factor. The linear term of the series is double-double; the
// quadratic and later terms (< 2^-19.8) are doubles, whose rounding sets the error
// of the value before the last rounding (2.7e-22 relative): one in 3e6 results is
// not the correctly rounded one. Powers that overflow give inf; other arguments as
// pow(x, gamma): +-0 -> 0, +-inf -> inf, negative and NaN -> NaN; subnormal
// arguments, whose power is below the smallest double, give 0.
//
// The range: rho*theta falls with height, over a constant-theta background from
// 350 at the ground to 65 at 15 km, 25 at 20 km, 0.8 at 28 km and 2^-6 at 30.2 km (at
// 30.7 km its pressure ends). A row touches the one or two entries near its value,
// so the rest of the 128 KB costs nothing. With four binades (64 <= x, 32 KB)
// every row above 15 km was computed twice; step of 2000 x 1000 in us, four / sixteen
// binades, column of 10 km 76.4 / 76.4, 20 km 132.8 / 76.1, 28 km 133.4 / 76.1;
// 800 x 400 23.4 / 23.4, 37.9 / 23.4, 38.2 / 23.4; 1003 x 517 with the inflow 32.7 /
// 32.8, 53.7 / 32.8, 54.2 / 32.8.
//
// The entry is a gather, and the flux kernels pay for its bytes. Three loads of
// 40 bytes a lane (c_j and double-doubles of c_j^-gamma and of every binade's
// factor) / this one of 16: a step of 2000 x 1000 84.5 / 82.7 us, of 8192 x
// 4096 1315 / 1277, of 1003 x 517 33.8 / 33.0. With uniform loads (a timing
// copy, wrong values) 2000 x 1000 takes 75.1.
//
// The x waves and the large z tiles take the value of the entry alone
// (PowGammaIn) and look at k once, after a wave's last face (x) or a stage's (z):
// a test and a branch in every face cost 4 to 5 % of a large launch (8192 x 4096
// x 523 / 497 us, z 769 / 738; 2000 x 1000 x 38.4 / 37.6, z 49.4 / 47.6).

// x^gamma = s + l for k < kGamEntries, else s + l times the binade's factor.
PMW_HD void pow_gamma_entry(double x, double& s, double& l, unsigned& k) {
  using namespace powt;
  k = (high_word(x) >> 11) - (1017u << 9);           // 2^-6 <= x < 1024: an index
  const GamQ t = kGamQ[k & (kGamEntries - 1u)];
  const double r = fma(significand(x), (double)t.c, -1.0);  // exact
  const double th = t.h, tl = t.l;
  // c_k = gamma (gamma-1) ... (gamma-k+1) / k!, k = 7..2; c_8 r^8 < 2^-80
  double q = fma_c(-0x1.2cfc9a75b3dd8p-8, r, 0x1.ca0d127e7ec8ep-8);
  q = fma_c(q, r, -0x1.7dbd21dc9384dp-7);
  q = fma_c(q, r, 0x1.6f188e3a5d3e0p-6);
  q = fma_c(q, r, -0x1.caf32d76b8deap-5);
  q = fma_c(q, r, 0x1.1efa23f1c08bep-2);
  // (1 + r)^gamma = 1 + ph + pl
  const double ph = 0x1.6678ae3cb2859p+0 * r;        // gamma
  const double pl = fma(r * r, q, fma(0x1.6678ae3cb2859p+0, r, -ph));
  // (th + tl)(1 + ph + pl) = s + l
  const double a = th * ph;
  s = th + a;                                        // Fast2Sum: th > |a|
  l = (((th - s) + a) + fma(th, ph, -a)) + fma(th, pl, fma(tl, ph, tl));
}

PMW_HD double pow_gamma(double x) {
  using namespace powt;
  double s, l;
  unsigned k;
  pow_gamma_entry(x, s, l, k);
  if (__builtin_expect(k >= kGamEntries, 0)) {
    // the last entry (NaN) serves powers past the largest, NaN and a set sign
    const unsigned e = ((high_word(x) >> 20) + 7u) >> 4;
    const double* te = kGamE + 2u * (e < kGamELast ? e : kGamELast);
    const double eh = te[0], el = te[1];
    const double h = s * eh;                         // (s + l)(eh + el)
    const double up = h + fma(l, eh, fma(s, el, fma(s, eh, -h)));
    const double res = e < 36u ? up * 0x1p-64 : e < 100u ? up : up * 0x1p64;  // as kGamE
    const double inf = __builtin_inf();
    if (res < inf) return res;
    return x == 0.0 ? 0.0 : (x > 0.0 || x == -inf) ? inf : __builtin_nan("");
  }
  return s + l;
}

// x^(gamma-1) to 4e-16 relative for positive normal x, by the same steps in
// plain double arithmetic: for the adjoint's dp/dq = gamma C0 q^(gamma-1),
// where a derivative needs no last bit. Other x give NaN. Two loads and no
// branch: with one entry per binade and the rare path in a branch the adjoint
// kernels, at their register limits, spill (16 of 400 x 200 112 -> 166 us).
PMW_HD double pow_gamma_minus_one(double x) {
  using namespace powt;
  const unsigned hi = high_word(x);
  const double* t = kGamM + 2u * ((hi >> 11) & 511u);
  const double d = t[0], c = t[1], e = kGamD[(hi >> 20) & 2047u];
  const double r = fma(significand(x), c, -1.0);  // exact, |r| <= 2^-9
  // c_k = a (a-1) ... (a-k+1) / k!, a = gamma - 1; c_6 r^6 < 2^-60
  double q = fma_c(0x1.eaabd5fa7fe8cp-6, r, -0x1.54c5337464d59p-5);
  q = fma_c(q, r, 0x1.0628bd48c9ba5p-4);
  q = fma_c(q, r, -0x1.eba2540426299p-4);
  q = fma_c(q, r, 0x1.99e2b8f2ca164p-2);
  const double pw = d * e;
  const bool normal = hi - 0x00100000u < 0x7fe00000u;
  return normal ? fma(pw, q * r, pw) : __builtin_nan("");
}

}  // namespace pmw
