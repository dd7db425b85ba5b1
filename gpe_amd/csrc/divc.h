// divc.h -- division of an FP64 field by a constant that the host knows, as
// the reference build rounds it, without a division in the kernel.
#pragma once
#include <cmath>
#include <cstdint>

#ifdef __HIPCC__
#define GPE_DIVC_HD __host__ __device__ __forceinline__
#else
#define GPE_DIVC_HD inline
#endif

namespace gpe {

// Division by a real constant s as the reference build evaluates it: the
// divisor is promoted to complex and divided by compiler-rt's logb-scaled
// quotient, i.e. ((a*c + b*0)/d, (b*c - a*0)/d) * 2^-e with c = s*2^-e,
// d = c*c + 0*0, e = logb(s).  d is known ahead, so t/d needs no division:
// with zh a neighbour of 1/d and zl the rest, fma(t, zh, t*zl) is t/d rounded
// to nearest (N. Brisebarre, J.-M. Muller, S. K. Raina, "Accelerating
// correctly rounded floating-point division when the divisor is known in
// advance", IEEE Trans. Computers 53, 2004), but for some d and zl on a few
// numerators whose quotient lies next to the middle of two doubles.
// make_divc enumerates those and takes a zh, zl for which every one rounds
// as it should; 0.08% of random divisors have none, and their quotients
// differ in the last bit on a handful of the 2^53 numerators.
// zh and zl carry the factor 2^-e, so the final * 2^-e costs nothing.
// Numerators may be as large as for the division itself; the smallest are
// 2^-900 for divisors from 2^-1022 to 2^100 (below, t*zl loses bits).  An
// infinite numerator gives an infinity, but NaN where zl < 0 (3% of random
// divisors: no zl >= 0 rounds every quotient).
struct DivC {
  double cs, zh, zl;
};

// t/d in the scaled form above: 2 operations where the general FP64 division
// issues 11 and takes about 70 cycles per wave (measured on an MI355X, 5
// cycles for a multiplication or an FMA).
GPE_DIVC_HD double div_const(double t, const DivC &d) { return std::fma(t, d.zh, t * d.zl); }

// Whether fma(t, zh, t*zl) is t/d rounded to nearest for every double t, d in
// [1, 4).  Its error before the last rounding is below 2^-51 ulp, so it can
// only differ for a t whose quotient is that close to the midpoint of two
// doubles: with t = T and d = B as 53-bit integers and X = 2Q+1 twice the
// midpoint, 2^(m+1) T - B X = N for m = 52 or 53 and a small N != 0.  For each
// N, X = -N/B modulo a power of two; every such T is tried.
inline bool division_exact(double d, double zh, double zl) {
  int eb = 0;
  const uint64_t B = (uint64_t)std::ldexp(std::frexp(d, &eb), 53);
  const double b = std::ldexp((double)B, -52), s = std::ldexp(1.0, eb - 1);  // d = b*s, b in [1, 2)
  const double h = zh * s, l = zl * s;                                        // of 1/b
  const int z = __builtin_ctzll(B);
  if (z > 4) return true;  // N is a multiple of 2^z
  const uint64_t odd = B >> z;
  uint64_t inv = odd;  // Newton: odd*inv = 1 mod 2^64
  for (int i = 0; i < 6; ++i) inv *= 2 - odd * inv;
  for (int N = -16; N <= 16; ++N) {
    if (N == 0 || (N & ((1 << z) - 1)) != 0) continue;
    for (int m = 52; m <= 53; ++m) {
      const uint64_t period = (uint64_t)1 << (m + 1 - z);
      for (uint64_t X = ((uint64_t)(-(int64_t)(N >> z)) * inv) & (period - 1); X < ((uint64_t)1 << 54); X += period) {
        if (X < ((uint64_t)1 << 53) || !(X & 1)) continue;
        const __int128 v = (__int128)B * X + N;
        const uint64_t T = (uint64_t)(v >> (m + 1));
        if (((__int128)T << (m + 1)) != v || T < ((uint64_t)1 << 52) || T >= ((uint64_t)1 << 53)) continue;
        const double t = std::ldexp((double)T, -52);
        if (std::fma(t, h, t * l) != t / b) return false;
      }
    }
  }
  return true;
}

// The constants of a divisor s.
inline DivC make_divc(double s) {
  DivC d{};
  if (s == 0.0 || !std::isfinite(s)) {  // (0/0, Inf/Inf, NaN: every quotient is NaN)
    d.cs = d.zh = d.zl = NAN;
    return d;
  }
  const int e = std::ilogb(s);
  const double c = std::ldexp(s, -e);
  const double den = c * c + 0.0 * 0.0;
  const double near = 1.0 / den, below = std::nextafter(near, 0.0), r = std::fma(-den, near, 1.0);
  // zh below 1/d first: with zl >= 0 a zero numerator keeps its sign
  const double high[2] = {r < 0.0 ? below : near, near};
  double zh = near, zl = r / den;
  bool found = false;
  for (int q = 0; q < 2 && !found; ++q) {
    const double l = std::fma(-den, high[q], 1.0) / den;
    const double low[3] = {l, std::nextafter(l, 1.0), std::nextafter(l, -1.0)};
    for (int i = 0; i < 3 && !found; ++i) {
      if (!division_exact(den, high[q], low[i]) || (q == 0 && low[i] < 0.0)) continue;
      zh = high[q];
      zl = low[i];
      found = true;
    }
  }
  if (zl == 0.0) zl = 0x1p-200;  // d = 1: too small to count, but an infinity times it is one
  d.cs = c;
  d.zh = std::ldexp(zh, -e);
  d.zl = std::ldexp(zl, -e);
  return d;
}

}  // namespace gpe
