// harm_chain.h -- a serial sum s = (((s + t0) + t1) + ...) in parallel, to the bit.
//
// While a running sum stays inside one binade, (2^e, 2^(e+1)), it is a multiple
// of u = 2^(e-52) and each addition rounds s + t to the nearest multiple, ties
// to the even one.  The change that a run of terms makes to s then depends on s
// only through its parity (s/u mod 2): moving s by an even number of u moves
// the exact sum, its nearest multiples and their parities with it.  So a run's
// effect is found without knowing s, by adding its terms to C = 1.5 2^e (even)
// and to C + u (odd): two changes, two parities after, and how far down and up
// the sums went.  Such maps compose associatively (a scan over lanes), and a
// run's map holds for the actual s if neither the sums from C nor those from s
// leave the binade.  Where one does not hold, that run's terms are added one
// by one.  Negative s: the same with all signs turned.
#pragma once
#include <string.h>
#include "harm_device.h"

namespace harm {

HARM_HD unsigned long long chain_bits(double x) {
#ifdef __HIP_DEVICE_COMPILE__
  return (unsigned long long)__double_as_longlong(x);
#else
  unsigned long long b;
  memcpy(&b, &x, 8);
  return b;
#endif
}
HARM_HD double chain_double(unsigned long long b) {
#ifdef __HIP_DEVICE_COMPILE__
  return __longlong_as_double((long long)b);
#else
  double x;
  memcpy(&x, &b, 8);
  return x;
#endif
}

struct ChainScale {
  int e;  // biased exponent and sign of s; -1: no binade to work in (zero, tiny, huge, not finite)
  double C, u, lo, hi;
  HARM_HD explicit ChainScale(double s) {
    const unsigned long long b = chain_bits(s);
    const unsigned x = (unsigned)(b >> 52) & 0x7ffu;
    e = (x < 64 || x > 2040) ? -1 : (int)(b >> 52);
    C = chain_double(((unsigned long long)x << 52) | (1ull << 51));
    u = chain_double((unsigned long long)(x - 52) << 52);
    lo = chain_double((unsigned long long)x << 52);
    hi = chain_double((unsigned long long)(x + 1) << 52);
  }
  HARM_HD double turned(double t) const { return chain_double(chain_bits(t) ^ ((unsigned long long)(e >> 11 & 1) << 63)); }
};

// a run's map: the change of an even and of an odd sum, bit 0/1 of q the parity
// after each, and the least and largest sums from C
struct ChainMap {
  double d0, d1, mn, mx;
  int q;
};
template <int N>
HARM_HD ChainMap chain_map(const ChainScale& c, const double (&t)[N]) {
  double x0 = c.C, x1 = c.C + c.u, mn = c.C, mx = c.C;
#pragma unroll
  for (int k = 0; k < N; k++) {
    const double v = c.turned(t[k]);
    x0 += v;
    x1 += v;
    mn = (x0 > mn) ? mn : x0;  // a NaN stays
    mx = (x1 < mx) ? mx : x1;
  }
  ChainMap m;
  m.d0 = x0 - c.C;
  m.d1 = x1 - (c.C + c.u);
  m.q = (int)(chain_bits(x0) & 1) | (int)(chain_bits(x1) & 1) << 1;
  m.mn = mn;
  m.mx = mx;
  return m;
}
// a, then b (the range is each run's own)
HARM_HD void chain_then(double a0, double a1, int aq, double& b0, double& b1, int& bq) {
  const double n0 = a0 + ((aq & 1) ? b1 : b0), n1 = a1 + ((aq & 2) ? b1 : b0);
  bq = (bq >> (aq & 1) & 1) | (bq >> (aq >> 1 & 1) & 1) << 1;
  b0 = n0;
  b1 = n1;
}
// the map holds for the sum s (its size, |s|) before the run
HARM_HD bool chain_holds(const ChainScale& c, double s, double mn, double mx) {
  const double down = s + (mn - c.C) - 2.0 * c.u, up = s + (mx - c.C) + 2.0 * c.u;
  return mn > c.lo && mx < c.hi && down > c.lo && up < c.hi;
}

}  // namespace harm
