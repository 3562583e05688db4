// vert_sources_chain.h -- the tridiagonal chains of the sources step
// (gitm_vert_sources.hip): divisions without range handling, the range tests
// that tell whether they were exact, and the sweeps of a solve (calc_conduction_1d,
// calc_conduction.f90:132-244), serial in altitude.  Also built for the host
// (GV_HOST_EMULATION).
#pragma once

#include "vert_column.h"

namespace gv {
namespace chain {

#ifdef GV_HOST_EMULATION
struct alignas(16) double2 {
  double x, y;
};
GV_FN double2 make_double2(double x, double y) { return {x, y}; }
// the hardware's reciprocal is good to about a float's precision
GV_FN double rcp_approx(double d) {
  return __builtin_bit_cast(double, __builtin_bit_cast(long long, 1.0 / d) & ~0x1fffffffLL);
}
#else
GV_FN double rcp_approx(double d) { return __builtin_amdgcn_rcp(d); }
#endif
GV_FN int high_word(double x) { return (int)(__builtin_bit_cast(long long, x) >> 32); }

// IEEE division without its range handling.  The hardware's sequence is:
// scale both operands, refine v_rcp_f64 twice, multiply, correct by the
// remainder, undo the scaling and fix special operands up.  The scalings are
// by powers of two, so where neither the operands nor the remainder leave the
// normal range the middle part alone gives the same bits: div_recip's refined
// reciprocal, which quotients by one divisor share, and a multiplication and
// correction.  div_pos is for divisors > 0 and div_neg for divisors < 0: they
// differ in the sign of a zero remainder, which makes the quotients of +0 and
// -0 right too.
GV_FN double div_recip(double d) {
  double r = rcp_approx(d);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
}
GV_FN double div_pos(double n, double d, double r) {
  const double q = n * r;
  return __builtin_fma(-__builtin_fma(d, q, -n), r, q);
}
GV_FN double div_neg(double n, double d, double r) {
  const double q = n * r;
  return __builtin_fma(__builtin_fma(-d, q, n), r, q);
}

// Whether the quick divisions may be used is decided by range.  Divisors
// known before the chains are positive and within 2^-200..2^200, numerators
// and the sub-diagonal zero or within 2^-200..2^200, the other matrix elements
// within 2^200; the pivots are negative and within 2^-240..2^240 (Pivots), each
// of the forward sweeps' values is zero or above 2^-600 (Values), and what
// comes out is finite.  Otherwise the column is done again with plain divisions.
// A zero value is a zero numerator's quotient, or the given one of level 0, and
// exact: a numerator d - dp a that is not zero is no less than 2^-800 (d = 0) or
// the last place of a d above 2^-401, so its quotient is no less than 2^-1040,
// which is not zero in the high word.
struct Range {
  double lo = 0x1p200, hi = 0.0;  // of the divisors, and of every magnitude
  bool tiny = false;
  GV_MEM void divisor(double x) {
    lo = fmin(lo, x);
    hi = fmax(hi, x);
  }
  GV_MEM void element(double x) { hi = fmax(hi, fabs(x)); }
  GV_MEM void numerator(double x) {
    element(x);
    tiny |= (x != 0.0) & (fabs(x) < 0x1p-200);
  }
  GV_MEM bool good() const { return (lo > 0x1p-200) & (hi < 0x1p200) & !tiny; }
};

// The ranges of a chain's pivots and values, from the high words of two
// levels at once (as integers negative doubles ascend with their magnitude;
// doubled as unsigned ones, less one, the words order by magnitude, but for zero,
// which comes last).
GV_FN int lesser(int a, int b) { return a < b ? a : b; }
GV_FN int greater(int a, int b) { return a > b ? a : b; }
struct Pivots {
  int lo = 0x7fffffff, hi = (int)0x80000000;
  GV_MEM void see(double x, double y) {
    lo = lesser(lesser(high_word(x), high_word(y)), lo);
    hi = greater(greater(high_word(x), high_word(y)), hi);
  }
  GV_MEM bool good() const { return lo >= high_word(-0x1p-240) && hi < high_word(-0x1p240); }
};
struct Values {
  unsigned lo = ~0u;
  // (on the device in the three instructions that it takes: the compiler makes
  // seven of it, in loops that issue one every 4 to 5 clocks)
  static GV_MEM unsigned order(double x) {
#ifdef GV_HOST_EMULATION
    return 2u * (unsigned)high_word(x) - 1u;
#else
    unsigned r;
    asm("v_lshl_add_u32 %0, %1, 1, -1" : "=v"(r) : "v"(high_word(x)));
    return r;
#endif
  }
  GV_MEM void see(double x, double y) {
    const unsigned u = order(x), v = order(y);
#ifdef GV_HOST_EMULATION
    lo = u < lo ? u : lo;
    lo = v < lo ? v : lo;
#else
    asm("v_min3_u32 %0, %0, %1, %2" : "+v"(lo) : "v"(u), "v"(v));
#endif
  }
  GV_MEM bool good() const { return lo >= 2u * (unsigned)high_word(0x1p-600) - 1u; }
};

// Two levels of a row from level i on, i odd: 16-byte aligned.
GV_FN double2 load2(const double *row, int i) {
  return *reinterpret_cast<const double2 *>(row + i);
}
GV_FN void store2(double *row, int i, double2 v) {
  *reinterpret_cast<double2 *>(row + i) = v;
}

// The chains take two levels at a time.  A lone wavefront issues one
// instruction of whatever kind every 4 to 5 clocks and an LDS read takes some
// 60, so the loops hold nothing but arithmetic, 16-byte LDS accesses and an
// address per row: a ring of P pairs holds operands on their way, a pair's
// slot is read anew as soon as its levels are done, U rounds of the ring are
// unrolled, and what is read past the last pair (within the LDS image, PAD
// doubles beyond its last row) is not used.  step(slot, i) works on levels i
// and i + 1 and read(slot, i) starts its reads; n pairs from level i0 on in
// steps of d levels.
template <int P, int U, class Slot, class Read, class Step>
GV_FN void ring(int n, int i0, int d, const Read &read, const Step &step) {
  Slot x[P];
#pragma unroll
  for (int p = 0; p < P; p++) read(x[p], i0 + p * d);
  int i = i0;
  for (; n >= P * U; n -= P * U, i += P * U * d) {
#pragma unroll
    for (int p = 0; p < P * U; p++) {
      step(x[p % P], i + p * d);
      GV_ORDER();
      read(x[p % P], i + (p + P) * d);
      GV_ORDER();
    }
  }
#pragma unroll
  for (int p = 0; p < P * U - 1; p++)
    if (p < n) {
      step(x[p % P], i + p * d);
      if (p + P < P * U - 1) read(x[p % P], i + (p + P) * d);
    }
}
constexpr int PAD = 16;  // ring reads at most P pairs past the last level

// The forward sweep of one solve (:232-241): cp to rb, dp to wd.  sc d is the
// solve's right side (sc is 1 or 2: the fma rounds once).
struct Fwd {
  double2 a, c, b, d;
};
// cp at one level, and dp at the level below, whose pivot is known by then:
// dp's five operations go between those of the pivot's reciprocal, each of
// which waits 6 to 22 clocks for the one before (88 a level).
struct Forward {
  double sc, cp, dp;
  double a, d, den, r;  // the level below's
  GV_MEM void level(double a1, double c1, double b1, double d1) {
    const double t = cp * a1;
    GV_ORDER();
    const double den1 = b1 - t;
    const double u = dp * a;
    GV_ORDER();
    const double r0 = rcp_approx(den1);
    const double n = __builtin_fma(d, sc, -u);
    GV_ORDER();
    const double q = n * r;
    const double e0 = __builtin_fma(-den1, r0, 1.0);
    GV_ORDER();
    const double m = __builtin_fma(-den, q, n);
    const double r1 = __builtin_fma(e0, r0, r0);
    GV_ORDER();
    dp = __builtin_fma(m, r, q);
    const double e1 = __builtin_fma(-den1, r1, 1.0);
    GV_ORDER();
    const double r2 = __builtin_fma(e1, r1, r1);
    const double qc = c1 * r2;
    const double mc = __builtin_fma(-den1, qc, c1);
    cp = __builtin_fma(mc, r2, qc);
    a = a1;
    d = d1;
    den = den1;
    r = r2;
  }
  GV_MEM double last() {
    const double n = __builtin_fma(d, sc, -(dp * a));
    return dp = div_neg(n, den, r);
  }
};
template <bool FAST>
GV_FN bool sweep(const double *ra, const double *rc, double *rb,
                                      const double *rd, double *wd, double sc, int nA, double &cp,
                                      double &dp) {
  const auto plain = [&](double a, double c, double b, double d) {
    const double den = b - cp * a;
    const double n = __builtin_fma(d, sc, -(dp * a));
    cp = c / den;
    dp = n / den;
    return den;
  };
  if (!FAST) {
    for (int i = 1; i <= nA; i++) {
      plain(ra[i], rc[i], rb[i], rd[i]);
      rb[i] = cp;
      wd[i] = dp;
    }
    return true;
  }
  Pivots pivots;
  Values values;
  // the odd level out, if there is one, is read before the ring runs
  const double a1 = ra[nA], c1 = rc[nA], b1 = rb[nA], d1 = rd[nA];
  // the level below level 1 gives dp = dp(0)
  Forward f{sc, cp, 0.0, 0.0, -dp / sc, -1.0, -1.0};
  double v0 = dp;
  ring<2, 4, Fwd>(
      nA / 2, 1, 2,
      [&](Fwd &x, int i) {
        x.b = load2(rb, i);
        x.a = load2(ra, i);
        x.c = load2(rc, i);
        x.d = load2(rd, i);
      },
      [&](Fwd &x, int i) {
        double2 c;
        f.level(x.a.x, x.c.x, x.b.x, x.d.x);
        const double p0 = f.den;
        c.x = f.cp;
        const double v1 = f.dp;
        f.level(x.a.y, x.c.y, x.b.y, x.d.y);
        c.y = f.cp;
        store2(rb, i, c);
        store2(wd, i - 2, make_double2(v0, v1));
        pivots.see(p0, f.den);
        values.see(v0, v1);
        v0 = f.dp;
      });
  const int top = nA & ~1;
  cp = f.cp;
  dp = f.last();
  values.see(v0, dp);
  store2(wd, top - 1, make_double2(v0, dp));
  if (nA & 1) {
    const double p = plain(a1, c1, b1, d1);
    pivots.see(p, p);
    values.see(dp, dp);
    rb[nA] = cp;
    wd[nA] = dp;
  }
  return pivots.good() && values.good();
}

// The forward sweep on known pivots: dp over the right side in rn.
struct Fwd2 {
  double2 a, n, den, r;
};
template <bool FAST>
GV_FN bool sweep2(const double *ra, double *rn, const double *rden,
                                       const double *rr, int nA, double &dp) {
  if (!FAST) {
    for (int i = 1; i <= nA; i++) rn[i] = dp = (rn[i] - dp * ra[i]) / rden[i];
    return true;
  }
  Values values;
  const double a1 = ra[nA], n1 = rn[nA], den1 = rden[nA];
  ring<3, 2, Fwd2>(
      nA / 2, 1, 2,
      [&](Fwd2 &x, int i) {
        x.a = load2(ra, i);
        x.n = load2(rn, i);
        x.r = load2(rr, i);
        x.den = load2(rden, i);
      },
      [&](Fwd2 &x, int i) {
        double2 v;
        v.x = dp = div_neg(x.n.x - dp * x.a.x, x.den.x, x.r.x);
        v.y = dp = div_neg(x.n.y - dp * x.a.y, x.den.y, x.r.y);
        values.see(v.x, v.y);
        store2(rn, i, v);
      });
  if (nA & 1) {
    rn[nA] = dp = (n1 - dp * a1) / den1;
    values.see(dp, dp);
  }
  return values.good();
}

// The back substitution (:243-247), levels nA..0: the solution over dp in
// rd; t the value at nA + 1.
struct Back {
  double2 cp, dp;
};
template <bool FAST>
GV_FN void back(const double *rc, double *rd, int nA, double t) {
  if (!FAST) {
    for (int i = nA; i >= 0; i--) rd[i] = t = rd[i] - rc[i] * t;
    return;
  }
  const double c0 = rc[0], d0 = rd[0], c1 = rc[nA], d1 = rd[nA];
  if (nA & 1) rd[nA] = t = d1 - c1 * t;
  const int n = nA / 2;
  ring<4, 2, Back>(
      n, 2 * n - 1, -2,
      [&](Back &x, int i) {
        x.cp = load2(rc, i);
        x.dp = load2(rd, i);
      },
      [&](Back &x, int i) {
        double2 v;
        v.y = t = x.dp.y - x.cp.y * t;
        v.x = t = x.dp.x - x.cp.x * t;
        store2(rd, i, v);
      });
  rd[0] = d0 - c0 * t;
}

}  // namespace chain
}  // namespace gv
