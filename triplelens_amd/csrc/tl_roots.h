// Root solver of the image polynomial on the GPU: Laguerre's iteration of the
// reference (laguerre.cc:18-198) with the same bits in every root, at a
// fraction of the instructions the operation-by-operation restatement in
// tl_math.h takes.
//
// What the reference's iteration computes falls in two kinds:
//   * values that enter x (the Horner sums, the quotients f/b and 2s/b, the
//     square root, the step m/g): these are computed with the reference's
//     rounding, operation for operation;
//   * values that are only compared (the error bound of |p(x)|, which of
//     g + sq and g - sq is larger, the product check of the roots, the image
//     test's residual): these are bracketed by cheap bounds, and the
//     reference's own expressions are evaluated only where a comparison falls
//     inside the bracket.
// The moduli of the second kind (14 correctly rounded hypots per iteration)
// were most of the chain's instructions.
//
// Quotients and square roots of operands in a safe range are taken without
// the pre-scaling and special-value fix-up of the IEEE sequences, and a
// square root hands its reciprocal on to the divisions by it (modulus
// correction, csqrt).  Operands outside the range or just below a power of two,
// signed zeros and everything else unusual go through the general iteration.
#pragma once

#include "tl_math.h"

namespace tl {

// Smaller and larger magnitude, one instruction each (fmin and fmax of the
// language quiet signalling NaNs first; a NaN operand here gives the other one
// or a NaN, and every caller compares the result so that a NaN in any of its
// operands is seen by another comparison).
__device__ __forceinline__ double min_abs(double a, double b) {
  double r;
  asm("v_min_f64 %0, |%1|, |%2|" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double max_abs(double a, double b) {
  double r;
  asm("v_max_f64 %0, |%1|, |%2|" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// Keeps both sides of a select computed (the compiler would otherwise branch
// around the shorter one: a taken branch costs one wavefront about 50 cycles).
__device__ __forceinline__ void keep(double& a) { asm volatile("" : "+v"(a)); }

// ---- in-range arithmetic ---------------------------------------------------
// The forms below round as the IEEE operations do, except for a few operands
// that all lie just below a power of two (see quot_near and sqrt_near).  So an
// iteration with an operand whose mantissa bits 32 to 47 are all ones (one
// iteration in 10^4) is left to the general form: edge(a) holds these bits,
// and the largest of several operands' is kEdge where one of them has them.
// (Three maxima of 16-bit halves and a sign in lag_step: a 200-point chain
// takes 3.95 ms instead of 3.91 without the check; with the compiler's packed
// maxima and a comparison of its own 4.06, with a shift per operand and both
// sides of a power of two 4.12.)
constexpr unsigned kEdge = 0xFFFF;
__device__ __forceinline__ unsigned edge_bits(double a) { return (unsigned)__double2hiint(a); }
__device__ __forceinline__ unsigned edge(double a) { return edge_bits(a) & 0xFFFFu; }
// (the lower halves' maximum, its upper half not defined)
__device__ __forceinline__ unsigned edge_max(unsigned a, unsigned b, unsigned c) {
  unsigned r;
  asm("v_max3_u16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// Reciprocal of b for 2^-900 <= |b| <= 2^900: the hardware estimate r0
// (e = 1 - b r0, |e| below 2^-22) and one third-order correction
// r0 (1 + e + e^2), within 2^-66 of 1/b before the last rounding.
__device__ __forceinline__ double rcp_near(double b) {
  const double r0 = __builtin_amdgcn_rcp(b);
  const double e = fma(-b, r0, 1.0);
  const double p = fma(e, e, e);
  return fma(r0, p, r0);
}
// a / b rounded to nearest from r = rcp_near(b), one correction by the exact
// residual, for operands and quotients within 2^-900 .. 2^900.  With r the
// nearest double to 1/b the result is rounded to nearest (Markstein).  For
// b = 2 - k 2^-52, k odd, 1/b lies k^2 2^-107 above a midpoint: where the
// estimate does not resolve that (k below 2^20), r is the double below, and
// for k >= 3 the quotients next to a midpoint may come out one unit off.
// These b have edge(b) == kEdge.
__device__ __forceinline__ double quot_near(double a, double b, double r) {
  const double q = a * r;
  return fma(fma(-b, q, a), r, q);
}
// s = sqrt(a) rounded to nearest and h close to 1 / (2 s), for
// 2^-600 <= a <= 2^600: the hardware reciprocal root y, s0 = a y, h0 = y/2 with
// h0 s0 = 1/2 - e, one third-order step (1 - 2e)^-1/2 = 1 + e + 3/2 e^2, and the
// exact residual.  The value before the last rounding is good to 3.4 2^-106 of
// the root: enough for all mantissas but the dozen whose roots lie closer to a
// midpoint.  Of those (enumerated: A 2^s = M^2 - j, |j| <= 27) the only one
// that comes out as the neighbouring double is 4 - 2^-51, edge(a) == kEdge.
__device__ __forceinline__ void sqrt_near(double a, double& s, double& h) {
  const double y = __builtin_amdgcn_rsq(a);
  const double s0 = a * y, h0 = 0.5 * y;
  const double e = fma(-h0, s0, 0.5);
  const double p = e * fma(1.5, e, 1.0);
  const double s1 = fma(s0, p, s0);
  h = fma(h0, p, h0);
  s = fma(fma(-s1, s1, a), h, s1);
}
// hyp_sel for 2^-240 <= ay <= ax <= 2^240 and ay > ax 2^-54, if the root's
// operand n (set here) has edge(n) != kEdge.  (1/w and, in
// csqrt_near, 1/q come from a root's reciprocal by a second-order step, good
// to 2^-103: of the b of quot_near only k = 1 is left, which is harmless.)
__device__ __forceinline__ double hyp_near(double ax, double ay, double& n) {
  double h, hi;
  n = ax * ax + ay * ay;
  sqrt_near(n, h, hi);
  const double w = 2.0 * h;
  const double r = fma(hi, fma(-w, hi, 1.0), hi);  // 1 / w
  const double d1 = h - ay;
  double ta = ax * (2.0 * d1 - ax) + (d1 - 2.0 * (ax - ay)) * d1;
  const double d2 = h - ax;
  double tb = 2.0 * d2 * (ax - 2.0 * ay) + ((4.0 * d2 - ay) * ay + d2 * d2);
  keep(ta);
  keep(tb);
  return h - quot_near(h <= 2.0 * ay ? ta : tb, w, r);
}
__device__ __forceinline__ bool hyp_in_range(double ax, double ay) {
  return (int(ay >= 0x1p-240) & int(ax <= 0x1p+240) & int(ay > ax * 0x1p-54)) != 0;
}
// csqrt_sel for re, im with hyp_in_range(max, min) of their magnitudes, if the
// operands n1, n2 of its roots have an edge other than kEdge.
__device__ __forceinline__ cx csqrt_near(double re, double im, double& n1, double& n2) {
  const double fr = fabs(re);
  const double d = hyp_near(max_abs(re, im), min_abs(re, im), n1);
  double q, h;
  n2 = 0.5 * (d + fr);
  sqrt_near(n2, q, h);
  h = 2.0 * h;
  const double w = 0.5 * quot_near(im, q, fma(h, fma(-q, h, 1.0), h));
  const bool pos = re > 0.0;
  return mk(pos ? q : fabs(w), copysign(pos ? w : q, im));
}

constexpr double kTinyOp = 0x1p-300, kHugeOp = 0x1p+300;

// ---- Laguerre --------------------------------------------------------------
// Horner sums of p at x: b[0] = p(x), and b[j + 1] is coefficient j of the
// polynomial deflated by x (laguerre.cc:133-139).
template <int M>
__device__ __forceinline__ void horner_sums(const cx (&p)[M + 1], cx x, cx (&b)[M + 1]) {
  b[M] = p[M];
#pragma unroll
  for (int j = M - 1; j >= 0; j--) b[j] = cadd(cmul(x, b[j + 1]), p[j]);
}

// The step dx from x with Laguerre's fractional kick (laguerre.cc:22) of
// iteration i, a multiple of kLagMT; the table is read modulo 8.
__device__ __forceinline__ cx lag_kick(cx x, cx dx, int i) {
  const int k = (i / kLagMT) & 7;
  const double frac = k == 0 ? 0.5 : k == 1 ? 0.23 : k == 2 ? 0.73 : k == 3 ? 0.13
                    : k == 4 ? 0.37 : k == 5 ? 0.61 : k == 6 ? 0.89 : 1.0;
  return csub(x, cmul(mk(frac, 0.0), dx));
}

// The reference's iteration i at x, every value as laguerre.cc computes it;
// b holds the Horner sums at x.  Returns true when x is accepted (and left
// unchanged), else x is the next point.
template <int M>
__device__ __forceinline__ bool lag_general(const cx (&b)[M + 1], cx& x, int i,
                                            const TrigTable* trig, bool& oob) {
  cx f = mk(0.0, 0.0), s = mk(0.0, 0.0);
#pragma unroll
  for (int j = M - 1; j >= 0; j--) {
    s = cadd(cmul(x, s), f);
    f = cadd(cmul(x, f), b[j + 1]);
  }
  const double md = (double)M;
  double err = cabs_(b[M]);
  const double ax = cabs_(x);
  double ab = err;
#pragma unroll
  for (int j = M - 1; j >= 0; j--) {
    ab = cabs_(b[j]);
    err = ab + ax * err;
  }
  if (ab <= err * kLagEps) return true;
  const cx g = cdiv_sel(f, b[0]);
  const cx h = csub(cmul(g, g), cdiv_sel(cscale(s, 2.0), b[0]));
  const cx rad = cscale(csub(cscale(h, md), cmul(g, g)), md - 1.0);
  const cx sq = csqrt_(rad);
  cx gp = cadd(g, sq);
  const cx gm = csub(g, sq);
  double agp = cabs_(gp);
  const double agm = cabs_(gm);
  if (agp < agm) {
    gp = gm;
    agp = agm;
  }
  cx dx;
  if (agp > 0.0) dx = cdiv_rc_sel(md, gp);
  else dx = cscale(mk(trig->c[i], trig->s[i]), 1.0 + ax);
  const cx x1 = csub(x, dx);
  if (x.re == x1.re && x.im == x1.im) return true;
  if (i % kLagMT) {
    x = x1;
  } else {
    oob |= i / kLagMT >= 8;
    x = lag_kick(x, dx, i);
  }
  return false;
}

// A polynomial whose constant term is NaN in both parts (a source position
// that is not finite) has NaN sums at every x: no comparison accepts x, and
// lag_general's step is that of a vanishing denominator.  The iterations from i
// to the last, with its results (the fresh solves of one such position took
// 26.7 ms by lag_general, and take 9.8).  The chains and the critical curves go
// on by lag_general: this branch in their code cost every one of them 2%.
__device__ __forceinline__ bool lag_is_lost(cx p0) {
  return p0.re != p0.re && p0.im != p0.im;
}
__device__ inline bool lag_lost(cx& x, int i, const TrigTable* trig, bool& oob) {
  for (; i <= kLagMaxIt; i++) {
    const cx dx = cscale(mk(trig->c[i], trig->s[i]), 1.0 + cabs_(x));
    const cx x1 = csub(x, dx);
    if (x.re == x1.re && x.im == x1.im) return true;
    if (i % kLagMT) {
      x = x1;
    } else {
      oob |= i / kLagMT >= 8;
      x = lag_kick(x, dx, i);
    }
  }
  return false;
}

// One iteration of Laguerre::laguerre at x, in the parts that its two drivers
// below share.
//
// An iteration first runs the b recurrence alone (lag_eval): the one that
// accepts x (one in two to three) needs no derivative.  The error bound
// sum |b_j| |x|^j is bracketed by its 1-norm form E1: E1 / sqrt 2 <= E <= E1
// (|x| from the hardware root, good to 1e-7; the bracket is widened by 1e-5).
// One evaluation in a hundred falls inside it and gets moduli from the
// hardware root, which leave a bracket of 1e-4 (lag_narrow).
struct LagEval {
  double ax;      // |x|, or NaN (which leaves every comparison undecided) where
                  // its square may have lost digits
  double nb, e2;  // |p(x)|^2 and the square of the bound on which x is accepted
};
template <int M>
__device__ __forceinline__ LagEval lag_eval(const cx (&p)[M + 1], cx x, cx (&b)[M + 1]) {
  LagEval v;
  const double n = cnorm(x);
  v.ax = n > 1e-280 ? __builtin_amdgcn_sqrt(n) : __builtin_nan("");
  b[M] = p[M];
  double e1 = fabs(p[M].re) + fabs(p[M].im);
#pragma unroll
  for (int j = M - 1; j >= 0; j--) {
    b[j] = cadd(cmul(x, b[j + 1]), p[j]);
    e1 = fma(v.ax, e1, fabs(b[j].re) + fabs(b[j].im));
  }
  v.nb = cnorm(b[0]);
  const double el = kLagEps * e1;
  v.e2 = el * el;
  return v;
}
// not accepted (nb above 1e-250 follows from lag_step's lower bound)
__device__ __forceinline__ bool lag_far(const LagEval& v) { return v.nb > v.e2 * 1.0001; }
__device__ __forceinline__ bool lag_near(const LagEval& v) {
  return (int(v.nb < v.e2 * 0.49999) & int(v.e2 > 1e-250)) != 0;
}
// inside the bracket: the sum with moduli from the hardware root
template <int M>
__device__ __forceinline__ void lag_narrow(const LagEval& v, const cx (&b)[M + 1], bool& far,
                                           bool& near) {
  double e = __builtin_amdgcn_sqrt(cnorm(b[M]));
#pragma unroll
  for (int j = M - 1; j >= 0; j--) e = fma(v.ax, e, __builtin_amdgcn_sqrt(cnorm(b[j])));
  const double eh = kLagEps * e;
  near = (int(v.nb < eh * eh * 0.9999) & int(eh * eh > 1e-250)) != 0;
  far = v.nb > eh * eh * 1.0001;
}

// The step from x: the next point x1 and x - x1 = step.  Returns whether
// everything is in range, every comparison decided and x1 another point; else
// the iteration is lag_general's.
template <int M>
__device__ __forceinline__ bool lag_step(const cx (&b)[M + 1], cx x, cx& x1, cx& step) {
  constexpr double md = (double)M;
  // the recurrences' first two steps, from s = f = 0, leave s = b[M] and
  // f = x b[M] + b[M - 1] (up to the sign of a zero, which the range check
  // below sends to lag_general wherever it could matter)
  cx s = b[M], f = cadd(cmul(x, b[M]), b[M - 1]);
#pragma unroll
  for (int j = M - 3; j >= 0; j--) {
    s = cadd(cmul(x, s), f);
    f = cadd(cmul(x, f), b[j + 1]);
  }
  // g = f / b and 2 s / b by Smith's quotient over one denominator
  const cx B = b[0];
  const bool ce = fabs(B.re) < fabs(B.im);
  const double num = ce ? B.re : B.im, den = ce ? B.im : B.re;
  const double ratio = quot_near(num, den, rcp_near(den));
  const double denom = (num * ratio) + den;
  const double rd = rcp_near(denom);
  const cx s2 = cscale(s, 2.0);
  const double far_ = f.re * ratio, fbr = f.im * ratio;
  const double sar = s2.re * ratio, sbr = s2.im * ratio;
  const double xf = ce ? far_ + f.im : fbr + f.re, yf = ce ? fbr - f.re : f.im - far_;
  const double xs = ce ? sar + s2.im : sbr + s2.re, ys = ce ? sbr - s2.re : s2.im - sar;
  const cx g = mk(quot_near(xf, denom, rd), quot_near(yf, denom, rd));
  const cx g2 = cmul(g, g);
  const cx h = csub(g2, mk(quot_near(xs, denom, rd), quot_near(ys, denom, rd)));
  const cx rad = cscale(csub(cscale(h, md), g2), md - 1.0);
  double n1, n2;
  const cx sq = csqrt_near(rad.re, rad.im, n1, n2);
  unsigned em = edge_max(edge_bits(den), edge_bits(denom), edge_bits(n1));
  const cx gp = cadd(g, sq), gm = csub(g, sq);
  const double np = cnorm(gp), nm = cnorm(gm);
  const bool minus = np < nm;
  const cx d = mk(minus ? gm.re : gp.re, minus ? gm.im : gp.im);
  // the step m / d: Smith's quotient of a real numerator
  const bool ce2 = fabs(d.re) < fabs(d.im);
  const double num2 = ce2 ? d.re : d.im, den2 = ce2 ? d.im : d.re;
  const double ratio2 = quot_near(num2, den2, rcp_near(den2));
  const double denom2 = (num2 * ratio2) + den2;
  em = edge_max(em, edge_bits(n2), edge_bits(den2));
  em = edge_max(em, edge_bits(denom2), 0);
  const double rd2 = rcp_near(denom2);
  const double mr = md * ratio2;
  const double qa = quot_near(mr, denom2, rd2), qb = quot_near(md, denom2, rd2);
  step = mk(ce2 ? qa : qb, ce2 ? -qb : -qa);
  x1 = mk(x.re - (ce2 ? qa : qb), x.im + (ce2 ? qb : qa));
  // (lo bounds den and den2 from below as well; f, s, g and den2 too large for
  // the quotients leave rad out of its range)
  double lo = min_abs(min_abs(min_abs(xf, yf), min_abs(xs, ys)), min_abs(num, num2));
  // (negative where the maximum is kEdge: a sign costs no comparison)
  lo = __builtin_copysign(lo, __hiloint2double((int)(((em & 0xFFFFu) + 1u) << 15), 0));
  const double rx = max_abs(rad.re, rad.im), ry = min_abs(rad.re, rad.im);
  // (ints: a chain of && would be a chain of branches)
  return (int(lo >= kTinyOp) & int(fabs(den) <= kHugeOp) & int(hyp_in_range(rx, ry)) &
          int(min_abs(np, nm) < max_abs(np, nm) * (1.0 - 1e-12)) &
          (int(x.re != x1.re) | int(x.im != x1.im))) != 0;
}

// Laguerre::laguerre for a polynomial of degree M >= 2 held in registers,
// every lane on its own x.  Leaves the Horner sums at the returned x in b,
// which are the coefficients of the deflated polynomial (b[j + 1] =
// coefficient j, laguerre.cc:133-139).  LOST: a polynomial of NaNs is left to
// lag_lost.
template <int M, bool LOST = false>
__device__ __forceinline__ bool lag_lane(const cx (&p)[M + 1], cx& x, cx (&b)[M + 1],
                                         const TrigTable* trig, bool& oob) {
  for (int i = 1; i <= kLagMaxIt; i++) {
    const LagEval v = lag_eval<M>(p, x, b);
    bool far = lag_far(v);
    if (__builtin_expect(!far, 0)) {
      bool near = lag_near(v);
      if (!near) lag_narrow<M>(v, b, far, near);
      if (near) return true;
    }
    cx x1, step;
    const int ok = int(lag_step<M>(b, x, x1, step)) & int(far);
    if (__builtin_expect(ok, 1)) {
      if (__builtin_expect(i % kLagMT == 0, 0)) {
        oob |= i / kLagMT >= 8;
        x = lag_kick(x, step, i);
      } else {
        x = x1;
      }
      continue;
    }
    keep(x.re);  // the general iteration shares nothing with the code above
    keep(x.im);
    if (LOST && lag_is_lost(p[0])) {
      const bool done = lag_lost(x, i, trig, oob);
      horner_sums<M>(p, x, b);
      return done;
    }
    if (lag_general<M>(b, x, i, trig, oob)) return true;
  }
  horner_sums<M>(p, x, b);  // not converged: the sums where it stopped
  return false;
}

// The same on a whole wavefront whose branches are all taken by the whole
// wave: SAME: every lane holds the same p and x; else each lane its own x
// (b is then not the sums at x, and the result means nothing: a lane that is
// done keeps x until the others are).  One wavefront alone on its SIMD waits
// 20 to 50 cycles at every branch; with lag_lane's returns the compiler made
// nine of an iteration, of which four were taken, one in four cycles of the
// chain.
template <int M, bool SAME>
__device__ __forceinline__ bool lag_wave(const cx (&p)[M + 1], cx& x, cx (&b)[M + 1],
                                         const TrigTable* trig, bool& oob) {
  unsigned long long run = ~0ull;  // lanes not done
  const unsigned long long me = 1ull << __lane_id();
  auto settle = [&](unsigned long long done) {
    run &= ~done;
    return SAME ? done != 0 : run == 0;
  };
  for (int i = 1; i <= kLagMaxIt; i++) {
    const LagEval v = lag_eval<M>(p, x, b);
    unsigned long long open = __ballot(!lag_far(v)) & run;
    if (__builtin_expect(open != 0, 0)) {
      unsigned long long done = __ballot(lag_near(v)) & open;
      if (open != done) {
        bool far, near;
        lag_narrow<M>(v, b, far, near);
        done |= __ballot(near) & open;
        open &= ~__ballot(far);
      }
      if (settle(done)) return true;
      open &= ~done;
    }
    cx x1, step;
    const bool ok = lag_step<M>(b, x, x1, step);
    const unsigned long long gen = (__ballot(!ok) | open) & run;
    if (__builtin_expect(i % kLagMT == 0, 0)) {
      const unsigned long long kick = run & ~gen;
      x1 = lag_kick(x, step, i);
      if (i / kLagMT >= 8) oob |= (kick & me) != 0;
    }
    if (__builtin_expect(gen != 0, 0)) {
      keep(x.re);  // the general iteration shares nothing with the code above
      keep(x.im);
      bool done = false;
      cx y = x;
      if (gen & me) done = lag_general<M>(b, y, i, trig, oob);
      if (gen & me) x1 = y;
      // (a lane that lag_general accepts keeps its x)
      const unsigned long long d = __ballot(done);
      if (SAME && d != 0) return true;
      if (run & me) x = x1;
      if (settle(d)) return true;
    } else if (SAME) {
      x = x1;
    } else {
      const bool mine = (run & me) != 0;
      x = mk(mine ? x1.re : x.re, mine ? x1.im : x.im);
    }
  }
  if (SAME) horner_sums<M>(p, x, b);  // not converged: the sums where it stopped
  return false;
}

}  // namespace tl
