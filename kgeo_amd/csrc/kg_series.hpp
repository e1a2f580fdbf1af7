// Sampling a ray along the uniform Mino-time grid by Taylor series.
//
// In Mino time the motion is polynomial.  With w = 1/r and c = cos(theta),
//
//   (dw/dtau)^2 = P(w) = 1 + A w^2 + B w^3 + C w^4,   A = a^2 - eta - lam^2,
//                 B = 2 (eta + (lam - a)^2),  C = -a^2 eta,
//   (dc/dtau)^2 = eta - E c^2 - a^2 c^4,              E = eta + lam^2 - a^2,
//
// so w'' = A w + 3/2 B w^2 + 2 C w^3 and c'' = -E c - 2 a^2 c^3, and the
// Taylor coefficients at any point follow from the ones before by the
// Cauchy products w^2, w^3, c^2, c^3.  The integrands of t, phi and sigma
// are rational in w and c; their series are the products' quotients,
// integrated term by term.  One expansion (about 5 P^2 multiply-adds for
// order P) replaces the elliptic functions and integrals of every sample on
// both sides of it, and a sample costs one polynomial per coordinate: the
// Gralla-Lupsasca formulas (kerr_raytracing_ana.py:126-683) are evaluated
// only at the rays' anchors (kg_sample.hpp).  w is regular at infinity,
// where r is not, and the poles of the integrands that the ray reaches or
// nearly reaches are taken out in closed form (below), so what limits a step
// is the distance to complex singularities: a ray needs about ten.
//
// Closed forms.  For a quartic motion y'^2 = k^2 + R1 y + R2 y^2 + R3 y^3 +
// R4 y^4 and either sign e, with N = k + e y' + (R1 / 2k) y, differentiating
// ln(N / y) gives
//
//   1/y = (1/k) [ -e (ln(N/y))' + (R3/2 y^2 + R4 y^3) / N ],
//
// whose last term is regular at y = 0 where N is not 0 (e y' > 0 there).
// It is used about infinity (y = w, k = 1: the log of I_1) or about the
// horizon (y = w - 1/r_+, k = (r_+^2 + a^2 - a lam)/r_+^2: the log of I_+),
// per lane, whichever is nearer.  1/w^2 = (-w'/w)' + B w / 2 + C w^2 takes
// out the double pole of I_2.  At the axis k is imaginary and the same
// identity, for y = 1 -+ c, k = i l, reads
//
//   l/y = -e (arg N)' - (T3/2 + T4 y)(4 l^3 - 2 l T1 y) /
//         (T1^2 + 4 l^2 (T2 + T3 y + T4 y^2)),   N = (2 l e y', 2 l^2 - T1 y),
//
// an angle that turns by 2 pi as the ray passes the axis.
//
// Everything is written in the grid's index (s = (tau - tau_0)/h), so a
// sample's offset is a small exact number.  Templated on the scalar type
// (kg_math.hpp); control follows the value.

#pragma once

#include "kg_geodesic.hpp"

namespace kg {

// A lane holds five coefficient arrays of kSeriesOrder + 1 doubles while it
// samples: at order 14 two waves per SIMD fit without spills (247 of 256
// registers; with sigma 14 values spill).  Measured at orders 12, 14 and 16
// (ms): 512 x 512 x 500 samples 2.14, 2.08, 2.11; 217 x 301 x 333 0.70, 0.69,
// 0.76; 64 x 64 x 100 0.31, 0.28, 0.26; a 16-image survey 8.0, 7.7, 7.8.
constexpr int kSeriesOrder = 14;
// Truncation: 1e-14 (of w, and in phi and t relative to 10 and 100), 3e-15 in
// cos(theta), whose error arccos magnifies next to the axis.  Against direct
// evaluation r and theta then agree to 1.4e-13 and 1.5e-14 or better at 99 % of the
// samples, phi to 2e-14 (the walk by addition theorems: 2.5e-13, 3e-14, 1.6e-13).
constexpr float kSeriesTolLog2 = -46.506993f;     // log2(1e-14)
constexpr float kSeriesTolPolarLog2 = -48.243958f;  // log2(3e-15)

// The fits' coefficients.  In the sample loops the number of instructions
// counts, not a chain's length (two waves per SIMD and several independent
// chains cover it), and so do registers: Horner's scheme with each constant
// as the multiply-add's scalar operand takes one instruction per coefficient.
// Left to itself the compiler keeps literal constants in vector registers
// across the loop and copies each before use, so the kernels read them from
// constant memory by scalar loads that it cannot hoist (fits()).
constexpr int kLogFit = 0, kLogTerms = 8, kAtanFit = 8, kAtanTerms = 11, kAcosFit = 19, kAcosTerms = 12;
#define KG_SERIES_FITS                                                                                       \
  0.6666666666666666, 0.4000000000000088, 0.28571428570803614, 0.22222222392713917, 0.18181795640132906,     \
      0.15386239702814658, 0.13268773138656886, 0.13086626147840102, -0.3333333333333333, 0.1999999999999552, \
      -0.14285714284666542, 0.11111111015256361, -0.09090904578123903, 0.07692183190826087,                  \
      -0.06664511447381948, 0.0585814891280221, -0.0508544973794026, 0.03923165829558719,                    \
      -0.01917687711906226, 0.1666666666666665, 0.07500000000020764, 0.044642857103423646,                   \
      0.03038194736709848, 0.02237204763174451, 0.017355259955786323, 0.013929652902326633,                  \
      0.011875494382636922, 0.0078029494773533175, 0.01603551434914882, -0.010749050339697808,               \
      0.028169218060881414
#if defined(__HIPCC__)
static __constant__ double kSeriesFits[31] = {KG_SERIES_FITS};
#endif
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(4))) const double FitCoef;
KG_INLINE const FitCoef* fits() {
  const FitCoef* p = (const FitCoef*)&kSeriesFits[0];
  asm volatile("" : "+s"(p));
  return p;
}
#else
typedef const double FitCoef;
inline const FitCoef* fits() {
  static const double c[31] = {KG_SERIES_FITS};
  return c;
}
#endif
template <int N> KG_INLINE double horner(const FitCoef* c, double z) {
  double p = c[N - 1];
#pragma unroll
  for (int n = N - 2; n >= 0; --n) {
#if defined(__HIP_DEVICE_COMPILE__)
    // as written: the compiler would copy c[n] to vector registers for v_fmac
    double q;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(q) : "v"(z), "v"(p), "s"(c[n]));
    p = q;
#else
    p = c[n] + z * p;
#endif
  }
  return p;
}

// sqrt(x) for 0 <= x <= 1 within an ulp: the hardware's reciprocal square root
// and two steps (Goldschmidt), without the scaling that denormals need.
KG_INLINE double sqrt_fast(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double y = __builtin_amdgcn_rsq(x + 1.0e-300);
  double g = x * y, h = 0.5 * y;
  double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  e = __builtin_fma(-g, g, x);
  return __builtin_fma(h, e, g);
#else
  return ::sqrt(x);
#endif
}

// acos_poly (kg_math.hpp) in as few instructions: the same reduction and
// coefficients, no branch.
KG_INLINE double acos_fast(double x) {
  const double ax = kfabs(x);
  const bool small = ax < 0.5;  // false for NaN
  // |x| an ulp above 1 (a sample on the axis) counts as 1
  const double z = small ? x * x : __builtin_fmax(0.5 - 0.5 * ax, 0.0);
  const double s = small ? ax : sqrt_fast(z);
  const double r = s + s * (z * horner<kAcosTerms>(fits() + kAcosFit, z));  // asin s
  // acos |x|: pi/2 - r, or 2 r; of x < 0: pi less that
  const double q = small ? kHalfPi - (r - 6.123233995736766e-17) : r + r;
  return x < 0.0 ? kPi - (q - 1.2246467991473532e-16) : q;
}
template <class T> KG_INLINE T acos_fast(const T& x) { return acos_poly(x); }

// x > 0 finite.  ln x = e ln 2 + 2 artanh(s), s = (m - 1)/(m + 1) for
// m = x / 2^e in [1/sqrt 2, sqrt 2) (e.g. Muller, Elementary Functions, ch. 4),
// 2 artanh(s) = 2 s + s z Q(z), z = s^2, Q a degree-7 Chebyshev fit (mpmath).
KG_INLINE double log_pos(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  double m = __builtin_amdgcn_frexp_mant(x);
  int e = __builtin_amdgcn_frexp_exp(x);
#else
  int e;
  double m = ::frexp(x, &e);
#endif
  const bool low = m < 0.7071067811865476;
  m = low ? 2.0 * m : m;
  const double k = static_cast<double>(low ? e - 1 : e);
  const double s = (m - 1.0) * frcp(m + 1.0);
  const double z = s * s;
  const double q = horner<kLogTerms>(fits() + kLogFit, z);
  // ln 2 in two parts, the first exact times any exponent
  return k * 0.6931471803691238 + (2.0 * s + (s * (z * q) + k * 1.9082149292705877e-10));
}

template <class T> KG_INLINE T log_pos(const T& x) { return klog(x); }

// atan2(y, x), within a few ulp; 0 for (0, 0).  The quotient of the smaller
// by the larger is brought below tan(pi/8) by atan t = pi/4 + atan((t - 1)/
// (t + 1)) (one division for both steps), atan t = t + t z R(z), z = t^2, R
// a degree-10 Chebyshev fit (mpmath, 7e-18).
KG_INLINE double atan2_fast(double y, double x) {
  const double ay = kfabs(y), ax = kfabs(x);
  const bool steep = ay > ax;
  const double lo = steep ? ax : ay, hi = steep ? ay : ax;
  const bool mid = lo > 0.41421356237309503 * hi;
  const double num = mid ? lo - hi : lo;
  const double den = mid ? lo + hi : hi;
  const double t = num * frcp(den + 1.0e-300);
  const double z = t * t;
  const double q = horner<kAtanTerms>(fits() + kAtanFit, z);
  double r = t + t * (z * q);
  r = mid ? r + 0.25 * kPi : r;
  r = steep ? kHalfPi - r : r;
  r = x < 0.0 ? kPi - r : r;
  return y < 0.0 ? -r : r;
}
template <class T> KG_INLINE T atan2_fast(const T& y, const T& x) { return katan2(y, x); }

// A lane's constants: SR_* of its ray, SF_* of its current expansion.  They
// are read where they are used: the kernels keep them in LDS (one column per
// lane), since the coefficient arrays fill the registers.
enum SeriesSlot : int {
  SR_A, SR_B, SR_C,           // the radial quartic in w
  SR_E, SR_Q,                 // the polar quartic: c'' = -E c + 2 Q c^3
  SR_l2,                      // minus its value at the axis
  SR_near,                    // 1 if the ray passes the axis closely enough for the angle, else 0
  SR_lam, SR_h, SR_ih,        // lambda, the grid step, 1/h
  SR_ap, SR_am, SR_bp, SR_bm, // residues of t' and phi' at 1 - r_+- w = 0
  SR_kh, SR_R1h,              // the radial quartic at the horizon: k and the slope R1
  SR_rm,                      // r_- (0: its pole taken as a constant, series_block_pixel)
  SF_n0, SF_n1, SF_eih, SF_b, // ln((n0 + e w' + n1 w)/(w - b)), e/h for the derivative per sample
  SF_kt, SF_kf,               // its factors in t and phi
  SF_sg,                      // y = 1 - sg c
  SF_ax,                      // -2 l sg/h
  SF_af, SF_wrap,             // the angle's factor in phi, and 2 pi of it past a pass
  SE_w, SE_v, SE_c, SE_u,     // the state where the last expansion ended
  SE_t, SE_f, SE_s,
  SE_q,                       // samples before this one (from the block's first) are queued
  SERIES_SLOTS
};

template <class T> struct LocalSlots {
  T v[SERIES_SLOTS];
  KG_INLINE void set(int q, const T& x) { v[q] = x; }
  KG_INLINE T operator()(int q) const { return v[q]; }
  KG_INLINE void fresh() const {}
};

// A, B, C: the radial quartic of the plan (radial_quartic).  The polar one is
// taken from the plan's rounded u_+, u_-, and not from eta and lam: u_+
// cancels for low spins and near-polar rays, and the samples of the reference
// (and of the direct evaluation) inherit that rounding, so the series does
// too: the axis value l2 from the plan's 1 - u_+.
template <class T, class Slots>
KG_INLINE void series_ray(const RayScalars<T>& c, const ThetaConsts<T>& tc, bool vortical, const T& lam, const T& A,
                          const T& B, const T& C, const T& h, Slots& k) {
  const T w2 = tc.v[TH_w] * tc.v[TH_w];
  const T& n = tc.v[TH_n];
  T E, Q, l2, om;  // om = 1 - u_+
  if (vortical) {  // c'^2 = a^2 (c^2 - u_-)(u_+ - c^2), a^2 = w^2/u_-
    const T um = tc.v[TH_A], up = um + tc.v[TH_B];
    const T q = w2 / um;
    E = -(q * (up + um));
    Q = -q;
    om = (1.0 - um) * (1.0 - n);
    l2 = q * (1.0 - um) * om;
  } else {  // c'^2 = w^2 (u_+ - c^2)(1 - k c^2/u_+)
    const T mu = tc.v[TH_k] / n;
    E = w2 * (1.0 + tc.v[TH_k]);
    Q = w2 * mu;
    om = 1.0 - n;
    l2 = w2 * om * (1.0 - mu);
  }
  k.set(SR_E, E);
  k.set(SR_Q, Q);
  k.set(SR_l2, l2);
  // the closest approach y1 = 1 - sqrt(u_+): N turns about 0 there if
  // T1 y1 < 2 l^2 (about l^2 for a close pass); rays that stay well away
  // take the pole of 1/(1 - c^2) in the series itself
  const T y1 = om / (1.0 + ksqrt(1.0 - om));
  k.set(SR_near, (val((2.0 * E - 4.0 * Q) * y1) < 1.5 * val(l2)) ? T(1.0) : T(0.0));
  k.set(SR_lam, lam);
  k.set(SR_A, A);
  k.set(SR_B, B);
  k.set(SR_C, C);
  k.set(SR_h, h);
  k.set(SR_ih, 1.0 / h);
  // t' = 1/w^2 + 2/w + (4 - 2 a lam w)/D + a^2 c^2, phi' = -lam + (lam +
  // 2 (a - lam) w)/D + lam/(1 - c^2), D = (1 - r_+ w)(1 - r_- w)
  const T idr = 1.0 / (c.rplus - c.rminus);
  k.set(SR_ap, 2.0 * (2.0 * c.rplus - c.a * lam) * idr);
  k.set(SR_am, -2.0 * (2.0 * c.rminus - c.a * lam) * idr);
  k.set(SR_bp, (lam * c.rplus + 2.0 * (c.a - lam)) * idr);
  k.set(SR_bm, -(lam * c.rminus + 2.0 * (c.a - lam)) * idr);
  k.set(SR_rm, c.rminus);
  // (r_+^2 + a^2 - a lam)/r_+^2, as this quartic has it: the closed form
  // holds for its own value at the horizon
  const T wh = 1.0 / c.rplus;
  const T ph = 1.0 + (wh * wh) * (A + wh * (B + wh * C));
  k.set(SR_kh, val(ph) > 0.0 ? ksqrt(ph) : T(0.0));
  k.set(SR_R1h, wh * (2.0 * A + wh * (3.0 * B + wh * (4.0 * C))));
}

// w, dw/dtau, c, dc/dtau and the integrals of t', phi', sigma' so far.
template <class T> struct SeriesState {
  T w, v, c, u;
  T t, f, s;
};

// One expansion: polynomials in the grid index about its centre.
template <class T, int P, bool SIG> struct Series {
  T w[P + 1], c[P + 1], t[P + 1], f[P + 1], s[SIG ? P + 1 : 1];
};

// Fixes a coefficient's value at this point of the program.  The compiler
// otherwise leaves a sum such as t's to its last use and keeps the arrays of
// every phase that adds to it alive until then (about ten arrays instead of
// six: the kernels would spill or hold one wave per SIMD).
KG_INLINE void settle(double& x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(x));
#endif
}
template <class T> KG_INLINE void settle(T&) {}

// Adds ft Z and ff Z, Z = 1/(l0 + l1 w), to the integrands t and f (from
// order 1; INIT: f starts here).
template <class T, int P, bool HAS_T, bool INIT>
KG_INLINE void series_reciprocal(const T& l0, const T& l1, const T (&w)[P + 1], const T& ft, const T& ff,
                                 T (&t)[P + 1], T (&f)[P + 1]) {
  T Z[P];
  Z[0] = 1.0 / (l0 + l1 * w[0]);
  const T g = -(l1 * Z[0]);
#pragma unroll
  for (int n = 0; n < P; ++n) {
    if (n > 0) {
      T z = w[1] * Z[n - 1];
#pragma unroll
      for (int j = 2; j <= n; ++j) z = z + w[j] * Z[n - j];
      Z[n] = g * z;
    }
    f[n + 1] = INIT ? ff * Z[n] : f[n + 1] + ff * Z[n];
    settle(f[n + 1]);
    if (HAS_T) {
      t[n + 1] = t[n + 1] + ft * Z[n];
      settle(t[n + 1]);
    }
  }
}

// The square's and the cube's order-n coefficients of x, given the square's
// lower ones.
template <class T, int P> KG_INLINE T series_square(const T (&x)[P + 1], int n) {
  T q = T(0.0);
  if (n > 0) q = x[0] * x[n];
#pragma unroll
  for (int j = 1; 2 * j < n; ++j) q = q + x[j] * x[n - j];
  if (n == 0) return x[0] * x[0];
  q = q + q;
  if (n % 2 == 0) q = q + x[n / 2] * x[n / 2];
  return q;
}
template <class T, int P> KG_INLINE T series_cube(const T (&x)[P + 1], const T (&x2)[P], int n) {
  T q = x[0] * x2[n];
#pragma unroll
  for (int j = 1; j <= n; ++j) q = q + x[j] * x2[n - j];
  return q;
}

// log2 |m| in single precision (finite m; -1e30 for 0).
KG_INLINE float series_log2(double m) {
#if defined(__HIP_DEVICE_COMPILE__)
  const float l = __builtin_amdgcn_logf(static_cast<float>(__builtin_amdgcn_frexp_mant(m))) +
                  static_cast<float>(__builtin_amdgcn_frexp_exp(m));
#else
  int e;
  const float l = ::log2f(static_cast<float>(::frexp(m, &e))) + static_cast<float>(e);
#endif
  return m == 0.0 ? -1.0e30f : l;
}

// x with |a| x^n = 2^ltol; 0 for NaN.
template <int N, class T> KG_INLINE float series_step(const T& a, float ltol) {
  const double m = kfabs(val(a));
  const float q = (ltol - series_log2(m)) * (1.0f / N);
#if defined(__HIP_DEVICE_COMPILE__)
  const float x = __builtin_amdgcn_exp2f(q);
#else
  const float x = ::exp2f(q);
#endif
  return m == m ? x : 0.0f;
}

// ln|(n0 + e v + n1 w)/(w - b)|, v the derivative per sample, iy = 1/(w - b)
template <class T, class Slots> KG_INLINE T series_log(const Slots& k, const T& w, const T& v, const T& iy) {
  return log_pos(kfabs((k(SF_n0) + k(SF_eih) * v + k(SF_n1) * w) * iy));
}

// The angle of N from the direction it has far from the pole, u the
// derivative per sample.  T1 y - 2 l^2 is written u'^2 - l^2 - (T2 y^2 +
// T3 y^3 + T4 y^4): next to the axis y = 1 -+ c has lost its digits and u
// has not.  The pass itself (y' = 0, N pointing back) is on the cut.
template <class T, class Slots> KG_INLINE T series_angle(const Slots& k, const T& c, const T& u) {
  const T y = 1.0 - k(SF_sg) * c;
  const T up = u * k(SR_ih);
  const T Q = k(SR_Q);
  const T d = (up * up - k(SR_l2)) - (y * y) * ((6.0 * Q - k(SR_E)) + Q * (y * (y - 4.0)));
  return atan2_fast(k(SF_ax) * u, d);
}

// The expansion about st, without the integrals' constants (series_match);
// returns the distance (in grid units, to both sides) over which the truncated
// terms stay below the tolerances.
template <class T, int P, bool SIG, class Slots>
KG_INLINE float series_expand(const RayScalars<T>& g, Slots& k, const SeriesState<T>& st, Series<T, P, SIG>& S) {
  const T &rp = g.rplus, &a2 = g.a2;
  const T h = k(SR_h);
  const T h2 = h * h;
  // polar motion
  {
    T c2[P];
    S.c[0] = st.c;
    S.c[1] = st.u * h;
    const T E = k(SR_E), Q = k(SR_Q);
    {
      const T hE = -(h2 * E), ha = h2 * (2.0 * Q);
#pragma unroll
      for (int n = 0; n < P; ++n) {
        c2[n] = series_square<T, P>(S.c, n);
        S.t[n + 1] = a2 * c2[n];
        settle(S.t[n + 1]);
        if (n + 2 <= P) S.c[n + 2] = (hE * S.c[n] + ha * series_cube<T, P>(S.c, c2, n)) * (1.0 / ((n + 1) * (n + 2)));
      }
    }
    // lam/(1 - c^2) = (lam/y + lam/(2 - y))/2, y = 1 - sg c; y'^2 = -l^2
    // + T1 y + T2 y^2 + T3 y^3 + T4 y^4, l > 0.  First 1/(2 - y) = 1/(1 + sg c)
    const T lam = k(SR_lam), l2 = k(SR_l2);
    const T sg = (val(st.c) >= 0.0) ? T(1.0) : T(-1.0);
    series_reciprocal<T, P, false, true>(T(1.0), sg, S.c, T(0.0), 0.5 * lam, S.t, S.f);
    // then lam/y: the angle's regular rest, a quotient of quadratics in y = 1
    // - sg c, y^2 = 1 - 2 sg c + c^2; away from the axis lam over 1 - sg c
    const bool nr = val(k(SR_near)) != 0.0;
    const T T1 = 2.0 * E - 4.0 * Q, T2 = 6.0 * Q - E, T3 = -4.0 * Q, T4 = Q;
    const T ll = lam * l2;
    const T p0 = -2.0 * T3 * ll, p1 = lam * (T1 * T3) - 4.0 * T4 * ll, p2 = 2.0 * lam * (T1 * T4);
    const T d0 = T1 * T1 + 4.0 * l2 * T2, d1 = 4.0 * l2 * T3, d2 = 4.0 * l2 * T4;
    const T Y2 = nr ? p2 : T(0.0), Y1 = nr ? -(sg * (p1 + 2.0 * p2)) : T(0.0), Y0 = nr ? p0 + p1 + p2 : lam;
    const T D2 = nr ? d2 : T(0.0), D1 = nr ? -(sg * (d1 + 2.0 * d2)) : -sg, D0 = nr ? d0 + d1 + d2 : T(1.0);
    T K[P];
#pragma unroll
    for (int n = 0; n < P; ++n) {
      K[n] = Y2 * c2[n] + Y1 * S.c[n];
      c2[n] = D2 * c2[n] + D1 * S.c[n];
      settle(K[n]);
      settle(c2[n]);
    }
    K[0] = K[0] + Y0;
    const T iD = 1.0 / (c2[0] + D0);
#pragma unroll
    for (int n = 0; n < P; ++n) {
      T x = K[n];
#pragma unroll
      for (int j = 1; j <= n; ++j) x = x - c2[j] * K[n - j];
      K[n] = x * iD;
      S.f[n + 1] = S.f[n + 1] + 0.5 * K[n];
      settle(S.f[n + 1]);
    }
    const T l = ksqrt(l2);
    k.set(SF_sg, sg);
    k.set(SF_ax, -(2.0 * l) * (sg * k(SR_ih)));
    k.set(SF_af, nr ? -0.5 * (lam / l) : T(0.0));
  }
  // radial motion.  About the horizon once it is the nearer pole and N there
  // is not near 0 (it vanishes on the other branch of the motion: rays that
  // linger at a photon orbit), else about infinity, where N = 1 + |v|
  const T wh = 1.0 / rp;
  const T A = k(SR_A), B = k(SR_B), C = k(SR_C), kh = k(SR_kh), R1h = k(SR_R1h);
  const bool hor = (val(st.w) > 0.4 * val(wh)) && (val(kh) > 0.01) &&
                   (val(kh * kfabs(st.v) + (kh * kh + 0.5 * R1h * (st.w - wh))) > 0.25 * val(kh * kh));
  const T b = hor ? wh : T(0.0);
  const T kb = hor ? kh : T(1.0);
  const T ikb = 1.0 / kb;
  const T n1 = hor ? 0.5 * R1h * ikb : T(0.0);
  const T n0 = kb - n1 * b;
  const T e = (val(st.v) >= 0.0) ? T(1.0) : T(-1.0);
  const T eih = e * k(SR_ih);
  const T ap = k(SR_ap), bp = k(SR_bp);
  // factors of q, Z = 1/(l0 + l1 w) and M = 1/(1 - r_- w) in t' and phi'
  const T tq = hor ? -(ap * wh) * ikb : T(2.0);
  const T pq = hor ? -(bp * wh) * ikb : T(0.0);
  k.set(SF_n0, n0);
  k.set(SF_n1, n1);
  k.set(SF_eih, eih);
  k.set(SF_b, b);
  k.set(SF_kt, -(e * tq));
  k.set(SF_kf, -(e * pq));
  S.w[0] = st.w;
  S.w[1] = st.v * h;
  {
    T q[P];  // the numerator (R3/2) y^2 + C y^3 in powers of w, then its quotient by N
    T w2[P];
    {
      const T R3 = B + 4.0 * C * b;
      const T m2 = 0.5 * R3 - 3.0 * C * b, m1 = b * (3.0 * C * b - R3), m0 = (b * b) * (0.5 * R3 - C * b);
      const T hA = h2 * A, hB = h2 * (1.5 * B), hC = h2 * (2.0 * C), hb = 0.5 * B;
#pragma unroll
      for (int n = 0; n < P; ++n) {
        w2[n] = series_square<T, P>(S.w, n);
        const T w3 = series_cube<T, P>(S.w, w2, n);
        if (n + 2 <= P) S.w[n + 2] = (hA * S.w[n] + hB * w2[n] + hC * w3) * (1.0 / ((n + 1) * (n + 2)));
        q[n] = m1 * S.w[n] + m2 * w2[n] + C * w3;
        S.t[n + 1] = S.t[n + 1] + (hb * S.w[n] + C * w2[n]);
        if (SIG) S.s[n + 1] = S.t[n + 1];
        settle(q[n]);
        settle(S.t[n + 1]);
      }
      q[0] = q[0] + m0;
    }
#pragma unroll
    for (int n = 0; n < P; ++n) {
      w2[n] = (eih * static_cast<double>(n + 1)) * S.w[n + 1] + n1 * S.w[n];  // N
      settle(w2[n]);
    }
    const T iN = 1.0 / (w2[0] + n0);
#pragma unroll
    for (int n = 0; n < P; ++n) {
      T x = q[n];
#pragma unroll
      for (int j = 1; j <= n; ++j) x = x - w2[j] * q[n - j];
      q[n] = x * iN;
      S.t[n + 1] = S.t[n + 1] + tq * q[n];
      S.f[n + 1] = S.f[n + 1] + pq * q[n];
      settle(S.t[n + 1]);
      settle(S.f[n + 1]);
    }
  }
  series_reciprocal<T, P, true, false>(hor ? T(0.0) : T(1.0), hor ? T(1.0) : -rp, S.w, hor ? T(2.0) : ap,
                                       hor ? T(0.0) : bp, S.t, S.f);
  series_reciprocal<T, P, true, false>(T(1.0), -k(SR_rm), S.w, k(SR_am), k(SR_bm), S.t, S.f);
  S.f[1] = S.f[1] - k(SR_lam);
#pragma unroll
  for (int n = 1; n <= P; ++n) {
    const T f = h * (1.0 / n);
    S.t[n] = S.t[n] * f;
    S.f[n] = S.f[n] * f;
    if (SIG) S.s[n] = S.s[n] * f;
  }
  // step: |coefficient| x^n at the two last orders below the tolerances
  constexpr float lt = kSeriesTolLog2;
  const float lw = lt + series_log2(kmax(kfabs(val(S.w[0])), kfabs(val(S.w[1]))));
  float x = series_step<P - 1>(S.w[P - 1], lw);
  const float xs[7] = {series_step<P>(S.w[P], lw),
                       series_step<P - 1>(S.c[P - 1], kSeriesTolPolarLog2),
                       series_step<P>(S.c[P], kSeriesTolPolarLog2),
                       series_step<P - 1>(S.t[P - 1], lt + 6.64386f),   // 100 times
                       series_step<P>(S.t[P], lt + 6.64386f),
                       series_step<P - 1>(S.f[P - 1], lt + 3.32193f),   // 10 times
                       series_step<P>(S.f[P], lt + 3.32193f)};
#pragma unroll
  for (int q = 0; q < 7; ++q) x = xs[q] < x ? xs[q] : x;
  return x;
}

// The state at offset x of the expansion (FULL: with v and u per unit of Mino
// time; otherwise a sample's values); an: the axis angle there.
template <class T, int P, bool SIG, bool FULL, class Slots>
KG_INLINE void series_at(const Slots& k, const Series<T, P, SIG>& S, const T& x, SeriesState<T>& o, T& r, T& an) {
  T w = S.w[P], c = S.c[P], t = S.t[P], f = S.f[P], s = S.s[SIG ? P : 0];
  T v = w, u = c;
#pragma unroll
  for (int n = P - 1; n >= 0; --n) {
    if (n < P - 1) {
      v = w + x * v;
      u = c + x * u;
    }
    w = S.w[n] + x * w;
    c = S.c[n] + x * c;
    t = S.t[n] + x * t;
    f = S.f[n] + x * f;
    if (SIG) s = S.s[n] + x * s;
  }
  const T y = w - k(SF_b);
  const T i = frcp(w * y);
  r = y * i;
  const T lg = series_log(k, w, v, w * i);
  const T ih = k(SR_ih);
  const T vr = v * (r * ih);
  o.t = t - vr + k(SF_kt) * lg;
  o.f = f + k(SF_kf) * lg;
  if (SIG) o.s = s - vr;
  an = series_angle(k, c, u);
  o.f = o.f + (k(SF_af) * an - (val(an) > 0.0 ? k(SF_wrap) : T(0.0)));
  o.w = w;
  o.c = c;
  if (FULL) {
    o.v = v * ih;
    o.u = u * ih;
  }
}

// The integrals' constants of a new expansion: t0, f0, s0 at its left end, the
// offset x (where the last one ended).  far (an observer at infinity): t0 and
// s0 are the reference's constants of the ray, infinite, NaN or about 1e16, of
// which the terms at the left end, infinite too, are a part already.
template <class T, int P, bool SIG, class Slots>
KG_INLINE void series_match(Slots& k, Series<T, P, SIG>& S, const T& x, const T& t0, const T& f0, const T& s0,
                            bool far) {
  S.t[0] = T(0.0);
  S.f[0] = T(0.0);
  S.s[0] = T(0.0);
  k.set(SF_wrap, T(0.0));
  SeriesState<T> o;
  T r, an;
  series_at<T, P, SIG, false>(k, S, x, o, r, an);
  S.t[0] = far ? t0 : t0 - o.t;
  S.f[0] = f0 - o.f;
  if (SIG) S.s[0] = far ? s0 : s0 - o.s;
  // approaching (an < 0): a later angle > 0 is past the pass, a turn further on
  k.set(SF_wrap, val(an) < 0.0 ? 2.0 * kPi * k(SF_af) : T(0.0));
}

// y and dy/dx at x of the motion y'' = q1 y + q2 y^2 + q3 y^3 from y, dy at 0.
template <class T, int P> KG_INLINE void series_motion(const T& q1, const T& q2, const T& q3, const T& x, T& y, T& dy) {
  T a[P + 1], a2[P];
  a[0] = y;
  a[1] = dy;
#pragma unroll
  for (int n = 0; n + 2 <= P; ++n) {
    a2[n] = series_square<T, P>(a, n);
    a[n + 2] = (q1 * a[n] + q2 * a2[n] + q3 * series_cube<T, P>(a, a2, n)) * (1.0 / ((n + 1) * (n + 2)));
  }
  T p = a[P], d = a[P];
#pragma unroll
  for (int n = P - 1; n >= 0; --n) {
    if (n < P - 1) d = p + x * d;
    p = a[n] + x * p;
  }
  y = p;
  dy = d;
}

// The motion x further on from the state kept in the SE slots, by its own
// series: a third of an expansion's work, where the integrals' series is then
// centred.
template <class T, class Slots> KG_INLINE void series_advance(const Slots& k, const T& x, SeriesState<T>& st) {
  constexpr int P = kSeriesOrder;
  const T h = k(SR_h), ih = k(SR_ih);
  const T h2 = h * h;
  st.c = k(SE_c);
  st.u = k(SE_u) * h;
  series_motion<T, P>(-(h2 * k(SR_E)), T(0.0), h2 * (2.0 * k(SR_Q)), x, st.c, st.u);
  st.u = st.u * ih;
  st.w = k(SE_w);
  st.v = k(SE_v) * h;
  series_motion<T, P>(h2 * k(SR_A), h2 * (1.5 * k(SR_B)), h2 * (2.0 * k(SR_C)), x, st.w, st.v);
  st.v = st.v * ih;
}

}  // namespace kg
