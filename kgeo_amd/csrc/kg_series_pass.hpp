// The sample passes of the linspace grid by Taylor series (kg_series.hpp),
// shared by the plain kernels (kgeo_raytrace.hip) and the batched survey
// (kgeo_batch.hip).
//
// A ray's grid is split into two blocks of consecutive samples.  The first
// starts from the observer, whose state is known in closed form, the second
// from an anchor, a direct evaluation (Landen ladder, Carlson duplications)
// of its first sample:
//   heads   one lane per (pixel, head): the anchors, and the last grid sample
//           (at 1e-10 of the horizon for captured rays, where only the
//           direct formulas reproduce the reference's rounding);
//   series  one lane per (pixel, block, part): samples of the block;
//   fixup   one lane per (queued range, sample): direct evaluation of what
//           the series leaves (kg_sample.hpp).
// The anchor keeps every sample within half a ray of the reference's own
// arithmetic: near the critical curve a difference in the last bit grows
// along the ray (by 1/d over a ray at distance d from the curve, 1/sqrt(d)
// over half of one), in the series and in the closed formulas alike.
//
// Where the rays are too few to fill the chip, the samples of a block are
// split into parts, one lane each, which all run the block's expansions up to
// their own samples' end: the results do not depend on the parts.  (More
// blocks instead of parts would run fewer expansions per lane, but more
// anchors, and would let near-critical rays change by 1e-9 with the number of
// pixels.)
//
// An expansion covers the samples on both sides of its centre, to which the
// motion alone is carried first (series_advance).
//
// The lanes of a wave take their steps together (the smallest any lane
// needs), so a sample index is uniform across the wave and every store is
// one contiguous row; a lane that would hold the others to steps below
// 1/kSeriesMinStep of its block leaves the rest of it to the fixup pass.  So a
// ray's last bits depend on the 64 rays of its wave: the same neighbours give
// the same bits for any number of pixels and parts, others (a ragged tail, a
// crop that moves the tiles) the same samples to the truncation.
// A queued range ends with its block (series_fixup_end).

#pragma once

#include "kg_sample.hpp"
#include "kg_series.hpp"

namespace kg {

constexpr int kSeriesBlocks = 2;
constexpr int kSeriesMaxParts = 8;
constexpr double kSeriesMinStep = 128.0;
// Rays followed past their end: |r - r_+|, and |r|/r_o on the way out, beyond
// which the closed forms are not used.
constexpr double kSeriesHorizon = 1.0e-3, kSeriesFar = 0.1;
// An expansion holds for the same distance x on both sides of its centre, so
// the next is centred ahead of where the last ended, by this part of its x:
// the distance to the nearest singularity (about 10 x) shrinks by at most the
// distance moved, so the new x is at least 1 - 1.8 / 10 of the old.
constexpr float kSeriesAhead = 0.8f;

#if defined(__HIPCC__)
// A lane's column of its wave's LDS (LocalSlots).  fresh() keeps the loads
// that follow it in their loop iteration: hoisted, the constants would hold
// registers through the sample loops.
struct LdsSlots {
  double (*s)[64];
  int lane;
  __device__ void set(int q, double x) { s[q][lane] = x; }
  __device__ double operator()(int q) const { return s[q][lane]; }
  __device__ void fresh() const { asm volatile("" ::: "memory"); }
};
#endif

// First sample of block b of nb (nb: the end, the last grid sample).
KG_INLINE int64_t series_start(int64_t ngeo, int64_t b, int64_t nb) {
  const int64_t last = ngeo - 1;
  return b >= nb ? last : (last * b + nb - 1) / nb;
}

// Blocks per ray: two, so that no sample is more than half a ray from its
// block's start (of 3 samples the middle one is not in any case).  Against direct
// evaluation, rays near the critical curve (four observers, 240 x 240 pixels,
// grids of 4 .. 16 samples) are off by up to 4e-9 of r in one block over the
// whole ray; in two of which the second started at a multiple of 8 samples
// (0.7 of the ray for grids of 32) by 2.5e-11; in two halves by 5e-12.
KG_INLINE int64_t series_blocks(int64_t ngeo) { return ngeo - 1 > kSeriesBlocks ? kSeriesBlocks : 1; }

// First sample of part q of `parts` of a block's samples js .. je - 1: inside
// the block a multiple of kFixupSpan, so that a queued range lies in one part.
KG_INLINE int64_t series_part(int64_t js, int64_t je, int64_t q, int64_t parts) {
  if (q <= 0) return js;
  if (q >= parts) return je;
  const int64_t s = (js + (je - js) * q / parts) / kFixupSpan * kFixupSpan;
  return s > js ? s : js;
}

// End of the queued range that starts at sample j: fixup_end, or the end of
// j's block before it.  far (an observer at infinity): sample 0 of the served
// rays is a range of its own.
KG_INLINE int64_t series_fixup_end(int64_t j, int64_t ngeo, bool walked, bool far) {
  const int64_t e = fixup_end(j, ngeo, walked), nb = series_blocks(ngeo);
  if (far && walked && j == 0) return 1;
  const int64_t s = nb > 1 ? series_start(ngeo, 1, nb) : 0;
  return (j < s && s < e) ? s : e;
}

// Queued ranges per pixel at most: one per window of kFixupSpan samples, one
// more for the window that the second block starts in and one for the sample 0
// of an observer at infinity.
constexpr int64_t kSeriesMoreItems = 2;
KG_INLINE int64_t series_items(int64_t ngeo) {
  return fixup_items(ngeo) + (series_blocks(ngeo) > 1 ? kSeriesMoreItems : 1);
}

// Queue samples j .. e - 1 of a block: from j to the next window, then one
// item per window.  walked: the last grid sample is a head's.
template <class Push> KG_INLINE void push_windows(Push& push, int64_t i, int64_t j, int64_t e, bool walked) {
  for (; j < e; j = (j / kFixupSpan + 1) * kFixupSpan) push(i, j, walked);
}

// Parts per block for npix rays (all images') sampled together on grids of
// ngeo samples: enough that 2^17 (ray, part) lanes fill the chip's 2048 places
// at two waves per SIMD.  More cost their expansions again.  Measured with 1,
// 2, 4 and 8 parts (ms): 1000 rays x 250 samples 0.361, 0.303, 0.272, 0.257;
// 64 x 64 x 100 0.316, 0.292, 0.286, 0.280; 217 x 301 x 333 0.81, 0.69, 0.72,
// 0.85; 512 x 512 x 500 2.03, 2.19, 2.51, 3.18; a survey of 16 images (64 .. 512
// pixels a side, 50 .. 400 samples) 7.6, 8.1, 8.1, 8.1.
inline int64_t pick_parts(int64_t npix, int64_t ngeo) {
  int64_t want = npix > 0 ? (1LL << 17) / npix : 1;
  const int64_t most = ngeo / series_blocks(ngeo) / kFixupSpan;
  if (want > kSeriesMaxParts) want = kSeriesMaxParts;
  if (want > most) want = most;
  return want < 1 ? 1 : want;
}

// Anchor records: theta (c, dc/dtau, G_phi, G_t), radial (r, I_+, I_-, I_1, I_2, dw/dtau);
// record 0 the last sample, record b the first sample of block b.
constexpr int kThSFields = 4;
constexpr int kRSFields = 6;

// Smallest x over the wave's lanes (all 64 must call), x >= 0.
KG_INLINE float wave_min(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  int v = __float_as_int(x);  // ordered as integers for x >= 0
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) {
    const int o = __shfl_xor(v, s);
    v = o < v ? o : v;
  }
  return __int_as_float(__builtin_amdgcn_readfirstlane(v));
#else
  return x;
#endif
}

// d cos(theta)/dtau from the Jacobi state at a sample (theta_out's cos theta).
template <class T>
KG_INLINE void theta_motion(const ThetaConsts<T>& tc, const ThState<T>& st, T& c, T& u) {
  const T* v = tc.v;
  if (tc.kind == THK_VORT) {
    c = v[TH_h] * ksqrt(v[TH_A] + v[TH_B] * (st.s * st.s));
    u = -(v[TH_w] * v[TH_B]) * (st.s * st.c * st.d) / c;
  } else {
    c = v[TH_A] * st.s;
    u = -(v[TH_w] * v[TH_A]) * (st.c * st.d);
  }
}

// d(1/r)/dtau from the Jacobi state at a sample (radial_out's r).
template <class T> KG_INLINE T radial_motion(const RadialConsts<T>& rc, const RState<T>& st) {
  const T* v = rc.v;
  const T& Xs = v[R_Xs];
  if (rc.rcase == 4) {
    const T& g0 = v[C4_g0];
    const T den = st.c + g0 * st.s;
    const T num = -v[C4_a2] * (g0 * st.c - st.s) - v[C4_b1] * den;  // r den
    return v[C4_a2] * Xs * st.d * (1.0 + g0 * g0) / (num * num);
  }
  if (rc.rcase == 3) {
    const T &AA = v[C3_AA], &BB = v[C3_BB], &r1 = v[C3_rr1], &r2 = v[C3_rr2];
    const T num = (BB * r2 - AA * r1) + (BB * r2 + AA * r1) * st.c;
    return 2.0 * AA * BB * (r2 - r1) * Xs * (st.s * st.d) / (num * num);
  }
  const T num = v[C2_rr4] * v[C2_rr31] - v[C2_rr3] * v[C2_rr41] * (st.s * st.s);
  return 2.0 * Xs * v[C2_rr41] * v[C2_rr31] * v[C2_rr43] * (st.s * st.c * st.d) / (num * num);
}

// Whether the heads and the series serve a pixel: its motion (theta_pick's
// walk) and PL_SERVED.  The same in every pass, block 0's included; the fixup
// pass takes the other pixels whole.
KG_INLINE bool series_serves(const double* __restrict__ plan, int64_t stride, int64_t p, const ThetaPick& tp) {
  return tp.walk && plan[static_cast<int64_t>(PL_SERVED) * stride + p] != 0.0;
}

// Theta head hd (0 the last sample, b the anchor of block b) of output pixel
// i: theta and the parked G_phi, G_t of its sample, and an anchor's motion.
template <class T = double>
KG_INLINE uint32_t series_theta_head_pixel(const double* __restrict__ plan, int64_t stride, int64_t p, uint32_t gflags,
                                           const SampleOut& o, int64_t i, int64_t hd, int64_t nb, const Records& rt) {
  ThetaConsts<T> tc;
  const ThetaPick tp = theta_pick(plan, stride, p, gflags, o, tc);
  if (!series_serves(plan, stride, p, tp)) return 0u;
  tc.kind = tp.kind;
  JacobiLadder<T> lad;
  jacobi_ladder(tc.v[TH_mp], lad);
  const int64_t j = hd == 0 ? o.ngeo - 1 : series_start(o.ngeo, hd, nb);
  WalkStep<T, 1> w;
  theta_init(tc, w);
  const double tau = mino_tau(j, o.ngeo, tp.stop, false);
  const T arg = theta_arg(tc, T(tau));
  ThState<T> ts;
  WalkState<T, 1> st;
  theta_direct<T, -1, true>(tc, lad, w, arg, ts, st);
  T th = T(0.0), Gph = T(0.0), Gt = T(0.0);
  theta_out<T, -1>(tc, arg, ts, true, th, Gph, Gt);
  if (hd > 0) {
    T c, u;
    theta_motion<T>(tc, ts, c, u);
    // next to a singularity of Pi (walk_enter) the anchor is not used
    if (!kfinite(val(st.P[0]))) c = T(NAN);
    *rt.at(hd, kThSFields, 0, p) = val(c);
    *rt.at(hd, kThSFields, 1, p) = val(u);
    *rt.at(hd, kThSFields, 2, p) = val(Gph);
    *rt.at(hd, kThSFields, 3, p) = val(Gt);
  }
  return loop_status(theta_store<T, true>(o, j * o.npix + i, tau, th, Gph, Gt), lad);
}

// Radial head hd: the sample's r and radial integrals, and an anchor's motion.
// Head 0 also stores r at sample 0, from the closed form (an ulp of its
// argument is up to 6e-11 of r_o for rays near the critical curve, where the
// plan's rounded roots place the observer; the closed form keeps sample 0
// with the samples it gives next to it).
template <class T = double>
KG_INLINE uint32_t series_radial_head_pixel(const double* __restrict__ plan, int64_t stride, int64_t p,
                                            uint32_t gflags, const SampleOut& o, int64_t i, int64_t hd, int64_t nb,
                                            const Records& rt) {
  if (!walk_ok(o, (gflags & GF_ANY_STEP_ZERO) != 0) || plan[static_cast<int64_t>(PL_SERVED) * stride + p] == 0.0)
    return 0u;
  RadialConsts<T> rc;
  T lam;
  double stop;
  radial_pick(plan, stride, p, rc, lam, stop);
  JacobiLadder<T> lad;
  jacobi_ladder(rc.v[R_k], lad);
  const int64_t j = hd == 0 ? o.ngeo - 1 : series_start(o.ngeo, hd, nb);
  const double tau = mino_tau(j, o.ngeo, stop, false);
  const T dv = rc.v[R_Xs] * tau;
  const T X = rc.v[R_U0] - dv;
  RState<T> rs;
  radial_state<T, -1>(rc, lad, X, dv, true, rs);
  const RadialOut<T> ro = radial_out<T, -1>(rc, T(tau), rs, true);
  T v = T(0.0);
  if (hd == 0 && o.r && o.ngeo > 1) {
    RState<T> r0;
    r0.s = rc.v[R_sn0];
    r0.c = rc.v[R_cn0];
    r0.d = rc.v[R_dn0];
    o.r[i] = val(radial_out<T, -1>(rc, T(0.0), r0, false).r);
  }
  if (hd > 0) {
    v = radial_motion<T>(rc, rs);
    // next to a singularity of an integral (walk_enter, block_log_enter)
    // the closed formulas lose digits: the anchor is not used
    bool ok = kfinite(val(v));
    WalkStep<T, 3> w;
    radial_init<T, -1>(rc, w);
    const bool blocks = rc.rcase == 3 || rc.rcase == 4;
    // below MINSPIN case 3 has no third-kind part of I_-
    const int np = (rc.rcase == 3 && val(rc.v[C3_hasm]) == 0.0) ? 2 : 3;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      WalkState<T, 3> st;
      walk_enter(w, q, rs.Pi[q], X, rs.s, rs.c, rs.d, st);
      const bool fine = kfinite(val(st.P[q])) & (!blocks | kfinite(val(block_log_enter(rs.lg[q]))));
      ok = ok & ((q >= np) | fine);
    }
    if (!ok) v = T(NAN);
  }
  *rt.at(hd, kRSFields, 0, p) = val(ro.r);
  *rt.at(hd, kRSFields, 1, p) = val(ro.Ip);
  *rt.at(hd, kRSFields, 2, p) = val(ro.Im);
  *rt.at(hd, kRSFields, 3, p) = val(ro.I1);
  *rt.at(hd, kRSFields, 4, p) = val(ro.I2);
  *rt.at(hd, kRSFields, 5, p) = val(v);
  return loop_status(false, lad);
}

// A head's sample: r and the combination of its radial record with the
// theta pass's parked G_phi, G_t (as radial_store).
template <class T>
KG_INLINE bool series_head_store(const SampleOut& o, const CombineConsts<T>& cmb, int64_t idx, double tau,
                                 const Records& rr, int64_t hd, int64_t col) {
  RadialOut<T> ro;
  ro.r = T(*rr.at(hd, kRSFields, 0, col));
  ro.Ip = T(*rr.at(hd, kRSFields, 1, col));
  ro.Im = T(*rr.at(hd, kRSFields, 2, col));
  ro.I1 = T(*rr.at(hd, kRSFields, 3, col));
  ro.I2 = T(*rr.at(hd, kRSFields, 4, col));
  return radial_store_g<T, true>(o, cmb, idx, tau, ro, T(o.ph[idx]), T(o.t[idx]));
}

// Part q of `parts` of block b of output pixel i (plan column p) by the
// series.  All lanes of a wave call together; `in` is false for a lane without a pixel
// (its i and p must be valid).  EARLY: block 0 of several, which reads nothing
// of the plan's radial constants (kg_setup_radial may still be writing them)
// and no record; not below MINSPIN, and for no observer at infinity, whose t
// and sigma start from the anchor's.  Returns the status bits.
template <bool SIG, bool EARLY, class Slots, class Push, class T = double>
KG_INLINE uint32_t series_block_pixel(const RayScalars<T>& c, const double* __restrict__ plan, int64_t stride,
                                      int64_t p, uint32_t gflags, const SampleOut& o, int64_t i, bool in, int64_t b,
                                      int64_t nb, int64_t q, int64_t parts, const Records& rth, const Records& rr,
                                      Slots& k, Push& push) {
  constexpr int P = kSeriesOrder;
  const int64_t last = o.ngeo - 1;
  const int64_t js = series_start(o.ngeo, b, nb), je = series_start(o.ngeo, b + 1, nb);
  if (js >= je) {  // a grid of one sample
    if (in && q + 1 == parts) push(i, js, false);
    return 0u;
  }
  const int64_t ps = series_part(js, je, q, parts), pe = series_part(js, je, q + 1, parts);
  const bool ends = b + 1 == nb && q + 1 == parts;  // the last sample is this part's too
  if (ps >= pe) return 0u;  // never the block's last part
  SeriesState<T> st;
  double stop;
  const bool far = !EARLY && c.r_o_inf;
  bool live = in;
  bool bad = false;
  {
    ThetaConsts<T> tc;
    const ThetaPick tp = theta_pick(plan, stride, p, gflags, o, tc);
    stop = tp.stop;
    const T lam = T(plan[static_cast<int64_t>(PL_LAM) * stride + p]);
    if (live && !series_serves(plan, stride, p, tp)) {
      // no heads for this pixel either: every sample, the last included
      push_windows(push, i, ps, ends ? o.ngeo : pe, false);
      live = false;
    }
    const T h = T(stop / static_cast<double>(o.ngeo - 1));
    series_ray(c, tc, tp.kind == THK_VORT, lam, T(plan[static_cast<int64_t>(PL_QA) * stride + p]),
               T(plan[static_cast<int64_t>(PL_QB) * stride + p]), T(plan[static_cast<int64_t>(PL_QC) * stride + p]), h, k);
    if (!EARLY && c.minspin && plan[static_cast<int64_t>(PL_RCASE) * stride + p] == 3.0) {
      // below MINSPIN the reference leaves the third-kind part of I_- out in
      // this case (kerr_raytracing_ana.py:529): 1/(r - r_-) is a constant
      const double* r0 = plan + static_cast<int64_t>(PL_R) * stride + p;
      const T kc = -(T(r0[C3_AA * stride]) + T(r0[C3_BB * stride])) * T(r0[C3_iImd * stride]);
      const T m0 = 1.0 + T(c.rminus) * kc;
      k.set(SR_am, k(SR_am) * m0);
      k.set(SR_bm, k(SR_bm) * m0);
      k.set(SR_rm, T(0.0));
    }
    const CombineConsts<T> cmb = combine_consts(c, lam);
    if (!EARLY && live && ends) bad = series_head_store<T>(o, cmb, last * o.npix + i, stop, rr, 0, p) || bad;
    const int64_t idx = js * o.npix + i;
    st.t = T(0.0);
    st.f = T(0.0);
    st.s = T(0.0);
    if (EARLY || b == 0) {
      // from infinity: 1/w and 1/w^2 finite, w as good as 0
      const T w0 = far ? T(1.0e-30) : 1.0 / T(c.r_o);
      st.w = w0;
      st.v = ksqrt(1.0 + w0 * w0 * (k(SR_A) + w0 * (k(SR_B) + w0 * k(SR_C))));
      st.c = c.cos_th;
      st.u = T(plan[static_cast<int64_t>(PL_U0) * stride + p]);
    } else {
      st.c = T(*rth.at(b, kThSFields, 0, p));
      st.u = T(*rth.at(b, kThSFields, 1, p));
      st.w = 1.0 / T(*rr.at(b, kRSFields, 0, p));
      st.v = T(*rr.at(b, kRSFields, 5, p));
    }
    if (!EARLY && live && nb > 1 && (b > 0 || far)) {
      const int64_t hd = b > 0 ? b : 1;
      RadialOut<T> ro;
      ro.r = T(*rr.at(hd, kRSFields, 0, p));
      ro.Ip = T(*rr.at(hd, kRSFields, 1, p));
      ro.Im = T(*rr.at(hd, kRSFields, 2, p));
      ro.I1 = T(*rr.at(hd, kRSFields, 3, p));
      ro.I2 = T(*rr.at(hd, kRSFields, 4, p));
      Sample<T> s;
      combine(cmb, T(mino_tau(series_start(o.ngeo, hd, nb), o.ngeo, stop, false)), ro, T(0.0),
              T(*rth.at(hd, kThSFields, 2, p)), T(*rth.at(hd, kThSFields, 3, p)), s);
      st.t = -s.t;
      st.s = -s.sig;
      if (b > 0) st.f = -s.ph;
    }
    // the series needs a pole at the axis (lam != 0) and a finite start; t and
    // sigma of an observer at infinity are what the anchor's are
    const bool fin = kfinite(val(st.t)) && kfinite(val(st.s));
    const bool ok = kfinite(val(st.w)) & kfinite(val(st.v)) & kfinite(val(st.c)) & kfinite(val(st.u)) &
                    (far ? nb > 1 : fin) & kfinite(val(st.f)) & (val(k(SR_l2)) > 0.0) & (val(lam) != 0.0) &
                    (val(st.w) > 0.0) & kfinite(val(k(SR_E))) & kfinite(val(h));
    bad = bad || (live && ok && !fin);
    // at infinity itself t and sigma are the difference of two infinite terms:
    // as the reference has it
    const int64_t first = far && b == 0 ? 1 : 0;
    if (live && ps < first) push(i, 0, true);
    if (live && !ok) {
      push_windows(push, i, ps < first ? first : ps, pe, true);
      live = false;
    }
    if (live && ps == js) {
      // the block's first sample
      const double tau = mino_tau(js, o.ngeo, stop, false);
      const T th = acos_poly(st.c);
      if (o.tau_out) o.tau_out[idx] = tau;
      if (o.th && b == 0) o.th[idx] = val(th);  // the anchor's head wrote it
      if (o.r && b > 0) o.r[idx] = *rr.at(b, kRSFields, 0, p);  // sample 0: radial head 0
      o.t[idx] = val(-st.t);
      o.ph[idx] = val(-st.f);
      if (SIG) o.sig[idx] = val(-st.s);
    }
    if (!live) {
      // a harmless motion for the lane's share of the wave's steps
      st.w = T(1.0e-3);
      st.v = T(0.0);
      st.c = T(0.0);
      st.u = T(0.0);
    }
  }
  const float floor_x = static_cast<float>(je - js) / static_cast<float>(kSeriesMinStep);
  k.set(SE_t, st.t);
  k.set(SE_f, st.f);
  k.set(SE_s, st.s);
  k.set(SE_q, T(0.0));
  const bool past = c.maxtaufrac > 1.0;
  // in samples from js, multiples of 2^-10 (exact): x0, up to where the
  // samples are done, and the expansion's centre x0 + d
  double x0 = 0.0, d = 0.0;
  int64_t j = js + 1;
  const double xe = static_cast<double>(je - js);
  while (j < pe) {
    Series<T, P, SIG> S;
    k.fresh();
    float x = series_expand<T, P, SIG>(c, k, st, S);
    if (!(x >= floor_x)) {  // also NaN
      if (live) {
        const int64_t from = j < ps ? ps : j, queued = js + static_cast<int64_t>(val(k(SE_q)));
        push_windows(push, i, from < queued ? queued : from, pe, true);
      }
      live = false;
    }
    x = live ? (x < 1.0e29f ? x : 1.0e29f) : 1.0e30f;  // all coefficients 0: no bound
    x = wave_min(x);
    if (x == 1.0e30f) break;  // no lane is left
    if (static_cast<double>(x) < d) {
      // it does not reach back to x0: centre it nearer
      d = kfloor(static_cast<double>(kSeriesAhead * x) * 1024.0) * (1.0 / 1024.0);
      series_advance<T>(k, T(d), st);
      continue;
    }
    series_match<T, P, SIG>(k, S, T(-d), k(SE_t), k(SE_f), k(SE_s), far);
    const double xc = x0 + d;
    double x1 = xc + static_cast<double>(x);
    if (x1 > xe) x1 = xe;
    x1 = kfloor(x1 * 1024.0) * (1.0 / 1024.0);
    const int64_t jn = js + static_cast<int64_t>(kfloor(x1)) + 1;  // the first sample after the step
    const int64_t jm = jn < pe ? jn : pe;
    if (j < ps) j = ps < jm ? ps : jm;
    double xj = static_cast<double>(j - js) - xc;
    for (; j < jm; ++j) {
      SeriesState<T> s;
      T r, an;
      k.fresh();
      series_at<T, P, SIG, false>(k, S, T(xj), s, r, an);
      xj += 1.0;
      const T th = acos_fast(s.c);
      if (live) {
        const int64_t idx = j * o.npix + i;
        if (o.tau_out) o.tau_out[idx] = mino_tau(j, o.ngeo, stop, false);
        if (o.th) o.th[idx] = val(th);
        if (o.r) o.r[idx] = val(r);
        o.t[idx] = val(-s.t);
        o.ph[idx] = val(-s.f);
        if (SIG) o.sig[idx] = val(-s.s);
        // a sample at a pole that the closed forms take out (0 times infinity) or,
        // of rays followed past their end, next to the horizon, where only the
        // direct formulas reproduce the reference's rounding: to the fixup
        // pass, with the rest of its window
        // (t has the same terms as r and phi)
        const bool odd = !(kfabs(val(r)) + kfabs(val(th)) + kfabs(val(s.f)) < INFINITY) ||
                         (past && kfabs(val(r) - val(c.rplus)) < kSeriesHorizon);
        if (odd && j - js >= static_cast<int64_t>(val(k(SE_q)))) {
          push(i, j, true);
          k.set(SE_q, T(static_cast<double>(series_fixup_end(j, o.ngeo, true, false) - js)));
        }
      }
    }
    if (j >= pe) break;
    {
      SeriesState<T> e;
      T r, an;
      series_at<T, P, SIG, true>(k, S, T(x1 - xc), e, r, an);
      // past the end of the ray the state may be handed on next to the horizon
      // or on the way through infinity, where the closed forms' terms have lost
      // the integrals' digits (an error of w by 1e-15 is one of r by 1e-15 r^2):
      // the rest is refused
      const bool lost = past && (kfabs(val(r) - val(c.rplus)) < kSeriesHorizon ||
                                 (val(e.v) < 0.0 && kfabs(val(r)) > kSeriesFar * c.r_o));
      k.set(SE_w, lost ? T(NAN) : e.w);
      k.set(SE_v, e.v);
      k.set(SE_c, e.c);
      k.set(SE_u, e.u);
      k.set(SE_t, e.t);
      k.set(SE_f, e.f);
      if (SIG) k.set(SE_s, e.s);
    }
    x0 = x1;
    d = static_cast<double>(kSeriesAhead * x);
    if (d > 0.5 * (xe - x0)) d = 0.5 * (xe - x0);
    d = kfloor(d * 1024.0) * (1.0 / 1024.0);
    series_advance<T>(k, T(d), st);
  }
  return bad ? ST_NONFINITE : 0u;
}

}  // namespace kg
