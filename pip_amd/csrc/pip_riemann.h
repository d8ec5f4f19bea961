// pip_riemann.h -- the face states and fluxes of pip_phys.h for bounded
// states, with fewer operations and the same results.
//
// "Bounded" means that every cell of the tile has density and pressure in
// (2^-100, 2^100) and the other variables below 2^100 in magnitude (no NaN,
// no infinity): stage_tile checks it once per cell while it loads the tile.
// Face states lie between cell values, so no intermediate of these functions
// overflows, no divisor is subnormal, and values equal those of the general
// function; the sign of a zero may differ (the median of slopes, and the normal
// field and the blends without the general form's terms in +0).  No later
// operation tells such zeros apart: none is divided by, and the one copysign,
// of the normal field, is reached only where that is not zero.  Where a function cannot
// vouch for that (a divisor that came out zero or infinite, an outer wave of
// HLLC's inside its switch band) it says so and the caller takes the general
// function for that face.  The stage kernels are bound by FP64 VALU issue (4 cycles a wave
// instruction, 16 for v_rcp_f64 and v_rsq_f64), so every identity below is
// one that removes instructions without changing a value:
//   - a product with a power of two is exact above the subnormal numbers, so
//     k x + y is one fma where the product is not subnormal or is added to a
//     pressure or energy (at least 2^-100, which no subnormal changes);
//   - max and the rounded square root commute (both are monotonic);
//   - finite non-zero divisors need no v_div_fixup_f64, positive arguments
//     no zero / infinity test in the square root;
//   - min(max(X, Y), 0) and min(X, Y) give minmod(X, Y) as a median;
//   - HLLC's switches |S| + S over max(2 S, eps) are exactly 0 or 1 outside
//     (0, eps / 2), so one side's flux and star state are enough there;
//   - 1 / sqrt(x) comes from the square root's own iteration.
#pragma once

#include "pip_phys.h"

namespace PIP_NS {

#if defined(__HIP_DEVICE_COMPILE__)
#if PIP_RELAXED
__device__ __forceinline__ double quob(double n, double, double r) { return n * r; }
#else
// n / d for finite n and finite non-zero d, r = qrcp(d): quo without the
// fixup of zero, infinite and NaN operands.
__device__ __forceinline__ double quob(double n, double d, double r) {
  const double q = n * r;
  return __builtin_fma(r, __builtin_fma(-d, q, n), q);
}
#endif
// sqrt(x) for positive finite x: qsqrt without its zero / infinity test;
// sqrt_rcp also gives a reciprocal of the root: h = 1 / (2 sqrt x) of the
// iteration is good to about 2^-47 (v_rsq_f64's 2^-24, squared by the step), so
// one Newton step replaces v_rcp_f64 and its two.  pip_check_arith_bounded runs
// these sequences beside the IEEE quotient and root.
__device__ __forceinline__ double sqrtb_h(double x, double& h) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y;
  h = y * 0.5;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}
__device__ __forceinline__ double sqrtb(double x) {
  double h;
  return sqrtb_h(x, h);
}
__device__ __forceinline__ double sqrt_rcp(double x, double& r) {
  double h;
  const double g = sqrtb_h(x, h);
  const double r0 = h + h;
  r = __builtin_fma(r0, __builtin_fma(-g, r0, 1.0), r0);
  return g;
}
#else
PIP_HD double quob(double n, double d, double) { return n / d; }
PIP_HD double sqrtb(double x) { return sqrt(x); }
PIP_HD double sqrt_rcp(double x, double& r) {
  r = 0.0;
  return sqrt(x);
}
#endif
PIP_HD double qdivb(double n, double d) { return quob(n, d, qrcp(d)); }

// minmod of the two one-sided differences: the median of X, Y and 0.
PIP_HD double minmod_med(double X, double Y) { return dmax(dmin(X, Y), dmin(dmax(X, Y), 0.0)); }

// The face states of get_Side (HLL_rot.f90:33-51) from the stencil a0..a3.
// POS: of a bounded tile's density or pressure, where half a slope is exact.
// Velocities and fields may be subnormal (ahead of a front), and half a
// subnormal slope rounds: one fma there put 1-D states 1e-323 off what the
// general face states give (its products cost a step 0.2 to 1 %).
template <bool POS = false>
PIP_HD void face_states(double a0, double a1, double a2, double a3, double& vl, double& vr) {
  const double d0 = a1 - a0, d1 = a2 - a1, d2 = a3 - a2;
  const double ml = minmod_med(d1, d0), mr = minmod_med(d2, d1);
  vl = POS ? fma2(0.5, ml, a1) : a1 + 0.5 * ml;
  vr = POS ? fma2(-0.5, mr, a2) : a2 - 0.5 * mr;
}

// Any active lane of the wave (host: this call).
PIP_HD bool wave_any(bool c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_ballot_w64(c) != 0ull;
#else
  return c;
#endif
}

// What a cell adds to the tile's check of boundedness: a sum of magnitudes
// (an infinity or NaN stays one) and the smaller of density and pressure.
constexpr double kBndHi = 1.2676506002282294e30;   // 2^100
constexpr double kBndLo = 7.8886090522101181e-31;  // 2^-100
PIP_HD bool bounded_cell(const double* v, int nv) {
  double s = fabs(v[0]);
  for (int n = 1; n < nv; n++) s = s + fabs(v[n]);
  return s < kBndHi && v[0] > kBndLo && v[4] > kBndLo;
}

// hllc_flux for bounded states, handed out as put(n, flux); false: not
// covered (take hllc_flux).  rg1 = 1 / (gm - 1).  Near rest, half of the
// contact speeds lie in (0, eps / 2), where the switch is a fraction and both
// star states count: such a wave forms its fluxes once for either side and
// blends them.  us per step with those faces left to the general function,
// which solves them again, with the blend, and with the general function
// alone, velocities up to 1e-13: 96 tubes 38.9 / 35.3 / 35.4, 300^2 47.4 / 43.2 /
// 56.0, 1024^2 326 / 290 / 355.  One loop for both kinds of wave cost moving
// flows 1.4 %.
template <class Put>
PIP_HD bool hllc_flux_b(const double* v_l, const double* v_r, double gm, double rg1, Put put) {
  const double ml = v_l[0] * v_l[1], mr = v_r[0] * v_r[1];
  const double ra = qrcp(v_l[0]), rb = qrcp(v_r[0]);
  const double cs_l = sqrtb(quob(gm * v_l[4], v_l[0], ra));
  const double cs_r = sqrtb(quob(gm * v_r[4], v_r[0], rb));
  const double vn_l = quob(ml, v_l[0], ra);
  const double vn_r = quob(mr, v_r[0], rb);
  const double sl = kAcc * dmin(vn_l - cs_l, vn_r - cs_r);
  const double sr = kAcc * dmax(vn_l + cs_l, vn_r + cs_r);
  const double al = sl - vn_l, ar = sr - vn_r;
  const double den = v_r[0] * ar - v_l[0] * al;
  const double sm = quob(mr * ar - ml * al + v_l[4] - v_r[4], den, qrcp(den));
  const double dl = sl - sm, dr = sr - sm;
  // thl, thr exactly 0 or 1, and neither star state divides by zero or
  // infinity (den passes through zero in supersonic flow)
  const double hb = 0.5 * kEpsi, dd = fabs(dl * dr);
  const bool ok = (sl <= 0.0 || sl >= hb) && (sr <= 0.0 || sr >= hb) && dd > 0.0 && dd < HUGE_VAL;
  if (!ok) return false;
  const double pr_m = sm * v_l[0] * al - ml * al + v_l[4];
  // the side whose states the flux is made of: left of the contact or, in a
  // supersonic flow (thl = 1, or thr = 1: that side's own flux), upstream
  const bool upl = sl > 0.0, upr = sr <= 0.0;
  auto side = [&](bool left, auto out) {
    const double r0 = left ? v_l[0] : v_r[0], r1 = left ? v_l[1] : v_r[1];
    const double r2 = left ? v_l[2] : v_r[2], r3 = left ? v_l[3] : v_r[3];
    const double pr = left ? v_l[4] : v_r[4], ri = left ? ra : rb;
    const double vn = left ? vn_l : vn_r, d = left ? dl : dr, as = left ? al : ar;
    double s = left ? sl : sr;
    const double m1 = r0 * r1, m2 = r0 * r2, m3 = r0 * r3;
    const double en = fma2(0.5, r0 * ((r1 * r1 + r2 * r2) + r3 * r3), quob(pr, gm - 1.0, rg1));
    const double rd = qrcp(d);
    const double st0 = quob(r0 * as, d, rd);
    const double st1 = st0 * sm;
    const double st2 = quob(st0 * m2, r0, ri);
    const double st3 = quob(st0 * m3, r0, ri);
    const double st4 = quob(as * en - pr * vn + pr_m * sm, d, rd);
    if (upl || upr) s = 0.0;
    out(0, m1 + s * (st0 - r0));
    out(1, (pr + quob(m1 * m1, r0, ri)) + s * (st1 - m1));
    out(2, quob(m1 * m2, r0, ri) + s * (st2 - m2));
    out(3, quob(m1 * m3, r0, ri) + s * (st3 - m3));
    out(4, quob(m1 * (en + pr), r0, ri) + s * (st4 - en));
  };
  const bool one = upl || (sm > 0.0 && !upr);
  const bool both = sm > 0.0 && sm < hb && !upl && !upr;  // thm is a fraction
  if (!wave_any(both)) {
    side(one, put);
    return true;
  }
  // the right side's flux first, then the left one's
  const double thm = both ? qdiv(sm + sm, kEpsi) : 1.0;
  double f_r[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
  for (int pass = 0; pass < 2; pass++) {
    double f[5];
    side(both ? pass == 1 : one, [&](int n, double x) { f[n] = x; });
    for (int n = 0; n < 5; n++) {
      if (pass == 0) f_r[n] = f[n];
      else put(n, thm * f[n] + (1.0 - thm) * f_r[n]);
    }
  }
  return true;
}

// What the wave speeds need of one side: normal momentum, its flux, energy,
// total pressure, v.B and the fast speed's square.
struct HlldSide {
  double m1, f1, en, pt, vb, cf2;
};
PIP_HD HlldSide hlld_side(const double* v, double gm, double rg1) {
  HlldSide s;
  const double b5 = v[5] * v[5], q1 = v[1] * v[1];
  const double b2 = (b5 + v[6] * v[6]) + v[7] * v[7];
  s.m1 = v[0] * v[1];
  s.en = fma2(0.5, b2, fma2(0.5, v[0] * ((q1 + v[2] * v[2]) + v[3] * v[3]), quob(v[4], gm - 1.0, rg1)));
  s.pt = fma2(0.5, b2, v[4]);
  s.vb = (v[1] * v[5] + v[2] * v[6]) + v[3] * v[7];
  s.f1 = fma2(0.5, b2, v[0] * q1 + v[4]) - b5;
  const double a = gm * v[4], ab = a + b2;
  // 2^-600 instead of 0: its root is lost in ab (> 2^-101)
  const double q = sqrtb(dmax(fma2(-4.0, a * b5, ab * ab), 2.409919865102884e-181));
  s.cf2 = qdivb(ab + q, 2.0 * v[0]);
  return s;
}
// The other components of a side: conserved m2, m3 and fluxes f2, f3, f4,
// f6, f7, formed where they are used (most faces use one side's).
struct HlldRest {
  double m2, m3, f2, f3, f4, f6, f7;
};
PIP_HD HlldRest hlld_rest(const double* v, const HlldSide& s) {
  return HlldRest{v[0] * v[2],
                  v[0] * v[3],
                  s.m1 * v[2] - v[5] * v[6],
                  s.m1 * v[3] - v[5] * v[7],
                  (s.en + s.pt) * v[1] - s.vb * v[5],
                  v[1] * v[6] - v[5] * v[2],
                  v[1] * v[7] - v[5] * v[3]};
}

// hlld_flux for bounded states, handed out as put(n, flux) (the caller's
// stores, so that no branch carries its results in registers to the end);
// false: not covered (take hlld_flux).  The wave speeds and the test for the
// central states run straight through for every face, so that the two sides'
// dependent chains overlap; every other region shares one branch.
template <int NV, class Put>
PIP_HD bool hlld_flux_b(const double* v_l, const double* v_r, double gm, double rg1, double cmax, Put put) {
  if (NV == 9) {
    put(5, 0.5 * ((v_l[NV - 1] + v_r[NV - 1]) - cmax * (v_r[5] - v_l[5])));
    put(NV - 1, 0.5 * (cmax * cmax * (v_l[5] + v_r[5]) - cmax * (v_r[NV - 1] - v_l[NV - 1])));
  }
  const HlldSide L = hlld_side(v_l, gm, rg1), R = hlld_side(v_r, gm, rg1);
  const double cf = sqrtb(dmax(L.cf2, R.cf2));
  const double sl = dmin(v_l[1], v_r[1]) - cf, sr = dmax(v_l[1], v_r[1]) + cf;
  const double fh = qdivb(1.0, sr - sl);
  auto hll = [&](double ul, double ur, double fl, double fr) { return fh * (((sr * ur - sl * ul) - fr) + fl); };
  const double ro_h = hll(v_l[0], v_r[0], L.m1, R.m1);
  const double m1_h = hll(L.m1, R.m1, L.f1, R.f1);
  const double bx = fh * (sr * v_r[5] - sl * v_l[5]);
  const double rh = qrcp(ro_h);
  const double sm = quob(m1_h, ro_h, rh);
  const double al = sl - v_l[1], ar = sr - v_r[1], dl = sl - sm, dr = sr - sm;
  const double ql = v_l[0] * al, qr = v_r[0] * ar;
  const double pt = L.pt + ql * (sm - v_l[1]);
  const double rdl = qrcp(dl), rdr = qrcp(dr);
  const double ro_l = quob(ql, dl, rdl), ro_r = quob(qr, dr, rdr);
  double rsl, rsr;
  const double ros_l = sqrt_rcp(ro_l, rsl), ros_r = sqrt_rcp(ro_r, rsr);
  const double sal = quob(fabs(bx), ros_l, rsl), sar = quob(fabs(bx), ros_r, rsr);
  const double sl1 = sm - sal, sr1 = sm + sar;
  const double ptm = pt * sm, bsm = sm * bx;
  // energy of a star state
  auto star_en = [&](const double* v, const HlldSide& S, double a, double d, double rd, double vy, double vz,
                     double by, double bz) {
    return quob(((a * S.en - S.pt * v[1]) + ptm) + bx * (((S.vb - bsm) - vy * by) - vz * bz), d, rd);
  };
  // HLLD intermediate states :810-843
  const double bh2 = bx * bx;
  struct Star {
    double by, bz, vy, vz;
  };
  auto star = [&](const double* v, double a, double q, double d) {
    const double f = qdivb(1.0, q * d - bh2), g = v[0] * (a * a) - bh2, fb = f * bx, c = sm - v[1];
    return Star{v[6] * f * g, v[7] * f * g, v[2] - fb * v[6] * c, v[3] - fb * v[7] * c};
  };
  // A side's part: taken by the wave where its lanes agree on the side, by
  // selects where they do not (two a value: 44 for the central states).
  auto by_side = [&](bool left, auto on_l, auto on_r, auto on_sel) {
    if (!wave_any(!left)) {
      on_l();
    } else if (!wave_any(left)) {
      on_r();
    } else {
      auto sel = [&](double x, double y) { return left ? x : y; };
      double v[8];
#pragma unroll
      for (int n = 0; n < 8; n++) v[n] = (n == 4) ? 0.0 : sel(v_l[n], v_r[n]);
      const HlldSide S = {sel(L.m1, R.m1), sel(L.f1, R.f1), sel(L.en, R.en), sel(L.pt, R.pt), sel(L.vb, R.vb), 0.0};
      on_sel(sel, v, S);
    }
  };
  // subsonic, positive star densities (so no divisor above or below is
  // zero), not HLLC-G's, and the contact between the two Alfven waves
  const bool subsonic = sl < 0.0 & sr > 0.0;
  const bool positive = ro_l > 0.0 & ro_r > 0.0;
  const bool stars = sl < sm - kHllg * sal & sm + kHllg * sar < sr;
  if (subsonic & positive & stars & sl1 < 0.0 & sr1 > 0.0) {
    // central states :861-898
    const Star l = star(v_l, al, ql, dl), r = star(v_r, ar, qr, dr);
    const double f1 = qdivb(1.0, ros_l + ros_r);
    const double f2 = copysign(1.0, bx);
    const double ww = ros_l * ros_r;
    const double vy = f1 * ((ros_l * l.vy + ros_r * r.vy) + (r.by - l.by) * f2);
    const double vz = f1 * ((ros_l * l.vz + ros_r * r.vz) + (r.bz - l.bz) * f2);
    const double by = f1 * ((ros_l * r.by + ros_r * l.by) + ww * (r.vy - l.vy) * f2);
    const double bz = f1 * ((ros_l * r.bz + ros_r * l.bz) + ww * (r.vz - l.vz) * f2);
    auto central = [&](const double* v, const HlldSide& S, const Star& t, double s, double s1, double a, double d,
                       double rd, double ro, double w) {
      const double ds = s1 - s;
      const double en1 = star_en(v, S, a, d, rd, t.vy, t.vz, t.by, t.bz);
      const double en2 = en1 + (w * (((t.vy * t.by + t.vz * t.bz) - vy * by) - vz * bz)) * f2;
      const HlldRest c = hlld_rest(v, S);
      const double m1s = ro * sm;
      auto out = [&](double u2, double us, double u) { return (s1 * u2 - ds * us) - s * u; };
      put(0, out(ro, ro, v[0]) + S.m1);
      put(1, out(m1s, m1s, S.m1) + S.f1);
      put(2, out(ro * vy, ro * t.vy, c.m2) + c.f2);
      put(3, out(ro * vz, ro * t.vz, c.m3) + c.f3);
      put(4, out(en2, en1, S.en) + c.f4);
      if (NV == 8) put(5, out(bx, bx, v[5]));
      put(6, out(by, t.by, v[6]) + c.f6);
      put(7, out(bz, t.bz, v[7]) + c.f7);
    };
    by_side(sm >= 0.0, [&] { central(v_l, L, l, sl, sl1, al, dl, rdl, ro_l, -ros_l); },
            [&] { central(v_r, R, r, sr, sr1, ar, dr, rdr, ro_r, ros_r); },
            [&](auto sel, const double* v, const HlldSide& S) {
              const Star t = {sel(l.by, r.by), sel(l.bz, r.bz), sel(l.vy, r.vy), sel(l.vz, r.vz)};
              central(v, S, t, sel(sl, sr), sel(sl1, sr1), sel(al, ar), sel(dl, dr), sel(rdl, rdr), sel(ro_l, ro_r),
                      sel(-ros_l, ros_r));
            });
    return true;
  }
  if (sl >= 0.0 || sr <= 0.0) {  // supersonic: the upstream side's flux
    auto up = [&](const double* v, const HlldSide& S) {
      const HlldRest c = hlld_rest(v, S);
      put(0, S.m1);
      put(1, S.f1);
      put(2, c.f2);
      put(3, c.f3);
      put(4, c.f4);
      if (NV == 8) put(5, 0.0);
      put(6, c.f6);
      put(7, c.f7);
    };
    if (sl >= 0.0) up(v_l, L);
    else up(v_r, R);
    return true;
  }
  if (!positive) return false;
  // one star state between the outer wave and the contact: HLLD's where both
  // Alfven waves lie on one side of the face, or HLLC-G's (:775-807)
  Star g = {0.0, 0.0, 0.0, 0.0};
  if (!stars) {
    const HlldRest cl = hlld_rest(v_l, L), cr = hlld_rest(v_r, R);
    g.by = hll(v_l[6], v_r[6], cl.f6, cr.f6);
    g.bz = hll(v_l[7], v_r[7], cl.f7, cr.f7);
    g.vy = quob(hll(cl.m2, cr.m2, cl.f2, cr.f2), ro_h, rh);
    g.vz = quob(hll(cl.m3, cr.m3, cl.f3, cr.f3), ro_h, rh);
  }
  auto one = [&](const double* v, const HlldSide& S, double s, double a, double q, double d, double rd, double ro) {
    const Star t = stars ? star(v, a, q, d) : g;
    const HlldRest c = hlld_rest(v, S);
    put(0, s * (ro - v[0]) + S.m1);
    put(1, s * (ro * sm - S.m1) + S.f1);
    put(2, s * (ro * t.vy - c.m2) + c.f2);
    put(3, s * (ro * t.vz - c.m3) + c.f3);
    put(4, s * (star_en(v, S, a, d, rd, t.vy, t.vz, t.by, t.bz) - S.en) + c.f4);
    if (NV == 8) put(5, s * (bx - v[5]));
    put(6, s * (t.by - v[6]) + c.f6);
    put(7, s * (t.bz - v[7]) + c.f7);
  };
  by_side(stars ? sl1 >= 0.0 : sm >= 0.0, [&] { one(v_l, L, sl, al, ql, dl, rdl, ro_l); },
          [&] { one(v_r, R, sr, ar, qr, dr, rdr, ro_r); },
          [&](auto sel, const double* v, const HlldSide& S) {
            one(v, S, sel(sl, sr), sel(al, ar), sel(ql, qr), sel(dl, dr), sel(rdl, rdr), sel(ro_l, ro_r));
          });
  return true;
}

}  // namespace PIP_NS
