// Per-point pieces of the SSB overlap shared by the object path and the
// exact per-BF loss path: the factorised Gamma (see ssb_device.h), the
// isotropic double-float aperture and the quadratic chi.
#pragma once

#include "ssb_internal.h"

namespace qssb {

// Balanced split of [0, nbf) into `groups` contiguous ranges.
__device__ __forceinline__ void group_range(int g, int groups, int nbf, int& b0, int& b1) {
  b0 = (int)(((long long)g * nbf) / groups);
  b1 = (int)(((long long)(g + 1) * nbf) / groups);
}

__device__ __forceinline__ float chi_quad(const QuadChi& m, float x, float y) {
  return m.mxx * x * x + 2.0f * m.mxy * x * y + m.myy * y * y;
}

// Aperture from d = Rout^2 - |u|^2 (double-float), where Rout is the radius
// at which the soft edge reaches 0.  For isotropic detector sampling the
// reference edge (semi - lambda|u|)/ang + 1/2 equals (Rout - |u|)*lambda/ang
// = d * (lambda/ang) / (Rout + |u|): the cancellation sits entirely in d,
// which is exact to ~1e-13 here, so ties (d == 0, A(Q-k) == A(Q+k)) resolve
// as exact arithmetic resolves them.
__device__ __forceinline__ float aperture_from_d(df d, const ApIso& a) {
  const float dh = d.hi + d.lo;
  if (dh >= a.d_in) return 1.0f;
  if (dh <= a.d_out) return 0.0f;
  const float r = sqrtf(fmaxf(a.rout2 - dh, 0.0f));
  const float e = dh * a.scale / (a.rout + r);
  return fminf(fmaxf(e, 0.0f), 1.0f);
}

// The aperture from a float32 estimate of d when it lies beyond the 1e-4
// margin of the soft band (exactly 0 or 1 there: the estimate is within a few
// 1e-6 of d for terms below 32 in magnitude); false when it is too close to the
// band to decide.
__device__ __forceinline__ bool aperture_decided(float est, const ApIso& ap, float& a) {
  constexpr float kMargin = 1e-4f;
  a = (est >= ap.d_in + kMargin) ? 1.0f : 0.0f;
  return est >= ap.d_in + kMargin || est <= ap.d_out - kMargin;
}

// The value unchanged, through an empty volatile asm: an expression built on
// it cannot be hoisted out of the branch that holds it.
__device__ __forceinline__ df df_in_branch(df x) {
  asm volatile("" : "+v"(x.hi), "+v"(x.lo));
  return x;
}

// Float32 estimates of the isotropic row terms of d(Q -/+ k),
// -qx^2 + 2 qx kx and -qx^2 - 2 qx kx (kx2 = 2 kx): within ~1e-5 of the
// double-float values for terms below 32 in magnitude, well inside the 1e-4
// margin that aperture_decided leaves.
__device__ __forceinline__ float row_estimate_minus(df qx, df kx2, df q2x) { return fmaf(qx.hi, kx2.hi, -q2x.hi); }
__device__ __forceinline__ float row_estimate_plus(df qx, df kx2, df q2x) { return -fmaf(qx.hi, kx2.hi, q2x.hi); }

// Isotropic aperture pair A(Q - k), A(Q + k) from d = row + col: decided
// from the estimates uq, vq of the row terms wherever d lies beyond the soft
// band's margin, otherwise from the double-float row terms, which are formed
// inside that branch only -- the few points near the soft edge pay for them,
// the rest do not.
__device__ __forceinline__ void iso_aperture_pair(float uq, float vq, df qx, df kx2, df q2x, const df& colA,
                                                  const df& colB, const ApIso& ap, float& am, float& app) {
  const bool da = aperture_decided(uq + colA.hi, ap, am);
  const bool dp = aperture_decided(vq + colB.hi, ap, app);
  if (!(da && dp)) {
    const df u = df_mul(df_in_branch(qx), kx2);
    if (!da) am = aperture_from_d(df_add(df_sub(u, q2x), colA), ap);
    if (!dp) app = aperture_from_d(df_add(df_neg(df_add(q2x, u)), colB), ap);
  }
}

// Aperture pair A(Q - k), A(Q + k).  ISO: from d = (Rout^2 - |k|^2) - |Q|^2
// +/- 2 Q.k; otherwise the general double-float soft-edge expression.
template <bool ISO>
__device__ __forceinline__ void aperture_pair(df qx, df qy, df kx, df ky, df cb, df q2, const ApIso& ap,
                                              const Optics& o, float& am, float& app) {
  if constexpr (ISO) {
    const df qk2 = df_mul(df_add(df_mul(qx, kx), df_mul(qy, ky)), df{2.0f, 0.0f});
    const df base = df_sub(cb, q2);
    am = aperture_from_d(df_add(base, qk2), ap);
    app = aperture_from_d(df_sub(base, qk2), ap);
  } else {
    am = aperture_at<false>(qx.hi, qx.lo, qy.hi, qy.lo, kx.hi, kx.lo, ky.hi, ky.lo, o);
    app = aperture_at<true>(qx.hi, qx.lo, qy.hi, qy.lo, kx.hi, kx.lo, ky.hi, ky.lo, o);
  }
}


// Normalised overlap Gamma^ = Gamma / |Gamma| of one (b, Q) from its
// factorised parts, Gamma = A(k) e^{i theta} [A(Q-k) e^{-i chi(Q)} - A(Q+k) e^{i chi(Q)}],
// with the guard |Gamma|^2 > 1e-16 ? rsqrt : 1e8 (cuda/kernels/common.py:227-230).
__device__ __forceinline__ float2 gamma_hat(float ak, float2 eth, float am, float app, float2 echi) {
  const float wr = (am - app) * echi.x;
  const float wi = -(am + app) * echi.y;
  float gr = ak * (eth.x * wr - eth.y * wi);
  float gi = ak * (eth.x * wi + eth.y * wr);
  const float mag2 = gr * gr + gi * gi;
  const float sc = (mag2 > 1e-16f) ? rsqrtf(mag2) : 1e8f;
  return make_float2(gr * sc, gi * sc);
}

// G * conj(g)
__device__ __forceinline__ float2 mul_conj(float2 G, float2 g) {
  return make_float2(G.x * g.x + G.y * g.y, G.y * g.x - G.x * g.y);
}

// sin(pi r) and cos(pi r) for |r| <= 1/2: minimax polynomials in r^2 (fitted
// for these functions by iteratively reweighted least squares; 5.3e-9 and
// 2.4e-10 before rounding, 1.6e-7 and 1.1e-7 evaluated in float32).
__device__ __forceinline__ void sincos_half_turns(float r, float& s, float& c) {
  const float u = r * r;
  float p = fmaf(0.07756020873785019f, u, -0.5982420444488525f);
  p = fmaf(p, u, 2.550069808959961f);
  p = fmaf(p, u, -5.167709827423096f);
  p = fmaf(p, u, 3.1415927410125732f);
  s = r * p;
  float q = fmaf(-0.024420656263828278f, u, 0.2349538952112198f);
  q = fmaf(q, u, -1.3352160453796387f);
  q = fmaf(q, u, 4.058709621429443f);
  q = fmaf(q, u, -4.934802055358887f);
  c = fmaf(q, u, 1.0f);
}

// Gamma^ from half the sum and half the difference of the two phases, in
// half turns: with s = (dp + dm) / 2pi, t = (dp - dm) / 2pi (dm, dp as in
// gamma_hat_chi below), Gamma = A(k) e^{i pi t} [A(Q-k) e^{-i pi s} - A(Q+k) e^{i pi s}].
// Outside the soft band one phasor is left: e^{i pi (t - s)} with A(Q-k)
// alone, -e^{i pi (t + s)} with A(Q+k) alone, and with both
// -2i sin(pi s) e^{i pi t}, whose normalised value is -i sign(sin(pi s)) e^{i pi t},
// sign = parity of floor(s).  For an even chi, t is odd and s even in k, so
// exchanging k and -k turns Gamma^ into -conj(Gamma^): one form, on the side
// where A(Q-k) is the larger, serves all.  Returns G * conj(Gamma^): `both`
// apertures 1 or A(Q-k) alone for `t` taken on that side, `flip` (a sign
// bit): the other side is meant.  It is normalised without the guard of
// gamma_hat, so the caller takes the points where Gamma can be that small
// through gamma_hat_st.
__device__ __forceinline__ float2 overlap_unit(float2 G, bool both, float s, float t, unsigned flip) {
  // (contracted, t's last product would round here by where this is inlined)
#pragma clang fp contract(off)
  const float a = t + (both ? -0.5f : -s);
  const float n = rintf(a);
  float sn, cs;
  sincos_half_turns(a - n, sn, cs);
  const unsigned turn = (unsigned)(int)(n + (both ? floorf(s) : 0.0f)) << 31;
  cs = __uint_as_float(__float_as_uint(cs) ^ flip);
  const float x = fmaf(G.x, cs, G.y * sn), y = fmaf(G.y, cs, -(G.x * sn));
  return make_float2(__uint_as_float(__float_as_uint(x) ^ turn), __uint_as_float(__float_as_uint(y) ^ turn));
}

// a + b, a not contracted into it: the C12 term m12c (qx - qy) (qx + qy) of s
// cancels a C10 term of its size to zero on an axis, and is zero on the diagonals.
// What rounding would leave has a sign, which overlap_unit would take.
__device__ __forceinline__ float add_cancelling(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}

// The general form of the same, with the guard of gamma_hat.
__device__ __forceinline__ float2 gamma_hat_st(float ak, float am, float app, float s, float t) {
  if (am == 0.0f && app == 0.0f) return make_float2(0.0f, 0.0f);
  auto turn = [](float x, float& sn, float& cs) {
    const float n = rintf(x);
    sincos_half_turns(x - n, sn, cs);
    const unsigned flip = (unsigned)(int)n << 31;
    sn = __uint_as_float(__float_as_uint(sn) ^ flip);
    cs = __uint_as_float(__float_as_uint(cs) ^ flip);
  };
  float ss, cc, st, ct;
  turn(s, ss, cc);
  turn(t, st, ct);
  const float wr = (am - app) * cc, wi = -(am + app) * ss;
  // contracted as written: the same bits wherever this is inlined
  const float gr = ak * fmaf(ct, wr, -(st * wi)), gi = ak * fmaf(ct, wi, st * wr);
  const float mag2 = fmaf(gr, gr, gi * gi);
  const float sc = (mag2 > 1e-16f) ? rsqrtf(mag2) : 1e8f;
  return make_float2(gr * sc, gi * sc);
}

// The term G * conj(Gamma^) of one point for an even chi.  near >= far: d =
// Rout^2 - |u|^2 of Q - k and Q + k, the larger first, as float32 estimates
// (an aperture is zero from d = 0 down and one from ap.d_in up); B: its sign
// says which of the two is the nearer (negative: Q + k); s, t as in
// overlap_unit, t on the nearer side.  One phasor serves where one aperture
// is zero, whatever the other's value (normalising takes it out), and where
// both are one; the general form at an outer edge and with the smaller aperture
// in its soft band, and wherever |Gamma| can meet the guard of gamma_hat, 1e-8:
// with both apertures one it is 2 A(k) |sin(pi s)|, at least 1.5e-7 for s further
// than kNearWhole from a whole number and A(k) from kSmallAk up (s is that near
// under no aberration, tiny ones, and on lines of the plane where C10 and C12
// cancel; next to 1 float32 itself is no finer than 6e-8).  A BF pixel of smaller
// A(k) goes there with all its points (margin = infinity).  whole: near_whole(s),
// if the caller cannot know that it isn't.  There both d
// come from exact(dn, df), to float32 of themselves: the float32 estimates, whose error grows
// with the terms and weighs by the width of the band, would give an aperture in its
// band to 1e-6 at 20 mrad and 1.25 mrad a pixel and to 1e-5 at 40 mrad and 0.25.
// They only say whether a point is within ap.edge of an edge, at least 1e-4 and
// 4e-6 Rout^2: they add up, for |Q| up to 2 Rout, to 2.5e-6 Rout^2.  B must not be a
// negative zero unless t is zero.
constexpr float kSmallAk = 1.2e-2f;
constexpr float kNearWhole = 2e-6f;
__device__ __forceinline__ bool near_whole(float s) { return fabsf(s - rintf(s)) <= kNearWhole; }
__device__ __forceinline__ float edge_margin(float ak, const ApIso& ap) { return ak < kSmallAk ? INFINITY : ap.edge; }

template <typename Exact>
__device__ __forceinline__ float2 overlap_term(float2 G, float near, float far, float B, float s, float t,
                                               bool whole, float margin, float ak, const ApIso& ap, Exact exact) {
  const float inner = ap.d_in + ap.edge;
  const bool both = far >= inner;
  const bool general = (fabsf(near) < margin) | ((far > -margin) & (far < inner)) | (both & whole);
  float2 z = overlap_unit(G, both, s, t, __float_as_uint(B) & 0x80000000u);
  if (general) {
    float dn = near, dfar = far;
    if (!both) {
      exact(dn, dfar);
      if (B < 0.0f) {
        const float x = dn;
        dn = dfar;
        dfar = x;
      }
    }
    float2 g = gamma_hat_st(ak, aperture_from_d(df{dn, 0.0f}, ap), aperture_from_d(df{dfar, 0.0f}, ap), s, t);
    if (B < 0.0f) g.x = -g.x;
    z = make_float2(fmaf(G.x, g.x, G.y * g.y), fmaf(G.y, g.x, -(G.x * g.y)));
  }
  return z;
}

// |q|^2 in double-float.
__device__ __forceinline__ df square_of(df x, df y) {
#pragma clang fp contract(off)
  const df xx = two_prod(x.hi, x.hi), yy = two_prod(y.hi, y.hi), q2 = two_sum(xx.hi, yy.hi);
  return df{q2.hi, q2.lo + (xx.lo + yy.lo) + 2.0f * (x.hi * x.lo + y.hi * y.lo)};
}

// d of Q - k and Q + k from double-float q, |q|^2, 2 k and Rout^2 - |k|^2, rounded once
// but for terms of 1e-14: the leading products and sums exactly, the rest in
// float32 (a third of the work of double-float throughout).  Equal where Q.k is
// zero.
__device__ __forceinline__ void exact_d(df x, df y, df q2, df kx2, df ky2, df cb, float& dm, float& dp) {
#pragma clang fp contract(off)
  const df xk = two_prod(x.hi, kx2.hi), yk = two_prod(y.hi, ky2.hi), qk2 = two_sum(xk.hi, yk.hi);
  const float qkl = qk2.lo + (xk.lo + yk.lo) + ((x.hi * kx2.lo + y.hi * ky2.lo) + (x.lo * kx2.hi + y.lo * ky2.hi));
  const df base = two_sum(cb.hi, -q2.hi);
  const float bl = base.lo + (cb.lo - q2.lo);
  dm = (base.hi + qk2.hi) + (bl + qkl);
  dp = (base.hi - qk2.hi) + (bl - qkl);
}

// What the terms of one BF pixel share under a quadratic chi: 2 k, Rout^2 -
// |k|^2, t as a linear form of q, the margin of overlap_term and A(k).  reach:
// |u|^2 up to which an aperture or its margin can be met (kReach above Rout^2).
struct QuadPixel {
  float kx2, ky2, cb, tx, ty, margin, ak;
  float kx2l, ky2l, cbl;   // low words, for exact_d
};
constexpr float kReachRel = 1.00002f, kReachAbs = 3e-4f;

__device__ __forceinline__ QuadPixel quad_pixel(const GeomPtrs& gp, int b, const QuadTurns& ev, df rout2,
                                                const ApIso& ap) {
  QuadPixel p;
  const df kx{gp.kx[b], gp.kxl[b]}, ky{gp.ky[b], gp.kyl[b]};
  p.kx2 = 2.0f * kx.hi;
  p.ky2 = 2.0f * ky.hi;
  p.kx2l = 2.0f * kx.lo;
  p.ky2l = 2.0f * ky.lo;
  const df cb = df_sub(rout2, df_add(df_mul(kx, kx), df_mul(ky, ky)));
  p.cb = cb.hi;
  p.cbl = cb.lo;
  p.tx = 2.0f * df_add(df_mul(ev.sxx, kx), df_mul(ev.sxy, ky)).hi;
  p.ty = 2.0f * df_add(df_mul(ev.syy, ky), df_mul(ev.sxy, kx)).hi;
  p.ak = gp.ak[b];
  p.margin = edge_margin(p.ak, ap);
  return p;
}

// Whether the apertures around k and -k can reach the frequencies
// [x0, x1] x [y0, y1].
__device__ __forceinline__ bool apertures_reach(const QuadPixel& p, float rout2, float x0, float x1, float y0,
                                                float y1) {
  const float kx = 0.5f * p.kx2, ky = 0.5f * p.ky2;
  const float ax = fmaxf(fmaxf(x0 - kx, kx - x1), 0.0f), ay = fmaxf(fmaxf(y0 - ky, ky - y1), 0.0f);
  const float bx = fmaxf(fmaxf(x0 + kx, -kx - x1), 0.0f), by = fmaxf(fmaxf(y0 + ky, -ky - y1), 0.0f);
  return p.ak != 0.0f && fminf(fmaf(ax, ax, ay * ay), fmaf(bx, bx, by * by)) < fmaf(rout2, kReachRel, kReachAbs);
}

// chi(u) split into its even part E and odd part O (ChiPoly).
__device__ __forceinline__ void chi_parts(const ChiPoly& cp, float ux, float uy, float& E, float& O) {
  const float r2 = ux * ux + uy * uy;
  float zr[7], zi[7];
  zr[0] = 1.0f;
  zi[0] = 0.0f;
#pragma unroll
  for (int m = 1; m < 7; ++m) {
    zr[m] = zr[m - 1] * ux - zi[m - 1] * uy;
    zi[m] = zr[m - 1] * uy + zi[m - 1] * ux;
  }
  const float r4 = r2 * r2, r6 = r4 * r2;
  auto t = [&](int i, int m) { return cp.ca[i] * zr[m] + cp.sa[i] * zi[m]; };
  E = cp.K[0] * r2 + cp.K[1] * t(1, 2) + cp.K[4] * r4 + cp.K[5] * r2 * t(5, 2) + cp.K[6] * t(6, 4) +
      cp.K[10] * r6 + cp.K[11] * r4 * t(11, 2) + cp.K[12] * r2 * t(12, 4) + cp.K[13] * t(13, 6);
  O = cp.K[2] * r2 * t(2, 1) + cp.K[3] * t(3, 3) + cp.K[7] * r4 * t(7, 1) + cp.K[8] * r2 * t(8, 3) +
      cp.K[9] * t(9, 5);
}

// Gamma^ from the phases: Gamma = A(k) [A(Q-k) e^{-i dm} - A(Q+k) e^{i dp}],
// dm = chi(Q-k) - chi(k), dp = chi(Q+k) - chi(k); same guard as gamma_hat.
__device__ __forceinline__ float2 gamma_hat_chi(float ak, float am, float app, float dm, float dp) {
  if (am == 0.0f && app == 0.0f) return make_float2(0.0f, 0.0f);
  float sm, cm, sp, cpp;
  sincosf(dm, &sm, &cm);
  sincosf(dp, &sp, &cpp);
  float gr = ak * (am * cm - app * cpp);
  float gi = ak * (-am * sm - app * sp);
  const float mag2 = gr * gr + gi * gi;
  const float sc = (mag2 > 1e-16f) ? rsqrtf(mag2) : 1e8f;
  return make_float2(gr * sc, gi * sc);
}

}  // namespace qssb
