// sarbp_poly.h -- row polynomials: the slant range over a wave's strip of pixels
// as a short polynomial in the pixel offsets, with the bounds that say where it
// holds.  Plain C++, so that the host tests check the setup that the kernels of
// sarbp_kernels.inc run.
#pragma once

#include <math.h>
#include <string.h>

#include "sarbp_internal.h"

#define SARBP_HD __host__ __device__ inline __attribute__((always_inline))

namespace sarbp {

SARBP_HD float float_of_bits(int v) {
  float f;
  memcpy(&f, &v, sizeof f);
  return f;
}

SARBP_HD float fract_of(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_fractf(v);
#else
  return v - floorf(v);
#endif
}

// 1 / sqrt(v) to 2^-23 or better.
SARBP_HD double rsqrt_estimate(double v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rsq(v);
#else
  return (double)(float)(1.0 / sqrt(v));
#endif
}

// 1 / v and sqrt(v) to an ulp (on the host: that ulp off), for bounds and first
// guesses.
SARBP_HD float rcp_estimate(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rcpf(v);
#else
  return nextafterf(1.0f / v, INFINITY);
#endif
}
SARBP_HD float sqrt_estimate(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_sqrtf(v);
#else
  return v > 0.0f ? nextafterf(sqrtf(v), INFINITY) : v;
#endif
}

// sqrt(v) in FP64: FP32's and two Newton steps, whose remainders (2^-23 and
// 2^-46 of the root) need FP32 only.  One step is good to 1e-8 m at 800 km,
// 4e-6 rad at X band.
SARBP_HD double range_root(double v) {
#pragma clang fp contract(off)
  const float s = sqrt_estimate((float)v), h = s > 0.0f ? 0.5f * rcp_estimate(s) : 0.0f;
  const double r = (double)s + (double)((float)fma(-(double)s, (double)s, v) * h);
  return r + (double)((float)fma(-r, r, v) * h);
}

template <int INTERP>
SARBP_HD constexpr double bin_scale() {
  return INTERP == kSinc8 ? 2.0 : 1.0;
}

// ---- row polynomials (SARBP_PREC_REF and _DF, linear and sinc8) -------------------------
//
// A wave's pixels of one pulse lie in a strip of 64 PX x PY pixels, over which
// the slant range is a short polynomial.  With the wave's centre pixel as the
// expansion point, x the (integer) column offset, y the row offset
// (half-integer), s = e.d, pp = |d|^2 - s^2 and g = 1 / (2 R0):
//   R - R0 = s + g pp - 2 g^2 s pp + g^3 (4 s^2 pp - pp^2) + O(d^5 / R0^4)
//          = s + sum c_ij x^i y^j,   2 <= i + j <= 4.
// One lane per (pulse, wave) computes the c_ij in FP64; a lane evaluates the
// terms in x once per pulse and the rows y = +-1/2, +-3/2 .. in pairs, so a
// pixel costs 3 FMA for its bin and phase together plus 13 / PY operations,
// where the expansion evaluated per pixel took 10 (order 2).  Terms of fourth
// and third order that are not kept whole are replaced by their best lower-
// order fit over the strip (x^3 -> 3/4 X^2 x and the like).
//   mode 0 keeps x^2 .. x^4, y x, y x^2, y^2, y^2 x;
//   mode 1 adds y x^3 and, in the phase, y^3;
//   mode 2 evaluates the exact two-step form per pixel, with its bin clamped.
// The setup takes the first mode whose dropped terms stay below kPolyTol of
// phase and kBinTol of a bin (mode 2 also where the window bound does not hold,
// as for antennas among the pixels or positions that are not numbers).  A
// polynomial's bins are not clamped: that bound and the bin of margin in a
// strip's positions keep them inside.
// 4096 x 4096 x 4096 pulses, 0.25 m, sinc8: 59 ms with the expansion per pixel
// (36.9 VALU instructions and 28.6 issue slots per pixel-pulse, 1 x 4 pixels
// per lane), 49.5-50.3 ms this way at 1 x 8 (30.1 and 23.8), bound by the VALU
// issue slots, 89% used, with the LDS pipe 66% busy beside them.
constexpr float kPolyTol[2] = {1.5e-6f, 5e-6f};  // rad, modes 0 and 1
// The bin has its own limit, which rules at low carriers and, against the
// phase's y^3, for rows that are long against dr: its y^3 is the best fit in y.
constexpr float kBinTol = 4e-6f;  // bins: a tenth of FP32's rounding of bin 500
// Record of a (pulse, wave), poly_rec16(PREC) float4:
// {c0, pa, A2, A3 | A4, pb, B1, B2 | C0, C1, bin0, alpha | beta, B3, D3, tag};
// phases in revolutions, ranges in bin units.  Mode 2: {c0, pa, 2 R0, last bin
// | g, pb, 2 g^2, - | first bin, -, bin0, alpha | beta, -, -, tag} with alpha and
// beta in m.  tag: the mode in bits 0-1, above them the byte offset of the
// position that the strip's bins count from, in the pulse's staged ones: the
// one below the centre's bin, so that FP32 rounds the bins at half their span
// (from the first position on, 1 m pixels with columns along range were up to
// 1.3 times further from the exact image than the double-float form).
//
// SARBP_PREC_DF takes the same expansion further (x^5, y x^3, y x^4, y^2 x^2,
// y^3) and evaluates the terms that reach many revolutions, pa x + a2 x^2, without
// rounding: pa and a2 are split into multiples of 1 / kCompGrid, whose products
// with the integers x and x^2 and their sum are exact in FP32 up to kCompExact
// revolutions and lose their whole ones exactly, and FP32 remainders.  The
// other terms are rounded and may reach kCompTurns revolutions.  The phase is
// then good to 5e-7 rad rms (1.3e-5 at most, 8e-6 of it left out), against
// 1.4e-6 rms of the double-float form per pixel.  Where a limit is passed, or
// without a bound, every pixel's range and phase are FP64 (mode 2).
// 1024 x 768 pixels of 1.6 m, 2048 pulses, sinc8: 6.95 ms per pixel in
// double-float, 3.9 by rows.
// Record: {c0, pa hi, pa lo, a2 hi | a2 lo, A2, A3, A4 | A5, pb, B1, B2 |
// B3, B4, C0, C1 | C2, D3, bin0, alpha | beta, -, -, tag}.  Mode 2: {antenna x, y
// (FP64) | z, range of the counted-from position (FP64) | .. | first bin, last
// bin, -, tag}.
constexpr float kCompTol = 8e-6f;  // rad, a bound: at it the error is ~1.2e-6 rms
constexpr double kCompGrid = 16384.0;
constexpr float kCompExact = 1000.0f;  // revolutions: below 2^24 / kCompGrid
constexpr float kCompTurns = 4.0f;

// Largest bin (the interpolator's unit) of n staged positions or samples.
template <int INTERP>
SARBP_HD constexpr int bin_last(int n) {
  return INTERP == kSinc8 ? 2 * n - 1 : (INTERP == kSinc8W ? n - 1 : n - 2);
}
// The setup's per-launch constants, opaque at each use: what is computed from
// them alone (S, FP32 copies) is made again per batch instead of being held in
// registers through the pixel loop, which spilled 11 of them.
struct SetupArgs {
  double inv_dr, k_rev, r0, dmax;
  int half, win;
  SARBP_HD explicit SetupArgs(const BpArgs& a)
      : inv_dr(a.inv_dr), k_rev(a.k_rev), r0(a.r0), dmax(a.dmax), half(a.half), win(a.win) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(inv_dr), "+s"(k_rev), "+s"(r0), "+s"(dmax), "+s"(half), "+s"(win));
#endif
  }
};

// Geometry of one pulse over a wave's strip and its expansion: FP64 where a
// term is large against the phase tolerance, FP32 for the terms of third order
// and above (at most a few revolutions over a strip).
template <int INTERP, int PREC, int PX, int PY>
struct PolySetup {
  static constexpr float X = kTileX * PX / 2, Y = 0.5f * (PY - 1);
  double R0, inv, al, be;  // centre range, 1 / R0, e.ux, e.uy
  double bin0;             // the centre's bin in the profile
  double c20;              // x^2 coefficient
  float alf, bef, a20, a11, a02, g2, g3, c31, c22, c03;
  float c50, c41;          // SARBP_PREC_DF
  bool bounded;            // the strip's bins are known and inside the planned window
  int first, n;            // the n positions (linear: samples) its pixels touch, from bin `first`
  int mode;

  // (wx, wy, wz): the strip's centre, yc rows from the tile reference pixel;
  // tc: {-, -, -, |ux|^2, ux.uy, |uy|^2}
  SARBP_HD PolySetup(const BpArgs& a, double wx, double wy, double wz, double yc, const double* tc,
                                       const double* pos) {
    // every kernel that images a job has to round this alike
#pragma clang fp contract(off)
    const SetupArgs c(a);
    const double ex = wx - pos[0], ey = wy - pos[1], ez = wz - pos[2];
    // 1 / R0 by Newton from the hardware's estimate, then R0 = R^2 / R0 with
    // its own correction: both to an ulp or two
    const double r2 = fma(ez, ez, fma(ey, ey, ex * ex));
    double y = rsqrt_estimate(r2);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const double h = 0.5 * y;
      y = fma(h, fma(-r2 * y, y, 1.0), y);
    }
    const double r = r2 * y;
    R0 = fma(0.5 * y, fma(-r, r, r2), r);
    inv = y;
    al = fma(ez, a.ux[2], fma(ey, a.ux[1], ex * a.ux[0])) * inv;
    be = fma(ez, a.uy[2], fma(ey, a.uy[1], ex * a.uy[0])) * inv;
    bin0 = (R0 - c.r0) * c.inv_dr;
    alf = (float)al;
    bef = (float)be;
    // R is convex in d: R0 + s <= R <= R0 + s + |d|^2 / (2 (R0 + s)), and s is
    // extremal at the strip's corners (the FP32 rounding of the offsets is
    // inside the margin of one bin)
    const float smin = fminf(-alf * X, alf * (X - 1.0f)) - fabsf(bef) * Y;
    const float smax = fmaxf(-alf * X, alf * (X - 1.0f)) + fabsf(bef) * Y;
    const float r0f = (float)R0, xlo = r0f + smin, dmax = (float)c.dmax;
    const float up = smax + 0.5f * dmax * dmax * rcp_estimate(xlo);
    const double ulo = fma((double)smin, c.inv_dr, bin0);
    const double uhi = fma((double)up, c.inv_dr, bin0);
    // The strip's positions have to lie inside the window that whole_window
    // gives the pulse (a.half bins below the tile reference pixel's): strips
    // decide one by one, alike in every kernel, and whatever they decide, a
    // tile's four never span more than that window.  `ref`: the reference
    // pixel's range from R0, by its difference of squares.  The tenth of a bin
    // covers the FP32 rounding here.
    constexpr int kOff = sinc_rows(INTERP) > 0 ? 3 : 0, kEnd = sinc_rows(INTERP) > 0 ? 2 : 3;
    const float ycf = (float)yc, inv_drf = (float)c.inv_dr;
    const float m = fmaf(ycf * ycf, (float)tc[5], -2.0f * ycf * bef * r0f);
    const float ref = m * rcp_estimate(r0f + sqrt_estimate(fmaf(r0f, r0f, m)));
    const bool inside = (smin - ref) * inv_drf >= (float)(kOff + 2 - c.half) + 0.1f &&
                        (up - ref) * inv_drf <= (float)(kOff + window_room(INTERP, c.win) - c.half - kEnd - 1) - 0.1f;
    bounded = inside && xlo > 0.5f * r0f && fabs(ulo) < 1.0e9 && fabs(uhi) < 1.0e9;
    // one bin of margin for the FP32 rounding of a pixel's bin; linear reads
    // one sample above it
    first = bounded ? (int)floor(ulo) - 1 : 0;
    n = bounded ? (int)floor(uhi) - first + (sinc_rows(INTERP) > 0 ? 2 : 3) : 0;
    const float uxx = (float)tc[3], uyy = (float)tc[5], invf = (float)inv;
    const double d20 = fma(-al, al, tc[3]);
    c20 = 0.5 * inv * d20;
    a20 = (float)d20;
    a11 = (float)(2.0 * (tc[4] - al * be));
    a02 = (float)(tc[5] - be * be);
    g2 = 0.5f * invf * invf;
    g3 = 0.25f * g2 * invf;
    c31 = g3 * (4.0f * alf * (alf * a11 + 2.0f * bef * a20) - 2.0f * a20 * a11);
    c22 = g3 * (4.0f * (alf * alf * a02 + bef * (2.0f * alf * a11 + bef * a20)) - 2.0f * a20 * a02 - a11 * a11);
    c03 = -g2 * bef * a02;
    const float lx = X * sqrt_estimate(uxx), ly = Y * sqrt_estimate(uyy), mu = fabsf(alf) * X * rcp_estimate(lx);
    const float q1 = lx * invf, q2 = q1 * q1, q4 = q2 * q2;
    const float rad = 6.2831853f * (float)c.k_rev;
    const float c13 = g3 * (4.0f * bef * (bef * a11 + 2.0f * alf * a02) - 2.0f * a11 * a02);
    const float c04 = g3 * a02 * (4.0f * bef * bef - a02);
    const float e13 = X * Y * Y * Y * fabsf(c13) + Y * Y * Y * Y * fabsf(c04);
    const float l = lx + ly, q = l * invf, ql4 = q * q * q * q;
    if constexpr (PREC == kDF) {
      const float r4 = 4.0f * g2 * g2;
      const float af2 = alf * alf;
      c50 = r4 * alf * a20 * (0.375f * a20 - 0.5f * af2);
      c41 = r4 * (0.375f * a20 * (bef * a20 + 2.0f * alf * a11) - 0.5f * af2 * (alf * a11 + 3.0f * bef * a20));
      // Dropped: x y^3 and y^4; the fifth order but for x^5 and x^4 y; the sixth,
      // along x (mu its cosine) and off it up to ly times the form's largest
      // gradient, 0.38 |d|^5 / R0^5; and from the seventh on |d| (d / R0)^6 / 16 /
      // (1 - d / R0).
      const float bf2 = bef * bef, ab = alf * bef, t22 = 2.0f * a20 * a02 + a11 * a11;
      const float c32 = r4 * (0.375f * (alf * t22 + 2.0f * bef * a20 * a11) -
                              0.5f * alf * (af2 * a02 + 3.0f * (ab * a11 + bf2 * a20)));
      const float c23 = r4 * (0.375f * (2.0f * alf * a11 * a02 + bef * t22) -
                              0.5f * bef * (3.0f * (af2 * a02 + ab * a11) + bf2 * a20));
      const float c14 = r4 * (0.375f * a02 * (alf * a02 + 2.0f * bef * a11) - 0.5f * bf2 * (3.0f * alf * a02 + bef * a11));
      const float c05 = r4 * bef * a02 * (0.375f * a02 - 0.5f * bf2);
      const float e5 = Y * Y * (X * X * (X * fabsf(c32) + Y * fabsf(c23)) + Y * Y * (X * fabsf(c14) + Y * fabsf(c05)));
      const float mu2 = mu * mu;
      const float e6 = q4 * q1 * lx * (0.0625f + 0.75f * mu2 + 0.5f * mu2 * mu2) + ql4 * q * (0.38f * ly + 0.125f * q * l);
      // Revolutions of the terms that FP32 rounds, and of those it does not.
      const float kr = (float)c.k_rev, g = 0.5f * invf;
      const float rounded = X * Y * (g * fabsf(a11) + X * g2 * (fabsf(alf * a11) + fabsf(bef) * a20) +
                                     Y * g2 * (fabsf(alf) * a02 + fabsf(bef * a11))) +
                            g * Y * Y * a02 + X * X * X * g2 * fabsf(alf) * a20;
      const float exact = kr * X * X * g * a20 + 0.5f * X;
      const float err = e13 + e5 + e6, e03 = 0.25f * Y * Y * Y * fabsf(c03);
      mode = bounded && q <= 0.5f && rad * err <= kCompTol && inv_drf * (err + e03) <= kBinTol &&
                     kr * rounded <= kCompTurns && exact <= kCompExact ? 0 : 2;
    } else {
      // Dropped: x y^3 and y^4 whole; x^2 y^2, x^3 y and y^3 but for their fits;
      // the fifth order, (3 mu - 10 mu^3 + 7 mu^5) / 8 of lx^5 / R0^4 along x
      // (mu its cosine), off it up to ly times the form's largest gradient, 0.42
      // |d|^4 / R0^4; and from the sixth on |d| (d / R0)^5 / 16 / (1 - d / R0).
      const float e5 = q4 * (0.375f * mu + 1.25f * mu * mu * mu) * lx + ql4 * (0.42f * ly + 0.125f * q * l);
      const float e22 = 0.5f * X * X * Y * Y * fabsf(c22);
      const float e31 = 0.25f * X * X * X * Y * fabsf(c31), e03 = 0.25f * Y * Y * Y * fabsf(c03);
      const float err1 = e5 + e22 + e13, err0 = err1 + e31 + e03;
      const bool mode0 = rad * err0 <= kPolyTol[0] && inv_drf * err0 <= kBinTol;
      const bool mode1 = rad * err1 <= kPolyTol[1] && inv_drf * (err1 + e03) <= kBinTol;
      mode = !(bounded && q <= 0.5f) ? 2 : (mode0 ? 0 : (mode1 ? 1 : 2));
    }
  }

  // Where the strip is not bounded: the planned window about the tile reference
  // pixel, every pixel's bin clamped into it.
  SARBP_HD void whole_window(const BpArgs& a, const double* tc, const double* pos) {
#pragma clang fp contract(off)
    const double ex = tc[0] - pos[0], ey = tc[1] - pos[1], ez = tc[2] - pos[2];
    const double bc = floor((sqrt(fma(ez, ez, fma(ey, ey, ex * ex))) - a.r0) * a.inv_dr) - (double)a.half;
    first = (int)fmax(fmin(bc, 2.0e9), -2.0e9) + (sinc_rows(INTERP) > 0 ? 3 : 0);
    n = window_room(INTERP, a.win);
    mode = 2;
  }

  // The record of a strip whose positions begin `offset` bytes into the
  // pulse's staged ones.
  SARBP_HD void store(const BpArgs& a, const double* pos, int offset, float4* r) const {
#pragma clang fp contract(off)
    const SetupArgs c(a);
    constexpr double kS = bin_scale<INTERP>();
    const float S = (float)(c.inv_dr * kS);
    // Phase increments per pixel reduced to one revolution, exact for the
    // integer x; y is half-integer, so the whole revolutions of a row step
    // leave (PY - 1) / 2 of themselves in the constant.
    double pa = c.k_rev * al;
    pa -= rint(pa);
    double pb = c.k_rev * be;
    const double turns = rint(pb);
    pb -= turns;
    double c0 = fma(c.k_rev, R0, -turns * (0.5 * (PY - 1)));
    c0 -= floor(c0);
    const int base = bounded ? (int)floor(bin0) - first : 0;
    const float b0 = (float)(kS * (bin0 - (double)(first + base)));
    const float lowest = (float)(-kS * base), highest = (float)(bin_last<INTERP>(n) - kS * base);
    const float tag = float_of_bits(((offset + base * room_bytes(INTERP)) << 2) | mode);
    const float g = (float)(0.5 * inv), f01 = 0.75f * Y * Y * c03;
    if constexpr (PREC == kDF) {
      if (mode == 2) {
        double* d = reinterpret_cast<double*>(r);
        for (int k = 0; k < 3; ++k) d[k] = pos[k];
        d[3] = fma((double)(first + base), a.dr, c.r0);
        r[5] = make_float4(lowest, highest, 0.0f, tag);
        return;
      }
      const double a2 = c.k_rev * c20;
      const double pah = rint(pa * kCompGrid) * (1.0 / kCompGrid), a2h = rint(a2 * kCompGrid) * (1.0 / kCompGrid);
      r[0] = make_float4((float)c0, (float)pah, (float)(pa - pah), (float)a2h);
      r[1] = make_float4((float)(a2 - a2h), (float)(c.inv_dr * kS * c20), -S * g2 * alf * a20,
                         S * g3 * a20 * (4.0f * alf * alf - a20));
      r[2] = make_float4(S * c50, (float)pb, S * g * a11, -S * g2 * (alf * a11 + bef * a20));
      r[3] = make_float4(S * c31, S * c41, S * g * a02, -S * g2 * (alf * a02 + bef * a11));
      r[4] = make_float4(S * c22, (float)c.k_rev * c03, b0, (float)(c.inv_dr * kS * al));
      r[5] = make_float4((float)(c.inv_dr * kS * be) + S * f01, 0.0f, 0.0f, tag);
      return;
    }
    if (mode == 2) {
      r[0] = make_float4((float)c0, (float)pa, (float)(2.0 * R0), highest);
      r[1] = make_float4(g, (float)pb, g2, 0.0f);
      r[2] = make_float4(lowest, 0.0f, b0, alf);
      r[3] = make_float4(bef, 0.0f, 0.0f, tag);
      return;
    }
    // mode 0: x^3 y and, in the phase too, y^3 as their best fits in x y and y
    const float f11 = mode == 0 ? 0.75f * X * X * c31 : 0.0f;
    r[0] = make_float4((float)c0, (float)pa, (float)(c.inv_dr * kS * c20), -S * g2 * alf * a20);
    r[1] = make_float4(S * g3 * a20 * (4.0f * alf * alf - a20), (float)pb + (mode == 0 ? (float)c.k_rev * f01 : 0.0f),
                       S * (g * a11 + f11), -S * g2 * (alf * a11 + bef * a20));
    r[2] = make_float4(S * (g * a02 + 0.5f * X * X * c22), -S * g2 * (alf * a02 + bef * a11), b0,
                       (float)(c.inv_dr * kS * al));
    r[3] = make_float4((float)(c.inv_dr * kS * be) + S * f01, S * c31, (float)c.k_rev * c03, tag);
  }
};

// The polynomial's terms in y at one column x of the strip: the phase is
// A + y (B + y^2 D) + y^2 C, the bin b0 + y b1 + y^2 b2.  rk: revolutions per bin
// unit.
struct RowTerms {
  float A, B, C, D, b0, b1, b2;
};

// Of a SARBP_PREC_REF record, mode 0 or 1.  pa x reaches 16 revolutions a column;
// taken to its fraction it is rounded once at that size and not again with each
// term added, for one instruction a column and pulse (0.4-0.9% of the time): 0.25
// to 0.8 m images are a third nearer to the FP64 ones (2500 x 1700 of 0.37 m,
// linear: 1.99e-6 -> 1.39e-6, 1.80e-6 with the expansion per pixel).
template <int MODE>
SARBP_HD RowTerms ref_row(const float4& p0, const float4& p1, const float4& p2, const float4& p3, float x, float x2,
                          float rk) {
#pragma clang fp contract(off)
  RowTerms t;
  const float qa = x2 * fmaf(fmaf(p1.x, x, p0.w), x, p0.z);
  t.A = fmaf(rk, qa, fract_of(fmaf(p0.y, x, p0.x)));
  t.b0 = fmaf(p2.w, x, p2.z) + qa;
  const float qb = x * (MODE == 1 ? fmaf(fmaf(p3.y, x, p1.w), x, p1.z) : fmaf(p1.w, x, p1.z));
  t.B = fmaf(rk, qb, p1.y);
  t.b1 = p3.x + qb;
  t.b2 = fmaf(p2.y, x, p2.x);
  t.C = rk * t.b2;
  t.D = MODE == 1 ? p3.z : 0.0f;
  return t;
}

// Of a SARBP_PREC_DF record, mode 0: the large phase terms exact modulo a
// revolution.
SARBP_HD RowTerms comp_row(const float4& p0, const float4& p1, const float4& p2, const float4& p3, const float4& p4,
                           const float4& p5, float x, float x2, float rk) {
#pragma clang fp contract(off)
  RowTerms t;
  const float turns = fract_of(fmaf(p0.y, x, p0.w * x2));  // exact
  const float qh = x * fmaf(fmaf(p2.x, x, p1.w), x, p1.z);
  t.A = turns + fmaf(x2, fmaf(rk, qh, p1.x), fmaf(p0.z, x, p0.x));
  t.b0 = fmaf(p4.w, x, p4.z) + x2 * (p1.y + qh);
  const float qb = x * fmaf(fmaf(fmaf(p3.y, x, p3.x), x, p2.w), x, p2.z);
  t.B = fmaf(rk, qb, p2.y);
  t.b1 = p5.x + qb;
  t.b2 = fmaf(fmaf(p4.x, x, p3.w), x, p3.z);
  t.C = rk * t.b2;
  t.D = p4.y;
  return t;
}

// A strip-pulse's work where its own wave stages its positions, over its work
// where a workgroup stages the tile's for four: `strip` and `tile` are the
// positions (samples) touched.  In units of a staged position, a row of 64
// pixels costs 6.25 (sinc8) or 37 (linear), again for every piece that the
// strip's positions are staged in.  Fitted to the throughput of 2048^2 images
// against split 768^2 and 1024^2 ones, columns across, along and at 45 degrees
// to range at 0.25 to 1.6 m: within 25% of the measured ratios of 0.9 to 3.3.
SARBP_HD float split_cost(int interp, int prec, int rows, float strip, float tile) {
#pragma clang fp contract(off)
  const bool sinc = sinc_rows(interp) > 0;
  const float pixels = (sinc ? 6.25f : 37.0f) * (float)rows;
  const float pieces = ceilf(strip / (float)(kSplitStage / room_bytes(interp)));
  const float scale = (sinc ? 1.0f : 0.88f) * (prec == kDF ? 1.1f : 1.0f);
  return scale * (pixels * fmaxf(pieces, 1.0f) + strip) / (pixels + 0.25f * tile);
}
// Positions that a strip of 64 columns by `rows` rows touches, of range steps dx
// and dy (m) a pixel.
SARBP_HD float touched(double dx, double dy, int rows, double inv_dr) {
#pragma clang fp contract(off)
  return (float)((dx * (kTileX - 1) + dy * (rows - 1)) * inv_dr) + 3.5f;
}

// Whether a job's strips cost less than `limit` split, by the mean range steps at
// two quarter points of the image from the first, the middle and the last of
// its antenna positions.  A position that is no number does not split.  Two
// launches of one call ask, and each images what the other leaves: they have to
// round alike, so here as in the functions above the compiler contracts nothing.
SARBP_HD bool split_wins(const BpArgs& a, const double* pos, int rows, float limit) {
#pragma clang fp contract(off)
  double dx = 0.0, dy = 0.0;
  for (int m = 0; m < 6; ++m) {
    const double* p = pos + 3 * (size_t)(m % 3 == 0 ? 0 : (m % 3 == 1 ? a.n_pulses / 2 : a.n_pulses - 1));
    const double at = m < 3 ? 0.25 : 0.75;
    double r2 = 0.0, al = 0.0, be = 0.0;
    for (int k = 0; k < 3; ++k) {
      const double e = a.origin[k] + at * a.nx * a.ux[k] + at * a.ny * a.uy[k] - p[k];
      r2 += e * e;
      al += e * a.ux[k];
      be += e * a.uy[k];
    }
    const double sixth = (1.0 / 6.0) * rsqrt_estimate(r2);
    dx += fabs(al) * sixth;
    dy += fabs(be) * sixth;
  }
  return split_cost(a.kernel_interp, a.kernel_prec, rows, touched(dx, dy, rows, a.inv_dr),
                    touched(dx, dy, kWaves * rows, a.inv_dr)) < limit;
}

SARBP_HD double dot_fma(const double* u, const double* v) { return fma(u[2], v[2], fma(u[1], v[1], u[0] * v[0])); }

// The setup's constants of one tile: its reference pixel and the grid steps'
// products (kept in LDS, not in 12 registers through the pixel loop).  Here, in
// strip_centre and in whole_window the FMAs are written out: left to the
// compiler, kernels that image the same job might round them differently.
SARBP_HD void tile_constants(const BpArgs& a, int x0, int y0, int tx, int ty, double* tc) {
  const int ic = x0 + tx / 2, jc = y0 + ty / 2;
  for (int k = 0; k < 3; ++k) tc[k] = fma((double)jc, a.uy[k], fma((double)ic, a.ux[k], a.origin[k]));
  tc[3] = dot_fma(a.ux, a.ux);
  tc[4] = dot_fma(a.ux, a.uy);
  tc[5] = dot_fma(a.uy, a.uy);
}

// A strip's centre, yc rows from the tile reference pixel.
SARBP_HD double strip_centre(const BpArgs& a, const double* tc, double yc, int k) { return fma(yc, a.uy[k], tc[k]); }

}  // namespace sarbp
