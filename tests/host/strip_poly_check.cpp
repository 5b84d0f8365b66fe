// strip_poly_check.cpp -- the row-polynomial setup of the BP kernels
// (csrc/sarbp_poly.h, planned by csrc/sarbp_plan.cpp) on random geometries,
// against the exact slant range (tests/test_strip_polynomials.py builds and
// runs it; no GPU).  Checks by name:
//   window   every strip's staged positions lie inside the pulse's planned
//            window, whatever the antenna positions, and a bounded strip's hold
//            every pixel's bin with half a bin to spare.
//   ref      SARBP_PREC_REF: what the accepted mode leaves out stays within its
//            tolerance, for pixels of any shape (aspect 1:100 to 100:1).
//   df       the same of SARBP_PREC_DF.
//   df_phase the FP32 phase of accepted SARBP_PREC_DF strips, as the kernel
//            evaluates it, against the exact one.
//   bins     the same of the bins, of REF and DF, at any carrier down to none:
//            within FP32 rounding (at their distance from the centre's) of the
//            exact ones and inside the positions.
//   split    whether a strip's pulses are shared out over waves: where its columns
//            lie across range on images too small to fill the chip, not where
//            each wave would stage a tile's positions; without the positions the
//            kernels decide alike.
//   launch   random planned launches, plain and batched: their LDS within the
//            budget, room for a whole window in it, every pulse in a partial sum,
//            the same sums in both.
//   root     the FP64 square root of the per-pixel fallback: two roundings.
// Exit status 0 when the named check passes.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "sarbp.h"
#include "sarbp_host.h"
#include "sarbp_poly.h"

using namespace sarbp;

namespace {

int g_failures = 0;
long g_strips = 0, g_bounded = 0;

#define CHECK(cond, ...)                                      \
  do {                                                        \
    if (!(cond) && ++g_failures <= 20) {                      \
      std::fprintf(stderr, "FAIL %s:%d: ", __FILE__, __LINE__); \
      std::fprintf(stderr, __VA_ARGS__);                      \
      std::fprintf(stderr, "\n");                             \
    }                                                         \
  } while (0)

using Rng = std::mt19937_64;
double uniform(Rng& r, double lo, double hi) { return std::uniform_real_distribution<double>(lo, hi)(r); }
double log_uniform(Rng& r, double lo, double hi) { return std::exp(uniform(r, std::log(lo), std::log(hi))); }

// A planned job and its antenna positions (which need not be the planned ones).
struct Job {
  BpArgs a;
  std::vector<double> pos;
};

// The strips of (tile x0, y0) and one pulse: calls f(setup, wave, yc) for each.
template <int INTERP, int PREC, int PY, class F>
void each_strip(const BpArgs& a, int tile, const double* pos, F&& f) {
  const int TY = kWaves * PY;
  double tc[6];
  tile_constants(a, tile % a.tiles_x * kTileX, tile / a.tiles_x * TY, kTileX, TY, tc);
  for (int w = 0; w < kWaves; ++w) {
    const double yc = w * PY + 0.5 * (PY - 1) - TY / 2;
    PolySetup<INTERP, PREC, 1, PY> ps(a, tc[0] + yc * a.uy[0], tc[1] + yc * a.uy[1], tc[2] + yc * a.uy[2], yc, tc, pos);
    f(ps, w, yc, tc);
  }
}

// Exact slant range of column x, row y (from the tile reference pixel tc).
long double range_at(const BpArgs& a, const double* tc, const double* pos, double x, double y) {
  long double s = 0;
  for (int k = 0; k < 3; ++k) {
    const long double d = (long double)tc[k] + x * (long double)a.ux[k] + y * (long double)a.uy[k] - pos[k];
    s += d * d;
  }
  return sqrtl(s);
}

template <int INTERP, int PREC, int PY>
void window_one(const Job& j) {
  const BpArgs& a = j.a;
  const bool sinc = sinc_rows(INTERP) > 0;
  for (int tile = 0; tile < a.tiles_x * a.tiles_y; ++tile)
    for (size_t m = 0; m < j.pos.size() / 3; ++m) {
      const double* pos = &j.pos[3 * m];
      each_strip<INTERP, PREC, PY>(a, tile, pos, [&](auto ps, int w, double yc, const double* tc) {
        auto whole = ps;
        whole.whole_window(a, tc, pos);
        ++g_strips;
        if (!ps.bounded) return;  // takes `whole` itself
        ++g_bounded;
        CHECK(ps.n >= 1 && ps.first >= whole.first && ps.first + ps.n <= whole.first + whole.n,
              "tile %d pulse %zu strip %d: positions [%d, %d + %d) outside the window [%d, %d + %d)", tile, m, w,
              ps.first, ps.first, ps.n, whole.first, whole.first, whole.n);
        for (int y = 0; y < PY; y += PY - 1)
          for (int x = -32; x < 32; x += 7) {
            const long double u = (range_at(a, tc, pos, x, yc + y - 0.5 * (PY - 1)) - a.r0) / a.dr - ps.first;
            CHECK(u >= 0.5L && u <= ps.n - (sinc ? 0.5L : 1.5L), "tile %d pulse %zu strip %d: bin %Lg of %d", tile, m,
                  w, u, ps.n);
          }
      });
    }
}

template <int PREC, int PY>
void window_interp(const Job& j) {
  if (j.a.kernel_interp == kLinear) window_one<kLinear, PREC, PY>(j);
  if (j.a.kernel_interp == kSinc8) window_one<kSinc8, PREC, PY>(j);
  if (j.a.kernel_interp == kSinc8W) window_one<kSinc8W, PREC, PY>(j);
}

void check_window() {
  Rng rng(7);
  for (int i = 0; i < 3000; ++i) {
    const int py = 2 << (int)(rng() % 3);
    const bool near = rng() % 2;
    sarbp_grid g{};
    const double sx = log_uniform(rng, 0.05, 4.0), sy = sx * log_uniform(rng, 0.2, 5.0);
    const double ang = uniform(rng, 0, 6.2831853);
    g.ux[0] = sx * std::cos(ang), g.ux[1] = sx * std::sin(ang), g.ux[2] = sx * uniform(rng, -0.2, 0.2);
    g.uy[0] = -sy * std::sin(ang), g.uy[1] = sy * std::cos(ang), g.uy[2] = sy * uniform(rng, -0.2, 0.2);
    g.nx = 1 + (int)(rng() % 130);
    g.ny = 1 + (int)(rng() % 100);
    sarbp_params p{};
    p.c = 299792458.0;
    p.fc = 9.6e9;
    p.dr = log_uniform(rng, 0.05, 2.0);
    p.n_pulses = 6;
    p.n_samples = 4096;
    p.r0 = uniform(rng, -100, 100);
    p.kaiser_beta = 6;
    p.interp = 1 + (int)(rng() % 2);
    p.precision = rng() % 2 ? SARBP_PREC_REF : SARBP_PREC_DF;
    Job j;
    j.pos.resize(18);
    const double R = near ? log_uniform(rng, 1e-4, 300.0) : log_uniform(rng, 300.0, 1e6);
    for (int m = 0; m < 6; ++m) {
      // above, beside or on the image, from a pixel, a strip's centre or anywhere
      const double px = (int)(rng() % 64) + (rng() % 2 ? 0.0 : uniform(rng, 0, 1)),
                   py_ = (int)(rng() % 32) + 0.5 * (int)(rng() % 2);
      double d[3] = {uniform(rng, -1, 1), uniform(rng, -1, 1), uniform(rng, 0, 1)};
      const double n = std::sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
      for (int k = 0; k < 3; ++k)
        j.pos[3 * m + k] = g.origin[k] + px * g.ux[k] + py_ * g.uy[k] + d[k] / n * R;
    }
    if (near && rng() % 20 == 0) j.pos[rng() % 18] = NAN;
    if (near && rng() % 20 == 0) j.pos[rng() % 18] = INFINITY;
    if (near && rng() % 20 == 0) j.pos[rng() % 18] = 1e300;
    // planned from the grid, from these positions, or from others
    std::vector<double> h = j.pos;
    if (rng() % 3 == 0)
      for (double& v : h) v = v * 1.5 + 50.0;
    const double* hp = rng() % 2 ? h.data() : nullptr;
    sarbp_tuning t{py, 1, 4};
    const Fitted f = fit_tuning(t, p.precision, &g, &p, hp);
    if (plan_args(hp, &g, &p, f.t, f.prec, &j.a, nullptr) != SARBP_OK) continue;
    if (f.t.rows_per_lane == 2) f.prec == kRef ? window_interp<kRef, 2>(j) : window_interp<kDF, 2>(j);
    if (f.t.rows_per_lane == 4) f.prec == kRef ? window_interp<kRef, 4>(j) : window_interp<kDF, 4>(j);
    if (f.t.rows_per_lane == 8) f.prec == kRef ? window_interp<kRef, 8>(j) : window_interp<kDF, 8>(j);
  }
  // both sides have to occur
  CHECK(g_bounded > g_strips / 20 && g_bounded < g_strips - g_strips / 20, "%ld of %ld strips bounded", g_bounded,
        g_strips);
}

// Kept terms of R - R0 (long double) of a strip: the Taylor expansion of
// sqrt((R0 + s)^2 + pp) in (s, pp) up to `fourth` order whole, its monomials
// x^i y^j of third order and above filtered by keep(i, j) -> factor on another
// monomial.  Coefficients c[i][j] by expanding the powers of s and pp.
struct Series {
  long double c[8][8] = {};  // c[i][j] x^i y^j, total degree <= 6
};
using Poly = Series;
Poly mul(const Poly& a, const Poly& b) {
  Poly r;
  for (int i = 0; i < 7; ++i)
    for (int j = 0; i + j < 7; ++j)
      if (a.c[i][j] != 0)
        for (int k = 0; i + j + k < 7; ++k)
          for (int l = 0; i + j + k + l < 7; ++l) r.c[i + k][j + l] += a.c[i][j] * b.c[k][l];
  return r;
}
Poly add(const Poly& a, const Poly& b, long double f) {
  Poly r = a;
  for (int i = 0; i < 8; ++i)
    for (int j = 0; j < 8; ++j) r.c[i][j] += f * b.c[i][j];
  return r;
}

// Strip geometry in long double.
struct Exact {
  long double R0, al, be, uxx, uxy, uyy;
  Exact(const BpArgs& a, const double* centre, const double* pos) {
    long double e[3], r2 = 0;
    al = be = uxx = uxy = uyy = 0;
    for (int k = 0; k < 3; ++k) e[k] = (long double)centre[k] - pos[k], r2 += e[k] * e[k];
    R0 = sqrtl(r2);
    for (int k = 0; k < 3; ++k) {
      al += e[k] * a.ux[k] / R0;
      be += e[k] * a.uy[k] / R0;
      uxx += (long double)a.ux[k] * a.ux[k];
      uxy += (long double)a.ux[k] * a.uy[k];
      uyy += (long double)a.uy[k] * a.uy[k];
    }
  }
  // R - R0 at (x, y), without cancellation
  long double at(long double x, long double y) const {
    const long double s = al * x + be * y, dd = uxx * x * x + 2 * uxy * x * y + uyy * y * y;
    const long double t = 2 * R0 * s + dd;
    return t / (R0 + sqrtl(R0 * R0 + t));
  }
  // R - R0 to sixth order
  Poly series() const {
    Poly s, pp, one;
    one.c[0][0] = 1;
    s.c[1][0] = al, s.c[0][1] = be;
    pp.c[2][0] = uxx - al * al, pp.c[1][1] = 2 * (uxy - al * be), pp.c[0][2] = uyy - be * be;
    // sqrt(1 + z), z = (2 R0 s + s^2 + pp) / R0^2, to z^6
    Poly z = add(add(Poly{}, s, 2 / R0), add(mul(s, s), pp, 1), 1 / (R0 * R0)), zp = one, r;
    long double b = 1;
    for (int k = 1; k <= 6; ++k) {
      zp = mul(zp, z);
      b *= (1.5L - k) / k;
      r = add(r, zp, R0 * b);
    }
    return r;
  }
};

long double eval(const Poly& p, double x, double y) {
  long double r = 0;
  for (int i = 7; i >= 0; --i) {
    long double t = 0;
    for (int j = 7; j >= 0; --j) t = t * y + p.c[i][j];
    r = r * x + t;
  }
  return r;
}

// A strip of PX x PY pixels per lane at range R: pixels of any shape and slant,
// a window that holds it.
template <int PX, int PY>
void random_strip(Rng& rng, BpArgs& a, double* tc, double* pos, double lx_max, double r_lo, double r_hi) {
  std::memset(&a, 0, sizeof a);
  const double R = log_uniform(rng, r_lo, r_hi);
  const double fc[] = {0.4e9, 1.3e9, 5.3e9, 9.6e9, 35e9};
  a.k_rev = 2 * fc[rng() % 5] / 299792458.0;
  const double aspect = log_uniform(rng, 0.01, 100.0), size = log_uniform(rng, 1e-4, 0.3) * R;
  const double ly_over_lx = (PY - 1) * aspect / (64.0 * PX);
  double lx = size / std::max(1.0, ly_over_lx);
  lx = std::min(lx, lx_max);
  const double sx = lx / (32.0 * PX), sy = sx * aspect, ang = uniform(rng, 0, 6.2831853),
               slant = uniform(rng, -0.5, 0.5) * (rng() % 2);
  a.ux[0] = sx * std::cos(ang), a.ux[1] = sx * std::sin(ang);
  a.uy[0] = -sy * std::sin(ang + slant), a.uy[1] = sy * std::cos(ang + slant);
  if (rng() % 2) a.ux[2] = sx * uniform(rng, -0.3, 0.3), a.uy[2] = sy * uniform(rng, -0.3, 0.3);
  const double el = rng() % 4 ? uniform(rng, 0.1, 1.5) : uniform(rng, 0, 0.1), az = rng() % 2 ? 0.0 : uniform(rng, -1.5, 1.5);
  const double d[3] = {std::cos(el) * std::sin(az), std::cos(el) * std::cos(az), std::sin(el)};
  tile_constants(a, 0, 0, 0, 0, tc);
  for (int k = 0; k < 3; ++k) pos[k] = -d[k] * R;
  const double l = 32.0 * PX * std::sqrt(tc[3]) + 4.0 * PY * std::sqrt(tc[5]);
  a.dmax = l;
  a.dr = log_uniform(rng, 1.0, 100.0) * l / 1000;
  a.inv_dr = 1 / a.dr;
  a.r0 = R - 100 * a.dr;
  a.win = 8192;
  a.half = 4095;
}

long g_taken[3];
double g_worst = 0;

// The terms that the kernel keeps of a strip's series in a mode.
template <int PREC, int PX, int PY>
Poly kept(Poly p, int mode) {
  const double X = 32.0 * PX, Y = 0.5 * (PY - 1);
  for (int i = 0; i < 7; ++i)
    for (int j = 0; i + j < 7; ++j) {
      const long double c = p.c[i][j];
      const int n = i + j;
      bool keep;
      if (PREC == kDF) {
        keep = n <= 3 || (n == 4 && j <= 2) || (n == 5 && j <= 1);
      } else {
        keep = n <= 3 || (n == 4 && j <= 1);
        if (i == 2 && j == 2) p.c[0][2] += 0.5 * X * X * c;
        if (mode == 0 && i == 3 && j == 1) p.c[1][1] += 0.75 * X * X * c, keep = false;
        if (mode == 0 && i == 0 && j == 3) p.c[0][1] += 0.75 * Y * Y * c, keep = false;
      }
      if (!keep) p.c[i][j] = 0;
    }
  return p;
}

template <int PREC, int PX, int PY>
void truncation_one(Rng& rng) {
  BpArgs a;
  double tc[6], pos[3];
  random_strip<PX, PY>(rng, a, tc, pos, PREC == kDF ? 1e5 : 512.0, 100.0, 8e5);
  PolySetup<kSinc8, PREC, PX, PY> ps(a, tc[0], tc[1], tc[2], 0.0, tc, pos);
  ++g_strips;
  g_bounded += ps.bounded;
  ++g_taken[ps.mode];
  if (ps.mode == 2) return;
  const Exact ex(a, tc, pos);
  const Poly p = kept<PREC, PX, PY>(ex.series(), ps.mode);
  const double X = 32.0 * PX, Y = 0.5 * (PY - 1), tol = PREC == kDF ? kCompTol : kPolyTol[ps.mode];
  double worst = 0;
  for (int n = 0; n < PY; ++n)
    for (int k = 0; k <= 16; ++k) {
      const double x = -X + k * (2 * X - 1) / 16, y = n - Y;
      worst = std::max(worst, std::fabs((double)(ex.at(x, y) - eval(p, x, y))));
    }
  const double rad = worst * 6.283185307179586 * a.k_rev;
  g_worst = std::max(g_worst, rad / tol);
  CHECK(rad <= 1.001 * tol, "PX %d PY %d mode %d: %.3g rad left out, |ux| %.3g |uy| %.3g R %.4g fc %.3g", PX, PY,
        ps.mode, rad, std::sqrt(tc[3]), std::sqrt(tc[5]), (double)ex.R0, a.k_rev * 1.5e8);
}

template <int PREC>
void check_truncation() {
  Rng rng(11);
  for (int i = 0; i < 60000; ++i) {
    truncation_one<PREC, 1, 2>(rng), truncation_one<PREC, 1, 4>(rng), truncation_one<PREC, 1, 8>(rng);
    if constexpr (PREC == kRef) {
      truncation_one<PREC, 2, 2>(rng), truncation_one<PREC, 2, 4>(rng), truncation_one<PREC, 2, 8>(rng);
      truncation_one<PREC, 4, 2>(rng), truncation_one<PREC, 4, 4>(rng);
    }
  }
  // every mode is taken, and the bounds are of the errors' size
  for (int m = 0; m < 3; ++m) CHECK(g_taken[m] > g_strips / 100 || (PREC == kDF && m == 1), "mode %d taken %ld", m, g_taken[m]);
  CHECK(g_worst > 0.5, "largest error %.2f of the tolerance", g_worst);
  std::printf("modes %ld %ld %ld, largest error %.2f of the tolerance\n", g_taken[0], g_taken[1], g_taken[2], g_worst);
}

// Row n's phase (revolutions) and bin from a record's terms, as the pixel loops
// form them.
float phase_of(const RowTerms& c, float y) { return fmaf(y, fmaf(y * y, c.D, c.B), fmaf(y * y, c.C, c.A)); }
float bin_of(const RowTerms& c, float y) { return fmaf(y, c.b1, fmaf(y * y, c.b2, c.b0)); }

double g_sum2 = 0;
long g_pixels = 0;

template <int PY>
void df_phase_one(Rng& rng) {
  BpArgs a;
  double tc[6], pos[3];
  random_strip<1, PY>(rng, a, tc, pos, 1e5, 1000.0, 8e5);
  PolySetup<kSinc8, kDF, 1, PY> ps(a, tc[0], tc[1], tc[2], 0.0, tc, pos);
  ++g_strips;
  g_bounded += ps.bounded;
  ++g_taken[ps.mode];
  if (ps.mode == 2) return;
  alignas(16) float4 r[6];
  ps.store(a, pos, 0, r);
  const Exact ex(a, tc, pos);
  const float rk = (float)(a.k_rev * a.dr / bin_scale<kSinc8>());
  double worst = 0;
  for (int n = 0; n < PY; ++n)
    for (int x = -32; x < 32; x += 3) {
      const float y = n - 0.5f * (PY - 1), xf = (float)x;
      const float ph = phase_of(comp_row(r[0], r[1], r[2], r[3], r[4], r[5], xf, xf * xf, rk), y);
      long double e = (long double)a.k_rev * (ex.R0 + ex.at(x, y)) - ph;
      e -= rintl(e);
      worst = std::max(worst, (double)fabsl(e) * 6.283185307179586);
      g_sum2 += (double)(e * e) * 39.4784176;
      ++g_pixels;
    }
  g_worst = std::max(g_worst, worst);
  // 8e-6 rad left out at most, and sums of up to 8 revolutions rounded a few
  // times to 2.4e-7 of one
  CHECK(worst <= 1.3e-5, "PY %d: phase off by %.3g rad, |ux| %.3g |uy| %.3g R %.4g fc %.3g: %.4g revolutions across", PY,
        worst, std::sqrt(tc[3]), std::sqrt(tc[5]), (double)ex.R0, a.k_rev * 1.5e8,
        1024 * a.k_rev * (double)(ex.uxx / (2 * ex.R0)));
}

void check_df_phase() {
  Rng rng(13);
  for (int i = 0; i < 60000; ++i) df_phase_one<2>(rng), df_phase_one<4>(rng), df_phase_one<8>(rng);
  CHECK(g_taken[0] > g_strips / 100 && g_taken[2] > g_strips / 100, "modes %ld %ld", g_taken[0], g_taken[2]);
  const double rms = std::sqrt(g_sum2 / g_pixels);
  // the double-float form per pixel: 1.4e-6 rad rms
  CHECK(rms <= 1.4e-6, "phase error %.3g rad rms", rms);
  std::printf("modes %ld %ld, phase error %.3g rad rms, %.3g at most\n", g_taken[0], g_taken[2], rms, g_worst);
}

template <int INTERP, int PREC, int PX, int PY>
void bins_one(Rng& rng) {
  BpArgs a;
  double tc[6], pos[3];
  random_strip<PX, PY>(rng, a, tc, pos, PREC == kDF ? 1e5 : 512.0, 100.0, 8e5);
  a.k_rev *= std::pow(10.0, -(int)(rng() % 8));
  if (rng() % 8 == 0) a.k_rev = 0;
  PolySetup<INTERP, PREC, PX, PY> ps(a, tc[0], tc[1], tc[2], 0.0, tc, pos);
  ++g_strips;
  g_bounded += ps.bounded;
  ++g_taken[ps.mode];
  if (ps.mode == 2) return;
  alignas(16) float4 r[6];
  ps.store(a, pos, 0, r);
  const Exact ex(a, tc, pos);
  int tag;
  std::memcpy(&tag, &r[poly_rec16(PREC) - 1].w, 4);
  const int base = (tag >> 2) / room_bytes(INTERP);  // the position the bins count from
  const double scale = bin_scale<INTERP>() * a.inv_dr;
  const double first = bin_scale<INTERP>() * ((ps.first + base) * a.dr + a.r0 - (double)ex.R0) * a.inv_dr;
  const float rk = (float)(a.k_rev * a.dr / bin_scale<INTERP>());
  double worst = 0, largest = 0;
  for (int n = 0; n < PY; ++n)
    for (int x = -32 * PX; x < 32 * PX; x += 5) {
      const float y = n - 0.5f * (PY - 1), xf = (float)x;
      RowTerms t;
      if constexpr (PREC == kDF)
        t = comp_row(r[0], r[1], r[2], r[3], r[4], r[5], xf, xf * xf, rk);
      else
        t = ps.mode == 1 ? ref_row<1>(r[0], r[1], r[2], r[3], xf, xf * xf, rk)
                         : ref_row<0>(r[0], r[1], r[2], r[3], xf, xf * xf, rk);
      const float bin = bin_of(t, y);
      const double exact = (double)(ex.at(x, y) * scale - first);
      worst = std::max(worst, std::fabs(bin - exact));
      largest = std::max(largest, std::fabs(exact + first));
      const double at = bin + bin_scale<INTERP>() * base;
      CHECK(at >= 0 && at < bin_last<INTERP>(ps.n) + (INTERP == kLinear ? 0 : 1), "bin %g outside the %d positions",
            at, ps.n);
    }
  // what is left out (kBinTol bins, at the interpolator's scale) and six
  // roundings of the largest distance from the centre's bin
  const double allowed = bin_scale<INTERP>() * kBinTol + 6 * std::ldexp(largest + 1, -24);
  g_worst = std::max(g_worst, worst / allowed);
  CHECK(worst <= allowed, "PREC %d PX %d PY %d mode %d: bin off by %.3g of %.4g, |ux| %.3g |uy| %.3g R %.4g fc %.3g dr %.3g", PREC, PX,
        PY, ps.mode, worst, largest, std::sqrt(tc[3]), std::sqrt(tc[5]), (double)ex.R0, a.k_rev * 1.5e8, a.dr);
}

void check_bins() {
  Rng rng(17);
  for (int i = 0; i < 30000; ++i) {
    bins_one<kLinear, kRef, 1, 2>(rng), bins_one<kSinc8, kRef, 1, 4>(rng), bins_one<kSinc8W, kRef, 1, 8>(rng);
    bins_one<kSinc8, kRef, 2, 8>(rng), bins_one<kLinear, kRef, 4, 4>(rng), bins_one<kSinc8, kDF, 1, 2>(rng);
    bins_one<kLinear, kDF, 1, 4>(rng), bins_one<kSinc8W, kDF, 1, 8>(rng);
  }
  for (long n : g_taken) CHECK(n > g_strips / 200, "modes taken %ld %ld %ld", g_taken[0], g_taken[1], g_taken[2]);
  std::printf("modes %ld %ld %ld, largest error %.2f of the allowed\n", g_taken[0], g_taken[1], g_taken[2], g_worst);
}

void check_root() {
  Rng rng(19);
  double worst = 0;
  for (int i = 0; i < 1000000; ++i) {
    const double r = log_uniform(rng, 1e-3, 1e8), v = r * r;
    const long double exact = sqrtl((long double)v);
    worst = std::max(worst, (double)(fabsl(range_root(v) - exact) / exact));
  }
  CHECK(worst <= std::ldexp(1.0, -52), "root off by 2^%.2f", std::log2(worst));
  CHECK(range_root(0.0) == 0.0, "root of 0 is %g", range_root(0.0));
  std::printf("largest error 2^%.2f\n", std::log2(worst));
}

void check_split() {
  const int sizes[] = {128, 256, 512, 768, 1024, 1536};
  for (int interp : {SARBP_INTERP_LINEAR, SARBP_INTERP_SINC8})
    for (double spacing : {0.25, 0.5, 1.0})
      for (int n : sizes)
        for (int along = 0; along < 2; ++along) {
          sarbp_grid g{};
          g.ux[along] = spacing;
          g.uy[1 - along] = spacing;
          g.nx = g.ny = n;
          g.origin[0] = g.origin[1] = -0.5 * n * spacing;
          sarbp_params p{};
          p.c = 299792458.0, p.fc = 9.6e9, p.dr = 0.1875, p.r0 = 4000, p.kaiser_beta = 6;
          p.n_pulses = 512, p.n_samples = 8192, p.interp = interp;
          std::vector<double> pos(3 * 512);
          for (int m = 0; m < 512; ++m) pos[3 * m] = (m - 256) * 0.15, pos[3 * m + 1] = -4000, pos[3 * m + 2] = 3000;
          for (int planned = 0; planned < 2; ++planned) {
            const double* h = planned ? pos.data() : nullptr;
            const sarbp_tuning t{4, 1, 4};
            BpArgs a;
            CHECK(plan_args(h, &g, &p, t, kRef, &a, nullptr) == SARBP_OK, "refused: %s", last_detail());
            bool split = a.parts > 1;
            if (split && a.split_limit > 0) split = split_wins(a, pos.data(), 4, a.split_limit);
            CHECK(!planned || a.split_limit == 0, "planned with positions, left to the kernels");
            CHECK(a.parts == 1 ? a.sum_pulses == INT32_MAX : (long)a.parts * a.sum_pulses >= 512, "%d sums of %d", a.parts,
                  a.sum_pulses);
            const bool sinc = interp == SARBP_INTERP_SINC8;
            // measured: 256^2 always gains, 768^2 across range; along it sinc8
            // loses from 768^2 on, linear from 1024^2; 1536^2 fills the chip
            if (n <= 256 || (!along && n <= 768))
              CHECK(split, "interp %d %g m %d^2 along %d planned %d: not split", interp, spacing, n, along, planned);
            if (n >= 1536 || (along && n >= (sinc ? 768 : 1024)))
              CHECK(!split, "interp %d %g m %d^2 along %d planned %d: split", interp, spacing, n, along, planned);
            ++g_strips;
          }
        }
}

void check_launch() {
  // registers allow 4 workgroups per CU; LDS in 512-B blocks
  set_occupancy_source([](int, int, int, int, int, size_t shm) {
    return std::max(1, std::min(4, (int)(160 * 1024 / 512 / ((shm + 16 + 511) / 512))));
  });
  Rng rng(23);
  long cut = 0, shared = 0, chosen = 0;
  for (int i = 0; i < 20000; ++i) {
    sarbp_grid g{};
    const double sx = log_uniform(rng, 0.02, 8.0), sy = sx * log_uniform(rng, 0.2, 5.0), ang = uniform(rng, 0, 6.2831853);
    g.ux[0] = sx * std::cos(ang), g.ux[1] = sx * std::sin(ang);
    g.uy[0] = -sy * std::sin(ang), g.uy[1] = sy * std::cos(ang);
    g.nx = (int)log_uniform(rng, 1, 9000);
    g.ny = (int)log_uniform(rng, 1, 9000);
    sarbp_params p{};
    p.c = 299792458.0, p.fc = 9.6e9, p.dr = log_uniform(rng, 0.05, 2.0), p.kaiser_beta = 6;
    p.n_pulses = rng() % 20 ? 1 + (int)(rng() % 300) : (int)(rng() % 2);
    p.n_samples = 4096;
    p.interp = 1 + (int)(rng() % 2);
    p.precision = rng() % 4 ? SARBP_PREC_REF : SARBP_PREC_DF;
    const double R = log_uniform(rng, 300, 1e6);
    std::vector<double> pos(3 * (size_t)p.n_pulses + 3);
    for (int m = 0; m < p.n_pulses; ++m) pos[3 * m] = m * 0.2, pos[3 * m + 1] = -0.8 * R, pos[3 * m + 2] = 0.6 * R;
    const double* h = rng() % 2 ? pos.data() : nullptr;
    const int cls = size_class(&g, &p, h);
    sarbp_tuning t = job_tuning(p.interp, cls, p.precision, h != nullptr, &g);
    const bool builtin = rng() % 2;
    if (!builtin) {
      static const int shapes[][2] = {{1, 2}, {1, 4}, {1, 8}, {2, 2}, {2, 4}, {2, 8}, {4, 2}, {4, 4}};
      const int* sh = shapes[rng() % 8];
      t = sarbp_tuning{sh[1], sh[0], 1 + (int)(rng() % 256)};
      if (check_tuning(p.precision, &t) != SARBP_OK) continue;
    }
    const Fitted f = fit_tuning(t, p.precision, &g, &p, h, builtin);
    BpArgs a, b, whole;
    const sarbp_status st = plan_args(h, &g, &p, f.launch, f.prec, &a, nullptr);
    // a cut tile is refused only where the tuned one is
    CHECK((plan_args(h, &g, &p, f.t, f.prec, &whole, nullptr) == SARBP_OK) == (st == SARBP_OK), "cut tile refused: %s", last_detail());
    if (st != SARBP_OK) continue;
    ++g_strips;
    CHECK(plan_args(h, &g, &p, f.launch, f.prec, &b, nullptr, true) == SARBP_OK, "batched plan refused");
    for (const BpArgs* x : {&a, &b}) {
      const int room = window_room(x->kernel_interp, x->win);
      CHECK(x->pool >= room, "%d staged positions, a window has %d", x->pool, room);
      CHECK(launch_lds(*x) <= kLdsBudget, "%zu bytes of LDS", launch_lds(*x));
      CHECK(x->parts >= 1 && x->parts <= kMaxParts && x->sum_pulses >= 1, "%d parts of %d", x->parts, x->sum_pulses);
      CHECK(x->parts == 1 ? x->sum_pulses >= p.n_pulses : (long)x->parts * x->sum_pulses >= p.n_pulses, "%d parts of %d, %d pulses",
            x->parts, x->sum_pulses, p.n_pulses);
      CHECK(x->parts == 1 || f.launch.cols_per_lane == 1, "parts of %d columns", f.launch.cols_per_lane);
      CHECK(x->split_limit == 0 || (x->parts > 1 && !h), "limit %g, %d parts", x->split_limit, x->parts);
    }
    CHECK(a.parts == b.parts && a.sum_pulses == b.sum_pulses && a.split_limit == b.split_limit && a.win == b.win &&
              a.kernel_interp == b.kernel_interp, "plain and batched plans differ");
    cut += f.launch.rows_per_lane != f.t.rows_per_lane;
    shared += a.parts > 1;
    chosen += a.split_limit > 0;
  }
  CHECK(cut > 100 && shared > 100 && chosen > 100, "%ld cut, %ld shared, %ld left to the kernels", cut, shared, chosen);
  set_occupancy_source(nullptr);
}

}  // namespace

int main(int argc, char** argv) {
  const char* name = argc > 1 ? argv[1] : "";
  if (!std::strcmp(name, "window")) check_window();
  else if (!std::strcmp(name, "ref")) check_truncation<kRef>();
  else if (!std::strcmp(name, "df")) check_truncation<kDF>();
  else if (!std::strcmp(name, "df_phase")) check_df_phase();
  else if (!std::strcmp(name, "bins")) check_bins();
  else if (!std::strcmp(name, "root")) check_root();
  else if (!std::strcmp(name, "split")) check_split();
  else if (!std::strcmp(name, "launch")) check_launch();
  else return std::fprintf(stderr, "unknown check %s\n", name), 2;
  std::printf("%s: %ld strips, %ld bounded, %d failures\n", name, g_strips, g_bounded, g_failures);
  return g_failures != 0;
}
