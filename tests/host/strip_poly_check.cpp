// strip_poly_check.cpp -- the row-polynomial setup of the BP kernels
// (csrc/sarbp_poly.h, planned by csrc/sarbp_plan.cpp) on random geometries,
// against the exact slant range (tests/test_strip_polynomials.py builds and
// runs it; no GPU).  Checks by name:
//   window   every strip's staged positions lie inside the pulse's planned
//            window, whatever the antenna positions, and a bounded strip's hold
//            every pixel's bin with half a bin to spare.
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

}  // namespace

int main(int argc, char** argv) {
  const char* name = argc > 1 ? argv[1] : "";
  if (!std::strcmp(name, "window")) check_window();
  else return std::fprintf(stderr, "unknown check %s\n", name), 2;
  std::printf("%s: %ld strips, %ld bounded, %d failures\n", name, g_strips, g_bounded, g_failures);
  return g_failures != 0;
}
