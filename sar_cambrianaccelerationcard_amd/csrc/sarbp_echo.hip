// sarbp_echo.hip -- point-target raw-echo generator on the device: the
// reference's generateEchoKernel / launchGenerateEcho
// (code/SAR_BP/CUDA/BPA_CUDA_kernels.cu:3-45, :79-89) behind the C ABI.
//
// Sample (i, j) of Srnm [Mslow][Nfast] is the sum over targets k of
// sigma_k exp(j (pi Kr t^2 - 4 pi R / lambda)) for the k inside the pulse
// (0 < t < Tr) and the beam (|Az| < La/2), Az = ta[i] vr - x_k,
// R = sqrt(Az^2 + y_k^2 + H^2), t = tr[j] - 2 R / c.  Range, gate and phase
// are FP64, in that order with one rounding per operation (no contraction),
// so the gate decisions are those of an FP64 evaluation of the formula; the
// phase is reduced to revolutions in FP64 and its sine and cosine are the
// hardware ones (which take revolutions).  The reference evaluates all of it
// in FP32, where 4 pi R / lambda ~ 1e6 rad carries ~0.1 rad of error.
//
// A wave owns one pulse and kEchoSamples x 64 consecutive fast-time samples.
// Range, delay and beam gate depend on the pulse and the target only, so they
// are evaluated once per wave, one target per lane, 64 targets at a time; the
// targets whose delay can fall inside the wave's samples are then taken in
// order, their values broadcast from the lane that holds them.
#include "sarbp.h"
#include "sarbp_host.h"

#include <cmath>

namespace sarbp {
namespace {

// Samples per lane.  More amortise the per-target geometry and delay test,
// fewer put less of a wave beside the pulse's edges: 2048 pulses x 2448
// samples x 64 targets (a chirp of 300 samples) ran 59 / 48.5 / 49.5 / 57.5 us
// at 1 / 2 / 4 / 8.
constexpr int kEchoSamples = 4;

struct EchoArgs {
  float2* out;
  const float* tg;  // [ntarget][3]: azimuth, ground range, sigma
  const float* ta;  // [mslow]
  const float* tr;  // [nfast]
  long long items;  // mslow * chunks: waves' worth of work
  int nfast, ntarget;
  int chunks;       // ceil(nfast / (64 kEchoSamples))
  double c, lambda, kr, tw, vr, h, la_half;
};

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Bound by the VALU: one FP64 delay difference, two compares and, inside the
// pulse, the phase and its sine and cosine per (sample, target near it); the
// square root and the two divisions of a (pulse, target) are paid once per
// wave instead of once per sample (one thread per sample over the whole
// target list: 485 us at 2048 x 2448 x 64, 49.5 us this way).
__global__ __launch_bounds__(256) void echo_kernel(EchoArgs a) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const long long step = (long long)gridDim.x * (blockDim.x >> 6);
  const long long first = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  for (long long item = first; item < a.items; item += step) {
    const int i = __builtin_amdgcn_readfirstlane((int)(item / a.chunks));
    const int j0 = __builtin_amdgcn_readfirstlane((int)(item - (long long)i * a.chunks)) * (64 * kEchoSamples);
    const double ta = a.ta[i];
    // A lane past the line's end holds a NaN time, which passes no gate and
    // leaves the minimum and maximum alone.
    double tr[kEchoSamples];
    double lo = __builtin_nan(""), hi = lo;
#pragma unroll
    for (int s = 0; s < kEchoSamples; ++s) {
      const unsigned j = (unsigned)j0 + lane + 64u * s;
      tr[s] = j < (unsigned)a.nfast ? (double)a.tr[j] : __builtin_nan("");
      lo = fmin(lo, tr[s]);
      hi = fmax(hi, tr[s]);
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
      lo = fmin(lo, __shfl_xor(lo, d));
      hi = fmax(hi, __shfl_xor(hi, d));
    }
    float sx[kEchoSamples] = {}, sy[kEchoSamples] = {};
    for (unsigned k0 = 0; k0 < (unsigned)a.ntarget; k0 += 64) {
      const unsigned k = k0 + lane;
      double delay = 0.0, carrier = 0.0;
      float sigma = 0.0f;
      bool heard = false;
      if (k < (unsigned)a.ntarget) {
        const double x = a.tg[3 * (size_t)k], y = a.tg[3 * (size_t)k + 1];
        sigma = a.tg[3 * (size_t)k + 2];
        const double az = ta * a.vr - x;
        const double r = sqrt(az * az + y * y + a.h * a.h);
        delay = 2.0 * r / a.c;
        carrier = 2.0 * r / a.lambda;
        // the rounded difference is monotonic in the time, so a target that
        // fails here fails the gate at every sample of the wave
        heard = fabs(az) < a.la_half && hi - delay > 0.0 && lo - delay < a.tw;
      }
      for (unsigned long long set = __ballot(heard); set; set &= set - 1) {
        const int l = __builtin_ctzll(set);
        const double dl = lane_value(delay, l), ca = lane_value(carrier, l);
        const float sg = lane_value(sigma, l);
#pragma unroll
        for (int s = 0; s < kEchoSamples; ++s) {
          const double t = tr[s] - dl;
          if (t > 0.0 && t < a.tw) {
            double rev = 0.5 * a.kr * t * t - ca;
            rev -= rint(rev);
            const float ph = (float)rev;
            sx[s] += sg * __builtin_amdgcn_cosf(ph);
            sy[s] += sg * __builtin_amdgcn_sinf(ph);
          }
        }
      }
    }
    float2* row = a.out + (size_t)i * a.nfast;
#pragma unroll
    for (int s = 0; s < kEchoSamples; ++s) {
      const unsigned j = (unsigned)j0 + lane + 64u * s;
      if (j < (unsigned)a.nfast) row[j] = make_float2(sx[s], sy[s]);
    }
  }
}

}  // namespace
}  // namespace sarbp

extern "C" {

sarbp_status sarbp_launch_generate_echo(sarbp_cf32* Srnm, const float* Ptarget, const float* ta, const float* tr,
                                        sarbp_sar_params p, int32_t Mslow, int32_t Nfast) {
  using namespace sarbp;
  if (Mslow < 0 || Nfast < 0 || p.Ntarget < 0)
    return fail(SARBP_ERR_INVALID_ARGUMENT, "Mslow %d, Nfast %d, Ntarget %d: negative", Mslow, Nfast, p.Ntarget);
  const long long total = (long long)Mslow * Nfast;
  if (total == 0) return SARBP_OK;
  if (!Srnm || !ta || !tr || (p.Ntarget > 0 && !Ptarget))
    return fail(SARBP_ERR_INVALID_ARGUMENT, "Srnm, Ptarget, ta or tr is NULL");
  if (!(std::isfinite(p.c) && p.c > 0.0f && std::isfinite(p.lambda) && p.lambda != 0.0f && std::isfinite(p.Kr) &&
        std::isfinite(p.Tr) && std::isfinite(p.vr) && std::isfinite(p.H) && std::isfinite(p.La)))
    return fail(SARBP_ERR_INVALID_ARGUMENT, "SARParams c, lambda, Kr, Tr, vr, H or La invalid");
  EchoArgs a{};
  a.out = reinterpret_cast<float2*>(Srnm);
  a.tg = Ptarget;
  a.ta = ta;
  a.tr = tr;
  a.nfast = Nfast;
  a.chunks = (int)(((long long)Nfast + 64 * kEchoSamples - 1) / (64 * kEchoSamples));
  a.items = (long long)Mslow * a.chunks;
  a.ntarget = p.Ntarget;
  a.c = p.c;
  a.lambda = p.lambda;
  a.kr = p.Kr;
  a.tw = p.Tr;
  a.vr = p.vr;
  a.h = p.H;
  a.la_half = (double)p.La / 2.0;
  const long long blocks = (a.items + 3) / 4;
  const unsigned grid = (unsigned)(blocks < 65536 ? blocks : 65536);
  hipLaunchKernelGGL(echo_kernel, dim3(grid), dim3(256), 0, nullptr, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "echo_kernel launch");
  // Synchronous, as the original (BPA_CUDA_kernels.cu:88).
  if ((e = hipDeviceSynchronize()) != hipSuccess) return hip_fail(e, "hipDeviceSynchronize");
  return SARBP_OK;
}

}  // extern "C"
