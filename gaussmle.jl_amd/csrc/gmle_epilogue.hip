// gmle_epilogue.hip -- per-emitter result conversion on the device.
//
// GaussMLE.jl finishes every fit on the host, one emitter at a time:
//   * goodness of fit: chi2 = -2 LLR with box^2 - P degrees of freedom,
//     p = 1 - Float32(cdf(Chisq(df), chi2))            (src/interface.jl:265-275)
//   * ROI -> camera coordinates: x_corner + x_roi - 1  (src/roi_batch.jl:29-34)
//   * camera -> microns: (x_camera - 1) * pixel_size, uncertainties and fitted
//     widths times the pixel size, z and its uncertainty unscaled
//                                                      (src/roi_batch.jl:125-302)
// gmle_epilogue_device does all of it for a whole batch in one launch, in the
// same arithmetic types (Float32 values, Float64 pixel size, Float64 CDF).
//
// The chi-square CDF is the regularized lower incomplete gamma function
// P(a, x), a = df/2, x = chi2/2, in Float64.  df is a whole number, so for
// x >= a/2 it is 1 - Q(a, x) with Q as the finite sum that the recurrence
// Q(a, x) = Q(a - 1, x) + x^(a-1) e^-x / Gamma(a) gives (DLMF 8.8.6),
//   Q(a, x) = x^(a-1) e^-x / Gamma(a) [1 + (a-1)/x + (a-1)(a-2)/x^2 + ...]
//             + (df odd) erfc(sqrt x),
// floor(df/2) positive terms that need no division.  Below a/2 (a fit far
// better than its noise) the terms would first grow by many orders of
// magnitude; there the power series
//   P(a, x) = x^a e^-x / Gamma(a + 1) * sum_n x^n / ((a + 1) ... (a + n))
// halves its terms at least and ends within 53.
//
// What bounds it: Float64 issue.  With the series below a + 1 and Legendre's
// continued fraction above, a wave ran both branches with one and two
// Float64 divisions per term.  A fit's chi2 lies within a few sqrt(2 df) of
// df, so all its lanes now take the finite sum, about three Float64 operations
// per term.  1,048,576 XYNBS results of 13 px on gfx950: 114 -> 27 us per call, of
// which 92 MB in and out take 20 us at the rate of a large copy.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "../../include/gaussmle.h"
#include "gmle_args.hpp"
#include "gmle_host.hpp"

namespace gmle {
namespace {

// Relative stopping tolerance of both sums: below half a Float64 ulp.
constexpr double kTol = 1e-16;
// erfc(sqrt x) is below 1e-17, and drops out of 1 - Q, from here on.
constexpr double kErfcEnd = 37.0;

// P(df/2, x); lg = lgamma(df/2).
// x <= 0 gives 0 (a chi^2 below zero, from an LLR rounded just above zero,
// has CDF 0 as in Distributions.jl, whose gamma CDF clamps x at 0); NaN stays NaN.
__host__ __device__ inline double gamma_p(int df, double x, double lg) {
  const double a = 0.5 * df;
  if (x != x) return x;
  if (!(x > 0.0)) return 0.0;
  if (isinf(x)) return 1.0;
  const double lx = log(x);
  if (x < 0.5 * a) {
    const double lead = exp(-x + a * lx - lg);
    double ap = a, del = 1.0 / a, sum = del;
    for (int n = 0; n < 1000; ++n) {
      ap += 1.0;
      del *= x / ap;
      sum += del;
      if (del < sum * kTol) break;
    }
    return sum * lead;
  }
  const int terms = df >> 1;
  const double ix = 1.0 / x;
  double c = a, t = 1.0, s = terms > 0 ? 1.0 : 0.0;
  int k = 1;
  // Four terms per step, t (r1 + r1 r2 + r1 r2 r3 + r1 r2 r3 r4) with
  // r_j = (c - j) / x: 12 operations instead of 16, and a shorter chain.  The
  // test holds only past the largest term, where they fall.
  for (; k + 4 <= terms; k += 4) {
    const double r0 = c * ix;
    const double r1 = r0 - ix, r2 = fma(-2.0, ix, r0), r3 = fma(-3.0, ix, r0), r4 = fma(-4.0, ix, r0);
    const double t1 = t * r1;
    s = fma(t1, fma(r2, fma(r3, 1.0 + r4, 1.0), 1.0), s);
    t = t1 * r2 * (r3 * r4);
    c -= 4.0;
    if (t < s * kTol) {
      k = terms;
      break;
    }
  }
  for (; k < terms; ++k) {
    c -= 1.0;
    t *= c * ix;
    s += t;
  }
  double q = s * exp(-x + (a - 1.0) * lx - lg);
  if ((df & 1) && x < kErfcEnd) q += erfc(sqrt(x));
  return q < 1.0 ? 1.0 - q : 0.0;
}

struct EpilogueArgs {
  int64_t n;
  int model, box;                 // used when models / boxes are null
  const int8_t* models;
  const int8_t* boxes;
  int stride;                     // params / crlb values per ROI
  const float* params;
  const float* crlb;
  const float* llr;
  const int32_t* xc;              // null: corners of fit(Array), x = 1 + k box, y = 1
  const int32_t* yc;
  double psx, psy;
  double lg;                      // lgamma(df/2) of (model, box), when both are the launch's
  float* out;                     // (kOut, n)
};

constexpr int kOut = 10;
constexpr int kBlock = 256;

// ROI k's results (kOut values).
__device__ __forceinline__ void epilogue_one(const EpilogueArgs& a, int64_t k, float* o) {
  const int model = a.models ? a.models[k] : a.model;
  const int box = a.boxes ? a.boxes[k] : a.box;
  const float qnan = __builtin_nanf("");
  if (model < XYNB || model > ASTIG || box < kMinBox || box > kMaxBox) {
#pragma unroll
    for (int q = 0; q < kOut; ++q) o[q] = qnan;
    return;
  }
  const float* p = a.params + k * a.stride;
  const float* u = a.crlb + k * a.stride;
  const int32_t xc = a.xc ? a.xc[k] : (int32_t)(1 + k * box);
  const int32_t yc = a.yc ? a.yc[k] : 1;
  // roi_to_camera_coords: Int32 corner + Float32 ROI coordinate - 1, in Float32
  const float xcam = ((float)xc + p[0]) - 1.0f;
  const float ycam = ((float)yc + p[1]) - 1.0f;
  o[0] = (float)((double)(xcam - 1.0f) * a.psx);
  o[1] = (float)((double)(ycam - 1.0f) * a.psy);
  o[2] = (float)((double)u[0] * a.psx);
  o[3] = (float)((double)u[1] * a.psy);
  const int P = n_params(model);
  const float chi2 = -2.0f * a.llr[k];
  const int df = box * box - P;
  const double lg = (a.models || a.boxes) ? lgamma(0.5 * (double)df) : a.lg;
  const double cdf = gamma_p(df, 0.5 * (double)chi2, lg);
  o[4] = 1.0f - (float)cdf;
  o[5] = o[6] = o[7] = o[8] = qnan;
  if (model == XYNBS) {   // one width, in x pixels (src/roi_batch.jl, Emitter2DFitSigma)
    o[5] = o[6] = (float)((double)p[4] * a.psx);
    o[7] = o[8] = (float)((double)u[4] * a.psx);
  } else if (model == XYNBSXSY) {
    o[5] = (float)((double)p[4] * a.psx);
    o[6] = (float)((double)p[5] * a.psy);
    o[7] = (float)((double)u[4] * a.psx);
    o[8] = (float)((double)u[5] * a.psy);
  }
  o[9] = chi2;
}

// One thread per ROI; a block's results go through LDS, so that the 40 bytes
// of each ROI leave in whole cache lines.  The LDS row is odd (kOut + 1), so
// a wave's writes meet different banks.
__global__ __launch_bounds__(kBlock) void epilogue_kernel(EpilogueArgs a) {
  __shared__ float rows[kBlock * (kOut + 1)];
  const int t = threadIdx.x;
  const int64_t first = (int64_t)blockIdx.x * kBlock;
  const int here = (int)min((int64_t)kBlock, a.n - first);
  if (t < here) {
    float o[kOut];
    epilogue_one(a, first + t, o);
#pragma unroll
    for (int q = 0; q < kOut; ++q) rows[t * (kOut + 1) + q] = o[q];
  }
  __syncthreads();
  float* dst = a.out + first * kOut;
#pragma unroll
  for (int i = 0; i < kOut; ++i) {
    const int e = t + i * kBlock;
    if (e < here * kOut) dst[e] = rows[e + e / kOut];
  }
}

// lgamma without the C library's process-wide sign.
double lgamma_of(double x) {
  int sign;
  return lgamma_r(x, &sign);
}

}  // namespace
}  // namespace gmle

using namespace gmle;

extern "C" {

int gmle_epilogue_device(int64_t n_rois, int model, int box, const int8_t* d_models, const int8_t* d_boxes,
                         int stride, const float* d_params, const float* d_crlb, const float* d_llr,
                         const int32_t* d_x_corners, const int32_t* d_y_corners, double pixel_size_x,
                         double pixel_size_y, float* d_out, void* stream) {
  if (n_rois <= 0) return fail(GMLE_ERR_ARG, "Input data array is empty");
  if (!d_params || !d_crlb || !d_llr || !d_out) return fail(GMLE_ERR_ARG, "device pointers must not be NULL");
  if (!d_models && (model < XYNB || model > ASTIG)) return fail(GMLE_ERR_ARG, "unknown PSF model %d", model);
  if (!d_boxes && (box < kMinBox || box > kMaxBox)) return fail(GMLE_ERR_ARG, "box size %d out of range", box);
  if ((d_x_corners == nullptr) != (d_y_corners == nullptr))
    return fail(GMLE_ERR_ARG, "pass both corner arrays or neither");
  const int pmax = d_models ? 6 : n_params(model);
  if (stride < pmax) return fail(GMLE_ERR_ARG, "stride %d is smaller than the parameter count %d", stride, pmax);
  if (!(pixel_size_x > 0.0) || !(pixel_size_y > 0.0)) return fail(GMLE_ERR_ARG, "pixel sizes must be > 0");
  EpilogueArgs a{n_rois, model, box, d_models, d_boxes, stride, d_params, d_crlb, d_llr, d_x_corners, d_y_corners,
                 pixel_size_x, pixel_size_y, 0.0, d_out};
  if (!d_models && !d_boxes) a.lg = lgamma_of(0.5 * (box * box - n_params(model)));
  const unsigned blocks = (unsigned)((n_rois + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(epilogue_kernel, dim3(blocks), dim3(kBlock), 0, (hipStream_t)stream, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GMLE_OK : hip_fail(e, "kernel launch");
}

// The chi-square survival function as the epilogue computes it, on the host
// (1 - Float32(P(df/2, chi2/2))): for callers and tests without a device.
float gmle_chi2_pvalue(float chi2, int df) {
  if (df <= 0) return __builtin_nanf("");
  return 1.0f - (float)gamma_p(df, 0.5 * (double)chi2, lgamma_of(0.5 * df));
}

}  // extern "C"
