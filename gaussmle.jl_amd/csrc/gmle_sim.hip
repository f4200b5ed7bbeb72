// gmle_sim.hip -- the simulator on the device: noisy ROI stacks for tests and
// benchmarks, as GaussMLE.jl's generate_roi_batch produces them
// (src/simulator.jl:35-345).
//
// Per pixel (i = row, j = column, 1-based), in Float32 as the reference:
//   expected = bg + photons * Phi(j; x, sigma_x) * Phi(i; y, sigma_y)
//              (src/simulator.jl:312-344; Phi as src/gausslib/baselibrary.jl:8-14,
//              astigmatic widths sigma0 sqrt(alpha((z -+ gamma) / d)))
//   Ideal camera: Poisson(expected) if expected > 0, else 0    (:259-275)
//   sCMOS: electrons = Poisson(expected * qe) + N(0, 1) * readnoise,
//          ADU = electrons / gain + offset                      (:281-307)
// Sensor maps are indexed the way the fitting kernel reads the variance map,
// [row = y_corner + i - 1, column = x_corner + j - 1] (src/unified_kernel.jl:
// 279-281); the reference simulator indexes [i + x_corner - 1, j + y_corner -
// 1] instead, which transposes them relative to the kernel.
// Random numbers come from Philox4x32-10 keyed by the seed and counted by
// (ROI, pixel, purpose), so the output depends on the seed only.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/gaussmle.h"
#include "gmle_args.hpp"
#include "gmle_host.hpp"
#include "gmle_rng.hpp"

namespace gmle {
namespace {

struct SimArgs {
  int model;
  float psf[8];
  int box;
  int64_t n;
  const float* params;   // per ROI: `stride` values, the model's parameters first
  int stride;
  int camera;
  const int32_t* xc;
  const int32_t* yc;
  const float* qe_map;   // (ny, nx) column-major, or null for the scalar
  const float* rn_map;
  const float* gain_map;
  const float* offset_map;
  int ny, nx;
  float qe, readnoise, gain, offset;
  uint64_t seed;
  int rois_per_wave;
  float* out;            // (box, box, n)
};

// integral_gaussian_1d (src/gausslib/baselibrary.jl:8-14) in Float32.
__host__ __device__ inline float pixel_integral(int k, float mu, float sigma) {
#pragma clang fp contract(off)
  const float s = sqrtf(0.5f / (sigma * sigma));
  return 0.5f * (erff(((float)k - mu + 0.5f) * s) - erff(((float)k - mu - 0.5f) * s));
}

__host__ __device__ inline float astig_alpha(float u, float A, float B) {
#pragma clang fp contract(off)
  return 1.0f + u * u + A * (u * u * u) + B * (u * u * u * u);
}

// Widths of one ROI's PSF on both axes.  The parameters come as values, and
// the model selects among values, not among pointers into the row.
__device__ __forceinline__ void sim_widths(const SimArgs& a, const float* t, float& sx, float& sy) {
#pragma clang fp contract(off)
  if (a.model == XYNB) {
    sx = sy = a.psf[0];
  } else if (a.model == XYNBS) {
    sx = sy = t[4];
  } else if (a.model == XYNBSXSY) {
    sx = t[4];
    sy = t[5];
  } else {
    const float z = t[2];
    sx = a.psf[0] * sqrtf(astig_alpha((z - a.psf[6]) / a.psf[7], a.psf[2], a.psf[4]));
    sy = a.psf[1] * sqrtf(astig_alpha((z + a.psf[6]) / a.psf[7], a.psf[3], a.psf[5]));
  }
}

// ---------------------------------------------------------------------------
// sample_poisson (gmle_rng.hpp) a Philox block at a time, in Float32 with
// guard bands.  Every comparison of the Float64 sampler is evaluated in Float32
// together with a bound on its rounding; a lane whose comparison falls inside
// the bound is `unsure` and its pixel is drawn again by the Float64 sampler
// itself, so the counts are the Float64 sampler's.  Uniforms are compared as
// the 32-bit integers they come from wherever both sides are uniforms or
// constants, which is exact.
// ---------------------------------------------------------------------------
constexpr float kFastMean = 1.0e6f;    // counts above 2^20: drawn in Float64
constexpr uint32_t kFastSteps = 200;   // passes on one pixel before the Float64 sampler takes over

struct PoissonState {
  bool knuth;
  float mean;
  float limit, prod, k;    // mean < 10: exp(-mean), product so far, draws so far - 1
  float b, ia, vr;         // mean >= 10: PTRS constants b, a and vr
};

__device__ __forceinline__ void poisson_start(float mean, PoissonState& s) {
  s.mean = mean;
  s.knuth = mean < 10.0f;
  s.limit = __builtin_amdgcn_exp2f(mean * -1.44269504f);
  s.prod = 1.0f;
  s.k = -1.0f;
  s.b = fmaf(2.53f, __builtin_amdgcn_sqrtf(mean), 0.931f);
  s.ia = fmaf(0.02483f, s.b, -0.059f);
  s.vr = fmaf(-3.6224f, __builtin_amdgcn_rcpf(s.b - 2.0f), 0.9277f);
}

// (x + 1/2) 2^-32, relative error 2^-24
__device__ __forceinline__ float unit(uint32_t x) { return fmaf((float)x, 0x1p-32f, 0x1p-33f); }

// Four uniforms of the multiplication method.  The product carries at most
// 2^-23 relative error per factor and the limit 2e-6, far within 2e-5 for the
// few dozen factors a mean below 10 takes.  The products fall, so the number
// of factors is one more than the products above the limit.
__device__ __forceinline__ void knuth_block(PoissonState& s, const U32x4& x, bool& done, bool& unsure) {
  const float p0 = s.prod * unit(x.v[0]), p1 = p0 * unit(x.v[1]), p2 = p1 * unit(x.v[2]), p3 = p2 * unit(x.v[3]);
  s.k += 1.0f + ((p0 > s.limit ? 1.0f : 0.0f) + (p1 > s.limit ? 1.0f : 0.0f) + (p2 > s.limit ? 1.0f : 0.0f));
  s.prod = p3;
  done = p3 <= s.limit;
  const float near = fminf(fminf(fabsf(p0 - s.limit), fabsf(p1 - s.limit)),
                           fminf(fabsf(p2 - s.limit), fabsf(p3 - s.limit)));
  unsure = near <= 2e-5f * s.limit;
}

// One attempt of the transformed rejection method, its steps in the order
// that needs the least: the tail rejection is exact on the integers.
__device__ __forceinline__ void ptrs_step(const PoissonState& s, uint32_t xu, uint32_t xv, bool& done, bool& unsure,
                                          float& value) {
  constexpr uint32_t kUs013 = (uint32_t)(0.013 * 4294967296.0 - 0.5);        // us < 0.013  <=>  w <= kUs013
  constexpr uint32_t kUs07 = (uint32_t)(0.07 * 4294967296.0 - 0.5) + 1u;     // us >= 0.07  <=>  w >= kUs07
  const bool neg = xu < 0x80000000u;
  const uint32_t w = neg ? xu : 0xFFFFFFFFu - xu;   // us = (w + 1/2) 2^-32
  if (w <= kUs013 && xv > w) return;                // rejected whatever k is
  const float us = unit(w);
  const uint32_t h = neg ? 0x7FFFFFFFu - xu : xu - 0x80000000u;   // |U| = (h + 1/2) 2^-32
  const float U = neg ? -unit(h) : unit(h);
  const float rus = __builtin_amdgcn_rcpf(us);
  // k = floor((2 a / us + b) U + mean + 0.43), the whole part of the mean
  // apart; the product's relative error is below 1e-6
  const float x0 = fmaf(2.0f * s.ia, rus, s.b) * U;
  const float mi = floorf(s.mean);
  const float f = x0 + ((s.mean - mi) + 0.43f);
  const float fl = floorf(f);
  const float k = mi + fl;
  const float band = fmaf(fabsf(x0), 3e-6f, 1e-6f);
  bool doubt = f - fl <= band || f - fl >= 1.0f - band;
  const float v = unit(xv);
  if (w >= kUs07) {
    doubt = doubt || fabsf(v - s.vr) <= 2e-6f;
    if (v <= s.vr) {
      done = true;
      unsure = unsure || doubt;
      value = k;
      return;
    }
  }
  if (doubt) {   // k itself is unsure
    done = unsure = true;
    return;
  }
  if (k < 0.0f) return;
  // log V + log(1/alpha) - log(a/us^2 + b) against log of the Poisson
  // probability of k.  The latter by its deviance k log(k/m) - (k - m), from
  // v = (k - m)/(k + m) where the two are close (Loader, "Fast and accurate
  // computation of binomial probabilities", 2000), and Stirling's series.
  const float invalpha = fmaf(1.1328f, __builtin_amdgcn_rcpf(s.b - 3.4f), 1.1239f);
  const float ln2 = 0.693147181f;
  const float q = fmaf(s.ia * rus, rus, s.b);
  const float lhs = ln2 * (__builtin_amdgcn_logf(v * invalpha) - __builtin_amdgcn_logf(q));
  const float m = s.mean, d = k - m;
  float rhs, eps = 4e-5f;
  if (k >= 4.0f) {
    const float r = d * __builtin_amdgcn_rcpf(k + m);
    const float r2 = r * r;
    float dev;
    if (r2 < 0.01f) {
      dev = fmaf(d, r, 2.0f * k * r * r2 * fmaf(r2, fmaf(r2, fmaf(r2, 1.0f / 9.0f, 1.0f / 7.0f), 0.2f), 1.0f / 3.0f));
      eps = fmaf(dev, 4e-6f, eps);
    } else {
      dev = fmaf(k, ln2 * __builtin_amdgcn_logf(k * __builtin_amdgcn_rcpf(m)), -d);
      eps = fmaf(k + m, 2e-6f, eps);
    }
    const float ik = __builtin_amdgcn_rcpf(k), ik2 = ik * ik;
    rhs = -dev - 0.5f * ln2 * __builtin_amdgcn_logf(6.28318531f * k) -
          ik * fmaf(ik2, fmaf(ik2, 1.0f / 1260.0f, -1.0f / 360.0f), 1.0f / 12.0f);
  } else {
    const float lfact = k < 2.0f ? 0.0f : k < 3.0f ? 0.693147181f : 1.79175947f;
    rhs = fmaf(k, ln2 * __builtin_amdgcn_logf(m), -m) - lfact;
    eps = fmaf(m, 4e-6f, eps);
  }
  if (fabsf(lhs - rhs) <= eps) {
    done = unsure = true;
  } else if (lhs < rhs) {
    done = true;
    value = k;
  }
}

// The Float64 samplers, out of line: few pixels (sCMOS read noise apart) reach
// them, and inlined their registers would halve the waves of the kernel.
__device__ __noinline__ float poisson64(uint64_t seed, int64_t roi, uint32_t pixel, float mean) {
  Stream shot(seed, roi, pixel, 0u);
  return (float)sample_poisson(shot, (double)mean);
}
__device__ __noinline__ float normal64(uint64_t seed, int64_t roi, uint32_t pixel) {
  Stream read(seed, roi, pixel, 1u);
  return (float)sample_normal(read);
}

// ---------------------------------------------------------------------------
// One wave draws a.rois_per_wave consecutive ROIs.
//
// What bounds it: instruction issue of Philox and the samplers.  A pixel takes
// one Philox block where the background is above 10 counts and up to eight
// below, so a wave that drew 64 pixels at a time waited for its slowest one.
// Instead every pass of the loop computes one Philox block per lane, and a
// lane whose pixel is finished takes the next pixel of the wave's list (its
// rank among the finished lanes gives the index), so that no lane idles until
// the list runs out.  The pixel integrals of each ROI and axis are computed
// once per ROI into LDS (2 box of them instead of 2 box^2).
// gfx950, 1,048,576 ROIs of 11 px, backgrounds 1-20: 7.78 -> 1.28 ms per call
// at 500-5000 photons, the same counts bit for bit.  Two
// attempts per pass instead of one: 1.57 ms.  Six waves per SIMD are asked
// for: 2, 4 and 8 gave 2.59, 1.76 and 1.57 ms against 1.57 for 6, before the
// one-attempt pass.
// ---------------------------------------------------------------------------
constexpr int kWavePixels = 2048;   // pixels of one wave's list, about: 32 per lane
constexpr int kWaveRois = 64;       // at most
constexpr int kTableFloats = 832;   // >= rois (2 box + 2) for every box (64 ROIs of 5 px, 57 of 6 px)

__host__ __device__ inline int sim_rois_per_wave(int box, int64_t n) {
  const int full = (kWavePixels + box * box - 1) / (box * box);
  const int64_t spread = (n + 8191) / 8192;   // small batches: one wave per slot of the chip first
  const int64_t r = full < spread ? full : spread;
  return (int)(r < 1 ? 1 : r > kWaveRois ? kWaveRois : r);
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6))) void sim_kernel(SimArgs a) {
#pragma clang fp contract(off)   // Float32 expected counts as written, like the reference
  __shared__ float table[kTableFloats];   // per ROI: Phi_x (box), Phi_y (box), photons, background
  const int lane = threadIdx.x;
  const int B = a.box, BB = a.box * a.box, row = 2 * B + 2;
  const int64_t first = (int64_t)blockIdx.x * a.rois_per_wave;
  const int rois = (int)min((int64_t)a.rois_per_wave, a.n - first);
  for (int e = lane; e < rois * row; e += 64) {
    const int k = e / row, c = e - k * row;
    const float* th = a.params + (first + k) * a.stride;
    const int np = a.stride < 6 ? a.stride : 6;
    float t[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) t[q] = q < np ? th[q] : 0.0f;
    const bool astig = a.model == ASTIG;
    float sx, sy;
    sim_widths(a, t, sx, sy);
    const bool on_x = c < B;
    const float phi = pixel_integral(on_x ? c + 1 : c - B + 1, on_x ? t[0] : t[1], on_x ? sx : sy);
    table[e] = c < 2 * B ? phi : c == 2 * B ? (astig ? t[3] : t[2]) : (astig ? t[4] : t[3]);
  }
  __syncthreads();

  const int total = rois * BB;
  int next = 64;       // first pixel nobody has taken (the same on every lane)
  int e = lane;        // this lane's pixel
  bool live = e < total;
  bool fresh = live;   // the pixel has to be set up
  int k = 0, p = 0;
  uint32_t step = 0;   // passes on this pixel: Philox blocks (mean < 10) or attempts, two of them from each block
  bool fixed = false;  // the count is `value` already
  float value = 0.0f;
  int64_t pix = 0;     // sCMOS: index into the sensor maps
  PoissonState st{};
  while (__ballot(live)) {
    if (fresh) {
      k = e / BB;
      p = e - k * BB;
      const int j = p / B, i = p - j * B;   // column, row (0-based)
      const float* r = table + k * row;
      float mean = r[2 * B + 1] + r[2 * B] * r[j] * r[B + i];
      fixed = false;
      value = 0.0f;
      if (a.camera == SCMOS) {
        const int cy = a.yc[first + k], cx = a.xc[first + k];
        if (cy < 1 || cx < 1 || cy > a.ny - B + 1 || cx > a.nx - B + 1) {   // off the sensor
          fixed = true;
          value = __builtin_nanf("");
        } else {
          pix = (int64_t)(cy - 1 + i) + (int64_t)a.ny * (int64_t)(cx - 1 + j);
          mean = mean * (a.qe_map ? a.qe_map[pix] : a.qe);
        }
      }
      if (!(mean > 0.0f)) fixed = true;
      step = 0;
      poisson_start(mean, st);
      fresh = false;
    }
    const uint64_t roi = (uint64_t)(first + k);
    const U32x4 x = philox4x32_10(U32x4{{(uint32_t)p, (uint32_t)roi, (uint32_t)(roi >> 32),
                                         st.knuth ? step : step >> 1}},
                                  (uint32_t)a.seed, (uint32_t)(a.seed >> 32));
    bool done = fixed, unsure = false;
    if (!fixed) {
      if (st.mean > kFastMean || step >= kFastSteps) {
        done = unsure = true;
      } else if (st.knuth) {
        knuth_block(st, x, done, unsure);
        value = st.k;
      } else {
        const bool second = step & 1;
        ptrs_step(st, second ? x.v[2] : x.v[0], second ? x.v[3] : x.v[1], done, unsure, value);
      }
      ++step;
      if (live && unsure) {
        value = poisson64(a.seed, first + k, (uint32_t)p, st.mean);
        done = true;
      }
    }
    done = done && live;
    if (done) {
      float out = value;
      if (a.camera == SCMOS && out == out) {
        const float rn = a.rn_map ? a.rn_map[pix] : a.readnoise;
        const float gain = a.gain_map ? a.gain_map[pix] : a.gain;
        const float offset = a.offset_map ? a.offset_map[pix] : a.offset;
        const float total_e = out + normal64(a.seed, first + k, (uint32_t)p) * rn;
        out = total_e / gain + offset;
      }
      a.out[first * BB + e] = out;
    }
    const uint64_t finished = __ballot(done);
    if (done) {
      e = next + __builtin_amdgcn_mbcnt_hi((uint32_t)(finished >> 32),
                                           __builtin_amdgcn_mbcnt_lo((uint32_t)finished, 0u));
      live = fresh = e < total;
    }
    next += __popcll(finished);
  }
}

int check_sim(int model, const float* psf, int box, int64_t n, int stride, int camera, int ny, int nx) {
  if (n <= 0) return fail(GMLE_ERR_ARG, "n_rois must be > 0");
  if (model < XYNB || model > ASTIG) return fail(GMLE_ERR_ARG, "unknown PSF model %d", model);
  if ((model == XYNB || model == ASTIG) && !psf) return fail(GMLE_ERR_ARG, "psf must not be NULL for this model");
  if (box < kMinBox || box > kMaxBox) return fail(GMLE_ERR_ARG, "box size %d out of range", box);
  if (stride < n_params(model)) return fail(GMLE_ERR_ARG, "stride %d < %d parameters", stride, n_params(model));
  if (camera != IDEAL && camera != SCMOS) return fail(GMLE_ERR_ARG, "camera must be 0 (ideal) or 1 (sCMOS)");
  if (camera == SCMOS && (ny < box || nx < box)) return fail(GMLE_ERR_ARG, "sensor %d x %d smaller than the box", ny, nx);
  return GMLE_OK;
}

}  // namespace
}  // namespace gmle

using namespace gmle;

extern "C" {

void gmle_philox4x32_10(const uint32_t* counter, const uint32_t* key, uint32_t* out) {
  const U32x4 r = philox4x32_10(U32x4{{counter[0], counter[1], counter[2], counter[3]}}, key[0], key[1]);
  for (int q = 0; q < 4; ++q) out[q] = r.v[q];
}

int gmle_simulate_device(int model, const float* psf, int box, int64_t n_rois, const float* d_params, int stride,
                         int camera, const int32_t* d_x_corners, const int32_t* d_y_corners, const float* d_qe,
                         const float* d_readnoise, const float* d_gain, const float* d_offset, int ny, int nx,
                         float qe, float readnoise, float gain, float offset, uint64_t seed, float* d_out,
                         void* stream) {
  int rc = check_sim(model, psf, box, n_rois, stride, camera, ny, nx);
  if (rc != GMLE_OK) return rc;
  if (!d_params || !d_out) return fail(GMLE_ERR_ARG, "params and out must not be NULL");
  if (camera == SCMOS && (!d_x_corners || !d_y_corners)) return fail(GMLE_ERR_ARG, "sCMOS needs ROI corners");
  if (camera == SCMOS && (!(gain != 0.0f) && !d_gain)) return fail(GMLE_ERR_ARG, "gain must be non-zero");
  SimArgs a{};
  a.model = model;
  // XYNB reads one float (sigma), ASTIG eight, the others none, as gmle_fit.
  if (model == XYNB) a.psf[0] = psf[0];
  if (model == ASTIG)
    for (int q = 0; q < 8; ++q) a.psf[q] = psf[q];
  a.box = box;
  a.n = n_rois;
  a.params = d_params;
  a.stride = stride;
  a.camera = camera;
  a.xc = d_x_corners;
  a.yc = d_y_corners;
  a.qe_map = d_qe;
  a.rn_map = d_readnoise;
  a.gain_map = d_gain;
  a.offset_map = d_offset;
  a.ny = ny;
  a.nx = nx;
  a.qe = qe;
  a.readnoise = readnoise;
  a.gain = gain;
  a.offset = offset;
  a.seed = seed;
  a.out = d_out;
  a.rois_per_wave = sim_rois_per_wave(box, n_rois);
  const int64_t blocks = (n_rois + a.rois_per_wave - 1) / a.rois_per_wave;
  hipLaunchKernelGGL(sim_kernel, dim3((unsigned)blocks), dim3(64), 0, (hipStream_t)stream, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GMLE_OK : hip_fail(e, "kernel launch");
}

}  // extern "C"
