// gmle_fit_kernel.hpp -- the per-ROI maximum-likelihood fitting kernel for gfx950.
//
// One kernel specialisation per (PSF model, camera, box size N, lanes per ROI L,
// precision).  It replaces GaussMLE.jl's unified_gaussian_mle_kernel!
// (src/unified_kernel.jl:285-434) together with everything it inlines:
// compute_pixel_derivatives (src/psf_derivatives.jl:6-187), the pixel-integrated
// Gaussian and its derivatives (src/gausslib/baselibrary.jl:8-67), the camera
// likelihood terms (src/camera_models.jl:19-96) and apply_constraints!
// (src/constraints.jl:172-177).
//
// Work mapping (wave64, one wave per workgroup):
//   * L lanes (1, 2, 4, 8 or 16, inside one DPP row) share one ROI; 64/L ROIs
//     per wave.
//   * Lane r of a group owns the contiguous column block [r*CB, r*CB + CB) with
//     CB = ceil(N/L); its CB*N pixels (and sCMOS variances) are loaded once and
//     stay in VGPRs for every Newton iteration and the final pass.
//   * The model is separable: value = bg + N*Phix[j]*Phiy[i].  Per iteration
//     each axis needs only N+1 edge evaluations (one erf and one exp each)
//     instead of the reference's 4 erf + 4-8 exp per pixel, and every gradient,
//     diagonal-Hessian and Fisher term is a product of a column value, a row
//     value and a pixel weight.  A pixel therefore only feeds a few weighted
//     column and row sums (accumulate); the tables multiply those sums.  Row
//     values are shared through LDS (publish_rows).  The P gradient and P
//     diagonal-Hessian values are summed across the L lanes with DPP permutes.
//   * The Newton update (exact division, step clamp, box clamp) is replicated
//     on the L lanes so they stay bit-identical.
//   * PREC_FP32 computes the final pass (LLR, full Fisher matrix, inversion,
//     CRLB) in Float32 like the reference; PREC_MIXED recomputes the model and
//     derivatives at the final estimate in Float64 and does the LLR, Fisher
//     accumulation and inversion in Float64.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "gmle_args.hpp"
#include "gmle_device.hpp"
#include "gmle_erf.hpp"

namespace gmle {

// ---------------------------------------------------------------------------
// Model traits.  EXTRA: 0 none (XYNB), 1 one sigma on both axes (XYNBS),
// 2 separate sigma per axis (XYNBSXSY), 3 astigmatic z (chain rule through
// sigma_x(z), sigma_y(z)).
// ---------------------------------------------------------------------------
template <int MODEL> struct MT;
template <> struct MT<XYNB> {
  static constexpr int P = 4, IX = 0, IY = 1, IN = 2, IBG = 3, IE1 = -1, IE2 = -1, EXTRA = 0;
};
template <> struct MT<XYNBS> {
  static constexpr int P = 5, IX = 0, IY = 1, IN = 2, IBG = 3, IE1 = 4, IE2 = -1, EXTRA = 1;
};
template <> struct MT<XYNBSXSY> {
  static constexpr int P = 6, IX = 0, IY = 1, IN = 2, IBG = 3, IE1 = 4, IE2 = 5, EXTRA = 2;
};
template <> struct MT<ASTIG> {
  static constexpr int P = 5, IX = 0, IY = 1, IN = 3, IBG = 4, IE1 = 2, IE2 = -1, EXTRA = 3;
};

// ---------------------------------------------------------------------------
// Scalar math per arithmetic type.
// ---------------------------------------------------------------------------
template <class T> struct DM;
template <> struct DM<float> {
  // Axis scales carry sqrt(log2 e): t * s is v = k u of gmle_erf.hpp, so the
  // Gaussian exp(-u^2) is exp2(-v^2).
  // exp(-u^2), and the edge's signed erfc and half-sign for the pixel
  // integrals (gmle_erf.hpp), which reuse the Gaussian
  static __device__ __forceinline__ void erf_gauss(float t, float s, float& se, float& hs, float& g) {
    const float v = t * s;
    g = fast_exp2((-v) * v);
    erf_edge(v, g, se, hs);
  }
  static __device__ __forceinline__ float inv_sqrt_2pi() { return kInvSqrt2Pi; }
  // a / b for the per-iteration width and axis constants: one v_rcp_f32
  // (1 ulp) and a multiply instead of the ~10-instruction IEEE division.
  static __device__ __forceinline__ float div(float a, float b) { return a * fast_rcp(b); }
  // 1 / b: v_rcp_f32 and one Newton step (correctly rounded but for rare last
  // bits), left out where the reciprocal is not finite.
  static __device__ __forceinline__ float inv(float b) {
    const float r = fast_rcp(b);
    const float e = fmaf(-b, r, 1.f);
    return fabsf(e) < 1.f ? fmaf(e, r, r) : r;
  }
  // The scale t -> v of an edge, k / (|sigma| sqrt 2): the reference's
  // sqrt(1 / (2 sigma^2)), which a negative width (bounds below 0 allow one)
  // does not turn round.
  static __device__ __forceinline__ float erf_rate(float, float inv_s) { return fabsf(inv_s) * kErfRate; }
};
template <> struct DM<double> {
  // Float64 keeps the reference's erf difference: its cancellation (~1e-16
  // absolute) is negligible, and tails that erf rounds to exactly +-1 stay
  // exactly 0 as in the reference.  se = -erf(u), hs = 0 in pixel_integral.
  static __device__ __forceinline__ void erf_gauss(double t, double s, double& se, double& hs, double& g) {
    const double u = t * s;
    g = exp(-(u * u));
    se = -erf(u);
    hs = 0.0;
  }
  static __device__ __forceinline__ double inv_sqrt_2pi() { return kInvSqrt2PiD; }
  static __device__ __forceinline__ double div(double a, double b) { return a / b; }
  static __device__ __forceinline__ double inv(double b) { return 1.0 / b; }
  static __device__ __forceinline__ double erf_rate(double sigma, double) { return sqrt(0.5 / (sigma * sigma)); }
};

// ---------------------------------------------------------------------------
// Per-axis tables for M consecutive pixels starting at 0-based index `first`
// (pixel k covers [k+1/2, k+3/2] in the reference's 1-based coordinates).  For
// pixel p with lower edge lo and upper edge hi (t = edge - mu):
//   phi = (erf(t_hi*s) - erf(t_lo*s)) / 2                  baselibrary.jl:8-14
//         (formed from signed complements, pixel_integral in gmle_erf.hpp)
//   D   = c (g_hi - g_lo),  c = -N/(sqrt(2pi) sigma)        baselibrary.jl:21-33
//   D2  = c/sigma^2 (t_hi g_hi - t_lo g_lo)
//   S   = c/sigma   (t_hi g_hi - t_lo g_lo)                 baselibrary.jl:40-52
//   SS  = -2/sigma S - N/(sqrt(2pi) sigma^5) (t_hi^3 g_hi - t_lo^3 g_lo)
// with g = exp(-t^2/(2 sigma^2)).  Pixel-level derivatives are these times the
// other axis' phi: dudt_x = D[j] phiy[i], d2udt2_x = D2[j] phiy[i], and the
// sigma derivative of one axis is S[j] phiy[i] (second: SS[j] phiy[i]).
// ---------------------------------------------------------------------------
template <class T, int M> struct AxisTab {
  T phi[M], D[M], D2[M], S[M], SS[M];
};

template <class T, int M, bool SIG>
__device__ __forceinline__ void axis_tables(T mu, T sigma, T nph, int first, AxisTab<T, M>& tb) {
  const T inv_s = DM<T>::div(T(1), sigma);
  static_assert(sizeof(T) == 8, "the Float32 edges are scaled (erf_rate)");
  const T s_erf = sqrt(DM<T>::div(T(0.5), sigma * sigma));
  const T c = -nph * DM<T>::inv_sqrt_2pi() * inv_s;
  const T c2 = c * inv_s * inv_s;
  const T cs = c * inv_s;
  const T css = c2 * inv_s * inv_s;
  const T m2s = T(-2) * inv_s;
  T se_prev = T(0), hs_prev = T(0), g_prev = T(0), tg_prev = T(0), t3g_prev = T(0);
#pragma unroll
  for (int e = 0; e <= M; ++e) {
    const T t = (T(first + e) + T(0.5)) - mu;
    T se, hs, g;
    DM<T>::erf_gauss(t, s_erf, se, hs, g);
    const T tg = t * g;
    const T t3g = SIG ? t * t * tg : T(0);
    if (e > 0) {
      const int p = e - 1;
      tb.phi[p] = pixel_integral<T>(se_prev, hs_prev, se, hs);
      tb.D[p] = c * (g - g_prev);
      const T w = tg - tg_prev;
      tb.D2[p] = c2 * w;
      if (SIG) {
        tb.S[p] = cs * w;
        tb.SS[p] = m2s * tb.S[p] + css * (t3g - t3g_prev);
      }
    }
    se_prev = se;
    hs_prev = hs;
    g_prev = g;
    tg_prev = tg;
    t3g_prev = t3g;
  }
}

// Axis constants of axis_tables() and single-edge evaluation, for computing
// one pixel's tables from its two edges on the fly (column side).
// The constants past c and 1/sigma are formed where they are used: an
// iteration needs them only after its pixel loop, where four values held
// across the loop would take registers from it.
template <class T> struct AxisK {
  T mu, s_erf, c, inv_s;
  __device__ __forceinline__ T c2() const { return c * inv_s * inv_s; }
  __device__ __forceinline__ T cs() const { return c * inv_s; }
  __device__ __forceinline__ T css() const { return c2() * inv_s * inv_s; }
  __device__ __forceinline__ T m2s() const { return T(-2) * inv_s; }
};
template <class T> struct Edge {
  T se, hs, g, tg, t3g;   // signed erfc, half-sign (gmle_erf.hpp), Gaussian, t g, t^3 g
};
template <class T>
__device__ __forceinline__ AxisK<T> axis_consts(T mu, T sigma, T nph) {
  AxisK<T> k;
  k.inv_s = DM<T>::inv(sigma);
  k.mu = mu;
  k.s_erf = DM<T>::erf_rate(sigma, k.inv_s);
  k.c = -nph * DM<T>::inv_sqrt_2pi() * k.inv_s;
  return k;
}
template <class T, bool SIG>
__device__ __forceinline__ Edge<T> edge_eval(const AxisK<T>& k, int e) {
  Edge<T> r;
  const T t = (T(e) + T(0.5)) - k.mu;
  DM<T>::erf_gauss(t, k.s_erf, r.se, r.hs, r.g);
  r.tg = t * r.g;
  r.t3g = SIG ? t * t * r.tg : T(0);
  return r;
}
// One pixel's tables (see axis_tables) from its lower / upper edges.
template <class T> struct Pix {
  T phi, D, D2, S, SS;
};
template <class T, bool SIG>
__device__ __forceinline__ Pix<T> pix_from_edges(const AxisK<T>& k, const Edge<T>& lo, const Edge<T>& hi) {
  Pix<T> p;
  p.phi = pixel_integral<T>(lo.se, lo.hs, hi.se, hi.hs);
  p.D = k.c * (hi.g - lo.g);
  const T w = hi.tg - lo.tg;
  p.D2 = k.c2() * w;
  p.S = SIG ? k.cs() * w : T(0);
  p.SS = SIG ? k.m2s() * p.S + k.css() * (hi.t3g - lo.t3g) : T(0);
  return p;
}

// ---------------------------------------------------------------------------
// One pixel row or column of an axis as plain differences of its two edges.
// The tables of axis_tables() are these times the axis constants:
//   D = c dg,  D2 = c2 w,  S = cs w,  SS = m2s cs w + css t3
// so sums weighted with them need the constants once per iteration, not once
// per row.
// ---------------------------------------------------------------------------
template <class T> struct Band {
  T phi, dg, w, t3;
};
template <class T, bool SIG>
__device__ __forceinline__ Edge<T> edge_at(const AxisK<T>& k, T pos) {
  Edge<T> r;
  const T t = pos - k.mu;
  DM<T>::erf_gauss(t, k.s_erf, r.se, r.hs, r.g);
  r.tg = t * r.g;
  r.t3g = SIG ? t * t * r.tg : T(0);
  return r;
}
template <class T, bool SIG>
__device__ __forceinline__ Band<T> band_from_edges(const Edge<T>& lo, const Edge<T>& hi) {
  Band<T> b;
  b.phi = pixel_integral<T>(lo.se, lo.hs, hi.se, hi.hs);
  b.dg = hi.g - lo.g;
  b.w = hi.tg - lo.tg;
  b.t3 = SIG ? hi.t3g - lo.t3g : T(0);
  return b;
}

// What the pixel loop and the row folds read of one row.
struct RowVals {
  float phi, phi2, pw, dg, w, t3, dg2, w2;   // phi^2, phi w, dg^2, w^2
};
template <bool SIG> __device__ __forceinline__ RowVals row_vals(const Band<float>& b) {
  RowVals v;
  v.phi = b.phi;
  v.phi2 = b.phi * b.phi;
  v.dg = b.dg;
  v.w = b.w;
  v.dg2 = b.dg * b.dg;
  v.pw = SIG ? b.phi * b.w : 0.f;
  v.t3 = SIG ? b.t3 : 0.f;
  v.w2 = SIG ? b.w * b.w : 0.f;
  return v;
}

// ---------------------------------------------------------------------------
// Row tables shared by the L lanes of an ROI.  Every lane needs every row's
// values, but evaluating the N + 1 row edges (one erf and one exp each) on all
// L lanes repeats the same work L times.  Instead lane r evaluates the rows
// [r RS, r RS + RS) and writes them to LDS, from where every lane of the ROI
// reads a row's values (one or two 16-byte reads at one address per ROI) when
// its loop reaches the row.  LDS reads issue beside the VALU, where the DPP
// moves used before took 5 VALU instructions per row at 2 and 4 lanes and 15
// at 8 (one per value at 16, where the read's latency counts instead: see
// rows_together).  The wave is its own only reader, and LDS operations of a wave stay in
// order, so no barrier is needed beyond the compiler's.  An ROI's rows take
// RS L slots (slots past row N - 1 are written and never read) plus 4 words,
// which spread the ROIs that one 16-lane phase of a read serves over the banks.
// ---------------------------------------------------------------------------
template <int N, int L> constexpr int row_slots() { return (N + L - 1) / L; }   // rows per lane
// Words of a row: its eight values with a width, four without.  One lane per
// ROI keeps four of the eight and forms the products again.
template <int MODEL, int L> constexpr int row_words() { return (MT<MODEL>::EXTRA != 0 && L > 1) ? 8 : 4; }
// Words from one row to the next: one lane per ROI interleaves the wave's 64
// ROIs, so that a read takes consecutive addresses.
template <int MODEL, int L> constexpr int row_stride() { return L == 1 ? 4 * kWave : row_words<MODEL, L>(); }
template <int MODEL, int N, int L> constexpr int roi_words() {
  return row_slots<N, L>() * L * row_words<MODEL, L>() + 4;
}
template <int MODEL, int N, int L> constexpr int rows_words() {
  return L == 1 ? N * 4 * kWave : kWave / L * roi_words<MODEL, N, L>();
}
// WORDS words of LDS; every caller with the same WORDS in a kernel gets the
// same array.
template <int WORDS> __device__ __forceinline__ float* wave_lds() {
  __shared__ float4 words[WORDS / 4];
  return reinterpret_cast<float*>(words);
}
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// This lane's rows, evaluated and written to its ROI's LDS words (and to own,
// unless null).
template <int MODEL, int N, int L>
__device__ __forceinline__ void publish_rows(const AxisK<float>& ky, int r, float* roi, RowVals* own = nullptr) {
  constexpr bool SIG = MT<MODEL>::EXTRA != 0;
  constexpr int RS = row_slots<N, L>();
  constexpr int W = row_stride<MODEL, L>();
  const float r0 = (float)(r * RS);
  float* dst = roi + r * RS * W;
  wave_lds_order();   // after the previous evaluation's reads
  Edge<float> lo = edge_at<float, SIG>(ky, r0 + 0.5f);
#pragma unroll
  for (int s = 0; s < RS; ++s) {
    const Edge<float> hi = edge_at<float, SIG>(ky, r0 + ((float)s + 1.5f));
    const RowVals v = row_vals<SIG>(band_from_edges<float, SIG>(lo, hi));
    lo = hi;
    if (own) own[s] = v;
    float4* q = reinterpret_cast<float4*>(dst + s * W);
    if constexpr (SIG && L > 1) {
      q[0] = make_float4(v.phi, v.phi2, v.pw, v.dg);
      q[1] = make_float4(v.w, v.t3, v.dg2, v.w2);
    } else {
      q[0] = make_float4(v.phi, v.dg, v.w, SIG ? v.t3 : v.dg2);
    }
  }
  wave_lds_order();
}

// Row i of the ROI, from LDS.
template <int MODEL, int L> __device__ __forceinline__ RowVals read_row(const float* roi, int i) {
  constexpr bool SIG = MT<MODEL>::EXTRA != 0;
  const float4* src = reinterpret_cast<const float4*>(roi + i * row_stride<MODEL, L>());
  const float4 a = src[0];
  if constexpr (SIG && L > 1) {
    const float4 b = src[1];
    return RowVals{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  } else if constexpr (SIG) {
    return row_vals<true>(Band<float>{a.x, a.y, a.z, a.w});
  } else {
    return RowVals{a.x, a.x * a.x, 0.f, a.y, a.z, 0.f, a.w, 0.f};
  }
}

// ---------------------------------------------------------------------------
// Tail split.  With N = L q + 1 the plain column blocks give each lane
// ceil(N / L) = q + 1 columns, and the group computes L (q + 1) columns for N:
// almost a whole padding column per lane (13 px on 4 lanes: 52 pixel slots
// per lane for 169 pixels).  Split instead, each lane holds q full columns
// [r q, r q + q) and, of the last column N - 1, the rows it evaluates itself: q N + ceil(N / L) slots (13 px on 4 lanes:
// 43).  The last column's partial sums are folded with that column's values on
// every lane and summed across the group with the rest (the fold is linear).
// ---------------------------------------------------------------------------
// From 4 lanes up: with 2 lanes a padding column is one in N + 1 and costs less
// than the tail's own row folds (XYNBS 11 px on 2 lanes, with the split 1.55 ns
// per ROI, as much as 12 px).
template <int N, int L> constexpr bool tail_split() { return L >= 4 && N > L && N % L == 1; }
// Register-resident full columns per lane.
template <int N, int L> constexpr int block_cols() {
  return tail_split<N, L>() ? N / L : (N + L - 1) / L;
}
// Rows whose pixel work the scheduler may mix, and that are read from LDS
// together, one such group ahead: a row of one column is a short dependent chain
// (model, reciprocal, weights, sums), so two go together.  us per launch on 16
// lanes with groups of 1, 2 and 4: sCMOS XYNB 13 px, 2,000 ROIs 24.5, 23.2, 23.2;
// XYNBSXSY 9 px, 4,000 ROIs 29.0, 28.8, 31.6.  From two columns on, one row at a time
// (sCMOS XYNBS 13 px, 3 columns, 1M ROIs 2.30 ms, two rows together 2.36;
// astigmatic 21 px, 2 columns on 16 lanes 59.3 us and 62.0).
template <int CB> constexpr int rows_together() { return CB == 1 ? 2 : 1; }
// Least waves per SIMD a fit kernel is built for: three where a lane's pixels (and
// variances) leave the loop enough of the 168 VGPRs that three waves have, and
// three waves' LDS fits a CU's 160 KB, else two up to 144 values (sCMOS XYNBS
// 16 px on 4 lanes, 128 values: 235 VGPRs; at one wave an earlier build of it took
// 4.19 ms per 1M ROIs, at two 2.93).  Above the first line the
// spills cost more than the third wave hides: sCMOS XYNBS 13 px
// on 4 lanes (86 values) runs 2.46 -> 2.34 ms per 1M ROIs with three waves and
// 164 B of scratch, XYNB 11 px on one lane (121 values) 1.51 -> 2.04 ms.
constexpr int kLds3Waves = 160 * 1024 / 12, kLds2Waves = 160 * 1024 / 8;
template <int MODEL, int CAM, int N, int L> constexpr int min_waves() {
  constexpr int px = (block_cols<N, L>() * N + (tail_split<N, L>() ? row_slots<N, L>() : 0)) * (CAM == SCMOS ? 2 : 1);
  return px <= 88 && rows_words<MODEL, N, L>() * 4 <= kLds3Waves ? 3 : px <= 144 ? 2 : 1;
}
// The pixel loop reads only phi (and phi^2) of a column; its other values wait
// in LDS until the fold, one quad per column and lane, where there is room for
// them beside the rows.
template <int MODEL, int CAM, int N, int L> constexpr int park_words() {
  constexpr int w = block_cols<N, L>() * (MT<MODEL>::EXTRA != 0 ? 4 : 2) * kWave;
  constexpr int room = min_waves<MODEL, CAM, N, L>() == 3 ? kLds3Waves : kLds2Waves;
  return (rows_words<MODEL, N, L>() + w) * 4 <= room ? w : 0;
}
// LDS words of one wave.
template <int MODEL, int CAM, int N, int L> constexpr int wave_words() {
  return rows_words<MODEL, N, L>() + park_words<MODEL, CAM, N, L>();
}
template <bool SIG> __device__ __forceinline__ void park_band(float* park, int cc, const Band<float>& b) {
  if constexpr (SIG) {
    reinterpret_cast<float4*>(park)[cc * kWave] = make_float4(b.dg, b.w, b.t3, 0.f);
  } else {
    reinterpret_cast<float2*>(park)[cc * kWave] = make_float2(b.dg, b.w);
  }
}
template <bool SIG> __device__ __forceinline__ Band<float> parked_band(const float* park, int cc, float phi) {
  if constexpr (SIG) {
    const float4 q = reinterpret_cast<const float4*>(park)[cc * kWave];
    return Band<float>{phi, q.x, q.y, q.z};
  } else {
    const float2 q = reinterpret_cast<const float2*>(park)[cc * kWave];
    return Band<float>{phi, q.x, q.y, 0.f};
  }
}

// Whether block column cc lies past the ROI on some lane (L does not divide
// N).  Such a column carries zero column values and adds nothing.
template <int N, int L> constexpr bool may_pad(int cc) {
  return !tail_split<N, L>() && (L - 1) * block_cols<N, L>() + cc >= N;
}

// Tail split: whether a lane keeps the values of the rows it evaluated in
// registers for its pixels of the last column, which then need not wait for LDS.
// Up to three of them, or under sCMOS: the two forms of the Poisson loop hold
// more, and four rows spilled there (XYNB 13 px on 4 lanes, 12,000 ROIs: 49.8 us
// through LDS, 56.2 from registers; sCMOS 51.9 and 50.1).
template <int CAM, int N, int L> constexpr bool keep_own_rows() {
  return tail_split<N, L>() && (CAM == SCMOS || row_slots<N, L>() <= 3);
}
// Rows 0 .. KR - 1, and in the loop the KR rows from i on while the next KR are
// in flight.
template <int MODEL, int N, int L, int KR>
__device__ __forceinline__ void first_rows(const float* roi, RowVals* next) {
#pragma unroll
  for (int k = 0; k < KR; ++k) next[k] = read_row<MODEL, L>(roi, k < N ? k : 0);
}
template <int MODEL, int N, int L, int KR>
__device__ __forceinline__ void take_rows(const float* roi, int i, RowVals* rows, RowVals* next) {
#pragma unroll
  for (int k = 0; k < KR; ++k) {
    rows[k] = next[k];
    if (i + KR + k < N) next[k] = read_row<MODEL, L>(roi, i + KR + k);
  }
}

// Per-ROI width parameters for one evaluation of the model.
template <class T> struct Widths {
  T sx, sy;          // sigma per axis (pixels)
  T dsx, dsy;        // astig: d sigma / dz
  T d2sx, d2sy;      // astig: d2 sigma / dz2
};

// psf_derivatives.jl:115-163: sigma_x(z), sigma_y(z) and their z derivatives.
template <class T>
__device__ __forceinline__ void astig_widths(T z, const float* psf, Widths<T>& w) {
  const T sx0 = (T)psf[0], sy0 = (T)psf[1], Ax = (T)psf[2], Ay = (T)psf[3];
  const T Bx = (T)psf[4], By = (T)psf[5], gamma = (T)psf[6], dd = (T)psf[7];
  const T zdx = DM<T>::div(z - gamma, dd);
  const T zdy = DM<T>::div(z + gamma, dd);
  const T zdx2 = zdx * zdx, zdy2 = zdy * zdy;
  const T ax = T(1) + zdx2 + Ax * (zdx2 * zdx) + Bx * (zdx2 * zdx2);
  const T ay = T(1) + zdy2 + Ay * (zdy2 * zdy) + By * (zdy2 * zdy2);
  const T sqax = sqrt(ax), sqay = sqrt(ay);
  w.sx = sx0 * sqax;
  w.sy = sy0 * sqay;
  const T dax = DM<T>::div(T(2) * zdx + T(3) * Ax * zdx2 + T(4) * Bx * (zdx2 * zdx), dd);
  const T day = DM<T>::div(T(2) * zdy + T(3) * Ay * zdy2 + T(4) * By * (zdy2 * zdy), dd);
  const T hx = DM<T>::div(sx0, T(2) * sqax), hy = DM<T>::div(sy0, T(2) * sqay);
  w.dsx = hx * dax;
  w.dsy = hy * day;
  const T d2ax = DM<T>::div(T(2) + T(6) * Ax * zdx + T(12) * Bx * zdx2, dd * dd);
  const T d2ay = DM<T>::div(T(2) + T(6) * Ay * zdy + T(12) * By * zdy2, dd * dd);
  w.d2sx = -DM<T>::div(sx0, T(4) * (ax * sqax)) * (dax * dax) + hx * d2ax;
  w.d2sy = -DM<T>::div(sy0, T(4) * (ay * sqay)) * (day * day) + hy * d2ay;
}

template <int MODEL, class T>
__device__ __forceinline__ void model_widths(const T* th, const float* psf, Widths<T>& w) {
  w.dsx = w.dsy = w.d2sx = w.d2sy = T(0);
  if constexpr (MODEL == XYNB) {
    w.sx = w.sy = (T)psf[0];
  } else if constexpr (MODEL == XYNBS) {
    w.sx = w.sy = th[4];
  } else if constexpr (MODEL == XYNBSXSY) {
    w.sx = th[4];
    w.sy = th[5];
  } else {
    astig_widths<T>(th[2], psf, w);
  }
}

// One pixel's likelihood weights (camera_models.jl:19-42): cf multiplies the
// model's derivatives in the gradient, df in the Hessian.  FAST (Poisson
// only): every model value exceeds 0.01 and neither 1e4 cap can bind; then
// cf = d/mu - 1 and df = d/mu^2 = (cf + 1)/mu are one FMA each.  Where no mask
// binds both forms give the same bits.
template <int CAM, bool FAST>
__device__ __forceinline__ void pixel_weights(float d, float var, float mu, float& cf, float& df) {
  if constexpr (CAM == IDEAL) {
    const float rc = fast_rcp(mu);
    const float a = fmaf(d, rc, -1.f), b = fmaf(a, rc, rc);
    if constexpr (FAST) {
      cf = a;
      df = b;
    } else {
      const bool pos = mu > 0.01f;   // camera_models.jl:23-32
      cf = pos ? (1.0e4f < a ? 1.0e4f : a) : 0.f;   // Julia's min: a NaN passes
      df = pos ? (1.0e4f < b ? 1.0e4f : b) : 0.f;
    }
  } else {
    const float v = mu + var;   // camera_models.jl:36-42
    const float rc = fast_rcp(v);
    cf = (d - mu) * rc;
    df = rc;
  }
}

// This lane's column values, and with the tail split those of the last column
// (from lane L - 1, whose block ends at edge N - 1).
template <int N, int L, bool SIG>
__device__ __forceinline__ void column_bands(const AxisK<float>& kx, int c0, Band<float>* cb, Band<float>& tl) {
  constexpr int CB = block_cols<N, L>();
  const float f0 = (float)c0;
  Edge<float> lo = edge_at<float, SIG>(kx, f0 + 0.5f);
#pragma unroll
  for (int cc = 0; cc < CB; ++cc) {
    const Edge<float> hi = edge_at<float, SIG>(kx, f0 + ((float)cc + 1.5f));
    cb[cc] = band_from_edges<float, SIG>(lo, hi);
    lo = hi;
    if (may_pad<N, L>(cc) && c0 + cc >= N) cb[cc] = Band<float>{0.f, 0.f, 0.f, 0.f};
  }
  if constexpr (tail_split<N, L>()) {
    const Band<float> b = band_from_edges<float, SIG>(lo, edge_at<float, SIG>(kx, (float)N + 0.5f));
    tl.phi = group_bcast<L, L - 1>(b.phi);
    tl.dg = group_bcast<L, L - 1>(b.dg);
    tl.w = group_bcast<L, L - 1>(b.w);
    tl.t3 = SIG ? group_bcast<L, L - 1>(b.t3) : 0.f;
  }
}

// ---------------------------------------------------------------------------
// One Newton iteration's gradient G[P] and diagonal Hessian H[P] over this
// lane's pixels (unified_kernel.jl:319-334):
//   G_k = sum_ij dudt_k cf,   H_k = sum_ij (d2udt2_k cf - dudt_k^2 df).
// Every term factors as (column value)(row value)(cf or df), so the pixels
// only feed six sums (seven where one parameter moves both widths):
//   C_j = sum_i phiy_i cf     CC_j = sum_i phiy_i^2 df      per column
//   R_i = sum_j phix_j cf     RR_i = sum_j phix_j^2 df      per row
//   sum cf, sum df            X_j = sum_i phiy_i wy_i df    per column
// and the derivatives of the x axis weight C and CC, those of the y axis R and
// RR: d/dx is sum_j Dx_j C_j, d/dy is sum_i Dy_i R_i, and so on.  Weighting
// the pixels with every row table instead took 7 (fixed width) to 11 sums per
// pixel and held them all per column.  Rows run in the outer loop: a row's R
// and RR are folded as soon as the row ends, and a lane keeps only its
// columns' five values and three sums.
// Bound by VALU issue.  gfx950, ms per launch against 7 to 11 sums per pixel
// with the row tables by DPP: sCMOS XYNBS 13 px, 1M ROIs 3.20 -> 2.36; astigmatic
// 15 px, 1M 6.07 -> 3.96; XYNBS 21 px, 200K 1.80 -> 1.02; XYNB 11 px on one lane,
// 1M 1.386 -> 1.144.
// ---------------------------------------------------------------------------
struct PixelSums {
  float a1, a2, a3, a4, a5;   // columns: dg C, w C, dg^2 CC, t3 C, w^2 CC
  float y1, y2, y3, y4, y5;   // rows: dg R, w R, t3 R, dg^2 RR, w^2 RR
  float gn, hn, xs;           // phi C, phi^2 CC, phi w X
  float scf, sdf;
};
template <int MODEL, int CAM, int N, int L, bool FAST>
__device__ __forceinline__ void accumulate(const float* dv, const float* vr, const float* dt, const float* vt, int c0,
                                           int r, float nph, float bg, const AxisK<float>& kx, const AxisK<float>& ky,
                                           const float* roi, const RowVals* own, float* park, PixelSums& out) {
  using Tr = MT<MODEL>;
  constexpr bool TAIL = tail_split<N, L>();
  constexpr int CB = block_cols<N, L>();
  constexpr int RS = row_slots<N, L>();
  constexpr bool SIG = Tr::EXTRA != 0;
  constexpr bool TWO = (Tr::EXTRA == 1 || Tr::EXTRA == 3);
  constexpr int KR = rows_together<CB>();
  // One column: its factor multiplies the row sums once, not every row's cf and
  // df.  With the rows read ahead in twos and the shorter Newton test below, us per
  // launch: sCMOS XYNB 13 px, 2,000 ROIs on 16 lanes 27.0 -> 23.2, ideal XYNB 7 px,
  // 100 ROIs 20.9 -> 19.5, XYNBSXSY 9 px, 4,000 ROIs 30.4 -> 28.8.
  constexpr bool ONE = CB == 1;
  constexpr bool OWN = keep_own_rows<CAM, N, L>();
  Band<float> cb[CB], tl{};
  column_bands<N, L, SIG>(kx, c0, cb, tl);
  constexpr bool PARK = park_words<MODEL, CAM, N, L>() != 0;
  if constexpr (PARK) {
#pragma unroll
    for (int cc = 0; cc < CB; ++cc) park_band<SIG>(park, cc, cb[cc]);
    wave_lds_order();
  }
  float px2[CB], C[CB], CC[CB], X[TWO ? CB : 1], pad_cf[CB], pad_df[CB];
#pragma unroll
  for (int cc = 0; cc < CB; ++cc) {
    px2[cc] = cb[cc].phi * cb[cc].phi;
    C[cc] = CC[cc] = 0.f;
    pad_cf[cc] = pad_df[cc] = 0.f;
    if constexpr (TWO) X[cc] = 0.f;
  }
  float y1 = 0.f, y2 = 0.f, y3 = 0.f, y4 = 0.f, y5 = 0.f;   // dg R, w R, t3 R, dg^2 RR, w^2 RR over the rows
  float scf = 0.f, sdf = 0.f;
  auto fold_row = [&](const RowVals& v, float R, float RR) __attribute__((always_inline)) {
    y1 = fmaf(v.dg, R, y1);
    y2 = fmaf(v.w, R, y2);
    y4 = fmaf(v.dg2, RR, y4);
    if constexpr (SIG) {
      y3 = fmaf(v.t3, R, y3);
      y5 = fmaf(v.w2, RR, y5);
    }
  };
  float a1 = 0.f, a2 = 0.f, a3 = 0.f, a4 = 0.f, a5 = 0.f, gn = 0.f, hn = 0.f, xs = 0.f;
  auto fold_col = [&](const Band<float>& b, float b2, float c, float cc2, float x) __attribute__((always_inline)) {
    a1 = fmaf(b.dg, c, a1);
    a2 = fmaf(b.w, c, a2);
    a3 = fmaf(b.dg * b.dg, cc2, a3);
    gn = fmaf(b.phi, c, gn);
    hn = fmaf(b2, cc2, hn);
    if constexpr (SIG) {
      a4 = fmaf(b.t3, c, a4);
      a5 = fmaf(b.w * b.w, cc2, a5);
      if constexpr (TWO) xs = fmaf(b.phi * b.w, x, xs);
    }
  };
  if constexpr (TAIL) {
    // the last column's pixels of this lane's own rows (slots past the last
    // row weigh nothing)
    const float npx = nph * tl.phi, tp2 = tl.phi * tl.phi;
    float Ct = 0.f, CCt = 0.f, Xt = 0.f;
#pragma unroll
    for (int s = 0; s < RS; ++s) {
      if (s % KR == 0) __builtin_amdgcn_sched_barrier(0);
      const RowVals v = OWN ? own[s] : read_row<MODEL, L>(roi, r * RS + s);
      const float mu = fmaf(npx, v.phi, bg);
      float cf, df;
      pixel_weights<CAM, FAST>(dt[s], CAM == SCMOS ? vt[s] : 0.f, mu, cf, df);
      if ((L - 1) * RS + s >= N) {   // some lane's slot lies past the last row
        const bool ok = r * RS + s < N;
        cf = ok ? cf : 0.f;
        df = ok ? df : 0.f;
      }
      Ct = fmaf(v.phi, cf, Ct);
      CCt = fmaf(v.phi2, df, CCt);
      if constexpr (TWO) Xt = fmaf(v.pw, df, Xt);
      fold_row(v, tl.phi * cf, tp2 * df);
      scf += cf;
      sdf += df;
    }
    fold_col(tl, tp2, Ct, CCt, Xt);
    // done here, not where the sums are next used
    asm volatile("" : "+v"(a1), "+v"(a2), "+v"(a3), "+v"(gn), "+v"(hn), "+v"(y1), "+v"(y2), "+v"(y4), "+v"(scf),
                 "+v"(sdf));
    if constexpr (SIG) asm volatile("" : "+v"(a4), "+v"(a5), "+v"(y3), "+v"(y5), "+v"(xs));
    __builtin_amdgcn_sched_barrier(0);
  }
  RowVals rows[KR], next[KR];
  first_rows<MODEL, N, L, KR>(roi, next);
  float z1 = 0.f, z2 = 0.f, z3 = 0.f, z4 = 0.f, z5 = 0.f;   // ONE: the row sums before their column factor
#pragma unroll
  for (int i = 0; i < N; ++i) {
    // Keep the rows' work apart: without this the scheduler hoists later rows'
    // values and pixel products and they all become live at once.
    if (i % KR == 0) {
      __builtin_amdgcn_sched_barrier(0);
      take_rows<MODEL, N, L, KR>(roi, i, rows, next);
    }
    const RowVals v = rows[i % KR];
    const float pn = nph * v.phi;
    float R = 0.f, RR = 0.f;
#pragma unroll
    for (int cc = 0; cc < CB; ++cc) {
      const float mu = fmaf(cb[cc].phi, pn, bg);
      float cf, df;
      pixel_weights<CAM, FAST>(dv[cc * N + i], CAM == SCMOS ? vr[cc * N + i] : 0.f, mu, cf, df);
      C[cc] = fmaf(v.phi, cf, C[cc]);
      CC[cc] = fmaf(v.phi2, df, CC[cc]);
      if constexpr (TWO) X[cc] = fmaf(v.pw, df, X[cc]);
      if constexpr (ONE) {
        z1 = fmaf(v.dg, cf, z1);
        z2 = fmaf(v.w, cf, z2);
        z4 = fmaf(v.dg2, df, z4);
        if constexpr (SIG) {
          z3 = fmaf(v.t3, cf, z3);
          z5 = fmaf(v.w2, df, z5);
        }
      } else {
        R = cc == 0 ? cb[cc].phi * cf : fmaf(cb[cc].phi, cf, R);
        RR = cc == 0 ? px2[cc] * df : fmaf(px2[cc], df, RR);
      }
      // A padding pixel has data 0; its weights are 0 under sCMOS (infinite
      // variance), and are dropped after the rows for the ideal camera.
      if (CAM == IDEAL && may_pad<N, L>(cc)) {
        pad_cf[cc] += cf;
        pad_df[cc] += df;
      } else {
        scf += cf;
        sdf += df;
      }
    }
    if constexpr (!ONE) fold_row(v, R, RR);
    // ... and tie this row's sums to the end of the row, or instruction
    // selection sinks the pixel work of every row below the last one.
    if (i % KR != KR - 1) continue;
#pragma unroll
    for (int cc = 0; cc < CB; ++cc) {
      asm volatile("" : "+v"(C[cc]), "+v"(CC[cc]));
      if constexpr (TWO) asm volatile("" : "+v"(X[cc]));
      if (CAM == IDEAL && may_pad<N, L>(cc)) asm volatile("" : "+v"(pad_cf[cc]), "+v"(pad_df[cc]));
    }
    asm volatile("" : "+v"(scf), "+v"(sdf));
    if constexpr (ONE) {
      asm volatile("" : "+v"(z1), "+v"(z2), "+v"(z4));
      if constexpr (SIG) asm volatile("" : "+v"(z3), "+v"(z5));
    } else {
      asm volatile("" : "+v"(y1), "+v"(y2), "+v"(y4));
      if constexpr (SIG) asm volatile("" : "+v"(y3), "+v"(y5));
    }
  }
  if constexpr (ONE) fold_row(RowVals{0.f, 0.f, 0.f, z1, z2, z3, z4, z5}, cb[0].phi, px2[0]);
#pragma unroll
  for (int cc = 0; cc < CB; ++cc) {
    fold_col(PARK ? parked_band<SIG>(park, cc, cb[cc].phi) : cb[cc], px2[cc], C[cc], CC[cc],
             TWO ? X[TWO ? cc : 0] : 0.f);
    if (CAM == IDEAL && may_pad<N, L>(cc)) {
      scf += c0 + cc < N ? pad_cf[cc] : 0.f;
      sdf += c0 + cc < N ? pad_df[cc] : 0.f;
    }
  }
  out = PixelSums{a1, a2, a3, a4, a5, y1, y2, y3, y4, y5, gn, hn, xs, scf, sdf};
}

// The gradient and diagonal Hessian from the sums: once for both forms of the
// pixel loop, so that an ROI's result does not depend on which one its wave took.
template <int MODEL>
__device__ __forceinline__ void gradient(const PixelSums& u, const AxisK<float>& kx, const AxisK<float>& ky,
                                         const Widths<float>& w, float* G, float* H) {
  using Tr = MT<MODEL>;
  constexpr bool SIG = Tr::EXTRA != 0;
  G[Tr::IX] = kx.c * u.a1;
  H[Tr::IX] = kx.c2() * u.a2 - (kx.c * kx.c) * u.a3;
  G[Tr::IY] = ky.c * u.y1;
  H[Tr::IY] = ky.c2() * u.y2 - (ky.c * ky.c) * u.y4;
  G[Tr::IN] = u.gn;
  H[Tr::IN] = -u.hn;
  G[Tr::IBG] = u.scf;
  H[Tr::IBG] = -u.sdf;
  if constexpr (SIG) {
    // width terms of each axis: first derivative ex w, second (m2s + d2) w + css t3
    const float csx = kx.cs() * u.a2, csy = ky.cs() * u.y2;                       // sum S C, sum S R
    const float ssx = kx.m2s() * csx + kx.css() * u.a4, ssy = ky.m2s() * csy + ky.css() * u.y3;   // sum SS C, sum SS R
    const float qx = kx.cs() * kx.cs() * u.a5, qy = ky.cs() * ky.cs() * u.y5;         // sum S^2 CC, sum S^2 RR
    const float qxy = 2.f * (kx.cs() * ky.cs()) * u.xs;
    if constexpr (MODEL == XYNBS) {
      G[Tr::IE1] = csx + csy;
      H[Tr::IE1] = ssx + ssy - qx - qy - qxy;
    } else if constexpr (MODEL == XYNBSXSY) {
      G[Tr::IE1] = csx;
      H[Tr::IE1] = ssx - qx;
      G[Tr::IE2] = csy;
      H[Tr::IE2] = ssy - qy;
    } else {
      G[Tr::IE1] = w.dsx * csx + w.dsy * csy;
      H[Tr::IE1] = (w.dsx * w.dsx) * (ssx - qx) + w.d2sx * csx + (w.dsy * w.dsy) * (ssy - qy) + w.d2sy * csy -
                   (w.dsx * w.dsy) * qxy;
    }
  }
}

// ---------------------------------------------------------------------------
// Final pass (unified_kernel.jl:353-431): at the estimate th, the LLR
// (camera_models.jl:60-85), the full Fisher matrix over pixels with model > 0
// (unified_kernel.jl:378-396) and its inversion into the CRLB, in arithmetic
// type TF.  Pixel data come from Src: VGPR arrays (RegSrc, in the iteration
// kernel) or global memory (GlobalSrc, in the Float64 final-pass kernel).
// ---------------------------------------------------------------------------
template <int N, bool SC> struct RegSrc {
  const float* dv;   // this lane's column block, [cc * N + i]
  const float* vr;
  __device__ __forceinline__ float d(int cc, int i) const { return dv[cc * N + i]; }
  __device__ __forceinline__ float var(int cc, int i) const { return SC ? vr[cc * N + i] : 0.f; }
};
// n consecutive floats from p (4-byte aligned) in 16- and 8-byte loads: gfx950
// global loads need only dword alignment, and one lane's run of a column then
// takes ceil(n / 4) load instructions instead of n.
template <int n> __device__ __forceinline__ void load_run(const float* p, float* out) {
#pragma unroll
  for (int i = 0; i + 4 <= n; i += 4) {
    float4 q;
    __builtin_memcpy(&q, p + i, sizeof(q));
    out[i] = q.x;
    out[i + 1] = q.y;
    out[i + 2] = q.z;
    out[i + 3] = q.w;
  }
  constexpr int b = n - n % 4;
  if constexpr (n % 4 >= 2) {
    float2 q;
    __builtin_memcpy(&q, p + b, sizeof(q));
    out[b] = q.x;
    out[b + 1] = q.y;
  }
  if constexpr (n % 2 == 1) out[n - 1] = p[n - 1];
}

template <int N, bool SC> struct GlobalSrc {
  const float* data = nullptr;   // the ROI, column-major
  const float* var = nullptr;    // var_map at the ROI's first pixel
  int ny = 0;
  // column cc's pixels and variances (both runs are contiguous)
  __device__ __forceinline__ void column(int cc, float* dcol, float* vcol) const {
    load_run<N>(data + cc * N, dcol);
    if constexpr (SC) load_run<N>(var + (int64_t)cc * ny, vcol);
  }
};
template <class TF, int P> struct FinalOut {
  TF crlb[P];
  TF llr;
};

// One pixel of the final pass (unified_kernel.jl:359-397): its LLR term
// (camera_models.jl:60-85) and, where the model is > 0, its Fisher
// contribution du du^T / v (v = model, or model + variance for sCMOS) to the
// upper triangle Fu.  du holds the pixel's P model derivatives.
template <int CAM, int P, class TF>
__device__ __forceinline__ void final_pixel(TF d, TF var, TF mu, const TF* du, bool cvalid, TF* Fu, TF& llr) {
  static_assert(sizeof(TF) == 8, "the Float32 pass sums its Fisher matrix by columns and rows");
  TF v = mu;
  TF lp;
  TF rv = TF(0);   // 1/mu, the ideal camera's Fisher weight
  if constexpr (CAM == IDEAL) {
    // camera_models.jl:60-71, as d log(mu/d) + d - mu with one log:
    // d log(mu/d) = -d log(d (1/mu)), and 1/mu is also the Fisher weight below.
    rv = mu > TF(0) ? TF(1) / mu : TF(0);
    lp = (mu > TF(0) && d > TF(0)) ? -d * log(d * rv) + (d - mu) : (mu > TF(0) && d == TF(0)) ? -mu : TF(0);
  } else {
    // camera_models.jl:73-85.  The Fisher weight below divides again, inside
    // its own block: a 1/v shared by both keeps it live across the block, and
    // the multi-shape kernel's largest sCMOS tiles then exceed 256 VGPRs.
    v = mu + var;
    const TF res = d - mu;
    lp = v > TF(0) ? TF(-0.5) * (res * res / v) : TF(0);
  }
  if (cvalid) llr += lp;
  if (cvalid && mu > TF(0)) {
    const TF wv = CAM == IDEAL ? rv : TF(1) / v;
    int q = 0;
#pragma unroll
    for (int k = 0; k < P; ++k) {
      const TF ak = du[k] * wv;
#pragma unroll
      for (int l = k; l < P; ++l) Fu[q++] += ak * du[l];
    }
  }
}

// The pixel's model derivatives from its column and row tables
// (psf_derivatives.jl:6-187): x, y, N, bg, and the sigma / z term.
template <int MODEL, class TF>
__device__ __forceinline__ void final_du(TF px, TF py, TF Dx, TF Dy, TF ax, TF ay, TF* du) {
  using Tr = MT<MODEL>;
  du[Tr::IX] = Dx * py;
  du[Tr::IY] = Dy * px;
  du[Tr::IN] = px * py;
  du[Tr::IBG] = TF(1);
  if constexpr (Tr::EXTRA == 2) {
    du[Tr::IE1] = ax * py;
    du[Tr::IE2] = ay * px;
  } else if constexpr (Tr::EXTRA != 0) {
    du[Tr::IE1] = ax * py + ay * px;
  }
}

// Sums across the group, the symmetric Fisher matrix and its inversion.
template <int L, int P, class TF>
__device__ __forceinline__ FinalOut<TF, P> final_reduce(TF* Fu, TF llr) {
  constexpr int NF = P * (P + 1) / 2;
  FinalOut<TF, P> out;
  out.llr = group_sum<L>(llr);
#pragma unroll
  for (int q = 0; q < NF; ++q) Fu[q] = group_sum<L>(Fu[q]);
  TF F[P * P];
  int q = 0;
#pragma unroll
  for (int k = 0; k < P; ++k)
#pragma unroll
    for (int l = k; l < P; ++l) {
      F[k + P * l] = Fu[q];
      F[l + P * k] = Fu[q];
      ++q;
    }
  invert_fisher<P, TF>(F, out.crlb);
  return out;
}

template <int MODEL, int CAM, int N, int L, class TF, class Src>
__device__ __forceinline__ FinalOut<TF, MT<MODEL>::P> final_pass(const float* th, const float* psf, int c0,
                                                               const Src& src) {
  using Tr = MT<MODEL>;
  constexpr int P = Tr::P;
  constexpr int CB = (N + L - 1) / L;
  constexpr bool SIG = Tr::EXTRA != 0;
  TF thf[P];
#pragma unroll
  for (int k = 0; k < P; ++k) thf[k] = (TF)th[k];
  Widths<TF> wf;
  model_widths<MODEL, TF>(thf, psf, wf);
  const TF nphf = thf[Tr::IN], bgf = thf[Tr::IBG];
  AxisTab<TF, N> fy;
  axis_tables<TF, N, SIG>(thf[Tr::IY], wf.sy, nphf, 0, fy);
  const AxisK<TF> kf = axis_consts<TF>(thf[Tr::IX], wf.sx, nphf);

  constexpr int NF = P * (P + 1) / 2;
  TF Fu[NF];
#pragma unroll
  for (int q = 0; q < NF; ++q) Fu[q] = TF(0);
  TF llr = TF(0);
  Edge<TF> flo = edge_eval<TF, false>(kf, c0);
  auto column = [&](int cc) __attribute__((always_inline)) {
    const Edge<TF> fhi = edge_eval<TF, false>(kf, c0 + cc + 1);
    const Pix<TF> fx = pix_from_edges<TF, SIG>(kf, flo, fhi);
    flo = fhi;
    const TF px = fx.phi;
    const bool cvalid = (L == 1) || (c0 + cc < N);
    TF ax = TF(0);
    if constexpr (SIG) ax = (MODEL == ASTIG) ? wf.dsx * fx.S : fx.S;
    float dcol[N], vcol[CAM == SCMOS ? N : 1];
    src.column(cc, dcol, vcol);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const TF py = fy.phi[i];
      TF ay = TF(0);
      if constexpr (SIG) ay = (MODEL == ASTIG) ? wf.dsy * fy.S[i] : fy.S[i];
      TF du[P];
      final_du<MODEL, TF>(px, py, fx.D, fy.D[i], ax, ay, du);
      const TF mu = bgf + nphf * px * py;
      final_pixel<CAM, P, TF>((TF)dcol[i], CAM == SCMOS ? (TF)vcol[i] : TF(0), mu, du, cvalid, Fu, llr);
    }
  };
  // One column at a time keeps only that column's loads in flight.
#pragma unroll 1
  for (int cc = 0; cc < CB; ++cc) column(cc);
  return final_reduce<L, P, TF>(Fu, llr);
}

// The same final pass with rows in the outer loop, for large boxes: each
// row's tables are built from its two edges where the row is used, and a lane
// holds only its CB columns' tables, instead of every row's (which for
// N > 16 would not fit the registers).  Pixels are register-resident.
template <int MODEL, int CAM, int N, int L, class TF, class Src>
__device__ __forceinline__ FinalOut<TF, MT<MODEL>::P> final_pass_rows(const float* th, const float* psf, int c0,
                                                                    const Src& src) {
  using Tr = MT<MODEL>;
  constexpr int P = Tr::P;
  constexpr int CB = (N + L - 1) / L;
  constexpr bool SIG = Tr::EXTRA != 0;
  TF thf[P];
#pragma unroll
  for (int k = 0; k < P; ++k) thf[k] = (TF)th[k];
  Widths<TF> wf;
  model_widths<MODEL, TF>(thf, psf, wf);
  const TF nphf = thf[Tr::IN], bgf = thf[Tr::IBG];
  const AxisK<TF> kx = axis_consts<TF>(thf[Tr::IX], wf.sx, nphf);
  const AxisK<TF> ky = axis_consts<TF>(thf[Tr::IY], wf.sy, nphf);
  Pix<TF> cx[CB];
  TF ax[CB];
  {
    Edge<TF> lo = edge_eval<TF, false>(kx, c0);
#pragma unroll
    for (int cc = 0; cc < CB; ++cc) {
      const Edge<TF> hi = edge_eval<TF, false>(kx, c0 + cc + 1);
      cx[cc] = pix_from_edges<TF, SIG>(kx, lo, hi);
      lo = hi;
      ax[cc] = SIG ? ((MODEL == ASTIG) ? wf.dsx * cx[cc].S : cx[cc].S) : TF(0);
    }
  }
  constexpr int NF = P * (P + 1) / 2;
  TF Fu[NF];
#pragma unroll
  for (int q = 0; q < NF; ++q) Fu[q] = TF(0);
  TF llr = TF(0);
  Edge<TF> rlo = edge_eval<TF, false>(ky, 0);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const Edge<TF> rhi = edge_eval<TF, false>(ky, i + 1);
    const Pix<TF> ry = pix_from_edges<TF, SIG>(ky, rlo, rhi);
    rlo = rhi;
    TF ay = TF(0);
    if constexpr (SIG) ay = (MODEL == ASTIG) ? wf.dsy * ry.S : ry.S;
#pragma unroll
    for (int cc = 0; cc < CB; ++cc) {
      const bool cvalid = (L == 1) || (c0 + cc < N);
      TF du[P];
      final_du<MODEL, TF>(cx[cc].phi, ry.phi, cx[cc].D, ry.D, ax[cc], ay, du);
      const TF mu = bgf + nphf * cx[cc].phi * ry.phi;
      final_pixel<CAM, P, TF>((TF)src.d(cc, i), CAM == SCMOS ? (TF)src.var(cc, i) : TF(0), mu, du, cvalid, Fu,
                              llr);
    }
  }
  return final_reduce<L, P, TF>(Fu, llr);
}

// One pixel's LLR term lp (camera_models.jl:60-85) and Fisher weight wv: 1/v
// where the model is > 0, else 0 (v = model, or model + variance for sCMOS).
template <int CAM> __device__ __forceinline__ void final_weights(float d, float var, float mu, float& lp, float& wv) {
  if constexpr (CAM == IDEAL) {
    // camera_models.jl:60-71, as d log(mu/d) + d - mu with one log:
    // d log(mu/d) = -d log(d (1/mu)), and 1/mu is also the Fisher weight.
    // 1/mu is v_rcp_f32 (1 ulp); the single log also avoids the cancellation of
    // d log(mu) against d log(d) in the two-log form.
    // ln x as v_log_f32 (log2) times ln 2.  x = d/mu of a pixel with d > 0
    // lies far above the denormal range; the clamp keeps even a denormal
    // product finite (its term is then ~0, as it would be).
    wv = mu > 0.f ? fast_rcp(mu) : 0.f;
    const float x = fmaxf(d * wv, 1.17549435e-38f);
    const float lnx = __builtin_amdgcn_logf(x) * 0.693147180559945309f;
    lp = (mu > 0.f && d >= 0.f) ? -d * lnx + (d - mu) : 0.f;   // -mu at d = 0 (lnx is finite there)
  } else {
    const float v = mu + var;   // camera_models.jl:73-85
    const float res = d - mu;
    const float rv = 1.f / v;
    // the clamp: 1 / v of a denormal v is infinite, and 0 x inf no LLR term
    lp = v > 0.f ? -0.5f * (res * res * fminf(rv, 3.40282347e38f)) : 0.f;
    wv = mu > 0.f ? rv : 0.f;
  }
}

// ---------------------------------------------------------------------------
// The Fisher matrix sum_ij du_k du_l wv (unified_kernel.jl:378-396) from
// weighted sums, as accumulate() forms the gradient: with the column sums
//   C = sum_i phiy wv, CC = sum_i phiy^2 wv, Y = sum_i phiy dgy wv, Z = sum_i phiy wy wv
// and the row sums R, RR, every entry is a sum over columns or rows.  Six sums
// per pixel (seven with a width) take the place of the P derivatives and the
// P (P + 1) / 2 products.
// ---------------------------------------------------------------------------
template <class T> struct FisherSums {
  T x = 0, xx = 0, xn = 0, n = 0, nn = 0, xy = 0;                        // columns
  T w = 0, xw = 0, nw = 0, ww = 0, xz = 0, wy = 0, wz = 0;               // columns, width terms
  T ry = 0, ryy = 0, ryn = 0, rw = 0, ryw = 0, rnw = 0, rww = 0;         // rows
  T s = 0;                                                               // sum of the weights
  template <bool SIG> __device__ __forceinline__ void column(const Band<T>& b, T C, T CC, T Y, T Z) {
    const T gp = b.dg * b.phi;
    x += b.dg * C;
    xx += b.dg * b.dg * CC;
    xn += gp * CC;
    n += b.phi * C;
    nn += b.phi * b.phi * CC;
    xy += gp * Y;
    if constexpr (SIG) {
      const T pw = b.phi * b.w;
      w += b.w * C;
      xw += b.dg * b.w * CC;
      nw += pw * CC;
      ww += b.w * b.w * CC;
      xz += gp * Z;
      wy += pw * Y;
      wz += pw * Z;
    }
  }
  template <bool SIG> __device__ __forceinline__ void row(const Band<T>& b, T R, T RR) {
    ry += b.dg * R;
    ryy += b.dg * b.dg * RR;
    ryn += b.dg * b.phi * RR;
    if constexpr (SIG) {
      rw += b.w * R;
      ryw += b.dg * b.w * RR;
      rnw += b.phi * b.w * RR;
      rww += b.w * b.w * RR;
    }
  }
};
// The upper triangle Fu (k <= l, row by row) from the sums and the axis
// constants: D = c dg, and the width or z derivative of an axis is e w.
template <int MODEL, class T>
__device__ __forceinline__ void fisher_entries(const FisherSums<T>& f, const AxisK<T>& kx, const AxisK<T>& ky,
                                               const Widths<T>& wd, T* Fu) {
  using Tr = MT<MODEL>;
  constexpr int P = Tr::P;
  auto set = [&](int k, int l, T v) __attribute__((always_inline)) {
    const int a = k < l ? k : l, b = k < l ? l : k;
    Fu[a * P - a * (a - 1) / 2 + (b - a)] = v;
  };
  set(Tr::IX, Tr::IX, kx.c * kx.c * f.xx);
  set(Tr::IX, Tr::IY, kx.c * ky.c * f.xy);
  set(Tr::IX, Tr::IN, kx.c * f.xn);
  set(Tr::IX, Tr::IBG, kx.c * f.x);
  set(Tr::IY, Tr::IY, ky.c * ky.c * f.ryy);
  set(Tr::IY, Tr::IN, ky.c * f.ryn);
  set(Tr::IY, Tr::IBG, ky.c * f.ry);
  set(Tr::IN, Tr::IN, f.nn);
  set(Tr::IN, Tr::IBG, f.n);
  set(Tr::IBG, Tr::IBG, f.s);
  if constexpr (Tr::EXTRA != 0) {
    const T ex = Tr::EXTRA == 3 ? wd.dsx * kx.cs() : kx.cs();
    const T ey = Tr::EXTRA == 3 ? wd.dsy * ky.cs() : ky.cs();
    const T xa = kx.c * ex * f.xw, xb = kx.c * ey * f.xz, ya = ky.c * ex * f.wy, yb = ky.c * ey * f.ryw;
    const T na = ex * f.nw, nb = ey * f.rnw, ba = ex * f.w, bb = ey * f.rw;
    const T aa = ex * ex * f.ww, ab = ex * ey * f.wz, bb2 = ey * ey * f.rww;
    if constexpr (Tr::EXTRA == 2) {
      set(Tr::IX, Tr::IE1, xa);
      set(Tr::IX, Tr::IE2, xb);
      set(Tr::IY, Tr::IE1, ya);
      set(Tr::IY, Tr::IE2, yb);
      set(Tr::IN, Tr::IE1, na);
      set(Tr::IN, Tr::IE2, nb);
      set(Tr::IBG, Tr::IE1, ba);
      set(Tr::IBG, Tr::IE2, bb);
      set(Tr::IE1, Tr::IE1, aa);
      set(Tr::IE1, Tr::IE2, ab);
      set(Tr::IE2, Tr::IE2, bb2);
    } else {
      set(Tr::IX, Tr::IE1, xa + xb);
      set(Tr::IY, Tr::IE1, ya + yb);
      set(Tr::IN, Tr::IE1, na + nb);
      set(Tr::IBG, Tr::IE1, ba + bb);
      set(Tr::IE1, Tr::IE1, aa + T(2) * ab + bb2);
    }
  }
}

// The Fisher sums of columns [c0, c0 + ncol) pixel by pixel, leaving out the
// pixels whose model is not > 0, as unified_kernel.jl:378-396 does.  The sums
// above give such pixels weight 0 instead, which a non-finite derivative
// (non-finite parameters, a width of 0) turns into NaN: an ROI whose matrix is
// not finite is done again here.  Rolled loops: rare, and small.
template <int MODEL, int CAM, int N, class T>
__device__ __forceinline__ void fisher_by_pixel(const T* th, const AxisK<T>& kx, const AxisK<T>& ky,
                                                const Widths<T>& wd, int c0, int ncol, const float* var, int ny,
                                                T* Fu) {
  using Tr = MT<MODEL>;
  constexpr int P = Tr::P;
  constexpr bool SIG = Tr::EXTRA != 0;
#pragma unroll
  for (int q = 0; q < P * (P + 1) / 2; ++q) Fu[q] = T(0);
#pragma unroll 1
  for (int cc = 0; cc < ncol; ++cc) {
    const T fc = (T)(c0 + cc);
    const Band<T> cx = band_from_edges<T, SIG>(edge_at<T, SIG>(kx, fc + T(0.5)), edge_at<T, SIG>(kx, fc + T(1.5)));
#pragma unroll 1
    for (int i = 0; i < N; ++i) {
      const Band<T> ry = band_from_edges<T, SIG>(edge_at<T, SIG>(ky, (T)i + T(0.5)), edge_at<T, SIG>(ky, (T)i + T(1.5)));
      const T mu = th[Tr::IBG] + th[Tr::IN] * cx.phi * ry.phi;
      if (mu > T(0)) {
        T wv = T(1) / mu;
        if constexpr (CAM == SCMOS) wv = T(1) / (mu + (T)var[(int64_t)(c0 + cc) * ny + i]);
        T du[P];
        du[Tr::IX] = kx.c * cx.dg * ry.phi;
        du[Tr::IY] = ky.c * ry.dg * cx.phi;
        du[Tr::IN] = cx.phi * ry.phi;
        du[Tr::IBG] = T(1);
        if constexpr (SIG) {
          const T ax = (Tr::EXTRA == 3 ? wd.dsx * kx.cs() : kx.cs()) * cx.w;
          const T ay = (Tr::EXTRA == 3 ? wd.dsy * ky.cs() : ky.cs()) * ry.w;
          if constexpr (Tr::EXTRA == 2) {
            du[Tr::IE1] = ax * ry.phi;
            du[Tr::IE2] = ay * cx.phi;
          } else {
            du[Tr::IE1] = ax * ry.phi + ay * cx.phi;
          }
        }
        int q = 0;
#pragma unroll
        for (int k = 0; k < P; ++k) {
          const T ak = du[k] * wv;
#pragma unroll
          for (int l = k; l < P; ++l) Fu[q++] += ak * du[l];
        }
      }
    }
  }
}

// Group sums of the Fisher entries and the LLR, with the pixel-by-pixel matrix
// where the summed one is not finite (every lane of an ROI takes the same
// turn: the group sums are the same on all of them).
template <int MODEL, int CAM, int N, int L, class T>
__device__ __forceinline__ FinalOut<T, MT<MODEL>::P> final_solve(const T* th, const AxisK<T>& kx, const AxisK<T>& ky,
                                                               const Widths<T>& wd, T* Fu, T llr, int c0, int ncol,
                                                               const float* var, int ny) {
  constexpr int P = MT<MODEL>::P;
  constexpr int NF = P * (P + 1) / 2;
  bool fin = true;
#pragma unroll
  for (int q = 0; q < NF; ++q) {
    Fu[q] = group_sum<L>(Fu[q]);
    fin = fin && __builtin_isfinite(Fu[q]);   // not x - x == 0: x is a product, which contracts into the difference
  }
  llr = group_sum<L>(llr);
  if (__builtin_amdgcn_ballot_w64(!fin) != 0) {
    T Fp[NF];
    fisher_by_pixel<MODEL, CAM, N, T>(th, kx, ky, wd, c0, fin ? 0 : ncol, var, ny, Fp);
#pragma unroll
    for (int q = 0; q < NF; ++q) {
      const T f = group_sum<L>(Fp[q]);
      Fu[q] = fin ? Fu[q] : f;
    }
  }
  FinalOut<T, P> out;
  out.llr = llr;
  T F[P * P];
  int q = 0;
#pragma unroll
  for (int k = 0; k < P; ++k)
#pragma unroll
    for (int l = k; l < P; ++l) {
      F[k + P * l] = Fu[q];
      F[l + P * k] = Fu[q];
      ++q;
    }
  invert_fisher<P, T>(F, out.crlb);
  return out;
}

// The Float32 final pass at the estimate th over this lane's register-resident
// pixels, rows outer and the row values shared as in accumulate().
template <int MODEL, int CAM, int N, int L>
__device__ __forceinline__ FinalOut<float, MT<MODEL>::P> final_pass_f32(const float* th, const float* psf, int c0,
                                                                      int r, const float* dv, const float* vr,
                                                                      const float* dt, const float* vt, float* roi,
                                                                      const float* var, int ny) {
  using Tr = MT<MODEL>;
  constexpr int P = Tr::P;
  constexpr bool TAIL = tail_split<N, L>();
  constexpr int CB = block_cols<N, L>();
  constexpr int RS = row_slots<N, L>();
  constexpr bool SIG = Tr::EXTRA != 0;
  Widths<float> wd;
  model_widths<MODEL, float>(th, psf, wd);
  const float nph = th[Tr::IN], bg = th[Tr::IBG];
  const AxisK<float> kx = axis_consts<float>(th[Tr::IX], wd.sx, nph);
  const AxisK<float> ky = axis_consts<float>(th[Tr::IY], wd.sy, nph);
  constexpr bool OWN = keep_own_rows<CAM, N, L>();
  RowVals own[OWN ? RS : 1];
  publish_rows<MODEL, N, L>(ky, r, roi, OWN ? own : nullptr);
  Band<float> cb[CB], tl{};
  column_bands<N, L, SIG>(kx, c0, cb, tl);
  float C[CB], CC[CB], Y[CB], Z[CB];
#pragma unroll
  for (int cc = 0; cc < CB; ++cc) C[cc] = CC[cc] = Y[cc] = Z[cc] = 0.f;
  FisherSums<float> f;
  float llr = 0.f;
  if constexpr (TAIL) {
    float Ct = 0.f, CCt = 0.f, Yt = 0.f, Zt = 0.f;
#pragma unroll
    for (int s = 0; s < RS; ++s) {
      const RowVals v = OWN ? own[s] : read_row<MODEL, L>(roi, r * RS + s);
      const Band<float> b{v.phi, v.dg, v.w, 0.f};
      const float mu = fmaf(nph * tl.phi, b.phi, bg);
      float lp, wv;
      final_weights<CAM>(dt[s], CAM == SCMOS ? vt[s] : 0.f, mu, lp, wv);
      if ((L - 1) * RS + s >= N) {
        const bool ok = r * RS + s < N;
        lp = ok ? lp : 0.f;
        wv = ok ? wv : 0.f;
      }
      llr += lp;
      const float pw = b.phi * wv, xw = tl.phi * wv;
      Ct += pw;
      CCt = fmaf(b.phi, pw, CCt);
      Yt = fmaf(b.dg, pw, Yt);
      if constexpr (SIG) Zt = fmaf(b.w, pw, Zt);
      f.s += wv;
      f.row<SIG>(b, xw, tl.phi * xw);
    }
    f.column<SIG>(tl, Ct, CCt, Yt, Zt);
  }
  RowVals next = read_row<MODEL, L>(roi, 0);   // with one column per lane, a row ahead
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_barrier(0);   // as in accumulate()
    const RowVals v = CB == 1 ? next : read_row<MODEL, L>(roi, i);
    if (CB == 1 && i + 1 < N) next = read_row<MODEL, L>(roi, i + 1);
    const Band<float> b{v.phi, v.dg, v.w, 0.f};
    const float pn = nph * b.phi;
    float R = 0.f, RR = 0.f;
#pragma unroll
    for (int cc = 0; cc < CB; ++cc) {
      const float mu = fmaf(cb[cc].phi, pn, bg);
      float lp, wv;
      final_weights<CAM>(dv[cc * N + i], CAM == SCMOS ? vr[cc * N + i] : 0.f, mu, lp, wv);
      if (may_pad<N, L>(cc)) {
        lp = c0 + cc < N ? lp : 0.f;
        wv = c0 + cc < N ? wv : 0.f;
      }
      llr += lp;
      const float pw = b.phi * wv, xw = cb[cc].phi * wv;
      C[cc] += pw;
      CC[cc] = fmaf(b.phi, pw, CC[cc]);
      Y[cc] = fmaf(b.dg, pw, Y[cc]);
      if constexpr (SIG) Z[cc] = fmaf(b.w, pw, Z[cc]);
      R += xw;
      RR = fmaf(cb[cc].phi, xw, RR);
      f.s += wv;
    }
    f.row<SIG>(b, R, RR);
#pragma unroll
    for (int cc = 0; cc < CB; ++cc) {
      asm volatile("" : "+v"(C[cc]), "+v"(CC[cc]), "+v"(Y[cc]));
      if constexpr (SIG) asm volatile("" : "+v"(Z[cc]));
    }
    asm volatile("" : "+v"(f.ry), "+v"(f.ryy), "+v"(f.ryn), "+v"(f.s), "+v"(llr));
  }
#pragma unroll
  for (int cc = 0; cc < CB; ++cc) f.column<SIG>(cb[cc], C[cc], CC[cc], Y[cc], Z[cc]);
  float Fu[P * (P + 1) / 2];
  fisher_entries<MODEL, float>(f, kx, ky, wd, Fu);
  // columns of this lane; the last lane takes the tail column whole
  int ncol = N - c0 < CB ? (N - c0 < 0 ? 0 : N - c0) : CB;
  if (TAIL && r == L - 1) ncol = CB + 1;
  if (CAM == SCMOS && var == nullptr) ncol = 0;   // outside the variance map: nothing to read
  return final_solve<MODEL, CAM, N, L, float>(th, kx, ky, wd, Fu, llr, c0, ncol, var, ny);
}

// Out-of-range sCMOS corner: no fit, NaN outputs.
template <class TF, int P> __device__ __forceinline__ void nan_outputs(float* th, FinalOut<TF, P>& fo) {
  const float qnan = __builtin_nanf("");
#pragma unroll
  for (int k = 0; k < P; ++k) {
    th[k] = qnan;
    fo.crlb[k] = TF(qnan);
  }
  fo.llr = TF(qnan);
}

template <int P, class TF>
__device__ __forceinline__ void store_outputs(const FitArgs& a, int64_t out, int stride, const float* th,
                                              const FinalOut<TF, P>& fo) {
#pragma unroll
  for (int k = 0; k < P; ++k) {
    a.params[out * stride + k] = th[k];
    a.crlb[out * stride + k] = (float)fo.crlb[k];
  }
  a.llr[out] = (float)fo.llr;
  for (int k = P; k < stride; ++k) {   // mixed-model batches: unused parameter slots
    a.params[out * stride + k] = __builtin_nanf("");
    a.crlb[out * stride + k] = __builtin_nanf("");
  }
}

// ---------------------------------------------------------------------------
// The kernel.
// ---------------------------------------------------------------------------
// Where one ROI's pixels live and where its results go.
struct RoiRef {
  const float* data;   // the ROI's first pixel (column-major N x N)
  int64_t out;         // output slot
  int stride;          // params / crlb values per slot
  int cx, cy;          // 1-based camera corner (sCMOS)
};

// One ROI, fitted by the L lanes of its group (lane r of the group owns
// columns [r*CB, r*CB + CB)).  Every lane of the wave must call this (the
// cross-lane sums use DPP); `active` lanes store the results.
template <int MODEL, int CAM, int N, int L, int PREC>
__device__ __forceinline__ void fit_one(const FitArgs& a, const RoiRef& ref, bool active, int r, float* lds) {
  using Tr = MT<MODEL>;
  constexpr int P = Tr::P;
  constexpr bool TAIL = tail_split<N, L>();
  constexpr int CB = block_cols<N, L>();   // full columns per lane
  constexpr int RS = row_slots<N, L>();                 // tail split: rows of the last column per lane
  constexpr bool SIG = Tr::EXTRA != 0;  // sigma / z terms present
  constexpr bool OWN = keep_own_rows<CAM, N, L>();
  const int c0 = r * CB;
  // this ROI's row values (publish_rows)
  const int lane = threadIdx.x & (kWave - 1);
  float* roi = L == 1 ? lds + 4 * lane : lds + lane / L * roi_words<MODEL, N, L>();
  float* park = lds + rows_words<MODEL, N, L>() + (SIG ? 4 : 2) * lane;   // its columns' (park_band)

  // ---- load this lane's column block (and variances) once ----------------
  float dv[CB * N];
  float vr[CAM == SCMOS ? CB * N : 1];
  float dt[TAIL ? RS : 1];
  float vt[(TAIL && CAM == SCMOS) ? RS : 1];
  const float* src = ref.data;
  float dmax_l = 0.f;
  int cxc = 1, cyc = 1;
  bool inb = true;   // sCMOS ROI inside the variance map
  if constexpr (CAM == SCMOS) {
    cxc = ref.cx;
    cyc = ref.cy;
    inb = (cxc >= 1) && (cyc >= 1) && (cxc <= a.nx - N + 1) && (cyc <= a.ny - N + 1);
  }
  // Each column is a contiguous run of N floats in the ROI and in the variance
  // map: read in 16-byte loads (load_run), since a wave's lanes are ROIs apart
  // and every load instruction touches one cache line per lane.
#pragma unroll
  for (int cc = 0; cc < CB; ++cc) {
    const int col = c0 + cc;
    const bool valid = (L == 1) || TAIL || (col < N);
    if (valid) {
      load_run<N>(src + col * N, dv + cc * N);
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) dv[cc * N + i] = 0.f;
    }
    if constexpr (CAM == SCMOS) {
      if (valid && inb) {
        load_run<N>(a.var_map + (int64_t)(cyc - 1) + (int64_t)a.ny * (int64_t)(cxc - 1 + col), vr + cc * N);
      } else {
        // an infinite variance gives a padding column's pixels weight 0
        const float fill = valid ? 0.f : __builtin_inff();
#pragma unroll
        for (int i = 0; i < N; ++i) vr[cc * N + i] = fill;
      }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) dmax_l = fmaxf(dmax_l, dv[cc * N + i]);
  }
  if constexpr (TAIL) {
    // rows [r RS, r RS + RS) of the last column; slots past the last row hold
    // zeros (the row index is clamped, so no load leaves the ROI)
#pragma unroll
    for (int s = 0; s < RS; ++s) {
      const int ri = r * RS + s;
      const bool ok = ri < N;
      const int rc = ok ? ri : N - 1;
      const float x = src[(N - 1) * N + rc];
      dt[s] = ok ? x : 0.f;
      if constexpr (CAM == SCMOS) {
        if (inb) {
          const float v = a.var_map[(int64_t)(cyc - 1 + rc) + (int64_t)a.ny * (int64_t)(cxc - 1 + N - 1)];
          vt[s] = ok ? v : 0.f;
        } else {
          vt[s] = 0.f;
        }
      }
      dmax_l = fmaxf(dmax_l, dt[s]);
    }
  }
  const float dmax = group_max<L>(dmax_l);

  // ---- initial estimates (unified_kernel.jl:158-255) ---------------------
  float th[P];
  {
    float esum = 0.f;
#pragma unroll
    for (int cc = 0; cc < CB; ++cc) {
      const int col = c0 + cc;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const bool edge = (i == 0) || (i == N - 1) || (col == 0) || (col == N - 1);
        if (edge) esum += dv[cc * N + i];   // invalid columns hold zeros
      }
    }
    if constexpr (TAIL) {
#pragma unroll
      for (int s = 0; s < RS; ++s) esum += dt[s];   // the last column is an edge column
    }
    esum = group_sum<L>(esum);
    const float bg0 = esum / (float)(4 * N - 4);
    float tot = 0.f, xw = 0.f, yw = 0.f;
#pragma unroll
    for (int cc = 0; cc < CB; ++cc) {
      const bool valid = (L == 1) || TAIL || (c0 + cc < N);
      const float fj = (float)(c0 + cc + 1);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const float s = valid ? fmaxf(0.f, dv[cc * N + i] - bg0) : 0.f;
        tot += s;
        xw += s * fj;
        yw += s * (float)(i + 1);
      }
    }
    if constexpr (TAIL) {
#pragma unroll
      for (int s = 0; s < RS; ++s) {
        const int ri = r * RS + s;
        const float v = ri < N ? fmaxf(0.f, dt[s] - bg0) : 0.f;
        tot += v;
        xw += v * (float)N;
        yw += v * (float)(ri + 1);
      }
    }
    tot = group_sum<L>(tot);
    xw = group_sum<L>(xw);
    yw = group_sum<L>(yw);
    const float center = (float)(N + 1) * 0.5f;
    float x0 = tot > 10.f ? xw / tot : center;
    float y0 = tot > 10.f ? yw / tot : center;
    x0 = jclamp(x0, 1.5f, (float)N - 0.5f);
    y0 = jclamp(y0, 1.5f, (float)N - 0.5f);
    const float ph = fmaxf(tot, 100.f);
    th[Tr::IX] = x0;
    th[Tr::IY] = y0;
    th[Tr::IN] = ph;
    th[Tr::IBG] = bg0;
    if constexpr (MODEL == XYNBS) th[4] = 1.3f;
    if constexpr (MODEL == XYNBSXSY) { th[4] = 1.3f; th[5] = 1.3f; }
    if constexpr (MODEL == ASTIG) {
      float mxx = 0.f, myy = 0.f;
      float b0 = bg0;   // s again from the pixel, instead of every pixel's s kept from above
      asm volatile("" : "+v"(b0));
#pragma unroll
      for (int cc = 0; cc < CB; ++cc) {
        const bool valid = (L == 1) || TAIL || (c0 + cc < N);
        const float dxp = (float)(c0 + cc + 1) - x0;
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const float s = valid ? fmaxf(0.f, dv[cc * N + i] - b0) : 0.f;
          const float dyp = (float)(i + 1) - y0;
          mxx += s * dxp * dxp;
          myy += s * dyp * dyp;
        }
      }
      if constexpr (TAIL) {
        const float dxp = (float)N - x0;
#pragma unroll
        for (int s = 0; s < RS; ++s) {
          const int ri = r * RS + s;
          const float v = ri < N ? fmaxf(0.f, dt[s] - b0) : 0.f;
          const float dyp = (float)(ri + 1) - y0;
          mxx += v * dxp * dxp;
          myy += v * dyp * dyp;
        }
      }
      mxx = group_sum<L>(mxx);
      myy = group_sum<L>(myy);
      float z0 = 0.f;
      if (tot > 10.f) {
        const float sxe = sqrtf(fmaxf(0.5f, mxx / tot));
        const float sye = sqrtf(fmaxf(0.5f, myy / tot));
        const float rx = sxe / a.psf[0], ry = sye / a.psf[1];
        const float dal = rx * rx - ry * ry;
        z0 = -dal * (a.psf[7] * a.psf[7]) / (4.f * a.psf[6]);
        z0 = jclamp(z0, -600.f, 600.f);
      }
      th[2] = z0;
    }
  }

  // ---- Newton-Raphson iterations (unified_kernel.jl:314-351) -------------
  for (int it = 0; it < a.iterations; ++it) {
    Widths<float> w;
    model_widths<MODEL, float>(th, a.psf, w);
    const float nph = th[Tr::IN];
    const float bg = th[Tr::IBG];

    // Poisson fast path: every pixel has model > 0.01 and no cap can bind.
    // model >= bg - N*tiny for N <= 1e5 (phi >= 0 up to erf rounding), so
    // bg >= 0.05 keeps it above 0.01, and dmax <= 5000 bg min(bg,1) keeps
    // data/model - 1 and data/model^2 below 1e4.
    bool fast = false;
    if constexpr (CAM == IDEAL) {
      bool fin = true;
#pragma unroll
      for (int k = 0; k < P; ++k) fin = fin && (fabsf(th[k]) < 3.0e38f);
      fast = fin && (bg >= 0.05f) && (nph >= 0.f) && (nph <= 1.0e5f) &&
             (dmax <= 5000.f * bg * fminf(bg, 1.f));
    }

    float G[P], H[P];
    const AxisK<float> kx = axis_consts<float>(th[Tr::IX], w.sx, nph);
    const AxisK<float> ky = axis_consts<float>(th[Tr::IY], w.sy, nph);
    RowVals own[OWN ? RS : 1];
    publish_rows<MODEL, N, L>(ky, r, roi, OWN ? own : nullptr);
    // One form for the whole wave: where some ROI needs the masks, running both
    // in turn would cost the others' pixel loop again (XYNB 11 px, backgrounds
    // of 1-20 photons: 1.271 -> 1.254 ms per 1M ROIs, 40.9 -> 39.7 us per 10,000).
    PixelSums u;
    if (__builtin_amdgcn_ballot_w64(CAM == IDEAL && !fast) == 0) {
      accumulate<MODEL, CAM, N, L, true>(dv, vr, dt, vt, c0, r, nph, bg, kx, ky, roi, own, park, u);
    } else {
      accumulate<MODEL, CAM, N, L, false>(dv, vr, dt, vt, c0, r, nph, bg, kx, ky, roi, own, park, u);
    }
    gradient<MODEL>(u, kx, ky, w, G, H);
#pragma unroll
    for (int k = 0; k < P; ++k) {
      G[k] = group_sum<L>(G[k]);
      H[k] = group_sum<L>(H[k]);
    }
    // Scalar Newton step with constraints (unified_kernel.jl:337-350, constraints.jl:172-177).
    // G / H is a v_rcp_f32 and a multiply (1 ulp more than the division) where
    // both are below 1e30 in magnitude; a lane with a NaN, an infinity or a
    // value beyond that takes the IEEE division, so those cases come out as
    // the division gives them.  The division runs only in a wave that has
    // such a lane.  One sum of the magnitudes is tested: it is NaN, infinite or
    // large where one of them is, and a test of each became a packed bit mask of
    // three instructions per value.
    float step[P], size = 0.f;
#pragma unroll
    for (int k = 0; k < P; ++k) {
      const float g = G[k], h = H[k];
      step[k] = fabsf(h) > 1e-10f ? g * __builtin_amdgcn_rcpf(h) : 0.f;
      size += fabsf(g) + fabsf(h);
    }
    const bool exact = size < 1e30f;
    if (__builtin_amdgcn_ballot_w64(!exact) != 0) {
#pragma unroll
      for (int k = 0; k < P; ++k)
        if (!exact) step[k] = fabsf(H[k]) > 1e-10f ? G[k] / H[k] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < P; ++k) {
      const float ms = a.max_step[k];
      const float t = th[k] - jclamp(step[k], -ms, ms);
      th[k] = jclamp(t, a.lower[k], a.upper[k]);
    }
  }

  // ---- final pass: LLR + Fisher + CRLB (unified_kernel.jl:353-433) --------
  // Float32 here; the Float64 final pass runs as its own kernel
  // (final_pass_kernel) so that its registers do not lower this kernel's
  // occupancy.
  if constexpr (PREC == PREC_FP32) {
    const float* var = nullptr;   // the ROI's corner of the variance map
    if constexpr (CAM == SCMOS) {
      if (inb) var = a.var_map + (int64_t)(cyc - 1) + (int64_t)a.ny * (int64_t)(cxc - 1);
    }
    FinalOut<float, P> fo =
        final_pass_f32<MODEL, CAM, N, L>(th, a.psf, c0, r, dv, vr, dt, vt, roi, var, a.ny);
    if (!inb) nan_outputs(th, fo);
    if (active && r == 0) store_outputs<P>(a, ref.out, ref.stride, th, fo);
  } else {
    if (!inb) {
#pragma unroll
      for (int k = 0; k < P; ++k) th[k] = __builtin_nanf("");
    }
    if (active && r == 0) {
#pragma unroll
      for (int k = 0; k < P; ++k) a.params[ref.out * ref.stride + k] = th[k];
    }
  }
}

// The ROI that lane group `j` of a launch fits, and whether it stores.
// Inactive groups (past the end, or skipped batch slots) fit a valid ROI of
// the same shape and discard the result.
template <int MODEL, int CAM, int N>
__device__ __forceinline__ bool locate_roi(const FitArgs& a, int64_t j, int64_t fallback, RoiRef& ref) {
  bool active = j < a.n_rois;
  int64_t roi = active ? j : fallback;
  int64_t off = roi * (int64_t)(N * N);
  if (a.order) {
    const int32_t k = a.order[a.first + roi];
    active = active && (k >= 0);
    roi = (k >= 0) ? k : a.order[a.first + fallback];
    off = a.offsets[roi];
  }
  ref.data = a.data + off;
  ref.out = roi;
  ref.stride = a.out_stride > 0 ? a.out_stride : MT<MODEL>::P;
  ref.cx = ref.cy = 1;
  if constexpr (CAM == SCMOS) {
    ref.cx = a.x_corners[roi];
    ref.cy = a.y_corners[roi];
  }
  return active;
}

// One launch over n ROIs of one shape: 64/L ROIs per wave, in wave-sized
// tiles (a grid smaller than the tile count strides over the rest).
template <int MODEL, int CAM, int N, int L, int PREC>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(min_waves<MODEL, CAM, N, L>())))
void fit_kernel(FitArgs a) {
  constexpr int RPW = kWave / L;
  const int lane = threadIdx.x;
  const int r = (L == 1) ? 0 : (lane & (L - 1));
  // A batch slot range whose first entry is empty holds no ROI of this shape.
  if (a.n_rois <= 0 || (a.order && __builtin_amdgcn_readfirstlane(a.order[a.first]) < 0)) return;
  for (int64_t base = (int64_t)blockIdx.x * RPW; base < a.n_rois; base += (int64_t)gridDim.x * RPW) {
    RoiRef ref;
    const bool active = locate_roi<MODEL, CAM, N>(a, base + lane / L, 0, ref);
    fit_one<MODEL, CAM, N, L, PREC>(a, ref, active, r, wave_lds<wave_words<MODEL, CAM, N, L>()>());
  }
}

// Float64 final pass at the estimates the iteration kernel wrote to params,
// one lane per ROI; the ROI is re-read from HBM (once) instead of being held
// in VGPRs.  Two waves per SIMD are requested: from 12 px up the compiler then
// spills a few dozen values to scratch (astig 15 px: 284 -> 256 VGPRs, 29
// spilled), which costs less than running one wave per SIMD (gfx950: the
// astigmatic 15 px pass 18 % faster).
template <int MODEL, int CAM, int N>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(2))) void final_pass_kernel(FitArgs a) {
  constexpr int P = MT<MODEL>::P;
  if (a.n_rois <= 0 || (a.order && __builtin_amdgcn_readfirstlane(a.order[a.first]) < 0)) return;
  RoiRef ref;
  const bool active = locate_roi<MODEL, CAM, N>(a, (int64_t)blockIdx.x * kWave + threadIdx.x, 0, ref);
  if (!active) return;
  const int64_t slot = ref.out;
  float th[P];
#pragma unroll
  for (int k = 0; k < P; ++k) th[k] = a.params[slot * ref.stride + k];
  GlobalSrc<N, CAM == SCMOS> src;
  src.data = ref.data;
  bool inb = true;
  if constexpr (CAM == SCMOS) {
    const int cx = ref.cx, cy = ref.cy;
    inb = (cx >= 1) && (cy >= 1) && (cx <= a.nx - N + 1) && (cy <= a.ny - N + 1);
    src.var = a.var_map + (int64_t)(cy - 1) + (int64_t)a.ny * (int64_t)(cx - 1);
    src.ny = a.ny;
    if (!inb) src.var = nullptr;
  }
  FinalOut<double, P> fo;
  if (inb) {
    fo = final_pass<MODEL, CAM, N, 1, double>(th, a.psf, 0, src);
  } else {
    nan_outputs(th, fo);
  }
  store_outputs<P>(a, slot, ref.stride, th, fo);
  if (a.crlb64) {
#pragma unroll
    for (int k = 0; k < P; ++k) a.crlb64[slot * ref.stride + k] = fo.crlb[k];
    for (int k = P; k < ref.stride; ++k) a.crlb64[slot * ref.stride + k] = __builtin_nan("");
  }
  if (a.llr64) a.llr64[slot] = fo.llr;
}

// The Float64 final pass of large boxes (N > kMaxSmallBox): L lanes per ROI
// as in the iteration kernel, each holding its column block in VGPRs (read
// once from HBM in 16-byte runs), rows in the outer loop.
template <int MODEL, int CAM, int N, int L>
__global__ __launch_bounds__(kWave) void final_pass_lanes_kernel(FitArgs a) {
  constexpr int P = MT<MODEL>::P;
  constexpr int RPW = kWave / L;
  constexpr int CB = (N + L - 1) / L;
  const int lane = threadIdx.x;
  const int r = lane & (L - 1);
  const int c0 = r * CB;
  if (a.n_rois <= 0 || (a.order && __builtin_amdgcn_readfirstlane(a.order[a.first]) < 0)) return;
  for (int64_t base = (int64_t)blockIdx.x * RPW; base < a.n_rois; base += (int64_t)gridDim.x * RPW) {
    RoiRef ref;
    const bool active = locate_roi<MODEL, CAM, N>(a, base + lane / L, 0, ref);
    const int64_t slot = ref.out;
    float th[P];
#pragma unroll
    for (int k = 0; k < P; ++k) th[k] = a.params[slot * ref.stride + k];
    bool inb = true;
    if constexpr (CAM == SCMOS)
      inb = (ref.cx >= 1) && (ref.cy >= 1) && (ref.cx <= a.nx - N + 1) && (ref.cy <= a.ny - N + 1);
    float dv[CB * N];
    float vr[CAM == SCMOS ? CB * N : 1];
#pragma unroll
    for (int cc = 0; cc < CB; ++cc) {
      const int col = c0 + cc;
      if (col < N) {
        load_run<N>(ref.data + col * N, dv + cc * N);
      } else {
#pragma unroll
        for (int i = 0; i < N; ++i) dv[cc * N + i] = 0.f;
      }
      if constexpr (CAM == SCMOS) {
        if (col < N && inb) {
          load_run<N>(a.var_map + (int64_t)(ref.cy - 1) + (int64_t)a.ny * (int64_t)(ref.cx - 1 + col), vr + cc * N);
        } else {
#pragma unroll
          for (int i = 0; i < N; ++i) vr[cc * N + i] = 0.f;
        }
      }
    }
    const RegSrc<N, CAM == SCMOS> src{dv, vr};
    FinalOut<double, P> fo = final_pass_rows<MODEL, CAM, N, L, double>(th, a.psf, c0, src);
    if (!inb) nan_outputs(th, fo);
    if (active && r == 0) {
      store_outputs<P>(a, slot, ref.stride, th, fo);
      if (a.crlb64) {
#pragma unroll
        for (int k = 0; k < P; ++k) a.crlb64[slot * ref.stride + k] = fo.crlb[k];
        for (int k = P; k < ref.stride; ++k) a.crlb64[slot * ref.stride + k] = __builtin_nan("");
      }
      if (a.llr64) a.llr64[slot] = fo.llr;
    }
  }
}

template <int MODEL, int CAM, int N, int L, int PREC>
bool describe_fit(KernelInfo* k) {
  k->fit = reinterpret_cast<const void*>(&fit_kernel<MODEL, CAM, N, L, PREC>);
  k->rois_per_block = kWave / L;
  k->final_pass = nullptr;
  k->final_rois_per_block = kWave;
  if constexpr (PREC == PREC_MIXED) {
    if constexpr (N > kMaxSmallBox) {
      k->final_pass = reinterpret_cast<const void*>(&final_pass_lanes_kernel<MODEL, CAM, N, L>);
      k->final_rois_per_block = kWave / L;
    } else {
      k->final_pass = reinterpret_cast<const void*>(&final_pass_kernel<MODEL, CAM, N>);
    }
  }
  return true;
}

template <int MODEL, int CAM, int N, int L, int PREC>
hipError_t launch_fit(const FitArgs& a, hipStream_t stream) {
  constexpr int RPW = kWave / L;
  const int64_t blocks = (a.n_rois + RPW - 1) / RPW;
  if (blocks <= 0) return hipSuccess;
  hipLaunchKernelGGL((fit_kernel<MODEL, CAM, N, L, PREC>), dim3((unsigned)blocks), dim3(kWave), 0, stream, a);
  if constexpr (PREC == PREC_MIXED) {
    if constexpr (N > kMaxSmallBox) {
      hipLaunchKernelGGL((final_pass_lanes_kernel<MODEL, CAM, N, L>), dim3((unsigned)blocks), dim3(kWave), 0, stream,
                         a);
    } else {
      const int64_t fblocks = (a.n_rois + kWave - 1) / kWave;
      hipLaunchKernelGGL((final_pass_kernel<MODEL, CAM, N>), dim3((unsigned)fblocks), dim3(kWave), 0, stream, a);
    }
  }
  return hipGetLastError();
}

}  // namespace gmle
