// gmle_boxer.hip -- candidate boxes cut from camera frames on the device.
//
// The step before the fit in GaussMLE.jl's pipeline is SMLMBoxer.getboxes
// (examples/full_pipeline_boxer.jl:70-80, examples/full_pipeline.jl:73-81):
// a difference-of-Gaussians filter, local maxima above `minval`, boxes of
// `boxsize` pixels around them that overlap by at most `overlap` pixels, cut
// from the raw frames into a ROIBatch.  Here every step runs on the device:
//
//   D = G(sigma_small) * I - G(sigma_large) * I
//     separable, replicated edges; 1-D weights exp(-k^2 / (2 sigma^2)) for
//     |k| <= floor(3 sigma + 0.5), normalised to sum 1 (computed on the host in
//     Float64: sum = g0 + 2 g1 + 2 g2 + ..., then each weight rounded to
//     Float32); each pass is v = w0 x0 + sum_k w_k (x_-k + x_k), accumulated
//     by fma in increasing k; columns (x) first, then rows (y).
//   detection: D(p) > minval and no pixel q of the frame within Chebyshev
//     distance r of p beats it, where q beats p if D(q) > D(p) or D(q) == D(p)
//     and q comes first in column-major order; r = ceil(boxsize - overlap) - 1
//     (at least 1), so kept detections are at least boxsize - overlap apart.
//   box: top-left corner (row, col) = detection - (boxsize - 1) / 2, clamped
//     into the frame; the ROI holds the raw input pixels.
//   order: by frame, then column-major pixel index (Julia's findall order).
//
// Kernels (all deterministic; no atomics):
//   1. boxer_detect: filters and finds the 3 x 3 maxima above minval (a
//      necessary condition) in one sweep.  Writes one 64-bit word of candidates
//      per column and word_rows rows.  D stays in LDS except around pixels
//      above minval: where a step of a wave has one, its D is stored and its
//      words are flagged.  (Anything not stored is at most minval and beats no
//      candidate.)
//   2. boxer_suppress: one candidate word per lane; a wave tests its lanes'
//      candidates one at a time, reading each window with all 64 lanes;
//      survivors per block of words.
//   3. boxer_scan: exclusive scan of the block counts; total detections.
//   4. boxer_place: each survivor's rank from the scan -> corners and frame;
//      then the block copies its boxes, one wave per box.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/gaussmle.h"
#include "gmle_args.hpp"
#include "gmle_host.hpp"

namespace gmle {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kMaxRadius = 12;     // weights radius limit: sigma <= 4 px
constexpr int kStep = 8;           // columns per step of the sweep
constexpr int kStrip = 8;          // rows per thread of the y pass
constexpr int kRing = 16;          // columns of D in LDS, at least kStep + 2
constexpr uint64_t kStored = 1ull << 63;   // candidate word: D of its rows is stored
constexpr int kWordsPerThread = 4; // boxer_suppress / boxer_place, at most
constexpr int kScanThreads = 1024;
constexpr int kTargetBlocks = 3 * 5 * 256;   // boxer_detect runs five blocks per CU
constexpr int kMinSweep = 24;
constexpr int64_t kManyWords = 1 << 19;

struct BoxerArgs {
  const float* frames;   // (ny, nx, nf) column-major
  int ny, nx, nf;
  int rs, rl;            // weight radii of the two kernels
  int halo;              // max(rs, rl)
  float ws[kMaxRadius + 1];
  float wl[kMaxRadius + 1];
  float minval;
  int win;               // suppression radius r
  int box;
  int word_rows;         // rows per word
  int wpc;               // words per column: ceil(ny / word_rows)
  int sweep;             // columns per block of boxer_detect
  int64_t n_words;       // nf * nx * wpc
  int64_t max_boxes;
  int wpt;               // words per thread of suppress / place: 1, or kWordsPerThread for large stacks
  float* dog;            // (ny, nx, nf), where the word is kStored
  uint64_t* cand;        // (wpc, nx, nf); bit b of word w <-> row word_rows w + b
  uint64_t* keep;        // (wpc, nx, nf)
  int64_t* block_base;   // per suppress / place block
  int64_t* count;        // total detections
  float* rois;           // (box, box, max_boxes)
  int32_t* xc;
  int32_t* yc;
  int32_t* frame;
  float* strength;       // D at the detection (may be null)
};

// Rows per candidate word: four words and a halo of radius + 1 above and below
// fit the 256 rows of a block.
__host__ __device__ constexpr int word_rows_of(int rmax) { return rmax <= 6 ? 60 : 56; }

// One Gaussian over a register strip: out[o] = w0 x[c+o] + sum_k w_k
// (x[c+o-k] + x[c+o+k]), fma in increasing k, c = RMAX.  The radius is FIXED,
// or the uniform R where FIXED is 0.
template <int RMAX, int FIXED, int N>
__device__ __forceinline__ void strip_filter(const float (&x)[N + 2 * RMAX], const float* w, int R, float (&out)[N]) {
#pragma clang fp contract(off)
  const float w0 = w[0];
#pragma unroll
  for (int o = 0; o < N; ++o) out[o] = w0 * x[RMAX + o];
#pragma unroll
  for (int k = 1; k <= (FIXED ? FIXED : RMAX); ++k) {
    if (FIXED || k <= R) {
      const float wk = w[k];
#pragma unroll
      for (int o = 0; o < N; ++o) out[o] = fmaf(wk, x[RMAX + o - k] + x[RMAX + o + k], out[o]);
    }
  }
}

// LDS layout of a column of 256 rows: the rows' even groups of four, then the
// odd groups.  The y pass reads and writes groups of four rows (16 bytes) with
// its lanes two groups apart, which in plain order meets every other bank only
// (measured: 21 conflict cycles per access); here those lanes lie next to each
// other.  The odd half is turned by 32 words, so that consecutive rows, as the
// x pass writes and the test reads them, meet different banks too.
constexpr int kColumn = 256;
constexpr int kHalf = kColumn / 2;
__device__ __forceinline__ int even_slot(int pair) { return 4 * pair; }
__device__ __forceinline__ int odd_slot(int pair) { return kHalf + ((4 * pair + 32) & (kHalf - 1)); }
__device__ __forceinline__ int row_slot(int r) {
  return ((r & 4) ? odd_slot(r >> 3) : even_slot(r >> 3)) + (r & 3);
}

// Filter and 3 x 3 maxima above minval, one sweep.
//
// Block (x, y, z): columns [sweep x, sweep (x + 1)), rows [4 word_rows y, ...)
// of frame z.  256 threads hold 256 consecutive rows (the contiguous axis),
// 1 + RMAX of them above the block's first; the block walks right in steps of
// kStep columns:
//   x pass: thread t keeps the last 2 RMAX columns of its row in registers,
//     loads kStep more (256 contiguous bytes per wave and column) and writes
//     both filtered rows to LDS;
//   y pass: thread (strip, column) filters 8 rows of one column from LDS in
//     16-byte reads and writes D to a ring of kRing columns;
//   test: the columns with both neighbours in the ring, one wave per word,
//     lanes over rows; a wave goes further only where a pixel exceeds minval.
// So every input pixel is read once per row band, and D goes to memory only
// around bright pixels.
// RS and RL are the two radii, or 0 where they come from `a`.
//
// What bounds it: VALU issue (45 of the 70 instructions per pixel are the taps)
// and the two barriers of a step.  32 frames of 2048 x 2048, boxsize 11: the
// whole call 0.594 -> 0.303 ms against 0.13 ms for one read of the frames.  The
// tile kernel before it (62 x 30 pixels, every value of three LDS images read
// one at a time, D of every pixel written and read back) took 0.54 of 0.60 ms.
// Suppressing in this kernel, with the halo and the ring that needs, took 0.47:
// a block then waits for its slowest wave at every candidate.  Filtering the
// window of each candidate again in boxer_suppress took 0.35, but three times
// as long as before where a low minval makes one pixel in fifteen a candidate.
template <int RMAX, int RS, int RL>
__global__ __launch_bounds__(kBlock) void boxer_detect(BoxerArgs a) {
#pragma clang fp contract(off)
  constexpr int kDRows = kBlock - 2 * RMAX;            // rows of D that are complete
  // 32 strips, so that half a wave is one column and its 16-byte accesses are
  // free of conflicts; the last strips' rows past kDRows are filtered from
  // whatever lies past row 255, and nothing uses them.
  constexpr int kStrips = kColumn / kStrip;
  static_assert(kStrips * kStep == kBlock, "y pass layout");
  static_assert(4 * word_rows_of(RMAX) + 2 <= kDRows && kRing >= kStep + 2, "halo");
  __shared__ __attribute__((aligned(16))) float lds[(2 * kStep + kRing) * kColumn];
  float* hs = lds;
  float* hl = hs + kStep * kColumn;
  float* ring = hl + kStep * kColumn;
  constexpr int kWord = word_rows_of(RMAX);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int f = blockIdx.z;
  const int band = blockIdx.y * 4 * kWord;             // first row tested
  const int first = blockIdx.x * a.sweep;              // first column tested
  const int last = min(first + a.sweep, a.nx);
  const size_t plane = (size_t)a.ny * a.nx;
  const float* src = a.frames + (size_t)f * plane + min(max(band - 1 - RMAX + t, 0), a.ny - 1);
  const int row0 = band - 1;                           // row of D's index 0
  const int col0 = first - 1;                          // column of D's ring index 0
  auto pixel = [&](int c) { return src[(size_t)min(max(c, 0), a.nx - 1) * a.ny]; };

  float x[kStep + 2 * RMAX];
#pragma unroll
  for (int i = 0; i < kStep + 2 * RMAX; ++i) x[i] = pixel(col0 - RMAX + i);
  const int steps = (last - first + 2 + kStep - 1) / kStep;
  const int ys = t % kStrips, yc = t / kStrips;        // y pass: strip and column of the step
  const int slot = row_slot(t);
  // the test's row, and the slots of the rows around it in a column of D
  const int gr = band + wave * kWord + lane;
  const bool mine = lane < kWord && gr < a.ny;
  const int own = row_slot(gr - row0), up = row_slot(gr - row0 - 1), down = row_slot(gr - row0 + 1);
  const bool has_up = gr >= 1, has_down = gr + 1 < a.ny;
  const float ninf = -__builtin_inff();
  const int wi = blockIdx.y * 4 + wave;                // word of the column
  for (int s = 0; s < steps; ++s) {
    const int base = s * kStep;                        // ring column (not wrapped) of the step's first column
    {
      float vs[kStep], vl[kStep];
      strip_filter<RMAX, RS>(x, a.ws, a.rs, vs);
      strip_filter<RMAX, RL>(x, a.wl, a.rl, vl);
#pragma unroll
      for (int o = 0; o < kStep; ++o) {
        hs[o * kColumn + slot] = vs[o];
        hl[o * kColumn + slot] = vl[o];
      }
    }
    // the next step's columns: in flight during the y pass and the test
#pragma unroll
    for (int i = 0; i < 2 * RMAX; ++i) x[i] = x[i + kStep];
    if (s + 1 < steps) {
#pragma unroll
      for (int i = 0; i < kStep; ++i) x[2 * RMAX + i] = pixel(col0 + base + kStep + RMAX + i);
    }
    __syncthreads();
    {
      float v[kStrip + 2 * RMAX], vs[kStrip], vl[kStrip];
      auto load = [&](const float* h) {
        const float* p = h + yc * kColumn;
#pragma unroll
        for (int i = 0; i < (kStrip + 2 * RMAX) / 4; ++i) {   // group 2 ys + i of the column
          const float4 q = *reinterpret_cast<const float4*>(p + (i & 1 ? odd_slot(ys + i / 2) : even_slot(ys + i / 2)));
          v[4 * i] = q.x;
          v[4 * i + 1] = q.y;
          v[4 * i + 2] = q.z;
          v[4 * i + 3] = q.w;
        }
      };
      load(hs);
      strip_filter<RMAX, RS>(v, a.ws, a.rs, vs);
      load(hl);
      strip_filter<RMAX, RL>(v, a.wl, a.rl, vl);
      float* d = ring + ((base + yc) & (kRing - 1)) * kColumn;
      *reinterpret_cast<float4*>(d + even_slot(ys)) =
          make_float4(vs[0] - vl[0], vs[1] - vl[1], vs[2] - vl[2], vs[3] - vl[3]);
      *reinterpret_cast<float4*>(d + odd_slot(ys)) =
          make_float4(vs[4] - vl[4], vs[5] - vl[5], vs[6] - vl[6], vs[7] - vl[7]);
    }
    __syncthreads();
    // Ring columns base - 1 .. base + kStep - 2 have both neighbours.
    float here[kStep + 2];   // column base - 2 + j (before the first step's: wrapped, not used)
    bool any = false;
#pragma unroll
    for (int j = 0; j < kStep + 2; ++j) here[j] = ring[((base - 2 + j) & (kRing - 1)) * kColumn + own];
#pragma unroll
    for (int j = 0; j < kStep; ++j) any = any || here[j + 1] > a.minval;
    uint64_t word = 0;       // lane j: the word of the step's column j
    if (__ballot(mine && any)) {
      float above[kStep + 2], below[kStep + 2];
#pragma unroll
      for (int j = 0; j < kStep + 2; ++j) {
        const float* col = ring + ((base - 2 + j) & (kRing - 1)) * kColumn;
        above[j] = col[up];
        below[j] = col[down];
      }
#pragma unroll
      for (int j = 0; j < kStep + 2; ++j) {   // out of the frame: -inf, which beats nothing
        const int gc = col0 + base - 2 + j;
        const bool in = gc >= 0 && gc < a.nx;
        above[j] = in && has_up ? above[j] : ninf;
        below[j] = in && has_down ? below[j] : ninf;
        here[j] = in ? here[j] : ninf;
      }
#pragma unroll
      for (int j = 0; j < kStep; ++j) {
        const int gc = col0 + base - 1 + j;
        const float p = here[j + 1];
        // the left column and the row above come first in column-major order
        const float before = fmaxf(fmaxf(fmaxf(above[j], here[j]), below[j]), above[j + 1]);
        const float after = fmaxf(fmaxf(fmaxf(above[j + 2], here[j + 2]), below[j + 2]), below[j + 1]);
        const bool cand = mine && gc >= first && gc < last && p > a.minval && !(before >= p) && !(after > p);
        const uint64_t m = __ballot(cand);
        word = lane == j ? m | kStored : word;
        if (mine && gc >= first && gc < last) a.dog[(size_t)f * plane + (size_t)gc * a.ny + gr] = p;
      }
    }
    const int gc = col0 + base - 1 + lane;
    if (lane < kStep && wi < a.wpc && gc >= first && gc < last) a.cand[((size_t)f * a.nx + gc) * a.wpc + wi] = word;
  }
}

// Block-wide exclusive scan of one int64 per thread (inclusive scans within
// each wave by shuffles, then the wave totals through LDS); returns the prefix
// and leaves the block total in *total.  sh holds at least blockDim.x / 64.
__device__ int64_t block_exclusive_scan(int64_t v, int64_t* sh, int64_t* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int64_t incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int64_t up = __shfl_up(incl, off);
    if (lane >= off) incl += up;
  }
  if (lane == 63) sh[wave] = incl;
  __syncthreads();
  int64_t before = 0, all = 0;
  for (int q = 0; q < nw; ++q) {
    const int64_t t = sh[q];
    before += q < wave ? t : 0;
    all += t;
  }
  *total = all;
  __syncthreads();
  return before + incl - v;
}

// One word per lane; the wave tests its lanes' candidates one at a time, all 64
// lanes reading the candidate's window together, four elements each at a time
// so that their reads overlap.
__global__ __launch_bounds__(kBlock) void boxer_suppress(BoxerArgs a) {
  __shared__ int64_t sh[kWaves];
  const int lane = threadIdx.x & 63;
  const int win = a.win, side = 2 * win + 1, area = side * side;
  const int inv = (65536 + side - 1) / side;   // e / side = e inv >> 16 for e < 1024, side <= 31
  const size_t plane = (size_t)a.ny * a.nx;
  int kept = 0;
  for (int i = 0; i < a.wpt; ++i) {
    const int64_t w = ((int64_t)blockIdx.x * a.wpt + i) * kBlock + threadIdx.x;
    uint64_t todo = w < a.n_words ? a.cand[w] & ~kStored : 0, keep = todo;
    for (;;) {
      const uint64_t busy = __ballot(todo != 0);
      if (!busy) break;
      const int lead = __builtin_ctzll(busy);
      // the candidate: lowest pending bit of lane `lead`
      const uint64_t ms = __shfl(todo, lead);
      const int64_t ws = __shfl(w, lead);
      const int b = __builtin_ctzll(ms);
      const int64_t fc = ws / a.wpc;
      const int gc = (int)(fc % a.nx), wi = (int)(ws - fc * a.wpc);
      const int gr = wi * a.word_rows + b;
      const float* D = a.dog + (size_t)(fc / a.nx) * plane;
      const float v = D[(size_t)gc * a.ny + gr];
      // which words of the window's columns are stored: lane l < 32 the upper
      // word of column gc - win + l, lane 32 + l the lower one (a window is
      // shorter than a word)
      const int w_lo = max(gr - win, 0) / a.word_rows, w_hi = min(gr + win, a.ny - 1) / a.word_rows;
      const int bound = w_hi * a.word_rows;   // first row of the lower word
      const int sc = (lane & 31) - win;
      const bool col = (lane & 31) < side && gc + sc >= 0 && gc + sc < a.nx;
      const uint64_t stored = __ballot(col && (a.cand[(fc + (col ? sc : 0)) * a.wpc + (lane < 32 ? w_lo : w_hi)] >> 63));
      bool beaten = false;
      for (int e0 = 0; e0 < area; e0 += 256) {
        float q[4];
        bool in[4], before[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int e = e0 + 64 * j + lane, ec = e * inv >> 16, er = e - ec * side;   // column, row of the window
          const int qc = gc - win + ec, qr = gr - win + er;
          in[j] = e < area && qr >= 0 && qr < a.ny && ((stored >> (ec + (qr >= bound ? 32 : 0))) & 1);
          before[j] = ec < win || (ec == win && er < win);
          q[j] = in[j] ? D[(size_t)qc * a.ny + qr] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) beaten |= in[j] && (q[j] > v || (q[j] == v && before[j]));
        if (__ballot(beaten)) break;
      }
      const bool lost = __ballot(beaten) != 0;
      if (lane == lead) {
        todo &= todo - 1;
        if (lost) keep &= ~(1ull << b);
      }
    }
    if (w < a.n_words) a.keep[w] = keep;
    kept += __popcll(keep);
  }
  int64_t total;
  block_exclusive_scan(kept, sh, &total);
  if (threadIdx.x == 0) a.block_base[blockIdx.x] = total;
}

// Exclusive scan of the per-block counts in place (one block); the total
// number of detections goes to *count.
__global__ __launch_bounds__(kScanThreads) void boxer_scan(int64_t* base, int64_t nb, int64_t* count) {
  __shared__ int64_t sh[kScanThreads / 64];
  const int t = threadIdx.x;
  const int64_t per = (nb + kScanThreads - 1) / kScanThreads;
  const int64_t lo = min(nb, (int64_t)t * per), hi = min(nb, lo + per);
  int64_t s = 0;
  for (int64_t i = lo; i < hi; ++i) s += base[i];
  int64_t total;
  int64_t run = block_exclusive_scan(s, sh, &total);
  for (int64_t i = lo; i < hi; ++i) {
    const int64_t v = base[i];
    base[i] = run;
    run += v;
  }
  if (t == 0) *count = total;
}

// The words of one suppress block, wpt consecutive ones per thread, in order;
// then the block's boxes, one wave each.
__global__ __launch_bounds__(kBlock) void boxer_place(BoxerArgs a) {
  __shared__ int64_t sh[kWaves];
  const int64_t w0 = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * a.wpt;
  uint64_t keep[kWordsPerThread];
  int n = 0;
#pragma unroll
  for (int i = 0; i < kWordsPerThread; ++i) {
    keep[i] = i < a.wpt && w0 + i < a.n_words ? a.keep[w0 + i] : 0;
    n += __popcll(keep[i]);
  }
  int64_t total;
  const int64_t begin = a.block_base[blockIdx.x];
  int64_t k = begin + block_exclusive_scan(n, sh, &total);
  const int B = a.box, BB = a.box * a.box, half = (a.box - 1) / 2;
  const size_t plane = (size_t)a.ny * a.nx;
  if (n) {
#pragma unroll
    for (int i = 0; i < kWordsPerThread; ++i) {
      const int64_t fc = (w0 + i) / a.wpc;
      const int wr = (int)((w0 + i) - fc * a.wpc);
      const int gc = (int)(fc % a.nx), f = (int)(fc / a.nx);
      const int c0 = min(max(gc - half, 0), a.nx - B);
      while (keep[i] && k < a.max_boxes) {
        const int gr = wr * a.word_rows + __builtin_ctzll(keep[i]);
        keep[i] &= keep[i] - 1;
        a.xc[k] = c0 + 1;
        a.yc[k] = min(max(gr - half, 0), a.ny - B) + 1;
        a.frame[k] = f + 1;
        if (a.strength) a.strength[k] = a.dog[(size_t)f * plane + (size_t)gc * a.ny + gr];
        ++k;
      }
    }
  }
  __syncthreads();   // the corners below are this block's own
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t end = min(begin + total, a.max_boxes);
  for (int64_t q = begin + wave; q < end; q += kWaves) {
    const float* src = a.frames + (size_t)(a.frame[q] - 1) * plane + (size_t)(a.xc[q] - 1) * a.ny + (a.yc[q] - 1);
    float* dst = a.rois + (size_t)q * BB;
    for (int e = lane; e < BB; e += 64) {
      const int col = e / B, row = e - col * B;
      dst[e] = src[(size_t)col * a.ny + row];
    }
  }
}

int radius_of(double sigma) { return (int)floor(3.0 * sigma + 0.5); }

// Half of a normalised Gaussian kernel, w[0..R], in the documented order.
void gaussian_half(double sigma, int R, float* w) {
  double g[kMaxRadius + 1];
  double sum = 0.0;
  for (int k = 0; k <= R; ++k) {
    g[k] = exp(-(double)k * (double)k / (2.0 * sigma * sigma));
    sum += k == 0 ? g[k] : 2.0 * g[k];
  }
  for (int k = 0; k <= R; ++k) w[k] = (float)(g[k] / sum);
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Workspace: D | candidate words | survivor words | block counts.
struct Layout {
  size_t dog, cand, keep, base, total;
};

Layout layout(int ny, int nx, int nf) {
  // room for the words of either word_rows_of
  const int64_t n_words = (int64_t)nf * nx * ((ny + word_rows_of(kMaxRadius) - 1) / word_rows_of(kMaxRadius));
  Layout L;
  L.dog = 0;
  L.cand = L.dog + align256((size_t)ny * nx * nf * sizeof(float));
  L.keep = L.cand + align256((size_t)n_words * sizeof(uint64_t));
  L.base = L.keep + align256((size_t)n_words * sizeof(uint64_t));
  L.total = L.base + align256((size_t)((n_words + kBlock - 1) / kBlock) * sizeof(int64_t));
  return L;
}

int check_params(int ny, int nx, int nf, int box, float overlap, float sigma_small, float sigma_large, float minval) {
  if (nf <= 0 || ny <= 0 || nx <= 0) return fail(GMLE_ERR_ARG, "frame stack %d x %d x %d is empty", ny, nx, nf);
  if (nf > 65535) return fail(GMLE_ERR_ARG, "at most 65535 frames per call, got %d", nf);
  if (box < kMinBox || box > kMaxBatchBox) return fail(GMLE_ERR_ARG, "boxsize %d out of range [%d, %d]", box, kMinBox, kMaxBatchBox);
  if (ny < box || nx < box) return fail(GMLE_ERR_ARG, "frames of %d x %d are smaller than the box %d", ny, nx, box);
  if (!(overlap >= 0.0f) || !(overlap < (float)box)) return fail(GMLE_ERR_ARG, "overlap must be in [0, boxsize)");
  if (!(sigma_small > 0.0f) || !(sigma_large > 0.0f)) return fail(GMLE_ERR_ARG, "sigmas must be > 0");
  if (radius_of(sigma_small) > kMaxRadius || radius_of(sigma_large) > kMaxRadius)
    return fail(GMLE_ERR_ARG, "sigmas above 4 px are not supported (kernel radius > %d)", kMaxRadius);
  if (isnan(minval)) return fail(GMLE_ERR_ARG, "minval is NaN");
  return GMLE_OK;
}

// Columns a block sweeps: long sweeps filter little halo (2 columns), short
// ones give a small stack enough blocks.
int sweep_columns(const BoxerArgs& a) {
  const int64_t rows = (int64_t)a.nf * ((a.wpc + 3) / 4);
  const int64_t parts = std::max<int64_t>(1, kTargetBlocks / rows);   // at most three full rounds
  const int64_t cols = (a.nx + parts - 1) / parts;
  return (int)std::min<int64_t>((std::max<int64_t>(cols, kMinSweep) + kStep - 1) / kStep * kStep, 1 << 20);
}

BoxerArgs make_args(const float* frames, int ny, int nx, int nf, int box, float overlap, float sigma_small,
                    float sigma_large, float minval, int64_t max_boxes, void* ws) {
  BoxerArgs a{};
  a.frames = frames;
  a.ny = ny;
  a.nx = nx;
  a.nf = nf;
  a.rs = radius_of(sigma_small);
  a.rl = radius_of(sigma_large);
  a.halo = std::max(a.rs, a.rl);
  gaussian_half(sigma_small, a.rs, a.ws);
  gaussian_half(sigma_large, a.rl, a.wl);
  a.minval = minval;
  a.win = std::max(1, (int)ceilf((float)box - overlap) - 1);
  a.box = box;
  a.word_rows = word_rows_of(a.halo);
  a.wpc = (ny + a.word_rows - 1) / a.word_rows;
  a.n_words = (int64_t)nf * nx * a.wpc;
  a.sweep = sweep_columns(a);
  a.wpt = a.n_words >= kManyWords ? kWordsPerThread : 1;
  const Layout L = layout(ny, nx, nf);
  a.max_boxes = max_boxes;
  char* w = (char*)ws;
  a.dog = (float*)(w + L.dog);
  a.cand = (uint64_t*)(w + L.cand);
  a.keep = (uint64_t*)(w + L.keep);
  a.block_base = (int64_t*)(w + L.base);
  return a;
}


template <int RMAX, int RS, int RL> void launch_detect(const BoxerArgs& a, hipStream_t stream) {
  const dim3 grid((a.nx + a.sweep - 1) / a.sweep, (a.wpc + 3) / 4, a.nf);
  hipLaunchKernelGGL((boxer_detect<RMAX, RS, RL>), grid, dim3(kBlock), 0, stream, a);
}

int enqueue_boxer(const BoxerArgs& a, hipStream_t stream) {
  // radii 3 and 6 are those of the default sigmas, 1 and 2 px; fixed, the taps
  // need no branches
  if (a.rs == 3 && a.rl == 6)
    launch_detect<6, 3, 6>(a, stream);
  else if (a.halo <= 6)
    launch_detect<6, 0, 0>(a, stream);
  else
    launch_detect<kMaxRadius, 0, 0>(a, stream);
  const int64_t n_blocks = (a.n_words + (int64_t)kBlock * a.wpt - 1) / ((int64_t)kBlock * a.wpt);
  hipLaunchKernelGGL(boxer_suppress, dim3((unsigned)n_blocks), dim3(kBlock), 0, stream, a);
  hipLaunchKernelGGL(boxer_scan, dim3(1), dim3(kScanThreads), 0, stream, a.block_base, n_blocks, a.count);
  if (a.max_boxes > 0) hipLaunchKernelGGL(boxer_place, dim3((unsigned)n_blocks), dim3(kBlock), 0, stream, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GMLE_OK : hip_fail(e, "kernel launch");
}

}  // namespace
}  // namespace gmle

using namespace gmle;

extern "C" {

int64_t gmle_boxer_workspace_bytes(int ny, int nx, int n_frames) {
  if (ny <= 0 || nx <= 0 || n_frames <= 0) return 0;
  return (int64_t)layout(ny, nx, n_frames).total;
}

int gmle_find_boxes_device(const float* d_frames, int ny, int nx, int n_frames, int boxsize, float overlap,
                           float sigma_small, float sigma_large, float minval, int64_t max_boxes, float* d_rois,
                           int32_t* d_x_corners, int32_t* d_y_corners, int32_t* d_frame_indices,
                           float* d_strength, int64_t* d_count, void* d_workspace, void* stream) {
  int rc = check_params(ny, nx, n_frames, boxsize, overlap, sigma_small, sigma_large, minval);
  if (rc != GMLE_OK) return rc;
  if (max_boxes < 0) return fail(GMLE_ERR_ARG, "max_boxes must be >= 0");
  if (!d_frames || !d_count || !d_workspace) return fail(GMLE_ERR_ARG, "frames, count and workspace must not be NULL");
  if (max_boxes > 0 && (!d_rois || !d_x_corners || !d_y_corners || !d_frame_indices))
    return fail(GMLE_ERR_ARG, "output arrays must not be NULL when max_boxes > 0");
  BoxerArgs a = make_args(d_frames, ny, nx, n_frames, boxsize, overlap, sigma_small, sigma_large, minval, max_boxes,
                          d_workspace);
  a.count = d_count;
  a.rois = d_rois;
  a.xc = d_x_corners;
  a.yc = d_y_corners;
  a.frame = d_frame_indices;
  a.strength = d_strength;
  return enqueue_boxer(a, (hipStream_t)stream);
}

int gmle_find_boxes(const float* frames, int ny, int nx, int n_frames, int boxsize, float overlap,
                    float sigma_small, float sigma_large, float minval, int64_t max_boxes, float* rois,
                    int32_t* x_corners, int32_t* y_corners, int32_t* frame_indices, float* strength,
                    int64_t* n_found) {
  int rc = check_params(ny, nx, n_frames, boxsize, overlap, sigma_small, sigma_large, minval);
  if (rc != GMLE_OK) return rc;
  if (max_boxes < 0) return fail(GMLE_ERR_ARG, "max_boxes must be >= 0");
  if (!frames || !n_found) return fail(GMLE_ERR_ARG, "frames and n_found must not be NULL");
  if (max_boxes > 0 && (!rois || !x_corners || !y_corners || !frame_indices))
    return fail(GMLE_ERR_ARG, "output arrays must not be NULL when max_boxes > 0");
  const size_t npix = (size_t)ny * nx * n_frames;
  const size_t BB = (size_t)boxsize * boxsize;
  const size_t ws = layout(ny, nx, n_frames).total;
  // one allocation: frames | workspace | count | outputs
  const size_t o_ws = align256(npix * sizeof(float));
  const size_t o_count = o_ws + align256(ws);
  const size_t o_rois = o_count + 256;
  const size_t o_xc = o_rois + align256((size_t)max_boxes * BB * sizeof(float));
  const size_t o_yc = o_xc + align256((size_t)max_boxes * sizeof(int32_t));
  const size_t o_fr = o_yc + align256((size_t)max_boxes * sizeof(int32_t));
  const size_t o_st = o_fr + align256((size_t)max_boxes * sizeof(int32_t));
  const size_t bytes = o_st + align256((size_t)max_boxes * sizeof(float));
  char* dev = nullptr;
  hipError_t e = hipMalloc((void**)&dev, bytes);
  if (e != hipSuccess) return hip_fail(e, "hipMalloc");
  hipStream_t s = nullptr;
  e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
  if (e != hipSuccess) {
    (void)hipFree(dev);
    return hip_fail(e, "hipStreamCreate");
  }
  auto done = [&](int code) {
    (void)hipStreamSynchronize(s);
    (void)hipStreamDestroy(s);
    (void)hipFree(dev);
    return code;
  };
  int64_t* d_count = (int64_t*)(dev + o_count);
  if ((e = hipMemcpyAsync(dev, frames, npix * sizeof(float), hipMemcpyHostToDevice, s)) != hipSuccess)
    return done(hip_fail(e, "hipMemcpy frames"));
  BoxerArgs a = make_args((const float*)dev, ny, nx, n_frames, boxsize, overlap, sigma_small, sigma_large, minval,
                          max_boxes, dev + o_ws);
  a.count = d_count;
  a.rois = (float*)(dev + o_rois);
  a.xc = (int32_t*)(dev + o_xc);
  a.yc = (int32_t*)(dev + o_yc);
  a.frame = (int32_t*)(dev + o_fr);
  a.strength = strength ? (float*)(dev + o_st) : nullptr;
  if ((rc = enqueue_boxer(a, s)) != GMLE_OK) return done(rc);
  int64_t n = 0;
  if ((e = hipMemcpyAsync(&n, d_count, sizeof(n), hipMemcpyDeviceToHost, s)) != hipSuccess ||
      (e = hipStreamSynchronize(s)) != hipSuccess)
    return done(hip_fail(e, "hipMemcpy count"));
  *n_found = n;
  const size_t m = (size_t)std::min(n, max_boxes);
  if (m > 0) {
    if ((e = hipMemcpyAsync(rois, dev + o_rois, m * BB * sizeof(float), hipMemcpyDeviceToHost, s)) != hipSuccess ||
        (e = hipMemcpyAsync(x_corners, dev + o_xc, m * sizeof(int32_t), hipMemcpyDeviceToHost, s)) != hipSuccess ||
        (e = hipMemcpyAsync(y_corners, dev + o_yc, m * sizeof(int32_t), hipMemcpyDeviceToHost, s)) != hipSuccess ||
        (e = hipMemcpyAsync(frame_indices, dev + o_fr, m * sizeof(int32_t), hipMemcpyDeviceToHost, s)) !=
            hipSuccess ||
        (strength &&
         (e = hipMemcpyAsync(strength, dev + o_st, m * sizeof(float), hipMemcpyDeviceToHost, s)) != hipSuccess))
      return done(hip_fail(e, "hipMemcpy results"));
  }
  if ((e = hipStreamSynchronize(s)) != hipSuccess) return done(hip_fail(e, "hipStreamSynchronize"));
  return done(GMLE_OK);
}

// Weights the filter uses for one sigma (w[0..R], R = floor(3 sigma + 0.5));
// returns R, or -1 when R is above the supported radius.
int gmle_boxer_weights(float sigma, float* w, int capacity) {
  if (!(sigma > 0.0f)) return -1;
  const int R = radius_of(sigma);
  if (R > kMaxRadius || !w || capacity < R + 1) return -1;
  gaussian_half(sigma, R, w);
  return R;
}

}  // extern "C"
