// pmc_stats.h -- in-situ size distributions of a box.
//
// bin_grid_histogram_1d (src/bin_grid.F90:225-248) over particle diameters
// with number-concentration weights, as extract_aero_size builds its number
// and mass distributions (src/extract_aero_size.F90:132-138): particle i
// adds w_i / width to the log-spaced diameter bin it falls in, where w_i is
// its number concentration (aero_state_num_concs, src/aero_state.F90:
// 1243-1261), times its mass or volume for the mass and volume
// distributions.
//
// Two passes, with no sort and no atomics, so a histogram does not depend on
// the order in which work lands:
//   k_dist_partial: DIST_BLOCKS workgroups each take a fixed slice of the
//     box's particles (slice b is [b n / NB, (b+1) n / NB)).  Each wavefront
//     keeps its own LDS histogram.  Lanes that hold the same bin find each
//     other with one ballot per bit of the bin; the first of them adds the
//     others' values in lane order and updates the bin, one writer per bin.
//     The workgroup adds its wavefronts' histograms in order and writes the
//     whole window (zeros included) to partials[b][.].
//   k_dist_reduce: adds partials[0..NB)[bin], RED_ROWS rows a thread and
//     the rows' sums in order.
// Bins are handled in windows of at most DIST_WIN, one pair of passes per
// window.  Both passes read the particle count from the box descriptor on
// the device, so the host never waits on the device to enqueue them.
#pragma once

#include "pmc_exact.h"

namespace pmc {

constexpr int DIST_NUM = 0, DIST_MASS = 1, DIST_VOL = 2;
constexpr int DIST_ITEMS = 3;     // particles a lane in flight together
constexpr int DIST_BLOCKS = 512;  // workgroups of the partial pass: fixed, so sums do not depend on the device
constexpr int DIST_WIN = 2048;    // bins per window: the LDS histogram and a row of partials

// bin (1-based, 0 / n_bin + 1 outside the grid) and weight / width of
// particle slot p, w_box the box's weights
__device__ inline int dist_item(const Weights &w_box, const Arrays &A, int64_t p,
                                int quantity, int n_bin, double log_lo, double log_hi,
                                double *val) {
  const int ns = A.n_spec;
  const int klass = A.klass[p];
  double v = 0.0, m = 0.0;
  for (int s0 = 0; s0 < ns; s0 += SPEC_CHUNK) {
    double x[SPEC_CHUNK];
#pragma unroll
    for (int u = 0; u < SPEC_CHUNK; ++u)
      x[u] = A.vol[(int64_t)(s0 + u < ns ? s0 + u : ns - 1) * A.total_cap + p];
#pragma unroll
    for (int u = 0; u < SPEC_CHUNK; ++u)
      if (s0 + u < ns) {
        v += x[u];
        m += x[u] * A.density[s0 + u];
      }
  }
  const double r = vol2rad(v);
  const int b = linspace_find(log_lo, log_hi, n_bin + 1, log(2.0 * r));
  double w = nc_at_radius(w_box, klass, r);
  if (quantity == DIST_MASS) w *= m;
  else if (quantity == DIST_VOL) w *= v;
  const double width = (log_hi - log_lo) / (double)n_bin;
  *val = w / width;
  return b;
}

// Wavefronts of a partial-pass workgroup: as many as fit their histograms of
// `win` bins in 64 KB of LDS, up to eight.  Two workgroups a compute unit
// then leave 16 wavefronts to hide the arithmetic's latency.
constexpr int DIST_WAVES = 8;
inline int dist_waves(int win) { return std::min(DIST_WAVES, 65536 / (win * 8)); }
static_assert(65536 / (DIST_WIN * 8) >= 1, "a window's histogram fits the LDS");

// The sum of `v` over the lanes of the wavefront that hold the same key, in
// lane order, on the first of them (which this returns true for); key < 0:
// this lane holds nothing.  Every lane takes part.
__device__ inline bool wave_key_sum(int key, int key_bits, double v, double *sum) {
  const int lane = threadIdx.x & 63;
  uint64_t peers = __ballot(key >= 0);
  if (!peers) return false;
  for (int b = 0; b < key_bits; ++b) {
    const uint64_t m = __ballot((key >> b) & 1);
    peers &= ((key >> b) & 1) ? m : ~m;
  }
  const bool first = key >= 0 && __ffsll((long long)peers) - 1 == lane;
  // the leaders walk their peers together, one peer each a pass
  uint64_t rest = first ? peers : 0ull;
  double s = 0.0;
  while (__ballot(rest != 0)) {
    const double x = __shfl(v, rest ? __ffsll((long long)rest) - 1 : lane);
    if (rest) {
      s += x;
      rest &= rest - 1;
    }
  }
  *sum = s;
  return first;
}

// partials[blockIdx.x][0 .. win): this workgroup's sums over bins
// [win_lo, win_lo + win) (0-based) of its slice of the box's particles.
// Bound by FP64 arithmetic (a pow, a log and the weight per particle): a
// lane takes DIST_ITEMS particles at a time, whose chains are independent.
// 1.5e6 particles of 4 species in 160 bins take 50 us, 20000 in 60 bins
// 7.7 us (68 and 21 us with a block sort and a segmented scan per tile of
// 1024; 63 us with 4 wavefronts a workgroup in place of 8).
__global__ void __launch_bounds__(DIST_WAVES * 64)
k_dist_partial(const BoxDesc *boxes, Arrays A, int box, int quantity, int n_bin, double log_lo,
               double log_hi, int win_lo, int win, int key_bits, double *partials) {
  extern __shared__ double s_hist[];  // [wavefronts][win]
  __shared__ Weights s_w;
  const BoxDesc *B = &boxes[box];
  const int64_t n = B->n_part, off = B->off;
  const int64_t lo = (int64_t)blockIdx.x * n / gridDim.x;
  const int64_t hi = (int64_t)(blockIdx.x + 1) * n / gridDim.x;
  const int t = threadIdx.x, threads = blockDim.x, waves = threads >> 6;
  for (int j = t; j < waves * win; j += threads) s_hist[j] = 0.0;
  for (int j = t; j < (int)(sizeof(Weights) / sizeof(int)); j += threads)
    ((int *)&s_w)[j] = ((const int *)&B->w)[j];
  __syncthreads();
  double *hist = s_hist + (t >> 6) * win;
  for (int64_t base = lo; base < hi; base += threads * DIST_ITEMS) {
    int key[DIST_ITEMS];
    double val[DIST_ITEMS];
#pragma unroll
    for (int k = 0; k < DIST_ITEMS; ++k) {
      const int64_t i = base + (int64_t)k * threads + t;
      key[k] = -1;  // past the slice or outside the window
      val[k] = 0.0;
      if (i < hi) {
        double x;
        const int b = dist_item(s_w, A, off + i, quantity, n_bin, log_lo, log_hi, &x) - 1 - win_lo;
        if (b >= 0 && b < win && b + win_lo < n_bin) {
          key[k] = b;
          val[k] = x;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < DIST_ITEMS; ++k) {
      double sum;
      if (wave_key_sum(key[k], key_bits, val[k], &sum)) hist[key[k]] += sum;
    }
  }
  __syncthreads();
  double *out = partials + (int64_t)blockIdx.x * win;
  for (int j = t; j < win; j += threads) {
    double s = s_hist[j];
    for (int w = 1; w < waves; ++w) s += s_hist[w * win + j];
    out[j] = s;
  }
}

// hist[win_lo + j] = sum over workgroups of partials[.][j]: RED_BINS bins
// (a 128-byte line of a row) a workgroup, each thread RED_ROWS consecutive
// rows with its loads in flight together, then the threads' sums in row
// order: 3.6 us for 60 bins and 5.9 for 160.  (One thread a bin waits for
// its 512 loads in turn, 124 us for any bin count.)
constexpr int RED_BINS = 16, RED_ROWS = 8;
constexpr int RED_THREADS = RED_BINS * (DIST_BLOCKS / RED_ROWS);
static_assert(RED_THREADS <= 1024 && DIST_BLOCKS % RED_ROWS == 0, "one workgroup covers the rows");

__global__ void __launch_bounds__(RED_THREADS)
k_dist_reduce(const double *partials, int win_lo, int win, int n_bin, double *hist) {
  __shared__ double s_sum[RED_THREADS];
  const int t = threadIdx.x, row0 = (t / RED_BINS) * RED_ROWS;
  const int j = blockIdx.x * RED_BINS + t % RED_BINS;
  double s = 0.0;
  if (j < win) {
    double x[RED_ROWS];
#pragma unroll
    for (int r = 0; r < RED_ROWS; ++r) x[r] = partials[(int64_t)(row0 + r) * win + j];
#pragma unroll
    for (int r = 0; r < RED_ROWS; ++r) s += x[r];
  }
  s_sum[t] = s;
  __syncthreads();
  if (t < RED_BINS && j < win && win_lo + j < n_bin) {
    for (int r = 1; r < RED_THREADS / RED_BINS; ++r) s += s_sum[r * RED_BINS + t];
    hist[win_lo + j] = s;
  }
}

}  // namespace pmc
