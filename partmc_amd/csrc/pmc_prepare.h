// pmc_prepare.h -- the sorted structure of the exact mode: bin grids and
// the (bin, class) lists with their forward maps.
//
// aero_sorted_remake_if_needed (src/aero_sorted.F90:214-373), explicit-grid
// sorts (:254-262, with aero_sorted_discard_outside_grid :153-180) and
// aero_sorted_sort_particles (:185-209).  The passes of one preparation, in
// order, each over every box (or one) at once:
//   k_prep_radii    radius extremes of boxes without current lists
//   k_prep_plan     the grid and whether the box sorts, one wavefront a box
//   k_prep_keys     bins, classes and per-segment list counts
//   k_prep_lists    list lengths, starts and capacities, one workgroup a box
//   k_prep_scatter  list entries and forward indices
// Lists are rebuilt into the other pool half every time, so every list
// starts the sweep with slack.
//
// A box's particles are cut into at most SORT_THREADS segments of a multiple
// of 64, each walked by one wavefront from its first particle up, so a
// stable rank is a running count per list plus the lanes below with the same
// list (found with one ballot per bit of the list number).  These passes
// read and write a few words a particle and are bound by the arithmetic of
// the bins and by launches: a set_bin_grid of 1e5 particles takes 50 us of
// device time, 102 us when some lie outside the grid, and 0.44 ms at 1.5e6.
// (One workgroup a box, with a single thread discarding particles outside
// the grid and laying out the lists, took 2.1, 18.9 and 278 ms.)
#pragma once

#include "pmc_scan.h"
#include "pmc_state.h"

namespace pmc {

// An explicit grid for one box to be sorted on.  It is an argument of the
// passes and never part of the box: a preparation that ends early (the box
// holds an error, a class is out of range) leaves no grid behind for a later
// step, which has no pass that discards.
struct GridRequest {
  int n_bin = -1;  // -1: none
  double r_min = 0.0, r_max = 0.0;
};

constexpr int PREP_WAVES = 4;      // wavefronts a workgroup of the segment passes
constexpr int PREP_RADII_WG = 32;  // workgroups a box of k_prep_radii
constexpr int PREP_LDS_KEYS = 3072;  // list counters of a wavefront kept in LDS up to here

// segment length and count for n particles
__host__ __device__ inline int prep_seg_len(int n) {
  const int per = (n + SORT_THREADS - 1) / SORT_THREADS;
  return (per + 63) / 64 * 64;
}
__device__ inline int prep_segs(int n) {
  const int s = prep_seg_len(n);
  return s > 0 ? (n + s - 1) / s : 0;
}

// whether the plan takes the occupied bins from the box's lists (lists left
// stale by the parallel mode count as unsorted)
__device__ inline bool prep_use_lists(const BoxDesc *B) { return B->valid_sort && B->xlists_valid; }

// bin_grid_make (log), src/bin_grid.F90:83-138 via logspace
// src/util.F90:497-520, by the lanes of a wavefront
__device__ inline void make_log_grid_wave(int n_bin, double rmin, double rmax, double *edges,
                                          double *centers, double *widths) {
  if (n_bin <= 0) return;
  const int lane = threadIdx.x & 63;
  const double lmin = log(rmin), lmax = log(rmax);
  const int n = n_bin + 1;
  for (int i = 2 + lane; i <= n - 1; i += 64) {
    const double a = (double)(i - 1) / (double)(n - 1);
    edges[i - 1] = exp((1.0 - a) * lmin + a * lmax);
  }
  const double c1 = exp(interp_linear_disc(lmin, lmax, 2 * n_bin + 1, 2));
  const double c2 = exp(interp_linear_disc(lmin, lmax, 2 * n_bin + 1, 2 * n_bin));
  const double lc1 = log(c1), lc2 = log(c2);
  for (int i = 2 + lane; i <= n_bin - 1; i += 64) {
    const double a = (double)(i - 1) / (double)(n_bin - 1);
    centers[i - 1] = exp((1.0 - a) * lc1 + a * lc2);
  }
  for (int i = lane; i < n_bin; i += 64) widths[i] = (lmax - lmin) / (double)n_bin;
  if (lane == 0) {
    edges[0] = rmin;
    edges[n - 1] = rmax;
    centers[0] = c1;
    centers[n_bin - 1] = c2;
  }
}

// smallest and largest value over the wavefront, on every lane
__device__ inline double wave_min(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o));
  return v;
}
__device__ inline double wave_max(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}

// scratch of the radius extremes: a (min, max) pair per wavefront
__device__ inline double *prep_radii_of(const Arrays &A, int box) {
  return (double *)(A.sort_scratch + (int64_t)box * SORT_THREADS * A.max_keys);
}

__global__ void __launch_bounds__(256)
k_prep_radii(const BoxDesc *boxes, Arrays A, int only_box) {
  const int box = only_box >= 0 ? only_box : (int)blockIdx.y;
  const BoxDesc *B = &boxes[box];
  if (B->error || prep_use_lists(B)) return;
  double lo = 1e300, hi = -1e300;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < B->n_part; i += gridDim.x * 256) {
    const double r = vol2rad(A.vtot[B->off + i]);
    lo = fmin(lo, r);
    hi = fmax(hi, r);
  }
  lo = wave_min(lo);
  hi = wave_max(hi);
  const int w = blockIdx.x * 4 + (threadIdx.x >> 6);
  if ((threadIdx.x & 63) == 0) {
    prep_radii_of(A, box)[2 * w] = lo;
    prep_radii_of(A, box)[2 * w + 1] = hi;
  }
}

__global__ void __launch_bounds__(64)
k_prep_plan(BoxDesc *boxes, Arrays A, int only_box, GridRequest req) {
  const int box = only_box >= 0 ? only_box : (int)blockIdx.x;
  const int lane = threadIdx.x;
  BoxDesc *B = &boxes[box];
  if (B->error) return;
  double *edges = A.edges + (int64_t)box * (A.max_bin + 1);
  double *centers = A.centers + (int64_t)box * A.max_bin;
  double *widths = A.widths + (int64_t)box * A.max_bin;
  const int n_class = B->w.n_class;
  int err = 0, sort = 0;
  // a new grid of nn bins, or none (-1)
  int nn = -1;
  double gmin = 0.0, gmax = 0.0;
  if (req.n_bin >= 0) {
    if (req.n_bin > A.max_bin) {
      err = ERR_CAPACITY;
    } else {
      nn = req.n_bin;
      gmin = req.r_min;
      gmax = req.r_max;
    }
  } else {
    const bool use_lists = prep_use_lists(B);
    const int nb = B->n_bin, n = B->n_part;
    double rmin = 0.0, rmax = 0.0;
    if (!use_lists && n > 0) {
      double lo = 1e300, hi = -1e300;
      for (int w = lane; w < PREP_RADII_WG * 4; w += 64) {
        lo = fmin(lo, prep_radii_of(A, box)[2 * w]);
        hi = fmax(hi, prep_radii_of(A, box)[2 * w + 1]);
      }
      rmin = wave_min(lo);
      rmax = wave_max(hi);
    }
    if (!use_lists && B->valid_sort && nb > 0) {
      // a valid sort without current lists: the occupied bins are those of
      // the radius extremes
      if (n == 0) {
        rmin = edges[nb];
        rmax = edges[0];
      } else {
        const int b_lo = bin_find_log(nb, B->log_lo, B->log_hi, rmin);
        const int b_hi = bin_find_log(nb, B->log_lo, B->log_hi, rmax);
        rmin = edges[max(b_lo, 1) - 1];
        rmax = edges[min(b_hi, nb)];
      }
    }
    if (use_lists) {
      const int *llen = A.llen + (int64_t)box * A.max_keys;
      int first = nb + 1, last = 0;
      for (int b = 1 + lane; b <= nb; b += 64) {
        int tot = 0;
        for (int c = 1; c <= n_class; ++c) tot += llen[(b - 1) + nb * (c - 1)];
        if (tot > 0) {
          first = min(first, b);
          last = max(last, b);
        }
      }
      for (int o = 32; o > 0; o >>= 1) {
        first = min(first, __shfl_xor(first, o));
        last = max(last, __shfl_xor(last, o));
      }
      if (last == 0) {
        if (nb > 0) {
          rmin = edges[nb];
          rmax = edges[0];
        }
      } else {
        rmin = edges[first - 1];
        rmax = edges[last];
      }
    }
    if (lane == 0) B->regridded = 0;
    if (rmax == 0.0) {
      if (!use_lists && lane == 0) {
        B->n_bin = 0;
        B->bounds_valid = 0;
        B->tables_valid = 0;
      }
    } else if (nb < 1 || rmin / edges[0] < 3.0 || edges[nb] / rmax < 3.0) {
      gmin = rmin / 10.0;
      gmax = rmax * 10.0;
      const double nbf = ceil((log10(gmax) - log10(gmin)) * 10.0);
      if (nbf < 0.0) err = 538534122;
      else if (nbf > (double)A.max_bin) err = ERR_CAPACITY;
      else nn = (int)nbf;
    } else if (!use_lists) {
      sort = 1;
    }
  }
  if (nn >= 0) {
    sort = 1;
    make_log_grid_wave(nn, gmin, gmax, edges, centers, widths);
  }
  if (lane == 0) {
    if (nn >= 0) {
      B->n_bin = nn;
      // the end points as they were stored
      B->log_lo = log(gmin);
      B->log_hi = log(gmax);
      B->bounds_valid = 0;
      B->tables_valid = 0;
      B->regridded = 1;
      // the old grid's lists and keys end here, also when the passes after
      // this one do not get as far as new ones
      B->valid_sort = 0;
      B->xlists_valid = 0;
      B->pkeys_valid = 0;
    }
    if (err) B->error = err;
    B->prep_sort = sort;
    B->prep_outside = 0;
  }
}

// the lanes of the wavefront with the same key (key >= 0)
__device__ inline uint64_t wave_peers(int key, int key_bits) {
  uint64_t peers = __ballot(key >= 0);
  for (int b = 0; b < key_bits; ++b) {
    const uint64_t m = __ballot((key >> b) & 1);
    peers &= ((key >> b) & 1) ? m : ~m;
  }
  return peers;
}

// A wavefront's list counters: its own row in LDS, or the segment's row of
// the scratch where the lists are too many for that.
__device__ inline int *prep_counters(const Arrays &A, int box, int seg, int *lds, int keys) {
  int *row = A.sort_scratch + ((int64_t)box * SORT_THREADS + seg) * A.max_keys;
  return lds ? lds + (threadIdx.x >> 6) * keys : row;
}

// one lane's counter writes before the other lanes' atomics, and back
template <bool LDS>
__device__ inline void prep_counters_fence() {
  if (LDS) __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  else __threadfence();
}

// Bins and classes of the box's particles, and how many of each segment go
// to each list.  Particles outside an explicit grid are counted (the host
// discards them and repeats the pass); without one they are an error, so that
// no particle without a list reaches k_prep_scatter.
template <bool LDS>
__global__ void __launch_bounds__(64 * PREP_WAVES)
k_prep_keys(BoxDesc *boxes, Arrays A, int only_box, int lds_keys, int explicit_grid) {
  extern __shared__ int s_prep[];
  const int box = only_box >= 0 ? only_box : (int)blockIdx.y;
  BoxDesc *B = &boxes[box];
  if (B->error || !B->prep_sort) return;
  const int lane = threadIdx.x & 63;
  const int seg = blockIdx.x * PREP_WAVES + (threadIdx.x >> 6);
  const int n = B->n_part, S = prep_seg_len(n);
  if (seg >= prep_segs(n)) return;
  const int nb = B->n_bin, nc = B->w.n_class, K = nb * nc;
  const int64_t base = B->off;
  int *row = A.sort_scratch + ((int64_t)box * SORT_THREADS + seg) * A.max_keys;
  int *cnt = prep_counters(A, box, seg, LDS ? s_prep : nullptr, lds_keys);
  for (int k = lane; k < K; k += 64) cnt[k] = 0;
  prep_counters_fence<LDS>();
  int outside = 0;
  const int end = min(n, (seg + 1) * S);
  for (int i = seg * S + lane; i < end; i += 64) {
    const int b = bin_find_log(nb, B->log_lo, B->log_hi, vol2rad(A.vtot[base + i]));
    const int c = A.klass[base + i];
    A.fwd_bin[base + i] = b;
    A.fwd_class[base + i] = c;
    if (b < 1 || b > nb) {
      if (explicit_grid) outside++;
      else atomicExch(&B->error, 708651144);
    } else if (c < 1 || c > nc) {
      atomicExch(&B->error, 233133947);  // weight class out of range
    } else {
      atomicAdd(&cnt[(b - 1) + nb * (c - 1)], 1);
    }
  }
  if (outside) atomicAdd(&B->prep_outside, outside);
  if (LDS) {
    prep_counters_fence<LDS>();
    for (int k = lane; k < K; k += 64) row[k] = cnt[k];
  }
}

// List lengths (the segments' counts become their exclusive sums), then
// starts and capacities in the other pool half.
__global__ void __launch_bounds__(SORT_THREADS)
k_prep_lists(BoxDesc *boxes, Arrays A, int only_box) {
  __shared__ scan_storage<SORT_THREADS, int> s;
  const int box = only_box >= 0 ? only_box : (int)blockIdx.x;
  const int t = threadIdx.x;
  BoxDesc *B = &boxes[box];
  if (B->error) return;
  const int K = B->n_bin * B->w.n_class;
  int *lstart = A.lstart + (int64_t)box * A.max_keys;
  int *llen = A.llen + (int64_t)box * A.max_keys;
  int *lcap = A.lcap + (int64_t)box * A.max_keys;
  if (B->prep_sort) {
    const int segs = prep_segs(B->n_part);
    int *scr = A.sort_scratch + (int64_t)box * SORT_THREADS * A.max_keys;
    for (int k = t; k < K; k += SORT_THREADS) {
      int run = 0;
      for (int g0 = 0; g0 < segs; g0 += 16) {
        int c[16];  // a group's loads in flight together
#pragma unroll
        for (int u = 0; u < 16; ++u)
          c[u] = scr[(int64_t)(g0 + u < segs ? g0 + u : segs - 1) * A.max_keys + k];
#pragma unroll
        for (int u = 0; u < 16; ++u)
          if (g0 + u < segs) {
            scr[(int64_t)(g0 + u) * A.max_keys + k] = run;
            run += c[u];
          }
      }
      llen[k] = run;
    }
  }
  const int h = 1 - B->pool_cur;
  const int64_t pbase = B->pool_off + (int64_t)h * B->pool_half;
  int64_t pos = 0;
  for (int k0 = 0; k0 < K; k0 += SORT_THREADS) {
    const int k = k0 + t;
    const int len = k < K ? llen[k] : 0;
    const int cap = k < K ? len + len / 4 + 8 : 0;
    int tot;
    const int ex = block_sum_excl<SORT_THREADS>(cap, s, &tot);
    if (k < K) {
      lstart[k] = (int)(pbase + pos + ex);
      lcap[k] = cap;
    }
    pos += tot;
  }
  __syncthreads();  // every thread has read the pool fields
  if (t != 0) return;
  B->pool_top = (int)pos;
  B->pool_cur = h;
  if (pos > B->pool_half) {
    B->error = ERR_CAPACITY;
    return;
  }
  B->valid_sort = 1;
  B->xlists_valid = 1;
  B->pkeys_valid = 0;
}

// List entries and forward indices: a new sort's from the segments' ranks,
// kept lists moved to their new starts by their forward maps.
template <bool LDS>
__global__ void __launch_bounds__(64 * PREP_WAVES)
k_prep_scatter(BoxDesc *boxes, Arrays A, int only_box, int lds_keys) {
  extern __shared__ int s_prep[];
  const int box = only_box >= 0 ? only_box : (int)blockIdx.y;
  BoxDesc *B = &boxes[box];
  if (B->error) return;
  const int n = B->n_part, nb = B->n_bin;
  const int64_t base = B->off;
  const int *lstart = A.lstart + (int64_t)box * A.max_keys;
  if (!B->prep_sort) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
      const int key = (A.fwd_bin[base + i] - 1) + nb * (A.fwd_class[base + i] - 1);
      A.pool[lstart[key] + A.fwd_idx[base + i] - 1] = i + 1;
    }
    return;
  }
  const int lane = threadIdx.x & 63;
  const int seg = blockIdx.x * PREP_WAVES + (threadIdx.x >> 6);
  const int S = prep_seg_len(n);
  if (seg >= prep_segs(n)) return;
  const int K = nb * B->w.n_class;
  int *cnt = prep_counters(A, box, seg, LDS ? s_prep : nullptr, lds_keys);
  if (LDS) {
    const int *row = A.sort_scratch + ((int64_t)box * SORT_THREADS + seg) * A.max_keys;
    for (int k = lane; k < K; k += 64) cnt[k] = row[k];
    prep_counters_fence<LDS>();
  }
  int key_bits = 0;
  while ((1 << key_bits) < K) key_bits++;
  const int end = min(n, (seg + 1) * S);
  for (int i0 = seg * S; i0 < end; i0 += 64) {
    const int i = i0 + lane;
    int key = -1;
    if (i < end) key = (A.fwd_bin[base + i] - 1) + nb * (A.fwd_class[base + i] - 1);
    const uint64_t peers = wave_peers(key, key_bits);
    const int leader = key >= 0 ? __ffsll((long long)peers) - 1 : lane;
    int at = 0;
    if (key >= 0 && lane == leader) at = atomicAdd(&cnt[key], __popcll(peers));
    at = __shfl(at, leader);
    if (key >= 0) {
      const int p = at + __popcll(peers & ((1ull << lane) - 1ull));
      A.pool[lstart[key] + p] = i + 1;
      A.fwd_idx[base + i] = p + 1;
    }
  }
}

}  // namespace pmc
