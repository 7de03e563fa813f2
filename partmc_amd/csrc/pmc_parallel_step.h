// pmc_parallel_step.h -- the parallel-mode coagulation step.
//
// Per step and for every box at once:
//   1. keys: each particle caches its (bin, class) list key, its total
//      volume and (FP32 mode) its FP64-derived kernel terms; they change
//      only when the particle is created, the grid is remade, or the
//      environment or kernel type changes.  Live list counts are kept
//      exact by atomics, so aero_sorted_remake_if_needed's occupancy test
//      (src/aero_sorted.F90:264-292,341-351) needs no particle pass.
//   2. sort: a stable counting sort of the keys (tile histograms, one
//      device-wide scan, tile-local radix ranks) gives every (bin, class)
//      list in particle order.
//   3. pairs: one thread per bin pair draws n_samp ~ Poisson(k_max dt n1 n2)
//      (compute_n_samp, src/coagulation.F90:648-702) from the pair's own
//      stream; a device scan lays the tests of all pairs of all boxes out in
//      the reference's loop order (src/coagulation.F90:74-94).
//   4. tests: one thread per test pair draws its two entries
//      (find_rand_pair, :766-803), evaluates the weighted kernel (FP64, or
//      FP32 with an FP64 recheck inside the band) and accepts with
//      probability k/k_max (maybe_coag_pair, :712-759).
//   5. claims: an accepted test claims both particles with atomicMin of its
//      sequential index; a test wins when it holds both claims, i.e. no
//      earlier accepted test in the reference order touched either
//      particle.  Winners merge (coagulate_weighting + coagulate,
//      :810-985); losers are re-drawn in another round against the
//      particles still untouched this step.
//   6. compaction: slots freed by merges are filled from the tail.
// The step is deterministic: every draw is addressed by (box, step, site,
// ordinal) and every conflict is resolved by sequential index.
#pragma once

#include <rocprim/block/block_load.hpp>
#include <rocprim/block/block_radix_sort.hpp>
#include <rocprim/device/device_radix_sort.hpp>

#include "pmc_scan.h"

#include <string>
#include <vector>

namespace pmc {

constexpr int TILE_THREADS = 256;
constexpr int TILE_ITEMS = 16;
constexpr int TILE = TILE_THREADS * TILE_ITEMS;
constexpr uint32_t UNCLAIMED = 0xFFFFFFFFu;
constexpr uint8_t ST_LIVE = 0, ST_HOLE = 1, ST_NEW = 2;
constexpr int PAR_ROUNDS = 2;  // device-wide claim rounds before the per-box tail
static_assert(PAR_ROUNDS >= 1, "the tail runs on the pending list of a round");
constexpr int MAX_REDRAW = 64;

// What the claims and the list bookkeeping of a step keep per particle slot,
// in one 32-byte record: an event that touches a particle at random then
// touches one line (and one page) for all of it, not one per field.  The
// second half is read as one 16-byte word.
struct alignas(32) SlotRec {
  uint32_t claim;     // earliest event that accesses the particle this round
  uint32_t claim_wr;  // ... and earliest that changes it
  uint32_t dead_t;    // test index of the winner that consumed it
  int dead_r;         // claim round (step-wide count) of that winner
  int key0;           // a touched slot's list key at step start
  uint32_t depart_t;  // when a touched slot's step-start particle left that list
  int arr_of;         // pool entry of the arrival a slot holds
  uint32_t st;        // (epoch << 2) | state; another step's epoch reads as live
};

// A target event's outcome, in one line.
struct alignas(64) EventRec {
  int nsamp, ncoag;    // samples and coagulations
  int nrm;             // removed sources
  int nchain, head;    // their chain: entries (with copy markers), first chunk
  int ndup, dhead;     // copies of the target, the first one's pool entry
  int flags, err;
  int nrd, rdhead;     // distinct sources read from small source lists
};
// A pool entry's fields beside its volumes and components.
struct alignas(32) PoolRec {
  int group, nprim, ncomp;
  int next;            // the next copy's entry, -1 after the last
  double least, greatest;
};

struct PW {  // device view of the parallel work arrays
  int K_stride;     // keys per box of the list tables (the allocation's grid)
  int K_hist;       // keys per box of this step's histogram (the step's grid)
  int64_t P_stride; // pair slots per box
  int tab_classes, max_bin;
  int *key;         // [total_cap] list key, -1 for no key
  SlotRec *slot;    // [total_cap]
  int epoch;        // this step's status epoch, 1..63
  int tag;          // this step's tag (RC_REGRID)
  float4 *terms;    // [total_cap]
  int *perm;        // [total_cap] global slots sorted by (box, key)
  int *tile_box, *tile_start, *tiles_in_box;
  int64_t *tile_first;  // [n_box] first tile of the box; its histogram starts at K_hist * this
  uint32_t *hist, *hist_scan;
  int *lstart, *lcnt, *live;  // [n_box * K_stride]
  uint32_t *pair_n, *pair_exc;  // [n_box * P_stride (+1)]
  int *acc, *acc_scan, *tp1, *tp2;
  uint32_t *tid, *pend;
  uint32_t *ev_t;
  int *ev_p1, *ev_p2, *ev_box, *ev_out;
  int *f_app, *f_id, *f_info, *f_hole, *f_pend, *s_pend;
  int *s_app, *s_id, *s_info, *s_hole;
  int *box_first;
  uint64_t *holes, *holes_sorted;  // (box << 32 | slot)
  int *cmp_lo, *cmp_hi, *cmp_head;  // [n_box] compaction: hole range and holes below the final count
  unsigned long long *acc_samp;  // samples drawn by the device-wide target walks
  // accelerated per-particle path (try_per_particle_coag): one test slot per
  // target particle, one event record per target slot of a batch
  uint8_t *pair_acc;           // [NP] 0 per-set; 1 targets in (b1, c1); 2 targets in (b2, c2)
  uint32_t *pair_accn;         // [NP + 1] target slots (first accelerated pair of a list)
  uint32_t *acc_exc;           // [NP + 1] their exclusive scan
  int *trec;                   // [T_cap] record of a test slot, -1 for per-set tests
  int *tns;                    // [T_cap] n_samp (+ ACC_WARN) of a target without effect
  int *ev_rec;                 // [T_cap] record of an event, -1 for per-set events
  int acc_cap, pool_cap;
  EventRec *ev;                // [acc_cap] event records
  // particle pool [pool_cap]: entry r < acc_cap is the final target of
  // record r; entries from acc_cap on are the copies (aero_state_dup_particle)
  double *q_vol;               // [pool_cap][n_spec]
  PoolRec *q;                  // [pool_cap]
  int *q_csrc;                 // [pool_cap][MAX_COMP]
  double *q_ctime;             // [pool_cap][MAX_COMP]
  int *dup_top;                // [1] copy allocator of the round
  int *rm_buf;                 // chunks: [0] next chunk or -1, [1..RM_CHUNK) removed slots
  int *rm_top;                 // [1] chunk allocator of the round
  int rm_cap;
  unsigned long long *hole_top;  // [8] hole counter; then tail_rounds and rstat
  int *pend_k;                 // [T_cap] pair of each pending test entering the tail
  uint32_t *tpair;             // [T_cap] pair of every test of a single-batch step
  int tpair_ok;                // tpair is current for this step
  unsigned long long *tail_rounds;  // [1] claim rounds run by the tail, summed over boxes
  // Particles that join a list within the step ("arrivals": a merged
  // particle that lands in another (bin, class) than its slot's list, an
  // appended particle).  The draws of every pair reserve acap entries after
  // each list's n step-start members; the j-th reserved entry is the list's
  // j-th arrival before the pair begins (in sequence order).
  int *acap;          // [n_box * K_stride] reserved arrival entries of the list this step
  int *arr_n;         // [n_box * K_stride] arrivals recorded this step
  int *arr_head;      // [n_box * K_stride] the list's arrivals beyond A_MAX: first entry, -1 none
  // arrival pool: list L's first A_MAX arrivals at L * A_MAX + i, the rest
  // from ap_ovf on, chained from arr_head[L]
  int *ap_p;          // the arrival's slot
  uint32_t *ap_t;     // sequence index at which it joined the list
  uint32_t *ap_dep;   // at which it left again (UNCLAIMED: still there)
  int *ap_next;       // next overflow arrival of the same list
  uint32_t *ap_top;   // [1] overflow entries used this step
  int64_t ap_ovf;     // n_box * K_stride * A_MAX
  uint32_t ap_cap;    // overflow entries
  uint8_t *thin;      // [T_cap] the test's last draw was thinned (per batch)
  // Per (box, bin): the lowest index of an event pending at the start of
  // this round whose results land in that bin or a lower one (tests on an
  // empty arrival entry excluded; particles only grow, so an event on bins
  // b1, b2 adds particles to bins from max(b1, b2) up), as a running
  // minimum over the bins; and the same, per bin, for the next round.
  uint32_t *minpend, *minpend_next;  // [n_box * K_stride] each
  uint32_t *scan_part;  // [SCAN_COLS * SCAN_MAX_BLOCKS] chunk totals of the device-wide scans
  // The counts that drive a batch's claim rounds, kept on the device so the
  // host launches every round without reading them back: RC_N tests of the
  // current device-wide round (0: the round does not run), RC_E its events,
  // RC_TAIL the tests left to the tail; RC_REGRID the tag of the last step
  // that gave a box a new grid.
  int *rc;                      // [RC_SIZE]
  unsigned long long *pstat;    // [2] device-wide rounds run, tests left to the tail
  // the batch's round sizes, read back with the hole count after the tail to
  // size the next step's grids: round 0's events, round 1's tests and
  // events, the tail's tests (in the allocation of hole_top, after
  // tail_rounds)
  unsigned long long *rstat;    // [4]
};

constexpr int RC_N = 0, RC_E = 1, RC_TAIL = 2, RC_REGRID = 3, RC_SIZE = 4;

constexpr int ACC_CAP = 1 << 18;
constexpr int DUP_CAP = 1 << 18;
constexpr int RM_CHUNK = 16;
constexpr int CHAIN_WAVE_MIN = 32;  // removal chains longer than this are applied by a wavefront
constexpr int RM_CAP = 1 << 24;
constexpr int ACC_WARN = 1 << 30;
constexpr int READ_TRACK = 128;  // source lists up to this size have their reads tracked
constexpr int RF_WARN = 1, RF_DIED = 2, RF_MERGED = 4;
constexpr int A_MAX = 128;      // arrival entries a list can reserve
constexpr int ARR_REACH = 3;    // an empty list reserves entries when a list at most this many bins below is occupied
constexpr int TNS_ATHIN = 1 << 29;  // tns bit of a test or target event on an empty arrival entry
constexpr int TNS_SIDE2 = 1 << 28;  // ... of the pair's second list

struct ParallelWork {
  int n_box = 0;
  int64_t T_cap = 1 << 22;
  int64_t hole_cap = 0;
  int64_t H = 0, NP = 0;
  int n_tiles = 0;
  PW d{};
  void *sort_tmp = nullptr;
  size_t sort_tmp_bytes = 0;
  std::vector<int> tiles_in_box;
  uint32_t *h_u32 = nullptr;  // pinned scalars
  unsigned long long *h_u64 = nullptr;
  // optional per-kernel timing hooks of the owning handle
  void (*tbegin)(void *, const char *, hipEvent_t *) = nullptr;
  void (*tend)(void *, const char *, hipEvent_t) = nullptr;
  void *tctx = nullptr;
  hipStream_t tst = nullptr;  // stream of the launch being timed, when not the handle's
  int epoch = 0;              // status epoch of the last step (0: the array is clear)
  // a second stream (default priority) for the target walks, which run
  // beside the per-set tests of the same round
  hipStream_t st2 = nullptr;
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  int64_t n_tail_rounds = 0;  // the tail's claim rounds, summed over boxes
  int64_t rid = 1;        // round identifiers: a fresh one for every claim round
  unsigned long long *pstat = nullptr;  // [2] device-wide rounds run, tests left to the tail
  // the last batch's round 0 events, round 1 tests and events, tail tests
  // (-1: none yet): the grids of the next step's rounds are sized from them
  int64_t est[4] = {-1, -1, -1, -1};
  // The last step left every box's keys, terms and tables current for this
  // kernel type and precision (0: not, or a call changed a box since), with
  // grids of at most mb_step bins.
  int clean_type = 0, clean_terms = 0, mb_step = 0;
  int tag = 0;                // the last step's tag (RC_REGRID)
};

#define PLAUNCH(W, name, ...)                                   \
  do {                                                          \
    hipEvent_t ev_;                                             \
    if ((W).tbegin) (W).tbegin((W).tctx, name, &ev_);           \
    hipLaunchKernelGGL(__VA_ARGS__);                            \
    if ((W).tend) (W).tend((W).tctx, name, ev_);                \
  } while (0)

static std::string g_parallel_error;
inline const char *parallel_last_error() { return g_parallel_error.c_str(); }

#define PCHECK(expr)                                                       \
  do {                                                                     \
    hipError_t e_ = (expr);                                                \
    if (e_ != hipSuccess) {                                                \
      g_parallel_error = std::string(#expr) + ": " + hipGetErrorString(e_); \
      return ERR_HIP;                                                      \
    }                                                                      \
  } while (0)

template <class T>
static hipError_t pmalloc(T **p, size_t n) {
  return hipMalloc((void **)p, (n > 0 ? n : 1) * sizeof(T));
}

// ------------------------------------------------------------ kernels
__device__ inline int par_key(int bin, int cls, int nb) { return (bin - 1) + nb * (cls - 1); }

// keys (and optionally FP32 terms and cached volumes) for every particle of
// boxes whose keys are stale; terms for boxes whose terms are stale.  A target
// event that ended in an error held claims and is in no list that releases
// them: the slots of a box that goes on after an error are released here (a
// claim left on a source holds up every event that reads it, for good).
__global__ void __launch_bounds__(TILE_THREADS)
k_par_rekey(BoxDesc *boxes, Arrays A, PW W, int type, int want_terms, int phase) {
  const int tile = blockIdx.x;
  const int box = W.tile_box[tile];
  BoxDesc *B = &boxes[box];
  if (B->error) return;
  if (phase == 0 && B->revived)
    for (int it = 0; it < TILE_ITEMS; ++it) {
      const int64_t i = W.tile_start[tile] + it * TILE_THREADS + threadIdx.x;
      if (i >= B->cap) continue;
      W.slot[B->off + i].claim = UNCLAIMED;
      W.slot[B->off + i].claim_wr = UNCLAIMED;
    }
  const bool do_keys = phase == 0 ? (!B->pkeys_valid && B->valid_sort && B->n_bin > 0)
                                  : (B->rekey != 0);
  const bool do_terms = want_terms && phase == 0 && B->terms_kernel != type;
  if (!do_keys && !do_terms) return;
  const int n = B->n_part;
  const int nb = B->n_bin;
  const Env env = B->env;
  const int64_t base = B->off;
  int *live = W.live + (int64_t)box * W.K_stride;
  for (int it = 0; it < TILE_ITEMS; ++it) {
    int i = W.tile_start[tile] + it * TILE_THREADS + threadIdx.x;
    if (i >= n) continue;
    int64_t p = base + i;
    double v = particle_volume(A, p);
    A.vtot[p] = v;
    if (do_keys) {
      int b = bin_find_log(nb, B->log_lo, B->log_hi, vol2rad(v));
      if (b < 1 || b > nb) {
        atomicExch(&B->error, 708651144);
        continue;
      }
      int cls = A.klass[p];
      if (cls < 1 || cls > B->w.n_class) {
        atomicExch(&B->error, 233133947);  // weight class out of range
        continue;
      }
      int k = par_key(b, cls, nb);
      W.key[p] = k;
      atomicAdd(&live[k], 1);
    }
    if (do_terms) {
      double m = 0.0;
      for (int s = 0; s < A.n_spec; ++s) m += A.vol[(int64_t)s * A.total_cap + p] * A.density[s];
      W.terms[p] = particle_terms(type, v, m / v, env);
    }
  }
}

__global__ void k_par_zero_live(BoxDesc *boxes, PW W, int n_box, int phase) {
  int box = blockIdx.y;
  BoxDesc *B = &boxes[box];
  bool do_keys = phase == 0 ? (!B->pkeys_valid && B->valid_sort && B->n_bin > 0) : (B->rekey != 0);
  if (!do_keys || B->error) return;
  for (int k = threadIdx.x; k < W.K_stride; k += blockDim.x) W.live[(int64_t)box * W.K_stride + k] = 0;
}

__global__ void k_par_finish_rekey(BoxDesc *boxes, int n_box, int type, int want_terms, int phase) {
  int box = blockIdx.x * blockDim.x + threadIdx.x;
  if (box >= n_box) return;
  BoxDesc *B = &boxes[box];
  if (phase == 0) {
    if (!B->pkeys_valid && B->valid_sort && B->n_bin > 0) B->pkeys_valid = 1;
    if (!B->error) B->revived = 0;
    // FP64 steps do not keep the terms of new particles current
    B->terms_kernel = want_terms ? type : 0;
  } else if (B->rekey) {
    B->rekey = 0;
    B->pkeys_valid = 1;
  }
}

// radius extremes of boxes without a valid sort (r_min/r_max loop of
// src/aero_sorted.F90:293-304); positive doubles order like their bits
__global__ void __launch_bounds__(TILE_THREADS)
k_par_minmax(BoxDesc *boxes, Arrays A, PW W) {
  const int tile = blockIdx.x;
  const int box = W.tile_box[tile];
  BoxDesc *B = &boxes[box];
  if (B->error || (B->valid_sort && B->pkeys_valid)) return;
  const int n = B->n_part;
  unsigned long long lo = ~0ull, hi = 0ull;
  for (int it = 0; it < TILE_ITEMS; ++it) {
    int i = W.tile_start[tile] + it * TILE_THREADS + threadIdx.x;
    if (i >= n) continue;
    double r = vol2rad(particle_volume(A, B->off + i));
    unsigned long long bits = (unsigned long long)__double_as_longlong(r);
    lo = min(lo, bits);
    hi = max(hi, bits);
  }
  if (hi) {
    atomicMin(&B->rmin_bits, lo);
    atomicMax(&B->rmax_bits, hi);
  }
}

__global__ void k_par_reset_minmax(BoxDesc *boxes, int n_box) {
  int box = blockIdx.x * blockDim.x + threadIdx.x;
  if (box >= n_box) return;
  boxes[box].rmin_bits = ~0ull;
  boxes[box].rmax_bits = 0ull;
}

// The start of a step, one wavefront a box: its counters, the round state it
// owns cleared, and aero_sorted_remake_if_needed
// (src/aero_sorted.F90:214-373) with the occupancy from the live counts.  A
// box that gets a new grid tags the step: what was launched behind this
// kernel for the old grid then does nothing, and the host starts over from
// the keys.  (One thread a box walked the live counts and made the grid:
// 25 us for 160 bins, 4 here.)
__global__ void __launch_bounds__(64) k_step_front(BoxDesc *boxes, Arrays A, PW W, int64_t NP) {
  const int box = blockIdx.x, lane = threadIdx.x;
  BoxDesc *B = &boxes[box];
  for (int k = lane; k < W.K_stride; k += 64) {
    // at the start of the first round every event of the batch is pending
    W.minpend[(int64_t)box * W.K_stride + k] = 0u;
    W.minpend_next[(int64_t)box * W.K_stride + k] = UNCLAIMED;
  }
  if (lane == 0) {
    W.box_first[box] = -1;
    B->step_samp = 0;
    B->step_coag = 0;
    B->part_steps += B->n_part;
    B->regridded = 0;
    B->rekey = 0;
    if (box == 0) {
      *W.hole_top = 0ull;
      *W.tail_rounds = 0ull;
      *W.ap_top = 0u;
      if (W.ev) {
        *W.rm_top = 0;
        *W.dup_top = 0;
      }
      if (NP > 0) {  // what the pair scans read as their last input
        W.pair_n[NP] = 0;
        W.pair_accn[NP] = 0;
      }
    }
  }
  if (B->error) return;
  double *edges = A.edges + (int64_t)box * (A.max_bin + 1);
  double *centers = A.centers + (int64_t)box * A.max_bin;
  double *widths = A.widths + (int64_t)box * A.max_bin;
  const int nb = B->n_bin, nc = B->w.n_class;
  const bool use_counts = B->valid_sort && B->pkeys_valid;
  double rmin = 0.0, rmax = 0.0;
  if (use_counts) {
    const int *live = W.live + (int64_t)box * W.K_stride;
    int first = nb + 1, last = 0;
    for (int b = 1 + lane; b <= nb; b += 64) {
      int tot = 0;
      for (int c = 1; c <= nc; ++c) tot += live[par_key(b, c, nb)];
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
  } else if (B->valid_sort && nb > 0) {
    // a valid sort whose keys were dropped (population control moved
    // particles): the occupied bins are those of the radius extremes
    rmin = edges[nb];
    rmax = edges[0];
    if (B->n_part > 0) {
      const int b_lo = bin_find_log(nb, B->log_lo, B->log_hi,
                                    __longlong_as_double((long long)B->rmin_bits));
      const int b_hi = bin_find_log(nb, B->log_lo, B->log_hi,
                                    __longlong_as_double((long long)B->rmax_bits));
      rmin = edges[max(b_lo, 1) - 1];
      rmax = edges[min(b_hi, nb)];
    }
  } else if (B->n_part > 0) {
    rmin = __longlong_as_double((long long)B->rmin_bits);
    rmax = __longlong_as_double((long long)B->rmax_bits);
  }
  if (rmax == 0.0) {
    if (lane == 0) {
      if (!use_counts) {
        B->n_bin = 0;
        B->bounds_valid = 0;
        B->tables_valid = 0;
      }
      B->valid_sort = 1;
      B->pkeys_valid = 1;
    }
    return;
  }
  const bool need = (nb < 1) || (rmin / edges[0] < 3.0) || (edges[nb] / rmax < 3.0);
  if (need) {
    const double gmin = rmin / 10.0, gmax = rmax * 10.0;
    const double nbf = ceil((log10(gmax) - log10(gmin)) * 10.0);
    if (nbf < 0.0 || nbf > (double)A.max_bin) {
      if (lane == 0) B->error = nbf < 0.0 ? 538534122 : ERR_CAPACITY;
      return;
    }
    const int nn = (int)nbf;
    make_log_grid_wave(nn, gmin, gmax, edges, centers, widths);
    if (lane == 0) {
      B->n_bin = nn;
      B->log_lo = log(gmin);
      B->log_hi = log(gmax);
      B->bounds_valid = 0;
      B->tables_valid = 0;
      B->regridded = 1;
      B->rekey = 1;
      W.rc[RC_REGRID] = W.tag;
    }
  } else if (!use_counts && lane == 0) {
    B->rekey = 1;
    W.rc[RC_REGRID] = W.tag;
  }
  if (lane == 0) {
    B->valid_sort = 1;
    B->xlists_valid = 0;
  }
}

// tile histogram of keys into hist[box][key][tile]
__global__ void __launch_bounds__(TILE_THREADS)
k_par_hist(BoxDesc *boxes, PW W) {
  const int tile = blockIdx.x;
  const int box = W.tile_box[tile];
  BoxDesc *B = &boxes[box];
  extern __shared__ int s_h[];
  const int K = W.K_hist;
  for (int k = threadIdx.x; k < K; k += TILE_THREADS) s_h[k] = 0;
  __syncthreads();
  const int n = B->error ? 0 : B->n_part;
  const int64_t base = B->off;
  for (int it = 0; it < TILE_ITEMS; ++it) {
    int i = W.tile_start[tile] + it * TILE_THREADS + threadIdx.x;
    if (i < n) atomicAdd(&s_h[W.key[base + i]], 1);
  }
  __syncthreads();
  const int t_in_box = W.tile_start[tile] / TILE;
  const int nt = W.tiles_in_box[box];
  uint32_t *h = W.hist + (int64_t)K * W.tile_first[box];
  for (int k = threadIdx.x; k < K; k += TILE_THREADS) h[(int64_t)k * nt + t_in_box] = (uint32_t)s_h[k];
}

// Stable scatter.  The tile's keys are loaded coalesced and transposed to a
// blocked arrangement (item order = index order), radix-sorted (stable), and
// each item's rank among equal keys of the tile is its sorted position minus
// that of the key's first item.  The first position and the list offset of
// every key present are kept in shared memory (dynamic, 2 * K_stride ints),
// written by the first item of each run.
__global__ void __launch_bounds__(TILE_THREADS)
k_par_scatter(BoxDesc *boxes, PW W, int key_bits) {
  using BLD = rocprim::block_load<int, TILE_THREADS, TILE_ITEMS,
                                  rocprim::block_load_method::block_load_transpose>;
  using BRS = rocprim::block_radix_sort<int, TILE_THREADS, TILE_ITEMS, int>;
  __shared__ union {
    typename BLD::storage_type load;
    typename BRS::storage_type sort;
  } tmp;
  __shared__ int s_keys[TILE];
  extern __shared__ int s_run[];  // [0, K): first sorted position; [K, 2K): list offset
  const int tile = blockIdx.x;
  const int box = W.tile_box[tile];
  BoxDesc *B = &boxes[box];
  const int n = B->error ? 0 : B->n_part;
  const int64_t base = B->off;
  const int sentinel = (1 << key_bits) - 1;
  const int start = W.tile_start[tile];
  const int valid = max(0, min(TILE, n - start));
  int keys[TILE_ITEMS], vals[TILE_ITEMS];
  // coalesced loads, exchanged so that each thread holds TILE_ITEMS
  // consecutive keys
  BLD().load(W.key + base + start, keys, (unsigned)valid, sentinel, tmp.load);
  for (int it = 0; it < TILE_ITEMS; ++it) vals[it] = start + threadIdx.x * TILE_ITEMS + it;
  __syncthreads();
  BRS().sort(keys, vals, tmp.sort, 0, key_bits);
  __syncthreads();
  for (int it = 0; it < TILE_ITEMS; ++it) s_keys[threadIdx.x * TILE_ITEMS + it] = keys[it];
  __syncthreads();
  const int K = W.K_stride;
  const int t_in_box = start / TILE;
  const int nt = W.tiles_in_box[box];
  const int64_t o = (int64_t)W.K_hist * W.tile_first[box];
  const uint32_t bbase = W.hist_scan[o];
  for (int it = 0; it < TILE_ITEMS; ++it) {
    const int pos = threadIdx.x * TILE_ITEMS + it;
    const int k = keys[it];
    if (k == sentinel) continue;
    if (pos == 0 || s_keys[pos - 1] != k) {
      s_run[k] = pos;
      s_run[K + k] = (int)(W.hist_scan[o + (int64_t)k * nt + t_in_box] - bbase);
    }
  }
  __syncthreads();
  for (int it = 0; it < TILE_ITEMS; ++it) {
    const int pos = threadIdx.x * TILE_ITEMS + it;
    const int k = keys[it];
    if (k == sentinel) continue;
    const int dst = s_run[K + k] + (pos - s_run[k]);
    W.perm[base + dst] = (int)(base + vals[it]);
  }
}

// 64-bit divisions take about five times a 32-bit one: used only where an
// operand needs them.
__device__ inline void decode_pair(int64_t q, int tc, int mb, int *c1, int *c2, int *b1, int *b2) {
  uint32_t cls, rem;
  if (((uint64_t)q >> 32) == 0) {
    const uint32_t mb2 = (uint32_t)mb * (uint32_t)mb;
    cls = (uint32_t)q / mb2;
    rem = (uint32_t)q - cls * mb2;
  } else {
    const int64_t mb2 = (int64_t)mb * mb;
    cls = (uint32_t)(q / mb2);
    rem = (uint32_t)(q % mb2);
  }
  const uint32_t k1 = cls / (uint32_t)tc, r1 = rem / (uint32_t)mb;
  *c1 = (int)k1 + 1;
  *c2 = (int)(cls - k1 * (uint32_t)tc) + 1;
  *b1 = (int)r1 + 1;
  *b2 = (int)(rem - r1 * (uint32_t)mb) + 1;
}

// the box of global pair k, and the pair's index in it
__device__ inline int pair_box(const PW &W, int64_t k, int64_t *q) {
  int box;
  if (((uint64_t)(k | W.P_stride) >> 32) == 0) box = (int)((uint32_t)k / (uint32_t)W.P_stride);
  else box = (int)(k / W.P_stride);
  *q = k - (int64_t)box * W.P_stride;
  return box;
}

// The step's arguments for the functions called out of line (target visits
// and their merges), in LDS: passed by reference they would live in each
// lane's private memory, and every pointer read from there waits for all
// loads in flight.  A kernel that calls them fills it first.  With this, the
// volumes in registers (RecN) and the records in one line each, a tail round
// of 1e5 Brownian particles spends 23 us on visits and tests (28 before).
struct StepCtx {
  Arrays A;
  PW W;
};
static __shared__ StepCtx s_ctx;
__device__ inline void step_ctx_fill(const Arrays &A, const PW &W) {
  for (int q = threadIdx.x; q < (int)(sizeof(Arrays) / sizeof(int)); q += blockDim.x)
    ((int *)&s_ctx.A)[q] = ((const int *)&A)[q];
  for (int q = threadIdx.x; q < (int)(sizeof(PW) / sizeof(int)); q += blockDim.x)
    ((int *)&s_ctx.W)[q] = ((const int *)&W)[q];
  __syncthreads();
}

// loops over a record's species: unrolled over NS where that is few, so
// that the record stays in registers
#define REC_FOR(s, ns) for (int s = 0; s < (NS <= FEW_SPEC ? NS : (ns)); ++s) if (NS > FEW_SPEC || s < (ns))

// the record without its components (they are read in a second pass
// that depends on ncomp, so a reader that may not need them defers it)
template <int NS>
__device__ inline void load_rec_head(const Arrays &A, int64_t p, RecN<NS> &r) {
  const int ns = A.n_spec;
  if (NS <= FEW_SPEC) {
    double x[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) x[s] = A.vol[(int64_t)(s < ns ? s : ns - 1) * A.total_cap + p];
#pragma unroll
    for (int s = 0; s < NS; ++s) r.vol[s] = x[s];
  } else {
    for (int s = 0; s < ns; ++s) r.vol[s] = A.vol[(int64_t)s * A.total_cap + p];
  }
  r.id = A.id[p];
  r.group = A.group[p];
  r.klass = A.klass[p];
  r.nprim = A.nprim[p];
  r.ncomp = A.ncomp[p];
  r.least = A.least[p];
  r.greatest = A.greatest[p];
}

template <int NS>
__device__ inline void load_rec_comps(const Arrays &A, int64_t p, RecN<NS> &r) {
  for (int c = 0; c < r.ncomp; ++c) {
    r.csrc[c] = A.csrc[comp_at(p, c)];
    r.ctime[c] = A.ctime[comp_at(p, c)];
  }
}

template <int NS>
__device__ inline void load_rec(const Arrays &A, int64_t p, RecN<NS> &r) {
  load_rec_head(A, p, r);
  load_rec_comps(A, p, r);
}

// aero_particle_coagulate for the parallel path (same rules as rec_coagulate)
template <int NS>
__device__ inline int par_rec_coagulate(int n_spec, Stream &s, const RecN<NS> &p1,
                                        const RecN<NS> &p2, RecN<NS> &o) {
  REC_FOR(k, n_spec) o.vol[k] = p1.vol[k] + p2.vol[k];
  o.group = 0;
  o.klass = 0;
  o.id = 0;
  int n1 = p1.ncomp, n2 = p2.ncomp;
  if (p1.nprim < n1) return 465791384;
  if (p2.nprim < n2) return 465791385;
  for (int c = 0; c < MAX_COMP; ++c) {
    o.csrc[c] = 0;
    o.ctime[c] = 0.0;
  }
  if (n1 + n2 > MAX_COMP) {
    int n1_new = prob_round(s, (double)p1.nprim / (double)(p1.nprim + p2.nprim) * (double)MAX_COMP);
    int n2_new = MAX_COMP - n1_new;
    int sample[MAX_COMP];
    sample_without_replacement(s, n1_new, n1, sample);
    for (int i = 0; i < n1_new; ++i) {
      o.csrc[i] = p1.csrc[sample[i] - 1];
      o.ctime[i] = p1.ctime[sample[i] - 1];
    }
    sample_without_replacement(s, n2_new, n2, sample);
    for (int i = 0; i < n2_new; ++i) {
      o.csrc[i + n1_new] = p2.csrc[sample[i] - 1];
      o.ctime[i + n1_new] = p2.ctime[sample[i] - 1];
    }
    o.ncomp = MAX_COMP;
  } else {
    for (int i = 0; i < n1; ++i) {
      o.csrc[i] = p1.csrc[i];
      o.ctime[i] = p1.ctime[i];
    }
    for (int i = 0; i < n2; ++i) {
      o.csrc[n1 + i] = p2.csrc[i];
      o.ctime[n1 + i] = p2.ctime[i];
    }
    o.ncomp = n1 + n2;
  }
  o.least = fmin(p1.least, p2.least);
  o.greatest = fmax(p1.greatest, p2.greatest);
  o.nprim = p1.nprim + p2.nprim;
  return 0;
}

// try_per_particle_coag's tests (src/coagulation.F90:150-215): monotone
// decreasing weights, target weight strictly below the source weight with
// the destination class the target's, at least one expected source per
// target, and at most 1.5x growth.  Returns 0 (per-set path), 1 (targets in
// (b1, c1)) or 2 (targets in (b2, c2)).
__device__ inline int accel_kind(const Weights &w, const double *edges, int b1, int b2, int c1,
                                 int c2, int cc, double k_max, double del_t, const int *cnt, int nb,
                                 double *n_spt_out) {
  for (int i = 0; i < w.n_group * w.n_class; ++i)
    if (w.type[i] == WEIGHT_POWER && w.expo[i] > 0.0) return 0;
  double a1 = nc_at_radius(w, c1, edges[b1 - 1]), a2 = nc_at_radius(w, c1, edges[b1]);
  double d1 = nc_at_radius(w, c2, edges[b2 - 1]), d2 = nc_at_radius(w, c2, edges[b2]);
  double nc1_min = fmin(a1, a2), nc1_max = fmax(a1, a2);
  double nc2_min = fmin(d1, d2), nc2_max = fmax(d1, d2);
  int kind = 0, bt = 0, bs = 0, cs = 0;
  if (nc1_max < nc2_min && cc == c1) {
    kind = 1; bt = b1; bs = b2; cs = c2;
  }
  if (nc2_max < nc1_min && cc == c2) {
    kind = 2; bt = b2; bs = b1; cs = c1;
  }
  if (!kind) return 0;
  double n_spt = k_max * del_t * (double)cnt[par_key(bs, cs, nb)];
  if (n_spt < 1.0) return 0;
  double min_tv = rad2vol(edges[bt - 1]);
  double max_sv = rad2vol(edges[bs]);
  if ((min_tv + max_sv * n_spt) / min_tv > 1.5) return 0;
  *n_spt_out = n_spt;
  return kind;
}

// The most tests a bin pair may expect: its draw stays within an int by more
// than a thousand standard deviations.
constexpr double MAX_PAIR_TESTS = 2.0e9;

// n_samp of every (box, c1, c2, b1, b2), compute_n_samp
// src/coagulation.F90:648-702 on the pair's own Poisson stream
__global__ void k_par_pairs(BoxDesc *boxes, Arrays A, PW W, double del_t, uint64_t seed,
                            uint32_t step) {
  const int box = blockIdx.y;
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= W.P_stride || W.rc[RC_REGRID] == W.tag) return;
  BoxDesc *B = &boxes[box];
  uint32_t ns = 0;
  int acc = 0;
  uint32_t na = 0;  // target events of an accelerated pair
  if (!B->error) {
    int c1, c2, b1, b2;
    decode_pair(q, W.tab_classes, W.max_bin, &c1, &c2, &b1, &b2);
    const int nb = B->n_bin, nc = B->w.n_class;
    if (c1 <= nc && c2 <= c1 && b1 <= nb && b2 <= nb && (c1 != c2 || b2 >= b1)) {
      const int *cnt = W.lcnt + (int64_t)box * W.K_stride;
      int n1 = cnt[par_key(b1, c1, nb)], n2 = cnt[par_key(b2, c2, nb)];
      const int64_t ti = table_index(A, box, nb, nc, b1, b2, c1, c2);
      double k_max = A.kw[ti];
      const double *edges = A.edges + (int64_t)box * (A.max_bin + 1);
      double n_spt;
      // eligibility needs only the source list: a target that grows into
      // an empty bin during the step still visits that bin's pairs
      acc = accel_kind(B->w, edges, b1, b2, c1, c2, A.cc[ti], k_max, del_t, cnt, nb, &n_spt);
      if (acc) {
        // one event per entry of the target list when the loop reaches the
        // pair: its reserved arrival entries, then its step-start members;
        // none when the source list is empty
        if (n1 > 0 && n2 > 0) atomicAdd((unsigned long long *)&B->n_accel_pairs, 1ull);
        const int kt = acc == 1 ? par_key(b1, c1, nb) : par_key(b2, c2, nb);
        const int n_src = acc == 1 ? n2 : n1;
        const int *acp = W.acap + (int64_t)box * W.K_stride;
        if (n_src > 0) na = (uint32_t)(cnt[kt] + acp[kt]);
        ns = na;
      } else {
        // the bound on the lists when the loop reaches the pair: step-start
        // members plus reserved arrival entries (draws thin to the members)
        const int *acp = W.acap + (int64_t)box * W.K_stride;
        const double N1 = (double)(n1 + acp[par_key(b1, c1, nb)]);
        const double N2 = (double)(n2 + acp[par_key(b2, c2, nb)]);
        bool same = (b1 == b2) && (c1 == c2);
        double n_possible = same ? N1 * (N2 - 1.0) / 2.0 : N1 * N2;
        double mean = k_max * del_t * n_possible;
        if (n_possible > 0.0 && !(mean <= MAX_PAIR_TESTS)) {  // past an int, or no number
          atomicExch(&B->error, ERR_CAPACITY);
          mean = 0.0;
        }
        Stream ps;
        ps.open(seed, box, step, pair_site(nb, nc, b1, b2, c1, c2), 0, RNG_POISSON);
        ns = n_possible > 0.0 ? (uint32_t)rand_poisson(ps, mean) : 0u;
        if (ns) {
          atomicAdd((unsigned long long *)&B->n_samp, (unsigned long long)ns);
          atomicAdd((unsigned long long *)&B->step_samp, (unsigned long long)ns);
        }
      }
    }
  }
  W.pair_n[(int64_t)box * W.P_stride + q] = ns;
  W.pair_acc[(int64_t)box * W.P_stride + q] = (uint8_t)acc;
  W.pair_accn[(int64_t)box * W.P_stride + q] = na;
}

__device__ inline int64_t find_pair(const uint32_t *exc, int64_t n, uint32_t t) {
  // last index k with exc[k] <= t  (exc has n + 1 entries, exc[n] = total)
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    int64_t mid = (lo + hi + 1) >> 1;
    if (exc[mid] <= t) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// the pair of test t: from the step's test-to-pair table when it covers
// the step, else by binary search
__device__ inline int64_t test_pair(const PW &W, int64_t NP, uint32_t t) {
  return W.tpair_ok ? (int64_t)W.tpair[t] : find_pair(W.pair_exc, NP, t);
}

// The pair of every test of a single-batch step, and the first batch's
// counts: each wavefront takes 64 pairs, a lane writes the tests of a pair
// with few, the wavefront together those of one with many.
constexpr int FEW_TESTS = 8;
__device__ inline void batch_begin(const PW &W, int n_batch) {
  W.rc[RC_N] = n_batch;
  W.rc[RC_E] = 0;
  W.rc[RC_TAIL] = 0;
  for (int q = 0; q < 4; ++q) W.rstat[q] = 0ull;
}
__global__ void __launch_bounds__(256) k_expand_pairs(PW W, int64_t NP, int table, int n_batch) {
  const int lane = threadIdx.x & 63;
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k == 0) batch_begin(W, n_batch);
  if (!table) return;
  const uint32_t n = k < NP ? W.pair_n[k] : 0u, t0 = k < NP ? W.pair_exc[k] : 0u;
  if (n <= (uint32_t)FEW_TESTS)
    for (uint32_t i = 0; i < n; ++i) W.tpair[t0 + i] = (uint32_t)k;
  uint64_t many = __ballot(n > (uint32_t)FEW_TESTS);
  while (many) {
    const int src = __ffsll((long long)many) - 1;
    many &= many - 1;
    const uint32_t nn = __shfl(n, src), tt = __shfl(t0, src);
    const uint32_t kk = (uint32_t)(k - lane + src);
    for (uint32_t i = lane; i < nn; i += 64) W.tpair[tt + i] = kk;
  }
}

__device__ inline void atomic_max_double(double *addr, double v) {
  unsigned long long *a = (unsigned long long *)addr;
  unsigned long long nv = (unsigned long long)__double_as_longlong(v);
  atomicMax(a, nv);  // v >= 0
}

// A particle's status this step.  Statuses carry the epoch of the step that
// set them, so a new step starts with every particle live without clearing
// the array (it is cleared when the epoch wraps).
__device__ inline void st_set(const PW &W, int64_t p, uint8_t s) {
  W.slot[p].st = (uint32_t)((W.epoch << 2) | s);
}

// a slot of a step-start list can be drawn while it holds a particle of
// that list's (bin, class): untouched, or changed in place by an earlier
// merge without leaving the list
__device__ inline bool drawable_as(const PW &W, uint32_t st, int key_p, int key) {
  return !((int)(st >> 2) == W.epoch && (st & 3) == ST_HOLE) && key_p == key;
}
__device__ inline bool drawable(const PW &W, int p, int key) {
  const uint32_t st = W.slot[p].st;
  const int key_p = W.key[p];
  return drawable_as(W, st, key_p, key);
}

// ---- list membership within a step
// In the reference a bin pair draws its test count from the lists as they
// are when the loop reaches it (src/coagulation.F90:615-626) and each test
// draws among the members at that moment (:766-803).  Here the count comes
// from an upper bound, each list's n step-start members plus acap reserved
// arrival entries, and a draw thins itself: a member that left before the
// pair began, or a reserved entry with no arrival before then, drops the
// test.  Poisson thinning keeps the surviving count Poisson with the mean
// of the members present when the pair begins.  Within the pair, a member
// that left after the pair began is drawn again among the present ones.

// The fields of slot p that the list bookkeeping reads, loaded together
// (one memory round trip instead of a chain of them).
struct SlotView {
  int key, key0, e;
  uint32_t dep, st;
};
__device__ inline SlotView slot_load(const PW &W, int64_t p) {
  const uint4 h = *(const uint4 *)&W.slot[p].key0;
  return SlotView{W.key[p], (int)h.x, (int)h.z, h.y, h.w};
}
// a slot first changed this step records its step-start list and no
// departure yet
__device__ inline void slot_touch(const PW &W, int64_t p, SlotView &v) {
  if ((int)(v.st >> 2) != W.epoch || (v.st & 3) == ST_LIVE) {
    v.key0 = v.key;
    v.dep = UNCLAIMED;
    W.slot[p].key0 = v.key;
    W.slot[p].depart_t = UNCLAIMED;
  }
}

// An arrival takes the next entry of its list's array, or past A_MAX of
// them an overflow entry linked into the list's chain.  Which entries the
// arrivals take depends on the order of the atomics, so readers use only
// the set: counts and choices by (sequence index, slot) or by a hash of the
// slot.  The entry is complete before the readers of a later round (a
// later kernel, or a tail round behind a barrier) look at it.
__device__ inline void record_arrival(const PW &W, BoxDesc *B, int box, int key, int64_t p,
                                      uint32_t t) {
  const int64_t L = (int64_t)box * W.K_stride + key;
  const int i = atomicAdd(&W.arr_n[L], 1);
  int64_t e;
  if (i < A_MAX) {
    e = L * A_MAX + i;
  } else {
    const uint32_t o = atomicAdd(W.ap_top, 1u);
    if (o >= W.ap_cap) {
      atomicExch(&B->error, ERR_CAPACITY);
      return;
    }
    e = W.ap_ovf + o;
  }
  W.ap_p[e] = (int)p;
  W.ap_t[e] = t;
  W.ap_dep[e] = UNCLAIMED;
  W.slot[p].arr_of = (int)e;
  atomicAdd((unsigned long long *)&B->n_arrivals, 1ull);
  if (i < A_MAX) return;
  W.ap_next[e] = atomicExch(&W.arr_head[L], (int)e);
}

// visit every arrival entry of list L: the array, then the overflow chain
template <class F>
__device__ inline void arrivals_each(const PW &W, int64_t L, F f) {
  const int n = W.arr_n[L];
  const int na = n < A_MAX ? n : A_MAX;
  for (int i = 0; i < na; ++i) f(L * A_MAX + i);
  if (n > A_MAX)
    for (int e = W.arr_head[L]; e >= 0; e = W.ap_next[e]) f((int64_t)e);
}

// the particle in slot p (as v shows it) leaves the list it is in, at
// sequence index t
__device__ inline void slot_leave_view(const PW &W, int64_t p, uint32_t t, const SlotView &v) {
  if (v.key < 0) return;
  if (v.key == v.key0 && v.dep == UNCLAIMED) {
    W.slot[p].depart_t = t;  // the slot's step-start member
    return;
  }
  const int e = v.e;  // an arrival of list v.key
  if (e >= 0 && e < W.ap_ovf + W.ap_cap && W.ap_p[e] == (int)p && W.ap_dep[e] == UNCLAIMED)
    W.ap_dep[e] = t;
}

__device__ inline void slot_leave(const PW &W, int64_t p, uint32_t t, SlotView v) {
  slot_touch(W, p, v);
  slot_leave_view(W, p, t, v);
}
__device__ inline void slot_leave(const PW &W, int64_t p, uint32_t t) {
  slot_leave(W, p, t, slot_load(W, p));
}

// slot p receives a particle of list new_key in place of the one it held
// (a merge into a parent's slot, a target merged in place): the old one
// leaves its list at t_leave, the new one joins at t_join
__device__ inline void slot_write(const PW &W, BoxDesc *B, int box, int64_t p, uint32_t t_leave,
                                  uint32_t t_join, int new_key, SlotView v) {
  slot_touch(W, p, v);
  if (v.key == new_key) return;  // changed in place, still in its list
  slot_leave_view(W, p, t_leave, v);
  if (new_key != v.key0) record_arrival(W, B, box, new_key, p, t_join);
}

// an appended slot receives a particle of list new_key at sequence index t
__device__ inline void slot_append(const PW &W, BoxDesc *B, int box, int64_t p, uint32_t t,
                                   int new_key) {
  W.slot[p].key0 = -1;
  W.slot[p].depart_t = 0;
  record_arrival(W, B, box, new_key, p, t);
}

constexpr int DRAW_THIN = -2, DRAW_ATHIN = -3, DRAW_AGAIN = -4;

// 32-bit mixing (the finalizer of MurmurHash3)
__device__ inline uint32_t mix32(uint32_t h) {
  h ^= h >> 16;
  h *= 0x85ebca6bu;
  h ^= h >> 13;
  h *= 0xc2b2ae35u;
  h ^= h >> 16;
  return h;
}

// A draw on reserved entry j of list L for a pair that begins at tau.  The
// entry holds an arrival when the list had at least j arrivals before tau;
// which one is drawn uniformly among them (not `exclude`, the first draw of
// a test on the same list) as the one whose slot hashes lowest under u.  So
// each arrival present at tau is drawn at the rate of a member.  Returns
// the pool entry and its slot, or -1.
constexpr int ACHUNK = 8;  // arrival entries loaded together

__device__ inline int64_t arrival_draw(const PW &W, int64_t L, int j, uint32_t tau, uint32_t u,
                                       int exclude, int *p_out) {
  int n_before = 0;
  int64_t best = -1;
  uint32_t best_h = 0;
  int best_p = 0;
  auto consider = [&](int64_t e, uint32_t te, int pe) {
    if (te >= tau) return;
    ++n_before;
    if (pe == exclude) return;
    const uint32_t h = mix32(u ^ ((uint32_t)pe * 0x9E3779B9u));
    if (best < 0 || h < best_h || (h == best_h && pe < best_p)) {
      best = e;
      best_h = h;
      best_p = pe;
    }
  };
  // the array part a chunk at a time, its loads issued before any is used
  // (index clamped to the last entry), entries in order as before
  const int n = W.arr_n[L];
  const int na = n < A_MAX ? n : A_MAX;
  const int64_t e0 = L * A_MAX;
  for (int i0 = 0; i0 < na; i0 += ACHUNK) {
    uint32_t te[ACHUNK];
    int pe[ACHUNK];
#pragma unroll
    for (int q = 0; q < ACHUNK; ++q) {
      const int64_t e = e0 + (i0 + q < na ? i0 + q : na - 1);
      te[q] = W.ap_t[e];
      pe[q] = W.ap_p[e];
    }
#pragma unroll
    for (int q = 0; q < ACHUNK; ++q)
      if (i0 + q < na) consider(e0 + i0 + q, te[q], pe[q]);
  }
  if (n > A_MAX)
    for (int e = W.arr_head[L]; e >= 0; e = W.ap_next[e]) consider((int64_t)e, W.ap_t[e], W.ap_p[e]);
  *p_out = best_p;
  return j <= n_before ? best : -1;
}

// The arrival of rank r (1-based, in (sequence index, slot) order) among
// list L's arrivals, if it came before tau: the pool entry, or -1.
__device__ inline int64_t arrival_rank(const PW &W, int64_t L, int r, uint32_t tau) {
  int64_t found = -1;
  arrivals_each(W, L, [&](int64_t e) {
    if (found >= 0) return;
    const uint32_t te = W.ap_t[e];
    const int pe = W.ap_p[e];
    int rank = 0;
    arrivals_each(W, L, [&](int64_t f) {
      const uint32_t tf = W.ap_t[f];
      if (tf < te || (tf == te && W.ap_p[f] < pe)) ++rank;
    });
    if (rank == r - 1) found = te < tau ? e : -2;
  });
  return found >= 0 ? found : -1;
}

// entry c (1-based) of list `key` (list index L, n step-start members
// starting at s) for a pair that begins at tau: the particle, or
// DRAW_THIN (a member that left before tau), DRAW_ATHIN (no arrival there
// before tau), DRAW_AGAIN (a member that left after tau: draw again).  A
// reserved entry takes one more draw from `ts` to pick its arrival.
__device__ inline int draw_entry(const PW &W, int64_t base, int64_t L, int key, int n, int s,
                                 int c, uint32_t tau, Stream &ts, int exclude) {
  // (the fields that decide are loaded together, needed or not)
  if (c <= n) {
    const int p = W.perm[base + s + c - 1];
    const uint32_t stv = W.slot[p].st;
    const int kp = W.key[p];
    const uint32_t dep = W.slot[p].depart_t;
    if (drawable_as(W, stv, kp, key)) return p;
    return dep < tau ? DRAW_THIN : DRAW_AGAIN;
  }
  const uint32_t u = (uint32_t)(ts.uniform() * 4294967296.0);
  int p;
  const int64_t e = arrival_draw(W, L, c - n, tau, u, exclude, &p);
  if (e < 0) return DRAW_ATHIN;
  const uint32_t dep = W.ap_dep[e];
  const uint32_t stv = W.slot[p].st;
  const int kp = W.key[p];
  if (dep < tau) return DRAW_ATHIN;
  return drawable_as(W, stv, kp, key) ? p : DRAW_AGAIN;
}

// List starts and counts of every (box, key) from the scanned histogram, then
// the lists' reserved arrival entries and a fresh arrival log, one workgroup
// a box: lists at most ARR_REACH bins above an occupied one (particles only
// grow) reserve 2 + n/64, and a list that received arrivals in the previous
// step (on the same grid) at least twice as many as it received then.
__global__ void __launch_bounds__(256) k_par_lists(BoxDesc *boxes, PW W) {
  if (W.rc[RC_REGRID] == W.tag) return;  // laid out for another grid
  const int box = blockIdx.x;
  const int nt = W.tiles_in_box[box];
  const int K = W.K_hist;
  const int64_t o = (int64_t)K * W.tile_first[box];
  const uint32_t base = W.hist_scan[o];
  int *cnt = W.lcnt + (int64_t)box * W.K_stride;
  for (int k = threadIdx.x; k < W.K_stride; k += blockDim.x) {
    // keys beyond the step's grid hold no particle: their lists start at the
    // end of the box's, as the last key's list ends
    const int kk = k < K ? k : K - 1;
    const uint32_t e = W.hist_scan[o + (int64_t)kk * nt + nt - 1] + W.hist[o + (int64_t)kk * nt + nt - 1];
    const uint32_t s = k < K ? W.hist_scan[o + (int64_t)k * nt] : e;
    W.lstart[(int64_t)box * W.K_stride + k] = (int)(s - base);
    cnt[k] = (int)(e - s);
  }
  __syncthreads();
  const BoxDesc *B = &boxes[box];
  const int nb = B->n_bin, nc = B->w.n_class;
  const bool fresh = B->regridded || B->rekey;
  for (int k = threadIdx.x; k < W.K_stride; k += blockDim.x) {
    const int64_t L = (int64_t)box * W.K_stride + k;
    const int prev = fresh ? 0 : W.arr_n[L];
    int cap = 0;
    if (!B->error && nb > 0 && k < nb * nc) {
      const int b = k % nb + 1;
      bool near = false;
      for (int c = 1; c <= nc && !near; ++c)
        for (int bb = max(1, b - ARR_REACH); bb <= b && !near; ++bb)
          near = cnt[par_key(bb, c, nb)] > 0;
      if (near) cap = 2 + cnt[k] / 64;
      if (prev > 0) cap = max(cap, 2 * prev + 2);
      cap = min(A_MAX, cap);
    }
    W.acap[L] = cap;
    W.arr_n[L] = 0;
    W.arr_head[L] = -1;
  }
}

// find_rand_pair + maybe_coag_pair (src/coagulation.F90:712-803) for test t
// of pair k (global pair index): the two entries, drawn from the step's
// lists skipping slots whose particle is gone or has left the list's
// (bin, class) -- with every particle present the first draw of each
// stands -- and the accept decision.  A re-run uses the test's own stream:
// on an unchanged state it repeats the earlier outcome, on a changed one it
// is what the sequential chain would draw there.
struct TestOut {
  int p1, p2;
  bool accept;
  bool warn;
  int thin;  // 0: drawn; 1: thinned on a member that left before the pair; 2 (3): on an empty
            // arrival entry of the first (second) list
};

__device__ __forceinline__ void perset_test(BoxDesc *B, const Arrays &A, const PW &W, int box,
                                            int64_t k, int64_t q, uint32_t t, int type,
                                            uint64_t seed, uint32_t step, int precision,
                                            double band, int validation, TestOut &o,
                                            const Weights &w) {
  o.p1 = o.p2 = -1;
  o.accept = false;
  o.warn = false;
  o.thin = 0;
  int c1, c2, b1, b2;
  decode_pair(q, W.tab_classes, W.max_bin, &c1, &c2, &b1, &b2);
  const uint32_t tau = W.pair_exc[k];  // where the pair begins in the sequence
  const uint32_t j = t - tau;
  const int nb = B->n_bin, nc = w.n_class;
  const int64_t ti = table_index(A, box, nb, nc, b1, b2, c1, c2);
  const int cc = A.cc[ti];
  const double accept_factor = 1.0 / A.kw[ti];
  const bool same = (b1 == b2) && (c1 == c2);
  const int64_t lb = (int64_t)box * W.K_stride;
  const int key1 = par_key(b1, c1, nb), key2 = par_key(b2, c2, nb);
  const int n1 = W.lcnt[lb + key1], n2 = W.lcnt[lb + key2];
  const int s1 = W.lstart[lb + key1], s2 = W.lstart[lb + key2];
  const int N1 = n1 + W.acap[lb + key1], N2 = n2 + W.acap[lb + key2];
  const int64_t base = B->off;
  Stream ts;
  ts.open(seed, box, step, pair_site(nb, nc, b1, b2, c1, c2), j, RNG_TEST);
  // each side's first draw thins the test or stands; a member that left
  // within the pair is drawn again among those present
  int p1 = -1, p2 = -1;
  int i1 = 0;
  for (int a = 0; a < MAX_REDRAW; ++a) {
    const int c = rand_int(ts, N1);
    const int p = draw_entry(W, base, lb + key1, key1, n1, s1, c, tau, ts, -1);
    if (p >= 0) {
      i1 = c;
      p1 = p;
      break;
    }
    if (a == 0 && p != DRAW_AGAIN) {
      o.thin = p == DRAW_THIN ? 1 : 2;
      return;
    }
  }
  if (p1 >= 0 && (!same || N2 > 1)) {
    for (int a = 0; a < MAX_REDRAW; ++a) {
      int c;
      if (same) {
        c = rand_int(ts, N2 - 1);
        if (c == i1) c = N2;
      } else {
        c = rand_int(ts, N2);
      }
      const int p = draw_entry(W, base, lb + key2, key2, n2, s2, c, tau, ts, same ? p1 : -1);
      if (p >= 0 && p != p1) {
        p2 = p;
        break;
      }
      if (a == 0 && p < 0 && p != DRAW_AGAIN) {
        o.thin = p == DRAW_THIN ? 1 : 3;
        return;
      }
    }
  }
  if (p1 < 0 || p2 < 0) {
    atomicAdd(&B->n_dropped, 1);
    return;
  }
  o.p1 = p1;
  o.p2 = p2;
  const Env env = B->env;
  double u = ts.uniform();
  double pr;
  if (precision == 0) {
    double k64;
    int err = weighted_kernel64(A, w, env, type, p1, p2, c1, c2, cc, &k64);
    if (err) atomicExch(&B->error, err);
    pr = k64 * accept_factor;
    o.accept = u < pr;
  } else {
    float k32 = weighted_kernel32(type, w, env, W.terms[p1], W.terms[p2], c1, c2, cc);
    double p32 = (double)k32 * accept_factor;
    bool need64 = !(fabs(u - p32) >= band) || validation;
    double k64 = 0.0;
    if (need64) {
      int err = weighted_kernel64(A, w, env, type, p1, p2, c1, c2, cc, &k64);
      if (err) atomicExch(&B->error, err);
    }
    if (!(fabs(u - p32) >= band)) {
      atomicAdd((unsigned long long *)&B->n_recheck, 1ull);
      pr = k64 * accept_factor;
      o.accept = u < pr;
    } else {
      pr = p32;
      o.accept = u < p32;
      if (validation && (o.accept != (u < k64 * accept_factor)))
        atomicAdd((unsigned long long *)&B->n_flip, 1ull);
    }
    if (validation && k64 > 0.0) {
      atomic_max_double(&B->max_rel_err, fabs((double)k32 - k64) / k64);
      atomic_max_double(&B->max_p_err, fabs(p32 - k64 * accept_factor));
    }
  }
  o.warn = !(pr <= 1.0);
}

// outcome bits of ev_out
constexpr int O_WIN = 1, O_RM1 = 2, O_RM2 = 4, O_NEW = 8, O_SLOT1 = 16, O_SLOT2 = 32,
              O_APPEND = 64, O_ID1 = 128, O_ID2 = 256, O_NEWID = 512, O_INFO1 = 1024,
              O_INFO2 = 2048;

struct MergeCtx {
  int box, c1, c2, b1, b2;
  uint32_t j;
};

__device__ inline MergeCtx merge_ctx(BoxDesc *boxes, const PW &W, int n_box, uint32_t t) {
  MergeCtx m;
  const int64_t NP = (int64_t)n_box * W.P_stride;
  const int64_t k = test_pair(W, NP, t);
  int64_t q;
  m.box = pair_box(W, k, &q);
  decode_pair(q, W.tab_classes, W.max_bin, &m.c1, &m.c2, &m.b1, &m.b2);
  m.j = t - W.pair_exc[k];
  return m;
}

// coagulate_weighting (src/coagulation.F90:810-922): decisions only
// w: the box's weights (the tail stages them in LDS)
__device__ inline int merge_decide(const Arrays &A, const PW &W, const BoxDesc *B, Stream &s,
                                   int64_t p1, int64_t p2, int c1, int c2, int cc,
                                   int *new_group, const Weights &w) {
  // the parents' volumes and lists, read together up front
  const double v1 = A.vtot[p1], v2 = A.vtot[p2];
  const int key_p1 = W.key[p1], key_p2 = W.key[p2];
  // With one group its draw always stands (its pdf over the largest is 1),
  // and the three uniforms after it come from blocks 1 and 2, drawn side by
  // side; s stands after them as it would draw by draw.
  const bool one = w.n_group == 1;
  uint32_t o1[4], o2[4];
  if (one) {
    s.philox_block(1, o1);
    s.philox_block(2, o2);
    s.seek(5, o2);
  }
  double r1 = vol2rad(v1);
  double r2 = vol2rad(v2);
  double rc = vol2rad(rad2vol(r1) + rad2vol(r2));
  double nc1 = nc_at_radius(w, c1, r1);
  double nc2 = nc_at_radius(w, c2, r2);
  double ncc = nc_at_radius(w, cc, rc);
  double u1, u2, u3;
  if (one) {
    *new_group = 1;
    u1 = u52(o1[0], o1[1]);
    u2 = u52(o1[2], o1[3]);
    u3 = u52(o2[0], o2[1]);
  } else {
    double pdf[MAX_GROUP];
    for (int g = 0; g < w.n_group; ++g) {
      int idx = g + w.n_group * (cc - 1);
      pdf[g] = 1.0 / weight_nc(w.type[idx], w.mag[idx], w.expo[idx], rc);
    }
    *new_group = sample_cts_pdf(s, w.n_group, pdf);
    u1 = s.uniform();
    u2 = s.uniform();
    u3 = s.uniform();
  }
  double nc_min = fmin(nc1, fmin(nc2, ncc));
  bool rm1 = u1 < nc_min / nc1;
  bool rm2 = u2 < nc_min / nc2;
  bool cr = u3 < nc_min / ncc;
  int o = 0;
  if (rm1) o |= O_RM1;
  if (rm2) o |= O_RM2;
  if (cr) o |= O_NEW;
  bool id1_lost, id2_lost;
  if (cr) {
    id1_lost = false;
    id2_lost = false;
    if (rm1 && rm2) {
      if (v1 > v2) id2_lost = true;
      else id1_lost = true;
    }
    if (rm1 && !id1_lost) o |= O_ID1;
    else if (rm2 && !id2_lost) o |= O_ID2;
    else o |= O_NEWID;
    // the new particle takes a freed slot when there is one: the slot of
    // the parent whose list it stays in, if any, so that it can still be
    // drawn from that list in this step (in the reference it joins its
    // bin's list)
    const int nb = B->n_bin;
    const int b_new = bin_find_log(nb, B->log_lo, B->log_hi, rc);
    const int k_new = (b_new >= 1 && b_new <= nb) ? par_key(b_new, cc, nb) : -1;
    if (rm1 && rm2) o |= (key_p2 == k_new && key_p1 != k_new) ? O_SLOT2 : O_SLOT1;
    else if (rm1) o |= O_SLOT1;
    else if (rm2) o |= O_SLOT2;
    else o |= O_APPEND;
  } else {
    id1_lost = rm1;
    id2_lost = rm2;
  }
  if (rm1 && id1_lost) o |= O_INFO1;
  if (rm2 && id2_lost) o |= O_INFO2;
  return o;
}

// A claim on a particle the test changes (removes, or a target it merges
// into): recorded as the earliest accessor and the earliest writer.  A
// particle a test only reads is claimed as accessor only: tests that read
// it win together, a test that changes it waits for earlier readers, and a
// reader waits for earlier writers.
__device__ inline void claim_write(const PW &W, int p, uint32_t t) {
  atomicMin(&W.slot[p].claim, t);
  atomicMin(&W.slot[p].claim_wr, t);
}
// the claim of a test that only reads p.  The few large-weight particles are
// read by thousands of a round's tests: claims only fall within a round, and
// a test that sees an earlier one does not queue at the word (a stale, larger
// value only costs the atomic): the first round's tests of 1e5 Brownian
// particles take 39 us in place of 92.
__device__ inline void claim_read(const PW &W, int p, uint32_t t) {
  if (W.slot[p].claim > t) atomicMin(&W.slot[p].claim, t);
}

// the merge decisions of an accepted per-set test (which parents it
// removes), on the particles as they are before the round's winners apply
__device__ inline int perset_decide(BoxDesc *B, const Arrays &A, const PW &W, int box, int64_t k,
                                    int64_t q, uint32_t t, int p1, int p2, uint64_t seed,
                                    uint32_t step, Stream &ms) {
  int c1, c2, b1, b2;
  decode_pair(q, W.tab_classes, W.max_bin, &c1, &c2, &b1, &b2);
  const int nb = B->n_bin, nc = B->w.n_class;
  const int cc = A.cc[table_index(A, box, nb, nc, b1, b2, c1, c2)];
  ms.open(seed, box, step, pair_site(nb, nc, b1, b2, c1, c2), t - W.pair_exc[k], RNG_MERGE);
  int g;
  return merge_decide(A, W, B, ms, p1, p2, c1, c2, cc, &g, B->w) | (g << 16);
}

// The kernels of a claim round read their item counts from device memory
// (d.rc), and their grids are sized on the host from a bound or an
// estimate: every thread strides over the items.
#define PAR_FOR(i, n) \
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += gridDim.x * blockDim.x)

// test i of the round: draw, evaluate, accept, claim
__device__ __forceinline__ void par_test(BoxDesc *boxes, const Arrays &A, const PW &W, int n_box, int type,
                                uint64_t seed, uint32_t step, uint32_t t0, const uint32_t *pend,
                                int precision, double band, int validation, int i) {
  const uint32_t t = pend ? pend[i] : t0 + (uint32_t)i;
  const int64_t NP = (int64_t)n_box * W.P_stride;
  const int64_t k = test_pair(W, NP, t);
  if (!pend) W.thin[i] = 0;
  if (W.pair_acc[k]) return;  // a target slot: k_par_acc_tests
  W.acc[i] = 0;
  W.tid[i] = t;
  W.tp1[i] = -1;
  W.tp2[i] = -1;
  W.trec[i] = -1;
  W.tns[i] = 0;
  int64_t q;
  const int box = pair_box(W, k, &q);
  BoxDesc *B = &boxes[box];
  if (B->error) return;
  TestOut o;
  perset_test(B, A, W, box, k, q, t, type, seed, step, precision, band, validation, o,
              B->w);
  W.tp1[i] = o.p1;
  W.tp2[i] = o.p2;
  W.thin[t - t0] = o.thin ? 1 : 0;
  // counted once the test is final; a test thinned on an arrival entry waits
  // for the tail, where earlier events are settled first
  W.tns[i] = (o.warn ? ACC_WARN : 0) | (o.thin >= 2 ? TNS_ATHIN : 0) | (o.thin == 3 ? TNS_SIDE2 : 0);
  if (o.accept) {
    W.acc[i] = 1;
    Stream ms;
    const int d = perset_decide(B, A, W, box, k, q, t, o.p1, o.p2, seed, step, ms);
    if (d & O_RM1) claim_write(W, o.p1, t);
    else claim_read(W, o.p1, t);
    if (d & O_RM2) claim_write(W, o.p2, t);
    else claim_read(W, o.p2, t);
  }
}

// STRIDE: the grid may be smaller than the count (a later round, sized from
// an estimate).  The first round's grid covers its tests exactly, and
// without the loop the kernel keeps half the registers.
template <bool STRIDE>
__global__ void __launch_bounds__(256)
k_par_tests(BoxDesc *boxes, Arrays A, PW W, int n_box, int type, uint64_t seed, uint32_t step,
            uint32_t t0, const uint32_t *pend, int precision, double band, int validation) {
  const int n = W.rc[RC_N];
  if (STRIDE) {
    PAR_FOR(i, n) par_test(boxes, A, W, n_box, type, seed, step, t0, pend, precision, band, validation, i);
  } else {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) par_test(boxes, A, W, n_box, type, seed, step, t0, pend, precision, band, validation, i);
  }
}

// ------------------------------------------------ accelerated target slots
// try_per_particle_coag (src/coagulation.F90:150-241).  In the reference
// loop a target particle is visited by every accelerated pair that has its
// current (bin, class) on the target side, in loop order; a target that
// grows into the next bin is visited again by the later pairs of that bin.
// Here each target particle is one test slot, placed in the first
// accelerated pair of its step-start list (targets e = n .. 1, :220-237).
// Its thread walks the remaining pairs in loop order, following the
// target's current bin; in each it samples a virtual source particle
// (sample_source_particle, :333-517) and merges it in
// (coag_target_with_source, :522-582, with aero_state_dup_particle,
// src/aero_state.F90:488-539).  The final target, its copies and the
// removed sources are applied when the event wins all of its claims.

// aero_weight_array_rand_group (src/aero_weight_array.F90:496-514)
__device__ inline int rand_group_w(Stream &s, const Weights &w, int cls, double r) {
  double pdf[MAX_GROUP];
  for (int g = 0; g < w.n_group; ++g) {
    int idx = g + w.n_group * (cls - 1);
    pdf[g] = 1.0 / weight_nc(w.type[idx], w.mag[idx], w.expo[idx], r);
  }
  return sample_cts_pdf(s, w.n_group, pdf);
}

template <int NS>
__device__ inline double rec_vol(int n_spec, const RecN<NS> &r) {
  double v = 0.0;
  REC_FOR(s, n_spec) v += r.vol[s];
  return v;
}

template <int NS>
__device__ inline double rec_density(const Arrays &A, const RecN<NS> &r) {
  double m = 0.0;
  REC_FOR(s, A.n_spec) m += r.vol[s] * A.density[s];
  return m / rec_vol(A.n_spec, r);
}

// the sources a target removes, in a chain of RM_CHUNK-int chunks
struct RmChain {
  int head, cur, fill, n;
  uint64_t bloom;
};

__device__ inline uint64_t rm_bit(int slot) {
  return 1ull << ((((uint32_t)slot * 2654435761u) >> 26) & 63u);
}

__device__ inline bool rm_push(const PW &W, RmChain &c, int slot) {
  if (c.fill == RM_CHUNK) {
    int nc = atomicAdd(W.rm_top, RM_CHUNK);
    if (nc + RM_CHUNK > W.rm_cap) return false;
    W.rm_buf[nc] = -1;
    if (c.cur >= 0) W.rm_buf[c.cur] = nc;
    else c.head = nc;
    c.cur = nc;
    c.fill = 1;
  }
  W.rm_buf[c.cur + c.fill] = slot;
  c.fill++;
  c.n++;
  if (slot >= 0) c.bloom |= rm_bit(slot);
  return true;
}

__device__ inline bool rm_has(const PW &W, const RmChain &c, int slot) {
  if (slot < 0 || !(c.bloom & rm_bit(slot))) return false;
  int left = c.n;
  for (int ch = c.head; ch >= 0 && left > 0; ch = W.rm_buf[ch]) {
    int m = left < RM_CHUNK - 1 ? left : RM_CHUNK - 1;
    for (int q = 1; q <= m; ++q)
      if (W.rm_buf[ch + q] == slot) return true;
    left -= m;
  }
  return false;
}

// entries of a chain loaded together, one memory round trip for all of them
// (and for what the merge reads of their slots): 30 steps of 1e5 Brownian
// particles 116 ms in place of 127 with one entry at a time
constexpr int WALK = 4;

// visit the entries of a list of `left` kept in chunks from `head` on
template <class F>
__device__ inline void chunk_walk(const PW &W, int head, int left, F f) {
  for (int ch = head; ch >= 0 && left > 0; ch = W.rm_buf[ch]) {
    const int m = left < RM_CHUNK - 1 ? left : RM_CHUNK - 1;
    for (int q = 1; q <= m; q += WALK) {
      int e[WALK];
#pragma unroll
      for (int u = 0; u < WALK; ++u) e[u] = W.rm_buf[ch + min(q + u, m)];
#pragma unroll
      for (int u = 0; u < WALK; ++u)
        if (q + u <= m) f(e[u]);
    }
    left -= m;
  }
}

// visit the removed sources of record r in removal order; its chain also
// holds owner markers (-1 - k: the removals that follow belong to copy k)
template <class F>
__device__ inline void rm_walk(const PW &W, int r, F f) {
  chunk_walk(W, W.ev[r].head, W.ev[r].nchain, [&](int q) {
    if (q >= 0) f(q);
  });
}

// visit the sources record r read from small lists
template <class F>
__device__ inline void rd_walk(const PW &W, int r, F f) {
  chunk_walk(W, W.ev[r].rdhead, W.ev[r].nrd, f);
}

template <int NS>
__device__ inline void pool_store(const PW &W, int n_spec, int i, const RecN<NS> &s) {
  REC_FOR(k, n_spec) W.q_vol[(int64_t)i * n_spec + k] = s.vol[k];
  PoolRec &q = W.q[i];
  q.group = s.group;
  q.nprim = s.nprim;
  q.ncomp = s.ncomp;
  for (int c = 0; c < s.ncomp; ++c) {
    W.q_csrc[comp_at(i, c)] = s.csrc[c];
    W.q_ctime[comp_at(i, c)] = s.ctime[c];
  }
  q.least = s.least;
  q.greatest = s.greatest;
}

// sample_source_particle (src/coagulation.F90:333-517) against the running
// target, drawing from the step's source list (list start ss, n_s entries)
// the particles still present that this target has not removed; returns
// an error code, 0 on success.  Sources it removes are pushed to `chain`
// and claimed with index t.
// The target's side of the weighted kernel (as weighted_kernel64), the same
// for every source drawn for one pair: its Brownian terms, volume, radius and weight.
struct TargetSide {
  BrownAir air;
  BrownTerms terms;
  double vol, rad, nc;
};

template <int NS>
__device__ inline TargetSide target_side(const Arrays &A, const Weights &w, const Env &env,
                                         int type, const RecN<NS> &b, int c2) {
  TargetSide ts;
  ts.vol = rec_vol(A.n_spec, b);
  if (type == KERNEL_BROWN) {
    ts.air = brown_air(env.temp, env.pressure);
    ts.terms = brown_terms(ts.air, ts.vol, rec_density(A, b), env.temp);
  }
  ts.rad = vol2rad(ts.vol);
  ts.nc = nc_at_radius(w, c2, ts.rad);
  return ts;
}

// the weighted kernel of a record a of class c1 and the target
template <int NS>
__device__ inline int weighted_kernel_tgt(const Arrays &A, const Weights &w, const Env &env,
                                          int type, const RecN<NS> &a, const TargetSide &ts,
                                          int c1, int cc, double *k_out) {
  double v1 = rec_vol(A.n_spec, a), v2 = ts.vol;
  double k = 0.0;
  int err = 0;
  switch (type) {
    case KERNEL_ADDITIVE: k = env.beta * (v1 + v2); break;
    case KERNEL_CONSTANT: k = C_BETA_0; break;
    case KERNEL_ZERO: k = 0.0; break;
    case KERNEL_BROWN:
      k = brown_combine(brown_terms(ts.air, v1, rec_density(A, a), env.temp), ts.terms);
      break;
    case KERNEL_SEDI: err = kernel_sedi_helper(v1, v2, &k); break;
    default: err = 200724934;
  }
  *k_out = k * coag_num_conc_factor_j(w, vol2rad(v1), rad2vol(ts.rad), ts.nc, c1, cc);
  return err;
}

template <int NS>
__device__ inline int acc_sample_source(const Arrays &A, const PW &W, BoxDesc *B, int type,
                                        const RecN<NS> &target, int ct, int cs, double nc_src_min,
                                        int64_t sbase, int skey, int n_s, double n_spt,
                                        double accept_factor, Stream &aps, Stream &smp,
                                        Stream &fin, uint32_t tau, uint32_t t, bool claim,
                                        RmChain &chain,
                                        RmChain &reads, int *n_samp_out,
                                        int *n_coag_out, int *warn, RecN<NS> &source) {
  const int ns = A.n_spec;
  const Weights &w = B->w;
  const Env env = B->env;
  *n_samp_out = 0;
  *n_coag_out = 0;
  const double nc_target = nc_at_radius(w, target.klass, vol2rad(rec_vol(ns, target)));
  const double prm = nc_target / nc_src_min;
  if (!(prm <= 1.0)) return 653606684;
  const int n_remove = rand_poisson(aps, prm * n_spt);
  const int n_extra = rand_poisson(aps, (1.0 - prm) * n_spt);
  const int n_total = n_remove + n_extra;
  int n_avg = 0, n_samp = 0, n_rm_here = 0, n_thin = 0, n_samp_rm = 0;
  double prob_coag_tot = 0.0;
  double vol_sq[NS], vol_cv[NS];
  REC_FOR(q, ns) {
    vol_sq[q] = 0.0;
    vol_cv[q] = 0.0;
    source.vol[q] = 0.0;
  }
  source.id = 0;
  source.group = source.klass = source.nprim = source.ncomp = 0;
  for (int c = 0; c < MAX_COMP; ++c) {
    source.csrc[c] = 0;
    source.ctime[c] = 0.0;
  }
  source.least = source.greatest = 0.0;
  RecN<NS> pi;
  TargetSide ts;  // formed at the first sample: many pairs draw none
  bool have_ts = false;
  int i_samp = 1;
  for (; i_samp <= n_total; ++i_samp) {
    if (n_rm_here >= n_s) break;  // every source removed
    // the reference's n_samp > n_samp_remove (:413) over the samples kept
    if (i_samp > n_remove && n_samp > n_samp_rm && n_avg >= 2) {
      double cvmax = 0.0;
      REC_FOR(q, ns) {
        double vm = source.vol[q] / (double)n_avg;
        if (vm > 0.0) vol_cv[q] = sqrt(vol_sq[q] / (double)n_avg - vm * vm) / vm;
        if (q == 0 || vol_cv[q] > cvmax) cvmax = vol_cv[q];
      }
      double m95 = cvmax / sqrt((double)n_avg) * student_t_95_coeff(n_avg);
      if (m95 < 0.1) break;
    }
    // a uniform draw among the sources still present.  The counts above
    // come from the step-start list; a source that left before the pair
    // began (tau) was not in the reference's count (compute_n_source,
    // src/coagulation.F90:288-328, reads the list as it is), so a first
    // draw that lands on one thins the sample.  Sources that earlier
    // targets of the pair, or this one, removed are drawn again, as in the
    // reference's loop.
    int ps = -1;
    bool thinned = false;
    for (int a = 0; a < MAX_REDRAW; ++a) {
      int c = rand_int(smp, n_s);
      int q = W.perm[sbase + c - 1];
      if (drawable(W, q, skey) && !rm_has(W, chain, q)) {
        ps = q;
        break;
      }
      if (a == 0 && !drawable(W, q, skey) && W.slot[q].depart_t < tau) {
        thinned = true;
        break;
      }
    }
    if (thinned) {
      n_thin++;
      continue;
    }
    if (ps < 0) {
      atomicAdd(&B->n_dropped, 1);
      break;
    }
    // in a small list a source another target removes changes this
    // target's draws: remember what was read
    if (n_s <= READ_TRACK && !rm_has(W, reads, ps) && !rm_push(W, reads, ps)) return ERR_CAPACITY;
    n_samp++;
    if (i_samp <= n_remove) n_samp_rm++;
    load_rec_head(A, ps, pi);
    double kk;
    if (!have_ts) {
      ts = target_side(A, w, env, type, target, ct);
      have_ts = true;
    }
    int err = weighted_kernel_tgt(A, w, env, type, pi, ts, cs, ct, &kk);
    if (err) return err;
    double prob_coag = kk * accept_factor;
    prob_coag_tot += prob_coag;
    if (smp.uniform() < prob_coag) {
      n_avg++;
      load_rec_comps(A, ps, pi);
      err = par_rec_coagulate(ns, smp, source, pi, source);
      if (err) return err;
      REC_FOR(q, ns) vol_sq[q] += pi.vol[q] * pi.vol[q];
      if (i_samp <= n_remove) {
        double nc_i = nc_at_radius(w, pi.klass, vol2rad(rec_vol(ns, pi)));
        double prob_remove_i = nc_target / nc_i;
        if (smp.uniform() < prob_remove_i / prm) {
          if (!rm_push(W, chain, ps)) return ERR_CAPACITY;
          n_rm_here++;
          if (claim) claim_write(W, ps, t);
        }
      }
    }
  }
  *n_samp_out = n_samp;
  if (n_avg == 0) return 0;
  // the samples the early exit left undrawn thin as the drawn ones did
  for (int i = i_samp; i <= n_total; ++i) {
    const int q = W.perm[sbase + rand_int(smp, n_s) - 1];
    if (!drawable(W, q, skey) && W.slot[q].depart_t < tau) n_thin++;
  }
  double prob_coag_mean = prob_coag_tot / (double)n_samp;
  if (!(prob_coag_mean <= 1.0)) *warn = 1;
  int n_coag = rand_binomial(fin, n_total - n_thin, prob_coag_mean);
  REC_FOR(q, ns) source.vol[q] = source.vol[q] * ((double)n_coag / (double)n_avg);
  source.nprim = prob_round(fin, (double)source.nprim * ((double)n_coag / (double)n_avg));
  const int n_comp = source.ncomp;
  const int n_comp_new = source.nprim < MAX_COMP ? source.nprim : MAX_COMP;
  int sample[MAX_COMP];
  int cs_src[MAX_COMP];
  double ct_src[MAX_COMP];
  for (int c = 0; c < MAX_COMP; ++c) {
    cs_src[c] = source.csrc[c];
    ct_src[c] = source.ctime[c];
  }
  if (n_comp_new < n_comp) {
    sample_without_replacement(fin, n_comp_new, n_comp, sample);
    for (int c = 0; c < n_comp_new; ++c) {
      source.csrc[c] = cs_src[sample[c] - 1];
      source.ctime[c] = ct_src[sample[c] - 1];
    }
    source.ncomp = n_comp_new;
  } else if (n_comp < MAX_COMP) {
    int i_comp = 1;
    while (i_comp <= n_comp_new) {
      if (i_comp + n_comp <= n_comp_new) {
        for (int c = 1; c <= n_comp; ++c) {
          source.csrc[i_comp + c - 2] = cs_src[c - 1];
          source.ctime[i_comp + c - 2] = ct_src[c - 1];
        }
        i_comp += n_comp;
      } else {
        int sample_size = n_comp_new - i_comp + 1;
        sample_without_replacement(fin, sample_size, n_comp, sample);
        for (int c = 1; c <= sample_size; ++c) {
          source.csrc[i_comp + c - 2] = cs_src[sample[c - 1] - 1];
          source.ctime[i_comp + c - 2] = ct_src[sample[c - 1] - 1];
        }
        i_comp = n_comp_new + 1;
      }
    }
    source.ncomp = n_comp_new;
  }
  if (source.nprim < source.ncomp) return 808144130;
  *n_coag_out = n_coag;
  return 0;
}

// One target of an accelerated pair: the body of try_per_particle_coag's
// target loop (src/coagulation.F90:216-237) as the event at sequence index
// t of pair k (record rec).  A pair's events are laid out as the reference
// loops over its target list at the pair's start: the list's arrivals of
// the step first, the latest first (they were appended last), then its
// step-start members from the last entry down.  Each visit of a target to
// a pair is its own event, so a visit sees the sources as the events
// before the pair left them, and a target that merged at an earlier pair
// is read as that pair's event left it.  Returns 1 when the event has an
// effect (record rec and the pool filled; the removed sources are claimed
// with index t when `claim`), 0 when it has none (*tns = its samples +
// ACC_WARN, or TNS_ATHIN for an arrival entry with no arrival yet), -1 on
// a box error.  *p_out is the target's slot, or -1 when there is none.
template <int NS>
__device__ __noinline__ int acc_visit(BoxDesc *boxes, int64_t k, uint32_t t, int rec, int type,
                                      uint64_t seed, uint32_t step, double del_t, bool claim,
                                      int *p_out, int *tns) {
  const Arrays &A = s_ctx.A;
  const PW &W = s_ctx.W;
  *p_out = -1;
  *tns = 0;
  int64_t q;
  const int box = pair_box(W, k, &q);
  BoxDesc *B = &boxes[box];
  if (B->error) return -1;
  const int nb = B->n_bin, nc = B->w.n_class;
  const int64_t lb = (int64_t)box * W.K_stride;
  const double *edges = A.edges + (int64_t)box * (A.max_bin + 1);
  int c1, c2, b1, b2;
  decode_pair(q, W.tab_classes, W.max_bin, &c1, &c2, &b1, &b2);
  const int kind = W.pair_acc[k];
  const int bt = kind == 1 ? b1 : b2, ct = kind == 1 ? c1 : c2;
  const int bs = kind == 1 ? b2 : b1, cs = kind == 1 ? c2 : c1;
  const int kt = par_key(bt, ct, nb), ks = par_key(bs, cs, nb);
  const uint32_t tau = W.pair_exc[k];
  const int j = (int)(t - tau);
  const int acap_t = W.acap[lb + kt];
  int p;
  if (j < acap_t) {
    const int64_t e = arrival_rank(W, lb + kt, acap_t - j, tau);
    if (e < 0 || W.ap_dep[e] < tau) {
      *tns = TNS_ATHIN;  // an earlier event not yet settled may still fill it
      return 0;
    }
    p = W.ap_p[e];
  } else {
    const int m = W.lcnt[lb + kt] - (j - acap_t);
    p = W.perm[B->off + W.lstart[lb + kt] + m - 1];
  }
  if (!drawable(W, p, kt)) return 0;  // left the list before the pair
  *p_out = p;
  // the record's chains start empty, so an attempt cut short by an error
  // leaves nothing to walk
  EventRec &ev = W.ev[rec];
  ev.nrd = 0;
  ev.rdhead = -1;
  ev.nchain = 0;
  ev.nrm = 0;
  ev.head = -1;
  const int ns = A.n_spec;
  const Weights &w = B->w;
  const uint32_t ordinal = (uint32_t)j + 1;
  const int64_t ti = table_index(A, box, nb, nc, b1, b2, c1, c2);
  const double k_max = A.kw[ti];
  const int cc = A.cc[ti];
  const int n_s = W.lcnt[lb + ks];
  const uint32_t site = pair_site(nb, nc, b1, b2, c1, c2);
  Stream aps, smp, fin;
  aps.open(seed, box, step, site, ordinal, RNG_ACC_POISSON);
  smp.open(seed, box, step, site, ordinal, RNG_ACC_SAMPLE);
  fin.open(seed, box, step, site, ordinal, RNG_ACC_FINISH);
  RecN<NS> target, source;
  load_rec(A, p, target);
  RmChain chain{-1, -1, RM_CHUNK, 0, 0ull};
  RmChain reads{-1, -1, RM_CHUNK, 0, 0ull};
  int n_samp = 0, n_coag = 0, warn = 0, flags = 0, err_code = 0;
  int err = acc_sample_source(A, W, B, type, target, ct, cs, nc_at_radius(w, cs, edges[bs - 1]),
                              B->off + W.lstart[lb + ks], ks, n_s, k_max * del_t * (double)n_s,
                              1.0 / k_max, aps, smp, fin, tau, t, claim, chain, reads, &n_samp,
                              &n_coag, &warn, source);
  if (err) {
    atomicExch(&B->error, err);
    return -1;
  }
  const int n_rm = chain.n;
  int n_dup = 0, dup_head = -1, dup_tail = -1;
  RecN<NS> np = target;
  if (n_coag > 0) {
    // coag_target_with_source (src/coagulation.F90:522-582)
    Stream ft;
    ft.open(seed, box, step, site, ordinal, RNG_ACC_TARGET);
    const double old_nc = nc_at_radius(w, target.klass, vol2rad(rec_vol(ns, target)));
    err = par_rec_coagulate(ns, ft, target, source, np);
    if (err) {
      atomicExch(&B->error, err);
      return -1;
    }
    np.id = target.id;
    const double r_new = vol2rad(rec_vol(ns, np));
    np.group = rand_group_w(ft, w, cc, r_new);
    np.klass = cc;
    flags |= RF_MERGED;
    const int new_bin = bin_find_log(nb, B->log_lo, B->log_hi, r_new);
    if (new_bin < 1 || new_bin > nb) {
      err_code = 765620746;
    } else {
      // aero_state_dup_particle (src/aero_state.F90:488-539): the copies
      // join the list of the target's new bin
      const int n_copies = prob_round(ft, old_nc / nc_at_radius(w, np.klass, r_new));
      if (n_copies == 0) flags |= RF_DIED;
      for (int c = 1; c < n_copies; ++c) {
        const int d = W.acc_cap + atomicAdd(W.dup_top, 1);
        if (d >= W.pool_cap) {
          atomicExch(&B->error, ERR_CAPACITY);
          return -1;
        }
        RecN<NS> cp = np;
        cp.group = rand_group_w(ft, w, np.klass, r_new);
        pool_store(W, ns, d, cp);
        W.q[d].next = -1;
        if (dup_tail >= 0) W.q[dup_tail].next = d;
        else dup_head = d;
        dup_tail = d;
        n_dup++;
      }
    }
  }
  if (warn) flags |= RF_WARN;
  W.ev[rec].rdhead = reads.head;
  W.ev[rec].nrd = reads.n;
  if (n_coag == 0 && n_rm == 0 && err_code == 0) {
    *tns = n_samp | (warn ? ACC_WARN : 0);
    return 0;
  }
  if (flags & RF_MERGED) pool_store(W, ns, rec, np);
  W.ev[rec].nsamp = n_samp;
  W.ev[rec].ncoag = n_coag;
  W.ev[rec].nrm = n_rm;
  W.ev[rec].nchain = chain.n;
  W.ev[rec].head = chain.head;
  W.ev[rec].ndup = n_dup;
  W.ev[rec].dhead = dup_head;
  W.ev[rec].flags = flags;
  W.ev[rec].err = err_code;
  if (claim) claim_write(W, p, t);
  return 1;
}

__device__ inline int run_visit(BoxDesc *boxes, const Arrays &A, int64_t k, uint32_t t, int rec,
                                int type, uint64_t seed, uint32_t step, double del_t, bool claim,
                                int *p_out, int *tns) {
  return A.n_spec <= FEW_SPEC
             ? acc_visit<FEW_SPEC>(boxes, k, t, rec, type, seed, step, del_t, claim, p_out, tns)
             : acc_visit<MAX_SPEC>(boxes, k, t, rec, type, seed, step, del_t, claim, p_out, tns);
}

// visits per wavefront: each is one lane's serial sample loop, and fewer a
// wavefront spread the first round's visits over more compute units
constexpr int ACC_LANES = 16;
// Round 0 runs one thread per target slot of the batch (record a maps to
// its slot through acc_exc); later rounds run over the pending slots.
__device__ inline void acc_test(BoxDesc *boxes, const Arrays &A, const PW &W, int n_box, int type,
                                uint64_t seed, uint32_t step, uint32_t t0, const uint32_t *pend,
                                double del_t, uint32_t acc_base, int idx) {
  const int64_t NP = (int64_t)n_box * W.P_stride;
  uint32_t t;
  int i;
  int64_t k;
  if (pend) {
    i = idx;
    t = pend[i];
    k = test_pair(W, NP, t);
    if (!W.pair_acc[k]) return;
  } else {
    const uint32_t a = acc_base + (uint32_t)idx;
    k = find_pair(W.acc_exc, NP, a);
    t = W.pair_exc[k] + (a - W.acc_exc[k]);
    i = (int)(t - t0);
  }
  const int rec = (int)(W.acc_exc[k] + (t - W.pair_exc[k]) - acc_base);
  W.acc[i] = 0;
  W.tid[i] = t;
  W.tp2[i] = -1;
  W.trec[i] = rec;
  int p, tns;
  const int r = run_visit(boxes, A, k, t, rec, type, seed, step, del_t, true, &p, &tns);
  W.tp1[i] = p;
  W.tns[i] = tns;
  if (r == 1) W.acc[i] = 1;
  // the visit's samples, for the algorithmic traffic of this kernel
  const int ns = (r == 1) ? W.ev[rec].nsamp : (tns & (TNS_SIDE2 - 1));
  if (ns > 0) atomicAdd(W.acc_samp, (unsigned long long)ns);
}

__global__ void __launch_bounds__(64)
k_par_acc_tests(BoxDesc *boxes, Arrays A, PW W, int n_box, int type, uint64_t seed,
                uint32_t step, uint32_t t0, const uint32_t *pend, double del_t,
                uint32_t acc_base, int n_acc) {
  // over a pending list most slots are per-set tests that return at once:
  // every lane takes one; over the first round's target slots, ACC_LANES a
  // wavefront
  const int lanes = pend ? 64 : ACC_LANES;
  const int count = pend ? W.rc[RC_N] : n_acc;
  if ((int)blockIdx.x * lanes >= count) return;
  step_ctx_fill(A, W);
  if ((int)threadIdx.x >= lanes) return;
  for (int idx = blockIdx.x * lanes + threadIdx.x; idx < count; idx += gridDim.x * lanes)
    acc_test(boxes, A, W, n_box, type, seed, step, t0, pend, del_t, acc_base, idx);
}

// the largest batch end t1 <= min(T, t0 + T_cap) whose target slots fit the
// records; out[0] = t1, out[1] = acc_count(t0), out[2] = acc_count(t1),
// out[3] and [4] the step's tests and target slots, out[5] 0, or why there is
// nothing else: BE_REGRID (a box got a new grid), BE_TESTS (the step's tests
// are more than their 32-bit indices; the boxes' own 64-bit counts tell)
constexpr uint32_t BE_REGRID = 1, BE_TESTS = 2;
__device__ inline uint32_t acc_count(const PW &W, int64_t NP, uint32_t T, uint32_t t) {
  if (t >= T) return W.acc_exc[NP];
  int64_t k = test_pair(W, NP, t);
  return W.acc_exc[k] + (W.pair_acc[k] ? t - W.pair_exc[k] : 0u);
}

__global__ void __launch_bounds__(64)
k_batch_end(const BoxDesc *boxes, PW W, int n_box, int64_t NP, uint32_t t0, uint32_t t_cap,
            uint32_t a_cap, uint32_t *out) {
  const bool regrid = W.rc[RC_REGRID] == W.tag;
  long long tests = 0;
  if (t0 == 0)  // the first batch's: step_samp holds this step's draws
    for (int b = threadIdx.x; b < n_box; b += 64) tests += boxes[b].step_samp;
  for (int o = 32; o > 0; o >>= 1) tests += __shfl_xor(tests, o);
  if (threadIdx.x != 0) return;
  tests += W.acc_exc[NP];
  out[5] = regrid ? BE_REGRID : tests > (long long)UINT32_MAX ? BE_TESTS : 0u;
  if (out[5]) return;
  const uint32_t T = W.pair_exc[NP];
  const uint32_t a0 = acc_count(W, NP, T, t0);
  uint32_t lo = t0 + 1, hi = (T - t0 < t_cap) ? T : t0 + t_cap;
  if (acc_count(W, NP, T, hi) - a0 <= a_cap) lo = hi;  // the usual case: all of it fits
  while (lo < hi) {  // largest t1 in [lo, hi] with acc_count(t1) - a0 <= a_cap
    uint32_t mid = lo + (hi - lo + 1) / 2;
    if (acc_count(W, NP, T, mid) - a0 <= a_cap) lo = mid; else hi = mid - 1;
  }
  out[0] = lo;
  out[1] = a0;
  out[2] = acc_count(W, NP, T, lo);
  out[3] = T;
  out[4] = W.acc_exc[NP];
}

// compact accepted tests into the event list (in test order), as the scan of
// their flags places them
struct GatherEvents {
  PW W;
  __device__ void operator()(int64_t i, uint32_t acc, uint32_t e) const {
    if (!acc) return;
    W.ev_t[e] = W.tid[i];
    W.ev_p1[e] = W.tp1[i];
    W.ev_p2[e] = W.tp2[i];
    W.ev_rec[e] = W.trec[i];
  }
};

__device__ inline void resolve_event(BoxDesc *boxes, const Arrays &A, const PW &W, int n_box,
                                     uint64_t seed, uint32_t step, int e) {
  uint32_t t = W.ev_t[e];
  int p1 = W.ev_p1[e], p2 = W.ev_p2[e];
  MergeCtx m = merge_ctx(boxes, W, n_box, t);
  W.ev_box[e] = m.box;
  // the first event of its box (events are in test order, so box-major)
  if (e == 0) {
    W.box_first[m.box] = 0;
  } else {
    int64_t q;
    if (pair_box(W, test_pair(W, (int64_t)n_box * W.P_stride, W.ev_t[e - 1]), &q) != m.box)
      W.box_first[m.box] = e;
  }
  const int r = W.ev_rec[e];
  if (r >= 0) {
    // a target event wins when it holds the target and every removed source
    // ... and no earlier event claimed a source it read
    bool win = W.slot[p1].claim == t;
    rm_walk(W, r, [&](int q) { win = win && W.slot[q].claim == t; });
    rd_walk(W, r, [&](int q) { win = win && W.slot[q].claim_wr >= t; });
    const int died = (W.ev[r].flags & RF_DIED) ? 1 : 0;
    W.ev_out[e] = win ? O_WIN : 0;
    W.f_app[e] = win ? W.ev[r].ndup : 0;
    W.f_id[e] = win ? W.ev[r].ndup : 0;
    W.f_info[e] = win ? W.ev[r].nrm + died : 0;
    W.f_hole[e] = win ? W.ev[r].nrm + died : 0;
    return;
  }
  // the decisions say which parents the merge changes (removes); a parent
  // it keeps is only read
  BoxDesc *B = &boxes[m.box];
  const int nb = B->n_bin, nc = B->w.n_class;
  int cc = A.cc[table_index(A, m.box, nb, nc, m.b1, m.b2, m.c1, m.c2)];
  Stream s;
  s.open(seed, m.box, step, pair_site(nb, nc, m.b1, m.b2, m.c1, m.c2), m.j, RNG_MERGE);
  int g;
  const int d = merge_decide(A, W, B, s, p1, p2, m.c1, m.c2, cc, &g, B->w);
  const bool win = ((d & O_RM1) ? W.slot[p1].claim == t : W.slot[p1].claim_wr > t) &&
                   ((d & O_RM2) ? W.slot[p2].claim == t : W.slot[p2].claim_wr > t);
  int o = 0;
  if (win) o = d | O_WIN | (g << 16) | (cc << 24);
  W.ev_out[e] = o;
  W.f_app[e] = (o & O_APPEND) ? 1 : 0;
  W.f_id[e] = (o & O_NEWID) ? 1 : 0;
  W.f_info[e] = ((o & O_INFO1) ? 1 : 0) + ((o & O_INFO2) ? 1 : 0);
  W.f_hole[e] = ((o & O_RM1) && !(o & O_SLOT1) ? 1 : 0) + ((o & O_RM2) && !(o & O_SLOT2) ? 1 : 0);
}

__global__ void k_par_resolve(BoxDesc *boxes, Arrays A, PW W, int n_box, uint64_t seed,
                              uint32_t step) {
  const int E = W.rc[RC_E];
  PAR_FOR(e, E) resolve_event(boxes, A, W, n_box, seed, step, e);
}

// A particle's components, all MAX_COMP of them in wide loads that go out
// together (a particle's 80 and 160 bytes are 16-byte aligned).  A load under
// `if (c < n)` becomes a branch, and the compiler waits for every load in
// flight at each one, one memory round trip per component.
__device__ inline void load_comps(const int *csrc, const double *ctime, int64_t p, int *s,
                                  double *t) {
  static_assert(MAX_COMP % 4 == 0, "whole 16-byte words");
  const int4 *ps = (const int4 *)(csrc + comp_at(p, 0));
  const double2 *pt = (const double2 *)(ctime + comp_at(p, 0));
#pragma unroll
  for (int c = 0; c < MAX_COMP / 4; ++c) {
    const int4 x = ps[c];
    s[4 * c] = x.x;
    s[4 * c + 1] = x.y;
    s[4 * c + 2] = x.z;
    s[4 * c + 3] = x.w;
  }
#pragma unroll
  for (int c = 0; c < MAX_COMP / 2; ++c) {
    const double2 x = pt[c];
    t[2 * c] = x.x;
    t[2 * c + 1] = x.y;
  }
}
__device__ inline void load_comps(const Arrays &A, int64_t p, int *s, double *t) {
  load_comps(A.csrc, A.ctime, p, s, t);
}

// Pool entry i written as the particle of class klass and identifier id in a
// slot: its old particle leaves its list at t_leave, the new one joins at
// t_join.  The slot's bookkeeping and the entry are read together.
__device__ inline void write_new_particle(const Arrays &A, const PW &W, BoxDesc *B, int box,
                                          uint32_t t_leave, uint32_t t_join, int64_t slot,
                                          bool appended, int i, int klass, int64_t id, int nb,
                                          int type, int want_terms, const SlotView &sv) {
  const PoolRec q = W.q[i];
  int cs[MAX_COMP];
  double ct[MAX_COMP];
  load_comps(W.q_csrc, W.q_ctime, i, cs, ct);
  double v = 0.0;
  double m = 0.0;
  const int ns = A.n_spec;
  for (int s0 = 0; s0 < ns; s0 += SPEC_CHUNK) {
    double x[SPEC_CHUNK], rho[SPEC_CHUNK];
#pragma unroll
    for (int u = 0; u < SPEC_CHUNK; ++u) {
      const int s = s0 + u < ns ? s0 + u : ns - 1;
      x[u] = W.q_vol[(int64_t)i * ns + s];
      rho[u] = A.density[s];
    }
#pragma unroll
    for (int u = 0; u < SPEC_CHUNK; ++u)
      if (s0 + u < ns) {
        A.vol[(int64_t)(s0 + u) * A.total_cap + slot] = x[u];
        v += x[u];
        m += x[u] * rho[u];
      }
  }
  A.vtot[slot] = v;
  A.id[slot] = id;
  A.group[slot] = q.group;
  A.klass[slot] = klass;
  A.nprim[slot] = q.nprim;
  A.ncomp[slot] = q.ncomp;
#pragma unroll
  for (int c = 0; c < MAX_COMP; ++c)
    if (c < q.ncomp) {
      A.csrc[comp_at(slot, c)] = cs[c];
      A.ctime[comp_at(slot, c)] = ct[c];
    }
  A.least[slot] = q.least;
  A.greatest[slot] = q.greatest;
  int b = bin_find_log(nb, B->log_lo, B->log_hi, vol2rad(v));
  if (b < 1 || b > nb) {
    atomicExch(&B->error, 134572570);
    st_set(W, slot, ST_NEW);
    W.key[slot] = 0;
    return;
  }
  int k = par_key(b, klass, nb);
  if (appended) slot_append(W, B, box, slot, t_join, k);
  else slot_write(W, B, box, slot, t_leave, t_join, k, sv);
  st_set(W, slot, ST_NEW);
  W.key[slot] = k;
  if (want_terms) W.terms[slot] = particle_terms(type, v, m / v, B->env);
}

// Where a merge puts what it creates.  In a claim round the positions come
// from the round's scans over the events (RankAlloc, one per event); in the
// sequential tail they come straight from the box's counters (SeqAlloc).
struct RankAlloc {
  BoxDesc *B;
  int64_t app, id, info, hole;  // this event's next ranks
  int *live;                    // the box's live counts per list key
  __device__ int64_t append_slot() {
    int64_t r = app++;
    return B->n_part + r < B->cap ? B->off + B->n_part + r : -1;
  }
  __device__ int64_t new_id() {
    return (B->next_id + id++ - 1) * B->id_stride + B->id_offset + 1;
  }
  __device__ int64_t info_index() { return B->n_info + info++; }
  __device__ int64_t hole_index() { return hole++; }
  __device__ void live_add(int key, int d) { atomicAdd(&live[key], d); }
  __device__ void count(int64_t samp, int64_t coag, int warn) {
    if (samp) {
      atomicAdd((unsigned long long *)&B->n_samp, (unsigned long long)samp);
      atomicAdd((unsigned long long *)&B->step_samp, (unsigned long long)samp);
    }
    if (coag) {
      atomicAdd((unsigned long long *)&B->n_coag, (unsigned long long)coag);
      atomicAdd((unsigned long long *)&B->step_coag, (unsigned long long)coag);
    }
    if (warn) atomicAdd((unsigned long long *)&B->n_warn, (unsigned long long)warn);
  }
};

// The round's allocator: counters kept in the lane and summed over the
// wavefront per box before they reach the box (thousands of winners of one
// box would otherwise serialise on the same counter words)
struct ApplyAlloc : RankAlloc {
  int64_t n_samp, n_coag, n_warn;
  int lk[3], ld[3], nl;  // the first live-count changes, summed per wavefront later
  __device__ void count(int64_t samp, int64_t coag, int warn) {
    n_samp += samp;
    n_coag += coag;
    n_warn += warn;
  }
  __device__ void live_add(int key, int d) {
    if (nl < 3) {
      lk[nl] = key;
      ld[nl] = d;
      ++nl;
    } else {
      atomicAdd(&live[key], d);
    }
  }
};

// Sum live-count changes over the wavefront per (list, key) and add each
// sum once; key < 0: nothing from this lane.  Every lane takes part.
__device__ inline void wave_flush_live(int *live, int key, int d) {
  const int lane = threadIdx.x & 63;
  const uint64_t addr = key >= 0 ? (uint64_t)(live + key) : 0ull;
  uint64_t pending = __ballot(key >= 0 && d != 0);
  while (pending) {
    const int leader = __ffsll((long long)pending) - 1;
    const uint64_t la = __shfl(addr, leader);
    const bool mine = ((pending >> lane) & 1ull) && addr == la;
    int td = mine ? d : 0;
    for (int off = 32; off > 0; off >>= 1) td += __shfl_xor(td, off);
    if (lane == leader && td) atomicAdd((int *)la, td);
    pending &= ~__ballot(mine);
  }
}

// Sum each box's counter changes over the wavefront and add them with one
// set of atomics per box (box < 0: nothing from this lane).  Every lane of
// the wavefront takes part.
__device__ inline void wave_flush_counts(BoxDesc *boxes, int box, int64_t s, int64_t c,
                                         int64_t w) {
  const int lane = threadIdx.x & 63;
  uint64_t pending = __ballot(box >= 0 && (s | c | w));
  while (pending) {
    const int leader = __ffsll((long long)pending) - 1;
    const int lb = __shfl(box, leader);
    const bool mine = ((pending >> lane) & 1ull) && box == lb;
    long long ts = mine ? s : 0, tc = mine ? c : 0, tw = mine ? w : 0;
    for (int off = 32; off > 0; off >>= 1) {
      ts += __shfl_xor(ts, off);
      tc += __shfl_xor(tc, off);
      tw += __shfl_xor(tw, off);
    }
    if (lane == leader) {
      BoxDesc *B = &boxes[lb];
      if (ts) {
        atomicAdd((unsigned long long *)&B->n_samp, (unsigned long long)ts);
        atomicAdd((unsigned long long *)&B->step_samp, (unsigned long long)ts);
      }
      if (tc) {
        atomicAdd((unsigned long long *)&B->n_coag, (unsigned long long)tc);
        atomicAdd((unsigned long long *)&B->step_coag, (unsigned long long)tc);
      }
      if (tw) atomicAdd((unsigned long long *)&B->n_warn, (unsigned long long)tw);
    }
    pending &= ~__ballot(mine);
  }
}

// The tail's allocator: ranks as in a round, live-count changes gathered
// in the workgroup's shared memory and counters in the lane, both flushed
// once (many winners of one box would otherwise contend on the same words)
struct TailAlloc : RankAlloc {
  int *s_live;
  int64_t n_samp, n_coag, n_warn;
  __device__ void live_add(int key, int d) { atomicAdd(&s_live[key], d); }
  __device__ void count(int64_t samp, int64_t coag, int warn) {
    n_samp += samp;
    n_coag += coag;
    n_warn += warn;
  }
};

template <class Alloc>
__device__ inline void put_info(const Arrays &A, BoxDesc *B, Alloc &al, int64_t id, int action,
                                int64_t other) {
  int64_t k = al.info_index();
  if (k < B->info_cap) {
    A.info_id[B->info_off + k] = id;
    A.info_action[B->info_off + k] = action;
    A.info_other[B->info_off + k] = other;
  }
}

// Which components the merged particle keeps when the parents hold more than
// MAX_COMP together (aero_particle_coagulate, src/aero_particle.F90:
// 917-1033): prob_round of the first parent's share, then two selection
// samples (sample_without_replacement keeps sorted order).  take: a bit per
// component of each parent; returns the first parent's share.
template <class S>
__device__ inline int resample_masks(S &s, int n1, int n2, int np1, int np2, uint32_t *take1,
                                     uint32_t *take2) {
  const int n1_new = prob_round(s, (double)np1 / (double)(np1 + np2) * (double)MAX_COMP);
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    const int n = side ? n2 : n1, want = side ? MAX_COMP - n1_new : n1_new;
    uint32_t take = 0;
    int m = 0;
    for (int c = 0; c < n && m < want; ++c) {
      const double r = s.uniform();
      if (!((double)(n - c) * r >= (double)(want - m))) {
        take |= 1u << c;
        m++;
      }
    }
    (side ? *take2 : *take1) = take;
  }
  return n1_new;
}

__device__ inline void resample_components(const Arrays &A, Stream &s, int64_t p1, int64_t p2,
                                           int64_t dst, int n1, int n2, int np1, int np2) {
  int s1[MAX_COMP], s2[MAX_COMP];
  double t1[MAX_COMP], t2[MAX_COMP];
  load_comps(A, p1, s1, t1);
  load_comps(A, p2, s2, t2);
  uint32_t take1, take2;
  const int n1_new = resample_masks(s, n1, n2, np1, np2, &take1, &take2);
  int m1 = 0, m2 = n1_new;
#pragma unroll
  for (int c = 0; c < MAX_COMP; ++c) {
    if ((take1 >> c) & 1u) {
      A.csrc[comp_at(dst, m1)] = s1[c];
      A.ctime[comp_at(dst, m1)] = t1[c];
      ++m1;
    }
  }
#pragma unroll
  for (int c = 0; c < MAX_COMP; ++c) {
    if ((take2 >> c) & 1u) {
      A.csrc[comp_at(dst, m2)] = s2[c];
      A.ctime[comp_at(dst, m2)] = t2[c];
      ++m2;
    }
  }
}

// Every lane's loads before any lane's stores after it.  The fence keeps the
// compiler from moving either across; the barrier is convergent, so branches
// before and after it on one condition stay two branches and no lane runs
// ahead to its stores.  Neither is an instruction.
__device__ inline void wave_handoff() {
  wave_fence();
  __builtin_amdgcn_wave_barrier();
}

// One lane's resampling by its whole wavefront: about 40 uniforms of one
// stream are 20 Philox blocks, one a lane, and the components go through the
// lanes.  Every lane takes part; the arguments are the resampling lane's,
// broadcast.  i0: the stream's next uniform.  A drizzle drop's merge spends
// 13 us on this alone on one lane, about 4 here.
struct LaneUniforms {
  double a, b;  // this lane's block
  int at;
  __device__ inline double uniform() {
    const double v = __shfl((at & 1) ? b : a, at >> 1);
    ++at;
    return v;
  }
};
__device__ inline void wave_resample(const Arrays &A, const Stream &s, int i0, int64_t p1,
                                     int64_t p2, int64_t dst, int n1, int n2, int np1, int np2) {
  const int lane = threadIdx.x & 63;
  int s1 = 0, s2 = 0;
  double t1 = 0.0, t2 = 0.0;
  if (lane < MAX_COMP) {
    s1 = A.csrc[comp_at(p1, lane)];
    t1 = A.ctime[comp_at(p1, lane)];
    s2 = A.csrc[comp_at(p2, lane)];
    t2 = A.ctime[comp_at(p2, lane)];
  }
  uint32_t o[4];
  s.philox_block((uint32_t)(i0 >> 1) + lane, o);
  LaneUniforms u{u52(o[0], o[1]), u52(o[2], o[3]), i0 & 1};
  uint32_t take1, take2;
  const int n1_new = resample_masks(u, n1, n2, np1, np2, &take1, &take2);
  const uint32_t below = lane < 32 ? (1u << lane) - 1u : 0u;
  wave_handoff();  // dst may be a parent's slot
  if (lane < MAX_COMP) {
    if ((take1 >> lane) & 1u) {
      const int c = __popc(take1 & below);
      A.csrc[comp_at(dst, c)] = s1;
      A.ctime[comp_at(dst, c)] = t1;
    }
    if ((take2 >> lane) & 1u) {
      const int c = n1_new + __popc(take2 & below);
      A.csrc[comp_at(dst, c)] = s2;
      A.ctime[comp_at(dst, c)] = t2;
    }
  }
}

// What a merge reads of its parents, loaded together before anything is
// written: one memory round trip where reading each field as it is needed,
// between the stores, costs one apiece (in the tail of 3e5-drop boxes 1.2 us
// left of 6.3, the rest behind the claims' barrier).  With the first
// species' volumes among them and the components loaded ahead of the sums,
// 20 steps of six such boxes take 43.1 ms in place of 53.8.
struct MergeParents {
  SlotView v1, v2;
  int64_t id1, id2;
  int n1, n2, np1, np2;
  double least1, least2, greatest1, greatest2;
  double x1[SPEC_CHUNK], x2[SPEC_CHUNK];  // the first species' volumes
};
__device__ inline MergeParents load_parents(const Arrays &A, const PW &W, int64_t p1, int64_t p2) {
  MergeParents P;
  P.v1 = slot_load(W, p1);
  P.v2 = slot_load(W, p2);
  P.id1 = A.id[p1];
  P.id2 = A.id[p2];
  P.n1 = A.ncomp[p1];
  P.n2 = A.ncomp[p2];
  P.np1 = A.nprim[p1];
  P.np2 = A.nprim[p2];
  P.least1 = A.least[p1];
  P.least2 = A.least[p2];
  P.greatest1 = A.greatest[p1];
  P.greatest2 = A.greatest[p2];
#pragma unroll
  for (int u = 0; u < SPEC_CHUNK; ++u) {
    const int64_t row = (int64_t)min(u, A.n_spec - 1) * A.total_cap;
    P.x1[u] = A.vol[row + p1];
    P.x2[u] = A.vol[row + p2];
  }
  return P;
}

// the merged particle of an accepted per-set test written straight from
// its parents' slots into dst (which may be either parent's slot):
// aero_particle_coagulate (src/aero_particle.F90:917-1033).  Components
// are concatenated, or resampled on `rs` (the merge stream after the merge
// decisions) when the parents hold more than MAX_COMP together, unless the
// wavefront has done so already.
__device__ inline int direct_merge(const Arrays &A, const PW &W, BoxDesc *B, int box, uint32_t t,
                                   int64_t p1, int64_t p2, int64_t dst, bool appended, int64_t id,
                                   int group, int klass, int type, int want_terms, Stream *rs,
                                   const MergeParents &P, bool in_place, int *key) {
  const int64_t tc = A.total_cap;
  const int n1 = P.n1, n2 = P.n2;
  *key = 0;
  if (P.np1 < n1) return 465791384;
  if (P.np2 < n2) return 465791385;
  // components: the first parent's, then the second's, all loaded before
  // any is written, and on their way while the volumes are added and the bin
  // is found; the first parent's are in place when it is the slot
  const bool all = n1 + n2 <= MAX_COMP;
  int s1[MAX_COMP], s2[MAX_COMP];
  double t1[MAX_COMP], t2[MAX_COMP];
  if (all && !in_place) {
    load_comps(A, p2, s2, t2);
    if (dst != p1) load_comps(A, p1, s1, t1);
  }
  // dst may be a parent's slot: each species' sum depends only on its own
  // row, so it is written once formed; a chunk's loads go out together
  double v = 0.0, m = 0.0;
  const int ns = A.n_spec;
#pragma unroll
  for (int u = 0; u < SPEC_CHUNK; ++u) {
    if (u < ns) {
      const double x = P.x1[u] + P.x2[u];
      A.vol[(int64_t)u * tc + dst] = x;
      v += x;
      m += x * A.density[u];
    }
  }
  for (int s0 = SPEC_CHUNK; s0 < ns; s0 += SPEC_CHUNK) {
    double x[SPEC_CHUNK], rho[SPEC_CHUNK];
#pragma unroll
    for (int u = 0; u < SPEC_CHUNK; ++u) {
      const int s = s0 + u < ns ? s0 + u : ns - 1;
      x[u] = A.vol[(int64_t)s * tc + p1] + A.vol[(int64_t)s * tc + p2];
      rho[u] = A.density[s];
    }
#pragma unroll
    for (int u = 0; u < SPEC_CHUNK; ++u) {
      if (s0 + u < ns) {
        A.vol[(int64_t)(s0 + u) * tc + dst] = x[u];
        v += x[u];
        m += x[u] * rho[u];
      }
    }
  }
  const int nb = B->n_bin;
  const int b = bin_find_log(nb, B->log_lo, B->log_hi, vol2rad(v));
  if (in_place) {
    // the components are in place
  } else if (all) {
    if (dst != p1) {
#pragma unroll
      for (int c = 0; c < MAX_COMP; ++c)
        if (c < n1) {
          A.csrc[comp_at(dst, c)] = s1[c];
          A.ctime[comp_at(dst, c)] = t1[c];
        }
    }
#pragma unroll
    for (int c = 0; c < MAX_COMP; ++c)
      if (c < n2) {
        A.csrc[comp_at(dst, n1 + c)] = s2[c];
        A.ctime[comp_at(dst, n1 + c)] = t2[c];
      }
  } else {
    resample_components(A, *rs, p1, p2, dst, n1, n2, P.np1, P.np2);
  }
  A.vtot[dst] = v;
  A.id[dst] = id;
  A.group[dst] = group;
  A.klass[dst] = klass;
  A.nprim[dst] = P.np1 + P.np2;
  A.ncomp[dst] = all ? n1 + n2 : MAX_COMP;
  A.least[dst] = fmin(P.least1, P.least2);
  A.greatest[dst] = fmax(P.greatest1, P.greatest2);
  if (b < 1 || b > nb) {
    st_set(W, dst, ST_NEW);
    W.key[dst] = 0;
    return 134572570;
  }
  const int k_new = par_key(b, klass, nb);
  if (appended) slot_append(W, B, box, dst, t, k_new);
  else slot_write(W, B, box, dst, t, t, k_new, dst == p1 ? P.v1 : P.v2);
  st_set(W, dst, ST_NEW);
  W.key[dst] = k_new;
  *key = k_new;
  if (want_terms) W.terms[dst] = particle_terms(type, v, m / v, B->env);
  return 0;
}

// coagulate_weighting + coagulate (src/coagulation.F90:810-985) of an
// accepted per-set test, o_group the decisions of merge_decide with the new
// particle's group and class from bits 16 and 24 on: removals become
// holes (or the slot the merged particle takes), the merged particle is
// written, removal records follow the reference's order.  post: the merge
// stream after the decisions, or null to find it again.  in_place: the
// merged particle's components are in its slot already.
template <class Alloc>
__device__ inline void perset_merge(BoxDesc *B, const Arrays &A, const PW &W, int box, int n_box,
                                    uint32_t t, int64_t p1, int64_t p2, uint64_t seed,
                                    uint32_t step, int type, int want_terms, int rid, Alloc &al,
                                    int o_group, const Stream *post, bool in_place,
                                    const MergeParents &P) {
  al.count(0, 1, 0);
  const int cc = o_group >> 24;
  const int o = o_group & 0xFFFF;
  int new_group = (o_group >> 16) & 0xFF;
  Stream s;
  if (post) {
    s = *post;
  } else if (P.n1 + P.n2 > MAX_COMP && !in_place) {
    const int64_t k = test_pair(W, (int64_t)n_box * W.P_stride, t);
    int c1, c2, b1, b2;
    decode_pair(k - (int64_t)box * W.P_stride, W.tab_classes, W.max_bin, &c1, &c2, &b1, &b2);
    s.open(seed, box, step, pair_site(B->n_bin, B->w.n_class, b1, b2, c1, c2), t - W.pair_exc[k],
           RNG_MERGE);
    (void)merge_decide(A, W, B, s, p1, p2, c1, c2, cc, &new_group, B->w);
  }
  int64_t info_other = 0;
  int64_t slot = -1;
  int key = 0;  // the merged particle's list
  if (o & O_NEW) {
    const int64_t nid = (o & O_ID1) ? P.id1 : (o & O_ID2) ? P.id2 : al.new_id();
    info_other = nid;
    if (o & O_SLOT1) slot = p1;
    else if (o & O_SLOT2) slot = p2;
    else {
      slot = al.append_slot();
      if (slot < 0) {
        atomicExch(&B->error, ERR_CAPACITY);
        return;
      }
    }
    const bool appended = !(o & (O_SLOT1 | O_SLOT2));
    const int err = direct_merge(A, W, B, box, t, p1, p2, slot, appended, nid, new_group, cc, type,
                                 want_terms, &s, P, in_place, &key);
    if (err) atomicExch(&B->error, err);
  }
  if (o & O_RM1) {
    W.slot[p1].dead_t = t;
    W.slot[p1].dead_r = rid;
    al.live_add(P.v1.key, -1);
    if (!(o & O_SLOT1)) {
      slot_leave(W, p1, t, P.v1);
      st_set(W, p1, ST_HOLE);
      W.holes[al.hole_index()] = ((uint64_t)box << 32) | (uint64_t)(p1 - B->off);
    }
  }
  if (o & O_RM2) {
    W.slot[p2].dead_t = t;
    W.slot[p2].dead_r = rid;
    al.live_add(P.v2.key, -1);
    if (!(o & O_SLOT2)) {
      slot_leave(W, p2, t, P.v2);
      st_set(W, p2, ST_HOLE);
      W.holes[al.hole_index()] = ((uint64_t)box << 32) | (uint64_t)(p2 - B->off);
    }
  }
  if (slot >= 0) al.live_add(key, 1);
  if (o & O_INFO1) put_info(A, B, al, P.id1, 2, info_other);
  if (o & O_INFO2) put_info(A, B, al, P.id2, 2, info_other);
}

// The components of a wavefront's winning per-set merges, by its lanes
// together while the merges are few.  Resamplings: each takes the wavefront
// about 2 us, where all of them side by side, a lane each, take 13.  The rest
// join their parents' components, three merges at once with a lane a
// component: one round trip, where a lane's own 40 conditional stores wait
// for its loads (six boxes of 3e5 drops 43.0 -> 41.7 ms, a scenario
// 16.7 -> 16.3); beyond JOIN_MOST, four such passes, the lanes side by side
// do as well.  win: this lane merges p1 and p2 with decisions o into an
// existing slot or the append_rank-th new one; ms: its merge stream after the
// decisions.  Returns whether this lane's components are done.  Every lane of
// the wavefront takes part.
constexpr int RESAMPLE_MOST = 6;
constexpr int JOIN_AT_ONCE = 64 / MAX_COMP, JOIN_MOST = 12;
__device__ inline bool wave_components(const Arrays &A, const BoxDesc *B, bool win, int o,
                                        int64_t p1, int64_t p2, int64_t append_rank,
                                        const Stream &ms, const MergeParents &P) {
  bool mine = false, join = false;
  int64_t dst = 0;
  int n1 = 0, n2 = 0, np1 = 0, np2 = 0;
  if (win && (o & O_NEW)) {
    n1 = P.n1;
    n2 = P.n2;
    np1 = P.np1;
    np2 = P.np2;
    bool ok = np1 >= n1 && np2 >= n2;
    if (ok) {
      if (o & O_SLOT1) dst = p1;
      else if (o & O_SLOT2) dst = p2;
      else if (B->n_part + append_rank < B->cap) dst = B->off + B->n_part + append_rank;
      else ok = false;  // the merge fails
    }
    mine = ok && n1 + n2 > MAX_COMP;
    join = ok && !mine;
  }
  // components that only join, JOIN_AT_ONCE merges in a pass of the lanes
  uint64_t cat = __ballot(join);
  if (__popcll(cat) > JOIN_MOST) {
    cat = 0;
    join = false;
  }
  const int lane = threadIdx.x & 63, slice = lane / MAX_COMP, c = lane % MAX_COMP;
  while (cat) {
    uint64_t m = cat;
    for (int q = 0; q < slice; ++q) m &= m - 1;
    const bool on = slice < JOIN_AT_ONCE && m != 0;
    const int src = on ? __ffsll((long long)m) - 1 : lane;
    const int a = __shfl((int)p1, src), b = __shfl((int)p2, src), d = __shfl((int)dst, src);
    const int na = __shfl(n1, src), nb = __shfl(n2, src);
    const bool in_a = on && c < na && d != a, in_b = on && c < nb;
    int sa = 0, sb = 0;
    double ta = 0.0, tb = 0.0;
    if (in_a) {
      sa = A.csrc[comp_at(a, c)];
      ta = A.ctime[comp_at(a, c)];
    }
    if (in_b) {
      sb = A.csrc[comp_at(b, c)];
      tb = A.ctime[comp_at(b, c)];
    }
    wave_handoff();  // d may be b: a lane's store is over another's load
    if (in_a) {
      A.csrc[comp_at(d, c)] = sa;
      A.ctime[comp_at(d, c)] = ta;
    }
    if (in_b) {
      A.csrc[comp_at(d, na + c)] = sb;
      A.ctime[comp_at(d, na + c)] = tb;
    }
    wave_handoff();
    for (int q = 0; q < JOIN_AT_ONCE; ++q) cat &= cat - 1;
  }
  uint64_t todo = __ballot(mine);
  if (__popcll(todo) > RESAMPLE_MOST) return join;
  while (todo) {
    const int src = __ffsll((long long)todo) - 1;
    todo &= todo - 1;
    Stream s;
    s.k0 = __shfl(ms.k0, src);
    s.k1 = __shfl(ms.k1, src);
    s.c0 = __shfl(ms.c0, src);
    s.c1 = __shfl(ms.c1, src);
    s.c2 = __shfl(ms.c2, src);
    s.c3 = __shfl(ms.c3, src);
    const int i0 = 2 * (int)__shfl(ms.block, src) - __shfl(ms.have, src);
    wave_resample(A, s, i0, __shfl((long long)p1, src), __shfl((long long)p2, src),
                  __shfl((long long)dst, src), __shfl(n1, src), __shfl(n2, src),
                  __shfl(np1, src), __shfl(np2, src));
  }
  return mine || join;
}

// a winning target event (coag_target_with_source and
// aero_state_dup_particle, src/coagulation.F90:522-582,
// src/aero_state.F90:488-539): removed sources become holes with a
// coagulation record naming the particle that took them (the target or one
// of its copies), the merged target replaces the old one in place, copies
// are appended with new identifiers in creation order, and a target or
// copy that kept no copy of itself is removed with a weighting record.
template <class Alloc>
__device__ __noinline__ void acc_apply(BoxDesc *B, int box, uint32_t t, int r, int64_t p, int type,
                                       int want_terms, int rid, Alloc &al,
                                       bool chain_elsewhere = false) {
  const Arrays &A = s_ctx.A;
  const PW &W = s_ctx.W;
  const int nb = B->n_bin;
  const int64_t target_id = A.id[p];
  const int klass = A.klass[p];
  const EventRec ev = W.ev[r];
  const int flags = ev.flags;
  // copy identifiers in creation order, drawn before any record names them
  int64_t id_first = 0;
  for (int kk = 0; kk < ev.ndup; ++kk) {
    int64_t v = al.new_id();
    if (kk == 0) id_first = v;
  }
  auto copy_id = [&](int kk) { return id_first + (int64_t)(kk - 1) * B->id_stride; };
  if (chain_elsewhere) {
    // the removed sources are applied by a wavefront (k_par_apply_chains)
    // at this event's first hole and record ranks
    al.hole += ev.nrm;
    al.info += ev.nrm;
  } else {
    int64_t owner = target_id;
    int left = ev.nchain;
    for (int ch = ev.head; ch >= 0 && left > 0; ch = W.rm_buf[ch]) {
      const int m = left < RM_CHUNK - 1 ? left : RM_CHUNK - 1;
      for (int q0 = 1; q0 <= m; q0 += WALK) {
        // WALK entries of the chain, then what is read of their slots,
        // together; the slots are distinct
        int e[WALK];
        SlotView sv[WALK];
        int64_t id[WALK];
#pragma unroll
        for (int u = 0; u < WALK; ++u) e[u] = W.rm_buf[ch + min(q0 + u, m)];
#pragma unroll
        for (int u = 0; u < WALK; ++u) {
          const int64_t q = e[u] >= 0 ? e[u] : p;
          sv[u] = slot_load(W, q);
          id[u] = A.id[q];
        }
#pragma unroll
        for (int u = 0; u < WALK; ++u) {
          if (q0 + u > m) continue;
          const int q = e[u];
          if (q < 0) {
            owner = copy_id(-1 - q);
            continue;
          }
          W.slot[q].dead_t = t;
          W.slot[q].dead_r = rid;
          al.live_add(sv[u].key, -1);
          slot_leave(W, q, t, sv[u]);
          st_set(W, q, ST_HOLE);
          W.holes[al.hole_index()] = ((uint64_t)box << 32) | (uint64_t)(q - B->off);
          put_info(A, B, al, id[u], 2, owner);
        }
      }
      left -= m;
    }
  }
  const unsigned long long n_samp = (unsigned long long)ev.nsamp;
  const unsigned long long n_coag = (unsigned long long)ev.ncoag;
  al.count((int64_t)n_samp, (int64_t)n_coag, (flags & RF_WARN) ? 1 : 0);
  atomicAdd((unsigned long long *)&B->n_acc_samp, n_samp);
  if (n_coag) atomicAdd((unsigned long long *)&B->n_acc_coag, n_coag);
  if (ev.err) atomicExch(&B->error, ev.err);
  if (!(flags & RF_MERGED)) return;
  const SlotView sv = slot_load(W, p);
  W.slot[p].dead_t = t;
  W.slot[p].dead_r = rid;
  al.live_add(sv.key, -1);
  write_new_particle(A, W, B, box, t, t, p, false, r, klass, target_id, nb, type, want_terms, sv);
  if (flags & RF_DIED) {
    slot_leave(W, p, t);
    st_set(W, p, ST_HOLE);
    W.holes[al.hole_index()] = ((uint64_t)box << 32) | (uint64_t)(p - B->off);
    put_info(A, B, al, target_id, 4, 0);
  } else {
    al.live_add(W.key[p], 1);
  }
  int kk = 0;
  for (int d = ev.dhead; d >= 0; d = W.q[d].next) {
    ++kk;
    const int64_t slot = al.append_slot();
    if (slot < 0) {
      atomicExch(&B->error, ERR_CAPACITY);
      return;
    }
    write_new_particle(A, W, B, box, t, t, slot, true, d, klass, copy_id(kk), nb, type, want_terms,
                       SlotView{});
    al.live_add(W.key[slot], 1);
  }
}

__device__ inline void apply_event(BoxDesc *boxes, const Arrays &A, const PW &W, int n_box,
                                   uint64_t seed, uint32_t step, int type, int want_terms, int rid,
                                   int E, int64_t hole_base, int e) {
  int box = -1;
  int64_t cs = 0, cc = 0, cw = 0;
  int nl = 0, lk[3] = {0, 0, 0}, ld[3] = {0, 0, 0};
  int *live = W.live;
  if (e < E && (W.ev_out[e] & O_WIN)) {
    const uint32_t t = W.ev_t[e];
    box = W.ev_box[e];
    BoxDesc *B = &boxes[box];
    const int first = W.box_first[box];
    ApplyAlloc al;
    al.B = B;
    al.app = W.s_app[e] - W.s_app[first];
    al.id = W.s_id[e] - W.s_id[first];
    al.info = W.s_info[e] - W.s_info[first];
    al.hole = hole_base + W.s_hole[e];
    al.live = W.live + (int64_t)box * W.K_stride;
    al.n_samp = al.n_coag = al.n_warn = 0;
    al.nl = 0;
    if (W.ev_rec[e] >= 0) {
      acc_apply(B, box, t, W.ev_rec[e], W.ev_p1[e], type, want_terms, rid, al,
                W.ev[W.ev_rec[e]].nchain > CHAIN_WAVE_MIN);
    } else {
      perset_merge(B, A, W, box, n_box, t, W.ev_p1[e], W.ev_p2[e], seed, step, type, want_terms,
                   rid, al, W.ev_out[e] & ~O_WIN, nullptr, false,
                   load_parents(A, W, W.ev_p1[e], W.ev_p2[e]));
    }
    cs = al.n_samp;
    cc = al.n_coag;
    cw = al.n_warn;
    nl = al.nl;
    for (int i = 0; i < 3; ++i) {
      lk[i] = al.lk[i];
      ld[i] = al.ld[i];
    }
    live = al.live;
  }
  wave_flush_counts(boxes, box, cs, cc, cw);
  for (int i = 0; i < 3; ++i) wave_flush_live(live, i < nl ? lk[i] : -1, i < nl ? ld[i] : 0);
}

// apply the round's winners, each at the positions its ranks give
__global__ void __launch_bounds__(256)
k_par_apply(BoxDesc *boxes, Arrays A, PW W, int n_box, uint64_t seed, uint32_t step,
            int type, int want_terms, int rid) {
  const int E = W.rc[RC_E];
  if ((int)(blockIdx.x * blockDim.x) >= E) return;
  step_ctx_fill(A, W);
  const int64_t hole_base = (int64_t)*W.hole_top;
  // the loop bound is uniform over the workgroup: every lane reaches the
  // wavefront flushes of each pass
  for (int base = blockIdx.x * blockDim.x; base < E; base += gridDim.x * blockDim.x)
    apply_event(boxes, A, W, n_box, seed, step, type, want_terms, rid, E, hole_base,
                base + (int)threadIdx.x);
}

// The removed sources of the round's winning target events with long
// removal chains, one wavefront per event: each chunk's entries go to
// lanes, the ranks of holes and removal records follow the chain order (a
// ballot count of the entries before a lane), and each record names the
// particle that took the source: the target, or the copy named by the last
// copy marker before it in the chain (a ballot of the markers).
__device__ inline void apply_chain(BoxDesc *boxes, const Arrays &A, const PW &W, int e, int lane,
                                   int64_t hole_base, int rid) {
  if (!(W.ev_out[e] & O_WIN)) return;
  const int r = W.ev_rec[e];
  if (r < 0 || W.ev[r].nchain <= CHAIN_WAVE_MIN) return;
  const uint32_t t = W.ev_t[e];
  const int box = W.ev_box[e];
  BoxDesc *B = &boxes[box];
  const int first = W.box_first[box];
  const int64_t hole0 = hole_base + W.s_hole[e];
  const int64_t info0 = B->n_info + (W.s_info[e] - W.s_info[first]);
  const int64_t id_first =
      (B->next_id + (W.s_id[e] - W.s_id[first]) - 1) * B->id_stride + B->id_offset + 1;
  int *live = W.live + (int64_t)box * W.K_stride;
  int64_t owner = A.id[W.ev_p1[e]];
  int done = 0;  // removed sources before this chunk
  int left = W.ev[r].nchain;
  for (int ch = W.ev[r].head; ch >= 0 && left > 0; ch = W.rm_buf[ch]) {
    const int m = left < RM_CHUNK - 1 ? left : RM_CHUNK - 1;
    const bool here = lane < m;
    const int q = here ? W.rm_buf[ch + 1 + lane] : 0;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint64_t marks = __ballot(here && q < 0);
    const uint64_t rems = __ballot(here && q >= 0);
    // the owner of this lane's entry: the last marker at or before it
    const uint64_t mk = marks & (below | (1ull << lane));
    // every lane shuffles (no divergence around the cross-lane read)
    const int src = mk ? 63 - __clzll((long long)mk) : lane;
    const int qm = __shfl(q, src);
    const int64_t own = mk ? id_first + (int64_t)(-1 - qm - 1) * B->id_stride : owner;
    if (here && q >= 0) {
      const int ord = done + __popcll(rems & below);
      W.slot[q].dead_t = t;
      W.slot[q].dead_r = rid;
      atomicAdd(&live[W.key[q]], -1);
      slot_leave(W, q, t);
      st_set(W, q, ST_HOLE);
      W.holes[hole0 + ord] = ((uint64_t)box << 32) | (uint64_t)(q - B->off);
      const int64_t ki = info0 + ord;
      if (ki < B->info_cap) {
        A.info_id[B->info_off + ki] = A.id[q];
        A.info_action[B->info_off + ki] = 2;
        A.info_other[B->info_off + ki] = own;
      }
    }
    const int last = marks ? 63 - __clzll((long long)marks) : 0;
    const int ql = __shfl(q, last);
    if (marks) owner = id_first + (int64_t)(-1 - ql - 1) * B->id_stride;
    done += __popcll(rems);
    left -= m;
  }
}

__global__ void __launch_bounds__(256)
k_par_apply_chains(BoxDesc *boxes, Arrays A, PW W, int rid) {
  const int lane = threadIdx.x & 63;
  const int E = W.rc[RC_E];
  const int64_t hole_base = (int64_t)*W.hole_top;
  // one wavefront per event, striding over the round's events
  for (int e = blockIdx.x * 4 + (threadIdx.x >> 6); e < E; e += gridDim.x * 4)
    apply_chain(boxes, A, W, e, lane, hole_base, rid);
}

// A box's count with `added` more particles.  Those beyond its capacity were
// not written (the box holds ERR_CAPACITY), and no pass after this one, nor a
// reader of the box, may go past the slots that were.
__device__ inline int grown(const BoxDesc *B, int64_t added) {
  return (int)min((int64_t)B->n_part + added, B->cap);
}

// per-box totals of a round: appended slots, new ids, records, winners
__device__ inline void box_totals(BoxDesc *boxes, const PW &W, int E, int box) {
  const int first = W.box_first[box];
  if (first < 0) return;
  int lo = first, hi = E - 1;  // last event of the box (ev_box sorted)
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (W.ev_box[mid] == box) lo = mid; else hi = mid - 1;
  }
  const int last = lo;
  BoxDesc *B = &boxes[box];
  B->n_part = grown(B, (int64_t)W.s_app[last] + W.f_app[last] - W.s_app[first]);
  B->next_id += W.s_id[last] + W.f_id[last] - W.s_id[first];
  B->n_info += W.s_info[last] + W.f_info[last] - W.s_info[first];
}

__device__ inline void release_event(const PW &W, int e) {
  W.slot[W.ev_p1[e]].claim = UNCLAIMED;
  W.slot[W.ev_p1[e]].claim_wr = UNCLAIMED;
  const int r = W.ev_rec[e];
  if (r >= 0) {
    rm_walk(W, r, [&](int q) {
      W.slot[q].claim = UNCLAIMED;
      W.slot[q].claim_wr = UNCLAIMED;
    });
  } else {
    W.slot[W.ev_p2[e]].claim = UNCLAIMED;
    W.slot[W.ev_p2[e]].claim_wr = UNCLAIMED;
  }
}

// Tests of the round that must be drawn again: accepted tests that lost a
// claim, and any other non-winning test that drew a particle which an
// earlier winner (smaller sequential index) of the same round removed or
// changed after the draw -- in the sequential chain that test would have
// seen the particles as that winner left them.  A particle changed in an
// earlier round was drawn in its changed state.
__device__ inline bool consumed_before(const PW &W, int p, uint32_t t, int rid) {
  if (p < 0) return false;
  const uint32_t st = W.slot[p].st, dead_t = W.slot[p].dead_t;
  const int dead_r = W.slot[p].dead_r;
  return (int)(st >> 2) == W.epoch && (st & 3) != ST_LIVE && dead_t < t && dead_r == rid;
}

// A test on an empty arrival entry of list L (bin bL) of a pair that
// begins at tau is final once no event with a smaller index than tau that
// could add a particle to L was pending at the start of the round that ran
// it: every arrival into L before tau had been applied then.  On the
// pair's second list the bound is the test's own index, since earlier
// tests of the pair can change the first list's draws (a member they
// removed is drawn again).  Such tests change no list until an earlier
// event fills their entry, so they do not hold back others.
// Returns the word of the next round's minima that the test's index lowers,
// or null.
__device__ inline uint32_t *pending_test(BoxDesc *boxes, const PW &W, int n_box, int rid, int i) {
  uint32_t t = W.tid[i];
  const int64_t NP = (int64_t)n_box * W.P_stride;
  const int64_t k = test_pair(W, NP, t);
  int64_t q;
  const int box = pair_box(W, k, &q);
  int c1, c2, b1, b2;
  decode_pair(q, W.tab_classes, W.max_bin, &c1, &c2, &b1, &b2);
  const int kind = W.pair_acc[k];
  // the lowest bin this event's results can land in
  const int b_lo = kind ? (kind == 1 ? b1 : b2) : max(b1, b2);
  const int64_t mb = (int64_t)box * W.K_stride;
  const bool athin = (W.tns[i] & TNS_ATHIN) && !W.acc[i];
  int f = 0;
  if (athin) {
    // an empty entry of the second list was reached after the first
    // list's draws, which earlier tests of the same pair can change
    const bool side2 = !kind && (W.tns[i] & TNS_SIDE2);
    const int b_list = kind ? b_lo : (side2 ? b2 : b1);
    f = (side2 ? t : W.pair_exc[k]) <= W.minpend[mb + b_list - 1] ? 0 : 1;
  } else if (W.acc[i]) {
    f = (W.ev_out[W.acc_scan[i]] & O_WIN) ? 0 : 1;
  } else if (W.trec[i] >= 0) {
    // a target event without effect: final unless an earlier winner of the
    // round changed its target; its samples count once final
    bool changed = consumed_before(W, W.tp1[i], t, rid);
    if (W.tp1[i] >= 0)
      rd_walk(W, W.trec[i], [&](int q) { changed = changed || consumed_before(W, q, t, rid); });
    f = changed ? 1 : 0;
    int v = W.tns[i];
    if (!f && v) {
      BoxDesc *B = &boxes[box];
      unsigned long long ns = (unsigned long long)(v & (ACC_WARN - 1));
      atomicAdd((unsigned long long *)&B->n_samp, ns);
      atomicAdd((unsigned long long *)&B->step_samp, ns);
      atomicAdd((unsigned long long *)&B->n_acc_samp, ns);
      if (v & ACC_WARN) atomicAdd((unsigned long long *)&B->n_warn, 1ull);
    }
  } else if (W.tp1[i] >= 0) {
    f = (consumed_before(W, W.tp1[i], t, rid) || consumed_before(W, W.tp2[i], t, rid)) ? 1 : 0;
  }
  if (!f && W.trec[i] < 0 && (W.tns[i] & ACC_WARN)) {
    // a per-set test's k_max warning (src/coagulation.F90:749-751), once final
    atomicAdd((unsigned long long *)&boxes[box].n_warn, 1ull);
  }
  W.f_pend[i] = f;
  // values only fall: most tests see a smaller one already and skip the atomic
  uint32_t *m = &W.minpend_next[mb + b_lo - 1];
  return f && !athin && *m > t ? m : nullptr;
}

// What follows the round's merges, in one launch: the boxes' totals, the
// claims released, and which tests stay pending (none of which reads what
// another writes).
__global__ void k_par_settle(BoxDesc *boxes, PW W, int n_box, int rid) {
  const int n = W.rc[RC_N], E = W.rc[RC_E];
  if (n == 0) return;
  PAR_FOR(b, n_box) box_totals(boxes, W, E, b);
  PAR_FOR(e, E) release_event(W, e);
  // The tests come in index order, so the first of a wavefront's lanes with
  // the same word has their minimum: one atomic for all of them (each on its
  // own: 54 us a round of 1e5 Brownian particles, now 21).  The loop bound is
  // uniform over the workgroup.
  for (int base = blockIdx.x * blockDim.x; base < n; base += gridDim.x * blockDim.x) {
    const int i = base + (int)threadIdx.x;
    uint32_t *m = i < n ? pending_test(boxes, W, n_box, rid, i) : nullptr;
    uint64_t todo = __ballot(m != nullptr);
    while (todo) {
      const int first = __ffsll((long long)todo) - 1;
      uint32_t *word = (uint32_t *)__shfl((unsigned long long)m, first);
      if ((int)(threadIdx.x & 63) == first) atomicMin(word, W.tid[i]);
      todo &= ~__ballot(m == word);
    }
  }
}

// the pending tests in order, with their pairs (which the tail reads)
struct GatherPending {
  PW W;
  int64_t NP;
  __device__ void operator()(int64_t i, uint32_t f, uint32_t at) const {
    if (!f) return;
    const uint32_t t = W.tid[i];
    W.pend[at] = t;
    W.pend_k[at] = (int)test_pair(W, NP, t);
  }
};

// The end of a device-wide round, one workgroup per box: the running minimum
// over the box's bins of the next round's minima, this round's cleared for
// the round after.  And, if the round ran, its holes join the step's count,
// and its pending tests go to another device-wide round while that settles
// most of the batch (at most half of it still pending, and not the last
// round), else to the tail.  A round without events leaves nothing
// pending: with no winner no test's inputs changed, and a test on an empty
// arrival entry stays thinned, as no particle arrived.
constexpr int PREFIX_THREADS = 256;
__global__ void __launch_bounds__(PREFIX_THREADS) k_round_end(PW W, int n_batch, int round) {
  __shared__ scan_storage<PREFIX_THREADS, uint32_t> tmp;
  __shared__ uint32_t carry;
  const int tid = threadIdx.x;
  uint32_t *m = W.minpend_next + (int64_t)blockIdx.x * W.K_stride;
  uint32_t *c = W.minpend + (int64_t)blockIdx.x * W.K_stride;
  for (int base = 0; base < W.K_stride; base += PREFIX_THREADS) {
    const int q = base + tid;
    uint32_t v = q < W.K_stride ? m[q] : UNCLAIMED;
    if (base > 0 && tid == 0) v = min(v, carry);
    uint32_t tot;
    const uint32_t r = block_scan_incl<PREFIX_THREADS>(v, OpMin(), tmp, &tot);
    if (q < W.K_stride) {
      m[q] = r;
      c[q] = UNCLAIMED;
    }
    if (tid == PREFIX_THREADS - 1) carry = r;
    __syncthreads();
  }
  if (tid != 0) return;
  W.box_first[blockIdx.x] = -1;
  if (blockIdx.x != 0) return;
  const int n = W.rc[RC_N];
  if (n == 0) return;  // the round did not run
  if (W.ev) {
    *W.rm_top = 0;
    *W.dup_top = 0;
  }
  const int E = W.rc[RC_E];
  const int p = E > 0 ? W.s_pend[n] : 0;
  *W.hole_top += (unsigned long long)W.s_hole[E];
  W.pstat[0] += 1ull;
  W.rstat[round == 0 ? 0 : 2] = (unsigned long long)E;
  if (p > 0 && round < PAR_ROUNDS - 1 && p <= n_batch / 2) {
    W.rc[RC_N] = p;
    W.rstat[1] = (unsigned long long)p;
  } else {
    W.rc[RC_N] = 0;
    W.rc[RC_TAIL] = p;
    W.rstat[3] = (unsigned long long)p;
    W.pstat[1] += (unsigned long long)p;
  }
}

// first index of the sorted list v[0..n) holding a value >= x
__device__ inline int lower_bound_u32(const uint32_t *v, int n, uint32_t x) {
  int lo = 0, hi = n;
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    if (v[mid] < x) lo = mid + 1; else hi = mid;
  }
  return lo;
}

constexpr int TAIL_THREADS = 512;
constexpr int TF_EFFECT = 1, TF_ACC = 2, TF_RUN = 4, TF_WARN = 8, TF_ATHIN = 16, TF_SIDE2 = 32,
              TF_WAIT = 64;

// claims inside one kernel are read and released with device-scope atomics,
// so they need no cache maintenance between the phases of a round
__device__ inline uint32_t claim_load(const PW &W, int p) {
  return __hip_atomic_load(&W.slot[p].claim, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline uint32_t claim_wr_load(const PW &W, int p) {
  return __hip_atomic_load(&W.slot[p].claim_wr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void claim_release(const PW &W, int p) {
  __hip_atomic_store(&W.slot[p].claim, UNCLAIMED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&W.slot[p].claim_wr, UNCLAIMED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}


// a phase boundary of the tail: earlier writes of the box's workgroup
// become visible to its next phase.  Only this workgroup touches the box,
// so a workgroup-scope fence suffices; claims go through device-scope
// atomics.
__device__ inline void tail_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  __syncthreads();
}

// The tail of a batch: the tests still pending after the device-wide claim
// rounds, mostly chains of tests on one particle (a large particle drawn by
// many tests of its bin pairs).  One workgroup per box runs claim rounds
// over a window of the box's next TAIL_THREADS pending tests, in sequential
// order, with barriers in place of launches.  A test is run again only when
// a particle it read or claimed was changed by an earlier winner; a test
// that lost with its inputs unchanged keeps its outcome and claims again.
// The window's earliest test always wins or is final, so every round makes
// progress.
// Claims distinguish reading from changing.  Every particle of an accepted
// test is claimed in W.claim (earliest accessor); the particles the test
// changes are also claimed in W.claim_wr (earliest writer).  A per-set
// merge changes only the parents it removes: a parent that stays is read
// and left as it was.  A test wins when it is the earliest accessor of
// every particle it changes and no earlier test changes a particle it only
// reads.  Tests that only read a particle therefore win together (the
// large-weight particle a bin pair draws over and over, which the
// weighting keeps), and a later test that changes it waits for them.
__global__ void __launch_bounds__(TAIL_THREADS)
k_par_tail(BoxDesc *boxes, Arrays A, PW W, int n_box, const uint32_t *pend, int type,
           uint64_t seed, uint32_t step, int precision, double band, double del_t,
           uint32_t acc_base, int want_terms, int rid0, unsigned long long *rounds_out,
           uint32_t batch_t0) {
  const int box = blockIdx.x;
  const int tid = threadIdx.x;
  BoxDesc *B = &boxes[box];
  const int64_t pb = (int64_t)box * W.P_stride;
  const int n = W.rc[RC_TAIL];
  if (n == 0) return;
  const int lo = lower_bound_u32(pend, n, W.pair_exc[pb]);
  const int hi = lower_bound_u32(pend, n, W.pair_exc[pb + W.P_stride]);
  if (lo >= hi) return;
  step_ctx_fill(A, W);
  __shared__ scan_storage<TAIL_THREADS, int> scan_tmp;
  __shared__ scan_storage<TAIL_THREADS, uint32_t> scan_tmp3;
  __shared__ uint32_t s_carry;
  __shared__ scan_storage<TAIL_THREADS, long long> scan_tmp2;
  __shared__ uint32_t w_t[TAIL_THREADS];
  __shared__ int w_k[TAIL_THREADS], w_p1[TAIL_THREADS], w_p2[TAIL_THREADS];
  __shared__ int w_tns[TAIL_THREADS], w_fl[TAIL_THREADS];
  __shared__ int s_tot[4];
  __shared__ long long s_hole_base;
  __shared__ int s_err;
  // the box's weights, read by every test and merge decision of the tail
  __shared__ Weights s_w;
  for (int q = tid; q < (int)(sizeof(Weights) / sizeof(int)); q += TAIL_THREADS)
    ((int *)&s_w)[q] = ((const int *)&B->w)[q];
  extern __shared__ int s_live[];  // live-count changes of the box's lists
  // then, per bin, the lowest index of an unsettled test of the window whose
  // results land in that bin or a lower one (a running minimum)
  uint32_t *s_pm = (uint32_t *)(s_live + W.K_stride);
  for (int q = tid; q < W.K_stride; q += TAIL_THREADS) s_live[q] = 0;
  int64_t c_samp = 0, c_coag = 0, c_warn = 0;  // this lane's counter changes
  int wn = 0, head = lo;
  int rid = rid0;
  unsigned long long n_rounds = 0;
  for (;;) {
    if (tid == 0) s_err = B->error;
    tail_barrier();
    if (s_err || (wn == 0 && head >= hi)) break;
    // refill the window from the queue, in order
    const int add = min(TAIL_THREADS - wn, hi - head);
    if (tid < add) {
      const uint32_t t = pend[head + tid];
      const int kl = (int)(W.pend_k[head + tid] - pb);
      w_t[wn + tid] = t;
      w_k[wn + tid] = kl;
      w_fl[wn + tid] = TF_RUN | (W.pair_acc[pb + kl] ? TF_ACC : 0);
      w_p1[wn + tid] = -1;
      w_p2[wn + tid] = -1;
      w_tns[wn + tid] = 0;
    }
    __syncthreads();
    wn += add;
    head += add;
    const bool active = tid < wn;
    uint32_t t = 0;
    int64_t k = pb;
    int fl = 0, p1 = -1, p2 = -1, tns = 0;
    if (active) {
      t = w_t[tid];
      k = pb + w_k[tid];
      fl = w_fl[tid];
      p1 = w_p1[tid];
      p2 = w_p2[tid];
      tns = w_tns[tid];
    }
    const bool is_acc = fl & TF_ACC;
    const int rec = is_acc ? (int)(W.acc_exc[k] + (t - W.pair_exc[k]) - acc_base) : -1;
    // 1. run the tests whose inputs are new or changed
    if (active && (fl & TF_RUN)) {
      fl &= ~(TF_RUN | TF_EFFECT | TF_WARN | TF_ATHIN | TF_SIDE2 | TF_WAIT);
      if (is_acc) {
        const int r = run_visit(boxes, A, k, t, rec, type, seed, step, del_t, false, &p1, &tns);
        if (r == 1) fl |= TF_EFFECT;
        if (tns & TNS_ATHIN) fl |= TF_ATHIN;
        p2 = -1;
      } else {
        TestOut o;
        perset_test(B, A, W, box, k, k - pb, t, type, seed, step, precision, band, 0, o,
                    s_w);
        p1 = o.p1;
        p2 = o.p2;
        W.thin[t - batch_t0] = o.thin ? 1 : 0;
        if (o.accept) fl |= TF_EFFECT;
        if (o.warn) fl |= TF_WARN;
        if (o.thin >= 2) fl |= TF_ATHIN;
        if (o.thin == 3) fl |= TF_SIDE2;
      }
    }
    const bool effect = fl & TF_EFFECT;
    // the merge decisions of an accepted per-set test, from the particles as
    // they are now: they say which parents it changes
    int o_win = -1;
    Stream ms{};  // a per-set test's merge stream, after its decisions
    if (effect && !is_acc) {
      int c1, c2, b1, b2;
      decode_pair(k - pb, W.tab_classes, W.max_bin, &c1, &c2, &b1, &b2);
      const int nb = B->n_bin, nc = B->w.n_class;
      const int cc = A.cc[table_index(A, box, nb, nc, b1, b2, c1, c2)];
      ms.open(seed, box, step, pair_site(nb, nc, b1, b2, c1, c2), t - W.pair_exc[k], RNG_MERGE);
      int g;
      o_win = merge_decide(A, W, B, ms, p1, p2, c1, c2, cc, &g, s_w) | (g << 16) | (cc << 24);
    }
    // 2. claims
    if (effect) {
      if (is_acc) {
        claim_write(W, p1, t);
        rm_walk(W, rec, [&](int q) { claim_write(W, q, t); });
      } else {
        if (o_win & O_RM1) claim_write(W, p1, t);
        else atomicMin(&W.slot[p1].claim, t);
        if (o_win & O_RM2) claim_write(W, p2, t);
        else atomicMin(&W.slot[p2].claim, t);
      }
    }
    // what a merge reads of its parents travels while the claims settle: no
    // winner of the round changes a particle that another one reads
    MergeParents par{};
    if (effect && !is_acc) par = load_parents(A, W, p1, p2);
    __syncthreads();
    // 3. resolve, and what each winner creates
    bool win = false;
    int c_app = 0, c_id = 0, c_info = 0, c_hole = 0;
    if (effect) {
      if (is_acc) {
        win = claim_load(W, p1) == t;
        rm_walk(W, rec, [&](int q) {
          const bool held = claim_load(W, q) == t;
          win = win && held;
        });
        rd_walk(W, rec, [&](int q) {
          const bool held = claim_wr_load(W, q) >= t;
          win = win && held;
        });
        if (win) {
          const int died = (W.ev[rec].flags & RF_DIED) ? 1 : 0;
          c_app = W.ev[rec].ndup;
          c_id = W.ev[rec].ndup;
          c_info = W.ev[rec].nrm + died;
          c_hole = W.ev[rec].nrm + died;
        }
      } else {
        const int o = o_win & 0xFFFF;
        win = ((o & O_RM1) ? claim_load(W, p1) == t : claim_wr_load(W, p1) > t) &&
              ((o & O_RM2) ? claim_load(W, p2) == t : claim_wr_load(W, p2) > t);
        if (win) {
          c_app = (o & O_APPEND) ? 1 : 0;
          c_id = (o & O_NEWID) ? 1 : 0;
          c_info = ((o & O_INFO1) ? 1 : 0) + ((o & O_INFO2) ? 1 : 0);
          c_hole = ((o & O_RM1) && !(o & O_SLOT1) ? 1 : 0) + ((o & O_RM2) && !(o & O_SLOT2) ? 1 : 0);
        }
      }
    }
    // ranks of what the winners create: two scans of packed counts
    long long ai = ((long long)c_id << 32) | (long long)c_app;
    long long ih = ((long long)c_hole << 32) | (long long)c_info;
    long long r_ai, r_ih, t_ai, t_ih;
    r_ai = block_sum_excl<TAIL_THREADS>(ai, scan_tmp2, &t_ai);
    r_ih = block_sum_excl<TAIL_THREADS>(ih, scan_tmp2, &t_ih);
    const int r_app = (int)(r_ai & 0xFFFFFFFFll), r_id = (int)(r_ai >> 32);
    const int r_info = (int)(r_ih & 0xFFFFFFFFll), r_hole = (int)(r_ih >> 32);
    int tot;
    if (tid == 0) {
      s_tot[0] = (int)(t_ai & 0xFFFFFFFFll);
      s_tot[1] = (int)(t_ai >> 32);
      s_tot[2] = (int)(t_ih & 0xFFFFFFFFll);
      s_tot[3] = (int)(t_ih >> 32);
      const int th = s_tot[3];
      s_hole_base = th ? (long long)atomicAdd(W.hole_top, (unsigned long long)th) : 0ll;
    }
    __syncthreads();
    // 4. apply the winners at their ranks
    const bool in_place =
        wave_components(A, B, win && !is_acc, o_win, p1, p2, r_app, ms, par);
    if (win) {
      TailAlloc al;
      al.B = B;
      al.app = r_app;
      al.id = r_id;
      al.info = r_info;
      al.hole = (int64_t)s_hole_base + r_hole;
      al.live = nullptr;
      al.s_live = s_live;
      al.n_samp = al.n_coag = al.n_warn = 0;
      if (is_acc) acc_apply(B, box, t, rec, p1, type, want_terms, rid, al);
      else perset_merge(B, A, W, box, n_box, t, p1, p2, seed, step, type, want_terms, rid, al,
                        o_win, &ms, in_place, par);
      c_samp += al.n_samp;
      c_coag += al.n_coag;
      c_warn += al.n_warn;
    }
    tail_barrier();
    if (tid == 0) {
      B->n_part = grown(B, s_tot[0]);
      B->next_id += s_tot[1];
      B->n_info += s_tot[2];
    }
    // 5. release the claims
    if (effect) {
      claim_release(W, p1);
      if (is_acc) rm_walk(W, rec, [&](int q) { claim_release(W, q); });
      else claim_release(W, p2);
    }
    // 6. what stays in the window: losers (run again only if an earlier
    // winner changed what they read) and tests whose inputs changed
    int keep = 0;
    bool athin = false;
    if (active && !win) {
      bool changed = consumed_before(W, p1, t, rid) || consumed_before(W, p2, t, rid);
      if (is_acc && effect && !changed)
        rm_walk(W, rec, [&](int q) { changed = changed || consumed_before(W, q, t, rid); });
      if (is_acc && p1 >= 0 && !changed)
        rd_walk(W, rec, [&](int q) { changed = changed || consumed_before(W, q, t, rid); });
      if (effect || changed) {
        keep = 1;
        if (changed) fl |= TF_RUN;
      } else if (fl & TF_ATHIN) {
        athin = true;  // decided below
      } else {
        // final without effect: its counts
        if (is_acc && tns) {
          c_samp += tns & (ACC_WARN - 1);
          atomicAdd((unsigned long long *)&B->n_acc_samp,
                    (unsigned long long)(tns & (ACC_WARN - 1)));
          if (tns & ACC_WARN) c_warn += 1;
        }
        if (!is_acc && (fl & TF_WARN)) c_warn += 1;
      }
    }
    if (win && !is_acc && (fl & TF_WARN)) c_warn += 1;
    // A test thinned on an empty arrival entry of list L (bin bL) is final
    // once no earlier test of the window that won this round (its arrivals
    // show from the next round on) or waits for another round could add a
    // particle to L: particles only grow, so a test on bins b1, b2 adds
    // them to bins from max(b1, b2) up, and a target event to bins from its
    // target's.  On the pair's second list the bound is the test's own
    // index (earlier tests of the pair can change the first list's draws).
    // Until then it waits, and it runs once more when it is no longer
    // blocked.
    for (int q = tid; q < W.K_stride; q += TAIL_THREADS) s_pm[q] = UNCLAIMED;
    __syncthreads();
    int b1 = 1, b2 = 1, kind = 0;
    if (active) {
      int c1, c2;
      decode_pair(k - pb, W.tab_classes, W.max_bin, &c1, &c2, &b1, &b2);
      kind = W.pair_acc[k];
    }
    const int b_lo = kind ? (kind == 1 ? b1 : b2) : max(b1, b2);
    if (active && (win || keep)) atomicMin(&s_pm[b_lo - 1], t);
    __syncthreads();
    // running minimum over the bins, TAIL_THREADS bins at a time
    const int nbin = B->n_bin;
    for (int base = 0; base < nbin; base += TAIL_THREADS) {
      const int q = base + tid;
      uint32_t v = q < nbin ? s_pm[q] : UNCLAIMED;
      if (base > 0 && tid == 0) v = min(v, s_carry);
      uint32_t tot_m;
      const uint32_t r = block_scan_incl<TAIL_THREADS>(v, OpMin(), scan_tmp3, &tot_m);
      if (q < nbin) s_pm[q] = r;
      if (tid == TAIL_THREADS - 1) s_carry = r;
      __syncthreads();
    }
    if (athin) {
      const bool side2 = !kind && (fl & TF_SIDE2);
      const int b_list = kind ? b_lo : (side2 ? b2 : b1);
      const bool blocked = (side2 ? t : W.pair_exc[k]) > s_pm[b_list - 1];
      if (blocked) {
        // wait, without running, until the events that block it settle
        keep = 1;
        fl |= TF_WAIT;
      } else if (fl & TF_WAIT) {
        // unblocked since its last run: run once more, on the settled lists
        keep = 1;
        fl = (fl & ~TF_WAIT) | TF_RUN;
      }
    }
    int r_keep;
    r_keep = block_sum_excl<TAIL_THREADS>(keep, scan_tmp, &tot);
    if (keep) {
      w_t[r_keep] = t;
      w_k[r_keep] = (int)(k - pb);
      w_fl[r_keep] = fl;
      w_p1[r_keep] = p1;
      w_p2[r_keep] = p2;
      w_tns[r_keep] = tns;
    }
    wn = tot;
    rid++;
    n_rounds++;
  }
  __syncthreads();
  // flush the gathered live-count and counter changes
  int *live = W.live + (int64_t)box * W.K_stride;
  for (int q = tid; q < W.K_stride; q += TAIL_THREADS)
    if (s_live[q]) atomicAdd(&live[q], s_live[q]);
  if (c_samp) {
    atomicAdd((unsigned long long *)&B->n_samp, (unsigned long long)c_samp);
    atomicAdd((unsigned long long *)&B->step_samp, (unsigned long long)c_samp);
  }
  if (c_coag) {
    atomicAdd((unsigned long long *)&B->n_coag, (unsigned long long)c_coag);
    atomicAdd((unsigned long long *)&B->step_coag, (unsigned long long)c_coag);
  }
  if (c_warn) atomicAdd((unsigned long long *)&B->n_warn, (unsigned long long)c_warn);
  if (tid == 0 && n_rounds) {
    atomicAdd(rounds_out, n_rounds);
    B->n_rounds += (int)n_rounds;
    B->n_tail_tests += hi - lo;
  }
}

// the largest bin count among the boxes (their pair space for this step),
// to the host
__global__ void __launch_bounds__(256) k_max_nbin(const BoxDesc *boxes, int n_box, uint32_t *out) {
  __shared__ scan_storage<256, int> tr;
  int m = 1;
  for (int b = threadIdx.x; b < n_box; b += 256)
    if (!boxes[b].error) m = max(m, boxes[b].n_bin);
  const int r = block_reduce<256>(m, OpMax(), tr);
  if (threadIdx.x == 0) out[0] = (uint32_t)r;
}

// Round state of a batch after the first (k_step_front clears the first's),
// and the entries after the pair space when its size is new.
__global__ void k_batch_reset(PW W, int n_box, int64_t NP, int n_batch) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (int64_t)n_box * W.K_stride) {
    W.minpend[i] = 0u;
    W.minpend_next[i] = UNCLAIMED;
  }
  if (i != 0) return;
  batch_begin(W, n_batch);
  *W.tail_rounds = 0ull;
  if (W.ev) {
    *W.rm_top = 0;
    *W.dup_top = 0;
  }
  W.pair_n[NP] = 0;
  W.pair_accn[NP] = 0;
}

__global__ void k_init_slots(SlotRec *p, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = SlotRec{UNCLAIMED, UNCLAIMED, 0u, 0, 0, 0u, 0, ST_LIVE};
}
__global__ void k_clear_status(SlotRec *p, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i].st = ST_LIVE;
}
// Tail-fill compaction over all holes at once.  Per box: the range of its
// holes in the sorted list and how many lie below the final count.  Then
// the j-th such head hole receives the j-th live slot of the tail
// [n_final, n) in slot order: v = n_final + j + m with m the number of the
// tail's holes below v, found by binary search over those holes.  Sources
// lie at or above n_final and destinations below it, so the moves run in
// place.  Live particles of the tail keep their slot order.
__device__ inline void compact_range(const BoxDesc *boxes, const PW &W, const uint64_t *sorted,
                                     int box, int n_holes) {
  auto lower = [&](uint64_t key, int lo, int hi) {
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (sorted[mid] < key) lo = mid + 1; else hi = mid;
    }
    return lo;
  };
  const int lo = lower((uint64_t)box << 32, 0, n_holes);
  const int hi = lower((uint64_t)(box + 1) << 32, lo, n_holes);
  const int n_final = boxes[box].n_part - (hi - lo);
  W.cmp_lo[box] = lo;
  W.cmp_hi[box] = hi;
  W.cmp_head[box] = lower(((uint64_t)box << 32) | (uint64_t)(uint32_t)n_final, lo, hi) - lo;
}

__global__ void k_compact_ranges(BoxDesc *boxes, PW W, int n_box, int n_holes) {
  const int box = blockIdx.x * blockDim.x + threadIdx.x;
  if (box < n_box) compact_range(boxes, W, W.holes_sorted, box, n_holes);
}

// Few holes are sorted and cut into the boxes' ranges by one workgroup: each
// thread counts the holes below its own in LDS, n reads a hole, 2 us for 1000
// of them (the device radix sort and the ranges: 14 + 4 us).  Beyond
// FEW_HOLES the quadratic count loses.
constexpr int FEW_HOLES = 2048;
__global__ void __launch_bounds__(1024) k_compact_few(BoxDesc *boxes, PW W, int n_box,
                                                      int n_holes) {
  __shared__ uint64_t s_in[FEW_HOLES], s_out[FEW_HOLES];
  for (int i = threadIdx.x; i < n_holes; i += 1024) s_in[i] = W.holes[i];
  __syncthreads();
  for (int i = threadIdx.x; i < n_holes; i += 1024) {
    const uint64_t h = s_in[i];
    int rank = 0;
    for (int j = 0; j < n_holes; ++j) rank += s_in[j] < h ? 1 : 0;
    s_out[rank] = h;
    W.holes_sorted[rank] = h;
  }
  __syncthreads();
  for (int box = threadIdx.x; box < n_box; box += 1024)
    compact_range(boxes, W, s_out, box, n_holes);
}

__global__ void k_compact_move(BoxDesc *boxes, Arrays A, PW W, int n_holes) {
  const int jg = blockIdx.x * blockDim.x + threadIdx.x;
  if (jg >= n_holes) return;
  const uint64_t h = W.holes_sorted[jg];
  const int box = (int)(h >> 32);
  const int lo = W.cmp_lo[box], hi = W.cmp_hi[box], head = W.cmp_head[box];
  const int j = jg - lo;
  if (j >= head) return;
  const BoxDesc *B = &boxes[box];
  const int n_final = B->n_part - (hi - lo);
  // tail holes: sorted slots at [lo + head, hi); the smallest m with
  // n_final + j + m < tail_hole[m] (or m = their count)
  int a = 0, b = hi - lo - head;
  while (a < b) {
    const int m = (a + b) >> 1;
    const int slot = (int)(W.holes_sorted[lo + head + m] & 0xFFFFFFFFu);
    if (n_final + j + m < slot) b = m; else a = m + 1;
  }
  const int from = n_final + j + a;
  const int hole = (int)(h & 0xFFFFFFFFu);
  const int64_t pf = B->off + from, pt = B->off + hole;
  copy_particle(A, pf, pt);
  W.key[pt] = W.key[pf];
  W.terms[pt] = W.terms[pf];
  W.slot[pt].st = W.slot[pf].st;
}

__global__ void k_par_invalidate(BoxDesc *boxes, int n_box) {
  int box = blockIdx.x * blockDim.x + threadIdx.x;
  if (box >= n_box) return;
  boxes[box].pkeys_valid = 0;
  boxes[box].terms_kernel = 0;
}

// The end of a step, one workgroup a box: the slots the compaction freed, the
// sort's flags, and the arrivals of the step beyond their list's reserved
// entries (not seen by the list's later pairs).
__global__ void __launch_bounds__(256) k_step_end(BoxDesc *boxes, PW W, int compacted) {
  const int box = blockIdx.x;
  BoxDesc *B = &boxes[box];
  int over = 0;
  for (int k = threadIdx.x; k < W.K_stride; k += 256) {
    const int64_t L = (int64_t)box * W.K_stride + k;
    over += max(0, W.arr_n[L] - W.acap[L]);
  }
  for (int off = 32; off > 0; off >>= 1) over += __shfl_xor(over, off);
  if ((threadIdx.x & 63) == 0 && over)
    atomicAdd((unsigned long long *)&B->n_arr_over, (unsigned long long)over);
  if (threadIdx.x != 0) return;
  if (compacted) B->n_part -= W.cmp_hi[box] - W.cmp_lo[box];
  B->valid_sort = 1;
  B->xlists_valid = 0;
}

// ------------------------------------------------------------ host side
// The reference's tot_n_samp counts each pair's Poisson draw over the
// members present when the loop reaches it (src/coagulation.F90:627): the
// batch's thinned tests come off the counts drawn over the bound.  The
// step's holes, the tail's rounds and the batch's round sizes go to the host.
__global__ void __launch_bounds__(256) k_batch_finish(BoxDesc *boxes, PW W, int64_t NP,
                                                      uint32_t t0, int n,
                                                      unsigned long long *to_host) {
  if (blockIdx.x == 0 && threadIdx.x < 6) to_host[threadIdx.x] = W.hole_top[threadIdx.x];
  // a wavefront keeps its count while its tests are one box's (they are in
  // box order): an add each 64 tests took 31 us for 50000 tests of one box
  int now = -1;
  int64_t sum = 0;
  for (int base = blockIdx.x * blockDim.x; base < n; base += gridDim.x * blockDim.x) {
    const int i = base + (int)threadIdx.x;
    int box = -1;
    int64_t q;
    if (i < n && W.thin[i]) box = pair_box(W, test_pair(W, NP, t0 + (uint32_t)i), &q);
    const uint64_t thin = __ballot(box >= 0);
    if (!thin) continue;
    const int lead = __shfl(box, __ffsll((long long)thin) - 1);
    const bool one = __ballot(box >= 0 && box != lead) == 0;
    if (!one || lead != now) {
      wave_flush_counts(boxes, (threadIdx.x & 63) == 0 ? now : -1, -sum, 0, 0);
      now = lead;
      sum = 0;
    }
    if (one) sum += __popcll(thin);
    else wave_flush_counts(boxes, box, -1, 0, 0);
  }
  wave_flush_counts(boxes, (threadIdx.x & 63) == 0 ? now : -1, -sum, 0, 0);
}

inline int parallel_init(ParallelWork &W, int n_box, int max_bin) {
  W.n_box = n_box;
  W.d.max_bin = max_bin;
  W.d.tab_classes = 1;
  if (hipHostMalloc((void **)&W.h_u32, 64 * sizeof(uint32_t)) != hipSuccess) return ERR_HIP;
  if (hipHostMalloc((void **)&W.h_u64, 8 * sizeof(unsigned long long)) != hipSuccess) return ERR_HIP;
  if (hipStreamCreate(&W.st2) != hipSuccess) return ERR_HIP;
  if (hipMalloc((void **)&W.pstat, 2 * sizeof(unsigned long long)) != hipSuccess) return ERR_HIP;
  if (hipMemset(W.pstat, 0, 2 * sizeof(unsigned long long)) != hipSuccess) return ERR_HIP;
  if (hipEventCreateWithFlags(&W.ev_fork, hipEventDisableTiming) != hipSuccess) return ERR_HIP;
  if (hipEventCreateWithFlags(&W.ev_join, hipEventDisableTiming) != hipSuccess) return ERR_HIP;
  return 0;
}

// the accelerated path's records, allocated when a step first has target slots
inline void parallel_free_records(ParallelWork &W) {
  PW &d = W.d;
  void *ptrs[] = {d.ev, d.q_vol, d.q, d.q_csrc, d.q_ctime, d.dup_top, d.rm_buf, d.rm_top};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  d.ev = nullptr;
  d.q = nullptr;
  d.q_vol = d.q_ctime = nullptr;
  d.q_csrc = nullptr;
  d.dup_top = d.rm_buf = d.rm_top = nullptr;
  d.acc_cap = d.pool_cap = d.rm_cap = 0;
}

inline int parallel_alloc_records(ParallelWork &W, int n_spec) {
  PW &d = W.d;
  const int64_t c = ACC_CAP, pc = (int64_t)ACC_CAP + DUP_CAP;
  PCHECK(pmalloc(&d.ev, c));
  PCHECK(pmalloc(&d.q, pc));
  PCHECK(pmalloc(&d.q_vol, (size_t)n_spec * pc));
  PCHECK(pmalloc(&d.q_csrc, (size_t)MAX_COMP * pc));
  PCHECK(pmalloc(&d.q_ctime, (size_t)MAX_COMP * pc));
  PCHECK(pmalloc(&d.dup_top, 1));
  PCHECK(pmalloc(&d.rm_buf, RM_CAP));
  PCHECK(pmalloc(&d.rm_top, 1));
  PCHECK(hipMemset(d.dup_top, 0, sizeof(int)));
  PCHECK(hipMemset(d.rm_top, 0, sizeof(int)));
  d.acc_cap = (int)c;
  d.pool_cap = (int)pc;
  d.rm_cap = RM_CAP;
  return 0;
}

inline void parallel_free_arrays(ParallelWork &W) {
  PW &d = W.d;
  void *ptrs[] = {d.key,  d.slot, d.terms, d.perm, d.tile_box, d.tile_start,
                  d.tiles_in_box, d.tile_first, d.hist, d.hist_scan, d.lstart, d.lcnt, d.live,
                  d.pair_n, d.pair_exc, d.acc, d.acc_scan, d.tp1, d.tp2, d.tid, d.pend, d.ev_t,
                  d.ev_p1, d.ev_p2, d.ev_box, d.ev_out, d.f_app, d.f_id, d.f_info, d.f_hole,
                  d.f_pend, d.s_pend, d.s_app, d.s_id, d.s_info, d.s_hole,
                  d.box_first,
                  d.holes, d.holes_sorted, d.cmp_lo, d.cmp_hi, d.cmp_head, d.acc_samp,
                  d.scan_part, W.sort_tmp, d.rc,
                  d.pair_acc, d.pair_accn, d.acc_exc, d.trec, d.tns, d.ev_rec,
                  d.hole_top, d.pend_k, d.tpair,
                  d.acap, d.arr_n, d.arr_head, d.ap_p, d.ap_t, d.ap_dep, d.ap_next, d.ap_top,
                  d.thin, d.minpend, d.minpend_next};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  parallel_free_records(W);
  int ks = d.K_stride;
  int64_t ps = d.P_stride;
  int tc = d.tab_classes, mb = d.max_bin;
  d = PW{};
  d.K_stride = ks;
  d.P_stride = ps;
  d.tab_classes = tc;
  d.max_bin = mb;
  W.sort_tmp = nullptr;
  W.sort_tmp_bytes = 0;
}

inline void parallel_free(ParallelWork &W) {
  parallel_free_arrays(W);
  if (W.h_u32) (void)hipHostFree(W.h_u32);
  if (W.h_u64) (void)hipHostFree(W.h_u64);
  W.h_u64 = nullptr;
  W.h_u32 = nullptr;
  if (W.ev_fork) (void)hipEventDestroy(W.ev_fork);
  if (W.ev_join) (void)hipEventDestroy(W.ev_join);
  if (W.st2) (void)hipStreamDestroy(W.st2);
  if (W.pstat) (void)hipFree(W.pstat);
  W.ev_fork = W.ev_join = nullptr;
  W.st2 = nullptr;
  W.pstat = nullptr;
}

// (re)allocate everything sized by particle capacities and the class count
inline int parallel_layout(ParallelWork &W, const Arrays &A, int n_box,
                           const std::vector<int64_t> &cap, int max_bin) {
  parallel_free_arrays(W);
  PW &d = W.d;
  d.max_bin = max_bin;
  d.K_stride = max_bin * d.tab_classes;
  d.P_stride = (int64_t)d.tab_classes * d.tab_classes * max_bin * max_bin;
  // the sort and the tail keep two ints per list of a box in LDS beside
  // their static LDS: refuse grids and class counts that do not fit
  {
    int dev = 0, lds_max = 0;
    PCHECK(hipGetDevice(&dev));
    PCHECK(hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    hipFuncAttributes fa_tail, fa_scatter;
    PCHECK(hipFuncGetAttributes(&fa_tail, reinterpret_cast<const void *>(&k_par_tail)));
    PCHECK(hipFuncGetAttributes(&fa_scatter, reinterpret_cast<const void *>(&k_par_scatter)));
    const size_t dyn = 2 * (size_t)d.K_stride * sizeof(int);
    if (fa_tail.sharedSizeBytes + dyn > (size_t)lds_max ||
        fa_scatter.sharedSizeBytes + dyn > (size_t)lds_max) {
      g_parallel_error = "parallel mode: " + std::to_string(max_bin) + " bins x " +
                         std::to_string(d.tab_classes) + " weight classes need " +
                         std::to_string(dyn) + " bytes of LDS per box list set, above the " +
                         std::to_string(lds_max) + " a workgroup has beside the kernels' own";
      return ERR_CAPACITY;
    }
  }
  const int64_t tc = A.total_cap;
  PCHECK(pmalloc(&d.key, tc));
  PCHECK(pmalloc(&d.slot, tc));
  PCHECK(pmalloc(&d.terms, tc));
  PCHECK(pmalloc(&d.perm, tc));
  // tiles over each box's capacity
  std::vector<int> tb, ts;
  std::vector<int64_t> hoff(n_box);
  W.tiles_in_box.assign(n_box, 0);
  int64_t H = 0;
  for (int b = 0; b < n_box; ++b) {
    int nt = (int)((cap[b] + TILE - 1) / TILE);
    if (nt < 1) nt = 1;
    W.tiles_in_box[b] = nt;
    for (int t = 0; t < nt; ++t) {
      tb.push_back(b);
      ts.push_back(t * TILE);
    }
    hoff[b] = (int64_t)tb.size() - nt;
    H += (int64_t)d.K_stride * nt;
  }
  W.n_tiles = (int)tb.size();
  W.H = H;
  PCHECK(pmalloc(&d.tile_box, tb.size()));
  PCHECK(pmalloc(&d.tile_start, ts.size()));
  PCHECK(pmalloc(&d.tiles_in_box, n_box));
  PCHECK(pmalloc(&d.tile_first, n_box));
  PCHECK(hipMemcpy(d.tile_box, tb.data(), tb.size() * sizeof(int), hipMemcpyHostToDevice));
  PCHECK(hipMemcpy(d.tile_start, ts.data(), ts.size() * sizeof(int), hipMemcpyHostToDevice));
  PCHECK(hipMemcpy(d.tiles_in_box, W.tiles_in_box.data(), n_box * sizeof(int), hipMemcpyHostToDevice));
  PCHECK(hipMemcpy(d.tile_first, hoff.data(), n_box * sizeof(int64_t), hipMemcpyHostToDevice));
  d.K_hist = d.K_stride;
  PCHECK(pmalloc(&d.hist, H));
  PCHECK(pmalloc(&d.hist_scan, H + 1));
  PCHECK(pmalloc(&d.lstart, (size_t)n_box * d.K_stride));
  PCHECK(pmalloc(&d.lcnt, (size_t)n_box * d.K_stride));
  PCHECK(pmalloc(&d.live, (size_t)n_box * d.K_stride));
  PCHECK(hipMemset(d.live, 0, sizeof(int) * (size_t)n_box * d.K_stride));
  PCHECK(pmalloc(&d.acap, (size_t)n_box * d.K_stride));
  PCHECK(pmalloc(&d.arr_n, (size_t)n_box * d.K_stride));
  PCHECK(hipMemset(d.arr_n, 0, sizeof(int) * (size_t)n_box * d.K_stride));
  PCHECK(pmalloc(&d.arr_head, (size_t)n_box * d.K_stride));
  W.NP = (int64_t)n_box * d.P_stride;
  PCHECK(pmalloc(&d.pair_n, W.NP + 1));
  PCHECK(pmalloc(&d.pair_exc, W.NP + 1));
  PCHECK(hipMemset(d.pair_n, 0, sizeof(uint32_t) * (W.NP + 1)));
  PCHECK(pmalloc(&d.pair_acc, W.NP));
  PCHECK(pmalloc(&d.pair_accn, W.NP + 1));
  PCHECK(pmalloc(&d.acc_exc, W.NP + 1));
  PCHECK(hipMemset(d.pair_accn, 0, sizeof(uint32_t) * (W.NP + 1)));
  PCHECK(pmalloc(&d.rc, RC_SIZE));
  PCHECK(hipMemset(d.rc, 0, sizeof(int) * RC_SIZE));
  d.pstat = W.pstat;
  PCHECK(pmalloc(&d.hole_top, 8));
  d.tail_rounds = d.hole_top + 1;
  d.rstat = d.hole_top + 2;
  const int64_t T = W.T_cap;
  PCHECK(pmalloc(&d.acc, T + 1));
  PCHECK(pmalloc(&d.acc_scan, T + 1));
  PCHECK(pmalloc(&d.tp1, T));
  PCHECK(pmalloc(&d.tp2, T));
  PCHECK(pmalloc(&d.tid, T));
  PCHECK(pmalloc(&d.pend, T));
  PCHECK(pmalloc(&d.ev_t, T));
  PCHECK(pmalloc(&d.ev_p1, T));
  PCHECK(pmalloc(&d.ev_p2, T));
  PCHECK(pmalloc(&d.ev_box, T));
  PCHECK(pmalloc(&d.ev_out, T));
  PCHECK(pmalloc(&d.trec, T));
  PCHECK(pmalloc(&d.pend_k, T));
  PCHECK(pmalloc(&d.tpair, T));
  PCHECK(pmalloc(&d.tns, T));
  PCHECK(pmalloc(&d.thin, T));
  PCHECK(pmalloc(&d.minpend, (size_t)n_box * d.K_stride));
  PCHECK(pmalloc(&d.minpend_next, (size_t)n_box * d.K_stride));
  // arrivals of one step: at most one per merge or copy, over every batch
  d.ap_cap = (uint32_t)std::min<int64_t>(2 * T + DUP_CAP, (int64_t)INT32_MAX / 2);
  d.ap_ovf = (int64_t)n_box * d.K_stride * A_MAX;
  if (d.ap_ovf + d.ap_cap > (int64_t)INT32_MAX) {
    g_parallel_error = "arrival pool larger than 2^31 entries";
    return ERR_CAPACITY;
  }
  PCHECK(pmalloc(&d.ap_p, d.ap_ovf + d.ap_cap));
  PCHECK(pmalloc(&d.ap_t, d.ap_ovf + d.ap_cap));
  PCHECK(pmalloc(&d.ap_dep, d.ap_ovf + d.ap_cap));
  PCHECK(pmalloc(&d.ap_next, d.ap_ovf + d.ap_cap));
  PCHECK(pmalloc(&d.ap_top, 1));
  PCHECK(pmalloc(&d.ev_rec, T));
  int **fl[] = {&d.f_app, &d.f_id, &d.f_info, &d.f_hole, &d.f_pend,
                &d.s_app, &d.s_id, &d.s_info, &d.s_hole, &d.s_pend};
  for (int **f : fl) PCHECK(pmalloc(f, T + 1));
  PCHECK(pmalloc(&d.box_first, n_box));
  int64_t total_cap = 0;
  for (int b = 0; b < n_box; ++b) total_cap += cap[b];
  W.hole_cap = total_cap + 1024;
  PCHECK(pmalloc(&d.holes, W.hole_cap));
  PCHECK(pmalloc(&d.holes_sorted, W.hole_cap));
  PCHECK(pmalloc(&d.cmp_lo, n_box));
  PCHECK(pmalloc(&d.acc_samp, 1));
  PCHECK(hipMemset(d.acc_samp, 0, sizeof(unsigned long long)));
  PCHECK(pmalloc(&d.cmp_hi, n_box));
  PCHECK(pmalloc(&d.cmp_head, n_box));
  // the chunk totals of the device-wide scans
  PCHECK(pmalloc(&d.scan_part, (size_t)SCAN_COLS * SCAN_MAX_BLOCKS));
  PCHECK(rocprim::radix_sort_keys(nullptr, W.sort_tmp_bytes, d.holes, d.holes_sorted,
                                  (unsigned)W.hole_cap, 0u, 64u, (hipStream_t)0));
  PCHECK(hipMalloc(&W.sort_tmp, W.sort_tmp_bytes));
  hipLaunchKernelGGL(k_init_slots, dim3((tc + 255) / 256), dim3(256), 0, 0, d.slot, tc);
  W.epoch = 0;
  PCHECK(hipGetLastError());
  PCHECK(hipDeviceSynchronize());
  return 0;
}

// more weight classes: the arrays go, so that nothing reads them with the new
// strides, and the next step lays them out again
inline int parallel_classes(ParallelWork &W, int n_box, int classes) {
  (void)n_box;
  parallel_free_arrays(W);
  W.d.tab_classes = classes;
  W.d.K_stride = W.d.max_bin * classes;
  W.d.P_stride = (int64_t)classes * classes * W.d.max_bin * W.d.max_bin;
  g_parallel_error = "";
  return 0;
}

// the sort of the step's keys into lists, and the pairs' test counts laid out
// in reference order; d.P_stride and W.NP are set for grids of mb_step bins
inline void parallel_sort_and_pairs(ParallelWork &W, const Arrays &A, BoxDesc *d_box, int n_box,
                                    hipStream_t st, double del_t, uint64_t seed, uint32_t step) {
  PW &d = W.d;
  const dim3 gt(W.n_tiles), bt(TILE_THREADS);
  // stable counting sort of the keys; the histogram spans the step's grid:
  // keys are below mb_step * classes
  d.K_hist = W.mb_step * d.tab_classes;
  PLAUNCH(W, "k_par_hist", k_par_hist, gt, bt, d.K_hist * sizeof(int), st, d_box, d);
  const int64_t nh = (int64_t)d.K_hist * W.n_tiles;
  scan_excl_sum(scan_job(d.hist, d.hist_scan, d.scan_part, nh), nh, st);
  hipLaunchKernelGGL(k_par_lists, dim3(n_box), dim3(256), 0, st, d_box, d);
  // the sentinel 2^key_bits - 1 lies above the keys
  int key_bits = 1;
  while ((1 << key_bits) <= d.K_hist) key_bits++;
  PLAUNCH(W, "k_par_scatter", k_par_scatter, gt, bt, 2 * d.K_stride * sizeof(int), st, d_box, d,
          key_bits);
  // Poisson test counts per bin pair
  PLAUNCH(W, "k_par_pairs", k_par_pairs, dim3((unsigned)((d.P_stride + 255) / 256), n_box),
          dim3(256), 0, st, d_box, A, d, del_t, seed, step);
  // both in one pass; each writes its total after the pair space
  ScanJob J = scan_job(d.pair_n, d.pair_exc, d.scan_part, W.NP);
  J.in[1] = d.pair_accn;
  J.out[1] = d.acc_exc;
  J.cols = 2;
  scan_excl_sum(J, W.NP, st);
  // the step's test count, its target slots and the first batch's bounds
  hipLaunchKernelGGL(k_batch_end, dim3(1), dim3(64), 0, st, d_box, d, n_box, W.NP, 0u,
                     (uint32_t)W.T_cap, (uint32_t)ACC_CAP, W.h_u32 + 4);
}

// the pair space of grids of up to mb bins
inline void parallel_pair_space(ParallelWork &W, int n_box, int mb) {
  W.mb_step = mb;
  W.d.max_bin = mb;
  W.d.P_stride = (int64_t)W.d.tab_classes * W.d.tab_classes * mb * mb;
  W.NP = (int64_t)n_box * W.d.P_stride;
}

// The whole parallel step.  The host waits twice: for the test counts, which
// size the claim rounds, and for the hole count, which sizes the compaction.
// A step that follows another with no call between that changes a box finds
// keys, terms and tables current: it launches straight through to the test
// counts on the last step's grids, and starts over from the keys only if a
// box turns out to need a new grid.  (About 35 dispatches a step; 83 with
// every pass a launch of its own and the checks for stale state in each
// step.)
inline int parallel_step(ParallelWork &W, const Arrays &A, BoxDesc *d_box, int n_box,
                         const std::vector<int64_t> &cap, int max_bin, hipStream_t st, int type,
                         double del_t, uint64_t seed, uint32_t step, int precision, double band,
                         int validation) {
  PW &d = W.d;
  const int want_terms = (precision != 0) ? 1 : 0;
  bool clean = W.clean_type == type && W.clean_terms == want_terms;
  W.clean_type = 0;  // set again at the end of a step that went through
  if (d.key == nullptr || d.K_stride != max_bin * d.tab_classes || W.NP != (int64_t)n_box * d.P_stride) {
    int e = parallel_layout(W, A, n_box, cap, max_bin);
    if (e) return e;
    hipLaunchKernelGGL(k_par_invalidate, dim3((n_box + 63) / 64), dim3(64), 0, st, d_box, n_box);
    clean = false;
  }
  const dim3 gb((n_box + 63) / 64), bb(64);
  const dim3 gt(W.n_tiles), bt(TILE_THREADS);
  d.tpair_ok = 0;  // built once the step's tests are laid out
  if (++W.tag == INT32_MAX) W.tag = 1;
  d.tag = W.tag;
  // 1. keys for boxes with a valid grid but stale keys, radius extremes for
  // unsorted boxes, the remake test, and keys again after a new grid
  if (!clean) {
    hipLaunchKernelGGL(k_par_zero_live, dim3(1, n_box), dim3(256), 0, st, d_box, d, n_box, 0);
    hipLaunchKernelGGL(k_par_rekey, gt, bt, 0, st, d_box, A, d, type, want_terms, 0);
    hipLaunchKernelGGL(k_par_finish_rekey, gb, bb, 0, st, d_box, n_box, type, want_terms, 0);
    hipLaunchKernelGGL(k_par_reset_minmax, gb, bb, 0, st, d_box, n_box);
    hipLaunchKernelGGL(k_par_minmax, gt, bt, 0, st, d_box, A, d);
  }
  hipLaunchKernelGGL(k_step_front, dim3(n_box), dim3(64), 0, st, d_box, A, d, clean ? W.NP : 0);
  if (clean) {
    // 2.-4. on the last step's grids; W.h_u32[9] tells whether they still hold
    parallel_sort_and_pairs(W, A, d_box, n_box, st, del_t, seed, step);
    PCHECK(hipStreamSynchronize(st));
    clean = W.h_u32[9] != BE_REGRID;
  }
  if (!clean) {
    if (++W.tag == INT32_MAX) W.tag = 1;
    d.tag = W.tag;
    hipLaunchKernelGGL(k_par_zero_live, dim3(1, n_box), dim3(256), 0, st, d_box, d, n_box, 1);
    hipLaunchKernelGGL(k_par_rekey, gt, bt, 0, st, d_box, A, d, type, 0, 1);
    hipLaunchKernelGGL(k_par_finish_rekey, gb, bb, 0, st, d_box, n_box, type, 0, 1);
    // The largest grid among the boxes this step: the pair space spans it
    // (not the allocation's max_bin) and the sort keys need only its bits.
    hipLaunchKernelGGL(k_max_nbin, dim3(1), dim3(256), 0, st, d_box, n_box, W.h_u32 + 12);
    PCHECK(hipStreamSynchronize(st));
    parallel_pair_space(W, n_box, std::max(1, std::min((int)W.h_u32[12], max_bin)));
    hipLaunchKernelGGL(k_batch_reset,
                       dim3((unsigned)(((int64_t)n_box * d.K_stride + 255) / 256)), dim3(256), 0,
                       st, d, n_box, W.NP, 0);
    // 2. majorant and pair tables (shared with the exact mode)
    const int mb = max_bin;
    hipLaunchKernelGGL(k_kbounds, dim3((mb * mb + 255) / 256, n_box), dim3(256), 0, st, d_box, A, type);
    hipLaunchKernelGGL(k_mark_bounds, gb, bb, 0, st, d_box, n_box, type);
    hipLaunchKernelGGL(k_pair_tables,
                       dim3((d.tab_classes * d.tab_classes * mb * mb + 255) / 256, n_box), dim3(256),
                       0, st, d_box, A);
    hipLaunchKernelGGL(k_mark_tables, gb, bb, 0, st, d_box, n_box);
    // 3. and 4.
    parallel_sort_and_pairs(W, A, d_box, n_box, st, del_t, seed, step);
    PCHECK(hipStreamSynchronize(st));
  }
  if (W.h_u32[9] == BE_TESTS) {
    g_parallel_error = "more than 2^32 - 1 tests in a step: reduce del_t or remake the grid";
    return ERR_CAPACITY;
  }
  const uint32_t T = W.h_u32[7];
  const uint32_t T_acc = W.h_u32[8];
  if (T_acc > 0 && d.ev == nullptr) {
    int e = parallel_alloc_records(W, A.n_spec);
    if (e) return e;
  }
  // every particle starts the step live: a fresh status epoch, and a clear
  // array when the 6-bit epoch wraps
  if (++W.epoch > 63) {
    W.epoch = 1;
    hipLaunchKernelGGL(k_clear_status, dim3((unsigned)((A.total_cap + 255) / 256)), dim3(256), 0,
                       st, d.slot, A.total_cap);
  }
  d.epoch = W.epoch;
  // 5. tests, claims and merges, in batches of T_cap tests.  The rounds of
  // a batch are launched without reading their counts back: each kernel
  // reads them from d.rc and a round that does not run finds a zero count.
  // Grids are sized from the previous batch's counts, and the kernels stride
  // over any excess.
  int64_t n_holes = 0;
  for (uint32_t t0 = 0; t0 < T;) {
    uint32_t t1, a0, a1;
    const bool first = t0 == 0;
    if (!first) {
      // the batch ends where its target slots would overflow the records
      hipLaunchKernelGGL(k_batch_end, dim3(1), dim3(64), 0, st, d_box, d, n_box, W.NP, t0,
                         (uint32_t)W.T_cap, (uint32_t)d.acc_cap, W.h_u32 + 4);
      PCHECK(hipStreamSynchronize(st));
    }
    t1 = W.h_u32[4];
    a0 = W.h_u32[5];
    a1 = W.h_u32[6];
    const int n_acc = (int)(a1 - a0);
    const int n_batch = (int)(t1 - t0);
    const uint32_t batch_t0 = t0;
    t0 = t1;
    if (first) {
      // the batch's counts, and the test-to-pair table when the step is one batch
      const int table = (int64_t)T <= W.T_cap ? 1 : 0;
      hipLaunchKernelGGL(k_expand_pairs, dim3(table ? (unsigned)((W.NP + 255) / 256) : 1u),
                         dim3(256), 0, st, d, W.NP, table, n_batch);
      d.tpair_ok = table;
    } else {
      hipLaunchKernelGGL(k_batch_reset,
                         dim3((unsigned)(((int64_t)n_box * d.K_stride + 255) / 256)), dim3(256), 0,
                         st, d, n_box, W.NP, n_batch);
    }
    const uint32_t *pend = nullptr;
    // a grid for at most `bound` items, `per` a workgroup, sized from the
    // last batch's count with a margin (the kernels stride over any excess)
    auto grid = [](int64_t bound, int64_t last, int per) -> unsigned {
      int64_t want = last >= 0 ? last + last / 4 + 1024 : bound;
      if (want > bound) want = bound;
      return (unsigned)std::max<int64_t>(1, (want + per - 1) / per);
    };
    for (int round = 0; round < PAR_ROUNDS; ++round) {
      // a later round runs only while at most half of the batch is pending
      const int nb = round == 0 ? n_batch : n_batch / 2;  // its largest test count
      if (nb <= 0) break;  // a batch of one test has no second round
      const unsigned g_n = round == 0 ? (unsigned)((nb + 255) / 256) : grid(nb, W.est[1], 256);
      const unsigned g_e = grid(nb, W.est[round == 0 ? 0 : 2], 256);
      W.rid++;
      // the target visits run on the second stream beside the per-set tests
      // (disjoint slots; both only claim with atomics)
      if (n_acc > 0) {
        PCHECK(hipEventRecord(W.ev_fork, st));
        PCHECK(hipStreamWaitEvent(W.st2, W.ev_fork, 0));
        W.tst = W.st2;
        const unsigned g_a = pend ? grid(nb, W.est[1], 64) : (unsigned)((n_acc + ACC_LANES - 1) / ACC_LANES);
        PLAUNCH(W, "k_par_acc_tests", k_par_acc_tests, dim3(g_a), dim3(64), 0, W.st2,
                d_box, A, d, n_box, type, seed, step, batch_t0, pend, del_t, a0, n_acc);
        W.tst = nullptr;
        PCHECK(hipEventRecord(W.ev_join, W.st2));
      }
      if (round == 0)
        PLAUNCH(W, "k_par_tests", k_par_tests<false>, dim3(g_n), dim3(256), 0, st, d_box, A, d,
                n_box, type, seed, step, batch_t0, pend, precision, band, validation);
      else
        PLAUNCH(W, "k_par_tests", k_par_tests<true>, dim3(g_n), dim3(256), 0, st, d_box, A, d,
                n_box, type, seed, step, batch_t0, pend, precision, band, validation);
      if (n_acc > 0) PCHECK(hipStreamWaitEvent(st, W.ev_join, 0));
      scan_excl_sum(scan_job(d.acc, d.acc_scan, d.scan_part, 0, d.rc + RC_N, d.rc + RC_E), nb, st,
                    GatherEvents{d});
      hipLaunchKernelGGL(k_par_resolve, dim3(g_e), dim3(256), 0, st, d_box, A, d, n_box, seed, step);
      {
        // the winners' ranks: the flag arrays in one pass
        const int *fs[4] = {d.f_app, d.f_id, d.f_info, d.f_hole};
        int *ss[4] = {d.s_app, d.s_id, d.s_info, d.s_hole};
        ScanJob J = scan_job(fs[0], ss[0], d.scan_part, 0, d.rc + RC_E);
        for (int q = 1; q < 4; ++q) {
          J.in[q] = (const uint32_t *)fs[q];
          J.out[q] = (uint32_t *)ss[q];
        }
        J.cols = 4;
        scan_excl_sum(J, nb, st);
      }
      // one wavefront per event, a few events each: most have no long chain
      if (n_acc > 0)
        hipLaunchKernelGGL(k_par_apply_chains, dim3(std::min(grid(nb, W.est[round == 0 ? 0 : 2], 16), 4096u)),
                           dim3(256), 0, st, d_box, A, d, (int)W.rid);
      PLAUNCH(W, "k_par_apply", k_par_apply, dim3(g_e), dim3(256), 0, st, d_box, A, d,
              n_box, seed, step, type, want_terms, (int)W.rid);
      hipLaunchKernelGGL(k_par_settle, dim3(g_n), dim3(256), 0, st, d_box, d, n_box, (int)W.rid);
      scan_excl_sum(scan_job(d.f_pend, d.s_pend, d.scan_part, 0, d.rc + RC_N), nb, st,
                    GatherPending{d, W.NP});
      hipLaunchKernelGGL(k_round_end, dim3(n_box), dim3(PREFIX_THREADS), 0, st, d, n_batch, round);
      std::swap(d.minpend, d.minpend_next);
      // the next round and the tail read the pending tests from d.pend: the
      // tests kernels copy them into tid before the round writes d.pend
      pend = d.pend;
    }
    // the rest per box, one workgroup each
    PLAUNCH(W, "k_par_tail", k_par_tail, dim3(n_box), dim3(TAIL_THREADS),
            2 * d.K_stride * sizeof(int), st, d_box, A, d,
            n_box, d.pend, type, seed, step, precision, band, del_t, a0,
            want_terms, (int)W.rid + 1, d.tail_rounds, batch_t0);
    // the holes, the tail's rounds and the batch's round sizes, to the host
    hipLaunchKernelGGL(k_batch_finish, dim3(std::min((n_batch + 255) / 256, 64)), dim3(256), 0, st, d_box, d,
                       W.NP, batch_t0, n_batch, W.h_u64);
    PCHECK(hipStreamSynchronize(st));
    n_holes = (int64_t)W.h_u64[0];
    W.n_tail_rounds += (int64_t)W.h_u64[1];
    for (int q = 0; q < 4; ++q) W.est[q] = (int64_t)W.h_u64[2 + q];
    W.rid += (int64_t)W.h_u64[1] + 2;  // past every round id the tail used
  }
  // 6. compaction
  if (n_holes > 0) {
    if (n_holes <= FEW_HOLES) {
      hipLaunchKernelGGL(k_compact_few, dim3(1), dim3(1024), 0, st, d_box, d, n_box, (int)n_holes);
    } else {
      PCHECK(rocprim::radix_sort_keys(W.sort_tmp, W.sort_tmp_bytes, d.holes, d.holes_sorted,
                                      (unsigned)n_holes, 0u, 64u, st));
      hipLaunchKernelGGL(k_compact_ranges, gb, bb, 0, st, d_box, d, n_box, (int)n_holes);
    }
    PLAUNCH(W, "k_par_compact", k_compact_move, dim3((unsigned)((n_holes + 255) / 256)), dim3(256),
            0, st, d_box, A, d, (int)n_holes);
  }
  hipLaunchKernelGGL(k_step_end, dim3(n_box), dim3(256), 0, st, d_box, d, n_holes > 0 ? 1 : 0);
  PCHECK(hipGetLastError());
  W.clean_type = type;
  W.clean_terms = want_terms;
  return 0;
}

}  // namespace pmc
