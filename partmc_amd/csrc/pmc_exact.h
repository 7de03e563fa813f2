// pmc_exact.h -- majorant and pair tables, and the exact sequential-order
// sweep (the lists it walks are made in pmc_prepare.h).
//
// The exact sweep replays mc_coag's loop order (src/coagulation.F90:74-94)
// inside one wavefront per box, and speculates on the state not changing:
//   - the lanes take the next 64 occupied bin pairs and draw their counts;
//     the pairs up to the first that changes the box stand, the rest are
//     drawn again on the lists as it left them;
//   - the tests of a pair are evaluated SWEEP_TESTS at a time, two lanes a
//     test, and stand up to the first accepted one;
//   - that one is merged by the whole wavefront with the reference's
//     swap-last bookkeeping.
// With the same per-site Philox streams as the oracle, the resulting
// integer state is bit-identical.
#pragma once

#include "pmc_state.h"
#include "pmc_prepare.h"

namespace pmc {

// ------------------------------------------------------------ helpers
// Species are read SPEC_CHUNK at a time, the loads of a chunk issued
// before any is used (index clamped to the last species): a load in the
// body of a loop with a runtime count costs one memory round trip each.
// Sums run in species order, as one at a time would.
constexpr int SPEC_CHUNK = 4;

__device__ inline double particle_volume(const Arrays &A, int64_t p) {
  const int ns = A.n_spec;
  double v = 0.0;
  for (int s0 = 0; s0 < ns; s0 += SPEC_CHUNK) {
    double x[SPEC_CHUNK];
#pragma unroll
    for (int u = 0; u < SPEC_CHUNK; ++u)
      x[u] = A.vol[(int64_t)(s0 + u < ns ? s0 + u : ns - 1) * A.total_cap + p];
#pragma unroll
    for (int u = 0; u < SPEC_CHUNK; ++u)
      if (s0 + u < ns) v += x[u];
  }
  return v;
}

__device__ inline double particle_density(const Arrays &A, int64_t p) {
  const int ns = A.n_spec;
  double m = 0.0, v = 0.0;
  for (int s0 = 0; s0 < ns; s0 += SPEC_CHUNK) {
    double x[SPEC_CHUNK], rho[SPEC_CHUNK];
#pragma unroll
    for (int u = 0; u < SPEC_CHUNK; ++u) {
      const int s = s0 + u < ns ? s0 + u : ns - 1;
      x[u] = A.vol[(int64_t)s * A.total_cap + p];
      rho[u] = A.density[s];
    }
#pragma unroll
    for (int u = 0; u < SPEC_CHUNK; ++u)
      if (s0 + u < ns) m += x[u] * rho[u];
  }
  v = particle_volume(A, p);
  return m / v;
}

// kernel (src/coag_kernel.F90:83-125) times coag_num_conc_factor
// (num_conc_weighted_kernel, src/coag_kernel.F90:175-209), FP64 from the
// raw species volumes.
__device__ inline int weighted_kernel64(const Arrays &A, const Weights &w,
                                        const Env &env, int type, int64_t p1,
                                        int64_t p2, int c1, int c2, int cc,
                                        double *k_out) {
  double v1 = particle_volume(A, p1);
  double v2 = particle_volume(A, p2);
  double k = 0.0;
  int err = 0;
  switch (type) {
    case KERNEL_ADDITIVE: k = env.beta * (v1 + v2); break;
    case KERNEL_CONSTANT: k = C_BETA_0; break;
    case KERNEL_ZERO: k = 0.0; break;
    case KERNEL_BROWN: {
      double d1 = particle_density(A, p1);
      double d2 = particle_density(A, p2);
      k = kernel_brown_helper(v1, d1, v2, d2, env.temp, env.pressure);
      break;
    }
    case KERNEL_SEDI: err = kernel_sedi_helper(v1, v2, &k); break;
    default: err = 200724934;
  }
  double r1 = vol2rad(v1);
  double r2 = vol2rad(v2);
  *k_out = k * coag_num_conc_factor(w, r1, r2, c1, c2, cc);
  return err;
}

// whole-record copy of particle slot `from` into slot `to`.  Fields are
// read in chunks before they are written: a store between two loads of
// the same arrays makes the second wait for the first, one memory round
// trip per field.
__device__ inline void copy_particle(const Arrays &A, int64_t from, int64_t to) {
  const int64_t tc = A.total_cap;
  for (int s0 = 0; s0 < A.n_spec; s0 += 8) {
    double x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s0 + j < A.n_spec) x[j] = A.vol[(int64_t)(s0 + j) * tc + from];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s0 + j < A.n_spec) A.vol[(int64_t)(s0 + j) * tc + to] = x[j];
  }
  const double vtot = A.vtot[from];
  const int64_t id = A.id[from];
  const int group = A.group[from], klass = A.klass[from], nprim = A.nprim[from];
  const int nco = A.ncomp[from];
  const double least = A.least[from], greatest = A.greatest[from];
  const int fb = A.fwd_bin[from], fc = A.fwd_class[from], fi = A.fwd_idx[from];
  A.vtot[to] = vtot;
  A.id[to] = id;
  A.group[to] = group;
  A.klass[to] = klass;
  A.nprim[to] = nprim;
  A.ncomp[to] = nco;
  A.least[to] = least;
  A.greatest[to] = greatest;
  A.fwd_bin[to] = fb;
  A.fwd_class[to] = fc;
  A.fwd_idx[to] = fi;
  for (int c0 = 0; c0 < nco; c0 += 10) {  // entries past n_comp are never read
    int cs[10];
    double ct[10];
#pragma unroll
    for (int j = 0; j < 10; ++j) {
      if (c0 + j < nco) {
        cs[j] = A.csrc[comp_at(from, c0 + j)];
        ct[j] = A.ctime[comp_at(from, c0 + j)];
      }
    }
#pragma unroll
    for (int j = 0; j < 10; ++j) {
      if (c0 + j < nco) {
        A.csrc[comp_at(to, c0 + j)] = cs[j];
        A.ctime[comp_at(to, c0 + j)] = ct[j];
      }
    }
  }
}

// ------------------------------------------------------------- k bounds
// est_k_minmax_binned_unweighted / est_k_minmax_for_bin_unweighted
// (src/coag_kernel.F90:253-341): one thread per (box, b1, b2).  Bounds
// are recomputed only after a new grid (or kernel type), as in the
// reference where env changes do not invalidate them (:64-70).
__global__ void k_kbounds(BoxDesc *boxes, Arrays A, int type) {
  const int box = blockIdx.y;
  BoxDesc *B = &boxes[box];
  if (B->error || (B->bounds_valid && B->bounds_kernel == type)) return;
  const int nb = B->n_bin;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= nb * nb) return;
  const int b1 = idx % nb + 1, b2 = idx / nb + 1;
  const double *edges = A.edges + (int64_t)box * (A.max_bin + 1);
  double v1_low = rad2vol(edges[b1 - 1]);
  double v1_high = rad2vol(edges[b1]);
  double v2_low = rad2vol(edges[b2 - 1]);
  double v2_high = rad2vol(edges[b2]);
  double kmin = 0.0, kmax = 0.0;
  Env env = B->env;
  for (int i = 1; i <= 3; ++i)
    for (int j = 1; j <= 3; ++j) {
      double v1 = interp_linear_disc(v1_low, v1_high, 3, i);
      double v2 = interp_linear_disc(v2_low, v2_high, 3, j);
      double a, b;
      int err = kernel_minmax(type, A.d_min, A.d_max, v1, v2, env, &a, &b);
      if (err) atomicExch(&B->error, err);
      if (i == 1 && j == 1) {
        kmin = a;
        kmax = b;
      } else {
        kmin = fmin(kmin, a);
        kmax = fmax(kmax, b);
      }
    }
  int64_t o = (int64_t)box * A.max_bin * A.max_bin + idx;
  A.kmin[o] = kmin;
  A.kmax[o] = kmax * 2.0;
}

__global__ void k_mark_bounds(BoxDesc *boxes, int n_box, int type) {
  int box = blockIdx.x * blockDim.x + threadIdx.x;
  if (box >= n_box) return;
  BoxDesc *B = &boxes[box];
  if (B->error) return;  // its bounds were not computed
  if (!B->bounds_valid || B->bounds_kernel != type) {
    B->bounds_valid = 1;
    B->bounds_kernel = type;
    B->tables_valid = 0;
  }
}

// coag_dest_class + max_coag_num_conc_factor per (c1, c2, b1, b2), times
// the unweighted k_max (mc_coag_for_bin, src/coagulation.F90:136-140).
// The reference evaluates these for every visited pair and step; they
// depend only on the grid and the weights, so they are tabled.
__global__ void k_pair_tables(BoxDesc *boxes, Arrays A) {
  const int box = blockIdx.y;
  BoxDesc *B = &boxes[box];
  if (B->error || B->tables_valid) return;
  const int nb = B->n_bin, nc = B->w.n_class;
  const int nn = nb * nb;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= nc * nc * nn) return;
  const int pair = idx % nn, cls = idx / nn;
  const int b2 = pair % nb + 1, b1 = pair / nb + 1;
  const int c2 = cls % nc + 1, c1 = cls / nc + 1;
  const double *edges = A.edges + (int64_t)box * (A.max_bin + 1);
  const double *centers = A.centers + (int64_t)box * A.max_bin;
  Weights w = B->w;
  int cc = coag_dest_class(w, centers, b1, c1, c2);
  double f_max = max_coag_num_conc_factor(w, edges, b1, b2, c1, c2, cc);
  double k_max = A.kmax[(int64_t)box * A.max_bin * A.max_bin + (b1 - 1) + nb * (b2 - 1)];
  int64_t o = (int64_t)box * A.tab_classes * A.tab_classes * A.max_bin * A.max_bin + idx;
  A.kw[o] = k_max * f_max;
  A.cc[o] = (int8_t)cc;
}

__global__ void k_mark_tables(BoxDesc *boxes, int n_box) {
  int box = blockIdx.x * blockDim.x + threadIdx.x;
  if (box >= n_box) return;
  if (!boxes[box].error) boxes[box].tables_valid = 1;  // else they were not computed
}

__device__ inline int64_t table_index(const Arrays &A, int box, int nb, int nc,
                                      int b1, int b2, int c1, int c2) {
  return (int64_t)box * A.tab_classes * A.tab_classes * A.max_bin * A.max_bin +
         (int64_t)((c1 - 1) * nc + (c2 - 1)) * nb * nb + (int64_t)(b1 - 1) * nb +
         (b2 - 1);
}

// --------------------------------------------------------- exact sweep
// A detached particle record, as aero_particle_t on the path.
// NS bounds the species it holds: the records of up to FEW_SPEC species keep
// their volumes in registers.
constexpr int FEW_SPEC = 4;
template <int NS>
struct RecN {
  double vol[NS];
  int64_t id;
  int group, klass, nprim, ncomp;
  int csrc[MAX_COMP];
  double ctime[MAX_COMP];
  double least, greatest;
};
using Rec = RecN<MAX_SPEC>;

struct ExactBox {
  const Arrays *A;
  BoxDesc *B;
  Tape *tape = nullptr;  // the box's tape when one records or replays, else null
  int box;
  int64_t base;
  int nb, nc;
  int *lstart, *llen, *lcap;
  uint64_t seed;
  uint32_t step;
  const double *edges;

  __device__ int key(int bin, int cls) const { return (bin - 1) + nb * (cls - 1); }
  __device__ int n_entry(int bin, int cls) const { return llen[key(bin, cls)]; }
  __device__ int entry(int bin, int cls, int i) const {  // 1-based domain
    return A->pool[lstart[key(bin, cls)] + i - 1];
  }

  __device__ void load(int dom0, Rec &r) const {
    int64_t p = base + dom0;
    for (int s = 0; s < A->n_spec; ++s) r.vol[s] = A->vol[(int64_t)s * A->total_cap + p];
    r.id = A->id[p];
    r.group = A->group[p];
    r.klass = A->klass[p];
    r.nprim = A->nprim[p];
    r.ncomp = A->ncomp[p];
    for (int c = 0; c < r.ncomp; ++c) {
      r.csrc[c] = A->csrc[comp_at(p, c)];
      r.ctime[c] = A->ctime[comp_at(p, c)];
    }
    r.least = A->least[p];
    r.greatest = A->greatest[p];
  }
  __device__ void store(int dom0, const Rec &r) const {
    int64_t p = base + dom0;
    double v = 0.0;
    for (int s = 0; s < A->n_spec; ++s) {
      A->vol[(int64_t)s * A->total_cap + p] = r.vol[s];
      v += r.vol[s];
    }
    A->vtot[p] = v;
    A->id[p] = r.id;
    A->group[p] = r.group;
    A->klass[p] = r.klass;
    A->nprim[p] = r.nprim;
    A->ncomp[p] = r.ncomp;
    for (int c = 0; c < r.ncomp; ++c) {
      A->csrc[comp_at(p, c)] = r.csrc[c];
      A->ctime[comp_at(p, c)] = r.ctime[c];
    }
    A->least[p] = r.least;
    A->greatest[p] = r.greatest;
  }
  __device__ double rec_volume(const Rec &r) const {
    double v = 0.0;
    for (int s = 0; s < A->n_spec; ++s) v += r.vol[s];
    return v;
  }
  __device__ double rec_radius(const Rec &r) const { return vol2rad(rec_volume(r)); }

  __device__ void add_info(int64_t id, int action, int64_t other) {
    int64_t k = B->n_info;
    if (k < B->info_cap) {
      A->info_id[B->info_off + k] = id;
      A->info_action[B->info_off + k] = action;
      A->info_other[B->info_off + k] = other;
    }
    B->n_info = k + 1;
  }

  // integer_varray_append with relocation when a list is full
  __device__ int list_append(int k, int val) {
    if (llen[k] == lcap[k]) {
      int ncap = lcap[k] * 2 + 8;
      if ((int64_t)B->pool_top + ncap > B->pool_half) return ERR_CAPACITY;
      int nstart = (int)(B->pool_off + (int64_t)B->pool_cur * B->pool_half + B->pool_top);
      for (int i = 0; i < llen[k]; ++i) A->pool[nstart + i] = A->pool[lstart[k] + i];
      lstart[k] = nstart;
      lcap[k] = ncap;
      B->pool_top += ncap;
    }
    A->pool[lstart[k] + llen[k]] = val;
    llen[k] += 1;
    return 0;
  }
  // integer_varray_remove_entry (1-based), src/integer_varray.F90:151-171
  __device__ void list_remove(int k, int index) {
    int n = llen[k];
    if (index < n) A->pool[lstart[k] + index - 1] = A->pool[lstart[k] + n - 1];
    A->pool[lstart[k] + n - 1] = 0;
    llen[k] = n - 1;
  }

  // aero_particle_array_remove_particle + integer_rmap2_remove
  // (src/aero_particle_array.F90:182-199, src/integer_rmap2.F90:197-246);
  // dom is 1-based.
  __device__ void remove(int dom) {
    int64_t pd = base + dom - 1;
    int r1_old = A->fwd_bin[pd], r2_old = A->fwd_class[pd], idx_old = A->fwd_idx[pd];
    int n_dom = B->n_part;
    int shifted = n_dom;
    int64_t ps = base + shifted - 1;
    if (shifted != dom) {
      int kf = key(A->fwd_bin[ps], A->fwd_class[ps]);
      A->pool[lstart[kf] + A->fwd_idx[ps] - 1] = dom;
      copy_particle(*A, ps, pd);  // particle record and forward maps
    }
    B->n_part = n_dom - 1;
    int kl = key(r1_old, r2_old);
    int idx_fix = llen[kl];
    int dom_fix = A->pool[lstart[kl] + idx_fix - 1];
    list_remove(kl, idx_old);
    if (idx_fix != idx_old) A->fwd_idx[base + dom_fix - 1] = idx_old;
  }

  // aero_sorted_add_particle (src/aero_sorted.F90:397-449) for a valid sort
  __device__ int add(const Rec &r) {
    if (B->n_part >= B->cap) return ERR_CAPACITY;
    int bin = bin_find_log(nb, B->log_lo, B->log_hi, rec_radius(r));
    int dom0 = B->n_part;
    store(dom0, r);
    B->n_part = dom0 + 1;
    if (bin < 1 || bin > nb) return 134572570;
    int k = key(bin, r.klass);
    int err = list_append(k, dom0 + 1);
    if (err) return err;
    A->fwd_bin[base + dom0] = bin;
    A->fwd_class[base + dom0] = r.klass;
    A->fwd_idx[base + dom0] = llen[k];
    return 0;
  }

  // integer_rmap2_change with the reference's range-1-only early return
  // (src/integer_rmap2.F90:136-191)
  __device__ int change(int dom, int bin, int cls) {
    int64_t pd = base + dom - 1;
    int r1_old = A->fwd_bin[pd], r2_old = A->fwd_class[pd];
    if (r1_old == bin) return 0;
    int idx_old = A->fwd_idx[pd];
    int kl = key(r1_old, r2_old);
    list_remove(kl, idx_old);
    if (idx_old <= llen[kl]) {
      int shifted = A->pool[lstart[kl] + idx_old - 1];
      A->fwd_idx[base + shifted - 1] = idx_old;
    }
    int kn = key(bin, cls);
    int err = list_append(kn, dom);
    if (err) return err;
    A->fwd_bin[pd] = bin;
    A->fwd_class[pd] = cls;
    A->fwd_idx[pd] = llen[kn];
    return 0;
  }

  __device__ int64_t new_id() {
    int64_t id = (B->next_id - 1) * B->id_stride + B->id_offset + 1;
    B->next_id += 1;
    return id;
  }

  // the same by the whole wavefront (a wave_fence follows before next_id is
  // read again)
  __device__ int64_t new_id_wave() {
    const int64_t next = B->next_id;
    if ((threadIdx.x & 63) == 0) B->next_id = next + 1;
    return (next - 1) * B->id_stride + B->id_offset + 1;
  }

  template <class S>
  __device__ int rand_group(S &s, const Weights &w, int cls, double r) const {
    double pdf[MAX_GROUP] = {1.0};  // one group: its pdf over the largest is 1
    for (int g = 0; w.n_group > 1 && g < w.n_group; ++g) {
      int idx = g + w.n_group * (cls - 1);
      pdf[g] = 1.0 / weight_nc(w.type[idx], w.mag[idx], w.expo[idx], r);
    }
    return sample_cts_pdf(s, w.n_group, pdf);
  }
};

// aero_particle_coagulate, src/aero_particle.F90:917-1033
__device__ inline int rec_coagulate(const ExactBox &E, Stream &s, const Rec &p1,
                                    const Rec &p2, Rec &out) {
  Rec o;
  for (int k = 0; k < E.A->n_spec; ++k) o.vol[k] = p1.vol[k] + p2.vol[k];
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
    int n1_new = prob_round(s, (double)p1.nprim / (double)(p1.nprim + p2.nprim) *
                                   (double)MAX_COMP);
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
  out = o;
  return 0;
}

// ---- a box's wavefront acting together
// One lane's writes before the other lanes' reads.  A wavefront's memory
// operations are carried out in program order, so this only keeps the
// compiler from reordering them: waiting for the stores (a workgroup-scope
// fence) costs a memory round trip each time.
__device__ inline void wave_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

// The value of one lane, the same lane for the whole wavefront: read into
// scalar registers, a few cycles where a shuffle through the LDS crossbar
// takes a hundred (two for a double): 2 steps of 20000 Brownian particles in
// the exact mode take 89.4 ms in place of 91.2.  Every lane of the wavefront
// is active.
__device__ inline int wave_value(int v, int lane) {
  return __builtin_amdgcn_readlane(v, __builtin_amdgcn_readfirstlane(lane));
}
__device__ inline int64_t wave_value(int64_t v, int lane) {
  const uint32_t lo = (uint32_t)wave_value((int)(uint32_t)v, lane);
  return ((int64_t)wave_value((int)(v >> 32), lane) << 32) | (int64_t)lo;
}
__device__ inline double wave_value(double v, int lane) {
  return __longlong_as_double(wave_value((int64_t)__double_as_longlong(v), lane));
}

// A call-site stream drawn by a whole wavefront: lane l holds block l, so 64
// blocks cost what one does on one lane.  Every lane calls uniform() and
// gets the same value.  With a tape, lane 0 draws.
struct WaveStream {
  Stream s;
  int at;       // next uniform of this lane set's 128
  double a, b;  // this lane's block

  __device__ inline void fill() {
    uint32_t o[4];
    philox4x32_10(s.c0, s.c1, s.c2, s.c3 | ((s.block + (threadIdx.x & 63)) & 0xFFFFFFu), s.k0,
                  s.k1, o);
    a = u52(o[0], o[1]);
    b = u52(o[2], o[3]);
    s.block += 64;
    at = 0;
  }
  __device__ inline void open(uint64_t seed, uint32_t box, uint32_t step, uint32_t site,
                              uint32_t ordinal, uint32_t kind, Tape *tape) {
    s.open(seed, box, step, site, ordinal, kind);
    s.tape = tape;
    a = b = 0.0;
    at = 0;
    if (!tape) fill();
  }
  __device__ inline double uniform() {
    if (s.tape) {
      double v = 0.0;
      if ((threadIdx.x & 63) == 0) v = s.uniform();
      return wave_value(v, 0);
    }
    if (at == 128) fill();
    const double v = wave_value((at & 1) ? b : a, at >> 1);
    ++at;
    return v;
  }
};

// ExactBox::remove by the whole wavefront, of the particle at entry idx of
// list kl: the moved particle's fields go through the lanes (a species or a
// component each), list fix-ups through lane 0.  Every value the bookkeeping
// needs is read before anything is written.  Returns the particle whose
// entry moved to idx (dom itself: none did).
__device__ inline int wave_remove(ExactBox &E, int dom, int kl, int idx) {
  const Arrays &A = *E.A;
  const int lane = threadIdx.x & 63;
  const int64_t tc = A.total_cap;
  const int n_dom = E.B->n_part;
  const int64_t pd = E.base + dom - 1, ps = E.base + n_dom - 1;
  const int n_kl = E.llen[kl], start_kl = E.lstart[kl];
  int dom_fix = A.pool[start_kl + n_kl - 1];
  const int fb = A.fwd_bin[ps], fc = A.fwd_class[ps], fi = A.fwd_idx[ps];
  const double x = lane < A.n_spec ? A.vol[(int64_t)lane * tc + ps] : 0.0;
  const int cs = lane < MAX_COMP ? A.csrc[comp_at(ps, lane)] : 0;
  const double ct = lane < MAX_COMP ? A.ctime[comp_at(ps, lane)] : 0.0;
  const double vtot = A.vtot[ps], least = A.least[ps], greatest = A.greatest[ps];
  const int64_t id = A.id[ps];
  const int group = A.group[ps], klass = A.klass[ps], nprim = A.nprim[ps], nco = A.ncomp[ps];
  const bool moved = n_dom != dom;
  if (moved && dom_fix == n_dom) dom_fix = dom;  // the last entry is the moved particle's
  if (moved) {
    if (lane < A.n_spec) A.vol[(int64_t)lane * tc + pd] = x;
    if (lane < nco) {
      A.csrc[comp_at(pd, lane)] = cs;
      A.ctime[comp_at(pd, lane)] = ct;
    }
  }
  if (lane == 0) {
    if (moved) {
      A.pool[E.lstart[E.key(fb, fc)] + fi - 1] = dom;
      A.vtot[pd] = vtot;
      A.id[pd] = id;
      A.group[pd] = group;
      A.klass[pd] = klass;
      A.nprim[pd] = nprim;
      A.ncomp[pd] = nco;
      A.least[pd] = least;
      A.greatest[pd] = greatest;
      A.fwd_bin[pd] = fb;
      A.fwd_class[pd] = fc;
      A.fwd_idx[pd] = fi;
    }
    E.B->n_part = n_dom - 1;
    if (idx < n_kl) A.pool[start_kl + idx - 1] = dom_fix;
    A.pool[start_kl + n_kl - 1] = 0;
    E.llen[kl] = n_kl - 1;
    if (idx != n_kl) A.fwd_idx[E.base + dom_fix - 1] = idx;
  }
  wave_fence();
  return idx != n_kl ? dom_fix : dom;
}

// What the accepted test knows of its two particles: their slots, the lists
// they were drawn from and at which entry, and their side of the kernel.
struct TestPair {
  int dom1, dom2, key1, key2, idx1, idx2;
  double v1, v2, r1, r2, rc, nc1, nc2, ncc;  // volumes, radii (rc: combined), weights
};

// coagulate_weighting + coagulate, src/coagulation.F90:810-985
// (dom1, dom2 1-based), with aero_particle_coagulate
// (src/aero_particle.F90:917-1033) and aero_sorted_add_particle
// (src/aero_sorted.F90:397-449), by the whole wavefront.  A merge is a chain
// of memory round trips and FP64 functions: the parents' fields are read
// together (a species or a component a lane), the radii and weights come
// from the test, and the merge stream's blocks are drawn at once.  7.4 us a
// merge (Brownian, 4 species); on one lane, with the three particles'
// records in private memory, 18.6.
__device__ inline int wave_coagulate(ExactBox &E, const Weights &w, WaveStream &s,
                                     const TestPair &T, int cc) {
  const Arrays &A = *E.A;
  BoxDesc *B = E.B;
  const int lane = threadIdx.x & 63, ns = A.n_spec;
  const int64_t tc = A.total_cap;
  const int64_t p1 = E.base + T.dom1 - 1, p2 = E.base + T.dom2 - 1;
  const int64_t id1 = A.id[p1], id2 = A.id[p2];
  const double x1 = lane < ns ? A.vol[(int64_t)lane * tc + p1] : 0.0;
  const double x2 = lane < ns ? A.vol[(int64_t)lane * tc + p2] : 0.0;
  int cs1 = 0, cs2 = 0;
  double ct1 = 0.0, ct2 = 0.0;
  if (lane < MAX_COMP) {
    cs1 = A.csrc[comp_at(p1, lane)];
    cs2 = A.csrc[comp_at(p2, lane)];
    ct1 = A.ctime[comp_at(p1, lane)];
    ct2 = A.ctime[comp_at(p2, lane)];
  }
  const int n1 = A.ncomp[p1], n2 = A.ncomp[p2], np1 = A.nprim[p1], np2 = A.nprim[p2];
  const double least = fmin(A.least[p1], A.least[p2]);
  const double greatest = fmax(A.greatest[p1], A.greatest[p2]);
  if (id1 == id2) return 371947172;
  // the merged volume's bin, which the random decisions do not change
  const double x = x1 + x2;
  double v = 0.0;
  for (int q = 0; q < ns; ++q) v += wave_value(x, q);
  const int bin = bin_find_log(E.nb, B->log_lo, B->log_hi, vol2rad(v));
  const int new_group = E.rand_group(s, w, cc, T.rc);
  const double nc_min = fmin(T.nc1, fmin(T.nc2, T.ncc));
  const bool remove_1 = s.uniform() < nc_min / T.nc1;
  const bool remove_2 = s.uniform() < nc_min / T.nc2;
  const bool create_new = s.uniform() < nc_min / T.ncc;
  bool id_1_lost, id_2_lost;
  if (create_new) {
    id_1_lost = false;
    id_2_lost = false;
    if (remove_1 && remove_2) {
      if (T.v1 > T.v2) id_2_lost = true;
      else id_1_lost = true;
    }
  } else {
    id_1_lost = remove_1;
    id_2_lost = remove_2;
  }
  int64_t info_other = 0;
  uint64_t take1 = 0, take2 = 0;  // components kept of each parent
  int n1_new = n1, n_out = n1 + n2;
  if (create_new) {
    if (np1 < n1) return 465791384;
    if (np2 < n2) return 465791385;
    if (n1 + n2 > MAX_COMP) {
      n1_new = prob_round(s, (double)np1 / (double)(np1 + np2) * (double)MAX_COMP);
      take1 = sample_mask(s, n1_new, n1);
      take2 = sample_mask(s, MAX_COMP - n1_new, n2);
      n_out = MAX_COMP;
    } else {
      take1 = (1ull << n1) - 1ull;
      take2 = (1ull << n2) - 1ull;
    }
    if (remove_1 && !id_1_lost) info_other = id1;
    else if (remove_2 && !id_2_lost) info_other = id2;
    else info_other = E.new_id_wave();
  }
  // removals from the larger index down; the first may move the second's entry
  int idx1 = T.idx1, idx2 = T.idx2;
  for (int q = 0; q < 2; ++q) {
    const bool second = (q == 0) == (T.dom2 > T.dom1);
    if (!(second ? remove_2 : remove_1)) continue;
    const int idx = second ? idx2 : idx1;
    const int fix = wave_remove(E, second ? T.dom2 : T.dom1, second ? T.key2 : T.key1, idx);
    if (fix == (second ? T.dom1 : T.dom2)) (second ? idx1 : idx2) = idx;
    if ((second ? id_2_lost : id_1_lost) && lane == 0) E.add_info(second ? id2 : id1, 2, info_other);
  }
  if (!create_new) {
    wave_fence();
    return 0;
  }
  const int dom0 = B->n_part;
  if (dom0 >= B->cap) return ERR_CAPACITY;
  const int64_t p = E.base + dom0;
  if (lane < ns) A.vol[(int64_t)lane * tc + p] = x;
  const uint64_t below = (1ull << lane) - 1ull;
  if (lane < MAX_COMP && ((take1 >> lane) & 1ull)) {
    const int c = __popcll(take1 & below);
    A.csrc[comp_at(p, c)] = cs1;
    A.ctime[comp_at(p, c)] = ct1;
  }
  if (lane < MAX_COMP && ((take2 >> lane) & 1ull)) {
    const int c = n1_new + __popcll(take2 & below);
    A.csrc[comp_at(p, c)] = cs2;
    A.ctime[comp_at(p, c)] = ct2;
  }
  int err = 0;
  if (lane == 0) {
    A.vtot[p] = v;
    A.id[p] = info_other;
    A.group[p] = new_group;
    A.klass[p] = cc;
    A.nprim[p] = np1 + np2;
    A.ncomp[p] = n_out;
    A.least[p] = least;
    A.greatest[p] = greatest;
    B->n_part = dom0 + 1;
    if (bin < 1 || bin > E.nb) {
      err = 134572570;
    } else {
      const int k = E.key(bin, cc);
      err = E.list_append(k, dom0 + 1);
      if (!err) {
        A.fwd_bin[p] = bin;
        A.fwd_class[p] = cc;
        A.fwd_idx[p] = E.llen[k];
      }
    }
  }
  wave_fence();
  return wave_value(err, 0);
}

// the copies of aero_state_dup_particle with random groups,
// src/aero_state.F90:488-539: n_copies - 1 more of the particle in slot dom
__device__ inline int exact_copies(ExactBox &E, const Weights &w, Stream &s, int dom,
                                   int n_copies) {
  for (int i_dup = 1; i_dup <= n_copies - 1; ++i_dup) {
    Rec np;
    E.load(dom - 1, np);
    np.id = E.new_id();
    np.group = E.rand_group(s, w, E.A->klass[E.base + dom - 1],
                            vol2rad(E.A->vtot[E.base + dom - 1]));
    int err = E.add(np);
    if (err) return err;
  }
  return 0;
}

// sample_source_particle, src/coagulation.F90:333-517 (one lane).  A dry run
// changes nothing: it ends with SOURCE_REMOVED where a source would go.
constexpr int SOURCE_REMOVED = -1;
__device__ inline int exact_sample_source(ExactBox &E, const Weights &w,
                                          const Env &env, const BrownAir &air, int type,
                                          uint32_t site,
                                          uint32_t ordinal, int bs, int cs,
                                          const Rec &target, double n_samp_mean,
                                          double accept_factor, bool dry, int *n_samp_out,
                                          int *n_coag_out, int *n_warn, Rec &source) {
  const int ns = E.A->n_spec;
  *n_samp_out = 0;
  *n_coag_out = 0;
  if (E.n_entry(bs, cs) == 0) return 0;
  Stream aps, smp, fin;
  aps.open(E.seed, E.box, E.step, site, ordinal, RNG_ACC_POISSON);
  smp.open(E.seed, E.box, E.step, site, ordinal, RNG_ACC_SAMPLE);
  fin.open(E.seed, E.box, E.step, site, ordinal, RNG_ACC_FINISH);
  aps.tape = smp.tape = fin.tape = E.tape;
  double nc_target = nc_at_radius(w, target.klass, E.rec_radius(target));
  int64_t target_id = target.id;
  int ct = target.klass;
  double nc_src_min = nc_at_radius(w, cs, E.edges[bs - 1]);
  double prm = nc_target / nc_src_min;
  if (!(prm <= 1.0)) return 653606684;
  int n_remove = rand_poisson(aps, prm * n_samp_mean);
  int n_extra = rand_poisson(aps, (1.0 - prm) * n_samp_mean);
  int n_total = n_remove + n_extra;
  int n_avg = 0, n_samp = 0;
  double prob_coag_tot = 0.0;
  double vol_sq[MAX_SPEC], vol_cv[MAX_SPEC];
  for (int k = 0; k < ns; ++k) {
    vol_sq[k] = 0.0;
    vol_cv[k] = 0.0;
  }
  for (int k = 0; k < ns; ++k) source.vol[k] = 0.0;
  source.id = 0;
  source.group = source.klass = source.nprim = source.ncomp = 0;
  for (int c = 0; c < MAX_COMP; ++c) {
    source.csrc[c] = 0;
    source.ctime[c] = 0.0;
  }
  source.least = source.greatest = 0.0;
  for (int i_samp = 1; i_samp <= n_total; ++i_samp) {
    if (E.n_entry(bs, cs) == 0) break;
    if (n_samp > n_remove && n_avg >= 2) {
      double cvmax = 0.0;
      for (int k = 0; k < ns; ++k) {
        double vm = source.vol[k] / (double)n_avg;
        if (vm > 0.0) vol_cv[k] = sqrt(vol_sq[k] / (double)n_avg - vm * vm) / vm;
        if (k == 0 || vol_cv[k] > cvmax) cvmax = vol_cv[k];
      }
      double m95 = cvmax / sqrt((double)n_avg) * student_t_95_coeff(n_avg);
      if (m95 < 0.1) break;
    }
    n_samp++;
    int i_unif = rand_int(smp, E.n_entry(bs, cs));
    int dom = E.entry(bs, cs, i_unif);
    Rec pi;
    E.load(dom - 1, pi);
    // the target is a detached copy (src/coagulation.F90:226-229): source
    // removals may move its slot, so the kernel is taken against the copy
    double k;
    int err = 0;
    {
      double v1 = E.rec_volume(pi), v2 = E.rec_volume(target);
      double kk = 0.0;
      err = 0;
      switch (type) {
        case KERNEL_ADDITIVE: kk = env.beta * (v1 + v2); break;
        case KERNEL_CONSTANT: kk = C_BETA_0; break;
        case KERNEL_ZERO: kk = 0.0; break;
        case KERNEL_BROWN: {
          double m1 = 0.0, m2 = 0.0;
          for (int q = 0; q < ns; ++q) {
            m1 += pi.vol[q] * E.A->density[q];
            m2 += target.vol[q] * E.A->density[q];
          }
          kk = brown_combine(brown_terms(air, v1, m1 / v1, env.temp),
                             brown_terms(air, v2, m2 / v2, env.temp));
          break;
        }
        case KERNEL_SEDI: err = kernel_sedi_helper(v1, v2, &kk); break;
        default: err = 200724934;
      }
      k = kk * coag_num_conc_factor(w, vol2rad(v1), vol2rad(v2), cs, ct, ct);
    }
    if (err) return err;
    double prob_coag = k * accept_factor;
    prob_coag_tot += prob_coag;
    if (smp.uniform() < prob_coag) {
      n_avg++;
      err = rec_coagulate(E, smp, source, pi, source);
      if (err) return err;
      for (int q = 0; q < ns; ++q) vol_sq[q] += pi.vol[q] * pi.vol[q];
      if (i_samp <= n_remove) {
        double nc_i = nc_at_radius(w, pi.klass, E.rec_radius(pi));
        double prob_remove_i = nc_target / nc_i;
        if (smp.uniform() < prob_remove_i / prm) {
          if (dry) return SOURCE_REMOVED;
          E.remove(dom);
          E.add_info(pi.id, 2, target_id);
        }
      }
    }
  }
  *n_samp_out = n_samp;
  if (n_avg == 0) return 0;
  double prob_coag_mean = prob_coag_tot / (double)n_samp;
  if (!(prob_coag_mean <= 1.0)) *n_warn = 1;
  int n_coag = rand_binomial(fin, n_total, prob_coag_mean);
  for (int q = 0; q < ns; ++q) source.vol[q] = source.vol[q] * ((double)n_coag / (double)n_avg);
  source.nprim = prob_round(fin, (double)source.nprim * ((double)n_coag / (double)n_avg));
  int n_comp = source.ncomp;
  int n_comp_new = source.nprim < MAX_COMP ? source.nprim : MAX_COMP;
  int sample[MAX_COMP];
  int cs_src[MAX_COMP];
  double ct_src[MAX_COMP];
  for (int c = 0; c < MAX_COMP; ++c) {
    cs_src[c] = source.csrc[c];
    ct_src[c] = source.ctime[c];
  }
  if (n_comp_new < n_comp) {
    sample_without_replacement(fin, n_comp_new, n_comp, sample);
    for (int i = 0; i < n_comp_new; ++i) {
      source.csrc[i] = cs_src[sample[i] - 1];
      source.ctime[i] = ct_src[sample[i] - 1];
    }
    source.ncomp = n_comp_new;
  } else if (n_comp < MAX_COMP) {
    int i_comp = 1;
    while (i_comp <= n_comp_new) {
      if (i_comp + n_comp <= n_comp_new) {
        for (int i = 1; i <= n_comp; ++i) {
          source.csrc[i_comp + i - 2] = cs_src[i - 1];
          source.ctime[i_comp + i - 2] = ct_src[i - 1];
        }
        i_comp += n_comp;
      } else {
        int sample_size = n_comp_new - i_comp + 1;
        sample_without_replacement(fin, sample_size, n_comp, sample);
        for (int i = 1; i <= sample_size; ++i) {
          source.csrc[i_comp + i - 2] = cs_src[sample[i - 1] - 1];
          source.ctime[i_comp + i - 2] = ct_src[sample[i - 1] - 1];
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

// coag_target_with_source, src/coagulation.F90:522-582, in two parts.  The
// merged target, its new bin and how many copies of it there are to be:
// nothing is changed.
__device__ inline int exact_target_merge(ExactBox &E, const Weights &w, Stream &s, const Rec &tp,
                                         const Rec &source, int cc, Rec &np, int *new_bin,
                                         int *n_copies) {
  const double old_nc = nc_at_radius(w, tp.klass, E.rec_radius(tp));
  int err = rec_coagulate(E, s, tp, source, np);
  if (err) return err;
  const double r = E.rec_radius(np);
  np.id = tp.id;
  np.group = E.rand_group(s, w, cc, r);
  np.klass = cc;
  *new_bin = bin_find_log(E.nb, E.B->log_lo, E.B->log_hi, r);
  if (*new_bin < 1 || *new_bin > E.nb) return 765620746;
  *n_copies = prob_round(s, old_nc / nc_at_radius(w, np.klass, r));
  return 0;
}

// ... and its place in the lists, with the copies (or without itself when
// there are none, src/aero_state.F90:488-539); the record is already in its
// slot
__device__ inline int exact_target_place(ExactBox &E, const Weights &w, Stream &s, int dom,
                                         int64_t target_id, int new_bin, int cc, int n_copies) {
  int err = E.change(dom, new_bin, cc);
  if (err) return err;
  if (n_copies == 0) {
    E.remove(dom);
    E.add_info(target_id, 4, 0);
  } else {
    err = exact_copies(E, w, s, dom, n_copies);
    if (err) return err;
  }
  return E.A->id[E.base + dom - 1] != target_id ? 654300924 : 0;
}

__device__ inline uint32_t pair_site(int nb, int nc, int b1, int b2, int c1, int c2) {
  return (uint32_t)((((c1 - 1) * nc + (c2 - 1)) * nb + (b1 - 1)) * nb + (b2 - 1));
}

// num_conc_weighted_kernel (as weighted_kernel64) of the two particles that
// a pair of neighbouring lanes holds, this lane's in slot p of class c_own:
// each lane forms its own particle's terms and both combine them (every
// combination is symmetric in its operands).  Every lane takes part; the
// value is the same on both.
struct PairSide {
  double v, r, nc;  // this lane's particle
  double rc, ncc;   // the combined radius and its weight
};
__device__ inline int weighted_kernel_pair(const Arrays &A, const Weights &w, const Env &env,
                                           const BrownAir &air, int type, int64_t p, int c_own,
                                           int cc, double *k_out, PairSide *side) {
  const double v = A.vtot[p];
  const double r = vol2rad(v);
  const double v_o = __shfl_xor(v, 1), r_o = __shfl_xor(r, 1);
  double k = 0.0;
  int err = 0;
  switch (type) {
    case KERNEL_ADDITIVE: k = env.beta * (v + v_o); break;
    case KERNEL_CONSTANT: k = C_BETA_0; break;
    case KERNEL_ZERO: k = 0.0; break;
    case KERNEL_BROWN: {
      const BrownTerms t = brown_terms(air, v, particle_density(A, p), env.temp);
      const BrownTerms o{r_o, __shfl_xor(t.diffus, 1), __shfl_xor(t.speedsq, 1),
                         __shfl_xor(t.deltasq, 1)};
      k = brown_combine(t, o);
      break;
    }
    case KERNEL_SEDI: {
      const double winf = fall_g(r), winf_o = __shfl_xor(winf, 1);
      double ec;
      err = effic(r, r_o, &ec);
      k = ec * C_PI * ((r + r_o) * (r + r_o)) * fabs(winf - winf_o);
      break;
    }
    default: err = 200724934;
  }
  const double nc = nc_at_radius(w, c_own, r), nc_o = __shfl_xor(nc, 1);
  const double rc = vol2rad(rad2vol(r) + rad2vol(r_o));
  const double ij_nc = nc_at_radius(w, cc, rc);
  *k_out = k * (nc * nc_o / fmin(nc, fmin(nc_o, ij_nc)));
  *side = PairSide{v, r, nc, rc, ij_nc};
  return err;
}

// Workspace of a box's sweep beside its static LDS: the lists' lengths,
// starts and capacities, the occupied bins of the two classes in hand and
// the weights at the bin edges.  It sits in LDS while it fits SWEEP_LDS
// bytes; beyond, the lists stay in global memory and the rest goes to the
// sort's scratch (free during a sweep).
constexpr int SWEEP_LDS = 49152;
constexpr int SWEEP_TESTS = 32;  // tests of a pair evaluated together, two lanes each
__host__ __device__ inline size_t sweep_bytes(int max_bin, int classes) {
  return sizeof(double) * (size_t)(max_bin + 1) * classes +
         sizeof(int) * ((size_t)3 * max_bin * classes + 2 * (size_t)max_bin);
}

// the bins of a class's occupied lists, in order, and `row` in any case
// (0: none); returns their number
__device__ inline int occupied_bins(const int *llen, int nb, int row, int *out) {
  const int lane = threadIdx.x & 63;
  int m = 0;
  for (int b0 = 0; b0 < nb; b0 += 64) {
    const int b = b0 + lane + 1;
    const bool in = b <= nb && (llen[b - 1] > 0 || b == row);
    const uint64_t mask = __ballot(in);
    if (in) out[m + __popcll(mask & ((1ull << lane) - 1ull))] = b;
    m += __popcll(mask);
  }
  return m;
}

// number of the sorted list's entries below x
__device__ inline int count_below(const int *v, int n, int x) {
  const int lane = threadIdx.x & 63;
  int m = 0;
  for (int i0 = 0; i0 < n; i0 += 64) m += __popcll(__ballot(i0 + lane < n && v[i0 + lane] < x));
  return m;
}

// The target loop of try_per_particle_coag (src/coagulation.F90:216-237)
// over the entries of list (bt, ct), from the last down, 64 at a time: each
// lane samples its target's source and forms the merged target as if the
// box did not change.  A merged target is written over the old one, and
// may join another list or leave copies at the ends of lists; none of that
// touches the source list, the entries still to come or their particles, so
// the lanes stand together up to the first that removes a source, removes
// its target, or adds to the source list.  That one runs alone, in order,
// and the lanes after it start again.  Returns whether anything changed.
// Up to 64 targets take about 110 us together; one lane walking them took
// 23 us each.
struct AccCounts {
  int64_t samp, coag, warn;
};

__device__ __noinline__ bool sweep_targets(ExactBox &E, const Weights &w, const Env &env,
                                           const BrownAir &air, int type, uint32_t site, int bt,
                                           int ct, int bs, int cs, double n_spt,
                                           double accept_factor, int cc, AccCounts *acc,
                                           int *err_out) {
  // what a lane's target needs: nothing, a merge that stands with the
  // others', or the box to itself (from the sampling, from the merge on, or
  // only to report an error)
  constexpr int T_NONE = 0, T_MERGE = 1, T_SAMPLE = 2, T_ALONE = 3, T_ERROR = 4;
  const int lane = threadIdx.x & 63;
  bool effect = false;
  int err = 0;
  for (int e0 = E.n_entry(bt, ct); e0 >= 1 && !err;) {
    const int e = e0 - lane;
    const bool mine = E.tape ? lane == 0 : e >= 1;
    int need = T_NONE, ns_ = 0, nco = 0, warn = 0, lerr = 0, dom = 1;
    int new_bin = bt, n_copies = 1;
    Rec target, source, np;
    Stream ts;
    if (mine) {
      dom = E.entry(bt, ct, e);
      E.load(dom - 1, target);
      if (E.tape) {
        need = T_SAMPLE;  // a tape's draws follow the call order
      } else {
        lerr = exact_sample_source(E, w, env, air, type, site, (uint32_t)e, bs, cs, target, n_spt,
                                   accept_factor, true, &ns_, &nco, &warn, source);
        if (lerr == SOURCE_REMOVED) {
          need = T_SAMPLE;
        } else if (lerr) {
          need = T_ERROR;
        } else if (nco > 0) {
          ts.open(E.seed, E.box, E.step, site, (uint32_t)e, RNG_ACC_TARGET);
          const int x = exact_target_merge(E, w, ts, target, source, cc, np, &new_bin, &n_copies);
          need = (x || n_copies == 0 || (new_bin == bs && cc == cs)) ? T_ALONE : T_MERGE;
        }
      }
    }
    const uint64_t alone = __ballot(need >= T_SAMPLE);
    const int stop = alone ? __ffsll((long long)alone) - 1 : 64;
    const bool stands = mine && lane < stop;
    if (stands) {
      acc->samp += ns_;
      acc->coag += nco;
      acc->warn += warn;
      if (need == T_MERGE) E.store(dom - 1, np);
    }
    wave_fence();
    // list changes in order, one lane at a time
    uint64_t lists = __ballot(stands && need == T_MERGE && (new_bin != bt || n_copies > 1));
    effect = effect || __ballot(stands && need == T_MERGE);
    while (lists && !err) {
      const int src = __ffsll((long long)lists) - 1;
      lists &= lists - 1;
      if (lane == src)
        lerr = exact_target_place(E, w, ts, dom, target.id, new_bin, cc, n_copies);
      wave_fence();
      err = wave_value(lerr, src);
    }
    if (stop < 64 && !err) {
      if (lane == stop) {
        if (need == T_SAMPLE) {
          warn = 0;
          lerr = exact_sample_source(E, w, env, air, type, site, (uint32_t)e, bs, cs, target,
                                     n_spt, accept_factor, false, &ns_, &nco, &warn, source);
        }
        if (!lerr && nco > 0) {
          dom = E.entry(bt, ct, e);  // removed sources may have moved it
          E.load(dom - 1, target);
          ts.open(E.seed, E.box, E.step, site, (uint32_t)e, RNG_ACC_TARGET);
          ts.tape = E.tape;
          lerr = exact_target_merge(E, w, ts, target, source, cc, np, &new_bin, &n_copies);
          // a target that grew out of the grid is stored before the error
          if (!lerr || lerr == 765620746) E.store(dom - 1, np);
          if (!lerr)
            lerr = exact_target_place(E, w, ts, dom, target.id, new_bin, cc, n_copies);
        }
        acc->samp += ns_;
        acc->coag += nco;
        acc->warn += warn;
      }
      wave_fence();
      err = wave_value(lerr, stop);
      effect = true;
    }
    e0 -= stop < 64 ? stop + 1 : 64;
  }
  *err_out = err;
  return effect;
}

// The sequential sweep: one 64-lane wavefront per box.  The box's descriptor
// and (SWEEP_LDS) its lists' bookkeeping live in LDS for its duration.  A
// pass over the next 64 pairs takes 2.5 us under flat weights and 9.5 under
// power weights (a pair at a time, most of it one lane's Poisson draw, took
// 4.5 and 5.3 us a pair); a batch of tests 4.2 us (additive) to 6.0
// (Brownian; 10.1 with a lane a test).
template <bool LDS>
__global__ void __launch_bounds__(64)
k_exact_sweep(BoxDesc *boxes, Arrays A, int type, double del_t, uint64_t seed, uint32_t step) {
  extern __shared__ double s_sweep[];
  const int box = blockIdx.x;
  const int lane = threadIdx.x;
  __shared__ BoxDesc s_box;
  for (int q = lane; q < (int)(sizeof(BoxDesc) / sizeof(int)); q += 64)
    ((int *)&s_box)[q] = ((const int *)&boxes[box])[q];
  __syncthreads();
  BoxDesc *B = &s_box;
  const int nb = B->n_bin, nc = B->w.n_class, K = nb * nc;
  // the workspace
  const int64_t kb = (int64_t)box * A.max_keys;
  double *nc_edge =
      LDS ? s_sweep : (double *)(A.sort_scratch + (int64_t)box * SORT_THREADS * A.max_keys);
  int *after = (int *)(nc_edge + (size_t)(A.max_bin + 1) * nc);
  int *L1 = after, *L2 = after + A.max_bin;
  int *llen = A.llen + kb, *lstart = A.lstart + kb, *lcap = A.lcap + kb;
  if (LDS) {
    int *at = L2 + A.max_bin;
    for (int k = lane; k < K; k += 64) {
      at[k] = llen[k];
      at[K + k] = lstart[k];
      at[2 * K + k] = lcap[k];
    }
    llen = at;
    lstart = at + K;
    lcap = at + 2 * K;
  }
  if (lane == 0) {
    B->step_samp = 0;
    B->step_coag = 0;
    B->part_steps += B->n_part;
  }
  const Weights &w = B->w;
  const Env env = B->env;
  // the target loop is called out of line: it gets copies, so that the
  // arguments and what the walk keeps stay in registers
  __shared__ Arrays s_A;
  for (int q = lane; q < (int)(sizeof(Arrays) / sizeof(int)); q += 64)
    ((int *)&s_A)[q] = ((const int *)&A)[q];
  ExactBox E;
  E.A = &A;
  E.B = B;
  E.tape = B->tape.mode != TAPE_OFF ? &B->tape : nullptr;
  E.box = box;
  E.base = B->off;
  E.nb = nb;
  E.nc = nc;
  E.lstart = lstart;
  E.llen = llen;
  E.lcap = lcap;
  E.seed = seed;
  E.step = step;
  E.edges = A.edges + (int64_t)box * (A.max_bin + 1);
  int64_t tot_samp = 0, tot_coag = 0, n_warn = 0;
  AccCounts acc{0, 0, 0};  // this lane's targets
  int err = 0;
  const bool run = !B->error;

  bool mono_dec = true;
  for (int i = 0; i < w.n_group * w.n_class; ++i) {
    if (w.type[i] == WEIGHT_POWER && w.expo[i] > 0.0) mono_dec = false;
  }
  if (run && mono_dec)
    for (int c = 1; c <= nc; ++c)
      for (int q = lane; q <= nb; q += 64)
        nc_edge[(c - 1) * (nb + 1) + q] = nc_at_radius(w, c, E.edges[q]);
  BrownAir air{0.0, 0.0};
  if (type == KERNEL_BROWN) air = brown_air(env.temp, env.pressure);
  __syncthreads();

  for (int c1 = 1; run && c1 <= nc && !err; ++c1)
    for (int c2 = 1; c2 <= c1 && !err; ++c2) {
      const bool tri = c1 == c2;  // b2 starts at b1
      int m1 = occupied_bins(llen + nb * (c1 - 1), nb, 0, L1);
      int m2 = tri ? m1 : occupied_bins(llen + nb * (c2 - 1), nb, 0, L2);
      const int *M2 = tri ? L1 : L2;
      wave_fence();
      int i0 = 0, j0 = 0;  // the next pair (L1[i0], M2[j0])
      while (i0 < m1 && !err) {
        // this lane's pair: the lane-th from there
        int i = i0, j = j0 + lane;
        while (i < m1 && j >= m2) {
          ++i;
          j += (tri ? i : 0) - m2;
        }
        const bool valid = i < m1 && (!E.tape || lane == 0);
        const int b1 = valid ? L1[i] : 1, b2 = valid ? M2[j] : 1;
        const int n1 = valid ? E.n_entry(b1, c1) : 0, n2 = valid ? E.n_entry(b2, c2) : 0;
        int kind = 0, n_samp = 0, cc = 1;  // kind 1 (2): targets in the first (second) list
        double k_max = 0.0, n_spt = 0.0;
        if (valid && n2 > 0) {
          const int64_t ti = table_index(A, box, nb, nc, b1, b2, c1, c2);
          cc = A.cc[ti];
          k_max = A.kw[ti];
          // try_per_particle_coag, src/coagulation.F90:150-241
          if (mono_dec) {
            const double a1 = nc_edge[(c1 - 1) * (nb + 1) + b1 - 1];
            const double a2 = nc_edge[(c1 - 1) * (nb + 1) + b1];
            const double d1 = nc_edge[(c2 - 1) * (nb + 1) + b2 - 1];
            const double d2 = nc_edge[(c2 - 1) * (nb + 1) + b2];
            const double nc1_min = fmin(a1, a2), nc1_max = fmax(a1, a2);
            const double nc2_min = fmin(d1, d2), nc2_max = fmax(d1, d2);
            int bt = 0, bs = 0, n_src = 0;
            if (nc1_max < nc2_min && cc == c1) {
              kind = 1; bt = b1; bs = b2; n_src = n2;
            }
            if (nc2_max < nc1_min && cc == c2) {
              kind = 2; bt = b2; bs = b1; n_src = n1;
            }
            if (kind) {
              n_spt = k_max * del_t * (double)n_src;
              bool ok = n_spt >= 1.0;
              if (ok) {
                const double min_tv = rad2vol(E.edges[bt - 1]);
                const double max_new = min_tv + rad2vol(E.edges[bs]) * n_spt;
                ok = !(max_new / min_tv > 1.5);
              }
              if (!ok) kind = 0;
            }
          }
          if (!kind) {
            // compute_n_samp, src/coagulation.F90:648-702
            const double n_possible = (tri && b1 == b2) ? (double)n1 * ((double)n2 - 1.0) / 2.0
                                                        : (double)n1 * (double)n2;
            Stream ps;
            ps.open(seed, box, step, pair_site(nb, nc, b1, b2, c1, c2), 0, RNG_POISSON);
            ps.tape = E.tape;
            n_samp = rand_poisson(ps, k_max * del_t * n_possible);
          }
        }
        const uint64_t vm = __ballot(valid);
        if (!vm) break;  // no pair left (the second class may have no particle)
        uint64_t todo = __ballot(kind != 0 || n_samp > 0);
        bool changed = false;
        int at = 63 - __clzll((long long)vm);  // the last pair settled by this pass
        while (todo && !changed && !err) {
          const int src = __ffsll((long long)todo) - 1;
          todo &= todo - 1;
          const int p_b1 = wave_value(b1, src), p_b2 = wave_value(b2, src);
          const int p_cc = wave_value(cc, src);
          const int p_kind = wave_value(kind, src);
          const double p_kmax = wave_value(k_max, src);
          const uint32_t site = pair_site(nb, nc, p_b1, p_b2, c1, c2);
          const double accept_factor = 1.0 / p_kmax;
          if (p_kind) {
            const double p_spt = wave_value(n_spt, src);
            const int bt = p_kind == 1 ? p_b1 : p_b2, ct = p_kind == 1 ? c1 : c2;
            const int bs = p_kind == 1 ? p_b2 : p_b1, cs = p_kind == 1 ? c2 : c1;
            if (lane == 0) B->n_accel_pairs += 1;
            ExactBox E2 = E;
            E2.A = &s_A;
            const Env env2 = env;
            const BrownAir air2 = air;
            AccCounts acc2{0, 0, 0};
            int err2 = 0;
            const bool effect = sweep_targets(E2, w, env2, air2, type, site, bt, ct, bs, cs, p_spt,
                                              accept_factor, p_cc, &acc2, &err2);
            acc.samp += acc2.samp;
            acc.coag += acc2.coag;
            acc.warn += acc2.warn;
            err = err2;
            if (effect) {
              changed = true;
              at = src;
            }
            continue;
          }

          // per_set_coag, src/coagulation.F90:587-645
          const bool same = tri && p_b1 == p_b2;
          const int ns_pair = wave_value(n_samp, src);
          const int key1 = E.key(p_b1, c1), key2 = E.key(p_b2, c2);
          if (lane == 0) tot_samp += ns_pair;
          int t = 1;
          while (t <= ns_pair && !err) {
            const int l1 = llen[key1], l2 = llen[key2];
            if ((l1 < 2 && same) || l1 < 1 || l2 < 1) break;
            // speculative batch: a pair of lanes takes test t + lane / 2 (one
            // test at a time on a tape, whose draws follow the call order)
            const int tj = t + (lane >> 1);
            const bool mine = tj <= ns_pair && (!E.tape || lane < 2);
            double u0 = 0.0, u1 = 0.0, u2 = 0.0;
            if (E.tape) {
              Stream ts;
              ts.open(seed, box, step, site, (uint32_t)(t - 1), RNG_TEST);
              ts.tape = E.tape;
              if (lane == 0) {
                u0 = ts.uniform();
                u1 = ts.uniform();
                u2 = ts.uniform();
              }
              u0 = wave_value(u0, 0);
              u1 = wave_value(u1, 0);
              u2 = wave_value(u2, 0);
            } else {
              // the test's three uniforms: block 0 on the even lane, block 1
              // on the odd one
              Stream ts;
              ts.open(seed, box, step, site, (uint32_t)(tj - 1), RNG_TEST);
              uint32_t o[4];
              philox4x32_10(ts.c0, ts.c1, ts.c2, ts.c3 | (uint32_t)(lane & 1), ts.k0, ts.k1, o);
              const double a = u52(o[0], o[1]), b = u52(o[2], o[3]);
              const double a_o = __shfl_xor(a, 1), b_o = __shfl_xor(b, 1);
              u0 = (lane & 1) ? a_o : a;
              u1 = (lane & 1) ? b_o : b;
              u2 = (lane & 1) ? a : a_o;
            }
            const int d1 = (int)(u0 * (double)l1) % l1 + 1;
            int d2;
            if (same) {
              d2 = (int)(u1 * (double)(l2 - 1)) % (l2 - 1) + 1;
              if (d2 == d1) d2 = l2;
            } else {
              d2 = (int)(u1 * (double)l2) % l2 + 1;
            }
            const int dom = A.pool[(lane & 1) ? lstart[key2] + d2 - 1 : lstart[key1] + d1 - 1];
            double k;
            PairSide side;
            const int lerr = weighted_kernel_pair(A, w, env, air, type, E.base + dom - 1,
                                                  (lane & 1) ? c2 : c1, p_cc, &k, &side);
            const double p = k * accept_factor;
            const bool warn = mine && !(p <= 1.0);
            const bool accept = mine && (u2 < p || lerr != 0);
            const uint64_t am = __ballot(accept);
            const int first = am ? (__ffsll((long long)am) - 1) & ~1 : 64;
            // warnings of the tests that happened (one lane of each pair)
            const uint64_t wm = __ballot(warn && !(lane & 1) && lane <= first);
            n_warn += __popcll(wm);
            if (first == 64) {
              t += E.tape ? 1 : SWEEP_TESTS;
              continue;
            }
            err = wave_value(lerr, first);
            if (err) break;
            const int f2 = first + 1, tt = t + (first >> 1);
            const TestPair T{wave_value(dom, first), wave_value(dom, f2), key1, key2,
                             wave_value(d1, first), wave_value(d2, first),
                             wave_value(side.v, first), wave_value(side.v, f2),
                             wave_value(side.r, first), wave_value(side.r, f2),
                             wave_value(side.rc, first), wave_value(side.nc, first),
                             wave_value(side.nc, f2), wave_value(side.ncc, first)};
            WaveStream ms;
            ms.open(seed, box, step, site, (uint32_t)(tt - 1), RNG_MERGE, E.tape);
            err = wave_coagulate(E, w, ms, T, p_cc);
            if (lane == 0) tot_coag += 1;
            changed = true;
            at = src;
            t = tt + 1;
          }
        }
        // go on after the last settled pair, on the lists as they are now
        const int a_i = wave_value(i, at), a_j = wave_value(j, at);
        if (changed) {
          const int row = L1[a_i], col = M2[a_j];
          wave_fence();
          // the reference tests the first list's length at the start of its
          // row only: a row emptied within is finished
          m1 = occupied_bins(llen + nb * (c1 - 1), nb, row, L1);
          m2 = tri ? m1 : occupied_bins(llen + nb * (c2 - 1), nb, 0, L2);
          wave_fence();
          i0 = count_below(L1, m1, row);
          j0 = count_below(M2, m2, col + 1);
        } else {
          i0 = a_i;
          j0 = a_j + 1;
        }
        if (j0 >= m2) {
          ++i0;
          j0 = tri ? i0 : 0;
        }
      }
    }
  for (int o = 32; o > 0; o >>= 1) {
    acc.samp += __shfl_xor((long long)acc.samp, o);
    acc.coag += __shfl_xor((long long)acc.coag, o);
    acc.warn += __shfl_xor((long long)acc.warn, o);
  }
  if (lane == 0 && run) {
    tot_samp += acc.samp;
    tot_coag += acc.coag;
    n_warn += acc.warn;
    B->n_acc_samp += acc.samp;
    B->n_acc_coag += acc.coag;
    if (err) B->error = err;
    B->step_samp = tot_samp;
    B->step_coag = tot_coag;
    B->n_samp += tot_samp;
    B->n_coag += tot_coag;
    B->n_warn += n_warn;
  }
  __syncthreads();
  if (LDS)
    for (int k = lane; k < K; k += 64) {
      A.llen[kb + k] = llen[k];
      A.lstart[kb + k] = lstart[k];
      A.lcap[kb + k] = lcap[k];
    }
  for (int q = lane; q < (int)(sizeof(BoxDesc) / sizeof(int)); q += 64)
    ((int *)&boxes[box])[q] = ((const int *)&s_box)[q];
}

}  // namespace pmc
