// pmc_transfer.h -- particles between the host's arrays and a box.
//
// The host keeps particles as records in arrays of its own (volumes
// particle-major, aero_particle_t%vol); the device keeps each field and each
// species contiguous over the slots.  They meet in a small ring of pinned
// memory: the host copies a chunk of its arrays into a part of the ring (or
// out of one) and a kernel reads it (or writes it) over the bus, while the
// host is at the next part.  The kernels do what the layouts ask for: the
// transposition of the volumes, through LDS so that the bus sees whole
// lines, the total volumes, and the defaults of absent fields.
//
// Bound by the bus and the host's copy, which overlap: 85000 particles of 4
// species go up in 0.13 ms and come back in 0.19 (volumes and identifiers).
// A pageable copy per field and species, with transpositions on the host,
// took 0.60 and 0.42 ms: below 1 MB such a copy costs 40 to 280 us, whatever
// its size.
// Components that a caller uploads need no transposition and are most of a
// record's bytes: they go straight to their slots by a copy of each array.
// 4e5 whole records of one species go up in 3.8 ms from pageable memory and
// 2.2 from pinned (7.1 with the components through the ring, where the kernel
// waits for the bus 20 times; 4.4 and 2.5 with a copy per field), and 100 of
// them in 0.05 ms either way (0.07 and 0.19).
#pragma once

#include "pmc_state.h"

namespace pmc {

constexpr int STAGE_PARTS = 4;
constexpr size_t STAGE_BYTES = 1 << 20;  // of a part: past it more does not pay, and 4 MB of a handle that moves particles stay pinned
constexpr int XFER_THREADS = 128;  // 32 KB of LDS for the most species

// the fields of a chunk of particles in a part; null: absent
struct Records {
  double *vol, *ctime, *least, *greatest;
  int64_t *id;
  int *group, *klass, *nprim, *ncomp, *csrc;
};
enum : unsigned {
  REC_VOL = 1, REC_ID = 2, REC_GROUP = 4, REC_KLASS = 8, REC_NPRIM = 16, REC_NCOMP = 32,
  REC_CSRC = 64, REC_CTIME = 128, REC_LEAST = 256, REC_GREATEST = 512
};

inline size_t record_bytes(unsigned fields, int ns) {
  auto has = [&](unsigned f) -> size_t { return (fields & f) ? 1 : 0; };
  return 8 * (has(REC_VOL) * ns + has(REC_ID) + has(REC_LEAST) + has(REC_GREATEST) +
              has(REC_CTIME) * MAX_COMP) +
         4 * (has(REC_GROUP) + has(REC_KLASS) + has(REC_NPRIM) + has(REC_NCOMP) +
              has(REC_CSRC) * MAX_COMP);
}

// the fields of m particles in a part, the 8-byte ones first
inline Records records_at(char *part, unsigned fields, int64_t m, int ns) {
  Records R{};
  auto take = [&](unsigned f, int64_t bytes) -> void * {
    if (!(fields & f)) return nullptr;
    void *p = part;
    part += m * bytes;
    return p;
  };
  R.vol = (double *)take(REC_VOL, 8 * ns);
  R.id = (int64_t *)take(REC_ID, 8);
  R.ctime = (double *)take(REC_CTIME, 8 * MAX_COMP);
  R.least = (double *)take(REC_LEAST, 8);
  R.greatest = (double *)take(REC_GREATEST, 8);
  R.group = (int *)take(REC_GROUP, 4);
  R.klass = (int *)take(REC_KLASS, 4);
  R.nprim = (int *)take(REC_NPRIM, 4);
  R.ncomp = (int *)take(REC_NCOMP, 4);
  R.csrc = (int *)take(REC_CSRC, 4 * MAX_COMP);
  return R;
}

// m records into the slots from base on; absent primaries and components are
// one of source 0, absent create times 0.  Given components are in their
// slots already (copied straight from the caller's arrays).  flag: a word to
// clear, or null.
__global__ void __launch_bounds__(XFER_THREADS)
k_put_records(Arrays A, int64_t base, int m, Records R, int *flag) {
  extern __shared__ double s_vol[];  // [XFER_THREADS * n_spec]
  const int t = threadIdx.x, i0 = blockIdx.x * XFER_THREADS, ns = A.n_spec;
  const int cnt = min(XFER_THREADS, m - i0);
  if (flag && blockIdx.x == 0 && t == 0) *flag = 0;
  for (int j = t; j < cnt * ns; j += XFER_THREADS) s_vol[j] = R.vol[(int64_t)i0 * ns + j];
  __syncthreads();
  if (t < cnt) {
    const int i = i0 + t;
    const int64_t p = base + i;
    if (R.id) A.id[p] = R.id[i];
    A.group[p] = R.group[i];
    A.klass[p] = R.klass[i];
    A.nprim[p] = R.nprim ? R.nprim[i] : 1;
    A.ncomp[p] = R.ncomp ? R.ncomp[i] : 1;
    const bool times = R.least && R.greatest;
    A.least[p] = times ? R.least[i] : 0.0;
    A.greatest[p] = times ? R.greatest[i] : 0.0;
    double v = 0.0;
    for (int s = 0; s < ns; ++s) {
      const double x = s_vol[t * ns + s];
      A.vol[(int64_t)s * A.total_cap + p] = x;
      v += x;
    }
    A.vtot[p] = v;
  }
  if (R.ncomp) return;
  const int64_t c0 = comp_at(base + i0, 0);
  for (int j = t; j < cnt * MAX_COMP; j += XFER_THREADS) {
    A.csrc[c0 + j] = 0;
    A.ctime[c0 + j] = 0.0;
  }
}

// the records of m slots from base on; the device keeps only the first ncomp
// components of a particle, the rest read as zero
__global__ void __launch_bounds__(XFER_THREADS)
k_get_records(Arrays A, int64_t base, int m, Records R) {
  extern __shared__ double s_vol[];  // [XFER_THREADS * n_spec] when volumes are asked for
  __shared__ int s_nco[XFER_THREADS];
  const int t = threadIdx.x, i0 = blockIdx.x * XFER_THREADS, ns = A.n_spec;
  const int cnt = min(XFER_THREADS, m - i0);
  if (t < cnt) {
    const int i = i0 + t;
    const int64_t p = base + i;
    if (R.vol)
      for (int s = 0; s < ns; ++s) s_vol[t * ns + s] = A.vol[(int64_t)s * A.total_cap + p];
    const int nco = A.ncomp[p];
    s_nco[t] = nco;
    if (R.id) R.id[i] = A.id[p];
    if (R.group) R.group[i] = A.group[p];
    if (R.klass) R.klass[i] = A.klass[p];
    if (R.nprim) R.nprim[i] = A.nprim[p];
    if (R.ncomp) R.ncomp[i] = nco;
    if (R.least) R.least[i] = A.least[p];
    if (R.greatest) R.greatest[i] = A.greatest[p];
  }
  __syncthreads();
  if (R.vol)
    for (int j = t; j < cnt * ns; j += XFER_THREADS) R.vol[(int64_t)i0 * ns + j] = s_vol[j];
  if (!R.csrc && !R.ctime) return;
  const int64_t c0 = comp_at(base + i0, 0), r0 = (int64_t)i0 * MAX_COMP;
  for (int j = t; j < cnt * MAX_COMP; j += XFER_THREADS) {
    const bool kept = j % MAX_COMP < s_nco[j / MAX_COMP];
    if (R.csrc) R.csrc[r0 + j] = kept ? A.csrc[c0 + j] : 0;
    if (R.ctime) R.ctime[r0 + j] = kept ? A.ctime[c0 + j] : 0.0;
  }
}

// A box's descriptor changed in stream order, its new values as arguments: a
// launch (2.5 us) where a copy to the device and its wait take 11 a field.
__global__ void k_set_env(BoxDesc *B, Env env) {
  if (threadIdx.x != 0) return;
  B->env = env;
  B->terms_kernel = 0;
}

// the class count changes the key space of the lists
__global__ void k_set_weights(BoxDesc *B, Weights w) {
  if (threadIdx.x != 0) return;
  B->w = w;
  B->tables_valid = 0;
  B->xlists_valid = 0;
  B->pkeys_valid = 0;
  B->valid_sort = 0;
}

__global__ void k_scale_weights(BoxDesc *B, double factor) {
  if ((int)threadIdx.x < B->w.n_group * B->w.n_class) B->w.mag[threadIdx.x] *= factor;
  if (threadIdx.x == 0) B->tables_valid = 0;
}

__global__ void k_set_next_id(BoxDesc *B, int64_t next_id, int64_t stride, int64_t offset) {
  if (threadIdx.x != 0) return;
  B->next_id = next_id;
  B->id_stride = stride;
  B->id_offset = offset;
}

// a box's particles were replaced by n_part new ones
__global__ void k_set_uploaded(BoxDesc *B, int n_part) {
  if (threadIdx.x != 0) return;
  B->n_part = n_part;
  B->valid_sort = 0;
  B->xlists_valid = 0;
  B->pkeys_valid = 0;
  B->terms_kernel = 0;
  B->n_info = 0;
  if (B->error) B->revived = 1;
  B->error = 0;
}

}  // namespace pmc
