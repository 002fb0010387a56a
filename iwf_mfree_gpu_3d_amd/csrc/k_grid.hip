// k_grid.hip -- blanking, cell hashing, stable counting sort, cell tables, permute + predict.
//
// Replaces (one pass each, all on one stream, no host round trip):
//   do_blanking + compute_hashes + adapt_particle_number   src/actions_gpu.cu:489-531,
//                                                          src/grid_gpu_base.cu:41-63,141-164
//   thrust::sort_by_key (stable) + find_cell_start         src/grid_gpu_green.cu:24-70,265-301
//   reorder_data + init + predict + material_eos +
//   do_corrector_artificial_stress                         src/grid_gpu_green.cu:72-125,
//                                                          src/leap_frog.cu:30-70,
//                                                          src/actions_gpu.cu:40-53,70-132
//
// Sort: keys are cell hashes < num_cell or INT_MAX.  A counting sort by cell gives the cell
// offsets directly (exclusive scan of the per-cell counts).  The atomic that counts a particle
// returns its slot inside the cell, in no particular order; the permutation then takes each
// particle to its place by previous index among its cell's, which makes the result identical to a
// stable sort.  INT_MAX keys go to the tail in previous-index order by a block-wise compaction.
// Cell start/end of the reference are off[c], off[c+1] for non-empty cells.
//
// Launches bound the sort of small sets and atomics that of large ones.  The counts are an array of
// their own that the scatter leaves zero for the next sort; the scan is one launch up to SCAN_ALONE
// cells and two above; the order inside the cells is the permutation's own work for small sets; and a
// run of particles of one cell is counted by one atomic, which also hands out their slots.  With the
// permutation: 8,000 particles 44 us in eight launches, now 29 in four; 1M 0.32 ms, now 0.25 (hash 33
// us, now 17: the particles come in the last sort's order; scatter 40, now 6.4: no atomics; fix-up and
// zeroing 17, now 7.6).
#include <algorithm>

#include "mfg_device.hpp"
#include "mfg_records.hpp"

namespace mfg {

constexpr int BS = 256;  // threads per block of the particle passes
constexpr int SCAN_ITEMS = SCAN_TILE / BS;
constexpr int SCAN_NT = 1024;  // threads of a tile without tile sums

template <class T>
__device__ __forceinline__ T wave_incl_scan(T v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const T t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}

// exclusive scan across a block of NT threads; lds must hold NT/64 + 1 values
template <int NT, class T>
__device__ __forceinline__ T block_excl_scan(T v, T *lds, T &total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const T incl = wave_incl_scan(v);
  if (lane == 63) lds[wid] = incl;
  __syncthreads();
  if (threadIdx.x == 0) {
    T acc = 0;
    for (int w = 0; w < NT / 64; w++) {
      const T t = lds[w];
      lds[w] = acc;
      acc += t;
    }
    lds[NT / 64] = acc;
  }
  __syncthreads();
  const T r = incl - v + lds[wid];
  total = lds[NT / 64];
  __syncthreads();
  return r;
}

__device__ __forceinline__ bool rates_invalid(const State &st, unsigned i) {
  auto bad = [](double v) { return isnan(v) || isinf(v); };
  return bad(st.xt[i]) || bad(st.yt[i]) || bad(st.zt[i]) || bad(st.vxt[i]) || bad(st.vyt[i]) ||
         bad(st.vzt[i]) || bad(st.St[0][i]) || bad(st.St[1][i]) || bad(st.St[2][i]) ||
         bad(st.St[3][i]) || bad(st.St[4][i]) || bad(st.St[5][i]) || bad(st.rho_t[i]) ||
         bad(st.T_t[i]);
}

// Each kernel below is a body run by workgroup `b` (blockIdx.x of a single-instance launch, the
// workgroup inside its instance's range of a batched launch) and a __global__ wrapper.
__device__ __forceinline__ void blank_hash_count(unsigned b, const State &st, unsigned n_init,
                                                 const GridInfo &g, int blanking, double b0,
                                                 double b1, double b2, double b3, double b4,
                                                 double b5, double vmax2, int *key, int *hist,
                                                 int *slot, int *blk, Counters *cnt) {
  __shared__ int lds[BS / 64 + 1];
  const unsigned i = b * BS + threadIdx.x;
  int blank_key = 0, k = KEY_BLANK;
  if (i < n_init) {
    uint32_t fl = st.flags[i];
    if (blanking) {
      double px = st.x[i], py = st.y[i], pz = st.z[i];
      double vx = st.vx[i], vy = st.vy[i], vz = st.vz[i];
      bool too_fast = vx * vx + vy * vy + vz * vz >= vmax2;
      bool in = px >= b0 && px <= b3 && py >= b1 && py <= b4 && pz >= b2 && pz <= b5;
      uint32_t nf = fl;
      if (too_fast || !in) nf |= FL_BLANKED;
      // inside and slow: finite rates unblank (src/actions_gpu.cu:506-529), non-finite ones keep
      // the flag as it is, so the rates matter only for a blanked particle
      else if ((fl & FL_BLANKED) && !rates_invalid(st, i)) nf &= ~FL_BLANKED;
      if (nf != fl) st.flags[i] = nf;
      fl = nf;
    }
    if ((fl & FL_BLANKED) && g.hard_blank) {
      k = KEY_BLANK;
    } else {
      int ix = (int)((st.x[i] - g.bbmin[0]) / g.dx);
      int iy = (int)((st.y[i] - g.bbmin[1]) / g.dx);
      int iz = (int)((st.z[i] - g.bbmin[2]) / g.dx);
      long hh = (long)ix * g.ny * g.nz + (long)iy * g.nz + iz;
      k = (int)hh;
      if (k < 0 || (long)k >= g.num_cell) {
        atomicOr(&cnt->err_grid, 1);
        k = KEY_BLANK;
      }
    }
    key[i] = k;
    blank_key = (k == KEY_BLANK) ? 1 : 0;
  }
  // one atomic for a run of lanes in the same cell (the particles come in the last sort's order, two
  // or three to a cell): the first lane adds the run's length, each takes its place in the run
  const int lane = threadIdx.x & 63;
  const int k_before = __shfl_up(k, 1, 64);  // by every lane: a lane that sits out gives 0
  const uint64_t heads = __ballot(lane == 0 || k_before != k);
  const int head = 63 - __clzll(heads & (~0ull >> (63 - lane)));
  const uint64_t later = lane == 63 ? 0ull : heads >> (lane + 1);
  int first = 0;
  if (head == lane && k != KEY_BLANK) first = atomicAdd(&hist[k], later ? __ffsll((unsigned long long)later) : 64 - lane);
  first = __shfl(first, head, 64);
  if (k != KEY_BLANK) slot[i] = first + lane - head;
  int total;
  block_excl_scan<BS>(blank_key, lds, total);
  if (threadIdx.x == 0) blk[b] = total;
}
__global__ void __launch_bounds__(BS)
    k_blank_hash_count(State st, unsigned n_init, GridInfo g, int blanking, double b0, double b1,
                       double b2, double b3, double b4, double b5, double vmax2, int *key,
                       int *hist, int *slot, int *blk, Counters *cnt) {
  blank_hash_count(blockIdx.x, st, n_init, g, blanking, b0, b1, b2, b3, b4, b5, vmax2, key, hist,
                   slot, blk, cnt);
}

// ITEMS consecutive entries from k on, those beyond n as 0 (k and the array 16-byte aligned)
template <int ITEMS>
__device__ __forceinline__ void load_items(const int *a, long k, long n, int (&v)[ITEMS]) {
  if (k + ITEMS <= n) {
#pragma unroll
    for (int q = 0; q < ITEMS; q += 4) {
      const int4 x = *(const int4 *)(a + k + q);
      v[q] = x.x; v[q + 1] = x.y; v[q + 2] = x.z; v[q + 3] = x.w;
    }
  } else {
#pragma unroll
    for (int q = 0; q < ITEMS; q++) v[q] = k + q < n ? a[k + q] : 0;
  }
}

// Block sums of a sort: a workgroup's base is the sum of those of all workgroups before it, which each adds
// up itself.  From PREFIX_CHUNKS of them on also sums over PREFIX_CHUNK of them each are made (one workgroup of
// CS_NT threads for both arrays), which keeps that linear: 68M particles of which every tenth is blanked 8.5 -> 0.5
// ms of scatter, 549M cells 10.0 -> 1.6 ms of scan; 8M without blanked particles 6 us more.
constexpr int CS_NT = 1024;
template <class T>
__device__ __forceinline__ void chunk_sums(const T *a, unsigned n, T *chunk) {
  const unsigned lane = threadIdx.x & 63, w = threadIdx.x >> 6, chunks = n / PREFIX_CHUNK;  // whole ones
  for (unsigned c = w; c < chunks; c += CS_NT / 64) {
    T s = 0;
#pragma unroll
    for (unsigned q = 0; q < PREFIX_CHUNK; q += 64) s += a[(size_t)c * PREFIX_CHUNK + q + lane];
    s = wave_incl_scan(s);
    if (lane == 63) chunk[c] = s;
  }
}
// this thread's share of the sum of a[0 .. b) among NT
template <int NT, class T>
__device__ __forceinline__ T sum_before(const T *a, const T *chunk, unsigned b) {
  T s = 0;
  unsigned first = 0;
  if (chunk) {
    for (unsigned k = threadIdx.x; k < b / PREFIX_CHUNK; k += NT) s += chunk[k];
    first = b / PREFIX_CHUNK * PREFIX_CHUNK;
  }
  for (unsigned k = first + threadIdx.x; k < b; k += NT) s += a[k];
  return s;
}

// Particles in the low and occupied cells in the high 32 bits: one scan gives both the offsets and the
// occupied cells' places in their list
typedef unsigned long long CellSum;
__device__ __forceinline__ CellSum cell_sum(int count) {
  return (CellSum)count | ((CellSum)(count > 0) << 32);
}

// tile reduction of the cell counts
__device__ __forceinline__ void scan_reduce(unsigned b, const int *hist, long n, CellSum *part) {
  __shared__ CellSum lds[BS / 64 + 1];
  int v[SCAN_ITEMS];
  CellSum s = 0;
  load_items<SCAN_ITEMS>(hist, (long)b * SCAN_TILE + (long)threadIdx.x * SCAN_ITEMS, n, v);
#pragma unroll
  for (int q = 0; q < SCAN_ITEMS; q++) s += cell_sum(v[q]);
  CellSum total;
  block_excl_scan<BS>(s, lds, total);
  if (threadIdx.x == 0) part[b] = total;
}
__global__ void __launch_bounds__(BS) k_scan_reduce(const int *hist, long n, CellSum *part) {
  scan_reduce(blockIdx.x, hist, n, part);
}

// the chunk sums that a sort needs
__device__ __forceinline__ void sort_chunks(const GridBuffers &gb, unsigned tiles) {
  if (gb.part_chunk) chunk_sums(gb.blk2, tiles, gb.part_chunk);
  if (gb.blk_chunk) chunk_sums(gb.blk, (unsigned)gb.nblk, gb.blk_chunk);
}
__global__ void __launch_bounds__(CS_NT) k_sort_chunks(GridBuffers gb, unsigned tiles) { sort_chunks(gb, tiles); }

// The offsets of tile b's cells (NT threads, ITEMS cells each), its occupied cells in the list of all
// (ascending; occ[n]: how many), and with the last tile the totals.  A tile's base is the sum of all
// before it: of the tile sums, or without them (part null: SCAN_ALONE) of the counts themselves, eight
// loads of a thread in flight (26,000 cells: 8.4 us, 62,000: 9.3, of which the list of occupied cells
// 1.8; in two launches 4.6 and 4.8, the gap between them, and the list).
template <int NT, int ITEMS>
__device__ __forceinline__ void scan_cells(unsigned b, const int *hist, long n, const CellSum *part,
                                           const CellSum *chunk, int *off, int *occ, unsigned n_init, Counters *cnt) {
  __shared__ CellSum lds[NT / 64 + 1];
  const long base = ((long)b * NT + threadIdx.x) * ITEMS;
  int v[ITEMS];
  CellSum s = 0, before = 0, total, prefix;
  load_items<ITEMS>(hist, base, n, v);
  if (part) {
    before = sum_before<NT>(part, chunk, b);
  } else {
    // b tiles of NT x ITEMS counts: ITEMS / 4 vectors a thread and tile
    const int4 *h = (const int4 *)hist + threadIdx.x;
#pragma unroll 8
    for (unsigned k = 0; k < b * (ITEMS / 4); k++) {
      const int4 x = h[(size_t)k * NT];
      before += cell_sum(x.x) + cell_sum(x.y) + cell_sum(x.z) + cell_sum(x.w);
    }
  }
#pragma unroll
  for (int q = 0; q < ITEMS; q++) s += cell_sum(v[q]);
  block_excl_scan<NT>(before, lds, prefix);
  const CellSum first = prefix + block_excl_scan<NT>(s, lds, total);
  if (threadIdx.x == 0 && (long)(b + 1) * NT * ITEMS >= n) {  // the last tile
    const unsigned N = (unsigned)(prefix + total);
    off[n] = (int)N;
    occ[n] = (int)((prefix + total) >> 32);
    cnt->N = N;
    cnt->n_blank_key = n_init - N;
    cnt->candidates = 0ull;
    cnt->pairs = 0ull;
  }
  int w[ITEMS], o = (int)(unsigned)first, place = (int)(first >> 32);
#pragma unroll
  for (int q = 0; q < ITEMS; q++) {
    w[q] = o;
    o += v[q];
    if (v[q] > 0) occ[place++] = (int)(base + q);
  }
  if (base + ITEMS <= n) {
#pragma unroll
    for (int q = 0; q < ITEMS; q += 4) *(int4 *)(off + base + q) = make_int4(w[q], w[q + 1], w[q + 2], w[q + 3]);
  } else {
#pragma unroll
    for (int q = 0; q < ITEMS; q++)
      if (base + q < n) off[base + q] = w[q];
  }
}
template <int NT, int ITEMS>
__global__ void __launch_bounds__(NT) k_scan_cells(const int *hist, long n, const CellSum *part, const CellSum *chunk,
                                                   int *off, int *occ, unsigned n_init, Counters *cnt) {
  scan_cells<NT, ITEMS>(blockIdx.x, hist, n, part, chunk, off, occ, n_init, cnt);
}

// particles to their cells (order: an INT_MAX key's particle at its final place, the others in any
// order within their cell), and the counts back to zero by all nb workgroups, of which those past the
// particles' only clear (scatter_blocks)
__device__ __forceinline__ void scatter(unsigned b, unsigned nb, unsigned n_init, long num_cell, const int *key,
                                        const int *off, const int *slot, int *hist, const int *blk,
                                        const int *chunk, const Counters *cnt, int *order) {
  __shared__ int lds[BS / 64 + 1];
  const unsigned i = b * BS + threadIdx.x;
  const int k = (i < n_init) ? key[i] : 0;
  const int is_blank = (i < n_init && k == KEY_BLANK) ? 1 : 0;
  int total;
  const int rank = block_excl_scan<BS>(is_blank, lds, total);
  if (total > 0) {
    int prefix;
    block_excl_scan<BS>(sum_before<BS>(blk, chunk, b), lds, prefix);
    if (is_blank) order[(int)cnt->N + prefix + rank] = (int)i;
  }
  if (i < n_init && !is_blank) order[off[k] + slot[i]] = (int)i;
  for (long c = (long)i; c < num_cell; c += (long)nb * BS) hist[c] = 0;
}
__global__ void __launch_bounds__(BS) k_scatter(unsigned n_init, long num_cell, const int *key, const int *off,
                                                const int *slot, int *hist, const int *blk, const int *chunk,
                                                const Counters *cnt, int *order) {
  scatter(blockIdx.x, gridDim.x, n_init, num_cell, key, off, slot, hist, blk, chunk, cnt, order);
}

// The place of the particle at scattered position t: by previous index among its cell's.
__device__ __forceinline__ unsigned place_in_cell(unsigned t, const int *scattered, const int *off, int particle,
                                                  int key) {
  if (key == KEY_BLANK) return t;
  const int s = off[key], e = off[key + 1];
  int place = s;
  for (int q = s; q < e; q++) place += scattered[q] < particle;
  return (unsigned)place;
}
__device__ __forceinline__ void order_cells(unsigned b, unsigned n_init, const int *scattered, const int *key,
                                            const int *off, int *order) {
  const unsigned t = b * BS + threadIdx.x;
  if (t >= n_init) return;
  const int s = scattered[t];
  order[place_in_cell(t, scattered, off, s, key[s])] = s;
}
__global__ void __launch_bounds__(BS) k_order(unsigned n_init, const int *scattered, const int *key,
                                              const int *off, int *order) {
  order_cells(blockIdx.x, n_init, scattered, key, off, order);
}

// gather the persistent state by the sort permutation, then predict the half step and build the
// pair records (EOS and artificial stress included)
template <class RecT>
__device__ __forceinline__ void permute_predict(unsigned b, const State &src, const State &dst,
                                                unsigned n_init, int *order, const int *scattered,
                                                const int *off, const int *key, int *key_sorted,
                                                const Counters *cnt, const Consts &c, int predict,
                                                RecT *rec, double4 *nl4, double2 *pse2,
                                                double4 *cs4, double *p_dbg, double *R_dbg) {
  unsigned i = b * BS + threadIdx.x;
  if (i >= n_init) return;
  const unsigned N = cnt->N;
  // from the scattered particles (the order inside the cells is found here and kept), from a
  // finished order, or, both null, the particles keep their places (a step between sorts)
  const int s = scattered ? scattered[i] : order ? order[i] : (int)i;
  if (scattered || order) {
    const int k = key[s];
    if (scattered) {
      i = place_in_cell(i, scattered, off, s, k);
      order[i] = s;
    }
    key_sorted[i] = k;
  }
  double x[3] = {src.x[s], src.y[s], src.z[s]};
  double v[3] = {src.vx[s], src.vy[s], src.vz[s]};
  double S[6], St[6];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    S[k] = src.S[k][s];
    St[k] = src.St[k][s];
  }
  double xt[3] = {src.xt[s], src.yt[s], src.zt[s]};
  double vt[3] = {src.vxt[s], src.vyt[s], src.vzt[s]};
  double rho = src.rho[s], T = src.T[s], rho_t = src.rho_t[s], T_t = src.T_t[s], h = src.h[s];
  uint32_t fl = src.flags[s];
  dst.x[i] = x[0]; dst.y[i] = x[1]; dst.z[i] = x[2];
  dst.vx[i] = v[0]; dst.vy[i] = v[1]; dst.vz[i] = v[2];
  dst.vbx[i] = src.vbx[s]; dst.vby[i] = src.vby[s]; dst.vbz[i] = src.vbz[s];
  dst.fcx[i] = src.fcx[s]; dst.fcy[i] = src.fcy[s]; dst.fcz[i] = src.fcz[s];
  dst.ftx[i] = src.ftx[s]; dst.fty[i] = src.fty[s]; dst.ftz[i] = src.ftz[s];
  dst.h[i] = h; dst.rho[i] = rho;
#pragma unroll
  for (int k = 0; k < 6; k++) {
    dst.S[k][i] = S[k];
    dst.St[k][i] = St[k];
  }
  dst.eps_pl[i] = src.eps_pl[s]; dst.eps_pl_dot[i] = src.eps_pl_dot[s]; dst.T[i] = T;
  dst.xt[i] = xt[0]; dst.yt[i] = xt[1]; dst.zt[i] = xt[2];
  dst.vxt[i] = vt[0]; dst.vyt[i] = vt[1]; dst.vzt[i] = vt[2];
  dst.rho_t[i] = rho_t; dst.T_t[i] = T_t;
  dst.flags[i] = fl;
  dst.id[i] = src.id[s];
  if (!predict) return;

  // predict (src/leap_frog.cu:42-70): half step from the rates of the previous step
  const bool blanked = (fl & FL_BLANKED) != 0;
  const bool tool = (fl & FL_TOOL) != 0;
  double xh[3], vh[3], Sh[6], rhoh = rho, Th = T;
  if (!blanked) {
    const double hdt = 0.5 * c.dt;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      xh[k] = x[k] + hdt * xt[k];
      vh[k] = v[k] + hdt * vt[k];
    }
#pragma unroll
    for (int k = 0; k < 6; k++) Sh[k] = S[k] + hdt * St[k];
    rhoh = rho + hdt * rho_t;
    Th = T + hdt * T_t;
  } else {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      xh[k] = x[k];
      vh[k] = v[k];
    }
#pragma unroll
    for (int k = 0; k < 6; k++) Sh[k] = S[k];
  }
  // equation of state and artificial stress (src/actions_gpu.cu:40-53,70-132)
  double p = 0., R[6] = {0., 0., 0., 0., 0., 0.};
  if (i < N && !blanked && !tool) {
    double c0 = sqrt_site(c.a_K / c.a_rho0, c.single_sqrt);
    p = c0 * c0 * (rhoh - c.a_rho0);
    if (c.a_stresseps != 0.) art_stress(c.a_stresseps, rhoh, p, Sh, R);
  }
  emit_record<RecT>(i, xh, h, vh, rhoh, Sh, p, R, Th, tool, blanked, c, rec, nl4, pse2, cs4);
  if (p_dbg) {
    p_dbg[i] = p;
#pragma unroll
    for (int k = 0; k < 6; k++) R_dbg[6 * (size_t)i + k] = R[k];
  }
}
template <class RecT>
__global__ void __launch_bounds__(BS)
    k_permute_predict(State src, State dst, unsigned n_init, int *order, const int *scattered,
                      const int *off, const int *key, int *key_sorted, const Counters *cnt, Consts c, int predict, RecT *rec,
                      double4 *nl4, double2 *pse2, double4 *cs4, double *p_dbg, double *R_dbg,
                      unsigned *list_n) {
  // the contact search's list, which the particle update fills, starts empty
  if (list_n && blockIdx.x == 0 && threadIdx.x == 0) *list_n = 0u;
  permute_predict<RecT>(blockIdx.x, src, dst, n_init, order, scattered, off, key, key_sorted, cnt, c, predict, rec,
                        nl4, pse2, cs4, p_dbg, R_dbg);
}

// Green (0xffffffff for empty cells) or Rothlin (start == end) tables from the offsets
__global__ void __launch_bounds__(BS) k_cells_to_tables(const int *off, long n, int rothlin,
                                                        int *start, int *end) {
  long c = (long)blockIdx.x * BS + threadIdx.x;
  if (c >= n) return;
  int s = off[c], e = off[c + 1];
  if (!rothlin && s == e) {
    start[c] = -1;
    end[c] = -1;
  } else {
    start[c] = s;
    end[c] = e;
  }
}

// bounding box and largest h over the first N particles (unlocked grids)
__global__ void __launch_bounds__(BS) k_bbox(State st, const Counters *cnt, double *part) {
  __shared__ double red[7][BS];
  const unsigned N = cnt->N;
  double mn[3] = {1e300, 1e300, 1e300}, mx[3] = {-1e300, -1e300, -1e300}, hm = -1e300;
  for (unsigned i = blockIdx.x * BS + threadIdx.x; i < N; i += gridDim.x * BS) {
    double p[3] = {st.x[i], st.y[i], st.z[i]};
#pragma unroll
    for (int k = 0; k < 3; k++) {
      mn[k] = fmin(mn[k], p[k]);
      mx[k] = fmax(mx[k], p[k]);
    }
    hm = fmax(hm, st.h[i]);
  }
  for (int k = 0; k < 3; k++) {
    red[k][threadIdx.x] = mn[k];
    red[3 + k][threadIdx.x] = mx[k];
  }
  red[6][threadIdx.x] = hm;
  __syncthreads();
  for (int o = BS / 2; o > 0; o >>= 1) {
    if (threadIdx.x < (unsigned)o) {
      for (int k = 0; k < 3; k++) red[k][threadIdx.x] = fmin(red[k][threadIdx.x], red[k][threadIdx.x + o]);
      for (int k = 3; k < 7; k++) red[k][threadIdx.x] = fmax(red[k][threadIdx.x], red[k][threadIdx.x + o]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int k = 0; k < 7; k++) part[7 * blockIdx.x + k] = red[k][0];
}

// ---------------------------------------------------------------------------------------------
static inline unsigned nblocks(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

void launch_blank_hash_count(hipStream_t s, const State &st, unsigned n_init, const GridInfo &g,
                             int blanking, const double *bb, double vmax2, GridBuffers &gb,
                             Counters *cnt) {
  double z[6] = {0, 0, 0, 0, 0, 0};
  const double *b = bb ? bb : z;
  hipLaunchKernelGGL(k_blank_hash_count, dim3(gb.nblk), dim3(BS), 0, s, st, n_init, g, blanking,
                     b[0], b[1], b[2], b[3], b[4], b[5], vmax2, gb.key, gb.hist, gb.order, gb.blk, cnt);
}

// The order inside the cells in a launch of its own or by the permutation, whose gathers then wait for
// four dependent reads more: 8,000 particles 2.5 us and a launch against 1.1 more; 1M 7.6 us against 28
bool order_apart(long particles) { return particles >= 128 * 1024; }

int scan_tiles(long num_cell, bool alone) {
  return (int)nblocks(num_cell, alone ? SCAN_TILE_ALONE : SCAN_TILE);
}

void launch_scan_cells(hipStream_t s, const GridInfo &g, GridBuffers &gb, unsigned n_init,
                       Counters *cnt) {
  const bool alone = g.num_cell <= SCAN_ALONE;
  const dim3 tiles((unsigned)scan_tiles(g.num_cell, alone));
  if (!alone) hipLaunchKernelGGL(k_scan_reduce, tiles, dim3(BS), 0, s, gb.hist, g.num_cell, gb.blk2);
  if (gb.part_chunk || gb.blk_chunk) hipLaunchKernelGGL(k_sort_chunks, dim3(1), dim3(CS_NT), 0, s, gb, tiles.x);
  if (alone) {
    hipLaunchKernelGGL((k_scan_cells<SCAN_NT, SCAN_TILE_ALONE / SCAN_NT>), tiles, dim3(SCAN_NT), 0, s, gb.hist, g.num_cell,
                       (const CellSum *)nullptr, (const CellSum *)nullptr, gb.count, gb.occ, n_init, cnt);
    return;
  }
  hipLaunchKernelGGL((k_scan_cells<BS, SCAN_ITEMS>), tiles, dim3(BS), 0, s, gb.hist, g.num_cell, gb.blk2,
                     gb.part_chunk, gb.count, gb.occ, n_init, cnt);
}

// A workgroup per 256 particles, and for a few particles in a large grid one per 4,096 cells, up to 2,048:
// cleared by the particles' four workgroups alone, 1,000 particles sorted in 266 us with 8M cells and 1,890 with
// 64M, now 74 and 280.
int scatter_blocks(unsigned n_init, long num_cell) {
  return (int)std::max<long>(nblocks(n_init, BS), std::min<long>(nblocks(num_cell, 4096), 2048));
}

void launch_scatter(hipStream_t s, unsigned n_init, const GridInfo &g, GridBuffers &gb,
                    Counters *cnt) {
  hipLaunchKernelGGL(k_scatter, dim3(scatter_blocks(n_init, g.num_cell)), dim3(BS), 0, s, n_init, g.num_cell, gb.key, gb.count,
                     gb.order, gb.hist, gb.blk, gb.blk_chunk, cnt, gb.scattered);
}

void launch_order(hipStream_t s, unsigned n_init, GridBuffers &gb) {
  hipLaunchKernelGGL(k_order, dim3(nblocks(n_init, BS)), dim3(BS), 0, s, n_init, gb.scattered, gb.key,
                     gb.count, gb.order);
}

void launch_permute_predict_ex(hipStream_t s, const State &src, const State &dst, unsigned n_init,
                               const GridBuffers &gb, const Counters *cnt, const Consts &c,
                               int predict, void *rec, double4 *nl4, double2 *pse2, double4 *cs4,
                               double *p_dbg, double *R_dbg, unsigned *list_n) {
  if (c.precision == MFG_FP64)
    hipLaunchKernelGGL(k_permute_predict<Rec64>, dim3(nblocks(n_init, BS)), dim3(BS), 0, s, src,
                       dst, n_init, gb.order, gb.scattered, gb.count, gb.key, gb.key_sorted, cnt, c, predict, (Rec64 *)rec,
                       nl4, pse2, cs4, p_dbg, R_dbg, list_n);
  else
    hipLaunchKernelGGL(k_permute_predict<Rec32>, dim3(nblocks(n_init, BS)), dim3(BS), 0, s, src,
                       dst, n_init, gb.order, gb.scattered, gb.count, gb.key, gb.key_sorted, cnt, c, predict, (Rec32 *)rec,
                       nl4, pse2, cs4, p_dbg, R_dbg, list_n);
}

void launch_cells_to_tables(hipStream_t s, const GridInfo &g, const int *offsets, int rothlin,
                            int *start, int *end) {
  hipLaunchKernelGGL(k_cells_to_tables, dim3(nblocks(g.num_cell, BS)), dim3(BS), 0, s, offsets,
                     g.num_cell, rothlin, start, end);
}

void launch_bbox_reduce(hipStream_t s, const State &st, const Counters *cnt, unsigned n_init,
                        double *partials, int nb) {
  (void)n_init;
  hipLaunchKernelGGL(k_bbox, dim3(nb), dim3(BS), 0, s, st, cnt, partials);
}

// ---------------------------------------------------------------------------------------------
// batched launches: the same bodies, arguments from each instance's descriptor.  Before the
// permutation an instance's state is buf[cur], after it buf[cur ^ 1].
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(BS) kb_blank_hash_count(const Inst *in, BatchMap m) {
  unsigned b, nb;
  const Inst &d = in[batch_locate(m, b, nb)];
  blank_hash_count(b, d.buf[d.cur], d.n_init, d.g, d.blanking, d.bb[0], d.bb[1], d.bb[2], d.bb[3],
                   d.bb[4], d.bb[5], d.vmax2, d.gb.key, d.gb.hist, d.gb.order, d.gb.blk, d.cnt);
}

__global__ void __launch_bounds__(BS) kb_scan_reduce(const Inst *in, BatchMap m) {
  unsigned b, nb;
  const Inst &d = in[batch_locate(m, b, nb)];
  scan_reduce(b, d.gb.hist, d.g.num_cell, d.gb.blk2);
}

__global__ void __launch_bounds__(CS_NT) kb_sort_chunks(const Inst *in, BatchMap m) {
  unsigned b, nb;
  const Inst &d = in[batch_locate(m, b, nb)];
  sort_chunks(d.gb, (unsigned)((d.g.num_cell + SCAN_TILE - 1) / SCAN_TILE));
}

template <int NT, int ITEMS>
__global__ void __launch_bounds__(NT) kb_scan_cells(const Inst *in, BatchMap m) {
  unsigned b, nb;
  const Inst &d = in[batch_locate(m, b, nb)];
  scan_cells<NT, ITEMS>(b, d.gb.hist, d.g.num_cell, NT == BS ? d.gb.blk2 : nullptr, d.gb.part_chunk, d.gb.count,
                        d.gb.occ, d.n_init, d.cnt);
}

__global__ void __launch_bounds__(BS) kb_scatter(const Inst *in, BatchMap m) {
  unsigned b, nb;
  const Inst &d = in[batch_locate(m, b, nb)];
  scatter(b, nb, d.n_init, d.g.num_cell, d.gb.key, d.gb.count, d.gb.order, d.gb.hist, d.gb.blk,
          d.gb.blk_chunk, d.cnt, d.gb.scattered);
}

__global__ void __launch_bounds__(BS) kb_order(const Inst *in, BatchMap m) {
  unsigned b, nb;
  const Inst &d = in[batch_locate(m, b, nb)];
  order_cells(b, d.n_init, d.gb.scattered, d.gb.key, d.gb.count, d.gb.order);
}

template <class RecT>
__global__ void __launch_bounds__(BS) kb_permute_predict(const Inst *in, BatchMap m) {
  unsigned b, nb;
  const Inst &d = in[batch_locate(m, b, nb)];
  permute_predict<RecT>(b, d.buf[d.cur], d.buf[d.cur ^ 1], d.n_init, d.gb.order, d.ordered ? nullptr : d.gb.scattered,
                        d.gb.count, d.gb.key, d.gb.key_sorted, d.cnt, d.c, 1, (RecT *)d.rec, d.nl4, d.pse2, d.cs4,
                        nullptr, nullptr);
}

// hash + blanking, scan and scatter of every instance, as sort_keys does for one
void launch_batch_sort(hipStream_t s, const BatchLaunch &L) {
  hipLaunchKernelGGL(kb_blank_hash_count, dim3(L.parts.blocks), dim3(BS), 0, s, L.inst, L.parts.m);
  if (!L.scan_alone) hipLaunchKernelGGL(kb_scan_reduce, dim3(L.tiles.blocks), dim3(BS), 0, s, L.inst, L.tiles.m);
  if (L.sort_chunks) hipLaunchKernelGGL(kb_sort_chunks, dim3(L.one.blocks), dim3(CS_NT), 0, s, L.inst, L.one.m);
  if (L.scan_alone) {
    hipLaunchKernelGGL((kb_scan_cells<SCAN_NT, SCAN_TILE_ALONE / SCAN_NT>), dim3(L.tiles.blocks), dim3(SCAN_NT), 0, s,
                       L.inst, L.tiles.m);
  } else {
    hipLaunchKernelGGL((kb_scan_cells<BS, SCAN_ITEMS>), dim3(L.tiles.blocks), dim3(BS), 0, s, L.inst, L.tiles.m);
  }
  hipLaunchKernelGGL(kb_scatter, dim3(L.scatter.blocks), dim3(BS), 0, s, L.inst, L.scatter.m);
  if (L.ordered) hipLaunchKernelGGL(kb_order, dim3(L.parts.blocks), dim3(BS), 0, s, L.inst, L.parts.m);
}

void launch_batch_permute(hipStream_t s, const BatchLaunch &L) {
  if (L.precision == MFG_FP64)
    hipLaunchKernelGGL(kb_permute_predict<Rec64>, dim3(L.parts.blocks), dim3(BS), 0, s, L.inst,
                       L.parts.m);
  else
    hipLaunchKernelGGL(kb_permute_predict<Rec32>, dim3(L.parts.blocks), dim3(BS), 0, s, L.inst,
                       L.parts.m);
}

}  // namespace mfg
