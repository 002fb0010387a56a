// k_pair.hip -- neighbour lists, PSE heat, and the fused pair + particle update pass.
//
// Neighbour pass (replaces the candidate loops of src/interactions_gpu.cu:89-150,227-336):
//   for particle i in cell (gi, gj, gk) the reference visits cells (ii, jj, kk) of the 5x5x5
//   stencil in ascending order and, inside a cell, particles in sorted order.  Cells along kk are
//   contiguous in the sorted order, so each (ii, jj) pair is ONE contiguous particle range
//   [off[c(ii,jj,klo)], off[c(ii,jj,khi)+1]); the 25 ranges in (ii, jj) order reproduce the
//   reference's visiting order exactly.  Candidates are kept if not blanked and inside the
//   cubic-spline support (1e-8 <= r^2 < 4 h_i^2, src/kernels.cuh:41), the only pairs whose terms
//   are non-zero.  The PSE heat sum (no cutoff, blanked j included, src/interactions_gpu.cu:
//   124-147) runs in the same candidate loop.
//
// Pair pass (src/interactions_gpu.cu:152-471 + src/actions_gpu.cu:134-300,302-331,371-449 +
// src/leap_frog.cu:72-100): per particle, CSPM matrix, velocity gradient, stress divergence with
// Gray artificial stress, Monaghan viscosity, XSPH, Brookshaw heat over the neighbour list, then
// in registers: Jaumann rate, continuity, momentum, advection, NaN/Inf invalidation, leap-frog
// correction and the Johnson-Cook radial return (FP64).
//
// Precision: FP64 throughout, or (FP32 modes) the relative position in FP64, the pair arithmetic in
// FP32 and every neighbour sum compensated; the particle update stays FP64.
//
// The FP64 pair pass at 1M particles (single-grain cut, about 103 neighbours each): 2.07 -> 0.98-1.02
// ms against one lane per particle with a walk of its own for B and the reference's order of evaluation
// (385 vector instructions per neighbour step and 110 of the B walk, now 150 and none); 8,000
// particles 198 -> 22 us (125 wavefronts of 100 steps, now 500 of 26).  At 1M it runs at 18 TB/s of
// record reads from the L2s; vector units busy half of the time, the L1 and LDS paths about two
// thirds, at two waves per SIMD (45 FP64 sums a lane; compiled for three it spills: 4.15 ms).
// Workgroups of 512 threads: 1.10 ms.
#include <algorithm>
#include <type_traits>

#include "mfg_device.hpp"

namespace mfg {

constexpr int BSP = 256;
// minimum waves per SIMD the pair kernels are compiled for (register budget)
#ifndef PAIR_WAVES
#define PAIR_WAVES 2
#endif

// ---------------------------------------------------------------------------------------------
// exp(a) for a <= 0, table-driven (P. T. P. Tang, "Table-driven implementation of the exponential
// function in IEEE floating-point arithmetic", ACM TOMS 15(2), 1989): a = (64 m + j) ln2/64 + r
// with n = 64 m + j = rint(a 64/ln2) and |r| <= ln2/128 (two-part ln2/64, fused), then
// exp(a) = 2^m 2^(j/64) (1 + p(r)), p the degree-5 Taylor polynomial of exp(r) - 1 (truncation
// r^6/720 < 3.5e-17 at |r| = ln2/128).  2^(j/64) is held as lead + trail, and the result is
// lead + (lead p + trail): within 0.85 ulp (the general library routine: 1 ulp), in 19 vector
// instructions and one 16-byte LDS read against that routine's 32, which also handles a > 0 and
// the overflow range.  a is clamped at -746, where exp already rounds to 0; this keeps n in int
// range.  A NaN argument (only from a non-finite record, whose stencil the neighbour pass poisons)
// gives 0, not NaN.  tab: EXP2_J64 in LDS.
// EXP2_J64[j] = {lead, trail}: lead = 2^(j/64) and trail = 2^(j/64) - lead, and the ln2
// constants, each correctly rounded (checked against a 60-digit evaluation by
// tests/test_exp_table.py, which reads them from this file).
// BEGIN EXP TABLE
constexpr double EXP_INV_LN2_64 = 0x1.71547652b82fep+6;  // 64 / ln 2
constexpr double EXP_LN2_64_HI = 0x1.62e42fefa39efp-7;   // ln 2 / 64, leading part
constexpr double EXP_LN2_64_LO = 0x1.abc9e3b39803fp-62;  // ln 2 / 64 - EXP_LN2_64_HI
__constant__ double2 EXP2_J64[64] = {
    {0x1.0000000000000p+0, 0x0p+0}, {0x1.02c9a3e778061p+0, -0x1.19083535b085dp-56},
    {0x1.059b0d3158574p+0, 0x1.d73e2a475b465p-55}, {0x1.0874518759bc8p+0, 0x1.186be4bb284ffp-57},
    {0x1.0b5586cf9890fp+0, 0x1.8a62e4adc610bp-54}, {0x1.0e3ec32d3d1a2p+0, 0x1.03a1727c57b53p-59},
    {0x1.11301d0125b51p+0, -0x1.6c51039449b3ap-54}, {0x1.1429aaea92de0p+0, -0x1.32fbf9af1369ep-54},
    {0x1.172b83c7d517bp+0, -0x1.19041b9d78a76p-55}, {0x1.1a35beb6fcb75p+0, 0x1.e5b4c7b4968e4p-55},
    {0x1.1d4873168b9aap+0, 0x1.e016e00a2643cp-54}, {0x1.2063b88628cd6p+0, 0x1.dc775814a8495p-55},
    {0x1.2387a6e756238p+0, 0x1.9b07eb6c70573p-54}, {0x1.26b4565e27cddp+0, 0x1.2bd339940e9d9p-55},
    {0x1.29e9df51fdee1p+0, 0x1.612e8afad1255p-55}, {0x1.2d285a6e4030bp+0, 0x1.0024754db41d5p-54},
    {0x1.306fe0a31b715p+0, 0x1.6f46ad23182e4p-55}, {0x1.33c08b26416ffp+0, 0x1.32721843659a6p-54},
    {0x1.371a7373aa9cbp+0, -0x1.63aeabf42eae2p-54}, {0x1.3a7db34e59ff7p+0, -0x1.5e436d661f5e3p-56},
    {0x1.3dea64c123422p+0, 0x1.ada0911f09ebcp-55}, {0x1.4160a21f72e2ap+0, -0x1.ef3691c309278p-58},
    {0x1.44e086061892dp+0, 0x1.89b7a04ef80d0p-59}, {0x1.486a2b5c13cd0p+0, 0x1.3c1a3b69062f0p-56},
    {0x1.4bfdad5362a27p+0, 0x1.d4397afec42e2p-56}, {0x1.4f9b2769d2ca7p+0, -0x1.4b309d25957e3p-54},
    {0x1.5342b569d4f82p+0, -0x1.07abe1db13cadp-55}, {0x1.56f4736b527dap+0, 0x1.9bb2c011d93adp-54},
    {0x1.5ab07dd485429p+0, 0x1.6324c054647adp-54}, {0x1.5e76f15ad2148p+0, 0x1.ba6f93080e65ep-54},
    {0x1.6247eb03a5585p+0, -0x1.383c17e40b497p-54}, {0x1.6623882552225p+0, -0x1.bb60987591c34p-54},
    {0x1.6a09e667f3bcdp+0, -0x1.bdd3413b26456p-54}, {0x1.6dfb23c651a2fp+0, -0x1.bbe3a683c88abp-57},
    {0x1.71f75e8ec5f74p+0, -0x1.16e4786887a99p-55}, {0x1.75feb564267c9p+0, -0x1.0245957316dd3p-54},
    {0x1.7a11473eb0187p+0, -0x1.41577ee04992fp-55}, {0x1.7e2f336cf4e62p+0, 0x1.05d02ba15797ep-56},
    {0x1.82589994cce13p+0, -0x1.d4c1dd41532d8p-54}, {0x1.868d99b4492edp+0, -0x1.fc6f89bd4f6bap-54},
    {0x1.8ace5422aa0dbp+0, 0x1.6e9f156864b27p-54}, {0x1.8f1ae99157736p+0, 0x1.5cc13a2e3976cp-55},
    {0x1.93737b0cdc5e5p+0, -0x1.75fc781b57ebcp-57}, {0x1.97d829fde4e50p+0, -0x1.d185b7c1b85d1p-54},
    {0x1.9c49182a3f090p+0, 0x1.c7c46b071f2bep-56}, {0x1.a0c667b5de565p+0, -0x1.359495d1cd533p-54},
    {0x1.a5503b23e255dp+0, -0x1.d2f6edb8d41e1p-54}, {0x1.a9e6b5579fdbfp+0, 0x1.0fac90ef7fd31p-54},
    {0x1.ae89f995ad3adp+0, 0x1.7a1cd345dcc81p-54}, {0x1.b33a2b84f15fbp+0, -0x1.2805e3084d708p-57},
    {0x1.b7f76f2fb5e47p+0, -0x1.5584f7e54ac3bp-56}, {0x1.bcc1e904bc1d2p+0, 0x1.23dd07a2d9e84p-55},
    {0x1.c199bdd85529cp+0, 0x1.11065895048ddp-55}, {0x1.c67f12e57d14bp+0, 0x1.2884dff483cadp-54},
    {0x1.cb720dcef9069p+0, 0x1.503cbd1e949dbp-56}, {0x1.d072d4a07897cp+0, -0x1.cbc3743797a9cp-54},
    {0x1.d5818dcfba487p+0, 0x1.2ed02d75b3707p-55}, {0x1.da9e603db3285p+0, 0x1.c2300696db532p-54},
    {0x1.dfc97337b9b5fp+0, -0x1.1a5cd4f184b5cp-54}, {0x1.e502ee78b3ff6p+0, 0x1.39e8980a9cc8fp-55},
    {0x1.ea4afa2a490dap+0, -0x1.e9c23179c2893p-54}, {0x1.efa1bee615a27p+0, 0x1.dc7f486a4b6b0p-54},
    {0x1.f50765b6e4540p+0, 0x1.9d3e12dd8a18bp-54}, {0x1.fa7c1819e90d8p+0, 0x1.74853f3a5931ep-55},
};
// END EXP TABLE

// In two halves, so that a wavefront starts the table reads of a whole particle group before it
// needs the first (waiting on each read where it is issued left the LDS latency exposed: slower
// than the library routine despite fewer instructions).  exp_reduce: n, r and the table read;
// exp_finish: the polynomial and the scaling.  n is rounded by adding 1.5 2^52, whose low mantissa
// word then holds it as an integer.
struct ExpPart {
  double r;
  int n;
  double2 s;
};
__device__ __forceinline__ ExpPart exp_reduce(double a, const double2 *tab) {
  a = __builtin_fmax(a, -746.);
  const double t = __builtin_fma(a, EXP_INV_LN2_64, 0x1.8p52);
  const double n = t - 0x1.8p52;
  ExpPart e;
  e.r = __builtin_fma(-n, EXP_LN2_64_LO, __builtin_fma(-n, EXP_LN2_64_HI, a));
  e.n = (int)__builtin_bit_cast(long long, t);
  e.s = tab[e.n & 63];
  return e;
}
__device__ __forceinline__ double exp_finish(const ExpPart &e) {
  const double r = e.r;
  double p = __builtin_fma(r, 1. / 120., 1. / 24.);
  p = __builtin_fma(p, r, 1. / 6.);
  p = __builtin_fma(p, r, 0.5);
  p = __builtin_fma(p, r, 1.);
  p = p * r;
  return __builtin_ldexp(e.s.x + __builtin_fma(e.s.x, p, e.s.y), e.n >> 6);
}

// ---------------------------------------------------------------------------------------------
// One wavefront per cell.  All particles of a cell share the 25 candidate ranges (in the reference's
// visiting order) and the wave's lanes take candidates: the candidate loads are coalesced.  The
// cell's particles are taken in groups of up to NB_GROUP; each 64-candidate chunk is loaded once
// (ahead, while the chunk before it is worked on) and tested against every particle of the group, which
// amortises the loads and gives the wave independent work to overlap.  For each particle the ballot
// of the kept candidates appends them in order to its row-major list; its PSE sum is a per-lane
// partial reduced over the wave.
//   PSE_MODE 0: no PSE sum; 1: FP64 PSE terms; 2: FP32 PSE terms accumulated in FP64
// Bound by vector issue (84 % busy at 1M).  1M single-grain cut, FP64 1.27 -> 0.94 ms, FP32 0.92 ->
// 0.74 ms, 65k FP64 131 -> 99 us: a group of four against 64 candidates took 211 vector instructions
// and 28 LDS reads with its particles' data in LDS, a branch per particle and the candidates listed
// in LDS beforehand; now 181 and 2 (+ 4 table reads), the listing included.
// Cells (wavefronts) per workgroup: neighbouring cells on one compute unit share most of their
// candidates in its L1.  1M cut, FP64 / FP32: one 0.91 / 0.75 ms, two 0.83 / 0.68, three 0.83 / 0.66,
// four 0.84 / 0.66, eight 0.90 / 0.71; 24 batched wedges 0.54, 0.52, 0.53, 0.54, 0.61.
constexpr int NB_WAVES = 3;
constexpr int NB_BLOCK = 64 * NB_WAVES;
#ifndef NB_GROUP_SIZE
#define NB_GROUP_SIZE 4
#endif
constexpr int NB_GROUP = NB_GROUP_SIZE;  // particles of a cell tested per candidate load

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Candidate q of a cell's list as the neighbour pass needs it: particle index, (x, y, z, flag)
// and (T, m / rho).
struct NbCand {
  int j;
  double4 pj;
  double2 tr;
};

// inclusive scan over the wavefront of ints >= 0: sums, or the largest so far
template <bool MAX>
__device__ __forceinline__ int wave_scan(int v) {
  auto step = [&](auto ctrl, auto rows) {
    const int t = __builtin_amdgcn_update_dpp(0, v, decltype(ctrl)::value, decltype(rows)::value, 0xf, false);
    v = MAX ? max(v, t) : v + t;
  };
  step(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{});  // row_shr 1, 2, 4, 8
  step(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});
  step(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});
  step(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});
  step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});  // row_bcast 15, 31
  step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
  return v;
}

// v of the lane at a fixed distance inside its row of 16
template <int CTRL>
__device__ __forceinline__ double dpp64(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// exchanges rows of 16 or 32 lanes between two registers and adds them: of 32, lanes 0-31 get
// a(l) + a(l + 32) and lanes 32-63 b(l - 32) + b(l); of 16, rows 0 and 2 get a's row pairs, rows 1
// and 3 b's
template <int ROWS>
__device__ __forceinline__ double swap_add(double a, double b) {
  const long long ia = __builtin_bit_cast(long long, a), ib = __builtin_bit_cast(long long, b);
  auto swap = [](unsigned x, unsigned y) {
    if constexpr (ROWS == 32) return __builtin_amdgcn_permlane32_swap(x, y, false, false);
    else return __builtin_amdgcn_permlane16_swap(x, y, false, false);
  };
  const auto lo = swap((unsigned)ia, (unsigned)ib), hi = swap((unsigned)(ia >> 32), (unsigned)(ib >> 32));
  return __builtin_bit_cast(double, (unsigned long long)hi[0] << 32 | lo[0]) +
         __builtin_bit_cast(double, (unsigned long long)hi[1] << 32 | lo[1]);
}

// The sums over the wavefront of four values: row r of 16 lanes gets that of a[row_sum_of(r)].  9
// instructions for the first two halvings of all four and 12 for the last four, against 18 per value.
constexpr int row_sum_of(int row) { return row == 1 ? 2 : row == 2 ? 1 : row; }
__device__ __forceinline__ double row_sums(const double a[4]) {
  double v = swap_add<16>(swap_add<32>(a[0], a[1]), swap_add<32>(a[2], a[3]));
  v += dpp64<0x128>(v);  // row_ror 8, 4, 2, 1
  v += dpp64<0x124>(v);
  v += dpp64<0x122>(v);
  v += dpp64<0x121>(v);
  return v;
}

// lane u's value in every lane, as a scalar
__device__ __forceinline__ double read_lane(double v, int u) {
  const long long b = __builtin_bit_cast(long long, v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, u);
  const unsigned hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), u);
  return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}

// The particles [s, e) of one cell against its T candidates (fetch(b0) gives each lane candidate
// b0 + lane, or past T any readable record, masked off; b0 ascends by 64 from 0): support test, PSE
// sum, ordered list write.  A group's
// particle data are scalars: read from LDS for every chunk of candidates they were two thirds of the
// LDS traffic, which returns a value per lane also where all lanes read one address.
template <int PSE_MODE, class Fetch>
__device__ __forceinline__ void cell_lists(int s, int e, int T, int lane, Fetch &&fetch, const double4 *__restrict__ nl4,
                                           const double2 *__restrict__ pse2,
                                           const double *__restrict__ h,
                                           const uint32_t *__restrict__ flags, const Consts &c,
                                           int *__restrict__ nbr, int cap, int *__restrict__ count,
                                           double *__restrict__ T_t, Counters *cnt,
                                           int *__restrict__ poison, const double2 *exp_tab,
                                           unsigned long long &n_cand, unsigned long long &n_pair) {
  static_assert(NB_GROUP == 4, "row_sums");
  // a group of GN particles from g0: GN is a compile-time constant, so that the work on one candidate
  // for all of them is one block of independent chains (behind a branch each, they ran one after the
  // other)
  auto group = [&](const int g0, auto gn_c) {
    constexpr int gn = decltype(gn_c)::value;
    // lane u: particle u of the group (the others repeat the last)
    const int pl = g0 + min(lane, gn - 1);
    const double4 pi = nl4[pl];
    const double hi = h[pl], h2 = hi * hi;
    double Tl = 0., il = 0., cl = 0.;
    if (PSE_MODE) {
      Tl = pse2[pl].x;
      il = rcp64(h2);
    }
    if (PSE_MODE == 2) cl = +4. / (hi * (h2 * h2) * PI_D * sqrt_rn(PI_D));
    // squared support; -1 (no candidate is inside) for a particle that gets no list: blanked, or its
    // own record non-finite.  A NaN smoothing length excludes nothing, so that its NaN reaches the sums
    // (rr2 >= 4 h^2 is false, src/kernels.cuh:41).  Not by fmin: the code around it gets worse (24 batched
    // wedges 530 us, 570 with fmin, 532 so).
    double fl = pi.w == 0. ? 4 * hi * hi : -1.;
    fl = isnan(fl) ? 0x1p1023 : fl;
    // per particle of the group (all wave-uniform but the PSE partial): position, squared support,
    // temperature, 1 / h^2, the FP32 PSE constants, list length so far
    double px[gn], py[gn], pz[gn], p4h2[gn], pT[gn], pih2[gn];
    float pc_f[gn], pih2_f[gn];
    int np[NB_GROUP] = {0, 0, 0, 0};
    double acc[NB_GROUP] = {0., 0., 0., 0.};
    int *const rows = nbr + (size_t)g0 * cap;
#pragma unroll
    for (int u = 0; u < gn; u++) {
      px[u] = read_lane(pi.x, u);
      py[u] = read_lane(pi.y, u);
      pz[u] = read_lane(pi.z, u);
      p4h2[u] = read_lane(fl, u);
      pT[u] = read_lane(Tl, u);
      pih2[u] = read_lane(il, u);
      pc_f[u] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, (float)cl), u));
      pih2_f[u] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, (float)il), u));
    }
    // a non-finite record among the candidates poisons every particle of the group (they share
    // the stencil)
    unsigned long long bad = 0;
    // one chunk of 64 candidates against the group; TAIL: the last chunk, lanes past T masked
    auto chunk = [&](const int b0, const NbCand &cd, auto tail) {
      constexpr bool TAIL = decltype(tail)::value;
      const bool valid = !TAIL || b0 + lane < T;
      const int j = cd.j;
      const double4 pj = cd.pj;
      double2 tr = cd.tr;
      unsigned long long in_chunk = ~0ull;
      if (TAIL) in_chunk = __builtin_amdgcn_ballot_w64(valid);
      const unsigned long long cand_ok = __builtin_amdgcn_ballot_w64(pj.w == 0.) & in_chunk;
      bad |= __builtin_amdgcn_ballot_w64(pj.w == 2.) & in_chunk;
      // masked lanes add zero, also where the record they hold is of an infinite temperature
      if (PSE_MODE && TAIL) tr = valid ? tr : make_double2(0., 0.);
      float try_f = 0.f;
      if (PSE_MODE == 2) try_f = (float)tr.y;
      // lapl_pse (src/kernels.cuh:71-92) times (T_j - T_i) m / rho_j
      // (src/interactions_gpu.cu:124-147); r^2 / h^2 as r^2 times 1 / h^2 and m / rho_j from the
      // record, each within two ulps of the reference's sqrt-square and divisions.  FP64: the kernel's
      // constant 4 / (h^5 pi sqrt(pi)) multiplies the sum; the exp of every particle of the
      // group is reduced (table reads started) in the first loop and finished in the second.
      ExpPart ex[gn];
#pragma unroll
      for (int u = 0; u < gn; u++) {
        const double xij = px[u] - pj.x, yij = py[u] - pj.y, zij = pz[u] - pj.z;
        const double rr2 = xij * xij + yij * yij + zij * zij;
        if (PSE_MODE == 1) ex[u] = exp_reduce(-rr2 * pih2[u], exp_tab);
        if (PSE_MODE == 2) {
          const float w2 = pc_f[u] * __expf(-(float)rr2 * pih2_f[u]);
          acc[u] += (double)((float)(tr.x - pT[u]) * w2 * try_f);
        }
        // ordered compaction: the candidates inside the support (src/kernels.cuh:41) go to the row in
        // lane order
        const unsigned long long m = __builtin_amdgcn_ballot_w64(rr2 < p4h2[u]) &
                                     ~__builtin_amdgcn_ballot_w64(rr2 < 1e-8) & cand_ok;
        const int n = __popcll(m);
        const unsigned pos = __builtin_amdgcn_mbcnt_hi(
            (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, (unsigned)(np[u] + u * cap)));
        if (np[u] + n <= cap) {
          if (__builtin_amdgcn_inverse_ballot_w64(m)) rows[pos] = j;
        } else if (__builtin_amdgcn_inverse_ballot_w64(m) && (int)pos < (u + 1) * cap) {
          rows[pos] = j;
        }
        np[u] += n;
      }
      if (PSE_MODE == 1) {
#pragma unroll
        for (int u = 0; u < gn; u++)
          acc[u] = __builtin_fma(tr.y * exp_finish(ex[u]), tr.x - pT[u], acc[u]);
      }
    };
    // the next chunk's candidates are loaded while a chunk is worked on
    NbCand cd = fetch(0);
    int b0 = 0;
    for (; b0 + 64 <= T; b0 += 64) {
      const NbCand nx = fetch(b0 + 64);
      chunk(b0, cd, std::false_type{});
      cd = nx;
    }
    if (b0 < T) chunk(b0, cd, std::true_type{});
    // row r of 16 lanes ends with the sum of particle row_sum_of(r), whose results its first lane
    // writes
    double sum = 0.;
    if (PSE_MODE) sum = row_sums(acc);
    const int row_id = lane >> 4;
    const int u = row_sum_of(row_id);
    const int n_u = u == 0 ? np[0] : u == 1 ? np[1] : u == 2 ? np[2] : np[3];
    if ((lane & 15) == 0 && u < gn) {
      const int p = g0 + u;
      poison[p] = bad != 0 ? 1 : 0;
      if (n_u > cap) {
        atomicOr(&cnt->err_capacity, 1);
        atomicMax(&cnt->max_count, n_u);
      }
      count[p] = min(n_u, cap);
      if (PSE_MODE) {
        if (PSE_MODE == 1) {
          const double hi = h[p], h2 = hi * hi;
          sum *= 4. * rcp64(h2 * h2 * hi * (PI_D * 1.7724538509055160273));  // sqrt(pi)
        }
        T_t[p] = ((flags[p] & FL_TOOL) ? c.alpha_tool : c.alpha_wp) * sum;
      }
    }
#pragma unroll
    for (int v = 0; v < gn; v++) {
      n_cand += (unsigned long long)T;
      n_pair += (unsigned long long)min(np[v], cap);
    }
  };
  int g0 = s;
  for (; g0 + NB_GROUP <= e; g0 += NB_GROUP) group(g0, std::integral_constant<int, NB_GROUP>{});
  switch (e - g0) {
    case 1: group(g0, std::integral_constant<int, 1>{}); break;
    case 2: group(g0, std::integral_constant<int, 2>{}); break;
    case 3: group(g0, std::integral_constant<int, 3>{}); break;
  }
}

// The candidate ranges of one cell: for stencil column r = lane < nr, the particles of rows
// [lo_k, hi_k) of grid column (lo_i + r / nj, lo_j + r % nj): each lane's first particle st, their
// number len and the exclusive prefix ex of the lengths; returns their sum T.
__device__ __forceinline__ int cell_ranges(const GridInfo &g, const int *__restrict__ off, int lane,
                                           int lo_i, int lo_j, int nj, int nr, int lo_k, int hi_k,
                                           int &st, int &len, int &ex) {
  const int nyz = g.ny * g.nz;
  st = 0;
  len = 0;
  if (lane < nr) {
    const int q = nj == 5 ? (lane * 52) >> 8 : lane / nj;  // lane / 5 for lane < 25
    const long cb = (long)(lo_i + q) * nyz + (long)(lo_j + lane - q * nj) * g.nz;
    st = off[cb + lo_k];
    len = off[cb + hi_k] - st;
  }
  const int incl = wave_scan<false>(len);  // lanes from nr on hold 0
  ex = incl - len;
  return __builtin_amdgcn_readlane(incl, 63);
}

// minimum waves per SIMD the kernel is compiled for (register budget): FP64 PSE 6, the others 7;
// 1M single-grain cut FP64 0.83 ms (5 waves 0.88), FP32 0.66 (8 waves 0.78)
#ifndef NB_WAVES_FP64_PSE
#define NB_WAVES_FP64_PSE 6
#endif
#ifndef NB_WAVES_OTHER
#define NB_WAVES_OTHER 7
#endif
// Body of workgroup b of nb (the single-instance kernel and the batched one below): each wavefront takes
// one cell of the occupied ones (occ, ascending; the scan of the sort lists them), each XCD one
// contiguous eighth of the list.  The launch is sized for the most cells the particles can occupy, not
// for the grid: its margins around the block are three quarters of the cells of a wedge cut.  Where that
// is more than a launch holds (NB_MOST_BLOCKS), further launches take the cells that follow (first: workgroups
// of the launches before; a loop in the kernel spills: FP64 PSE 6 registers, then 14).  Against
// a wavefront for every cell: 8,000 particles 27 -> 13 us, 19,000 35 -> 18, 64,000 with PSE 100 -> 65;
// 24 batched wedges, where a wavefront took 16 cells in turn, 0.77 -> 0.53 ms.
template <int PSE_MODE, bool FAR>
__device__ __forceinline__ void cell_neighbours(
    unsigned b, const GridInfo &g, const int *__restrict__ off, const int *__restrict__ occ,
    const double4 *__restrict__ nl4, const double2 *__restrict__ pse2,
    const double *__restrict__ h, const uint32_t *__restrict__ flags, const Consts &c,
    int *__restrict__ nbr, int cap, int *__restrict__ count, double *__restrict__ T_t,
    Counters *cnt, unsigned long long *__restrict__ stat_part, int *__restrict__ poison) {
  __shared__ int s_start[NB_WAVES][64];
  __shared__ unsigned long long s_stat[NB_WAVES][2];
  __shared__ double2 s_exp[PSE_MODE == 1 ? 64 : 1];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (PSE_MODE == 1) {
    if (threadIdx.x < 64) s_exp[threadIdx.x] = EXP2_J64[threadIdx.x];
    __syncthreads();
  }
  // workgroups x, x + 8, ... (XCD x) take the list's groups of NB_WAVES cells from x per on
  const unsigned n_occ = min((unsigned)occ[g.num_cell], (unsigned)g.num_cell);
  const unsigned groups = (n_occ + NB_WAVES - 1) / NB_WAVES;
  const unsigned per = (groups + 7) / 8, slot = b >> 3, at = ((b & 7) * per + slot) * NB_WAVES + w;
  unsigned long long n_cand = 0, n_pair = 0;
  // the particles [s, e) of one cell against its stencil's candidates
  auto do_cell = [&](const long c_, const int s, const int e) {
    const unsigned cell = (unsigned)c_, nyz = (unsigned)(g.ny * g.nz);  // cell hashes are 32-bit
    const int gi = (int)(cell / nyz), rem = (int)(cell - gi * nyz);
    const int gj = rem / g.nz, gk = rem - gj * g.nz;
    const int lo_i = gi - 2 < 0 ? 0 : gi - 2, hi_i = gi + 3 > g.nx ? g.nx : gi + 3;
    const int lo_j = gj - 2 < 0 ? 0 : gj - 2, hi_j = gj + 3 > g.ny ? g.ny : gj + 3;
    const int lo_k = gk - 2 < 0 ? 0 : gk - 2, hi_k = gk + 3 > g.nz ? g.nz : gk + 3;
    const int nj = hi_j - lo_j, nr = (hi_i - lo_i) * nj;
    int st, len, ex;
    const int T = cell_ranges(g, off, lane, lo_i, lo_j, nj, nr, lo_k, hi_k, st, len, ex);
    // Candidate q of range r is particle q + (st - ex), and st - ex ascends over the non-empty
    // ranges: of the 64 candidates from b0, those a range starts at get its st - ex from LDS, the rest
    // by a running maximum (16 instructions, against a loop over the 25 ranges before).
    int carry = 0;
    auto fetch = [&](int b0) {
      if (b0 == 0) carry = 0;
      s_start[w][lane] = 0;
      wave_lds_sync();
      if (len > 0 && (unsigned)(ex - b0) < 64u) s_start[w][ex - b0] = st - ex;
      wave_lds_sync();
      const int d = max(wave_scan<true>(s_start[w][lane]), carry);
      wave_lds_sync();
      carry = __builtin_amdgcn_readlane(d, 63);
      const int q = b0 + lane;
      NbCand cd;
      cd.j = q < T ? d + q : s;
      // byte offsets of 32 bits up to 2^27 particles (neighbours_far): 64 bits cost 1M FP64 with PSE 0.79 ->
      // 0.83 ms, 65k 63 -> 66 us
      typedef std::conditional_t<FAR, uint64_t, unsigned> Offset;
      cd.pj = *(const double4 *)((const char *)nl4 + (Offset)(unsigned)cd.j * 32u);
      cd.tr = make_double2(0., 1.);
      if (PSE_MODE) cd.tr = *(const double2 *)((const char *)pse2 + (Offset)(unsigned)cd.j * 16u);
      return cd;
    };
    cell_lists<PSE_MODE>(s, e, T, lane, fetch, nl4, pse2, h, flags, c, nbr, cap, count,
                         T_t, cnt, poison, s_exp, n_cand, n_pair);
  };
  if (slot < per && at < n_occ) {
    const int cell = occ[at];
    do_cell(cell, off[cell], off[cell + 1]);
  }
  if (!stat_part) return;
  // candidate / pair totals of this workgroup (work accounting of the roofline figures)
  if (lane == 0) {
    s_stat[w][0] = n_cand;
    s_stat[w][1] = n_pair;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long a = 0, bb = 0;
#pragma unroll
    for (int k = 0; k < NB_WAVES; k++) {
      a += s_stat[k][0];
      bb += s_stat[k][1];
    }
    stat_part[2 * (size_t)b] = a;
    stat_part[2 * (size_t)b + 1] = bb;
  }
}
template <int PSE_MODE, bool FAR>
__global__ void __launch_bounds__(NB_BLOCK)
    __attribute__((amdgpu_waves_per_eu(PSE_MODE == 1 ? NB_WAVES_FP64_PSE : NB_WAVES_OTHER)))
    k_cell_neighbours(unsigned first, GridInfo g, const int *__restrict__ off, const int *__restrict__ occ,
                      const double4 *__restrict__ nl4,
                      const double2 *__restrict__ pse2, const double *__restrict__ h,
                      const uint32_t *__restrict__ flags, Consts c, int *__restrict__ nbr, int cap,
                      int *__restrict__ count, double *__restrict__ T_t, Counters *cnt,
                      unsigned long long *__restrict__ stat_part, int *__restrict__ poison) {
  cell_neighbours<PSE_MODE, FAR>(first + blockIdx.x, g, off, occ, nl4, pse2, h, flags, c, nbr, cap, count, T_t, cnt,
                            stat_part, poison);
}

// ---------------------------------------------------------------------------------------------
// particle update after the neighbour sums (FP64 for both precisions)
struct PairSums {
  M3 vd, sd;
  double vt[3], xt[3], Tl;
};

// x: the new position; false if the particle was invalidated
__device__ __forceinline__ bool particle_update(const State &st, unsigned i, uint32_t fl,
                                                const Consts &c, const PairSums &ps,
                                                bool brook, double thermal_alpha, double (&x)[3]) {
  const bool tool = (fl & FL_TOOL) != 0;
  const double dt = c.dt, hdt = 0.5 * c.dt;
  double x0[3] = {st.x[i], st.y[i], st.z[i]};
  double v0[3] = {st.vx[i], st.vy[i], st.vz[i]};
  double S0[6], Sto[6];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    S0[k] = st.S[k][i];
    Sto[k] = st.St[k][i];
  }
  double vto[3] = {st.vxt[i], st.vyt[i], st.vzt[i]};
  double rho0 = st.rho[i], T0 = st.T[i], rho_to = st.rho_t[i], T_to = st.T_t[i];
  double nxt[3], nvt[3], nSt[6], nrho_t, nT_t;
  if (!tool) {
    double Sh[6], vh[3];
#pragma unroll
    for (int k = 0; k < 6; k++) Sh[k] = S0[k] + hdt * Sto[k];
#pragma unroll
    for (int k = 0; k < 3; k++) vh[k] = v0[k] + hdt * vto[k];
    double rhoh = rho0 + hdt * rho_to;
    // Jaumann, continuity, momentum, advection (src/actions_gpu.cu:134-300)
    jaumann(c.a_G, ps.vd, Sh, nSt);
    nrho_t = -rhoh * (ps.vd.m[0][0] + ps.vd.m[1][1] + ps.vd.m[2][2]);
    const double m = c.a_mass;
    double fc[3] = {st.fcx[i], st.fcy[i], st.fcz[i]};
    double ft[3] = {st.ftx[i], st.fty[i], st.ftz[i]};
#pragma unroll
    for (int a = 0; a < 3; a++) {
      nvt[a] = ps.vt[a] + (ps.sd.m[a][0] + ps.sd.m[a][1] + ps.sd.m[a][2] + fc[a] / m + ft[a] / m);
      nxt[a] = ps.xt[a] + vh[a];
    }
  } else {
#pragma unroll
    for (int a = 0; a < 3; a++) {
      nvt[a] = ps.vt[a];
      nxt[a] = ps.xt[a];
    }
#pragma unroll
    for (int k = 0; k < 6; k++) nSt[k] = Sto[k];
    nrho_t = rho_to;
  }
  nT_t = brook ? thermal_alpha * ps.Tl : T_to;
  st.xt[i] = nxt[0]; st.yt[i] = nxt[1]; st.zt[i] = nxt[2];
  st.vxt[i] = nvt[0]; st.vyt[i] = nvt[1]; st.vzt[i] = nvt[2];
#pragma unroll
  for (int k = 0; k < 6; k++) st.St[k][i] = nSt[k];
  st.rho_t[i] = nrho_t;
  st.T_t[i] = nT_t;
  // debug_invalidate (src/actions_gpu.cu:302-331)
  auto bad = [](double v) { return isnan(v) || isinf(v); };
  bool invalid = bad(nxt[0]) || bad(nxt[1]) || bad(nxt[2]) || bad(nvt[0]) || bad(nvt[1]) ||
                 bad(nvt[2]) || bad(nSt[0]) || bad(nSt[1]) || bad(nSt[2]) || bad(nSt[3]) ||
                 bad(nSt[4]) || bad(nSt[5]) || bad(nrho_t) || bad(nT_t);
  if (invalid) {
    st.flags[i] = fl | FL_BLANKED;
    return false;
  }
  // correct (src/leap_frog.cu:72-100)
  double v[3], S[6];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    x[k] = x0[k] + dt * nxt[k];
    v[k] = v0[k] + dt * nvt[k];
  }
#pragma unroll
  for (int k = 0; k < 6; k++) S[k] = S0[k] + dt * nSt[k];
  double rho = rho0 + dt * nrho_t;
  double T = T0 + dt * nT_t;
  // Johnson-Cook radial return (src/actions_gpu.cu:371-449)
  if (c.plastic && !tool) jc_radial_return(c, dt, st, i, S, T, rho);
  st.x[i] = x[0]; st.y[i] = x[1]; st.z[i] = x[2];
  st.vx[i] = v[0]; st.vy[i] = v[1]; st.vz[i] = v[2];
#pragma unroll
  for (int k = 0; k < 6; k++) st.S[k][i] = S[k];
  st.rho[i] = rho;
  st.T[i] = T;
  return true;
}

// The pair kernels end by storing a particle's neighbour sums (SoA, PAIR_SUMS doubles per
// particle: vd[9], sd[9], vt[3], xt[3], Tl); the per-particle kernel below reads them back and
// runs the update.  Split this way, neither kernel carries the other's registers.
constexpr int PAIR_SUMS = 25;

__device__ __forceinline__ void store_sums(double *__restrict__ sums, size_t stride, unsigned i,
                                           const PairSums &ps) {
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) {
      sums[(3 * a + b) * stride + i] = ps.vd.m[a][b];
      sums[(9 + 3 * a + b) * stride + i] = ps.sd.m[a][b];
    }
#pragma unroll
  for (int a = 0; a < 3; a++) {
    sums[(18 + a) * stride + i] = ps.vt[a];
    sums[(21 + a) * stride + i] = ps.xt[a];
  }
  sums[24 * stride + i] = ps.Tl;
}

// Jaumann rate, continuity, momentum, advection, invalidation, leap-frog correction and the
// Johnson-Cook radial return of every particle the pair pass summed (not blanked, in a cell), and its
// entry in the contact search's list (list_n null: none)
__device__ __forceinline__ void update_body(unsigned b, unsigned n_init, const State &st,
                                            const double *__restrict__ sums, size_t stride,
                                            const int *__restrict__ poison, const Consts &c,
                                            const Counters *cnt, const ToolSet &ts,
                                            const ContactSearch &cs) {
  const unsigned i = b * blockDim.x + threadIdx.x;
  if (i >= cnt->N || i >= n_init) return;
  const uint32_t fl = st.flags[i];
  if (fl & FL_BLANKED) return;
  PairSums ps;
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) {
      ps.vd.m[a][b] = sums[(3 * a + b) * stride + i];
      ps.sd.m[a][b] = sums[(9 + 3 * a + b) * stride + i];
    }
#pragma unroll
  for (int a = 0; a < 3; a++) {
    ps.vt[a] = sums[(18 + a) * stride + i];
    ps.xt[a] = sums[(21 + a) * stride + i];
  }
  ps.Tl = sums[24 * stride + i];
  // a non-finite record in the particle's stencil: the reference's sums carry it (0 * NaN), so
  // its rates are non-finite and the invalidation blanks it
  if (poison[i]) ps.vd.m[0][0] = __builtin_nan("");
  const bool tool_nz = (fl & FL_TOOL_NZ) != 0;
  const double thermal_alpha = tool_nz ? c.alpha_tool : c.alpha_wp;
  const bool brook = c.heat == MFG_HEAT_BROOKSHAW && thermal_alpha != 0.;
  double x[3];
  if (particle_update(st, i, fl, c, ps, brook, thermal_alpha, x) && cs.list_n && !(fl & FL_TOOL))
    contact_list(i, v3(x[0], x[1], x[2]), n_init, ts, cs);
}
// The workgroups past the particles' move the tools' triangles, one a thread.  Both would be launches of
// their own, and a third to clear the list's counter (the permutation does): at 8,000 particles 13 us
// of launches against none measurable here, at 1M 17 against 2; 24 batched instances list 29 against 12.
__global__ void __launch_bounds__(BSP)
    k_particle_update(unsigned n_init, State st, const double *__restrict__ sums, size_t stride,
                      const int *__restrict__ poison, Consts c, const Counters *cnt, ToolSet ts,
                      ContactSearch cs, ToolMoves mv) {
  const unsigned blocks = (n_init + blockDim.x - 1) / blockDim.x;
  if (blockIdx.x < blocks) {
    update_body(blockIdx.x, n_init, st, sums, stride, poison, c, cnt, ts, cs);
    return;
  }
  const int k = (int)((blockIdx.x - blocks) * blockDim.x + threadIdx.x);
  int first = 0;
  for (int a = 0; a < mv.n; a++) {
    if (k >= first && k < mv.end[a]) move_tri(mv.tris[a], mv.p_init[a], k - first, mv.t, mv.vel[a]);
    first = mv.end[a];
  }
}

// ---------------------------------------------------------------------------------------------
// Neighbour sums of the pair pass.
//
// The reference walks the stencil twice: for the CSPM matrix B, then for sums of the corrected
// gradient w = B^-1 w0.  Every sum is linear in w, so the pass walks the list once and sums with
// the uncorrected gradient w0 instead, one sum per component c of w0; finish_sums applies B^-1
// (or the identity) once per particle.  The stress sum needs its symmetric 3x3 factor per
// component of w0 (6 x 3 sums), from which the neighbours' part alone is summed: the particle's own
// stress and artificial stress multiply sum(w0) and sum(f^4 w0) at the end.  Constant factors of a
// particle (kernel normalisation, mass, viscosity and XSPH factors) are applied at the end as well.
struct PairAcc {
  double W[3], F[3];  // sum w0_c, sum fab w0_c
  double M[6][3];     // sum (A_j + fab R_j)_ab w0_c
  double D[3][3];     // sum (v_j - v_i)_a vol_j w0_c
  double V[3];        // sum Pi_ij w0_c
  double X[3];        // sum W / (rho_i + rho_j) (v_j - v_i)_a
  double B[6];        // sum vol_j x_a w0_c (symmetric: w0 is along x)
  double Q[6];        // sum vol_j (T_i - T_j) / r^2 x_a w0_c (Brookshaw heat)
};

// the scale of w0 in PairAcc: the sums hold w0 = (dW/dq)(q) x / r without the kernel's
// normalisation and 1/h (k1), W without the normalisation (fac)
struct PairScale {
  double k1, fac, mass, eps;
};

// adds up the partial sums of a particle's lanes (4 or 16, aligned); every lane gets the total
template <int LANES>
__device__ __forceinline__ double lanes_sum(double v) {
  if (LANES == 16) {
    v += dpp64<0x140>(v);  // row_mirror: the other eight of a row
    v += dpp64<0x141>(v);  // row_half_mirror: the other quad of eight lanes
  }
  v += dpp64<0xb1>(v);  // quad_perm 1,0,3,2
  v += dpp64<0x4e>(v);  // quad_perm 2,3,0,1
  return v;
}

// the reference's sums of one particle from its PairAcc: B and its inverse
// (src/interactions_gpu.cu:262-292), then every sum with the corrected gradient
// (src/interactions_gpu.cu:294-471).  A, R: the particle's own stress terms and artificial stress.
template <bool BROOK>
__device__ __forceinline__ void finish_sums(const Consts &c, const PairAcc &p, const PairScale &k,
                                            const double A[6], const double R[6], bool tool_nz,
                                            bool brook, PairSums &ps) {
  M3 B, inv;
  constexpr int sym[3][3] = {{0, 3, 5}, {3, 1, 4}, {5, 4, 2}};
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) {
      B.m[a][b] = -(k.k1 * p.B[sym[a][b]]);
      inv.m[a][b] = a == b ? 1. : 0.;
    }
  // tool particles (tool != 0) keep the identity correction
  if (c.cspm && !tool_nz && det3(B) > 1e-8) inv3(B, inv);
  auto correct = [&](const double s[3], int b) {
    return __builtin_fma(s[2], inv.m[2][b], __builtin_fma(s[1], inv.m[1][b], s[0] * inv.m[0][b]));
  };
  const double km = k.mass * k.k1;
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) {
      const int ab = sym[a][b];
      ps.vd.m[a][b] = k.k1 * correct(p.D[a], b);
      double t[3];
#pragma unroll
      for (int q = 0; q < 3; q++)
        t[q] = __builtin_fma(A[ab], p.W[q], __builtin_fma(R[ab], p.F[q], p.M[ab][q]));
      ps.sd.m[a][b] = km * correct(t, b);
    }
  const double kx = 2. * k.eps * k.mass * k.fac;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    ps.vt[a] = -(km * correct(p.V, a));
    ps.xt[a] = kx * p.X[a];
  }
  ps.Tl = 0.;
  if (BROOK && brook) {
    double s = 0.;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const double q[3] = {p.Q[sym[a][0]], p.Q[sym[a][1]], p.Q[sym[a][2]]};
      s += correct(q, a);
    }
    ps.Tl = 2. * k.k1 * s;
  }
}

// r = sqrt(r2) as the reference's sqrt site evaluates it, and 1 / r.  single: the float root of
// the float-rounded r2.  From v_rsq_f32 with one residual step it equals the correctly rounded
// root for every mantissa and both exponent parities (all 2^24 compared with __builtin_sqrtf; r2 in
// a list is at least 1e-8, far from the denormals).  FP64: the coupled iteration from v_rsq_f64.
__device__ __forceinline__ void root64(double r2, int single, double &rad, double &rinv) {
  if (single) {
    const float x = (float)r2, y = __builtin_amdgcn_rsqf(x);
    float s = x * y;
    s = __builtin_fmaf(__builtin_fmaf(-s, s, x), 0.5f * y, s);
    rad = (double)s;
    const double r0 = (double)y;
    double d = __builtin_fma(-rad, r0, 1.);
    d = __builtin_fma(d, d, d);
    rinv = __builtin_fma(r0, d, r0);
  } else {
    const double y = __builtin_amdgcn_rsq(r2);
    double g = r2 * y, h = 0.5 * y;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    rad = __builtin_fma(__builtin_fma(-g, g, r2), h, g);
    h = 2. * h;
    rinv = __builtin_fma(h, __builtin_fma(-rad, h, 1.), h);
  }
}

// FP64 terms.  The spline as the difference of two truncated powers, W = (2-q)^3/4 - (1-q)_+^3:
// both branches without a selection.
template <bool BROOK>
struct Pair64 {
  double x, y, z, vx, vy, vz, rho, cs, h, T, h1, kfab;
  double va, vb, ve;
  int single;

  __device__ __forceinline__ Pair64(const Consts &c, const Rec64 &r)
      : x(r.x), y(r.y), z(r.z), vx(r.vx), vy(r.vy), vz(r.vz), rho(r.rho), cs(r.c), h(r.h), T(r.T) {
    h1 = 1. / h;
    const double fac = INV_PI_D * h1 * h1 * h1;
    kfab = c.wdeltap > 0 ? fac / c.wdeltap : 0.;
    // halves of the pair means folded into the constants: mu = (h_i + h_j) v.x / (2 D),
    // D = r^2 + eta^2 (h_i + h_j)^2 / 4, Pi = 2 mu (beta mu - alpha (c_i + c_j) / 2) / (rho_i + rho_j)
    va = c.v_alpha;
    vb = 2. * c.v_beta;
    ve = 0.25 * (c.v_eta * c.v_eta);
    single = c.single_sqrt;
  }
  __device__ __forceinline__ PairScale scale(const Consts &c) const {
    const double fac = INV_PI_D * h1 * h1 * h1;
    return {fac * h1, fac, c.i_mass, c.xspheps};
  }
  __device__ __forceinline__ void term(PairAcc &p, const Rec64 &j, bool mech) const {
    const double dx = x - j.x, dy = y - j.y, dz = z - j.z;
    const double r2 = dx * dx + dy * dy + dz * dz;  // rounded as the list's support test rounds it
    double rad, rinv;
    root64(r2, single, rad, rinv);
    const double q = rad * h1;
    const double a = 2. - q, b = __builtin_fmax(1. - q, 0.);
    const double a2 = a * a, b2 = b * b;
    const double val = __builtin_fma(a2, 0.25 * a, -(b2 * b));
    const double g = __builtin_fma(3., b2, -0.75 * a2) * rinv;
    const double w0[3] = {g * dx, g * dy, g * dz};
    const double vol = j.vol;
    if (BROOK) {
      const double s = vol * (T - j.T) * rcp64(r2);
      const double sx = s * dx, sy = s * dy, sz = s * dz;
      p.Q[0] = __builtin_fma(sx, w0[0], p.Q[0]);
      p.Q[1] = __builtin_fma(sy, w0[1], p.Q[1]);
      p.Q[2] = __builtin_fma(sz, w0[2], p.Q[2]);
      p.Q[3] = __builtin_fma(sx, w0[1], p.Q[3]);
      p.Q[4] = __builtin_fma(sy, w0[2], p.Q[4]);
      p.Q[5] = __builtin_fma(sx, w0[2], p.Q[5]);
    }
    if (!mech || j.tool == 1.) return;
    const double vw[3] = {vol * w0[0], vol * w0[1], vol * w0[2]};
    p.B[0] = __builtin_fma(dx, vw[0], p.B[0]);
    p.B[1] = __builtin_fma(dy, vw[1], p.B[1]);
    p.B[2] = __builtin_fma(dz, vw[2], p.B[2]);
    p.B[3] = __builtin_fma(dx, vw[1], p.B[3]);
    p.B[4] = __builtin_fma(dy, vw[2], p.B[4]);
    p.B[5] = __builtin_fma(dx, vw[2], p.B[5]);
    const double dv[3] = {j.vx - vx, j.vy - vy, j.vz - vz};
    double fab = val * kfab;
    fab *= fab;
    fab *= fab;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      p.W[k] += w0[k];
      p.F[k] = __builtin_fma(fab, w0[k], p.F[k]);
#pragma unroll
      for (int e = 0; e < 3; e++) p.D[e][k] = __builtin_fma(dv[e], vw[k], p.D[e][k]);
    }
#pragma unroll
    for (int e = 0; e < 6; e++) {
      const double t = __builtin_fma(fab, j.R[e], j.A[e]);
#pragma unroll
      for (int k = 0; k < 3; k++) p.M[e][k] = __builtin_fma(t, w0[k], p.M[e][k]);
    }
    // one reciprocal serves 1 / D and 1 / (rho_i + rho_j)
    const double vr = -__builtin_fma(dv[2], dz, __builtin_fma(dv[1], dy, dv[0] * dx));
    const double hs = h + j.h, rs = rho + j.rho;
    const double d = __builtin_fma(ve * hs, hs, r2);
    const double inv = rcp64(rs * d);
    const double irs = inv * d;
    const double mu = 0.5 * hs * __builtin_fmin(vr, 0.) * (inv * rs);
    // a pair that recedes has no viscosity, also where a sound speed is NaN (a negative density); selected
    // here and not at pi, which waits for the reciprocal (8,000 particles 21.4 us without, 21.6 with, 22.0 at pi)
    const double ca = vr < 0. ? cs + j.c : 0.;
    const double pi = mu * __builtin_fma(vb, mu, -va * ca) * irs;
    const double xw = val * irs;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      p.V[k] = __builtin_fma(pi, w0[k], p.V[k]);
      p.X[k] = __builtin_fma(xw, dv[k], p.X[k]);
    }
  }
};

// ---------------------------------------------------------------------------------------------
// Neighbour sums of one particle, FP32 pair arithmetic.  Positions stay FP64 until the relative
// position is formed; the pair arithmetic is FP32 (contracted to FMA); every neighbour sum is
// compensated, either
//   AccKahan  FP32 running sum with Kahan's correction term (4 operations per term), or
//   AccWide   the FP32 term widened and added in FP64 (2 operations per term: on CDNA4 an FP64
//             add issues at the FP32 rate; the summation error, n 2^-53 sum|t|, is below
//             Kahan's 2 2^-24 sum|t|).
struct AccKahan {
  float s, e;
  __device__ __forceinline__ void zero() { s = e = 0.f; }
  __device__ __forceinline__ void add(float v) {
    float y = v - e;
    float t = s + y;
    e = (t - s) - y;
    s = t;
  }
  __device__ __forceinline__ double val() const { return (double)s - (double)e; }
};
struct AccWide {
  double s;
  __device__ __forceinline__ void zero() { s = 0.; }
  __device__ __forceinline__ void add(float v) { s += (double)v; }
  __device__ __forceinline__ double val() const { return s; }
};

// The CSPM entry of a neighbour (cs4): position, tool flag and volume
struct ToolVol {
  float tool, vol;
};

// One neighbour's terms of every sum, in FP32.  Where they round is fixed: the Johnson-Cook solve of
// the update stops at 1e-6, so a sum that differs in its last bit can end it
// an iteration earlier and move a result by more than its rounding.
template <bool BROOK>
struct Pair32 {
  Rec32 ri;
  float h1, fac, mass, inv_wdp, eps, va, vb, ve2;
  float iB[9];  // inverse CSPM matrix, [col][row] flattened

  __device__ __forceinline__ Pair32(const Consts &c, const Rec32 &r) : ri(r) {
    h1 = __builtin_amdgcn_rcpf(ri.h);
    fac = (float)INV_PI_D * h1 * h1 * h1;
    mass = (float)c.i_mass;
    inv_wdp = c.wdeltap > 0 ? (float)(1.0 / c.wdeltap) : 0.f;
    eps = (float)c.xspheps;
    va = (float)c.v_alpha;
    vb = (float)c.v_beta;
    ve2 = (float)(c.v_eta * c.v_eta);
#pragma unroll
    for (int q = 0; q < 9; q++) iB[q] = (q % 4 == 0) ? 1.f : 0.f;
  }
  // r / h, rounded: never fused into what follows
  __device__ __forceinline__ float ratio(float rad) const { return rad * h1; }
  // derivative of the cubic spline over its factor: both branches are x y h1 / r
  __device__ __forceinline__ float spline_der(float q, float rinv) const {
#pragma clang fp contract(fast)
    const bool outer = q > 1.f;
    const float a = 2.f - q, b = 1.f - 0.75f * q;
    const float x = outer ? -0.75f * a : -3.0f * q;
    const float y = outer ? a : b;
    return x * y * h1 * rinv;
  }
  // x_first: r^2 begins with x^2 rounded and y^2 fused on, not the other way round
  __device__ __forceinline__ void cspm_term(const double4 &g, float vol, bool x_first, float (&b)[9]) const {
#pragma clang fp contract(fast)
    float xij = (float)(ri.x - g.x), yij = (float)(ri.y - g.y), zij = (float)(ri.z - g.z);
    const float u = x_first ? xij : yij, v = x_first ? yij : xij;
    float rr2 = __builtin_fmaf(zij, zij, __builtin_fmaf(v, v, u * u));
    float rad = __builtin_amdgcn_sqrtf(rr2);
    float rinv = __builtin_amdgcn_rcpf(rad);
    float dw = spline_der(ratio(rad), rinv) * fac * vol;
    float gx = dw * xij, gy = dw * yij, gz = dw * zij;
    b[0] = -xij * gx; b[3] = -xij * gy; b[6] = -xij * gz;
    b[1] = -yij * gx; b[4] = -yij * gy; b[7] = -yij * gz;
    b[2] = -zij * gx; b[5] = -zij * gy; b[8] = -zij * gz;
  }
  __device__ __forceinline__ void invert(const double (&B)[9]) {
    M3 Bd, inv;
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++) Bd.m[a][b] = B[3 * a + b];
    if (det3(Bd) > 1e-8) {
      inv3(Bd, inv);
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) iB[3 * a + b] = (float)inv.m[a][b];
    }
  }
  // v: the 24 mechanical terms by slot (0 .. 8 vd, 9 .. 17 sd, 18 19 23 xt, 20 .. 22 vt); approach: the viscous ones count; heat, hot: the
  // Brookshaw term and whether it counts
  __device__ __forceinline__ void term(const Rec32 &rj, float (&v)[24], bool &approach, float &heat,
                                       bool &hot) const {
#pragma clang fp contract(fast)
    float xij = (float)(ri.x - rj.x), yij = (float)(ri.y - rj.y), zij = (float)(ri.z - rj.z);
    float rr2 = xij * xij + yij * yij + zij * zij;
    float rad = __builtin_amdgcn_sqrtf(rr2);
    float rinv = __builtin_amdgcn_rcpf(rad);
    float q = ratio(rad);
    float a = 2.f - q;
    float v_out = 0.25f * a * a * a;
    float v_in = 1.f - 1.5f * q * q * (1.f - 0.5f * q);
    float w = (q > 1.f ? v_out : v_in) * fac;
    float d = spline_der(q, rinv) * fac;
    float wx0 = d * xij, wy0 = d * yij, wz0 = d * zij;
    float w_x = wx0 * iB[0] + wy0 * iB[3] + wz0 * iB[6];
    float w_y = wx0 * iB[1] + wy0 * iB[4] + wz0 * iB[7];
    float w_z = wx0 * iB[2] + wy0 * iB[5] + wz0 * iB[8];
    const float volj = rj.vol;
    float vijx = ri.vx - rj.vx, vijy = ri.vy - rj.vy, vijz = ri.vz - rj.vz;
    float dvx = -vijx * volj, dvy = -vijy * volj, dvz = -vijz * volj;
    v[0] = dvx * w_x; v[1] = dvx * w_y; v[2] = dvx * w_z;
    v[3] = dvy * w_x; v[4] = dvy * w_y; v[5] = dvy * w_z;
    v[6] = dvz * w_x; v[7] = dvz * w_y; v[8] = dvz * w_z;
    float fab = w * inv_wdp;
    fab *= fab;
    fab *= fab;
    float Rxx = fab * (ri.R[0] + rj.R[0]), Ryy = fab * (ri.R[1] + rj.R[1]);
    float Rzz = fab * (ri.R[2] + rj.R[2]), Rxy = fab * (ri.R[3] + rj.R[3]);
    float Ryz = fab * (ri.R[4] + rj.R[4]), Rxz = fab * (ri.R[5] + rj.R[5]);
    float mx = mass * w_x, my = mass * w_y, mz = mass * w_z;
    float Txx = ri.A[0] + rj.A[0] + Rxx, Tyy = ri.A[1] + rj.A[1] + Ryy, Tzz = ri.A[2] + rj.A[2] + Rzz;
    float Txy = ri.A[3] + rj.A[3] + Rxy, Tyz = ri.A[4] + rj.A[4] + Ryz, Txz = ri.A[5] + rj.A[5] + Rxz;
    v[9] = Txx * mx; v[10] = Txy * my; v[11] = Txz * mz;
    v[12] = Txy * mx; v[13] = Tyy * my; v[14] = Tyz * mz;
    v[15] = Txz * mx; v[16] = Tyz * my; v[17] = Tzz * mz;
    float vijposij = vijx * xij + vijy * yij + vijz * zij;
    float rhoij_inv = __builtin_amdgcn_rcpf(0.5f * (ri.rho + rj.rho));
    approach = vijposij < 0.f;
    float cij = 0.5f * (ri.c + rj.c);
    float hij = 0.5f * (ri.h + rj.h);
    float muij = (hij * vijposij) * __builtin_amdgcn_rcpf(rr2 + ve2 * hij * hij);
    float piij = (-va * cij * muij + vb * muij * muij) * rhoij_inv;
    float f = -mass * piij;
    v[20] = f * w_x;
    v[21] = f * w_y;
    v[22] = f * w_z;
    float g = -eps * w * mass * rhoij_inv;
    v[18] = g * vijx;
    v[19] = g * vijy;
    v[23] = g * vijz;
    if (BROOK) {
      float e_w = (xij * w_x + yij * w_y + zij * w_z) * rinv;
      heat = 2.0f * rj.vol * (ri.T - rj.T) * rinv * e_w;
      hot = rad > 1e-8f;
    }
  }
};

// ---------------------------------------------------------------------------------------------
// Visiting order of the list-gather pair pass.  In the sorted order (x slowest, then y, then z)
// a neighbour record is read again by the particles of the 5 x 5 grid columns around it, up to
// four x-rows later; for a 1M-particle block that window holds about 7 MB of FP64 records, more
// than the 4 MB L2 of an XCD, so records are fetched again from beyond the L2.  The pass
// therefore visits the particles in strips of `strip` grid columns along y: strip by strip, and
// inside a strip x-row by x-row.  Each (strip, x-row) segment is one contiguous range of the
// sorted order, and the window shrinks to about 5 x (strip + 4) columns.  trav[t] is the
// particle visited at position t < N.  The order changes which particle a thread takes, never
// the sums of a particle.
constexpr int TRAV_BLOCK = 1024;

__device__ __forceinline__ int trav_segment_start(const GridInfo &g, const int *off, int strip,
                                                  int q, int &size) {
  const int nx = g.nx, s = q / nx, gi = q - s * nx;
  const int j0 = s * strip, j1 = min(j0 + strip, g.ny);
  const int a = off[((long)gi * g.ny + j0) * g.nz], b = off[((long)gi * g.ny + j1) * g.nz];
  size = b - a;
  return a;
}

// exclusive prefix of the segment sizes in visiting order (segment q = strip * nx + x-row);
// one workgroup
__global__ void __launch_bounds__(TRAV_BLOCK)
    k_trav_segments(GridInfo g, const int *__restrict__ off, int strip, int nseg,
                    int *__restrict__ seg_pos) {
  __shared__ int s_part[TRAV_BLOCK];
  const int per = (nseg + TRAV_BLOCK - 1) / TRAV_BLOCK;
  const int beg = threadIdx.x * per, end = min(beg + per, nseg);
  int sum = 0, size;
  for (int q = beg; q < end; q++) {
    trav_segment_start(g, off, strip, q, size);
    sum += size;
  }
  s_part[threadIdx.x] = sum;
  __syncthreads();
  for (int o = 1; o < TRAV_BLOCK; o <<= 1) {
    const int v = threadIdx.x >= (unsigned)o ? s_part[threadIdx.x - o] : 0;
    __syncthreads();
    s_part[threadIdx.x] += v;
    __syncthreads();
  }
  int run = s_part[threadIdx.x] - sum;
  for (int q = beg; q < end; q++) {
    trav_segment_start(g, off, strip, q, size);
    seg_pos[q] = run;
    run += size;
  }
}

__global__ void __launch_bounds__(BSP)
    k_trav_scatter(GridInfo g, const int *__restrict__ off, const int *__restrict__ key_sorted,
                   const int *__restrict__ seg_pos, int strip, const Counters *cnt,
                   int *__restrict__ trav) {
  const unsigned p = blockIdx.x * BSP + threadIdx.x;
  if (p >= cnt->N) return;
  const int col = key_sorted[p] / g.nz;  // cell index of a particle in a cell
  const int gi = col / g.ny, s = (col - gi * g.ny) / strip;
  const int q = s * g.nx + gi;
  int size;
  const int a = trav_segment_start(g, off, strip, q, size);
  trav[seg_pos[q] + ((int)p - a)] = (int)p;
}

// ---------------------------------------------------------------------------------------------
// A 16-byte piece of a record (the unit of the cooperative gathers through LDS below).
typedef unsigned piece16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void glb_void;

// A record array for the gathers: 16 bytes of every lane at record j, byte off + line, go to LDS.  A
// buffer descriptor's stride is the record size, so the load unit forms index x stride + offset; an
// index beyond n_rec reads zeros instead of faulting.  It forms them in 32 bits: an array of more than
// 4 GiB (22.4M FP64 records, 38.3M FP32) is read by 64-bit addresses (FAR), two vector instructions a
// load more, which at that size costs nothing (23.4M particles of 92 neighbours FP64 23.6 ms, 39.3M FP32
// 42.8, with 32-bit offsets and wrong records 23.6 and 43.0).
template <class Rec, bool FAR>
struct RecordArray {
  __amdgpu_buffer_rsrc_t rsrc;
  // word 3: the untyped 32-bit data format the load-to-LDS path needs on gfx9-family parts
  __device__ __forceinline__ RecordArray(const Rec *rec, unsigned n_rec)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc((void *)rec, (short)sizeof(Rec), (int)n_rec, 0x00020000)) {}
  __device__ __forceinline__ void load(int j, int off, int line, char *lds) const {
    __builtin_amdgcn_struct_ptr_buffer_load_lds(rsrc, (lds_void *)lds, 16, j, off, line, 0, 0);
  }
};
template <class Rec>
struct RecordArray<Rec, true> {
  const char *rec;
  __device__ __forceinline__ RecordArray(const Rec *r, unsigned) : rec((const char *)r) {}
  __device__ __forceinline__ void load(int j, int off, int line, char *lds) const {
    __builtin_amdgcn_global_load_lds((glb_void *)(rec + (uint64_t)(unsigned)j * sizeof(Rec) + off + line),
                                     (lds_void *)lds, 16, 0, 0);
  }
};

__device__ __forceinline__ void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Four lanes (a quad) per particle: lane s of the quad takes neighbours s, s + 4, ... of the list
// and the quad adds up its four partial sums at the end (lanes_sum).  A wavefront holds 16 particles,
// so 8,000 particles fill 500 wavefronts instead of 125, the longest list of a wavefront is that of
// 16 particles, not 64, and the four neighbours a quad holds at a time are mostly consecutive
// records.  Small sets take 16 lanes (lanes64).

// The gather.  Each lane of a quad needs one record per step; the quad loads its four records
// together, straight into LDS (buffer_load_dwordx4 ... lds writes lane l's 16 bytes at 16 l of the
// load's 1 KB block).  Load (r, line) of a step fetches 64-byte line `line` of the record of lane r
// of every quad, one 64-byte line per quad: one L1 access each, where a lane loading its own record
// makes one per 16-byte piece.  The index of lane r reaches the quad by a quad permutation.  Lane e of
// the quad fetches piece (e + r) mod 4
// of the line, so piece p of lane s's record lies in slot (p - s) mod 4 of its quad's 64 bytes in
// block (s, line): the four lanes of a quad read four different slots, and the 16-byte reads of any
// two (or four) quads fall on distinct banks.
template <class Rec, bool FAR, int LINES = sizeof(Rec) / 64>
struct QuadGather {
  static constexpr int P = 4 * LINES;  // LINES: lines of a record fetched, from its first
  static constexpr int AREA = 4 * LINES * 1024;
  static_assert(sizeof(Rec) % 64 == 0 && (int)sizeof(Rec) >= 64 * LINES, "whole 64-byte lines");
  struct Pieces {
    piece16 p[P];
  };
  RecordArray<Rec, FAR> array;
  char *area;
  int off[4];  // byte offset within a line of the piece this lane fetches, per record r
  int rd[4];   // LDS offset of piece p of line 0 of this lane's record
  __device__ __forceinline__ QuadGather(const Rec *rec, unsigned n_rec, char *lds, int lane)
      : array(rec, n_rec), area(lds) {
    const int s = lane & 3;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      off[r] = 16 * ((s + r) & 3);
      rd[r] = s * LINES * 1024 + 64 * (lane >> 2) + 16 * ((r - s) & 3);
    }
  }
  // fetches record j of every lane (all lanes active)
  __device__ __forceinline__ void issue(int j) const {
    const int jr[4] = {__builtin_amdgcn_mov_dpp(j, 0x00, 0xf, 0xf, true),
                       __builtin_amdgcn_mov_dpp(j, 0x55, 0xf, 0xf, true),
                       __builtin_amdgcn_mov_dpp(j, 0xaa, 0xf, 0xf, true),
                       __builtin_amdgcn_mov_dpp(j, 0xff, 0xf, 0xf, true)};
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int l = 0; l < LINES; l++) array.load(jr[r], off[r], 64 * l, area + (r * LINES + l) * 1024);
  }
  // this lane's record, once the loads have arrived
  __device__ __forceinline__ Pieces read() const {
    Pieces pc;
#pragma unroll
    for (int p = 0; p < P; p++) pc.p[p] = *(const piece16 *)(area + rd[p & 3] + (p >> 2) * 1024);
    return pc;
  }
};

// What a lane needs to begin its walk.  Of a particle past N or blanked it is loaded like any other (the
// arrays hold n_init) and not used, so that the loads go out together; N, the flags, the list's length
// and its first entry waited for one another: 512 particles 11.7 -> 10.3 us, 8,000 22.6 -> 21.9, 1M FP32
// 1.25 -> 1.23 ms, 24 batched wedges 1.26 -> 1.22 ms.  An entry is read inside its row, however short.
template <int F>
struct PairHead {
  unsigned i;   // the particle, below n_init
  uint32_t fl;  // its flags, FL_BLANKED past N
  bool act;
  int nl;
  int j[F];  // neighbours q0, q0 + dq, ... of the list; past its end the particle itself
  __device__ __forceinline__ PairHead(unsigned t, unsigned n_init, const State &st, const Counters *cnt,
                                      const int *__restrict__ trav, const int *__restrict__ nbr, int stride,
                                      const int *__restrict__ count, int q0, int dq) {
    const unsigned N = cnt->N;
    i = min(t, n_init - 1);
    if (trav) i = min((unsigned)trav[i], n_init - 1);  // trav holds no particles past N
    uint32_t f = st.flags[i];
    int n = count[i];
    const int *row = nbr + (size_t)i * stride;
#pragma unroll
    for (int k = 0; k < F; k++) j[k] = row[min(q0 + k * dq, stride - 1)];
    // the loads stay together and ahead of what their results decide
    asm volatile("" : "+v"(f), "+v"(n));
#pragma unroll
    for (int k = 0; k < F; k++) asm volatile("" : "+v"(j[k]));
    const bool in_range = t < N && t < n_init;
    fl = in_range ? f : FL_BLANKED;
    act = in_range && !(f & FL_BLANKED);
    nl = act ? n : 0;
#pragma unroll
    for (int k = 0; k < F; k++) j[k] = q0 + k * dq < nl ? j[k] : (int)i;
  }
};

// LANES: lanes of a particle, 4 or 16 (lanes64); area: QuadGather::AREA bytes a wavefront
template <bool BROOK, int LANES, int BS, bool FAR>
__device__ __forceinline__ void pair_sums(unsigned b, unsigned nb, unsigned n_init, const State &st,
                                          const Rec64 *__restrict__ rec,
                                          const int *__restrict__ nbr, int stride,
                                          const int *__restrict__ count, const Consts &c,
                                          const Counters *cnt, double *__restrict__ sums,
                                          size_t sstride, const int *__restrict__ trav, char *area) {
  typedef QuadGather<Rec64, FAR> Gather;
  const unsigned t = xcd_map(b, nb) * (BS / LANES) + threadIdx.x / LANES;
  // the wave index as a scalar: the scalar unit forms the LDS destinations of the loads
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = lane & (LANES - 1);
  const PairHead<1> hd(t, n_init, st, cnt, trav, nbr, stride, count, s, LANES);
  const unsigned i = hd.i, ic = hd.i;
  const uint32_t fl = hd.fl;
  const bool act = hd.act;
  const int nl = hd.nl, j0 = hd.j[0];
  int steps = (nl + LANES - 1) / LANES;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) steps = max(steps, __shfl_xor(steps, o, 64));
  steps = __builtin_amdgcn_readfirstlane(steps);
  const int *row = nbr + (size_t)ic * stride + s;
  // neighbour s + LANES k of the list; past its end the particle itself, which is loaded and not used
  auto index = [&](int k) -> int { return s + LANES * k < nl ? row[LANES * k] : (int)ic; };
  const Pair64<BROOK> P(c, rec[ic]);
  const bool tool_i = (fl & FL_TOOL) != 0, tool_nz = (fl & FL_TOOL_NZ) != 0;
  const bool brook = BROOK && c.heat == MFG_HEAT_BROOKSHAW && (tool_nz ? c.alpha_tool : c.alpha_wp) != 0.;
  PairAcc acc = {};
  const Gather g(rec, n_init, area + w * Gather::AREA, lane);
  if (steps > 0) {
    g.issue(j0);
    int jn = steps > 1 ? index(1) : 0;
    for (int k = 0; k < steps; k++) {
      __builtin_amdgcn_s_waitcnt(0);  // this step's records are in LDS
      const Rec64 rj = __builtin_bit_cast(Rec64, g.read());
      __builtin_amdgcn_s_waitcnt(0);  // every lane's reads are done before the area is refilled
      wave_sync_lds();
      if (k + 1 < steps) {
        g.issue(jn);
        if (k + 2 < steps) jn = index(k + 2);
      }
      if (s + LANES * k < nl) P.term(acc, rj, !tool_i);
    }
  }
  if (!act) return;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    acc.W[k] = lanes_sum<LANES>(acc.W[k]);
    acc.F[k] = lanes_sum<LANES>(acc.F[k]);
    acc.V[k] = lanes_sum<LANES>(acc.V[k]);
    acc.X[k] = lanes_sum<LANES>(acc.X[k]);
#pragma unroll
    for (int e = 0; e < 3; e++) acc.D[e][k] = lanes_sum<LANES>(acc.D[e][k]);
#pragma unroll
    for (int e = 0; e < 6; e++) acc.M[e][k] = lanes_sum<LANES>(acc.M[e][k]);
  }
#pragma unroll
  for (int e = 0; e < 6; e++) {
    acc.B[e] = lanes_sum<LANES>(acc.B[e]);
    if (BROOK) acc.Q[e] = lanes_sum<LANES>(acc.Q[e]);
  }
  if (s != 0) return;
  double A[6], R[6];
#pragma unroll
  for (int e = 0; e < 6; e++) {
    A[e] = rec[i].A[e];
    R[e] = rec[i].R[e];
  }
  // without neighbours the sums are zero, whatever the kernel's scale (infinite for h = 0)
  PairScale scale = P.scale(c);
  if (nl == 0) scale.k1 = scale.fac = 0.;
  PairSums ps;
  finish_sums<BROOK>(c, acc, scale, A, R, tool_nz, brook, ps);
  store_sums(sums, sstride, i, ps);
}
// BS: threads per workgroup (64, 128 or 256; each wavefront works alone, so the sums do not
// depend on it)
template <bool BROOK, int LANES, int BS, bool FAR>
__global__ void __launch_bounds__(BS, PAIR_WAVES)
    k_pair_sums(unsigned n_init, State st, const Rec64 *__restrict__ rec,
                const int *__restrict__ nbr, int stride, const int *__restrict__ count, Consts c,
                const Counters *cnt, double *__restrict__ sums, size_t sstride,
                const int *__restrict__ trav) {
  __shared__ __align__(16) char s_area[(BS / 64) * QuadGather<Rec64, FAR>::AREA];
  pair_sums<BROOK, LANES, BS, FAR>(blockIdx.x, gridDim.x, n_init, st, rec, nbr, stride, count, c, cnt, sums,
                              sstride, trav, s_area);
}

// ---------------------------------------------------------------------------------------------
// The FP64 sums in the reference's own order of evaluation: one lane per particle, one neighbour
// after the other, B first, every product and division rounded as the reference writes it
// (src/interactions_gpu.cu:152-471).  An unlocked grid takes its origin and cell size from the
// particles, to the last bit of the outermost position, so there the positions of every step must
// round as the reference's do for its cell tables to be the reference's; the sums above differ from
// these in the last bits.  On a locked grid nothing depends on those bits.  B is summed from the records'
// first 64-byte lines: from 32-byte entries of its own the pass took 3 % less (1M 1.98 against 1.92 ms, a step
// 3.19 ms against 3.65 with the neighbour pass and the sort of that time).
struct PairOrdered64 {
  Rec64 ri;
  bool tool_i, tool_nz, brook;
  double thermal_alpha, hi, h1, fac, Ti;
  M3 B, invB;
  PairSums ps;

  __device__ __forceinline__ PairOrdered64(const Consts &c, const Rec64 &r, uint32_t fl) : ri(r) {
    tool_i = ri.tool == 1.;
    tool_nz = (fl & FL_TOOL_NZ) != 0;
    thermal_alpha = tool_nz ? c.alpha_tool : c.alpha_wp;
    brook = c.heat == MFG_HEAT_BROOKSHAW && thermal_alpha != 0.;
    hi = ri.h;
    h1 = 1 / hi;
    fac = (INV_PI_D)*h1 * h1 * h1;
    Ti = brook ? ri.T : 0.;
#pragma unroll
    for (int a = 0; a < 3; a++) {
#pragma unroll
      for (int b = 0; b < 3; b++) {
        invB.m[a][b] = (a == b) ? 1. : 0.;
        B.m[a][b] = 0.;
        ps.vd.m[a][b] = 0.;
        ps.sd.m[a][b] = 0.;
      }
      ps.vt[a] = 0.;
      ps.xt[a] = 0.;
    }
    ps.Tl = 0.;
  }
  // tool particles (tool != 0) keep the identity correction
  __device__ __forceinline__ bool cspm_sum() const { return !tool_nz; }
  __device__ __forceinline__ void cspm_add(const Consts &c, double xj, double yj, double zj,
                                           double volj) {
    double xij = ri.x - xj, yij = ri.y - yj, zij = ri.z - zj;
    double rr2 = xij * xij + yij * yij + zij * zij;
    double w, wx, wy, wz;
    cubic_spline64(xij, yij, zij, rr2, h1, fac, c.single_sqrt, w, wx, wy, wz);
    B.m[0][0] -= volj * xij * wx; B.m[1][0] -= volj * xij * wy; B.m[2][0] -= volj * xij * wz;
    B.m[0][1] -= volj * yij * wx; B.m[1][1] -= volj * yij * wy; B.m[2][1] -= volj * yij * wz;
    B.m[0][2] -= volj * zij * wx; B.m[1][2] -= volj * zij * wy; B.m[2][2] -= volj * zij * wz;
  }
  __device__ __forceinline__ void cspm_end() {
    if (det3(B) > 1e-8) inv3(B, invB);
  }
  __device__ __forceinline__ void term(const Consts &c, const Rec64 &rj) {
    const double mass = c.i_mass, wdeltap = c.wdeltap, eps = c.xspheps;
    double xij = ri.x - rj.x, yij = ri.y - rj.y, zij = ri.z - rj.z;
    double rr2 = xij * xij + yij * yij + zij * zij;
    double w, wx0, wy0, wz0;
    cubic_spline64(xij, yij, zij, rr2, h1, fac, c.single_sqrt, w, wx0, wy0, wz0);
    double w_x, w_y, w_z;
    if (!c.cspm) {
      w_x = wx0; w_y = wy0; w_z = wz0;
    } else {
      w_x = (wx0 * invB.m[0][0] + wy0 * invB.m[1][0] + wz0 * invB.m[2][0]);
      w_y = (wx0 * invB.m[0][1] + wy0 * invB.m[1][1] + wz0 * invB.m[2][1]);
      w_z = (wx0 * invB.m[0][2] + wy0 * invB.m[1][2] + wz0 * invB.m[2][2]);
    }
    if (!tool_i && !(rj.tool == 1.)) {
      const double volj = rj.vol;
      double dvx = rj.vx - ri.vx, dvy = rj.vy - ri.vy, dvz = rj.vz - ri.vz;
      ps.vd.m[0][0] += dvx * w_x * volj; ps.vd.m[0][1] += dvx * w_y * volj; ps.vd.m[0][2] += dvx * w_z * volj;
      ps.vd.m[1][0] += dvy * w_x * volj; ps.vd.m[1][1] += dvy * w_y * volj; ps.vd.m[1][2] += dvy * w_z * volj;
      ps.vd.m[2][0] += dvz * w_x * volj; ps.vd.m[2][1] += dvz * w_y * volj; ps.vd.m[2][2] += dvz * w_z * volj;
      double Rxx = 0., Ryy = 0., Rzz = 0., Rxy = 0., Rxz = 0., Ryz = 0.;
      if (wdeltap > 0) {
        double fab = w / wdeltap;
        fab *= fab;
        fab *= fab;
        Rxx = fab * (ri.R[0] + rj.R[0]);
        Rxy = fab * (ri.R[3] + rj.R[3]);
        Ryy = fab * (ri.R[1] + rj.R[1]);
        Rxz = fab * (ri.R[5] + rj.R[5]);
        Ryz = fab * (ri.R[4] + rj.R[4]);
        Rzz = fab * (ri.R[2] + rj.R[2]);
      }
      ps.sd.m[0][0] += mass * (ri.A[0] + rj.A[0] + Rxx) * w_x;
      ps.sd.m[0][1] += mass * (ri.A[3] + rj.A[3] + Rxy) * w_y;
      ps.sd.m[0][2] += mass * (ri.A[5] + rj.A[5] + Rxz) * w_z;
      ps.sd.m[1][0] += mass * (ri.A[3] + rj.A[3] + Rxy) * w_x;
      ps.sd.m[1][1] += mass * (ri.A[1] + rj.A[1] + Ryy) * w_y;
      ps.sd.m[1][2] += mass * (ri.A[4] + rj.A[4] + Ryz) * w_z;
      ps.sd.m[2][0] += mass * (ri.A[5] + rj.A[5] + Rxz) * w_x;
      ps.sd.m[2][1] += mass * (ri.A[4] + rj.A[4] + Ryz) * w_y;
      ps.sd.m[2][2] += mass * (ri.A[2] + rj.A[2] + Rzz) * w_z;
      double vijx = ri.vx - rj.vx, vijy = ri.vy - rj.vy, vijz = ri.vz - rj.vz;
      double vijposij = vijx * xij + vijy * yij + vijz * zij;
      double rhoij = 0.5 * (ri.rho + rj.rho);
      if (vijposij < 0.) {
        double cij = 0.5 * (ri.c + rj.c);
        double hij = 0.5 * (hi + rj.h);
        double r2ij = xij * xij + yij * yij + zij * zij;
        double muij = (hij * vijposij) / (r2ij + c.v_eta * c.v_eta * hij * hij);
        double piij = (-c.v_alpha * cij * muij + c.v_beta * muij * muij) / rhoij;
        ps.vt[0] += -mass * piij * w_x;
        ps.vt[1] += -mass * piij * w_y;
        ps.vt[2] += -mass * piij * w_z;
      }
      ps.xt[0] += -eps * w * mass / rhoij * vijx;
      ps.xt[1] += -eps * w * mass / rhoij * vijy;
      ps.xt[2] += -eps * w * mass / rhoij * vijz;
    }
    if (brook) {
      double rij = sqrt_rn(xij * xij + yij * yij + zij * zij);
      if (rij > 1e-8) {
        double ex = xij / rij, ey = yij / rij, ez = zij / rij;
        double rij1 = 1. / rij;
        ps.Tl += 2.0 * (rj.vol) * (Ti - rj.T) * rij1 * (ex * w_x + ey * w_y + ez * w_z);
      }
    }
  }
};

// walks the list of a lane with record gathers of LINES lines; step(k, pieces) for k < nl
template <bool FAR, int LINES, class Step>
__device__ __forceinline__ void ordered_walk(const QuadGather<Rec64, FAR, LINES> &g, const int *row, int nl,
                                             int nmax, int ic, Step &&step) {
  typedef int iv4 __attribute__((ext_vector_type(4)));
  if (nmax <= 0) return;
  // indices in windows of four, one window ahead (rows hold a multiple of four entries)
  iv4 cur = {ic, ic, ic, ic}, nxt = cur;
  if (nl > 0) cur = *(const iv4 *)row;
  if (nl > 4) nxt = *(const iv4 *)(row + 4);
  auto index = [&](int k) -> int {
    if ((k & 3) == 0 && k > 0) {
      cur = nxt;
      if (k + 4 < nl) nxt = *(const iv4 *)(row + k + 4);
    }
    const int q = k & 3;
    return k < nl ? (q == 0 ? cur.x : q == 1 ? cur.y : q == 2 ? cur.z : cur.w) : ic;
  };
  g.issue(index(0));
  for (int k = 0; k < nmax; k++) {
    __builtin_amdgcn_s_waitcnt(0);  // this step's records are in LDS
    const auto pc = g.read();
    __builtin_amdgcn_s_waitcnt(0);  // every lane's reads are done before the area is refilled
    wave_sync_lds();
    if (k + 1 < nmax) g.issue(index(k + 1));
    if (k < nl) step(pc);
  }
}

template <int BS, bool FAR>
__global__ void __launch_bounds__(BS, PAIR_WAVES)
    k_pair_ordered(unsigned n_init, State st, const Rec64 *__restrict__ rec,
                   const int *__restrict__ nbr, int stride, const int *__restrict__ count, Consts c,
                   const Counters *cnt, double *__restrict__ sums, size_t sstride,
                   const int *__restrict__ trav) {
  typedef QuadGather<Rec64, FAR> Gather;
  __shared__ __align__(16) char s_area[BS / 64][Gather::AREA];
  const unsigned t = xcd_map(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  const bool in_range = t < cnt->N && t < n_init;
  const unsigned i = in_range && trav ? (unsigned)trav[t] : t;
  const uint32_t fl = in_range ? st.flags[i] : FL_BLANKED;
  const bool act = in_range && !(fl & FL_BLANKED);
  const unsigned ic = act ? i : 0u;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  PairOrdered64 P(c, rec[ic], fl);
  const int nl = act ? count[i] : 0;
  const int *row = nbr + (size_t)ic * stride;
  int nmax = nl;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) nmax = max(nmax, __shfl_xor(nmax, o, 64));
  nmax = __builtin_amdgcn_readfirstlane(nmax);
  if (c.cspm) {
    // x, y, z, h, T, vol, c, tool: the record's first line
    ordered_walk(QuadGather<Rec64, FAR, 1>(rec, n_init, s_area[w], lane), row, P.cspm_sum() ? nl : 0,
                 nmax, (int)ic, [&](const auto &pc) {
                   struct Line {
                     double x, y, z, h, T, vol, c, tool;
                   };
                   const Line j = __builtin_bit_cast(Line, pc);
                   if (j.tool != 1.) P.cspm_add(c, j.x, j.y, j.z, j.vol);
                 });
    P.cspm_end();
  }
  ordered_walk(Gather(rec, n_init, s_area[w], lane), row, nl, nmax, (int)ic,
               [&](const auto &pc) { P.term(c, __builtin_bit_cast(Rec64, pc)); });
  if (act) store_sums(sums, sstride, i, P.ps);
}

// ---------------------------------------------------------------------------------------------
// FP32 pair pass.  Every sum runs over the list in its order (the Kahan sums depend on it), first
// the nine of B, then the 24 with the corrected gradient; so a sum is one lane's, and a lane per
// particle would keep 25 of them.  Here a particle has L lanes (four or, in small sets, eight: pair_lanes),
// one in each of the L groups of consecutive lanes of its wavefront: in step k the lane of group n forms
// all terms of neighbour L k + n, the groups exchange them (spread: for four, four registers in four
// instructions), and every lane then adds the L neighbours' terms of its own share of the sums, in list
// order.
//
// Against one lane per particle, the same sums to the bit: 19,000 particles 137 -> 50 us (300 wavefronts
// of 100 steps, now 2,400 of 13; with four lanes 59), 255k with wide sums 396 -> 324 us, 1M 1.35 -> 1.23 ms.  At 1M the
// vector units are full: 424 instructions per 64 pairs, the exchanges and the transcendentals counting
// double and fourfold; one lane per particle needs 345 but runs at the pace of its list reads (each
// lane walks its own row: 1.42 ms).  115 registers: four waves per SIMD (three: 1.25 ms; five spill).
// The index of a lane's next neighbour is one 4-byte read two steps ahead: reading them by fours and
// exchanging them waits longer (1.86 ms).
// (FAR: three, its addresses take the registers that would otherwise spill.)
constexpr int pair32_waves(bool far) { return far ? 3 : 4; }

// L groups of 64 / L lanes (rows of 16 for four, half rows for eight): on return v[n] in group r holds
// what v[r] held in group n
template <int L>
__device__ __forceinline__ void spread(float (&v)[L]) {
  unsigned u[L];
#pragma unroll
  for (int r = 0; r < L; r++) u[r] = __builtin_bit_cast(unsigned, v[r]);
  // exchange bit by bit of the group number: halves of the wavefront, rows, half rows
#pragma unroll
  for (int r = 0; r < L / 2; r++) {
    const auto x = __builtin_amdgcn_permlane32_swap(u[r], u[r + L / 2], false, false);
    u[r] = x[0];
    u[r + L / 2] = x[1];
  }
#pragma unroll
  for (int b = 0; b < L; b += L / 2)
#pragma unroll
    for (int r = b; r < b + L / 4; r++) {
      const auto x = __builtin_amdgcn_permlane16_swap(u[r], u[r + L / 4], false, false);
      u[r] = x[0];
      u[r + L / 4] = x[1];
    }
  if constexpr (L == 8) {
#pragma unroll
    for (int r = 0; r < L; r += 2) {
      const int a = (int)u[r], b = (int)u[r + 1];  // row_ror:8 into the upper, the lower half of a row
      u[r] = (unsigned)__builtin_amdgcn_update_dpp(a, b, 0x128, 0xf, 0xc, false);
      u[r + 1] = (unsigned)__builtin_amdgcn_update_dpp(b, a, 0x128, 0xf, 0x3, false);
    }
  }
#pragma unroll
  for (int r = 0; r < L; r++) v[r] = __builtin_bit_cast(float, u[r]);
}
// v[n] = x of group n, in every group
template <int L>
__device__ __forceinline__ void rows_of(float x, float (&v)[L]) {
#pragma unroll
  for (int n = 0; n < L; n++) v[n] = x;
  spread(v);
}
template <int L>
__device__ __forceinline__ void rows_of(double x, double (&v)[L]) {
  const uint64_t w = __builtin_bit_cast(uint64_t, x);
  const unsigned w0 = (unsigned)w, w1 = (unsigned)(w >> 32);
  float lo[L], hi[L];
  rows_of(__builtin_bit_cast(float, w0), lo);
  rows_of(__builtin_bit_cast(float, w1), hi);
#pragma unroll
  for (int n = 0; n < L; n++)
    v[n] = __builtin_bit_cast(double, ((uint64_t)__builtin_bit_cast(unsigned, hi[n]) << 32) |
                                          __builtin_bit_cast(unsigned, lo[n]));
}
// the lanes of the particles for which group n's bit of m is set
template <int L>
__device__ __forceinline__ uint64_t row_mask(uint64_t m, int n) {
  if constexpr (L == 8) return ((m >> (8 * n)) & 0xff) * 0x0101010101010101ull;
  const uint64_t r = (m >> (16 * n)) & 0xffff;
  const uint64_t h = r | (r << 16);
  return h | (h << 32);
}
// adds neighbours 0 .. L - 1 to M sums; m: the lanes whose own neighbour counts.  With all of them in,
// no masks (a masked sum costs a fifth operation)
template <int M, int L, class Acc>
__device__ __forceinline__ void add_rows(Acc (&a)[M], const float (&v)[M][L], uint64_t m) {
  if (m == ~0ull) {
#pragma unroll
    for (int n = 0; n < L; n++)
#pragma unroll
      for (int q = 0; q < M; q++) a[q].add(v[q][n]);
  } else {
#pragma unroll
    for (int n = 0; n < L; n++)
      if (__builtin_amdgcn_inverse_ballot_w64(row_mask<L>(m, n))) {
#pragma unroll
        for (int q = 0; q < M; q++) a[q].add(v[q][n]);
      }
  }
}

// The records of a step: 64 in LDS one after the other (record of lane L at 112 L), as seven 1 KB
// blocks: load q fetches piece g = 64 q + lane of that image (record g / 7, piece g mod 7), so every
// lane loads and no piece is fetched twice.  At the 112-byte stride the 16-byte reads of a lane's own
// record fall on distinct banks for the lanes one read phase serves.
template <bool FAR>
struct RecGather {
  static constexpr int P = 7, AREA = P * 1024;
  static_assert(sizeof(Rec32) == 16 * P, "FP32 record image");
  struct Pieces {
    piece16 p[P];
  };
  RecordArray<Rec32, FAR> array;
  char *area;
  int src[P], off[P], lane;
  __device__ __forceinline__ RecGather(const Rec32 *rec, unsigned n_rec, char *lds, int l)
      : array(rec, n_rec), area(lds), lane(l) {
#pragma unroll
    for (int q = 0; q < P; q++) {
      const int g = 64 * q + lane, r = g / P;
      src[q] = 4 * r;
      off[q] = 16 * (g - P * r);
    }
  }
  __device__ __forceinline__ void issue(int j) const {
    int jm[P];
#pragma unroll
    for (int q = 0; q < P; q++) jm[q] = __builtin_amdgcn_ds_bpermute(src[q], j);
#pragma unroll
    for (int q = 0; q < P; q++) array.load(jm[q], off[q], 0, area + 1024 * q);
  }
  __device__ __forceinline__ Rec32 read() const {
    Pieces pc;
#pragma unroll
    for (int p = 0; p < P; p++) pc.p[p] = *(const piece16 *)(area + (int)sizeof(Rec32) * lane + 16 * p);
    return __builtin_bit_cast(Rec32, pc);
  }
};
// The CSPM entries of a step likewise, 32 bytes a lane in two loads (load q: piece g = 64 q + lane of
// the 2 KB image, entry g / 2).  The two pieces of an entry swap slots every eight entries, so that the
// 16-byte reads of 16 consecutive lanes fall on distinct bank groups.  The terms are light, so the
// walk holds CSPM_BLOCK steps in LDS while the next CSPM_BLOCK load.
constexpr int CSPM_BLOCK = 2, CSPM_STEP = 64 * 32, CSPM_AREA = 2 * CSPM_BLOCK * CSPM_STEP;
template <bool FAR>
struct EntryGather {
  struct Pieces {
    piece16 p[2];
  };
  RecordArray<double4, FAR> array;
  int src[2], off[2], rd[2];
  __device__ __forceinline__ EntryGather(const double4 *cs4, unsigned n_rec, int lane) : array(cs4, n_rec) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const int g = 64 * q + lane, r = g >> 1;
      src[q] = 4 * r;
      off[q] = 16 * (((g & 1) + (r >> 3)) & 1);
      rd[q] = 32 * lane + 16 * (((lane >> 3) + q) & 1);
    }
  }
  __device__ __forceinline__ void issue(int j, char *area) const {
#pragma unroll
    for (int q = 0; q < 2; q++)
      array.load(__builtin_amdgcn_ds_bpermute(src[q], j), off[q], 0, area + 1024 * q);
  }
  __device__ __forceinline__ double4 read(const char *area) const {
    Pieces pc;
#pragma unroll
    for (int q = 0; q < 2; q++) pc.p[q] = *(const piece16 *)(area + rd[q]);
    return __builtin_bit_cast(double4, pc);
  }
};

template <class Acc, bool BROOK, int L, int BS, bool FAR>
__device__ __forceinline__ void pair_rows(unsigned b, unsigned nb, unsigned n_init, const State &st,
                                          const Rec32 *__restrict__ rec, const int *__restrict__ nbr,
                                          int stride, const int *__restrict__ count, const Consts &c,
                                          const Counters *cnt, double *__restrict__ sums,
                                          size_t sstride, const int *__restrict__ trav,
                                          const double4 *__restrict__ cs4) {
  constexpr int AREA = CSPM_AREA > RecGather<FAR>::AREA ? CSPM_AREA : RecGather<FAR>::AREA;
  __shared__ __align__(16) char s_area[BS / 64][AREA];
  // the wave index as a scalar: the scalar unit forms the LDS destinations of the loads
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int PER = 64 / L;  // particles of a wavefront
  constexpr int NB = 8 / L, NA = 20 / L;  // sums of a lane: B, and those without the viscous ones
  const int n = lane / PER;
  const unsigned t = xcd_map(b, nb) * (BS / L) + PER * w + lane % PER;
  const PairHead<2> hd(t, n_init, st, cnt, trav, nbr, stride, count, n, L);
  const unsigned i = hd.i, ic = hd.i;
  const uint32_t fl = hd.fl;
  const bool act = hd.act;
  const int nl = hd.nl, j0 = hd.j[0], j1 = hd.j[1];
  int steps = (nl + L - 1) / L;
#pragma unroll
  for (int o = PER / 2; o > 0; o >>= 1) steps = max(steps, __shfl_xor(steps, o, 64));
  steps = __builtin_amdgcn_readfirstlane(steps);
  const int *row = nbr + (size_t)ic * stride + n;
  // neighbour L k + n of the list; past its end the particle itself, which is loaded and not used
  auto index = [&](int k) -> int { return n + L * k < nl ? row[L * k] : (int)ic; };
  Pair32<BROOK> P(c, rec[ic]);
  const bool tool_i = P.ri.tool == 1.f, tool_nz = (fl & FL_TOOL_NZ) != 0;
  char *area = s_area[w];
  if (c.cspm && steps > 0) {
    const EntryGather<FAR> g(cs4, n_init, lane);
    // No numerical reason (either order errs alike): the one-lane kernel's unrolled walk rounded the terms so for
    // all but every fourth neighbour, and results are to keep their bits (tests/golden/wide_pair_sums.npz)
    const bool x_first = std::is_same<Acc, AccWide>::value && (n & 3) != 0;
    Acc a2[NB], a1[1];  // B[L q + n] and, in every group, B[8]
#pragma unroll
    for (int q = 0; q < NB; q++) a2[q].zero();
    a1[0].zero();
    const int nb = (steps + CSPM_BLOCK - 1) / CSPM_BLOCK;
    int jn[CSPM_BLOCK];
#pragma unroll
    for (int s = 0; s < CSPM_BLOCK; s++)
      g.issue(s == 0 ? j0 : s == 1 ? j1 : index(s), area + s * CSPM_STEP);
#pragma unroll
    for (int s = 0; s < CSPM_BLOCK; s++) jn[s] = index(CSPM_BLOCK + s);
    for (int b = 0; b < nb; b++) {
      __builtin_amdgcn_s_waitcnt(0);  // this block's entries have arrived, and the next indices
      wave_sync_lds();
      const char *here = area + (b & 1) * CSPM_BLOCK * CSPM_STEP;
      if (b + 1 < nb) {  // into the half that block b - 1 used, read before
        char *next = area + ((b + 1) & 1) * CSPM_BLOCK * CSPM_STEP;
#pragma unroll
        for (int s = 0; s < CSPM_BLOCK; s++) g.issue(jn[s], next + s * CSPM_STEP);
#pragma unroll
        for (int s = 0; s < CSPM_BLOCK; s++) jn[s] = index((b + 2) * CSPM_BLOCK + s);
      }
#pragma unroll
      for (int s = 0; s < CSPM_BLOCK; s++) {
        const double4 e = g.read(here + s * CSPM_STEP);
        const ToolVol tv = __builtin_bit_cast(ToolVol, e.w);
        float B[9], v2[NB][L], v1[1][L];
        P.cspm_term(e, tv.vol, x_first, B);
        const uint64_t m = 
            __builtin_amdgcn_ballot_w64(n + L * (b * CSPM_BLOCK + s) < nl && !tool_nz && tv.tool != 1.f);
#pragma unroll
        for (int q = 0; q < NB; q++) {
#pragma unroll
          for (int r = 0; r < L; r++) v2[q][r] = B[L * q + r];
          spread(v2[q]);
        }
        rows_of(B[8], v1[0]);
        add_rows(a2, v2, m);
        add_rows(a1, v1, m);
      }
    }
    wave_sync_lds();  // the area is free for the next walk
    double B[9], of[L];
#pragma unroll
    for (int q = 0; q < NB; q++) {
      rows_of(a2[q].val(), of);
#pragma unroll
      for (int r = 0; r < L; r++) B[L * q + r] = of[r];
    }
    B[8] = a1[0].val();
    P.invert(B);
  }
  // slots L q + n of the 24 (Pair32::term): the first NA, and the last, with the viscous sums; heat
  Acc am[NA], av[1], ah[1];
#pragma unroll
  for (int q = 0; q < NA; q++) am[q].zero();
  av[0].zero();
  ah[0].zero();
  const RecGather<FAR> g(rec, n_init, area, lane);
  const bool brook = BROOK && (tool_nz ? c.alpha_tool : c.alpha_wp) != 0.;
  if (steps > 0) {
    g.issue(j0);
    int jn = j1;
    for (int k = 0; k < steps; k++) {
      __builtin_amdgcn_s_waitcnt(0);  // this step's records are in LDS
      const Rec32 rj = g.read();
      __builtin_amdgcn_s_waitcnt(0);  // every lane's reads are done before the area is refilled
      wave_sync_lds();
      if (k + 1 < steps) {
        g.issue(jn);
        jn = index(k + 2);
      }
      float v[24], vm[NA][L], vv[L], heat = 0.f;
      bool approach, hot = false;
      P.term(rj, v, approach, heat, hot);
      const bool in_list = n + L * k < nl, mech = in_list && !tool_i && !(rj.tool == 1.f);
      const uint64_t m = __builtin_amdgcn_ballot_w64(mech), mv = __builtin_amdgcn_ballot_w64(mech && approach);
#pragma unroll
      for (int q = 0; q < NA; q++) {
#pragma unroll
        for (int r = 0; r < L; r++) vm[q][r] = v[L * q + r];
        spread(vm[q]);
      }
#pragma unroll
      for (int r = 0; r < L; r++) vv[r] = v[24 - L + r];
      spread(vv);
      add_rows(am, vm, m);
      // the last slots: 20 .. 22 the viscous sums, 23 (and for eight lanes 16 .. 19) others
      constexpr uint64_t VISC = L == 8 ? 0x00ffffff00000000ull : 0x0000ffffffffffffull;
#pragma unroll
      for (int q = 0; q < L; q++) {
        const uint64_t keep = (row_mask<L>(mv, q) & VISC) | (row_mask<L>(m, q) & ~VISC);
        if (__builtin_amdgcn_inverse_ballot_w64(keep)) av[0].add(vv[q]);
      }
      if (BROOK) {
        float vh[1][L];
        rows_of(heat, vh[0]);
        add_rows(ah, vh, __builtin_amdgcn_ballot_w64(in_list && brook && hot));
      }
    }
  }
  if (!act) return;
  // slots: vd 0 .. 8, sd 0 .. 8, xt 0, xt 1, vt 0 .. 2, xt 2
  auto place = [](int s) { return s < 18 || s == 23 ? s : s < 20 ? s + 3 : s - 2; };
#pragma unroll
  for (int q = 0; q < NA; q++) sums[place(L * q + n) * sstride + i] = am[q].val();
  sums[place(24 - L + n) * sstride + i] = av[0].val();
  if (n == 0) sums[24 * sstride + i] = BROOK ? ah[0].val() : 0.;
}
// BS: threads per workgroup (64, 128 or 256; each wavefront works alone, so the sums do not
// depend on it).  Small instances spread over more compute units with smaller workgroups.
template <class Acc, bool BROOK, int L, int BS, bool FAR>
__global__ void __launch_bounds__(BS, pair32_waves(FAR))
    k_pair_rows(unsigned n_init, State st, const Rec32 *__restrict__ rec,
                const int *__restrict__ nbr, int stride, const int *__restrict__ count,
                Consts c, const Counters *cnt, double *__restrict__ sums, size_t sstride,
                const int *__restrict__ trav, const double4 *__restrict__ cs4) {
  pair_rows<Acc, BROOK, L, BS, FAR>(blockIdx.x, gridDim.x, n_init, st, rec, nbr, stride, count, c, cnt, sums,
                            sstride, trav, cs4);
}

// ---------------------------------------------------------------------------------------------
static inline unsigned nb(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// a multiple of 8 workgroups: eight equal shares of the list
unsigned neighbour_blocks(const GridInfo &g, unsigned n_init) {
  const long cells = std::min<long>(g.num_cell, n_init);
  return (unsigned)((cells + 8 * NB_WAVES - 1) / (8 * NB_WAVES) * 8);
}
bool neighbours_far(unsigned n_init) { return n_init > 1u << 27; }
static_assert((long)NB_MOST_BLOCKS * NB_BLOCK < 1L << 32, "a launch holds fewer than 2^32 threads");

void launch_neighbours(hipStream_t s, unsigned n_init, const GridInfo &g, const int *offsets,
                       const int *occ, const double4 *nl4,
                       const double2 *pse2, const double *h, const uint32_t *flags,
                       const Consts &c, int *nbr, int cap, int *count, double *T_t, Counters *cnt,
                       int want_pse, unsigned long long *stat_part, int *poison) {
  const unsigned blocks = neighbour_blocks(g, n_init);
  auto launch_as = [&](auto mode_c, auto far_c) {
    for (unsigned first = 0; first < blocks; first += NB_MOST_BLOCKS)
      hipLaunchKernelGGL((k_cell_neighbours<decltype(mode_c)::value, decltype(far_c)::value>),
                         dim3(std::min(blocks - first, NB_MOST_BLOCKS)), dim3(NB_BLOCK), 0, s, first, g, offsets, occ,
                         nl4, pse2, h, flags, c, nbr, cap, count, T_t, cnt, stat_part, poison);
  };
  auto launch = [&](auto mode_c) {
    if (neighbours_far(n_init)) launch_as(mode_c, std::true_type{});
    else launch_as(mode_c, std::false_type{});
  };
  if (!want_pse) launch(std::integral_constant<int, 0>{});
  else if (c.precision == MFG_FP64) launch(std::integral_constant<int, 1>{});
  else launch(std::integral_constant<int, 2>{});
}

// Lanes per particle.  Few particles leave SIMDs without a wavefront, and a wavefront alone on its SIMD
// waits at every step of its lists: more lanes shorten them.
// FP64: 16 below 4,096 particles (one wavefront per SIMD then; 512 particles 18.5 -> 11.7 us), else 4.
// Eight lanes would take 17 us at 8,000 particles against 22.5, but the order of the sums is part of the
// result in their last bits, and with it a single-precision rounding of the Johnson-Cook solve turns
// within 1,000 steps of the cut that four lanes follow the oracle through to 1e-10.
__host__ __device__ static inline int lanes64(unsigned n) { return n < 4096 ? 16 : 4; }
// FP32 (the same sums for either): 8 below 24k particles, else 4: 19,000 particles 50 us against 58,
// 32,000 60 against 58, 255k 362 against 322.
int pair_lanes(int precision, long particles) {
  if (precision == MFG_FP64) return lanes64((unsigned)std::min<long>(particles, 0xffffffffL));
  return particles < 24 * 1024 ? 8 : 4;
}
int pair_blocks(unsigned n_init, int lanes, int block) { return (int)nb((long)n_init * lanes, block); }
// whether the record array is beyond the gathers' 32-bit offsets (RecordArray)
bool pair_far(int precision, unsigned n_init) {
  return (uint64_t)n_init * (precision == MFG_FP64 ? sizeof(Rec64) : sizeof(Rec32)) > 1ull << 32;
}

void launch_pair(hipStream_t s, unsigned n_init, const State &st, const void *rec, const int *nbr,
                 int nl_stride, const int *count, const Consts &c, const Counters *cnt,
                 double *sums, size_t sstride, const int *trav, const double4 *cs4, int block,
                 bool ordered) {
  const int bs = block == 64 || block == 128 ? block : BSP;
  const int lanes = pair_lanes(c.precision, n_init);
  const dim3 blk(bs), grid((unsigned)pair_blocks(n_init, lanes, bs));
  const bool brook = c.heat == MFG_HEAT_BROOKSHAW, far = pair_far(c.precision, n_init);
  constexpr std::false_type NEAR{};
  constexpr std::true_type FAR{};
  auto launch = [&](auto bs_c, auto brook_c) {
    constexpr int BS = decltype(bs_c)::value;
    constexpr bool BROOK = decltype(brook_c)::value;
    auto sums64 = [&](auto lanes_c, auto far_c) {
      hipLaunchKernelGGL((k_pair_sums<BROOK, decltype(lanes_c)::value, BS, decltype(far_c)::value>), grid, blk, 0, s,
                         n_init, st, (const Rec64 *)rec, nbr, nl_stride, count, c, cnt, sums, sstride, trav);
    };
    auto ordered64 = [&](auto far_c) {  // one lane per particle
      hipLaunchKernelGGL((k_pair_ordered<BS, decltype(far_c)::value>), dim3(nb(n_init, bs)), blk, 0, s, n_init, st,
                         (const Rec64 *)rec, nbr, nl_stride, count, c, cnt, sums, sstride, trav);
    };
    auto rows = [&](auto acc) {
      auto with = [&](auto lanes_c, auto far_c) {
        hipLaunchKernelGGL((k_pair_rows<decltype(acc), BROOK, decltype(lanes_c)::value, BS, decltype(far_c)::value>),
                           grid, blk, 0, s, n_init, st, (const Rec32 *)rec, nbr, nl_stride, count, c, cnt, sums,
                           sstride, trav, cs4);
      };
      // a set beyond the 32-bit offsets is far too large for eight lanes
      if (far) with(std::integral_constant<int, 4>{}, FAR);
      else if (lanes == 4) with(std::integral_constant<int, 4>{}, NEAR);
      else with(std::integral_constant<int, 8>{}, NEAR);
    };
    if (c.precision == MFG_FP32_KAHAN) rows(AccKahan{});
    else if (c.precision == MFG_FP32_WIDE) rows(AccWide{});
    else if (ordered && far) ordered64(FAR);
    else if (ordered) ordered64(NEAR);
    else if (far) sums64(std::integral_constant<int, 4>{}, FAR);
    else if (lanes == 4) sums64(std::integral_constant<int, 4>{}, NEAR);
    else sums64(std::integral_constant<int, 16>{}, NEAR);
  };
  auto sized = [&](auto bs_c) {
    if (brook) launch(bs_c, std::true_type{});
    else launch(bs_c, std::false_type{});
  };
  if (bs == 64) sized(std::integral_constant<int, 64>{});
  else if (bs == 128) sized(std::integral_constant<int, 128>{});
  else sized(std::integral_constant<int, BSP>{});
}

// ---------------------------------------------------------------------------------------------
// batched launches (after the permutation an instance's state is buf[cur ^ 1]): neighbour lists
// (+ PSE), the pair sums in the list form and sorted visiting order, and the particle update
// ---------------------------------------------------------------------------------------------
// fewer waves per SIMD than the single-instance kernel (FP64 PSE 5, FP32 PSE 6, no PSE 7): the
// instance lookup and descriptor take the registers that would otherwise spill
template <int PSE_MODE, bool FAR>
__global__ void __launch_bounds__(NB_BLOCK)
    __attribute__((amdgpu_waves_per_eu(PSE_MODE == 1   ? NB_WAVES_FP64_PSE - 1
                                       : PSE_MODE == 2 ? NB_WAVES_OTHER - 2
                                                       : NB_WAVES_OTHER - 1)))
    kb_cell_neighbours(const Inst *in, BatchMap m, unsigned first) {
  unsigned b, nb;
  const Inst &d = in[batch_locate(m, b, nb)];
  const State &st = d.buf[d.cur ^ 1];
  cell_neighbours<PSE_MODE, FAR>(first + b, d.g, d.gb.count, d.gb.occ, d.nl4, d.pse2, st.h, st.flags, d.c, d.nbr,
                            d.nl_stride, d.count, st.T_t, d.cnt, nullptr, d.poison);
}

// the instances that have LANES lanes a particle alone: the sums depend on it in their last bits
template <bool BROOK, int LANES, bool FAR>
__global__ void __launch_bounds__(BSP, PAIR_WAVES) kb_pair_sums(const Inst *in, BatchMap m) {
  __shared__ __align__(16) char s_area[(BSP / 64) * QuadGather<Rec64, FAR>::AREA];
  unsigned b, nb;
  const Inst &d = in[batch_locate(m, b, nb)];
  if (lanes64(d.n_init) != LANES) return;
  pair_sums<BROOK, LANES, BSP, FAR>(b, nb, d.n_init, d.buf[d.cur ^ 1], (const Rec64 *)d.rec, d.nbr, d.nl_stride,
                               d.count, d.c, d.cnt, d.sums, d.sum_stride, nullptr, s_area);
}

template <class Acc, bool BROOK, int L, bool FAR>
__global__ void __launch_bounds__(BSP, pair32_waves(FAR)) kb_pair_rows(const Inst *in, BatchMap m) {
  unsigned b, nb;
  const Inst &d = in[batch_locate(m, b, nb)];
  pair_rows<Acc, BROOK, L, BSP, FAR>(b, nb, d.n_init, d.buf[d.cur ^ 1], (const Rec32 *)d.rec, d.nbr, d.nl_stride,
                                d.count, d.c, d.cnt, d.sums, d.sum_stride, nullptr, d.cs4);
}

__global__ void __launch_bounds__(BSP) kb_particle_update(const Inst *in, BatchMap m) {
  unsigned b, nb;
  const Inst &d = in[batch_locate(m, b, nb)];
  ContactSearch cs = d.cs;
  if (!d.search) cs.list_n = nullptr;
  update_body(b, d.n_init, d.buf[d.cur ^ 1], d.sums, d.sum_stride, d.poison, d.c, d.cnt, d.ts, cs);
}

// The kernels of the single-instance step in the sorted visiting order; the PSE mode as
// run_neighbours picks it.  One Brookshaw instance selects the kernel with its sum for all: the
// others' sums are the same in both.
void launch_batch_pair(hipStream_t s, const BatchLaunch &L) {
  auto neighbours_as = [&](auto mode_c, auto far_c) {
    for (unsigned first = 0; first < L.nbr_blocks; first += L.nbr_most)
      hipLaunchKernelGGL((kb_cell_neighbours<decltype(mode_c)::value, decltype(far_c)::value>), dim3(L.nbrs8.blocks),
                         dim3(NB_BLOCK), 0, s, L.inst, L.nbrs8.m, first);
  };
  auto neighbours = [&](auto mode_c) {
    if (L.nbr_far) neighbours_as(mode_c, std::true_type{});
    else neighbours_as(mode_c, std::false_type{});
  };
  if (!L.pse) neighbours(std::integral_constant<int, 0>{});
  else if (L.precision == MFG_FP64) neighbours(std::integral_constant<int, 1>{});
  else neighbours(std::integral_constant<int, 2>{});
  const dim3 gp(L.pairs8.blocks), bp(BSP);
  auto sums64 = [&](auto brook_c) {
    constexpr bool BROOK = decltype(brook_c)::value;
    if ((L.pair_lanes & 4) && L.pair_far)
      hipLaunchKernelGGL((kb_pair_sums<BROOK, 4, true>), gp, bp, 0, s, L.inst, L.pairs8.m);
    else if (L.pair_lanes & 4)
      hipLaunchKernelGGL((kb_pair_sums<BROOK, 4, false>), gp, bp, 0, s, L.inst, L.pairs8.m);
    if (L.pair_lanes & 16) hipLaunchKernelGGL((kb_pair_sums<BROOK, 16, false>), gp, bp, 0, s, L.inst, L.pairs8.m);
  };
  auto rows = [&](auto acc, auto brook_c) {
    constexpr bool BROOK = decltype(brook_c)::value;
    if (L.pair_far)
      hipLaunchKernelGGL((kb_pair_rows<decltype(acc), BROOK, 4, true>), gp, bp, 0, s, L.inst, L.pairs8.m);
    else if (L.pair_lanes == 4)
      hipLaunchKernelGGL((kb_pair_rows<decltype(acc), BROOK, 4, false>), gp, bp, 0, s, L.inst, L.pairs8.m);
    else
      hipLaunchKernelGGL((kb_pair_rows<decltype(acc), BROOK, 8, false>), gp, bp, 0, s, L.inst, L.pairs8.m);
  };
  auto launch = [&](auto brook_c) {
    constexpr bool BROOK = decltype(brook_c)::value;
    if (L.precision == MFG_FP64)
      sums64(brook_c);
    else if (L.precision == MFG_FP32_KAHAN)
      rows(AccKahan{}, brook_c);
    else
      rows(AccWide{}, brook_c);
  };
  if (L.brook) launch(std::true_type{});
  else launch(std::false_type{});
  hipLaunchKernelGGL(kb_particle_update, dim3(L.parts.blocks), dim3(BSP), 0, s, L.inst, L.parts.m);
}

int pair_order_segments(const GridInfo &g, int strip) {
  return (int)(((long)g.ny + strip - 1) / strip * g.nx);
}

void launch_pair_order(hipStream_t s, unsigned n_init, const GridInfo &g, const int *offsets,
                       const int *key_sorted, const Counters *cnt, int strip, int *seg_pos,
                       int *trav) {
  hipLaunchKernelGGL(k_trav_segments, dim3(1), dim3(TRAV_BLOCK), 0, s, g, offsets, strip,
                     pair_order_segments(g, strip), seg_pos);
  hipLaunchKernelGGL(k_trav_scatter, dim3(nb(n_init, BSP)), dim3(BSP), 0, s, g, offsets,
                     key_sorted, seg_pos, strip, cnt, trav);
}

void launch_particle_update(hipStream_t s, unsigned n_init, const State &st, const double *sums,
                            size_t sstride, const int *poison, const Consts &c,
                            const Counters *cnt, const ToolSet &ts, const ContactSearch &cs,
                            const ToolMoves &mv) {
  // one wavefront per workgroup: the few wavefronts with particles in the Johnson-Cook solve run for
  // six iterations of 1.6 us and more while the others are done, and hold back only themselves (256
  // threads: 8,000 particles 25 us, now 19; 19,000 26, 22.5; 1M 172, 156; 64,000 27, 28)
  constexpr int BS = 64;
  const unsigned blocks = nb(n_init, BS) + (mv.n > 0 ? nb(mv.end[mv.n - 1], BS) : 0);
  hipLaunchKernelGGL(k_particle_update, dim3(blocks), dim3(BS), 0, s, n_init, st, sums, sstride, poison, c,
                     cnt, ts, cs, mv);
}

}  // namespace mfg
