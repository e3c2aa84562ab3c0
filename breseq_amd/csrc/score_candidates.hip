// score_candidates.hip -- the exact FP64 scorer of candidate (column, insert slot) pairs on CDNA4
// (gfx950): allele-frequency EM, variant presence score, profile-likelihood frequency bounds,
// Fisher strand and KS quality tests (identify_mutations.cpp:1669-1910, 3009-3318; stats.cpp
// 2144-2284).
//
// One block of four wavefronts per candidate.  A candidate is a chain of EM loops (50 passes over
// its reads at most), so the kernel is bound by the latency of a pass, not by bandwidth.
//
//   * The reference forms every sum in read order, and its output is decided by comparisons and by
//     printed digits.  The EM loops run with sums in any order, over the candidate's distinct table
//     keys weighted with their reads (em_full, em_tasks): the same iterations, whose results differ from
//     the reference's by rounding, by more the more reads a sum has.  Every decision and every printed
//     digit is then checked to lie farther from its boundary than a bound on that (the guards below);
//     the candidates where one does not, about one in a hundred at 100 reads and 8 printed digits, are
//     done once more with the reference's sums, as are all of them when the screen is off.
//   * em_exact makes the reference's sums: row g of a wavefront (16 lanes) holds allele g's terms of 16
//     reads, and a chain of 16 additions whose operand is broadcast from lane k of the row
//     (v_fmac_f64 with row_newbcast, times 1.0, which rounds like an addition) adds them in order,
//     the fifth allele in a second chain beside the first; some 500 cycles per 16 reads.
//   * The frequency bounds are bisections, 20 levels each.  The midpoints a round evaluates lie on
//     one predicted path per bound: the crossing point is solved from the profile's likelihood with
//     the other alleles' proportions held (model_root), and the path holds the midpoints a sequential
//     bisection visits if every decision agrees with it.  The walk afterwards keeps every level up to
//     the first one where a decision leaves the path.  From the second round on the first levels are a
//     full tree, so a round always gains some.
//
// Phases: full fit (wavefront 0) | pure-genotype sums and call, in order (1); then rounds of the EM
// tasks (0-2): the null fit, the profiles at the ML frequency, 0 and 1 and the bounds' midpoints, 24
// tasks of eight lanes or 48 of four | KS and Fisher (3, first round).
//
// The distinct keys come from a hash of the column's own, so that they cost the same whatever the size of the
// table; a column of more of them than LDS holds rows for reads the table, a row per read, in the same loops
// (31 candidates of 3,000 reads and 40 MAPQs: 5.5 ms, where 45 ordered loops one after the other and
// all candidates took 34 ms, and two ordered tasks per wavefront 26 ms).
//
// With 669 candidates of about 100 reads the kernel takes 0.26 ms (1.23 ms with two ordered EM tasks per
// wavefront in LDS and three rounds of bisection); 28 candidates of 206 reads take 0.15 ms (1.40 ms),
// 36 of 3,000 reads 0.39 ms.
//
// Fisher terms are evaluated across lanes and added in order by one lane; the exact KS lattice is
// filled one anti-diagonal at a time (each cell is one addition of two neighbours, so the order of
// the cells does not change any value).
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "kernels.h"

namespace bsq {

namespace {

constexpr int kSW = kScoreWaves;
static_assert(kSW == 4, "phase roles are laid out for four wavefronts");
constexpr int kTaskWaves = 3;            // wavefronts of the EM tasks; the fourth has the statistics
constexpr int kTaskSlots = 48;           // most tasks of a round: 4 lanes each, or 24 of 8 lanes
constexpr int kKsDiag = 100;             // exact KS runs when m*n < 10000, so min(m, n) <= 99
constexpr uint32_t kNoKey = 0xffffffffu;
constexpr int kScoreProbes = 256;        // hash slots tried before a column counts as having too many distinct keys
constexpr double kDrop = 0.587566;       // kProfileLikelihoodLog10Drop (identify_mutations.cpp:3173)
// How far a result of sums in any order may be from the reference's, which adds n terms one after the
// other: every addition rounds by up to 2^-53 of the sum so far, and where the terms are alike, as those
// of reads that agree, all in one direction.  The sums here are of fewer, larger terms.
//   * A pass moves a frequency by up to n 2^-53 of itself, and EM forgets most of what earlier passes moved (in
//     the frequencies' logarithms a step is the identity less a mean over the reads).  Measured against correctly
//     rounded sums over qualities of 2 to 40 and 30 to 20,000 reads: at most 0.2 n 2^-53 in up to 5 passes, 0.9
//     in 20, 1.2 in 50.  Guard: (2 + passes / 8) n 2^-53, relative.
//   * A log10 likelihood is off by up to n 2^-53 of its size, and by up to n^2 2^-53 because the
//     frequencies add up to 1 only within n 2^-53; measured: at most 0.09 n 2^-53 (n + |log10 likelihood|).
//     Guard: eleven times that, for a score with the likelihoods of both its fits.
//   * A loop ends when no frequency moved by tol.  A step may be off by n 2^-53 for every pass up to it, and
//     for those of the full fit that a profile starts from.  Where one is that close to tol, the full fit is done
//     again in read order; the null fit and the profiles go on until a step is clearly below, and what the
//     passes since can have added to the likelihood is added to the value's guard.
// A decision or a printed digit closer to its boundary than its guard is made on exact sums.  Up to
// some 6,000 reads the least guards of a launch hold (ImParams::guard_log, guard_rel).
constexpr double kHalfUlp = 0x1p-53;
constexpr double kSumSlack = 64.0;       // additions besides those of the reads: a term's own operations

struct ScoreShared {
  double full_f[5];
  double fit[6];                   // frequencies an EM loop starts from and leaves; em_full: its passes
  double full_ll, null_ll;
  double gscore;                   // pure-genotype score
  double lp_best;                  // log10 likelihood of the best pure genotype
  double guard_rel, guard_log;     // the candidate's guards; the score's own size comes on top
  double val[kTaskSlots];          // profile values of the round's tasks (without the lpmax sum)
  double more[kTaskSlots];         // how far the reference's values may be below them for its last pass
  double null_more, target_more, end_more[2];
  double pts[2][kTaskSlots];       // bisection midpoints of the round, per bound
  double vlo[2], vhi[2];           // profile values at the ends of each bound's interval
  double lo[2], hi[2];
  double out[2];                   // the bounds as reported so far
  double target, ks_p, fisher_p;
  double exact_x[2], exact_v, exact_target;
  double ks_a[kKsDiag + 1], ks_b[kKsDiag + 1];
  double fisher[64];
  double ks_log_total;
  uint32_t ks_bnd[(10000 + 2 + 31) / 32 + 1];
  uint32_t qh[2][128];
  uint32_t cov[6][3];
  uint32_t obs[5];                 // reads per observed class (both strands)
  uint32_t wcount[kSW];
  int32_t n_keys;
  int32_t best;                    // pure-genotype best allele
  int32_t iter[2];
  int32_t active[2];
  int32_t depth[2];                // midpoints evaluated this round, per bound
  int32_t slot0[2];                // first task slot of each bound's midpoints
  int32_t n_tree;                  // the first of each bound's midpoints are a full tree's nodes
  int32_t exact;                   // bounds: 0 a round of tasks, 1 + side: an exact comparison is needed
  int32_t exact_have;              // exact_target is known
  int32_t bad_r;                   // a ratio outside the fast division's range
  int32_t crowded;                 // a key found no slot in the hash
  int32_t unsure;                  // a result too close to a boundary: the candidate is done again exactly
  int32_t emitted;
  int32_t done;
};

// LDS views.  Helpers that are not inlined reach shared memory through these, so their accesses
// compile to LDS instructions rather than generic (flat) ones, whose waits also cover memory loads.
typedef __attribute__((address_space(3))) double LdsDouble;
typedef __attribute__((address_space(3))) uint32_t LdsU32;
typedef __attribute__((address_space(3))) ScoreShared LdsShared;

static_assert(sizeof(ScoreShared) <= kScoreStaticLds, "scorer static LDS above its declared bound");

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ double readlane_d(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ double readfirstlane_d(double v) { return readlane_d(v, 0); }

template <int kCtrl>
__device__ __forceinline__ double dpp_add(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffLL), kCtrl, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), kCtrl, 0xf, 0xf, true);
  return v + __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Cross-lane sum over aligned groups of kN lanes; every lane of the group gets the same value.
template <int kN>
__device__ __forceinline__ double sum_lanes(double v) {
  v = dpp_add<0x4E>(dpp_add<0xB1>(v));            // quad_perm: lane ^ 1, lane ^ 2
  if constexpr (kN >= 8) v = dpp_add<0x141>(v);   // row_half_mirror: the other quad of eight lanes
  if constexpr (kN == 64) {
    v = dpp_add<0x140>(v);                        // row_mirror: the other eight of a row
    v = (readlane_d(v, 0) + readlane_d(v, 16)) + (readlane_d(v, 32) + readlane_d(v, 48));
  }
  return v;
}

// 1/s within about an ulp for a normal s well inside the exponent range: the hardware's reciprocal
// estimate and two fused Newton steps.  em_terms, which needs it correctly rounded, adds the correction
// step of a division by s (numerator 1).
__device__ __forceinline__ double recip_newton(double s) {
  double y = __builtin_amdgcn_rcp(s);
  y = fma(fma(-s, y, 1.0), y, y);
  y = fma(fma(-s, y, 1.0), y, y);
  return y;
}

template <bool kListGlobal>
__device__ __forceinline__ uint32_t list_at(const uint32_t* list, int i) {
  if constexpr (kListGlobal) return list[i];
  else return ((const __attribute__((address_space(3))) uint32_t*)list)[i];
}

// The candidate's reads.  A read's likelihoods depend on its table key alone, so the rows
// r[0..4] = 10^(lp_b - lpmax), r[5] = lpmax are kept once per distinct key, with the number of its
// reads, and the reads' list holds each read's row.  Where the rows are is a compile-time choice
// of the loops over them:
//   kRowsLds     in LDS (they fit)
//   kRowsGlobal  in the table in HBM (more distinct keys than rows fit): the list holds keys, and every read is a
//                row of its own
enum { kRowsLds = 0, kRowsGlobal = 1 };

struct Rows {
  const uint32_t* list;         // per read: its row (kRowsLds) or its key (kRowsGlobal)
  const double* lds;            // rows, six doubles each
  const uint32_t* reads;        // per row: its reads (kRowsLds)
  const double* __restrict__ tab_r;
  template <int kKind>
  __device__ __forceinline__ void row(int k, double r[6]) const {   // k: a row or a key
    typedef __attribute__((address_space(3))) const double LdsD;
    if constexpr (kKind == kRowsGlobal) {
      const double* p = tab_r + (size_t)k * 6;
#pragma unroll
      for (int c = 0; c < 6; c++) r[c] = p[c];
    } else {
      const LdsD* p = (const LdsD*)lds + k * 6;
#pragma unroll
      for (int c = 0; c < 6; c++) r[c] = p[c];
    }
  }
  // row `i` of the distinct rows, and its reads
  template <int kKind, bool kListGlobal>
  __device__ __forceinline__ uint32_t distinct(int i, double r[6]) const {
    if constexpr (kKind == kRowsGlobal) {
      row<kKind>((int)list_at<kListGlobal>(list, i), r);
      return 1u;
    } else {
      row<kKind>(i, r);
      return ((const __attribute__((address_space(3))) uint32_t*)reads)[i];
    }
  }
};

// Arguments of functions that are not inlined arrive in vector registers; a wave-uniform one is
// made scalar again, so that the branches and loops on it are scalar too.
__device__ __forceinline__ int uniform_i(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <class T>
__device__ __forceinline__ T* uniform_p(T* q) {
  const uint64_t u = (uint64_t)q;
  const uint32_t lo = (uint32_t)uniform_i((int)(uint32_t)u), hi = (uint32_t)uniform_i((int)(uint32_t)(u >> 32));
  return (T*)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ Rows uniform_rows(const Rows& R) {
  return Rows{uniform_p(R.list), uniform_p(R.lds), uniform_p(R.reads), uniform_p(R.tab_r)};
}

// One step of the two in-order chains: a += (lane K of this lane's row of ta), b likewise.
// v_fmac_f64 rounds ta * 1.0 + a once, as an addition does.
#define BSQ_CHAIN(K)                                                                                  \
  asm("v_fmac_f64_dpp %0, %2, %4 row_newbcast:" #K " row_mask:0xf bank_mask:0xf\n\t"                  \
      "v_fmac_f64_dpp %1, %3, %4 row_newbcast:" #K " row_mask:0xf bank_mask:0xf"                       \
      : "+v"(a), "+v"(b)                                                                              \
      : "v"(ta), "v"(tb), "v"(one))
// the first step waits out the VALU-write-to-DPP-read hazard of its operands, the last one the
// VALU-write-to-readlane hazard of its results
#define BSQ_CHAIN_FIRST                                                                               \
  asm("s_nop 1\n\t"                                                                                   \
      "v_fmac_f64_dpp %0, %2, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"                       \
      "v_fmac_f64_dpp %1, %3, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf"                            \
      : "+v"(a), "+v"(b)                                                                              \
      : "v"(ta), "v"(tb), "v"(one))
#define BSQ_CHAIN_LAST                                                                                \
  asm("v_fmac_f64_dpp %0, %2, %4 row_newbcast:15 row_mask:0xf bank_mask:0xf\n\t"                      \
      "v_fmac_f64_dpp %1, %3, %4 row_newbcast:15 row_mask:0xf bank_mask:0xf\n\t"                      \
      "s_nop 1"                                                                                       \
      : "+v"(a), "+v"(b)                                                                              \
      : "v"(ta), "v"(tb), "v"(one))

// The terms of 16 reads (one per lane of a row, the same reads in every row): ta the row's allele
// w_i(g), tb the fifth allele's, w_i(b) = f_b r_i(b) / s_i with s_i = Sum_b f_b r_i(b) in allele
// order, each quotient correctly rounded (the SharedDiv step: one reciprocal per read, then an FMA
// correction); f_b where s_i = 0; -0.0, which changes no sum, past the last read.  An allele that
// is not allowed has f_b = 0, so its products add nothing to s_i and its terms are 0.
struct Freq {
  double f0, f1, f2, f3, f4;
  double fg;      // the frequency of this lane's row
  bool slow;      // a product f_b r_i(b) may be too small for the shared reciprocal
};

__device__ __forceinline__ double row_value(double v0, double v1, double v2, double v3, int g) {
  return g < 2 ? (g == 0 ? v0 : v1) : (g == 2 ? v2 : v3);
}

struct Terms {
  double ta, tb;
  double s, xg, x4;
};

__device__ __forceinline__ Terms em_terms(const double r[6], const Freq& F, int g, bool live) {
  Terms T;
  const double x0 = F.f0 * r[0], x1 = F.f1 * r[1], x2 = F.f2 * r[2], x3 = F.f3 * r[3];
  T.x4 = F.f4 * r[4];
  T.s = (((x0 + x1) + x2) + x3) + T.x4;
  T.xg = row_value(x0, x1, x2, x3, g);
  const double y0 = recip_newton(T.s);
  const double y = fma(fma(-T.s, y0, 1.0), y0, y0);
  const double qa = T.xg * y, qb = T.x4 * y;
  const double ta = fma(fma(-T.s, qa, T.xg), y, qa);
  const double tb = fma(fma(-T.s, qb, T.x4), y, qb);
  T.ta = live ? ta : -0.0;
  T.tb = live ? tb : -0.0;
  return T;
}

// The terms by ordinary division, f_b where s_i = 0: what the fast quotients do not cover.
__device__ __forceinline__ void em_terms_slow(Terms& T, const Freq& F, bool live) {
  const double ta = (T.s > 0.0) ? T.xg / T.s : F.fg;
  const double tb = (T.s > 0.0) ? T.x4 / T.s : F.f4;
  T.ta = live ? ta : -0.0;
  T.tb = live ? tb : -0.0;
}

// One EM loop of the reference with its sums in read order, by one wavefront; returns the log10
// likelihood it reports and leaves the final frequencies in fit[].
//   mode 1: fit_allele_frequencies (identify_mutations.cpp:3240-3318) from the frequencies in fit[];
//           allele v (if any) is held out, with frequency zero.
//   mode 2: profile_log10_likelihood (:3094-3143): fit[v] pinned to x.
// 50 passes at most; a loop ends when no frequency moved by tol, and the likelihood is that of the
// last pass's frequencies: Sum_i (log10 s_i + lpmax_i) over reads with s_i > 0, in read order.
template <int kKind, bool kListGlobal>
__device__ __noinline__ double em_exact(const Rows Rv, int nv, int modev, int vv, double xv, LdsDouble* fit, double tolv,
                                        int bad_rv) {
  const Rows R = uniform_rows(Rv);
  const int n = uniform_i(nv), mode = uniform_i(modev), v = uniform_i(vv), bad_r = uniform_i(bad_rv);
  const double x = readfirstlane_d(xv), tol = readfirstlane_d(tolv);
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
  auto L = [&](int i) { return (int)list_at<kListGlobal>(R.list, i); };
  Freq F;
  F.f0 = readfirstlane_d(fit[0]);
  F.f1 = readfirstlane_d(fit[1]);
  F.f2 = readfirstlane_d(fit[2]);
  F.f3 = readfirstlane_d(fit[3]);
  F.f4 = readfirstlane_d(fit[4]);
  double l0, l1, l2, l3, l4;   // frequencies of the last pass
  const double dn = (double)n, one = 1.0;
  const SharedDiv by_n(dn);
  // the first two groups of 16 reads, which every pass begins with
  double r0[6], r1[6];
  R.row<kKind>(L(min(j, n - 1)), r0);
  R.row<kKind>(L(min(16 + j, n - 1)), r1);
  const int third = L(min(32 + j, n - 1));
  F.fg = row_value(F.f0, F.f1, F.f2, F.f3, g);
  for (int it = 0;;) {
    // with a ratio of at least 2^-100 or 0, a frequency of at least 2^-800 or 0 keeps every product
    // inside the range where the fast quotients are correctly rounded
    F.slow = bad_r || __any((F.fg != 0.0 && F.fg < 0x1p-800) || (F.f4 != 0.0 && F.f4 < 0x1p-800));
    double a = 0.0, b = 0.0;
    double r[6];
    Terms T = em_terms(r0, F, g, j < n);
    if (F.slow || __any(!(T.s > 0.0))) em_terms_slow(T, F, j < n);
#pragma unroll
    for (int k = 0; k < 6; k++) r[k] = r1[k];
    int next = third;
    for (int c0 = 0; c0 < n; c0 += 16) {
      // the chain over these 16 reads, with the next 16 reads' terms computed between its steps
      // (the compiler interleaves them) and the reads after those loaded
      const double ta = T.ta, tb = T.tb;
      const bool live = c0 + 16 + j < n;
      BSQ_CHAIN_FIRST;
      BSQ_CHAIN(1);
      BSQ_CHAIN(2);
      BSQ_CHAIN(3);
      T = em_terms(r, F, g, live);
      R.row<kKind>(next, r);
      next = L(min(c0 + 48 + j, n - 1));
      BSQ_CHAIN(4);
      BSQ_CHAIN(5);
      BSQ_CHAIN(6);
      BSQ_CHAIN(7);
      BSQ_CHAIN(8);
      BSQ_CHAIN(9);
      BSQ_CHAIN(10);
      BSQ_CHAIN(11);
      BSQ_CHAIN(12);
      BSQ_CHAIN(13);
      BSQ_CHAIN(14);
      BSQ_CHAIN_LAST;
      // the usual terms are final here, in the chain's own block; without this the compiler moves
      // their divisions behind the branch below
      asm volatile("" : "+v"(T.ta), "+v"(T.tb));
      if (F.slow || __any(!(T.s > 0.0))) em_terms_slow(T, F, live);
    }
    // the reference's loop body: new frequencies, and whether any moved by tol
    double fa = F.fg, fb = F.f4;
    if (mode == 1) {
      if (g != v) fa = by_n(a);
      if (4 != v) fb = by_n(b);
    } else {
      const double s0 = readlane_d(a, 0), s1 = readlane_d(a, 16), s2 = readlane_d(a, 32), s3 = readlane_d(a, 48), s4 = b;
      double others = 0.0;
      if (v != 0) others += s0;
      if (v != 1) others += s1;
      if (v != 2) others += s2;
      if (v != 3) others += s3;
      if (v != 4) others += s4;
      const SharedDiv d(others);
      const double rest = (1.0 - x) / 4.0;
      if (g != v) fa = (others > 0.0) ? d((1.0 - x) * a) : rest;
      if (4 != v) fb = (others > 0.0) ? d((1.0 - x) * b) : rest;
    }
    const bool moved = __any(fabs(fa - F.fg) >= tol || fabs(fb - F.f4) >= tol);
    l0 = F.f0;
    l1 = F.f1;
    l2 = F.f2;
    l3 = F.f3;
    l4 = F.f4;
    F.f0 = readlane_d(fa, 0);
    F.f1 = readlane_d(fa, 16);
    F.f2 = readlane_d(fa, 32);
    F.f3 = readlane_d(fa, 48);
    F.f4 = readlane_d(fb, 0);
    F.fg = fa;
    if (++it >= 50 || !moved) break;
  }
  if (lane == 0) {
    fit[0] = F.f0;
    fit[1] = F.f1;
    fit[2] = F.f2;
    fit[3] = F.f3;
    fit[4] = F.f4;
  }
  // the likelihood: 64 reads' terms at a time, added row by row
  double ll = 0.0;
  for (int c0 = 0; c0 < n; c0 += 64) {
    double r[6];
    R.row<kKind>(L(min(c0 + lane, n - 1)), r);
    const double s = (((l0 * r[0] + l1 * r[1]) + l2 * r[2]) + l3 * r[3]) + l4 * r[4];
    double ta = (s > 0.0) ? log10(s) + r[5] : 0.0;
    if (c0 + lane >= n) ta = -0.0;
    const double tb = -0.0;
    double b = 0.0;
#pragma unroll 1
    for (int row = 0; row < 64; row += 16) {
      double a = ll;
      BSQ_CHAIN_FIRST;
      BSQ_CHAIN(1);
      BSQ_CHAIN(2);
      BSQ_CHAIN(3);
      BSQ_CHAIN(4);
      BSQ_CHAIN(5);
      BSQ_CHAIN(6);
      BSQ_CHAIN(7);
      BSQ_CHAIN(8);
      BSQ_CHAIN(9);
      BSQ_CHAIN(10);
      BSQ_CHAIN(11);
      BSQ_CHAIN(12);
      BSQ_CHAIN(13);
      BSQ_CHAIN(14);
      BSQ_CHAIN_LAST;
      ll = readlane_d(a, row);
    }
  }
  return ll;
}

// The in-order sums of the reads' log10 likelihoods under each hypothesis (identify_mutations.cpp:
// 1669-1689), by one wavefront: lane g*16 + j reads hypothesis g of read j, as em_exact's rows.
template <bool kListGlobal>
__device__ __noinline__ void genotype_sums(const uint32_t* list, const uint32_t* key_of, const double* __restrict__ tab_lp,
                                           int nv, double* lps) {
  const int n = uniform_i(nv);
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
  const double one = 1.0;
  double a = 0.0, b = 0.0;
  for (int c0 = 0; c0 < n; c0 += 64) {
    double va[4], vb[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int i = c0 + 16 * q + j;
      const uint32_t e = list_at<kListGlobal>(list, min(i, n - 1));
      const double* lp = tab_lp + (size_t)(key_of ? key_of[e] : e) * 5;
      va[q] = lp[g];
      vb[q] = lp[4];
      if (i >= n) va[q] = vb[q] = -0.0;
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const double ta = va[q], tb = vb[q];
      BSQ_CHAIN_FIRST;
      BSQ_CHAIN(1);
      BSQ_CHAIN(2);
      BSQ_CHAIN(3);
      BSQ_CHAIN(4);
      BSQ_CHAIN(5);
      BSQ_CHAIN(6);
      BSQ_CHAIN(7);
      BSQ_CHAIN(8);
      BSQ_CHAIN(9);
      BSQ_CHAIN(10);
      BSQ_CHAIN(11);
      BSQ_CHAIN(12);
      BSQ_CHAIN(13);
      BSQ_CHAIN(14);
      BSQ_CHAIN_LAST;
    }
  }
  lps[0] = readlane_d(a, 0);
  lps[1] = readlane_d(a, 16);
  lps[2] = readlane_d(a, 32);
  lps[3] = readlane_d(a, 48);
  lps[4] = readlane_d(b, 0);
}

// Sum_i log10 s_i over distinct rows with their reads, s_i > 2^-100: the products of the powers,
// exponents kept apart, one logarithm at the end.
struct LogSum {
  double p = 1.0;
  int e = 0;
  __device__ __forceinline__ void add(double s, uint32_t h) {
    double q = s;
    int eq = 0;
    for (;;) {
      if (h & 1u) {
        p *= q;
        e += __builtin_amdgcn_frexp_exp(p) + eq;
        p = __builtin_amdgcn_frexp_mant(p);
      }
      h >>= 1;
      if (!h) break;
      q *= q;
      const int x = __builtin_amdgcn_frexp_exp(q);
      q = __builtin_amdgcn_frexp_mant(q);
      eq = 2 * eq + x;
    }
  }
  __device__ __forceinline__ double value() const { return log10(p) + (double)e * 0.30102999566398119521; }
};

// fit_allele_frequencies (identify_mutations.cpp:3240-3318) over all alleles with sums in any order,
// by one wavefront: 64 lanes share the distinct rows.  Leaves the frequencies in f and returns the
// log10 likelihood without the sum of the reads' lpmax; NaN where the loop cannot stand for the
// reference's (a read with s_i = 0, or a step too close to tol).  nu: (n + kSumSlack) 2^-53; fit[5]: the passes
// made.
template <int kKind, bool kListGlobal>
__device__ __noinline__ double em_full(const Rows Rv, int Kv, int nv, LdsDouble* fit, double tol, double nu) {
  const Rows R = uniform_rows(Rv);
  const int K = uniform_i(Kv), lane = threadIdx.x & 63;
  const double per_n = 1.0 / (double)uniform_i(nv);
  double f[5], fl[5];
#pragma unroll
  for (int b = 0; b < 5; b++) f[b] = fl[b] = fit[b];
  bool bad = false;
  int it = 1;
  for (;; it++) {
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int i = lane; i < K; i += 64) {
      double r[6];
      const uint32_t h = R.distinct<kKind, kListGlobal>(i, r);
      double s = f[0] * r[0];
#pragma unroll
      for (int b = 1; b < 5; b++) s = fma(f[b], r[b], s);
      const double y = recip_newton(s) * (double)h;
#pragma unroll
      for (int b = 0; b < 5; b++) acc[b] = fma(r[b], y, acc[b]);
    }
    double most = 0.0, sum = 0.0;
#pragma unroll
    for (int b = 0; b < 5; b++) {
      fl[b] = f[b];
      f[b] = f[b] * sum_lanes<64>(acc[b]) * per_n;
      sum += f[b];
      most = fmax(most, fabs(f[b] - fl[b]));
    }
    bad = bad || !(sum > 0.5 && sum < 2.0) || (it < 50 && fabs(most - tol) < fmax(1e-6 * tol, (double)(it + 1) * nu));
    if (!(most >= tol) || it >= 50) break;
  }
  LogSum L;
  for (int i = lane; i < K; i += 64) {
    double r[6];
    const uint32_t h = R.distinct<kKind, kListGlobal>(i, r);
    double s = fl[0] * r[0];
#pragma unroll
    for (int b = 1; b < 5; b++) s = fma(fl[b], r[b], s);
    bad = bad || !(s > 0x1p-100);
    L.add(s, h);
  }
  const double ll = sum_lanes<64>(L.value());
  if (lane == 0) {
#pragma unroll
    for (int b = 0; b < 5; b++) fit[b] = f[b];
    fit[5] = (double)it;
  }
  return __any(bad) ? __longlong_as_double(0x7ff8000000000000LL) : ll;
}

// The rows of em_tasks: get() returns row i's ratios, the variant's first and the other four alleles' in
// order, and its reads.
struct TaskRowsLds {      // six doubles a row, laid out so
  const LdsDouble* prow;
  __device__ __forceinline__ TaskRowsLds uniform() const { return *this; }
  __device__ __forceinline__ double get(int i, double r[5]) const {
    typedef __attribute__((address_space(3))) const char LdsChar;
    const LdsDouble* p = (const LdsDouble*)((LdsChar*)prow + __umul24((uint32_t)i, 48u));
#pragma unroll
    for (int b = 0; b < 5; b++) r[b] = p[b];
    return p[5];
  }
};
template <bool kListGlobal>
struct TaskRowsGlobal {   // rows of the table, a read each: the variant comes first through the columns' addresses
  const uint32_t* list;
  const double* __restrict__ tab_r;
  int variant;
  __device__ __forceinline__ TaskRowsGlobal uniform() const { return {uniform_p(list), uniform_p(tab_r), uniform_i(variant)}; }
  __device__ __forceinline__ double get(int i, double r[5]) const {
    const uint32_t at = list_at<kListGlobal>(list, i) * 48u;
    r[0] = *(const double*)((const char*)(tab_r + variant) + at);
#pragma unroll
    for (int b = 0; b < 4; b++) r[b + 1] = *(const double*)((const char*)(tab_r + b + (b >= variant ? 1 : 0)) + at);
    return 1.0;
  }
};

// The EM tasks of one wavefront, kSub lanes each: the null fit (the variant held out, from the counts
// of the reads' observations) or profile_log10_likelihood (identify_mutations.cpp:3094-3143: the
// variant pinned to x, the others from the full fit rescaled), the same iterations as em_exact's with
// sums in any order over the candidate's K rows (Src: TaskRowsLds or TaskRowsGlobal).  Returns log10 of the likelihood without
// the sum of the reads' lpmax, which every such value of a candidate shares, NaN where it cannot
// stand for the reference's (a read with s_i = 0), and how far below it the reference's may be because it may
// have ended some passes earlier: a step from f to g adds at most Sum_b (g_b - f_b) Sum_i r_i(b) / s_i to the likelihood's
// natural logarithm, which is concave.
//   nu: (n + kSumSlack) 2^-53; passes: those before the start, and one
//   start[4]: the other alleles' starting frequencies; scale: 1 / n in the null fit, else 0
struct TaskValue {
  double ll, more;
};

template <int kSub, class Src>
__device__ __noinline__ TaskValue em_tasks(const Src Sv, int Kv, double x, double start0, double start1, double start2,
                                        double start3, double scale_null, bool active, double tol, double nu, double passes) {
  const Src rows = Sv.uniform();
  const int K = uniform_i(Kv), sub = threadIdx.x & (kSub - 1);
  double f1 = start0, f2 = start1, f3 = start2, f4 = start3;
  const double rest = (1.0 - x) / 4.0;
  const bool null_fit = scale_null != 0.0;
  bool run = active, bad = false, ended = false;   // ended: the reference's loop may have
  double more = 0.0;
  for (int it = 1; __any(run); it++) {
    double a1 = 0.0, a2 = 0.0, a3 = 0.0, a4 = 0.0;
    // Four rows of a lane at a time, step by step: a row's chain (five products, a reciprocal, four
    // sums) is some 250 cycles of latency and 16 instructions, so four in flight fill each other's
    // waits.  The barriers keep the steps apart: left to itself the compiler runs the rows one after
    // the other.
    for (int i0 = sub; i0 < K; i0 += 4 * kSub) {
      double r[4][5], h[4], s[4], y[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        h[u] = rows.get(min(i0 + u * kSub, K - 1), r[u]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; u++) s[u] = x * r[u][0];
#pragma unroll
      for (int u = 0; u < 4; u++) s[u] = fma(f1, r[u][1], s[u]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; u++) s[u] = fma(f2, r[u][2], s[u]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; u++) s[u] = fma(f3, r[u][3], s[u]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; u++) s[u] = fma(f4, r[u][4], s[u]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; u++) y[u] = __builtin_amdgcn_rcp(s[u]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int step = 0; step < 2; step++) {   // recip_newton
        double e[4];
#pragma unroll
        for (int u = 0; u < 4; u++) e[u] = fma(-s[u], y[u], 1.0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 4; u++) y[u] = fma(e[u], y[u], y[u]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) y[u] *= (i0 + u * kSub < K) ? h[u] : 0.0;   // here: the loads' last values
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        a1 = fma(r[u][1], y[u], a1);
        a2 = fma(r[u][2], y[u], a2);
        a3 = fma(r[u][3], y[u], a3);
        a4 = fma(r[u][4], y[u], a4);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    const double q1 = sum_lanes<kSub>(a1), q2 = sum_lanes<kSub>(a2), q3 = sum_lanes<kSub>(a3), q4 = sum_lanes<kSub>(a4);
    a1 = f1 * q1;
    a2 = f2 * q2;
    a3 = f3 * q3;
    a4 = f4 * q4;
    const double others = (a1 + a2) + (a3 + a4);
    const double scale = null_fit ? scale_null : (1.0 - x) * recip_newton(others);
    const bool some = others > 0.0;
    const double g1 = some ? scale * a1 : rest, g2 = some ? scale * a2 : rest;
    const double g3 = some ? scale * a3 : rest, g4 = some ? scale * a4 : rest;
    const double most = fmax(fmax(fabs(g1 - f1), fabs(g2 - f2)), fmax(fabs(g3 - f3), fabs(g4 - f4)));
    // (not-a-number sums fail the first test)
    bad |= run & (!(others >= 0.0) | ((others > 0.0) & (others < 0x1p-500)));
    const double room = fmax(1e-6 * tol, ((double)it + passes) * nu);
    ended |= run & (most < tol + room);
    run &= (most >= tol - room) & (it < 50);
    if (__any(run & ended)) {
      const double gain = ((g1 - f1) * q1 + (g2 - f2) * q2) + ((g3 - f3) * q3 + (g4 - f4) * q4);
      if (run & ended) more += fmax(gain, 0.0);
    }
    // a task that ends keeps this pass's frequencies: the likelihood is theirs
    f1 = run ? g1 : f1;
    f2 = run ? g2 : f2;
    f3 = run ? g3 : f3;
    f4 = run ? g4 : f4;
  }
  LogSum L;
  for (int i = sub; i < K; i += kSub) {
    double p[5];
    const double reads = rows.get(i, p);
    const double s = fma(f4, p[4], fma(f3, p[3], fma(f2, p[2], fma(f1, p[1], x * p[0]))));
    bad = bad || !(s > 0x1p-100);
    L.add(s, (uint32_t)reads);
  }
  const double ll = sum_lanes<kSub>(L.value());
  // one lane that saw a read it cannot stand for spoils its task
  const unsigned long long m = __ballot(bad);
  const int base = (threadIdx.x & 63) & ~(kSub - 1);
  return {((m >> base) & ((1ull << kSub) - 1ull)) ? __longlong_as_double(0x7ff8000000000000LL) : ll, 0.5 * more};
}

// Where the profile likelihood is predicted to cross the target inside the interval of bound
// `side` (lanes 0-31: the lower bound, lanes 32-63: the upper one), used only to choose which
// midpoints to evaluate.  Model: m(x) = Sum_i log10(t_i + x d_i), the likelihood with the other
// alleles' proportions held at the full fit's (t_i their mixture, d_i = r_i(v) - t_i), with FP32
// logarithms, whose rounding moves the prediction by about 1e-7.  It is evaluated at 32 points per
// interval, the one bracketing the crossing is divided again, three times over, and the last
// bracket's ends are joined by a line.  Once profile values are known at the interval's ends, the model
// is corrected by the line through its errors there.  On 669 candidates of a 100x sample the path it
// gives is right to the last of some 20 levels for 96% of the bounds.
//   pre: per row d_i, t_i; prow: per row, its reads at [5] (null: one each)
//   Kv: the rows, or as many of them as pre holds: fewer than all only predict less well
//   known: the values vlo / vhi hold (else the target is m at the ML frequency, minus the drop)
template <bool kOnes>
__device__ __noinline__ double model_root(const LdsDouble* prow, const LdsDouble* pre, int Kv, double lo, double hi, bool known,
                                          double vlo, double vhi, double target) {
  const int K = uniform_i(Kv);
  const int lane = threadIdx.x & 63, side = lane >> 5, k = lane & 31;
  double a = lo, b = hi, d0 = 0.0, d1 = 0.0, va = 0.0, vb = 0.0;
#pragma unroll 1
  for (int round = 0; round < 3; round++) {
    const double x = a + (b - a) * ((double)k * (1.0 / 31.0));
    double l2 = 0.0;
#pragma unroll 4
    for (int i = 0; i < K; i++)
      l2 = fma(kOnes ? 1.0 : prow[6 * i + 5], (double)__builtin_amdgcn_logf((float)fma(x, pre[2 * i], pre[2 * i + 1])), l2);
    const double m = l2 * 0.30102999566398119521;
    if (round == 0) {
      const double m_lo = __shfl(m, 32 * side, 64), m_hi = __shfl(m, 32 * side + 31, 64);
      if (known) {
        d0 = vlo - m_lo;
        d1 = vhi - m_hi;
        if (!isfinite(d0)) d0 = isfinite(d1) ? d1 : 0.0;
        if (!isfinite(d1)) d1 = d0;
      } else {
        target = ((side == 0) ? m_hi : m_lo) - kDrop;   // the ML frequency is the inner end
      }
    }
    const double y = m + d0 + (hi > lo ? (d1 - d0) * ((x - lo) / (hi - lo)) : 0.0);
    // lower bound: the profile rises towards the ML frequency; upper bound: it falls away from it
    const bool before = (side == 0) ? (y < target) : (y >= target);
    const uint32_t half = (uint32_t)(__ballot(before) >> (32 * side));
    int c = __popc(half);
    c = min(max(c, 1), 31);
    va = __shfl(y, 32 * side + c - 1, 64);
    vb = __shfl(y, 32 * side + c, 64);
    const double na = a + (b - a) * ((double)(c - 1) * (1.0 / 31.0)), nb = a + (b - a) * ((double)c * (1.0 / 31.0));
    a = na;
    b = nb;
  }
  const double t = (target - va) / (vb - va);
  return a + (b - a) * ((t >= 0.0 && t <= 1.0) ? t : 0.5);
}

__device__ __noinline__ double lgamma_w(double x) { return lgamma(x); }

// fisher_exact_test_2x2 (stats.cpp:2144-2169) and the logarithm of KS's lattice count: terms across
// lanes, summed in order by lane 0.  The nine logarithms of factorials that every lane needs (and
// three for KS) are one lgamma evaluated on twelve lanes, and the four that a term needs of its own
// one each: an lgamma is some thousand cycles, and the chain of eighteen was the longest part of
// the statistics.  log C(n, k) is lgamma(n + 1) - lgamma(k + 1) - lgamma(n - k + 1), as the reference
// forms it.
//   choose_ks: returns log C(ks_n, ks_k) too
__device__ __noinline__ double fisher_2x2_w(uint32_t a, uint32_t b, uint32_t c, uint32_t d, LdsDouble* buf, uint32_t ks_n,
                                            uint32_t ks_k, LdsDouble* choose_ks) {
  const int lane = threadIdx.x & 63;
  const uint32_t row1 = a + b, row2 = c + d, col1 = a + c, col2 = b + d;
  const uint32_t n = row1 + row2;
  const uint32_t a_min = (row1 > col2) ? (row1 - col2) : 0;
  const uint32_t a_max = min(row1, col1);
  // arguments as the reference's doubles: whole numbers, exact
  double arg = 1.0;
  if (lane == 0) arg = (double)n + 1;
  if (lane == 1) arg = (double)row1 + 1;
  if (lane == 2) arg = (double)n - (double)row1 + 1;
  if (lane == 3) arg = (double)col1 + 1;
  if (lane == 4) arg = (double)a + 1;
  if (lane == 5) arg = (double)col1 - (double)a + 1;
  if (lane == 6) arg = (double)col2 + 1;
  if (lane == 7) arg = (double)(row1 - a) + 1;
  if (lane == 8) arg = (double)col2 - (double)(row1 - a) + 1;
  if (lane == 9) arg = (double)ks_n + 1;
  if (lane == 10) arg = (double)ks_k + 1;
  if (lane == 11) arg = (double)ks_n - (double)ks_k + 1;
  const double lg = lgamma_w(arg);
  if (lane == 0) *choose_ks = readlane_d(lg, 9) - readlane_d(lg, 10) - readlane_d(lg, 11);
  const double g_col1 = readlane_d(lg, 3), g_col2 = readlane_d(lg, 6);
  const double log_denom = readlane_d(lg, 0) - readlane_d(lg, 1) - readlane_d(lg, 2);
  const double lpo = (g_col1 - readlane_d(lg, 4) - readlane_d(lg, 5)) + (g_col2 - readlane_d(lg, 7) - readlane_d(lg, 8)) - log_denom;
  const double lre = log(1.0 + 1e-7);
  double total = 0.0;
  for (uint32_t base = a_min; base <= a_max; base += 64) {
    const uint32_t ai = min(base + (uint32_t)lane, a_max);
    const double l1 = g_col1 - lgamma_w((double)ai + 1) - lgamma_w((double)col1 - (double)ai + 1);
    const double l2 = g_col2 - lgamma_w((double)(row1 - ai) + 1) - lgamma_w((double)col2 - (double)(row1 - ai) + 1);
    const double lp = l1 + l2 - log_denom;
    buf[lane] = (lp <= lpo + lre) ? exp(lp) : 0.0;
    wave_sync();
    if (lane == 0) {
      const uint32_t m = min<uint32_t>(64u, a_max - base + 1u);
      for (uint32_t j = 0; j < m; j++) total += buf[j];
    }
    wave_sync();
  }
  return fmin(readlane_d(total, 0), 1.0);
}

// ks_test_two_sample_less (stats.cpp:2190-2284) from per-quality histograms of x (minor allele) and
// y (major allele); pooled ties are whole quality values.  log_total: log C(nx + ny, ny).
__device__ __noinline__ double ks_less_w(LdsShared* SS, uint32_t nxv, uint32_t nyv, double log_total) {
  const int lane = threadIdx.x & 63;
  const uint32_t nx = (uint32_t)uniform_i((int)nxv), ny = (uint32_t)uniform_i((int)nyv);
  // the counts up to qualities 2 * lane and 2 * lane + 1
  const uint32_t hx0 = SS->qh[0][2 * lane], hx1 = SS->qh[0][2 * lane + 1];
  const uint32_t hy0 = SS->qh[1][2 * lane], hy1 = SS->qh[1][2 * lane + 1];
  uint32_t cx1 = hx0 + hx1, cy1 = hy0 + hy1;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t ux = __shfl_up(cx1, o, 64), uy = __shfl_up(cy1, o, 64);
    if (lane >= o) {
      cx1 += ux;
      cy1 += uy;
    }
  }
  const uint32_t cx0 = cx1 - hx1, cy0 = cy1 - hy1;
  // the statistic: the least z over the qualities that occur, the first of equal ones
  const bool on0 = hx0 + hy0 != 0, on1 = hx1 + hy1 != 0;
  const double z0 = on0 ? (double)cx0 / nx - (double)cy0 / ny : INFINITY;
  const double z1 = on1 ? (double)cx1 / nx - (double)cy1 / ny : INFINITY;
  const double z = (z1 < z0) ? z1 : z0;
  const uint32_t zx = (z1 < z0) ? cx1 : cx0, zy = (z1 < z0) ? cy1 : cy0;
  double min_z = z;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) min_z = fmin(min_z, __shfl_xor(min_z, o, 64));
  const int at = __builtin_ctzll(__ballot(z == min_z) | (1ull << 63));
  const uint32_t bx = (uint32_t)__builtin_amdgcn_readlane((int)zx, at), by = (uint32_t)__builtin_amdgcn_readlane((int)zy, at);
  min_z = readlane_d(min_z, 0);
  const double stat = -min_z;
  if ((double)nx * ny >= 10000) {
    const double neff = ((double)nx * ny) / (nx + ny);
    return exp(-2.0 * stat * stat * neff);
  }
  const uint32_t m = ny, n = nx;   // cells (i, j), i <= m over y, j <= n over x
  const int64_t thr = (int64_t)by * n - (int64_t)bx * m;
  const uint32_t D = m + n;
  // m * n < 10000 bounds the lattice: min(m, n) <= 99 cells per diagonal, D <= 10000 boundary bits
  if (min(m, n) > (uint32_t)kKsDiag || D > 10000u) return __longlong_as_double(0x7ff8000000000000LL);
  // boundary(d): d is 0 or the pooled count at the end of a tie group
  const uint32_t nw = D / 32 + 1;
  for (uint32_t k = lane; k < nw; k += 64) SS->ks_bnd[k] = (k == 0) ? 1u : 0u;
  wave_sync();
  if (on0) __hip_atomic_fetch_or(&SS->ks_bnd[(cx0 + cy0) >> 5], 1u << ((cx0 + cy0) & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  if (on1) __hip_atomic_fetch_or(&SS->ks_bnd[(cx1 + cy1) >> 5], 1u << ((cx1 + cy1) & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  wave_sync();
  // the diagonal index runs over the smaller dimension
  const bool by_i = (m <= n);
  const uint32_t small = by_i ? m : n, large = by_i ? n : m;
  double umn;
  if (small < 64u) {
    // A diagonal in registers, cell s on lane s: a cell is its own and the lane before's value on the
    // diagonal before.  A cell that does not exist yet is 0; one that has left the lattice is not
    // read again by a cell inside it.
    const int32_t ti = (int32_t)thr;
    double u = (lane == 0) ? 1.0 : 0.0;
    int32_t lvl = by_i ? lane * (int32_t)(n + m) : -lane * (int32_t)(n + m);   // i*n - j*m on diagonal 0
    const int32_t step = by_i ? -(int32_t)m : (int32_t)n;
    uint32_t word = 0;
    for (uint32_t d = 0; d <= D; d++) {
      if ((d & 31u) == 0) word = (uint32_t)uniform_i((int)SS->ks_bnd[d >> 5]);
      if (d > 0) {
        const long long bits = __double_as_longlong(u);
        const int lo = __builtin_amdgcn_mov_dpp((int)(bits & 0xffffffffLL), 0x138, 0xf, 0xf, true);   // wave_shr:1
        const int hi = __builtin_amdgcn_mov_dpp((int)(bits >> 32), 0x138, 0xf, 0xf, true);
        u = __longlong_as_double(((long long)hi << 32) | (unsigned int)lo) + u;
      }
      if (((word >> (d & 31u)) & 1u) && lvl >= ti) u = 0.0;
      lvl += step;
    }
    umn = readlane_d(u, (int)small);
  } else {
    LdsDouble* A = SS->ks_a;   // diagonal d-1
    LdsDouble* B = SS->ks_b;   // diagonal d
    for (uint32_t d = 0; d <= D; d++) {
      const bool bnd = (SS->ks_bnd[d >> 5] >> (d & 31)) & 1u;
      const uint32_t s_lo = (d > large) ? d - large : 0u;
      const uint32_t s_hi = min(small, d);
      for (uint32_t s = s_lo + lane; s <= s_hi; s += 64) {
        const uint32_t i = by_i ? s : d - s;
        const uint32_t j = by_i ? d - s : s;
        double val;
        if (d == 0) {
          val = 1.0;
        } else {
          // u[i-1][j] + u[i][j-1], both on diagonal d-1
          const double up = (i > 0) ? A[by_i ? s - 1 : s] : 0.0;
          const double left = (j > 0) ? A[by_i ? s : s - 1] : 0.0;
          val = up + left;
        }
        const int64_t lvl = (int64_t)i * n - (int64_t)j * m;
        if (lvl >= thr && bnd) val = 0.0;
        B[s] = val;
      }
      wave_sync();
      LdsDouble* t = A;
      A = B;
      B = t;
    }
    umn = A[small];
  }
  const double total = exp(log_total);
  const double pv = 1.0 - umn / total;
  return fmin(fmax(pv, 0.0), 1.0);
}

// pure_genotype_call kept out of line: its FP64 pow/log10 would otherwise set the register
// footprint of the whole kernel.
__device__ __noinline__ void pure_genotype_call(const double* lps, uint32_t n, int* best, double* score) {
  double l[5];
  for (int b = 0; b < 5; b++) l[b] = lps[b];
  pure_genotype(l, n, *best, *score);
}

// allele_model::major_index / next_index (identify_mutations.cpp:3061-3086)
__device__ __forceinline__ int major_index(const double f[5], uint32_t n) {
  if (n == 0) return 5;
  int best = 0;
  for (int b = 1; b < 5; b++)
    if (f[b] > f[best]) best = b;
  return (f[best] > 0.0) ? best : 5;
}

__device__ __forceinline__ int next_index(const double f[5], uint32_t n, int excl) {
  if (n == 0) return 5;
  const double thr = 0.5 / (double)n;
  int best = 5;
  for (int b = 0; b < 5; b++) {
    if (b == excl) continue;
    if (f[b] < thr) continue;
    if (best == 5 || f[b] > f[best]) best = b;
  }
  return best;
}

// KS quality and Fisher strand p values of the entry (annotate_polymorphism_statistics,
// identify_mutations.cpp:3009-3033), by one wavefront.
// key_of, reads: the distinct keys and their reads, or (null) every one of the K list entries a key.
__device__ __noinline__ void stats_w(LdsShared* SS, const uint32_t* list, const uint32_t* key_of, const uint32_t* reads, int K,
                                     int Q, int major, int minor) {
  const int lane = threadIdx.x & 63;
  for (int i = lane; i < 256; i += 64) (&SS->qh[0][0])[i] = 0;
  wave_sync();
  uint32_t nx = 0, ny = 0;
  for (int i = lane; i < K; i += 64) {
    const uint32_t k = key_of ? key_of[i] : list[i];
    const uint32_t h = key_of ? reads[i] : 1u;
    const int ob = (int)((k % 10u) / 2u);
    const int q = (int)((k / 10u) % (uint32_t)Q);
    if (ob == major && q < 128) {
      __hip_atomic_fetch_add(&SS->qh[1][q], h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      ny += h;
    }
    if (ob == minor && q < 128) {
      __hip_atomic_fetch_add(&SS->qh[0][q], h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      nx += h;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    nx += __shfl_xor(nx, o, 64);
    ny += __shfl_xor(ny, o, 64);
  }
  wave_sync();
  const uint32_t mjt = (major < 5) ? SS->cov[major][2] : 0, mjb = (major < 5) ? SS->cov[major][0] : 0;
  const uint32_t mnt = (minor < 5) ? SS->cov[minor][2] : 0, mnb = (minor < 5) ? SS->cov[minor][0] : 0;
  const double fs = fisher_2x2_w(mnt, mnb, mjt, mjb, SS->fisher, nx + ny, ny, &SS->ks_log_total);
  wave_sync();
  const double ks = (nx > 0 && ny > 0) ? ks_less_w(SS, nx, ny, SS->ks_log_total) : 1.0;
  if (lane == 0) {
    SS->ks_p = ks;
    SS->fisher_p = fs;
  }
}

// Whether a value known within `rel` of itself prints as the reference's: %.*e with `places` digits, whose
// rounding boundary must not lie within the error.  A decade's end is no boundary: both sides of it
// print alike.
__device__ __noinline__ bool prints_surely_e(double v, int places, double rel) {
  if (v == 0.0) return true;
  if (!(v > 1e-280) || places > 12) return false;
  const double e = floor(log10(v));
  const double scaled = v * pow(10.0, (double)places - e);
  return fabs(scaled - floor(scaled) - 0.5) > rel * scaled;
}

// The same of a score known within `err`, printed with one decimal.
__device__ __forceinline__ bool prints_surely_f1(double v, double err) {
  const double scaled = 10.0 * fabs(v);
  return fabs(scaled - floor(scaled) - 0.5) > 10.0 * err;
}

// Whether the full fit's decisions (which alleles count, and their order) hold for any frequencies
// within `rel` of these, and the frequencies that are printed print alike.
__device__ __noinline__ bool fit_is_sure(const LdsDouble* f, uint32_t n, int places, double rel) {
  const double thr = 0.5 / (double)n;
  for (int a = 0; a < 5; a++) {
    if (f[a] < fmin(0.5 * thr, 0.01)) continue;
    if (fabs(f[a] - thr) <= 2.0 * rel * thr) return false;
    for (int b = 0; b < a; b++)
      if (fabs(f[a] - f[b]) <= 2.0 * rel * f[a]) return false;
    if (f[a] >= thr && !prints_surely_e(f[a], places, rel)) return false;
  }
  return true;
}

// The search of one bound (write_RA_frequency_bounds, identify_mutations.cpp:3175-3217), in
// registers of the lane that walks it.
struct Bound {
  double lo, hi, vlo, vhi;
  double out;       // the bound as reported so far
  int active;       // 0 ended, 1 between midpoints, 2 its end of the range is still to be compared
  int iter;
  // One comparison with the target: at the end of the range, which opens the search when the profile
  // there is below the target, or at the midpoint m of the interval.
  __device__ __forceinline__ void step(int side, bool ge, double m, double v, double tol, double fh) {
    if (active == 2) {
      active = (!ge && (hi - lo) > tol) ? 1 : 0;
      if (!ge) out = fh;
      return;
    }
    // lower bound: a profile >= target moves hi down; upper bound: it moves lo up
    const bool left = (side == 0) ? ge : !ge;   // the interval kept is [lo, m]
    if (left) {
      hi = m;
      vhi = v;
    } else {
      lo = m;
      vlo = v;
    }
    iter++;
    active = (iter < 40 && (hi - lo) > tol) ? 1 : 0;
    out = (side == 0) ? hi : lo;
  }
};

}  // namespace

// kKeysGlobal: the candidate's read list is this block's slice of a device scratch list (columns
// too deep for LDS), else it is in LDS.  The location is a compile-time choice, so that each
// instantiation's accesses to the list keep their address space (LDS instructions in the usual
// case); one pointer that may be either would make them all generic (flat) accesses.
template <bool kKeysGlobal>
__global__ void __launch_bounds__(kSW * 64) __attribute__((amdgpu_waves_per_eu(4))) k_score_candidates_t(ImParams P) {
  extern __shared__ __align__(16) unsigned char dyn[];
  uint32_t* list;   // the candidate's reads, in order: table keys, then rows
  size_t key_lds;
  if constexpr (kKeysGlobal) {
    list = P.key_scratch + (size_t)blockIdx.x * (size_t)P.key_cap;
    key_lds = 0;
  } else {
    list = (uint32_t*)dyn;
    key_lds = ((size_t)P.key_cap * sizeof(uint32_t) + 15) & ~(size_t)15;
  }
  // P.rows_cap rows (six doubles each), the same with the variant first (em_tasks), their two model
  // values, their keys and reads; before the rows are filled, the hash of the distinct keys lies in
  // their place (a key and its first read, then its row, per slot); where they don't fit, the model values of the
  // first pre_cap reads
  double* rows = (double*)(dyn + key_lds);
  double* prow = rows + (size_t)P.rows_cap * 6;
  double* pre = prow + (size_t)P.rows_cap * 6;
  uint32_t* key_of = (uint32_t*)(pre + (size_t)P.rows_cap * 2);
  uint32_t* row_reads = key_of + P.rows_cap;
  const int pre_cap = (int)((size_t)P.rows_cap * kScoreRowBytes / 16);
  constexpr bool kLG = kKeysGlobal;
  __shared__ ScoreShared SS;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int S = P.read_set_max, Q = P.quality_max;
  const double tol = P.precision_decimal;
  const int n_cand = min(*P.n_score, P.cand_cap);
  uint32_t err = 0;
  // Blocks take candidates from the pass's work counter, one at a time: a candidate's cost varies
  // several-fold, so a fixed stride over the grid would leave blocks idle while others work through a
  // run of costly candidates.
  __shared__ int s_next;
  for (;;) {
    if (tid == 0) s_next = atomicAdd(P.score_next, 1);
    __syncthreads();
    const int ci = __builtin_amdgcn_readfirstlane(s_next);
    __syncthreads();   // every wavefront has read s_next before the next draw overwrites it
    if (ci >= n_cand) break;
    // every index the candidate leads to is checked before it is used: a column inside the
    // sample, a window inside the index, a read range inside the alignments.  The values are read
    // as wave-uniform scalars, so the checks are uniform branches: a skip decided on per-lane
    // copies of the same value is a divergent branch to the compiler, and around the block's
    // barriers that has paired barriers across wavefronts wrongly (results read stale LDS).
    const int2 cd0 = P.score[ci];
    const int2 cd = make_int2(__builtin_amdgcn_readfirstlane(cd0.x), __builtin_amdgcn_readfirstlane(cd0.y));
    if (cd.x < 0 || cd.x >= P.n_pos || cd.y < 0) {
      err |= kErrIndex;
      continue;
    }
    const int p = cd.x, slot = cd.y;
    const int64_t w = p / 64;
    if (w >= P.n_windows) {
      err |= kErrIndex;
      continue;
    }
    const int rb = __builtin_amdgcn_readfirstlane(P.win_rb[w]), re = __builtin_amdgcn_readfirstlane(P.win_re[w]);
    if (rb < 0 || re < rb || re > P.n_reads) {
      err |= kErrIndex;
      continue;
    }
    if (tid < 18) SS.cov[tid / 3][tid % 3] = 0;
    if (tid == 0) {
      SS.n_keys = 0;
      SS.bad_r = 0;
      SS.unsure = 0;
      SS.best = -1;    // not computed yet
      SS.ks_p = 2.0;   // not computed yet
      SS.fisher_p = 1.0;
    }
    __syncthreads();
    // ---- pdata in file order (identify_mutations.cpp:1561-1657): order-preserving compaction
    for (int r0 = rb; r0 < re; r0 += kSW * 64) {
      const int r = r0 + tid;
      bool use = false;
      uint32_t key = 0;
      int obs = 0, strand_idx = 0;
      if (r < re) {
        const DRead R = P.reads[r];
        use = pdata_key(R, P.cigar, P.bases, P.quals, p, slot, S, Q, P.base_quality_cutoff, key, obs, strand_idx, err);
      }
      const unsigned long long mask = __ballot(use);
      if (lane == 0) SS.wcount[wave] = (uint32_t)__popcll(mask);
      __syncthreads();
      int base = SS.n_keys;
      for (int k = 0; k < wave; k++) base += (int)SS.wcount[k];
      if (use && key >= (uint32_t)P.tab_keys) {
        err |= kErrIndex;   // a key outside the likelihood tables: counted, never looked up
        key = 0;
      }
      if (use) {
        const int idx = base + __popcll(mask & ((1ull << lane) - 1ull));
        if (idx < P.key_cap) list[idx] = key;
        else err |= kErrCapacity;
        atomicAdd(&SS.cov[obs][strand_idx], 1u);
      }
      __syncthreads();
      if (tid == 0) {
        int tot = 0;
        for (int k = 0; k < kSW; k++) tot += (int)SS.wcount[k];
        SS.n_keys += tot;
      }
      __syncthreads();
    }
    const int n = __builtin_amdgcn_readfirstlane(min(SS.n_keys, P.key_cap));
    if (tid < 5) SS.obs[tid] = SS.cov[tid][0] + SS.cov[tid][2];
    // ---- the distinct keys, numbered in the order of their first reads, through a hash of the keys
    int K = n;
    bool dedup = true;
    {
      // half full at most, unless the rows' LDS holds fewer slots
      const int slots = min(1 << (32 - __clz(max(2 * n, 512) - 1)), 1 << (31 - __clz(P.rows_cap * 12)));
      const int shift = __clz(slots) + 1;
      uint32_t *hkey = (uint32_t*)rows, *hrow = hkey + slots;
#pragma unroll 1
      for (int i = tid; i < slots; i += kSW * 64) hkey[i] = hrow[i] = kNoKey;
      if (tid == 0) SS.crowded = 0;
      __syncthreads();
      // the slot of a key: its own, or the next free one (atomics only where a look does not settle it: most
      // reads of a deep column share a few keys)
      auto slot_of = [&](uint32_t key, bool insert) {
        uint32_t at = (key * 0x9E3779B1u) >> shift;
#pragma unroll 1
        for (int probe = 0; probe < kScoreProbes; probe++) {
          uint32_t old = hkey[at];
          if (insert && old == kNoKey) {
            old = atomicCAS(&hkey[at], kNoKey, key);
            if (old == kNoKey) return at;
          }
          if (old == key) return at;
          at = (at + 1u) & (uint32_t)(slots - 1);
        }
        return kNoKey;
      };
#pragma unroll 1
      for (int i = tid; i < n; i += kSW * 64) {
        const uint32_t at = slot_of(list[i], true);
        if (at == kNoKey) SS.crowded = 1;
        else if (hrow[at] > (uint32_t)i) atomicMin(&hrow[at], (uint32_t)i);
      }
      __syncthreads();
      dedup = uniform_i(SS.crowded) == 0;
      if (dedup) {
        // a key's row: how many first reads come before its own.  (A slot whose row is already there holds
        // less than any read still to be looked at.)
        K = 0;
#pragma unroll 1
        for (int i0 = 0; i0 < n; i0 += kSW * 64) {
          const int i = i0 + tid;
          const uint32_t at = (i < n) ? slot_of(list[i], false) : kNoKey;
          const bool first = at != kNoKey && hrow[at] == (uint32_t)i;
          const unsigned long long m = __ballot(first);
          if (lane == 0) SS.wcount[wave] = (uint32_t)__popcll(m);
          __syncthreads();
          int row = K + __popcll(m & ((1ull << lane) - 1ull));
          for (int k = 0; k < kSW; k++) {
            if (k < wave) row += (int)SS.wcount[k];
            K += (int)SS.wcount[k];
          }
          if (first) {
            hrow[at] = (uint32_t)row;
            if (row < P.rows_cap) {
              key_of[row] = list[i];
              row_reads[row] = 0;
            }
          }
          __syncthreads();
        }
        K = uniform_i(K);
        dedup = K <= P.rows_cap;
      }
      if (dedup)
#pragma unroll 1
        for (int i = tid; i < n; i += kSW * 64) {
          const uint32_t row = hrow[slot_of(list[i], false)];
          list[i] = row;
          atomicAdd(&row_reads[row], 1u);
        }
    }
    const int kind = (dedup || n <= P.rows_cap) ? kRowsLds : kRowsGlobal;
    if (!dedup) {
      K = n;
      if (kind == kRowsLds)
        for (int i = tid; i < n; i += kSW * 64) {
          key_of[i] = list[i];
          row_reads[i] = 1u;
          list[i] = (uint32_t)i;
        }
    }
    __syncthreads();
    bool bad_r = false;
    const int n_check = K * 6;   // (every read a row of its own where the rows are not in LDS)
#pragma unroll 1
    for (int i = tid; i < n_check; i += kSW * 64) {
      const double r = P.tab_r[(size_t)(kind == kRowsLds ? key_of[i / 6] : list[i / 6]) * 6 + i % 6];
      if (kind == kRowsLds) rows[i] = r;
      bad_r = bad_r || (i % 6 != 5 && r != 0.0 && !(r >= 0x1p-100 && r <= 2.0));
    }
    if (bad_r) SS.bad_r = 1;
    const Rows RR{list, rows, row_reads, P.tab_r};
    const uint32_t* keys = (kind == kRowsLds) ? key_of : nullptr;
    auto fit_exact = [&](int mode, int v, double x) {
      return kind == kRowsLds ? em_exact<kRowsLds, kLG>(RR, n, mode, v, x, (LdsDouble*)SS.fit, tol, SS.bad_r)
                              : em_exact<kRowsGlobal, kLG>(RR, n, mode, v, x, (LdsDouble*)SS.fit, tol, SS.bad_r);
    };
    const char refc = (slot == 0) ? P.ref[p] : '.';
    const int ref_idx = char_index(refc) < 0 ? 5 : char_index(refc);
    __syncthreads();
    // ---- the candidate, with sums in any order; then, when a decision or a printed digit lies too
    // close to its boundary (or every candidate is to be exact), once more with the reference's sums
    int major = 5, minor = 5, variant = 5;
    bool have_v = false;
    const double nu = ((double)n + kSumSlack) * kHalfUlp;
    // level 0: sums in any order; 1: the full fit and close comparisons with the reference's sums; 2: the
    // score's likelihoods too
    int level = P.screen_off ? 2 : 0;
    for (;;) {
      const bool in_order = level > 0;
      if (wave == 0) {
        // full fit, from 0.5 + one per observing read, normalized (identical values from every lane)
        double f[5], total = 0.0;
#pragma unroll
        for (int b = 0; b < 5; b++) {
          f[b] = 0.5 + (double)SS.obs[b];
          total += f[b];
        }
#pragma unroll
        for (int b = 0; b < 5; b++) SS.fit[b] = (n > 0) ? f[b] / total : 0.0;
        wave_sync();
        double ll = 0.0;
        bool unsure = false;
        if (n > 0) {
          if (in_order) {
            ll = fit_exact(1, -1, 0.0);
          } else {
            ll = kind == kRowsLds ? em_full<kRowsLds, kLG>(RR, K, n, (LdsDouble*)SS.fit, tol, nu)
                                  : em_full<kRowsGlobal, kLG>(RR, K, n, (LdsDouble*)SS.fit, tol, nu);
            unsure = !(fabs(ll) < 1e300);
          }
        }
        wave_sync();
        if (lane < 5) SS.full_f[lane] = SS.fit[lane];
        if (lane == 0) {
          if (level != 1) SS.full_ll = ll;   // level 1 keeps the value that goes with the null task's
          SS.unsure = unsure ? 2 : 0;
        }
      } else if (wave == 1 && (level == 0 || SS.best < 0)) {
        double lps[5];
        genotype_sums<kLG>(list, keys, P.tab_lp, n, lps);
        int best;
        double gscore;
        pure_genotype_call(lps, (uint32_t)n, &best, &gscore);
        if (lane == 0) {
          SS.best = best;
          SS.gscore = gscore;
          SS.lp_best = (n > 0) ? lps[best] : 0.0;
        }
      }
      __syncthreads();
      // every thread derives the same calls from the shared results
      bool cons;
      {
        double full_f[5];
        for (int b = 0; b < 5; b++) full_f[b] = SS.full_f[b];
        const double cbs = SS.gscore - P.log10_ref_length;
        cons = (SS.best != ref_idx) && !isnan(cbs) && (cbs > 0.0);
        major = uniform_i(major_index(full_f, (uint32_t)n));
        minor = uniform_i(next_index(full_f, (uint32_t)n, major));
        variant = uniform_i(next_index(full_f, (uint32_t)n, ref_idx));
      }
      have_v = variant != 5 && n > 0;
      const double fh = have_v ? SS.full_f[variant] : 0.0;
      double other = 0.0;   // the other alleles' share of the full fit
#pragma unroll
      for (int b = 0; b < 5; b++)
        if (b != variant) other += SS.full_f[b];
      if (have_v && kind == kRowsLds) {
        for (int i = tid; i < K; i += kSW * 64) {
          double r[6], t = 0.0;
          RR.row<kRowsLds>(i, r);
          int at = 1;
#pragma unroll
          for (int b = 0; b < 5; b++) {
            const bool mine = b == variant;
            prow[6 * i + (mine ? 0 : at)] = r[b];
            if (!mine) {
              t = fma((other > 0.0) ? SS.full_f[b] / other : 0.25, r[b], t);
              at++;
            }
          }
          prow[6 * i + 5] = (double)row_reads[i];
          pre[2 * i] = rows[6 * i + variant] - t;
          pre[2 * i + 1] = t;
        }
      } else if (have_v) {
        for (int i = tid; i < min(n, pre_cap); i += kSW * 64) {
          double r[6], t = 0.0, rv = 0.0;
          RR.row<kRowsGlobal>((int)list[i], r);
#pragma unroll
          for (int b = 0; b < 5; b++) {
            if (b == variant) rv = r[b];
            else t = fma((other > 0.0) ? SS.full_f[b] / other : 0.25, r[b], t);
          }
          rows[2 * i] = rv - t;
          rows[2 * i + 1] = t;
        }
      }
      if (tid == 0) {
        SS.done = 0;
        SS.emitted = 0;
        SS.exact = SS.exact_have = 0;
        SS.active[0] = SS.active[1] = 0;
        SS.depth[0] = SS.depth[1] = 0;
        SS.out[0] = 0.0;
        SS.out[1] = 1.0;
        if (level == 0) SS.guard_rel = fmax(P.guard_rel, (2.0 + 0.125 * SS.fit[5]) * nu);
        SS.guard_log = fmax(P.guard_log, nu * ((double)n + fabs(SS.lp_best)));
        if (!in_order && n > 0 && SS.unsure == 0 &&
            !fit_is_sure((LdsDouble*)SS.full_f, (uint32_t)n, P.places, SS.guard_rel))
          SS.unsure = 1;
      }
      __syncthreads();
      // ---- rounds: the null fit, the profiles at the ML frequency, 0 and 1 and the bounds' midpoints |
      // KS and Fisher; then more midpoints.  Nothing of an unsure fit is worth going on with.
      const bool go = uniform_i(SS.unsure) == 0;
      for (int round = 0; go; round++) {
        const int exact = uniform_i(SS.exact);
        const bool search = round == 0 || SS.active[0] || SS.active[1];
        if (have_v && wave == kTaskWaves && (exact || (level == 2 && round == 0))) {
          // the null fit, or both sides of a comparison too close for the tasks' values
          if (exact) {
            for (int part = SS.exact_have ? 1 : 0; part < 2; part++) {
              const double x = part ? SS.exact_x[exact - 1] : fh;
#pragma unroll
              for (int b = 0; b < 5; b++)
                SS.fit[b] = (b == variant) ? x : (other > 0.0) ? (1.0 - x) * SS.full_f[b] / other : (1.0 - x) / 4.0;
              wave_sync();
              const double ll = fit_exact(2, variant, x);
              wave_sync();
              if (lane == 0) {
                if (part) SS.exact_v = ll;
                else SS.exact_target = ll - kDrop;
              }
            }
          } else {
            double f[5], total = 0.0;
#pragma unroll
            for (int b = 0; b < 5; b++) {
              f[b] = (b == variant) ? 0.0 : 0.5 + (double)SS.obs[b];
              total += f[b];
            }
#pragma unroll
            for (int b = 0; b < 5; b++) SS.fit[b] = f[b] / total;
            wave_sync();
            const double ll = fit_exact(1, variant, 0.0);
            if (lane == 0) SS.null_ll = ll;
          }
        }
        if (!exact) {
          if (wave == kTaskWaves) {
            // annotate_polymorphism_statistics (identify_mutations.cpp:3009-3033); used if emitted
            if (round == 0 && n > 0 && !(in_order && SS.ks_p != 2.0))
              stats_w((LdsShared*)&SS, list, keys, row_reads, K, Q, major, minor);
          } else if (have_v && search) {
            // task slots of the round.  Round 0: the profiles at the ML frequency, 0 and 1 and the null
            // fit, then the first path of each bound that may be searched.  Later: per open bound
            // the first levels of the full tree, whatever the prediction, then a path.  A bound needs
            // 20 levels at most for its 1e-6; with one open, 24 tasks of eight lanes hold them.
            const int s0 = (round == 0) ? 4 : 0;
            const bool open0 = (round == 0) ? fh > tol : SS.active[0] != 0;
            const bool open1 = (round == 0) ? (1.0 - fh) > tol : SS.active[1] != 0;
            const bool both = open0 && open1;
            const int shift = both ? 2 : 3;   // lanes per task: 4 or 8
            const int share = both ? (kTaskSlots - s0) / 2 : kTaskSlots / 2 - s0;
            const int n_tree = (round == 0) ? 0 : 7;
            const int side_l = lane >> 5;
            const double lo_l = (round == 0) ? (side_l ? fh : 0.0) : SS.lo[side_l];
            const double hi_l = (round == 0) ? (side_l ? 1.0 : fh) : SS.hi[side_l];
            const LdsDouble *pr = (const LdsDouble*)prow, *pm = (const LdsDouble*)pre;
            const double root =
                kind == kRowsLds ? model_root<false>(pr, pm, K, lo_l, hi_l, round > 0, SS.vlo[side_l], SS.vhi[side_l], SS.target)
                                 : model_root<true>(nullptr, (const LdsDouble*)rows, min(n, pre_cap), lo_l, hi_l, round > 0,
                                                    SS.vlo[side_l], SS.vhi[side_l], SS.target);
            const double root0 = readlane_d(root, 0), root1 = readlane_d(root, 32);
            const int slot_i = (wave * 64 + lane) >> shift;
            const bool first = (lane & ((1 << shift) - 1)) == 0;
            double x = 0.0;
            bool active = false;
            const bool null_task = round == 0 && slot_i == 3;
            if (slot_i < s0) {
              x = (slot_i == 0) ? fh : (slot_i == 2) ? 1.0 : 0.0;
              active = !(null_task && level == 2);
            } else {
              const int side = (open0 && slot_i - s0 < share) ? 0 : 1;
              const int rel = slot_i - s0 - ((open0 && side == 1) ? share : 0);
              if (rel < share && (side ? open1 : open0)) {
                double a = (round == 0) ? (side ? fh : 0.0) : SS.lo[side], b = (round == 0) ? (side ? 1.0 : fh) : SS.hi[side];
                const int it0 = (round == 0) ? 0 : SS.iter[side];
                const double fs = side ? root1 : root0;
                // a tree node's turns are the bits of its breadth-first number below the leading one,
                // a path's those of the prediction
                const bool tree = rel < n_tree;
                const int node = rel + 1;
                const int deep = tree ? 31 - __clz(node) : rel - n_tree;
                double m = 0.5 * (a + b);
                active = true;
                for (int d = 0; d < deep; d++) {
                  const bool left = tree ? !((node >> (deep - 1 - d)) & 1) : (side == 0) ? (fs <= m) : (fs < m);
                  if (left) b = m;
                  else a = m;
                  if (!(it0 + d + 1 < 40 && (b - a) > tol)) active = false;
                  m = 0.5 * (a + b);
                }
                x = m;
                if (first) SS.pts[side][rel] = active ? m : -1.0;
              }
            }
            if (tid == 0) {
              SS.n_tree = n_tree;
              for (int side = 0; side < 2; side++) {
                SS.depth[side] = (side ? open1 : open0) ? share : 0;
                SS.slot0[side] = s0 + ((side == 1 && open0) ? share : 0);
              }
            }
            if (__any(active)) {
              // the other alleles' starting frequencies, in order
              double st[4], total = 0.0;
              int at = 0;
#pragma unroll
              for (int b = 0; b < 5; b++) total += (b == variant) ? 0.0 : 0.5 + (double)SS.obs[b];
#pragma unroll
              for (int q = 0; q < 4; q++) {
                at = q + (q >= variant ? 1 : 0);
                st[q] = null_task ? (0.5 + (double)SS.obs[at]) / total
                                  : (other > 0.0) ? (1.0 - x) * SS.full_f[at] / other : (1.0 - x) / 4.0;
              }
              const double sc = null_task ? 1.0 / (double)n : 0.0;
              const double passes = (level == 0 ? SS.fit[5] : 0.0) + 1.0;
              auto tasks_over = [&](auto src) {
                typedef decltype(src) Src;
                return both ? em_tasks<4, Src>(src, K, x, st[0], st[1], st[2], st[3], sc, active, tol, nu, passes)
                            : em_tasks<8, Src>(src, K, x, st[0], st[1], st[2], st[3], sc, active, tol, nu, passes);
              };
              const TaskValue val = kind == kRowsLds ? tasks_over(TaskRowsLds{pr})
                                                     : tasks_over(TaskRowsGlobal<kLG>{list, P.tab_r, variant});
              if (first && active) {
                (null_task ? SS.null_ll : SS.val[slot_i]) = val.ll;
                (null_task ? SS.null_more : SS.more[slot_i]) = val.more;
              }
            }
          }
        }
        __syncthreads();
        if (wave == 0) {
          // lanes 0 and 32 walk the lower and the upper bound side by side
          const int side = lane >> 5;
          const bool walker = (lane & 31) == 0;
          bool close = false;   // a comparison the tasks' values do not decide
          const double guard = P.screen_off ? INFINITY : SS.guard_log;
          Bound B;
          if (round == 0) {
            // (used if emitted)
            B.lo = side ? fh : 0.0;
            B.hi = side ? 1.0 : fh;
            B.vlo = side ? SS.val[0] : SS.val[1];
            B.vhi = side ? SS.val[2] : SS.val[0];
            B.out = side ? 1.0 : 0.0;
            B.iter = 0;
            B.active = have_v ? 2 : 0;
          } else {
            B.lo = SS.lo[side];
            B.hi = SS.hi[side];
            B.vlo = SS.vlo[side];
            B.vhi = SS.vhi[side];
            B.out = SS.out[side];
            B.iter = SS.iter[side];
            B.active = SS.active[side];
          }
          const double target = (round == 0) ? SS.val[0] - kDrop : SS.target;
          const double target_more = (round == 0) ? SS.more[0] : SS.target_more;
          const double end_more = (round == 0) ? SS.more[side ? 2 : 1] : SS.end_more[side];
          const int n_tree = SS.n_tree, slot0 = SS.slot0[side];
          if (exact == 1 + side) {
            // the exact comparison decides this side's end of the range, or its midpoint.  (The values
            // are within the guard of the target; the exact ones hold the lpmax sum.)
            B.step(side, SS.exact_v >= SS.exact_target, SS.exact_x[side], target, tol, fh);
          }
          if (walker && (!exact || P.screen_off) && B.active) {
            const int depth = exact ? 0 : SS.depth[side];
            if (B.active == 2) {
              const double v = side ? B.vhi : B.vlo;
              close = !(fabs(v - target) > guard + end_more + target_more);
              if (!close) B.step(side, v >= target, 0.0, v, tol, fh);
            }
            // down the evaluated levels: every level is one sequential bisection step (the interval
            // halved at 0.5 * (lo + hi), 40 steps at most, until it is no wider than tol)
            int node = 0;
            for (int level = 0; B.active == 1 && !close; level++) {
              // a tree's node is the sequential midpoint by construction; a path's only while every
              // earlier decision followed the path (off it, the interval and so its midpoint differ)
              const int k = node < n_tree ? node : n_tree + level;
              if (k >= depth) break;
              const double m = 0.5 * (B.lo + B.hi), at = SS.pts[side][k], v = SS.val[slot0 + k];
              if (m != at) break;
              close = !(fabs(v - target) > guard + SS.more[slot0 + k] + target_more);
              if (close) break;
              const bool ge = v >= target;
              B.step(side, ge, m, v, tol, fh);
              node = 2 * node + (((side == 0) ? ge : !ge) ? 1 : 2);
            }
            if (B.active == 1 && P.screen_off) close = true;   // every step exactly
          }
          // neither end of the search may hang on the last bits of the ML frequency
          const double width = B.hi - B.lo;
          const double bits = fmax(1e-11, 4.0 * SS.guard_rel);
          if (!in_order && (fabs(width - tol) < bits || fabs(2.0 * width - tol) < bits)) close = true;
          if (walker) {
            SS.lo[side] = B.lo;
            SS.hi[side] = B.hi;
            SS.vlo[side] = B.vlo;
            SS.vhi[side] = B.vhi;
            SS.out[side] = B.out;
            SS.iter[side] = B.iter;
            SS.active[side] = B.active;
            SS.end_more[side] = end_more;
            SS.exact_x[side] = (B.active == 2) ? (side ? 1.0 : 0.0) : 0.5 * (B.lo + B.hi);
          }
          const unsigned long long u = __ballot(walker && close), open = __ballot(walker && B.active != 0);
          const double out0 = readlane_d(B.out, 0), out1 = readlane_d(B.out, 32);
          if (lane == 0) {
            SS.target = target;
            SS.target_more = target_more;
            if (exact) SS.exact_have = 1;
            SS.exact = (in_order && u) ? ((u & 1ull) ? 1 : 2) : 0;
            // emitted: a consensus call, or a presence score at the cutoff
            const double score = (SS.full_ll - SS.null_ll) - P.log10_ref_length;
            const bool emitted = cons || (have_v && score >= P.polymorphism_cutoff);
            SS.emitted = emitted ? 1 : 0;
            SS.done = (!emitted || !have_v || !open) ? 1 : 0;
            int unsure = 0;
            if (level < 2 && have_v) {
              const double err = SS.guard_log + nu * fabs(score) + SS.null_more;
              if (!(fabs(score - P.polymorphism_cutoff) > err) || (emitted && !prints_surely_f1(score, err))) unsure = 2;
            }
            if (level == 0 && have_v && emitted && unsure == 0) {
              if (u) unsure = 1;
              if (SS.done && !(prints_surely_e(out0, P.places, SS.guard_rel) &&
                                (out1 == 1.0 || prints_surely_e(out1, P.places, SS.guard_rel))))
                unsure = 1;
            }
            SS.unsure = unsure;
            if (unsure) SS.done = 1;
          }
        }
        __syncthreads();
        if (SS.done) break;
      }
      const int unsure = uniform_i(SS.unsure);
      if (level == 2 || unsure == 0) break;
      level = max(level + 1, unsure);
      __syncthreads();   // every wavefront has read the verdict before it is cleared
    }
    if (tid == 0) {
      RaOut out;
      const bool emitted = SS.emitted != 0;
      out.gpos = p;
      out.slot = slot;
      out.emitted = emitted ? 1 : 0;
      out.ref_idx = (uint8_t)ref_idx;
      out.major = (uint8_t)major;
      out.minor = (uint8_t)minor;
      out.variant = (uint8_t)variant;
      out.pad[0] = out.pad[1] = out.pad[2] = 0;
      out.n = (uint32_t)n;
      for (int b = 0; b < 5; b++) out.f[b] = SS.full_f[b];
      out.variant_score = have_v ? (SS.full_ll - SS.null_ll) - P.log10_ref_length : __longlong_as_double(0x7ff8000000000000LL);
      out.lower = emitted ? SS.out[0] : 0.0;
      out.upper = emitted ? SS.out[1] : 1.0;
      out.ks_p = (emitted && n > 0) ? SS.ks_p : 1.0;
      out.fisher_p = (emitted && n > 0) ? SS.fisher_p : 1.0;
      int tt = 0, tb = 0;
      for (int b = 0; b < 5; b++) {
        out.cov[b][0] = SS.cov[b][2];
        out.cov[b][1] = SS.cov[b][0];
        tt += (int)SS.cov[b][2];
        tb += (int)SS.cov[b][0];
      }
      out.total_top = tt;
      out.total_bot = tb;
      P.ra_out[ci] = out;
      atomicAdd(&P.n_level[level], 1);
    }
    __syncthreads();
  }
  if (err) atomicOr(P.err, err);
}

template __global__ void k_score_candidates_t<false>(ImParams P);
template __global__ void k_score_candidates_t<true>(ImParams P);

}  // namespace bsq
