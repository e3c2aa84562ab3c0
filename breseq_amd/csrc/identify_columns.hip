// identify_columns.hip -- pass 2, insert slot 0 of every reference column, on CDNA4 (gfx950):
// coverage tallies, the per-genotype log10 likelihood sums, the pure-genotype call and a
// conservative screen that routes columns to the exact FP64 scorer
// (identify_mutations_pileup::pileup_callback, identify_mutations.cpp:1561-1821).
//
// One 64-wide wavefront owns a window of 64 consecutive columns.  The unique single-run alignments
// whose bytes are all legal (kIdPlain) go first, eight at a time: eight lanes per alignment, eight
// columns per lane.  Their positions' classes, ranges and counts are byte-wise operations on whole words
// (v_perm_b32 lookups, shifted masks of bit 7), so only the table row of a position and its six sums are
// per-position work; the rare observations other than the reference base go to LDS sums.  The eight
// groups' sums then meet in one lane per column, and the other alignments follow one at a time, lane =
// column, in file order, so the FP64 1/X1 sums keep the read order.
//
// The likelihood sums are FP32 (a 24-byte table row per read); the column's predicted and consensus
// decisions are certified against an explicit bound on the difference to the reference's FP64 sums,
// which holds for any order of the sums, and the rare columns within that bound of a threshold are
// decided by k_fix_columns from exact FP64 sums in read order.  Coverage counts are integers and the
// 1/X1 redundancy sums stay FP64 in read order, so those outputs are the reference's exactly.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device_common.h"
#include "kernels.h"

namespace bsq {

namespace {

constexpr int kWaveCols = 64;

__device__ __forceinline__ uint32_t rdlane(uint32_t v, int j) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, j);
}

// BAM 4-bit base code -> A0 C1 G2 T3; every other code -> 15.
__device__ __forceinline__ uint32_t base_idx4(uint32_t b) {
  const uint32_t i = (uint32_t)(0xFFFFFFF3FFF2F10FULL >> ((b & 15u) * 4u)) & 15u;
  return b > 15u ? 15u : i;
}

// Screening sums of one column (FP32).  Only observations other than the reference base update the
// per-class sums; the reference class follows from n.
struct Screen {
  uint32_t n;          // reads with a likelihood term
  uint32_t cnt[5];     // per observed class, reference class excluded
  float SL;            // Sum_i max_b log10 P_i(b)
  float G[5];          // per observed class v: Sum (log10 P_i(reference) - log10 P_i(v))
  float Gabs;          // Sum |terms of G| (rounding bound)
};

// What one alignment contributes to one lane's column at insert slot 0.
struct Entry {
  bool cover;          // the alignment has a pileup entry at this column
  bool is_del;
  int qpos;            // clamped into the read when !cover
  int ondel;           // -1 deletion, else max(indel, 0)
  uint32_t b, q;       // base code and quality at qpos (b = '.' for deletions)
  uint32_t qd;         // deletions: quality of the next read base in read direction
  bool del_ok;         // deletions: that base exists and is not N
  bool del_oob;        // deletions: that base lies outside the read (an error if the entry is used)
  bool trimmed;        // is_trimmed at slot 0 (alignment.h:389-410)
};

// The likelihood table as the kernel addresses it, in bytes: the rows of quality q of a (MAPQ, read
// file) block from (q + 1) * kStride on, those of class o 32 * o further.  The rows before quality 0
// are zeros, the rows of a read that adds nothing.  In LDS a row keeps its 24 bytes of values and the
// stride is 38 words, so that qualities spread over the banks.
constexpr uint32_t kFoldStride = 5 * sizeof(FoldRow), kFoldLdsStride = 152;
static_assert(kFoldLdsStride >= 4 * sizeof(FoldRow) + 24, "class 4's row ends before the next quality's first");

template <bool kLds>
struct Table {
  // `at` of a row: its byte in the table in memory, or its LDS address (base is added by the caller,
  // once per alignment)
  const unsigned char* p;
  uint32_t base;
  static constexpr uint32_t kStride = kLds ? kFoldLdsStride : kFoldStride;
  __device__ __forceinline__ float at(uint32_t off) const {
    if constexpr (kLds) {
      typedef __attribute__((address_space(3))) const float LdsFloat;
      return *(LdsFloat*)off;
    } else {
      return *(const float*)(p + off);
    }
  }
  __device__ __forceinline__ void row(uint32_t off, float t[6]) const {
    typedef float Pair __attribute__((ext_vector_type(2)));
    Pair v[3];
    if constexpr (kLds) {
      typedef __attribute__((address_space(3))) const Pair LdsPair;
      const LdsPair* r = (LdsPair*)off;
      v[0] = r[0];
      v[1] = r[1];
      v[2] = r[2];
    } else {
      typedef float Four __attribute__((ext_vector_type(4)));
      const Four a = *(const Four*)(p + off);
      v[0] = a.xy;
      v[1] = a.zw;
      v[2] = *(const Pair*)(p + off + 16);
    }
    t[0] = v[0].x;
    t[1] = v[0].y;
    t[2] = v[1].x;
    t[3] = v[1].y;
    t[4] = v[2].x;
    t[5] = v[2].y;
  }
};

}  // namespace

// Screen (identify_mutations.cpp:3240-3344 bounded from above): true unless no allele v can reach
// the presence-score cutoff.
//   * The full model's log likelihood is at most Sum_i max_b log10 P_i(b) = SL.
//   * The null model (v held out) starts EM from Laplace-smoothed counts f0 and EM never lowers the
//     likelihood, so its value is at least the likelihood at f0, which per read is at least
//     log10 f0(c) + log10 P_i(c) for any held-in class c: the read's own class, or the reference
//     class for reads that observe v.  Summed: Sum_{b!=v} cnt_b log10 f0_b + cnt_v log10 f0_ref
//     + D + G[v], where D = Sum_i log10 P_i(observed class) = lps[ref] - Sum_u G[u].
// The FP32 rounding of every sum is bounded explicitly and added to the margin.  Columns whose
// reference base is N go to the exact scorer whenever they have reads.
__device__ __forceinline__ bool screen_passes(const Screen& A, const float lps[5], int ref_idx, double log10_ref_len,
                                              double cutoff, double margin) {
  if (A.n == 0) return false;
  if (ref_idx < 0 || ref_idx > 4) return true;
  // class counts; the reference class is what the other classes leave of n
  float cnt[5], Lb[5];
  uint32_t others = 0;
#pragma unroll
  for (int b = 0; b < 5; b++) others += (b == ref_idx) ? 0u : A.cnt[b];
  float sumL = 0.0f, magL = 0.0f, Lref = 0.0f, lref = 0.0f, sumG = 0.0f;
#pragma unroll
  for (int b = 0; b < 5; b++) {
    cnt[b] = (float)((b == ref_idx) ? A.n - others : A.cnt[b]);
    // log10 f0_b = log10(0.5 + cnt_b) - log10(init_total)
    Lb[b] = log10f(0.5f + cnt[b]);
    sumL += cnt[b] * Lb[b];
    magL += cnt[b] * fabsf(Lb[b]);
    if (b == ref_idx) Lref = Lb[b];
    if (b == ref_idx) lref = lps[b];
    sumG += A.G[b];
  }
  const float n = (float)A.n;
  const float u = 5.9604645e-08f;   // 2^-24
  const float D = lref - sumG;
  const float mag0 = fabsf(A.SL) + fabsf(lref) + 2.0f * A.Gabs + magL;
#pragma unroll
  for (int v = 0; v < 5; v++) {
    if (v == ref_idx) continue;
    const float Li = log10f(2.0f + (n - cnt[v]));
    // Sum_{b!=v} cnt_b log10 f0_b + cnt_v log10 f0_ref, regrouped
    const float lb = D + A.G[v] + (sumL - cnt[v] * Lb[v]) + cnt[v] * Lref - n * Li;
    const float mag = mag0 + n * fabsf(Li) + cnt[v] * (fabsf(Lb[v]) + fabsf(Lref));
    // every FP32 term carries at most (n + 16) u of relative error through its sums, the
    // conversions from FP64 and log10f; doubled for safety
    const double bound = 2.0 * (double)(n + 16.0f) * (double)u * (double)mag;
    const double ub = (double)A.SL - (double)lb - log10_ref_len;
    if (ub >= cutoff - margin - bound) return true;
  }
  return false;
}

// Entry of alignment R at column p for the general (non-simple) CIGAR path; loads issued here.
__device__ __forceinline__ void prepare_general(const ImParams& P, const DRead& R, int p, Entry& e, uint32_t& err) {
  int qpos = 0, indel = 0;
  bool is_del = false;
  e.cover = entry_at(R, P.cigar, p, qpos, indel, is_del, err);
  e.is_del = e.cover && is_del;
  e.ondel = is_del ? -1 : (indel < 0 ? 0 : indel);
  e.qpos = e.cover ? qpos : 0;
  const uint8_t* sq = P.bases + R.seq_off;
  const uint8_t* ql = P.quals + R.seq_off;
  e.b = '.';
  e.q = 0;
  e.qd = 0;
  e.del_ok = false;
  e.del_oob = false;
  e.trimmed = is_trimmed(R, e.qpos, e.ondel < 0);
  if (e.cover && !is_del) {
    e.b = sq[e.qpos];
    e.q = ql[e.qpos];
  } else if (e.is_del) {
    // deletion: quality of the next read base in read direction (error_count.cpp:1075-1080)
    const int rev = (R.flags & kReadReversed) ? 1 : 0;
    const int qq = qpos + 1 - rev;
    if (qq < 0 || qq >= (int)R.l_qseq) {
      // reported only if the entry is used: breseq skips redundant and trimmed reads before it
      // looks at this base (identify_mutations.cpp:1591-1626)
      e.del_oob = true;
    } else if (sq[qq] != 15) {
      e.qd = ql[qq];
      e.del_ok = true;
    }
  }
}

// The per-call alignment view of the column pass (thread per alignment).
__global__ void __launch_bounds__(256) k_prep_reads(const DRead* reads, const uint8_t* byte_max, int64_t n, int32_t S,
                                                    int32_t Q, IdRec* out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const DRead R = reads[i];
    IdRec c;
    c.gpos = R.gpos;
    c.gend = R.gend;
    c.seq_off = (uint32_t)(uint64_t)R.seq_off;
    c.qoff = (int32_t)R.y0 - R.gpos;
    // q1 = qpos + 1 <= XL  <=>  qpos < XL;  l_qseq - q1 + 1 <= XR  <=>  qpos >= l_qseq - XR.
    // Query positions are below 65535, so 0xFFFF stands for "no right trim".
    const uint32_t lo = (R.xl >= 0) ? (uint32_t)R.xl : 0u;
    const uint32_t hi = (R.xr >= 0) ? (uint32_t)max(0, (int32_t)R.l_qseq - (int32_t)R.xr) : 0xFFFFu;
    c.trim = lo | (hi << 16);
    const bool file_ok = (int)R.rfile < S;
    c.row_block = file_ok ? (uint32_t)R.mslot * (uint32_t)S + R.rfile : 0xffffffffu;
    // the word-wise path takes qualities below 128 and needs no check of a position's bytes
    const bool plain = (R.flags & kReadSimple) && R.x1 == 1 && file_ok && Q <= 128 && (int)byte_max[i] < Q;
    c.x1_flags = (uint32_t)R.x1 | ((uint32_t)R.flags << 16) | (plain ? kIdPlain : 0u);
    c.pad = 0;
    out[i] = c;
  }
}

// Certified pure_genotype_call (identify_mutations.cpp:3398-3433) from FP32 sums.
//   * Each FP32 sum lps[b] adds n terms of one sign, each rounded once from FP64, in n - 1 rounded
//     additions: with u = 2^-24 and g = (n + 2) u it is within g / (1 - g) |lps[b]| of the exact sum
//     (the recursive-summation bound gamma_n = n u / (1 - n u), with two more u for the term
//     roundings and the reference's own FP64 summation error).  E is the largest such bound; a
//     column so deep that g reaches 1/2 is never certified.
//   * The reference's best is certain when the top sum leads the next by more than 2E.
//   * Its score lps[best] - log10 Sum_{b != best} 10^lps[b] moves by at most 2E when every sum moves
//     by at most E; here each 10^d (d <= 0) is evaluated from (float)d, adding at most 3e-6 (terms
//     below 10^-38 of the total underflow, which changes the total by less than that).
// A decision within 2E + kScoreSlack of its threshold is left to k_fix_columns, which recomputes
// the column's sums exactly in read order.
constexpr double kScoreSlack = 1e-4;

__device__ __forceinline__ double genotype_score_approx(const float lps[5], int best) {
  float off = -3.4028235e38f;
#pragma unroll
  for (int b = 0; b < 5; b++)
    if (b != best) off = fmaxf(off, lps[b]);
  float tot = 0.0f;
#pragma unroll
  for (int b = 0; b < 5; b++)
    if (b != best) tot += exp10f((float)((double)lps[b] - (double)off));
  return ((double)lps[best] - (double)off) - (double)log10f(tot);
}

// A mask of lanes as one of columns, where lane 8 a + b has column 8 b + a: the transpose of the mask as
// eight rows of eight bits, by swaps of 1x1, 2x2 and 4x4 blocks.
__device__ __forceinline__ unsigned long long lanes_to_columns(unsigned long long m) {
  unsigned long long t = (m ^ (m >> 7)) & 0x00AA00AA00AA00AAull;
  m ^= t ^ (t << 7);
  t = (m ^ (m >> 14)) & 0x0000CCCC0000CCCCull;
  m ^= t ^ (t << 14);
  t = (m ^ (m >> 28)) & 0x00000000F0F0F0F0ull;
  return m ^ t ^ (t << 28);
}

__device__ __forceinline__ void finish_column(const ImParams& P, int p, int t, int ref_idx, const float lps[5],
                                              double red_bot, double red_top, int uniq, bool insert_slot,
                                              const Screen& A, uint32_t& err) {
  if (P.audit) {
    // diagnostics: the column's FP32 sums and read count, for the precision audit
    float4* a = (float4*)(P.audit + (size_t)8 * p);
    a[0] = make_float4(lps[0], lps[1], lps[2], lps[3]);
    a[1] = make_float4(lps[4], __uint_as_float(A.n), 0.0f, 0.0f);
  }
  // position_coverage::sum (identify_mutations.h:115-120)
  const double r1 = red_bot + red_top;
  const int total = (int)round((double)uniq) + (int)round(r1);
  if (ref_idx < 0) err |= kErrRefChar;
  uint8_t fl = kPosValid;
  bool cons = false, cons_unsure = false;
  if (A.n > 0) {
    int best = 0;
    float E = 0.0f;
#pragma unroll
    for (int b = 0; b < 5; b++) {
      if (lps[b] > lps[best]) best = b;
      E = fmaxf(E, fabsf(lps[b]));
    }
    const double g = ((double)A.n + 2.0) * 5.9604644775390625e-08;
    const double err_sum = (g < 0.5) ? g / (1.0 - g) * (double)E * 1.0001 : INFINITY;
    float second = -3.4028235e38f;
#pragma unroll
    for (int b = 0; b < 5; b++)
      if (b != best) second = fmaxf(second, lps[b]);
    const bool best_unsure = ((double)lps[best] - (double)second) <= 2.0 * err_sum;
    const double margin = 2.0 * err_sum + kScoreSlack;
    const double cbs = genotype_score_approx(lps, best) - P.log10_ref_length;
    const bool pred_unsure = best_unsure || fabs(cbs - P.mutation_cutoff) <= margin;
    if (cbs >= P.mutation_cutoff) fl |= kPosPredicted;
    if (best != ref_idx) cons = cbs > 0.0;
    cons_unsure = best_unsure || (best != ref_idx && fabs(cbs) <= margin);
    if (cons) fl |= kPosConsensus;
    if (pred_unsure || cons_unsure) {
      const int k = atomicAdd(P.n_fix, 1);
      if (k < P.fix_cap) P.fix[k] = p;
      else err |= kErrCapacity;
    }
  }
  if (r1 > 0.0) fl |= kPosRedundant;
  if (insert_slot) fl |= kPosInsert;
  if ((double)total <= P.targets[t].seed_cutoff) fl |= kPosSeed;
  // an uncertain consensus call goes to the exact scorer, which makes the call itself
  const bool sure = cons || cons_unsure || (P.screen_off && A.n > 0);
  const bool cand = sure || screen_passes(A, lps, ref_idx, P.log10_ref_length, P.polymorphism_cutoff, P.screen_margin);
  if (cand) {
    fl |= kPosCandidate;
    // In column order, for the candidate test: four neighbouring columns share a block of it, and so
    // the lines of the same alignments.  (In lane order, columns eight apart, the test of 19,731
    // candidates at 3,000x took 1814 us, in column order 1025.)
    const unsigned long long m = __ballot(true);
    const int leader = __builtin_ctzll(m);
    int first = 0;
    if ((int)(threadIdx.x & 63) == leader) first = atomicAdd(P.n_cand, __popcll(m));
    const int slot = __builtin_amdgcn_readlane(first, leader) +
                     __popcll(lanes_to_columns(m) & ((1ull << (p & (kWaveCols - 1))) - 1ull));
    if (slot < P.cand_cap) P.cand[slot] = make_int2(p, sure ? 0 : kCandScreened);
    else err |= kErrCapacity;
  }
  if (insert_slot) {
    const int slot = atomicAdd(P.n_ins, 1);
    if (slot < P.ins_cap) P.ins[slot] = p;
    else err |= kErrCapacity;
  }
  P.col_flags[p] = fl;
  P.col_unique[p] = uniq;
  P.col_total[p] = total;
}

// The exact FP64 genotype sums of column p (slot 0), in read order, by one wavefront: its pdata
// gathered by order-preserving compaction into keys[], then five lanes add the FP64 likelihoods in
// that order (identify_mutations.cpp:1561-1657, 1669-1689).  Every lane returns the sums in lps[]
// and the number of reads.  sums[5] is LDS scratch of the wavefront.
__device__ __forceinline__ int exact_column_sums(const ImParams& P, int p, uint32_t* keys, double* sums, double lps[5],
                                                 uint32_t& err) {
  const int lane = threadIdx.x & 63;
  const int S = P.read_set_max, Q = P.quality_max;
  const int64_t w = p / kWaveCols;
  const int rb = P.win_rb[w], re = P.win_re[w];
  if (rb < 0 || re < rb || re > P.n_reads) {
    err |= kErrIndex;
    for (int b = 0; b < 5; b++) lps[b] = 0.0;
    return 0;
  }
  int n = 0;
  for (int r0 = rb; r0 < re; r0 += 64) {
    const int r = r0 + lane;
    bool use = false;
    uint32_t key = 0;
    int obs = 0, strand_idx = 0;
    if (r < re) use = pdata_key(P.reads[r], P.cigar, P.bases, P.quals, p, 0, S, Q, P.base_quality_cutoff, key, obs,
                                strand_idx, err);
    if (use && key >= (uint32_t)P.tab_keys) {
      err |= kErrIndex;
      key = 0;
    }
    const unsigned long long mask = __ballot(use);
    if (use) {
      const int idx = n + __popcll(mask & ((1ull << lane) - 1ull));
      if (idx < P.key_cap) keys[idx] = key;
      else err |= kErrCapacity;
    }
    n += __popcll(mask);
  }
  n = min(n, P.key_cap);
  __syncthreads();
  if (lane < 5) {
    double acc = 0.0;
    for (int j = 0; j < n; j++) acc += P.tab_lp[(size_t)keys[j] * 5 + lane];
    sums[lane] = acc;
  }
  __syncthreads();
  for (int b = 0; b < 5; b++) lps[b] = sums[b];
  __syncthreads();
  return n;
}

// The read list of a column's wavefront: in LDS, or (kKeysGlobal, deep samples) this block's slice
// of the device scratch list.  A compile-time choice, so that the list's accesses keep their address
// space.
template <bool kKeysGlobal>
__device__ __forceinline__ uint32_t* column_key_list(const ImParams& P, uint32_t* lds) {
  if constexpr (kKeysGlobal) return P.key_scratch + (size_t)blockIdx.x * (size_t)P.key_cap;
  else return lds;
}

// Exact pure-genotype decisions for the columns the column kernel could not certify: one wavefront
// per column, the reference's call made from its exact sums.
template <bool kKeysGlobal>
__global__ void __launch_bounds__(64) k_fix_columns_t(ImParams P) {
  extern __shared__ uint32_t fix_lds_keys[];   // P.key_cap, unless the list is in device scratch
  uint32_t* fix_keys = column_key_list<kKeysGlobal>(P, fix_lds_keys);
  __shared__ double fix_lps[5];
  const int lane = threadIdx.x;
  const int n_fix = min(*P.n_fix, P.fix_cap);
  uint32_t err = 0;
  for (int i = blockIdx.x; i < n_fix; i += gridDim.x) {
    const int p = P.fix[i];
    if (p < 0 || p >= P.n_pos || p / kWaveCols >= P.n_windows) {
      err |= kErrIndex;
      continue;
    }
    double lps[5];
    const int n = exact_column_sums(P, p, fix_keys, fix_lps, lps, err);
    int best;
    double score;
    pure_genotype(lps, (uint32_t)n, best, score);
    const double cbs = score - P.log10_ref_length;
    const int ref_idx = char_index(P.ref[p]);
    if (lane == 0) {
      uint8_t fl = P.col_flags[p] & (uint8_t)~(kPosPredicted | kPosConsensus);
      if (cbs >= P.mutation_cutoff) fl |= kPosPredicted;
      if ((best != ref_idx) && !isnan(cbs) && (cbs > 0.0)) fl |= kPosConsensus;
      P.col_flags[p] = fl;
    }
    __syncthreads();
  }
  if (err) atomicOr(P.err, err);
}

// Precision audit (diagnostics, after an identify pass that wrote P.audit): for every listed
// column, the exact FP64 sums beside the column pass's FP32 ones, and whether the final predicted
// and consensus flags equal the calls the exact sums make.  out[6*i .. 6*i+4] = FP64 sums,
// out[6*i+5] = reads; *mismatches counts columns whose flags differ.
template <bool kKeysGlobal>
__global__ void __launch_bounds__(64) k_audit_columns_t(ImParams P, const int32_t* cols, int32_t n_cols, double* out,
                                                        uint32_t* mismatches) {
  extern __shared__ uint32_t audit_lds_keys[];
  uint32_t* keys = column_key_list<kKeysGlobal>(P, audit_lds_keys);
  __shared__ double sums[5];
  const int lane = threadIdx.x;
  uint32_t err = 0;
  for (int i = blockIdx.x; i < n_cols; i += gridDim.x) {
    const int p = cols[i];
    if (p < 0 || p >= P.n_pos || p / kWaveCols >= P.n_windows) {
      err |= kErrIndex;
      continue;
    }
    double lps[5];
    const int n = exact_column_sums(P, p, keys, sums, lps, err);
    int best;
    double score;
    pure_genotype(lps, (uint32_t)n, best, score);
    const double cbs = score - P.log10_ref_length;
    const int ref_idx = char_index(P.ref[p]);
    if (lane == 0) {
      uint8_t want = 0;
      if (cbs >= P.mutation_cutoff) want |= kPosPredicted;
      if ((best != ref_idx) && !isnan(cbs) && (cbs > 0.0)) want |= kPosConsensus;
      const uint8_t have = P.col_flags[p] & (kPosPredicted | kPosConsensus);
      if (have != want) atomicAdd(mismatches, 1u);
      for (int b = 0; b < 5; b++) out[(size_t)6 * i + b] = lps[b];
      out[(size_t)6 * i + 5] = (double)n;
    }
    __syncthreads();
  }
  if (err) atomicOr(P.err, err);
}

// LDS of a block: the table, then per wavefront kColWords (or kColSplitWords) words per column, the
// lists of alignments, and three bytes per column.
//
// Word of a column in LDS: the rare observations' sums per class, then the counts.
enum : int { kWG = 0, kWCnt = 4, kWGabs = 8, kWUniq = 9, kWN = 10 };
// The words that the wavefronts sharing a window add up.
enum : int { kXLps = 0, kXSL = 5, kXN = 6, kXUniq = 7, kXCnt = 8, kXG = 13, kXGabs = 18, kXIns = 19 };
static_assert(kWN + 1 == kColWords && kXIns + 1 == kColSplitWords, "words of a column");

__device__ __forceinline__ float swap32_add(float a, float b) {
  // lanes 0-31: a summed over the two halves of the wavefront; lanes 32-63: b
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap16_add(float a, float b) {
  // rows of 16 lanes: even rows a, odd rows b, each summed over its pair of rows
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// Eight values per lane summed over the eight groups of eight lanes: the lane of group g keeps value
// 4*(g>>2) + 2*((g>>1)&1) + (g&1).
__device__ __forceinline__ float sum_groups(const float v[8], bool odd8) {
  float r[4], q[2];
#pragma unroll
  for (int k = 0; k < 4; k++) r[k] = swap32_add(v[k], v[k + 4]);
#pragma unroll
  for (int k = 0; k < 2; k++) q[k] = swap16_add(r[k], r[k + 2]);
  const float keep = odd8 ? q[1] : q[0], give = odd8 ? q[0] : q[1];
  // row_ror:8
  return keep + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(give), 0x128, 0xF, 0xF, false));
}

// The lane's number, computed anew where it is used: in the word-wise loops the sums take most
// registers, and an address kept across them would be spilled (a reload from scratch memory waits for
// the alignments' bytes that are on the way).
__device__ __forceinline__ int lane_anew() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(l));
  return l;
}

// Bits 7 of the bytes [lo8/8, hi8/8) of eight, as two words; lo8 and hi8 are multiples of 8 of any
// size (a shift of 63 leaves no bit 7, as one of 64 would).
__device__ __forceinline__ uint2 byte_range(int lo8, int hi8) {
  constexpr uint64_t kHigh = 0x8080808080808080ull;
  const uint64_t m = (kHigh << min(max(lo8, 0), 63)) & ~(kHigh << min(max(hi8, 0), 63));
  return make_uint2((uint32_t)m, (uint32_t)(m >> 32));
}

// What bounds it: 4.6 Mb at 100x takes 1042 us, with the vector unit 67% and the LDS 64% busy (24 vector
// instructions and 24 bytes of table per position of an alignment's column; 293 M instructions in all, half
// of the LDS time bank conflicts between rows of different qualities).  With a lane per column and an
// alignment per step the same took 453 M instructions and 1421 us.  Eight columns to a lane: the ranges
// and counts are shared by eight positions, and eight alignments go at once, so that the 48 sums still
// leave four wavefronts to a SIMD (128 registers).  Measured before -> now, in us: 2.05 Mb at 83x of 36
// bases 834 -> 553, 1 Mb at 300x 882 -> 625, 1.3 Mb at 90x 507 -> 425, 701 kb of 300 bases 182 -> 187.
template <bool kLds, int kWaves>
__global__ void __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) k_identify_columns_t(ImParams P) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const bool split = P.col_split != 0;
  const int n_words = split ? kColSplitWords : kColWords;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  // the table comes first, at the offsets that the row reads can hold
  uint32_t* const words0 = (uint32_t*)(smem_raw + (kLds ? (size_t)P.fold_rows / 5 * kFoldLdsStride + 15 & ~(size_t)15 : 0));
  uint32_t* const words = words0 + wave * n_words * 64;             // [word][64]
  uint4* const list = (uint4*)(words0 + kWaves * n_words * 64) + wave * kColList;
  unsigned char* const info = (unsigned char*)(words0 + kWaves * (n_words * 64 + kColList * 4)) +
                              wave * 192;                           // per column: 0x80 scored, class, hypothesis
  Table<kLds> tab;
  constexpr uint32_t kStride = Table<kLds>::kStride;
  if constexpr (kLds) {
    // 24 of a row's 32 bytes, as three pairs
    const uint2* src = (const uint2*)P.fold;
    for (int i = threadIdx.x; i < P.fold_rows * 3; i += blockDim.x) {
      const int row = i / 3, part = i - row * 3, q = row / 5, o = row - q * 5;
      *(uint2*)(smem_raw + q * kFoldLdsStride + o * 32 + part * 8) = src[row * 4 + part];
    }
    __syncthreads();
    typedef __attribute__((address_space(3))) unsigned char LdsByte;
    tab.base = (uint32_t)(uintptr_t)(LdsByte*)smem_raw;
  } else {
    tab.base = 0;
  }
  tab.p = (const unsigned char*)P.fold;
  // the block's windows; a wavefront takes every kWaves-th, or all share each
  const int64_t chunk = (P.n_windows + gridDim.x - 1) / gridDim.x;
  const int64_t w_begin = (int64_t)xcd_major_block() * chunk;
  const int64_t w_end = min<int64_t>(w_begin + chunk, P.n_windows);
  uint32_t err = 0;
  const int S = P.read_set_max, Q = P.quality_max;
  const int qcut = P.base_quality_cutoff;
  const uint32_t block_bytes = (uint32_t)(Q + 1) * kStride;   // table bytes of a (MAPQ, read file) block
  // lane of group g = lane / 8 in the word-wise loops: columns 8 * (lane % 8) + 0..7 of the window;
  // afterwards the lane's one column
  const int j8 = 8 * (lane & 7);
  const bool odd8 = (lane & 8) != 0;
  const int my = j8 + 4 * (lane >> 5) + 2 * ((lane >> 4) & 1) + ((lane >> 3) & 1);
  const uint32_t q_sub = (uint32_t)__builtin_amdgcn_readfirstlane(min(max(qcut, 0), 128)) * 0x01010101u;

  for (int64_t w = w_begin + (split ? 0 : wave); w < w_end; w += split ? 1 : kWaves) {
    const int p0 = (int)(w * kWaveCols);
    // target of the lane's column, or -1 when it is not scored; looked up again after the word-wise
    // loops, which need the registers
    auto scored_target = [&]() {
      const int p = p0 + my;
      const int t = (p < P.n_pos) ? P.pos_target[p] : -1;
      return (t >= 0 && P.targets[t].scored && P.targets[t].prop_cutoff >= 0.0) ? t : -1;
    };
    // index of the reference base, negative when it is none
    auto reference = [&](int t) { return (t >= 0) ? char_index(P.ref[p0 + my]) : 0; };
    const int rb = __builtin_amdgcn_readfirstlane(P.win_rb[w]);
    const int re = __builtin_amdgcn_readfirstlane(P.win_re[w]);
    {
      const int t = scored_target(), ref_idx = reference(t);
      info[my] = (t >= 0) ? 0x80 : 0;
      info[64 + my] = (ref_idx >= 0 && ref_idx < 4) ? (uint8_t)(32 * (3 - ref_idx)) : 1;   // as the read's class below
      info[128 + my] = (ref_idx >= 0 && ref_idx < 5) ? (uint8_t)ref_idx : 0;               // hypothesis of the reference
    }
#pragma unroll
    for (int i = 0; i < kColWords; i++) words[64 * i + lane] = 0u;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");

    float lps[5][8], SL[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      SL[k] = 0.0f;
#pragma unroll
      for (int b = 0; b < 5; b++) lps[b][k] = 0.0f;
    }
    // counts of up to 255 steps, a byte each; n4 is 255 times them (modulo 2^32)
    uint2 uniq4 = make_uint2(0u, 0u), n4 = make_uint2(0u, 0u);
    int steps = 0;
    auto flush_counts = [&]() {
      n4.x *= 0xFEFEFEFFu;   // the inverse of 255
      n4.y *= 0xFEFEFEFFu;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        atomicAdd(&words[64 * kWUniq + j8 + k], ((k < 4 ? uniq4.x : uniq4.y) >> (8 * (k & 3))) & 0xFFu);
        atomicAdd(&words[64 * kWN + j8 + k], ((k < 4 ? n4.x : n4.y) >> (8 * (k & 3))) & 0xFFu);
      }
      uniq4 = n4 = make_uint2(0u, 0u);
      steps = 0;
    };
    struct Group {
      uint64_t b, q;
    };
    auto fetch = [&](const uint4 rec, int j8) {
      Group g;
      // the lane's eight bytes, or the nearest that touch the alignment
      const int s = (int)(int16_t)rec.y >> 3, e = (int)rec.y >> 19;
      const int r = min(max(j8, s - 7), e - 1);
      const uint32_t at = rec.x + (uint32_t)r + kBytesFrontPad;
      __builtin_memcpy(&g.b, P.bases - kBytesFrontPad + at, 8);
      __builtin_memcpy(&g.q, P.quals - kBytesFrontPad + at, 8);
      return g;
    };
    // an observation of class o in read direction, other than the reference base, at column col
    auto add_one = [&](uint32_t row, uint32_t col, uint32_t o, bool rev) {
      const uint32_t et = info[128 + col];
      const float e = tab.at(row + 4u * (rev && et < 4u ? 3u - et : et)), d = tab.at(row + 4u * o);
      const uint32_t obs = rev ? 3u - o : o;
      atomicAdd((float*)&words[64 * (kWG + obs) + col], e - d);
      atomicAdd(&words[64 * (kWCnt + obs) + col], 1u);
      atomicAdd((float*)&words[64 * kWGabs + col], fabsf(e) + fabsf(d));
    };
    auto add = [&](auto rev_c, const uint4 rec, const Group& g, int j8) {
      constexpr bool rev = decltype(rev_c)::value;
      // the aligned and the untrimmed columns, times 8, from this lane's first
      const uint2 span = byte_range((int)(int16_t)rec.y - 8 * j8, ((int)rec.y >> 16) - 8 * j8);
      const uint2 kept = byte_range((int)(int16_t)rec.z - 8 * j8, ((int)rec.z >> 16) - 8 * j8);
      const uint2 scored = *(const uint2*)(info + j8), refs = *(const uint2*)(info + 64 + j8);
      uint32_t qz[2], cz[2], nr[2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const uint32_t b = (uint32_t)(g.b >> (32 * h)), q = (uint32_t)(g.q >> (32 * h));
        // 32 * class of the base (T0 G1 C2 A3), N 0xFF
        const uint32_t cls = __builtin_amdgcn_perm(0x00000020u, 0x00406000u, b);
        const uint32_t valid = (h ? span.y : span.x) & (h ? scored.y : scored.x) & ~cls;
        const uint32_t ok = valid & (h ? kept.y : kept.x) & ((q | 0x80808080u) - q_sub);
        (h ? uniq4.y : uniq4.x) += valid >> 7;
        const uint32_t m = __builtin_amdgcn_perm(ok, ok << 8, 0x0B090A08u);   // bit 7 spread over its byte
        (h ? n4.y : n4.x) += m;
        // The zero rows where nothing is added.  Counted qualities are below 128; bytes before the alignment
        // are another's and may be 255, which must not carry into its first.
        qz[h] = ((q & 0x7F7F7F7Fu) + 0x01010101u) & m;
        // the row of the class in read direction: A0 C1 G2 T3 forward, the complement reverse
        cz[h] = (rev ? cls : cls ^ 0x60606060u) & m;
        nr[h] = (cls ^ (h ? refs.y : refs.x)) & m;
      }
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const uint32_t qk = (qz[k >> 2] >> (8 * (k & 3))) & 0xFFu, ck = (cz[k >> 2] >> (8 * (k & 3))) & 0xFFu;
        float T[6];
        tab.row(__umul24(qk, kStride) + (rec.w + ck), T);
#pragma unroll
        for (int b = 0; b < 4; b++) lps[b][k] += T[rev ? 3 - b : b];
        lps[4][k] += T[4];
        SL[k] += T[5];
      }
      // Observations other than the reference base, a few of a step's 512 positions.  (Queued and added
      // by 64 lanes at a time they took as long.)
      uint64_t odd = ((uint64_t)nr[1] << 32) | nr[0];
      while (odd) {
        const int sh = __builtin_ctzll(odd) & ~7;
        odd &= ~(0xFFull << sh);
        const uint32_t qk = (uint32_t)((((uint64_t)qz[1] << 32) | qz[0]) >> sh) & 0xFFu;
        const uint32_t ck = (uint32_t)((((uint64_t)cz[1] << 32) | cz[0]) >> sh) & 0xFFu;
        add_one(__umul24(qk, kStride) + rec.w + ck, (uint32_t)(j8 + (sh >> 3)), ck >> 5, rev);
      }
    };
    // Alignments go through the list eight at a time, the forward ones from its front and the reverse
    // ones from its end, so that the strand is a compile-time constant; what does not make up eight
    // stays for the next batch.
    int n_fwd = 0, n_rev = 0;
    auto drain = [&](auto rev_c, int groups) {
      constexpr bool rev = decltype(rev_c)::value;
      auto rec = [&](int i, int l) {
        const int k = 8 * i + (l >> 3);
        return list[rev ? kColList - 1 - k : k];
      };
      if (groups <= 0) return;
      int l = lane_anew();
      Group a = fetch(rec(0, l), 8 * (l & 7));
      for (int i = 1; i < groups; i++) {   // the next alignments' bytes are on the way while these are added
        l = lane_anew();
        const Group b = fetch(rec(i, l), 8 * (l & 7));
        add(rev_c, rec(i - 1, l), a, 8 * (l & 7));
        a = b;
      }
      l = lane_anew();
      add(rev_c, rec(groups - 1, l), a, 8 * (l & 7));
    };
    const int n_reads = re - rb;
    // alignments per turn: all 64 lanes' worth, or an even share of a shared window
    const int batch = split ? min(64, max(8, ((n_reads + kWaves - 1) / kWaves + 7) & ~7)) : 64;
    const int first = rb + (split ? wave * batch : 0), stride = split ? kWaves * batch : batch;
    bool others = false;
    for (int r0 = first; r0 < re; r0 += stride) {
      const int m = min(batch, re - r0);
      uint4 ra = make_uint4(0u, 0u, 0u, 0u), rc = make_uint4(0u, 0u, 0u, 0u);
      if (lane < m) {
        const uint4* src = (const uint4*)(P.idrec + r0 + lane);
        ra = src[0];
        rc = src[1];
      }
      // ra = {gpos, gend, seq_off, qoff}, rc = {trim, row_block, x1_flags, pad}
      const bool here = (int)ra.y > p0 && lane < m;
      const bool plain = here && (rc.z & kIdPlain);
      const bool rev = ((rc.z >> 16) & kReadReversed) != 0;
      const unsigned long long fm = __ballot(plain && !rev), rm = __ballot(plain && rev);
      others |= __ballot(here && !plain) != 0;
      if (plain) {
        // columns of the window, times 8; what lies outside [-64, 128] is as good as the limit
        auto edge = [&](int c) { return (uint32_t)(8 * min(max(c, -64), 128)) & 0xFFFFu; };
        const int q0 = (int)ra.w + p0;   // query position at the window's first column
        const int lo = (int)(rc.x & 0xFFFFu), hi = (int)(rc.x >> 16);
        const unsigned long long before = (1ull << lane) - 1ull;
        const int at = rev ? kColList - 1 - (n_rev + __popcll(rm & before)) : n_fwd + __popcll(fm & before);
        list[at] = make_uint4(ra.z + (uint32_t)q0, edge((int)ra.x - p0) | (edge((int)ra.y - p0) << 16),
                              edge(lo - q0) | (edge(max(hi, lo) - q0) << 16), tab.base + rc.y * block_bytes);
      }
      n_fwd += __popcll(fm);
      n_rev += __popcll(rm);
      const bool last = r0 + stride >= re;
      if (last) {   // fill up with alignments of no columns
        const uint4 none = make_uint4(0u, 0u, 0u, tab.base);
        if (lane < ((-n_fwd) & 7)) list[n_fwd + lane] = none;
        else if (lane >= 32 && lane - 32 < ((-n_rev) & 7)) list[kColList - 1 - (n_rev + lane - 32)] = none;
        n_fwd = (n_fwd + 7) & ~7;
        n_rev = (n_rev + 7) & ~7;
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      const int gf = n_fwd >> 3, gr = n_rev >> 3;
      if (steps + gf + gr > 255) flush_counts();
      steps += gf + gr;
      drain(std::integral_constant<bool, false>{}, gf);
      drain(std::integral_constant<bool, true>{}, gr);
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      const uint4 keep_f = list[min(8 * gf + lane, kColList - 1)], keep_r = list[max(kColList - 1 - (8 * gr + lane), 0)];
      n_fwd &= 7;
      n_rev &= 7;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      if (lane < n_fwd) list[lane] = keep_f;
      if (lane < n_rev) list[kColList - 1 - lane] = keep_r;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    flush_counts();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    // from here on: lane = column
    const int p = p0 + my, t = scored_target(), ref_idx = reference(t);
    const bool lane_ok = t >= 0;
    // hypothesis index of the reference base for a forward / reverse read
    const int e_top = (ref_idx >= 0 && ref_idx < 5) ? ref_idx : 0;
    const int e_bot = (e_top < 4) ? 3 - e_top : e_top;
    float l0 = sum_groups(lps[0], odd8), l1 = sum_groups(lps[1], odd8), l2 = sum_groups(lps[2], odd8);
    float l3 = sum_groups(lps[3], odd8), l4 = sum_groups(lps[4], odd8);
    Screen A;
    A.SL = sum_groups(SL, odd8);
    A.n = words[64 * kWN + my];
    int uniq = (int)words[64 * kWUniq + my];
    A.Gabs = __uint_as_float(words[64 * kWGabs + my]);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      A.cnt[i] = words[64 * (kWCnt + i) + my];
      A.G[i] = __uint_as_float(words[64 * (kWG + i) + my]);
    }
    A.cnt[4] = 0;
    A.G[4] = 0.0f;
    double red_bot = 0.0, red_top = 0.0;
    bool insert_slot = false;
    // The other alignments, one at a time in file order.  Where wavefronts share the window, each takes
    // those of its batches, except those with X1 != 1, whose 1/X1 the first adds in file order.
    for (int turn = 0; turn < (split ? 2 : 1); turn++) {
      if (turn == 0 ? !others : wave != 0) continue;
      const int from = (turn == 0) ? first : rb, step = (turn == 0) ? stride : 64, width = (turn == 0) ? batch : 64;
      for (int r0 = from; r0 < re; r0 += step) {
        const int m = min(width, re - r0);
        uint4 ra = make_uint4(0u, 0u, 0u, 0u), rc = make_uint4(0u, 0u, 0u, 0u);
        if (lane < m) {
          const uint4* src = (const uint4*)(P.idrec + r0 + lane);
          ra = src[0];
          rc = src[1];
        }
        const bool one = (rc.z & 0xFFFFu) == 1u;
        unsigned long long sm =
            __ballot(lane < m && (int)ra.y > p0 && !(rc.z & kIdPlain) && (!split || one == (turn == 0)));
        while (sm) {
          const int j = __builtin_ctzll(sm);
          sm &= sm - 1ull;
          const uint32_t xf = rdlane(rc.z, j);
          const uint32_t x1 = xf & 0xFFFFu, rflags = (xf >> 16) & 0xFFu;
          const uint32_t row_block = rdlane(rc.y, j);
          // entry bits: 1 cover, 2 deletion, 4 deletion quality usable, 8 trimmed, 16 insertion follows,
          // 32 deletion quality base outside the read
          uint32_t eb, bq, qq, qd = 0u;
          if (rflags & kReadSimple) {
            const int gpos = (int)rdlane(ra.x, j), gend = (int)rdlane(ra.y, j);
            const int qpos = p + (int)rdlane(ra.w, j);
            const uint32_t tr = rdlane(rc.x, j);
            const uint32_t dj = (uint32_t)(p - gpos), len = (uint32_t)(gend - gpos);
            // the byte at this lane's column, or the last aligned one when the column is outside
            const uint32_t at = rdlane(ra.z, j) + rdlane(ra.w, j) + (uint32_t)gpos + min(dj, len - 1u);
            bq = P.bases[at];
            qq = P.quals[at];
            const bool cover = lane_ok && dj < len;
            const bool trimmed = qpos < (int)(tr & 0xFFFFu) || qpos >= (int)(tr >> 16);
            eb = (cover ? 1u : 0u) | (trimmed ? 8u : 0u);
          } else {
            Entry E;
            prepare_general(P, load_read(P.reads, r0 + j), p, E, err);
            eb = ((E.cover && lane_ok) ? 1u : 0u) | (E.is_del ? 2u : 0u) | (E.del_ok ? 4u : 0u) |
                 (E.trimmed ? 8u : 0u) | (E.ondel > 0 ? 16u : 0u) | (E.del_oob ? 32u : 0u);
            bq = E.b;
            qq = E.q;
            qd = E.qd;
          }
          const bool is_del = (eb & 2u) != 0u;
          const bool top = !(rflags & kReadReversed);
          const uint32_t base = is_del ? (uint32_t)'.' : bq;
          const bool valid = (eb & 1u) && base != 15u;
          if (x1 != 1u) {
            // coverage of a read with X1 != 1 is 1/X1 (identify_mutations.cpp:1606-1614); a redundant
            // read (X1 > 1) adds nothing else
            const double inv = 1.0 / (double)x1;
            if (top) red_top += valid ? inv : 0.0;
            else red_bot += valid ? inv : 0.0;
            if (x1 > 1u) continue;
          } else {
            uniq += valid ? 1 : 0;
            insert_slot = insert_slot || (valid && (eb & 16u));
          }
          // observed class (reference strand) and quality (error_count.cpp:1049-1105), as selects;
          // a base code other than A C G T N, a read file beyond the table or a quality beyond its
          // maximum is reported (the reference asserts)
          const uint32_t o4 = base_idx4(bq);
          const uint32_t obs = is_del ? 4u : o4;
          const uint32_t q = is_del ? qd : qq;
          // a deletion whose quality base lies outside the read, on an untrimmed unique read
          if (valid && !(eb & 8u) && (eb & 32u)) err |= kErrQueryIndex;
          const bool cand = valid && !(eb & 8u) && (!is_del || (eb & 4u));
          const bool bad_base = cand && !is_del && o4 > 3u;
          bool ok = cand && !bad_base && (int)q >= qcut;
          const bool bad_rs = ok && row_block == 0xffffffffu;
          const bool bad_q = ok && !bad_rs && q >= (uint32_t)Q;
          err |= (bad_base ? kErrBaseCode : 0u) | (bad_rs ? kErrReadSet : 0u) | (bad_q ? kErrQuality : 0u);
          ok = ok && !bad_rs && !bad_q;
          const uint32_t o_rs = (obs < 4u && !top) ? (obs ^ 3u) : obs;
          const uint32_t row = tab.base + (ok ? row_block * block_bytes + (q + 1u) * kStride + 32u * o_rs : 0u);
          float T[6];
          tab.row(row, T);
          if (top) {
            l0 += T[0];
            l1 += T[1];
            l2 += T[2];
            l3 += T[3];
          } else {
            l0 += T[3];
            l1 += T[2];
            l2 += T[1];
            l3 += T[0];
          }
          l4 += T[4];
          A.SL += T[5];
          A.n += ok ? 1u : 0u;
          if (ok && (int)obs != ref_idx) {
            const float e = tab.at(row + 4u * (uint32_t)(top ? e_top : e_bot)), d = tab.at(row + 4u * o_rs);
            const float g = e - d;
            A.Gabs += fabsf(e) + fabsf(d);
#pragma unroll
            for (int o = 0; o < 5; o++) {
              const bool hit = (int)obs == o;
              A.G[o] += hit ? g : 0.0f;
              A.cnt[o] += hit ? 1u : 0u;
            }
          }
        }
      }
    }
    float L5[5] = {l0, l1, l2, l3, l4};
    if (split) {
      auto put = [&](int i, uint32_t v) { words[64 * i + my] = v; };
#pragma unroll
      for (int b = 0; b < 5; b++) {
        put(kXLps + b, __float_as_uint(L5[b]));
        put(kXCnt + b, A.cnt[b]);
        put(kXG + b, __float_as_uint(A.G[b]));
      }
      put(kXSL, __float_as_uint(A.SL));
      put(kXN, A.n);
      put(kXUniq, (uint32_t)uniq);
      put(kXGabs, __float_as_uint(A.Gabs));
      put(kXIns, insert_slot ? 1u : 0u);
      __syncthreads();
      for (int i = wave; i < kColSplitWords; i += kWaves) {   // word i over all wavefronts
        const bool whole = (i >= kXN && i < kXG) || i == kXIns;
        uint32_t v = words0[64 * i + lane];
        for (int k = 1; k < kWaves; k++) {
          const uint32_t x = words0[64 * (k * kColSplitWords + i) + lane];
          v = whole ? v + x : __float_as_uint(__uint_as_float(v) + __uint_as_float(x));
        }
        words0[64 * i + lane] = v;
      }
      __syncthreads();
      if (wave != 0) continue;
      auto got = [&](int i) { return words[64 * i + my]; };
#pragma unroll
      for (int b = 0; b < 5; b++) {
        L5[b] = __uint_as_float(got(kXLps + b));
        A.cnt[b] = got(kXCnt + b);
        A.G[b] = __uint_as_float(got(kXG + b));
      }
      A.SL = __uint_as_float(got(kXSL));
      A.n = got(kXN);
      uniq = (int)got(kXUniq);
      A.Gabs = __uint_as_float(got(kXGabs));
      insert_slot = got(kXIns) != 0u;
    }
    if (!lane_ok) {
      if (p < P.n_pos) {
        P.col_flags[p] = 0;
        P.col_unique[p] = 0;
        P.col_total[p] = 0;
      }
    } else {
      finish_column(P, p, t, ref_idx, L5, red_bot, red_top, uniq, insert_slot, A, err);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  if (err) atomicOr(P.err, err);
}

template __global__ void k_fix_columns_t<false>(ImParams P);
template __global__ void k_fix_columns_t<true>(ImParams P);
template __global__ void k_audit_columns_t<false>(ImParams P, const int32_t*, int32_t, double*, uint32_t*);
template __global__ void k_audit_columns_t<true>(ImParams P, const int32_t*, int32_t, double*, uint32_t*);
template __global__ void k_identify_columns_t<true, 8>(ImParams P);
template __global__ void k_identify_columns_t<false, 8>(ImParams P);
template __global__ void k_identify_columns_t<true, 4>(ImParams P);
template __global__ void k_identify_columns_t<false, 4>(ImParams P);

}  // namespace bsq
