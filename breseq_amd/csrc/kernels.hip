// kernels.hip -- CDNA4 (gfx950) kernels of pass 2 that follow the column kernel.
//
//  k_route_candidates the exact scorer's candidates: insert slots >= 1 of columns whose unique reads
//                     carry insertions, and the columns of the column pass that can be emitted
//  k_runs             MC and UN interval detection (identify_mutations.cpp:2262-2344, 2972-3007)
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "kernels.h"

namespace bsq {

#define WAVE 64

__device__ __forceinline__ int uniform_i(int v) { return __builtin_amdgcn_readfirstlane(v); }

/* ------------------------------------------------------------------------------------------ */
/* Candidates of the exact scorer                                                              */

// Insert slots >= 1 of column p, whose unique reads carry insertions (one wavefront): the slots the
// reference visits (identify_mutations.cpp:1359-1361, 1598-1599), slot 1 always, and slot s+1 while
// some unique read with a longer insertion has a base other than N at slot s.  Lanes take the
// window's alignments.  Every visited slot goes to the exact scorer, which makes the consensus and
// polymorphism calls itself.
__device__ __forceinline__ void route_insert_slots(const ImParams& P, int p, int lane, uint32_t& err) {
  const int64_t w = p / WAVE;
  if (p < 0 || p >= P.n_pos || w >= P.n_windows) {
    err |= kErrIndex;
    return;
  }
  const int rb = P.win_rb[w], re = P.win_re[w];
  if (rb < 0 || re < rb || re > P.n_reads) {
    err |= kErrIndex;
    return;
  }
  for (int slot = 1; slot < 65536; slot++) {
    if (lane == 0) {
      const int c = atomicAdd(P.n_score, 1);
      if (c < P.cand_cap) P.score[c] = make_int2(p, slot);
      else err |= kErrCapacity;
    }
    bool next = false;
    for (int r0 = rb; r0 < re; r0 += WAVE) {
      const int r = r0 + lane;
      if (r >= re) continue;
      const DRead R = P.reads[r];
      if (R.x1 != 1) continue;
      int qpos, indel;
      bool is_del;
      if (!entry_at(R, P.cigar, p, qpos, indel, is_del, err) || is_del || indel <= slot) continue;
      if (P.bases[R.seq_off + qpos + slot] != 15) next = true;
    }
    if (!__any(next)) break;
  }
}

template <int kCtrl>
__device__ __forceinline__ double dpp_add(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffLL), kCtrl, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), kCtrl, 0xf, 0xf, true);
  return v + __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ double lane_d(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Sum over the wavefront: within each row of 16 lanes by DPP (lane ^ 1, ^ 2, ^ 7, ^ 15), then the
// four rows' sums.  A sixth of the latency of six shuffles, which go through the LDS crossbar.
__device__ __forceinline__ double wave_sum_d(double v) {
  v = dpp_add<0xB1>(v);    // quad_perm [1,0,3,2]
  v = dpp_add<0x4E>(v);    // quad_perm [2,3,0,1]
  v = dpp_add<0x141>(v);   // row_half_mirror
  v = dpp_add<0x140>(v);   // row_mirror
  return (lane_d(v, 0) + lane_d(v, 16)) + (lane_d(v, 32) + lane_d(v, 48));
}

// Orders a wavefront's own LDS accesses (its lanes read what other lanes wrote).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A wavefront's count per distinct key of a column, in LDS.  kHash: slots found by linear probing from the key's
// hash (tables of many keys); else a slot per key of the table.
template <bool kHash>
struct KeyCounts {
  uint32_t* count;     // per slot; 0: unused
  uint32_t* keys;      // kHash: the slot's key
  uint16_t* list;      // the used slots
  int slots;           // kHash: a power of two
  int shift;           // kHash: 32 - log2 slots
  static constexpr uint32_t kNone = 0xffffffffu;
  __device__ __forceinline__ uint32_t key(uint32_t slot) const { return kHash ? keys[slot] : slot; }
  // counts the key of every lane with `use`; false when one found no slot
  __device__ __forceinline__ bool add(bool use, uint32_t k) const {
    if constexpr (!kHash) {
      if (use) atomicAdd(&count[k], 1u);
      return true;
    } else {
      uint32_t slot = (k * 0x9E3779B1u) >> shift;
      for (int probe = 0; probe < kRouteProbes && __any(use); probe++) {
        if (use) {
          const uint32_t old = atomicCAS(&keys[slot], kNone, k);
          if (old == kNone || old == k) {
            atomicAdd(&count[slot], 1u);
            use = false;
          } else {
            slot = (slot + 1u) & (uint32_t)(slots - 1);
          }
        }
      }
      return !__any(use);
    }
  }
};

// One EM pass over a column's distinct keys (lane = key, 64 at a time): S[b] = Sum_i r_i(b) / s_i,
// s_i = Sum_b f_b r_i(b), and the log10 likelihood Sum_i log10 s_i (without the lpmax sum), each key
// weighted with its reads.  The logarithms are FP32: within an ulp of log2 s_i, 3.8e-6 below 64, and the
// rounding of s_i, so each log10 within 2e-6 for s_i between 2^-64 and 2^64.  False when a read's is not.
template <bool kHash>
__device__ __forceinline__ bool key_pass(const ImParams& P, const KeyCounts<kHash>& C, int K, int lane, const double f[5],
                                         double S[5], double& ll) {
  double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, l2 = 0.0;
  bool bad = false;
  for (int k0 = 0; k0 < K; k0 += WAVE) {
    const int k = k0 + lane;
    if (k >= K) continue;
    const uint32_t slot = C.list[k];
    const double h = (double)C.count[slot];
    const double* t = P.tab_r + (size_t)C.key(slot) * 6;
    double r[5], s = 0.0;
#pragma unroll
    for (int b = 0; b < 5; b++) {
      r[b] = t[b];
      s = fma(f[b], r[b], s);
    }
    bad = bad || !(s > 0x1p-64 && s < 0x1p64);
    double y = __builtin_amdgcn_rcp(s);
    y = fma(fma(-s, y, 1.0), y, y);
    y = fma(fma(-s, y, 1.0), y, y) * h;
#pragma unroll
    for (int b = 0; b < 5; b++) acc[b] = fma(r[b], y, acc[b]);
    l2 = fma(h, (double)log2f((float)s), l2);
  }
#pragma unroll
  for (int b = 0; b < 5; b++) S[b] = wave_sum_d(acc[b]);
  ll = wave_sum_d(l2) * 0.30102999566398119521;
  return !__any(bad);
}

// Whether a column that only the column pass's bound let through can reach the presence-score cutoff
// (identify_mutations.cpp:3240-3344): false only if no allele v can, from bounds on the two
// likelihoods of its score that follow the reference's own EM loops a few passes (one wavefront).
//   * Full fit: the likelihood is concave in the frequencies, so its maximum is at most
//     LL(f) + (max_b Sum_i r_i(b) / s_i - n) / ln 10 at any f.  f: the EM iterates from the
//     reference's starting point, the least bound of the first four.
//   * Null fit of v: EM never lowers the likelihood, and the reference reports that of its last
//     pass's frequencies, so any earlier iterate's likelihood is at most the reported one.  The k-th
//     iterate is used only when every step before it moved a frequency by more than 2 tol, which makes
//     the reference take that pass too.
// The reads' likelihoods depend on their table keys alone, so the passes run over the distinct keys
// with their counts.  The comparison keeps the margin of the column pass's screen, plus the
// rounding of the FP32 logarithms (2e-6 a read and likelihood).
template <bool kHash>
__device__ __forceinline__ bool may_be_emitted(const ImParams& P, const KeyCounts<kHash>& C, int K, const uint32_t cnt[5],
                                               int ref_idx, int lane) {
  double n = 0.0;
#pragma unroll
  for (int b = 0; b < 5; b++) n += (double)cnt[b];
  const double need = P.polymorphism_cutoff - P.screen_margin - 4e-6 * n + P.log10_ref_length;
  double upper = INFINITY;
  {
    double f[5], S[5], ll, total = 0.0;
#pragma unroll
    for (int b = 0; b < 5; b++) {
      f[b] = 0.5 + (double)cnt[b];
      total += f[b];
    }
#pragma unroll
    for (int b = 0; b < 5; b++) f[b] /= total;
    for (int it = 0; it < 4; it++) {
      if (!key_pass(P, C, K, lane, f, S, ll)) return true;
      double g = 0.0;
#pragma unroll
      for (int b = 0; b < 5; b++) {
        g = fmax(g, S[b]);
        f[b] = f[b] * S[b] / n;
      }
      const double gap = (g - n) * 0.43429448190325182765;
      upper = fmin(upper, ll + fmax(gap, 0.0));
      if (gap < 0.02) break;
    }
  }
#pragma unroll 1
  for (int v = 0; v < 5; v++) {
    if (v == ref_idx) continue;
    double f[5], S[5], ll, total = 0.0;
#pragma unroll
    for (int b = 0; b < 5; b++) {
      f[b] = (b == v) ? 0.0 : 0.5 + (double)cnt[b];
      total += f[b];
    }
#pragma unroll
    for (int b = 0; b < 5; b++) f[b] /= total;
    bool clear = false;
    for (int it = 0; it < 8; it++) {
      if (!key_pass(P, C, K, lane, f, S, ll)) return true;
      if (upper - ll < need) {
        clear = true;
        break;
      }
      double most = 0.0;
#pragma unroll
      for (int b = 0; b < 5; b++) {
        const double fn = f[b] * S[b] / n;
        most = fmax(most, fabs(fn - f[b]));
        f[b] = fn;
      }
      if (!(most > 2.0 * P.precision_decimal)) break;
    }
    if (!clear) return true;
  }
  return false;
}

// The exact scorer's candidates (one wavefront per column): insert slots of the columns with
// insertions, and the column pass's candidates, those that its bound alone let through tested
// again by may_be_emitted.  At 3,000 reads a column the bound of the column pass rules out next to
// nothing (19,743 of 20,011 columns passed it, of which some 30 are emitted) and the exact null fit of
// each took the scorer 35.6 ms; this test takes 1.02 ms and leaves 36 (1 Mb at 300x with
// 390 variants: 7,852 candidates, 0.17 ms, leaves 451).
// LDS per wavefront: a count per table key and the list of those that occur; where the table has more than
// kRouteKeys keys (from three MAPQs of paired reads on), a hash of the column's own keys (kHash), so that
// the test does not depend on the table's size.  While such tables went without the test, all screened columns
// went to the scorer (before -> now test and scorer, in ms; paired reads): 1 Mb at 300x, 3 MAPQs 1.6 -> 0.20 + 0.57,
// 10 MAPQs 9.6 -> 0.24 + 0.65, 40 MAPQs 10.0 -> 0.28 + 0.69; 20 kb at 3,000x, 3 MAPQs 14.9 -> 1.35 + 0.66,
// 40 MAPQs 34.1 -> 3.9 + 5.5.
template <bool kHash>
__global__ void __launch_bounds__(64 * kRouteWaves) k_route_candidates_t(ImParams P) {
  extern __shared__ uint32_t route_lds[];
  const int lane = threadIdx.x & (WAVE - 1), wave = uniform_i((int)threadIdx.x / WAVE), waves = (int)blockDim.x / WAVE;
  const int wv = blockIdx.x * waves + wave, n_wv = gridDim.x * waves;
  KeyCounts<kHash> C;
  C.slots = kHash ? P.route_slots : P.tab_keys;
  C.shift = kHash ? __clz(P.route_slots) + 1 : 0;
  C.count = route_lds + (size_t)wave * route_words(kHash, C.slots);
  C.keys = C.count + C.slots;
  C.list = (uint16_t*)(kHash ? C.keys + C.slots : C.keys);
  uint32_t err = 0;
  const int n_ins = min(*P.n_ins, P.ins_cap);
  for (int i = wv; i < n_ins; i += n_wv) route_insert_slots(P, uniform_i(P.ins[i]), lane, err);
  for (int i = lane; i < C.slots; i += WAVE) {
    C.count[i] = 0;
    if (kHash) C.keys[i] = C.kNone;
  }
  wave_lds_sync();
  const int n_cand = min(*P.n_cand, P.cand_cap);
  for (int ci = wv; ci < n_cand; ci += n_wv) {
    const int2 cd = P.cand[ci];
    const int p = uniform_i(cd.x);
    const int64_t w = p / WAVE;
    if (p < 0 || p >= P.n_pos || w >= P.n_windows) {
      err |= kErrIndex;
      continue;
    }
    bool keep = true;
    if (uniform_i(cd.y) == kCandScreened) {
      const int rb = uniform_i(P.win_rb[w]), re = uniform_i(P.win_re[w]);
      if (rb < 0 || re < rb || re > P.n_reads) {
        err |= kErrIndex;
        continue;
      }
      const uint32_t qspan = (uint32_t)max(0, P.quality_max - P.base_quality_cutoff);
      uint32_t cnt[5] = {0, 0, 0, 0, 0};
      bool full = false;
      for (int r0 = rb; r0 < re && !full; r0 += WAVE) {
        const int r = r0 + lane;
        bool use = false;
        uint32_t key = 0;
        int obs = 0;
        bool past = true;   // starts after the column: so do all later ones
        if (r < re) {
          const uint4* src = (const uint4*)(P.idrec + r);
          const uint4 ra = src[0], rc = src[1];
          past = (int)ra.x > p;
          const uint32_t xf = rc.z, flags = xf >> 16;
          // X1 of 0 or 1, as pdata_key
          if ((uint32_t)p - ra.x < ra.y - ra.x && (xf & 0xFFFFu) <= 1u) {
            if (flags & kReadSimple) {
              const uint32_t qpos = (uint32_t)p + ra.w;
              const uint32_t b = P.bases[ra.z + qpos], q = P.quals[ra.z + qpos];
              const int o = bam_index((uint8_t)b);
              use = o >= 0 && o < 4 && qpos >= (rc.x & 0xFFFFu) && qpos < (rc.x >> 16) &&
                    q - (uint32_t)P.base_quality_cutoff < qspan && rc.y != 0xffffffffu;
              obs = o;
              key = (rc.y * (uint32_t)P.quality_max + q) * 10u + (uint32_t)o * 2u + ((flags & kReadReversed) ? 1u : 0u);
            } else {
              // data errors of this read were reported by the column pass
              int strand_idx = 0;
              uint32_t e = 0;
              use = pdata_key(P.reads[r], P.cigar, P.bases, P.quals, p, 0, P.read_set_max, P.quality_max,
                              P.base_quality_cutoff, key, obs, strand_idx, e);
            }
          }
        }
        use = use && key < (uint32_t)P.tab_keys;
        const bool counted = C.add(use, key);
        full = full || !counted;
#pragma unroll
        for (int b = 0; b < 5; b++) cnt[b] += (uint32_t)__popcll(__ballot(use && obs == b));
        if (__all(past)) break;
      }
      wave_lds_sync();
      int K = 0;
      for (int k0 = 0; k0 < C.slots; k0 += WAVE) {
        const bool on = k0 + lane < C.slots && C.count[k0 + lane] != 0;
        const unsigned long long m = __ballot(on);
        if (on) C.list[K + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)(k0 + lane);
        K += __popcll(m);
      }
      wave_lds_sync();
      const int c = char_index(P.ref[p]);
      keep = full || (K > 0 && may_be_emitted(P, C, K, cnt, c < 0 ? 5 : c, lane));
      wave_lds_sync();
      for (int k = lane; k < K; k += WAVE) {
        const uint32_t slot = C.list[k];
        C.count[slot] = 0;
        if (kHash) C.keys[slot] = C.kNone;
      }
      wave_lds_sync();
    }
    if (keep && lane == 0) {
      const int k = atomicAdd(P.n_score, 1);
      if (k < P.cand_cap) P.score[k] = make_int2(p, 0);
      else err |= kErrCapacity;
    }
  }
  if (err) atomicOr(P.err, err);
}

/* ------------------------------------------------------------------------------------------ */
/* MC / UN runs                                                                                */

// Runs are found by the columns that open them and walked by a whole wavefront, 256 columns a step
// (four coalesced loads per lane), so a run of L columns costs L / 256 dependent steps:
//   MC: maximal runs with unique coverage <= the propagation cutoff; the seed is reached if any
//       column of the run, or the column closing it, has total coverage <= the seed cutoff
//       (identify_mutations.cpp:2270-2281); the redundant sub-range follows :2326-2343.
//   UN: maximal runs of columns without a predicted base (:2972-3007).
// The reference's walk over an MC run keeps red_start at the column before the first column without
// redundant coverage and red_end at the column after the last one, each -1 when the run starts
// (ends) there; a run with redundant coverage throughout has red_start at its last column.  The
// walk below gets both from the first and last such column of the run.
constexpr int kRunSpan = 4 * WAVE;

__device__ __forceinline__ int first_in(uint64_t m) { return __builtin_ctzll(m); }
__device__ __forceinline__ int last_in(uint64_t m) { return 63 - __builtin_clzll(m); }

__device__ void walk_mc_run(const RunParams& P, int s, int lane) {
  const TargetInfo T = P.targets[P.pos_target[s]];
  const int first = T.off, last = T.off + T.len - 1;
  bool seed = false;
  int fz = -1, lz = -1, e = last;
  for (int q0 = s;; q0 += kRunSpan) {
    bool in[4];
    uint8_t fl[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int q = q0 + j * WAVE + lane;
      const bool valid = q <= last;
      const int32_t u = valid ? P.col_unique[q] : 0;
      fl[j] = valid ? P.col_flags[q] : 0;
      in[j] = valid && (double)u <= T.prop_cutoff;
    }
    int end = kRunSpan;   // first index of this step outside the run
#pragma unroll
    for (int j = 3; j >= 0; j--) {
      const uint64_t out = __ballot(!in[j]);
      if (out) end = j * WAVE + first_in(out);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const bool member = j * WAVE + lane < end;
      seed |= member && (fl[j] & kPosSeed);
      const uint64_t nr = __ballot(member && !(fl[j] & kPosRedundant));
      if (nr) {
        if (fz < 0) fz = q0 + j * WAVE + first_in(nr);
        lz = q0 + j * WAVE + last_in(nr);
      }
    }
    if (end < kRunSpan) {
      e = q0 + end - 1;
      break;
    }
  }
  const bool any_seed = __any(seed);
  if (lane != 0) return;
  RunRec R;
  R.kind = 0;
  R.s = s;
  R.e = e;
  R.seed = (any_seed || (e < last && (P.col_flags[e + 1] & kPosSeed))) ? 1 : 0;
  R.red_start = fz < 0 ? e : (fz > s ? fz - 1 : -1);
  R.red_end = (fz >= 0 && lz < e) ? lz + 1 : -1;
  R.lo = (s > first) ? P.col_unique[s - 1] : -1;
  R.li = P.col_unique[s];
  R.ri = P.col_unique[e];
  R.ro = (e < last) ? P.col_unique[e + 1] : -1;
  const int k = atomicAdd(P.n_runs, 1);
  if (k < P.run_cap) P.runs[k] = R;
  else atomicOr(P.err, kErrCapacity);
}

__device__ void walk_un_run(const RunParams& P, int s, int lane) {
  const TargetInfo T = P.targets[P.pos_target[s]];
  const int last = T.off + T.len - 1;
  int e = last;
  for (int q0 = s;; q0 += kRunSpan) {
    int end = kRunSpan;
#pragma unroll
    for (int j = 3; j >= 0; j--) {
      const int q = q0 + j * WAVE + lane;
      const bool in = q <= last && !(P.col_flags[q] & kPosPredicted);
      const uint64_t out = __ballot(!in);
      if (out) end = j * WAVE + first_in(out);
    }
    if (end < kRunSpan) {
      e = q0 + end - 1;
      break;
    }
  }
  if (lane != 0) return;
  RunRec R;
  R.kind = 1;
  R.s = s;
  R.e = e;
  R.seed = 0;
  R.red_start = R.red_end = -1;
  R.lo = R.li = R.ri = R.ro = 0;
  const int k = atomicAdd(P.n_runs, 1);
  if (k < P.run_cap) P.runs[k] = R;
  else atomicOr(P.err, kErrCapacity);
}

// One lane per column marks the runs that open there; the wavefront then walks each of its marked
// runs in column order.  Every lane stays to the end: the walks need all 64.
__global__ void __launch_bounds__(256) k_runs(RunParams P) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & (WAVE - 1);
  bool mc_open = false, un_open = false;
  if (p < P.n_pos) {
    const int t = P.pos_target[p];
    if (t >= 0) {
      const TargetInfo T = P.targets[t];
      if (T.scored && T.prop_cutoff >= 0.0) {
        const bool at_first = p == T.off;
        if (P.do_mc && (double)P.col_unique[p] <= T.prop_cutoff)
          mc_open = at_first || !((double)P.col_unique[p - 1] <= T.prop_cutoff);
        if (!(P.col_flags[p] & kPosPredicted)) un_open = at_first || (P.col_flags[p - 1] & kPosPredicted);
      }
    }
  }
  const int base = uniform_i(p - lane);
  for (uint64_t m = __ballot(mc_open); m; m &= m - 1) walk_mc_run(P, base + first_in(m), lane);
  for (uint64_t m = __ballot(un_open); m; m &= m - 1) walk_un_run(P, base + first_in(m), lane);
}

template __global__ void k_route_candidates_t<false>(ImParams P);
template __global__ void k_route_candidates_t<true>(ImParams P);

}  // namespace bsq
