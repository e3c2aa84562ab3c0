// error_count.hip -- pass 1 of the pileup path on CDNA4 (gfx950): the covariate count table and the
// unique-only coverage histogram (error_count_pileup::pileup_callback, error_count.cpp:125-199, with
// cErrorTable::count_alignment_position, :854-986).
//
// Both outputs are integer sums, so they do not depend on the order in which pileup entries are
// visited.  Pass 1 therefore walks each alignment once (read-parallel) instead of walking columns:
//
//   k_ec_reads       64 consecutive alignments per work item of a wavefront, which steps through
//                    their M/=/X runs together.  The runs become items of eight query positions that
//                    the 64 lanes share evenly.  Bases and qualities are 8-byte loads from 8-byte
//                    aligned groups.  Covariates go to an LDS-privatized count table.  The lane of an
//                    alignment adds +1/-1 at the ends of each aligned run to a per-column difference
//                    array (unique or redundant).
//   k_cov_tile_sums  phase 1 of the prefix scan of the difference arrays (per 4096-column tile)
//   k_cov_tile_scan  phase 2: exclusive scan of the tile sums (one block)
//   k_cov_hist       phase 3: per-column unique and redundant coverage -> histogram of the unique
//                    coverage of columns without redundant reads (LDS-privatized)
//
// Deleted reference bases (is_del entries) never count, so only M/=/X runs contribute to either
// output; the entry of the last base of a run carries the run's indel (next CIGAR operations), as
// htslib's resolve_cigar2 reports it.
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "kernels.h"

namespace bsq {

// Copies each alignment's bases and qualities to its 8-byte aligned offset (DRead::seq_off) in the
// device layout, the bytes behind its last group's end as zeros.  Sixteen lanes take an alignment, in
// groups of eight bytes, and note its largest quality (byte_max; 255 as well when a base code is none of
// A, C, G, T and N): 4.6 Mb at 100x (1.85 GB moved) in 580 us, where a byte per lane took
// 1530 us.
// Reads up to seven bytes past the end of src_b and src_q.
__global__ void __launch_bounds__(256) k_repack_reads(const DRead* reads, const int64_t* raw_off, int64_t n_reads,
                                                      const uint8_t* src_b, const uint8_t* src_q, uint8_t* dst_b,
                                                      uint8_t* dst_q, uint8_t* byte_max) {
  const int l = threadIdx.x & 15;
  const int64_t step = ((int64_t)gridDim.x * blockDim.x) >> 4;
  for (int64_t r = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 4; r < n_reads; r += step) {
    const int len = (int)reads[r].l_qseq;
    const int64_t d = reads[r].seq_off, s = raw_off[r];
    uint32_t top = 0, bad = 0;
    for (int j = 8 * l; j < len; j += 128) {
      uint64_t b, q;
      __builtin_memcpy(&b, src_b + s + j, 8);   // one load; the hardware takes any alignment
      __builtin_memcpy(&q, src_q + s + j, 8);
      const uint64_t in = ~0ull >> (64 - 8 * min(len - j, 8));
      b &= in;
      q &= in;
      *(uint64_t*)(dst_b + d + j) = b;
      *(uint64_t*)(dst_q + d + j) = q;
#pragma unroll
      for (int k = 0; k < 8; k++) top = max(top, (uint32_t)(q >> (8 * k)) & 0xFFu);
      bad |= not_bases((uint32_t)(b | (0x0F0F0F0F0F0F0F0Full & ~in)));
      bad |= not_bases((uint32_t)((b | (0x0F0F0F0F0F0F0F0Full & ~in)) >> 32));
    }
    if (bad) top = 255;
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, o, 64));
    if (l == 0) byte_max[r] = (uint8_t)top;
  }
}

__global__ void k_fill_i32(int32_t* p, int64_t n, int32_t v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}

__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Inclusive scan across the 64 lanes of a wavefront.
__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  return v;
}


// Indel carried by the entry of the last base of the reference-consuming operation at index k
// (htslib resolve_cigar2 as breseq reads it; same rule as entry_at).
__device__ __forceinline__ int run_end_indel(const uint32_t* c, int k, int n) {
  if (k + 1 >= n) return 0;
  const uint32_t op2 = c[k + 1] & 15u;
  int indel = 0;
  if (op2 == OP_D) {
    indel = -(int)(c[k + 1] >> 4);
    for (int kk = k + 2; kk < n; ++kk) {
      if ((c[kk] & 15u) != OP_D) break;
      indel -= (int)(c[kk] >> 4);
    }
  } else if (op2 == OP_I) {
    indel = (int)(c[k + 1] >> 4);
    for (int kk = k + 2; kk < n; ++kk) {
      const uint32_t o3 = c[kk] & 15u;
      if (o3 == OP_I) indel += (int)(c[kk] >> 4);
      else if (o3 != OP_P) break;
    }
  } else if (op2 == OP_P && k + 2 < n) {
    int l3 = 0;
    for (int kk = k + 2; kk < n; ++kk) {
      const uint32_t o3 = c[kk] & 15u;
      if (o3 == OP_I) l3 += (int)(c[kk] >> 4);
      else if (is_ref_op(o3)) break;
    }
    if (l3 > 0) indel = l3;
  }
  return indel;
}

__device__ __forceinline__ uint32_t byte_of(uint32_t w, int k) { return (w >> (8 * k)) & 0xFFu; }

// Strand-folded base indices as 4-bit lookup tables: read bases by BAM code (A1 C2 G4 T8), reference
// bases by kRef* code (A0 C1 G2 T3 '.'4 N5).  The reverse-strand tables complement A<->T, C<->G, as
// count_alignment_position does before indexing (error_count.cpp:887-903).  15 = not a base.
constexpr uint64_t kReadLutFwd = 0xFFFFFFF3FFF2F10FULL;
constexpr uint64_t kReadLutRev = 0xFFFFFFF0FFF1F23FULL;
constexpr uint32_t kRefLutFwd = 0xFF543210u;
constexpr uint32_t kRefLutRev = 0xFF540123u;

// A block's count table in LDS: 25 words per (read set, quality) row, ri + 5*oi, and after the rows
// one signed word per row for the '..' pairs (below).
constexpr uint32_t kEcRow = 25;

struct EcTable {
  uint32_t* bins;
  int32_t* pairs;
  __device__ __forceinline__ void add(uint32_t row, uint32_t ri, uint32_t oi) const {
    atomicAdd(&bins[row * kEcRow + ri + 5u * oi], 1u);
  }
};

// Four positions' table offsets: bytes of (ri + 5*oi) * 4, or 96 where nothing is counted (N base,
// N reference).  Byte-wise on whole words: v_perm_b32 looks four codes up at once, the strand is an XOR
// (the classes are numbered T0 G1 C2 A3, the complement of A0 C1 G2 T3).  `odd` becomes nonzero when a byte needs the
// position-wise path: a code that is no base, a reference that is neither base nor N, or a quality
// that may be at or above the maximum.
__device__ __forceinline__ uint32_t ec_classes(uint32_t b, uint32_t q, uint32_t r, uint32_t strand, uint32_t q_add,
                                               uint32_t& odd) {
  const uint32_t rd = read_classes(b);
  const uint32_t rf = __builtin_amdgcn_perm(0x40408040u, 0x0004080Cu, r);   // 4 * class, N 0x80, other 0x40
  const uint32_t u = rd | rf;
  odd |= not_bases(b, rd);
  odd |= u & ~(u >> 1) & 0x40404040u;
  odd |= (((q & 0x7F7F7F7Fu) + q_add) | q) & 0x80808080u;
  const uint32_t x = (u ^ strand) & 0x3C3C3C3Cu;
  const uint32_t c = x + ((x >> 2) & 0x0C0C0C0Cu);
  const uint32_t none = __builtin_amdgcn_perm(u, u << 8, 0x0B090A08u);      // bit 7 spread over its byte
  return (none & 0x60606060u) | (c & ~none);
}

// Counts base against reference (count_alignment_position's first observation, error_count.cpp:
// 877-903) of eight consecutive query positions: bytes [lo, hi) of the base, quality and reference
// words, all in the run.  Nothing-counted bytes go to bin 24 of their row, which is never read.
__device__ __forceinline__ void ec_eight(uint2 b, uint2 q, const uint2 r, int lo, int hi, bool rev, uint32_t row0,
                                         uint32_t Q, const EcTable& T, uint32_t& err) {
  const uint64_t in = (~0ull << (8 * max(lo, 0))) & (~0ull >> (64 - 8 * min(hi, 8)));
  const uint32_t in0 = (uint32_t)in, in1 = (uint32_t)(in >> 32);
  b.x = (b.x & in0) | (0x0F0F0F0Fu & ~in0);   // outside the run: N bases of quality 0
  b.y = (b.y & in1) | (0x0F0F0F0Fu & ~in1);
  q.x &= in0;
  q.y &= in1;
  const uint32_t strand = rev ? 0u : 0x3C3C3C3Cu;
  const uint32_t q_add = (Q <= 128u) ? (128u - Q) * 0x01010101u : 0u;
  uint32_t odd = 0;
  const uint32_t c0 = ec_classes(b.x, q.x, r.x, strand, q_add, odd);
  const uint32_t c1 = ec_classes(b.y, q.y, r.y, strand, q_add, odd);
  unsigned char* base = (unsigned char*)(T.bins + row0 * kEcRow);
  if (odd == 0) {
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const uint32_t off = __umul24(byte_of(k < 4 ? q.x : q.y, k & 3), 4u * kEcRow) + byte_of(k < 4 ? c0 : c1, k & 3);
      atomicAdd((uint32_t*)(base + off), 1u);
    }
    return;
  }
  const uint64_t rlut = rev ? kReadLutRev : kReadLutFwd;
  const uint32_t flut = rev ? kRefLutRev : kRefLutFwd;
  for (int k = 0; k < 8; k++) {
    const uint32_t bk = byte_of(k < 4 ? b.x : b.y, k & 3), qk = byte_of(k < 4 ? q.x : q.y, k & 3);
    const uint32_t rk = byte_of(k < 4 ? r.x : r.y, k & 3);
    if (bk == 15u || rk == kRefN) continue;
    const uint32_t oi = (bk > 15u) ? 15u : (uint32_t)(rlut >> (4u * bk)) & 15u;
    const uint32_t ri = (flut >> (4u * rk)) & 15u;
    if (oi > 3u) err |= kErrBaseCode;
    else if (ri > 3u) err |= kErrRefChar;
    else if (qk >= Q) err |= kErrQuality;
    else T.add(row0 + qk, ri, oi);
  }
}

// The '..' pair observation (error_count.cpp:909-928) of a position takes the base after it in read
// direction against the reference after it in reference direction: for a forward read position
// j = qpos + 1, for a reverse read j = qpos, and both count the quality at j where neither the base
// nor the reference at j is N -- the condition under which the base observation counts j.  So over a
// run [y, last] the pairs are the run's base observations except one at the run's first position
// (forward) or last (reverse), and one more where the pairs reach past the run.  The flush adds the
// 16 base bins of a row up, and `pairs` holds these corrections: one LDS atomic per run in place of
// one per position.  q_end is never before a run's last base, since only soft clips behind it are
// taken off it.
__device__ __forceinline__ void ec_pair(const EcParams& P, const uint8_t* sq, const uint8_t* ql, int j, int col,
                                        uint32_t row0, int v, const EcTable& T, uint32_t& err) {
  const uint32_t b = sq[j], q = ql[j];
  if (b == 15u || P.ref_idx[col] == kRefN) return;
  if (q >= (uint32_t)P.quality_max) err |= kErrQuality;
  else atomicAdd(&T.pairs[row0 + q], v);
}

__device__ __forceinline__ void ec_run_pairs(const EcParams& P, const uint8_t* sq, const uint8_t* ql, bool rev, int x,
                                             int y, int len, int last_indel, int qe0, uint32_t row0, const EcTable& T,
                                             uint32_t& err) {
  const int last = y + len - 1;
  const bool past = last_indel == 0 && qe0 > last;   // the run's last position has a pair
  if (!rev) ec_pair(P, sq, ql, y, x, row0, -1, T, err);
  if (past != rev) ec_pair(P, sq, ql, past ? last + 1 : last, past ? x + len : x + len - 1, row0, past ? 1 : -1, T, err);
}

// a[at] += v from every lane with at >= 0, one atomic for consecutive lanes of the same address: in a
// deep sample dozens of neighbouring alignments start (and, of equal length, end) at one column.
__device__ __forceinline__ void add_equal(int32_t* a, int at, int v) {
  const int lane = threadIdx.x & 63;
  const int prev = __shfl_up(at, 1, 64);
  const bool head = lane == 0 || prev != at;
  const unsigned long long later = __ballot(head) & ~((2ull << lane) - 1ull);
  const int n = (later ? __builtin_ctzll(later) : 64) - lane;
  if (head && at >= 0) atomicAdd(&a[at], v * n);
}

__device__ __forceinline__ uint2 load8(const uint8_t* p) {
  uint2 v;
  __builtin_memcpy(&v, p, 8);   // one load; the hardware takes any alignment
  return v;
}

// The one-base deletion (error_count.cpp:934-956) or insertion (:963-982) after a run's last base.
__device__ __forceinline__ void ec_run_indel(const EcParams& P, const uint8_t* sq, const uint8_t* ql, const DRead& R,
                                             int x, int y, int len, int last_indel, uint32_t row0, const EcTable& T,
                                             uint32_t& err) {
  const uint32_t Q = (uint32_t)P.quality_max;
  const bool rev = (R.flags & kReadReversed) != 0;
  const int last = y + len - 1;
  if (last_indel == -1) {
    if (!rev && last + 1 >= (int)R.l_qseq) {
      err |= kErrQueryIndex;
      return;
    }
    const uint32_t b = sq[rev ? last : last + 1], q = ql[rev ? last : last + 1];
    const uint32_t r = P.ref_idx[x + len];
    if (b == 15u || r == kRefN) return;
    const uint32_t rd = ((rev ? kRefLutRev : kRefLutFwd) >> (4u * r)) & 15u;
    if (rd > 4u) err |= kErrRefChar;
    else if (q >= Q) err |= kErrQuality;
    else if (rd == 4u) atomicAdd(&T.pairs[row0 + q], 1);   // the bin of the pairs
    else T.add(row0 + q, rd, 4u);
  } else if (last_indel == 1) {
    const int mq = last + 1;
    if (mq >= (int)R.l_qseq) {
      err |= kErrQueryIndex;
      return;
    }
    if (mq > (int)R.qe0 || mq < (int)R.qs0) return;
    const uint32_t b = sq[mq], q = ql[mq];
    if (b == 15u) return;
    const uint32_t oi = (b > 15u) ? 15u : (uint32_t)((rev ? kReadLutRev : kReadLutFwd) >> (4u * b)) & 15u;
    if (oi > 3u) err |= kErrBaseCode;
    else if (q >= Q) err |= kErrQuality;
    else T.add(row0 + q, 4u, oi);
  }
}

// What bounds it: 4.6 Mb at 100x of 150-base reads needs 1.0 GB and moves 1.8 GB in 360 us, 5.1 TB/s, the
// rate of a large copy (a run's ends are read a second time, by ec_run_pairs, when their lines have left the
// L2), with the vector unit about 60% busy (17 instructions a position, 125 M in all) and the LDS 30%
// (one atomic a position).  One alignment of up to 168 bases to 21 lanes, position-wise selects and an atomic each
// for the base and its pair took 409 M instructions and 871 us; alignments with an indel went one at a
// time, and a wavefront whose alignments all cross one took 165 us alone.  Measured before -> now, in
// us: 2.05 Mb at 83x of 36 bases (five of 21 lanes had work) 1166 -> 226, 48 kb at 206x of 100 bases
// 165 -> 29, 701 kb at 57x of 300 bases (one alignment at a time) 248 -> 63, 1 Mb at 300x 553 -> 259,
// 20 kb at 3,000x 137 -> 82 (the difference array's atomics, hence add_equal).  64 alignments a work
// item rather than 32: the loads before the items (record, target) are paid once for twice the items.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) k_ec_reads(EcParams P) {
  extern __shared__ uint32_t ec_lds[];
  // A run as the lanes that share it read it, in terms of the wavefront's item number i (eight
  // positions each, the runs' items one after the other): first byte at + 8 i, its column col + 8 i,
  // and the bytes from begin - 8 i to end - 8 i in the run: {at, col, end, begin * 2 + reversed}.
  __shared__ uint4 ec_rec[kEcWaves][kEcChunk];
  __shared__ uint32_t ec_row[kEcWaves][kEcChunk];
  __shared__ uint32_t ec_first[kEcWaves][2 * kEcSteps];   // bit i: item i is its run's first
  const int S = P.read_set_max, Q = P.quality_max, rows = S * Q;
  const EcTable T{ec_lds, (int32_t*)(ec_lds + (size_t)rows * kEcRow)};
  for (int i = threadIdx.x; i < rows * (int)(kEcRow + 1); i += blockDim.x) ec_lds[i] = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t gw = ((int64_t)xcd_major_block() * blockDim.x + threadIdx.x) >> 6;
  const int64_t nw = ((int64_t)gridDim.x * blockDim.x) >> 6;
  uint32_t err = 0;
  for (int64_t c0 = gw * kEcChunk; c0 < P.n_reads; c0 += nw * kEcChunk) {
    // Lane i takes alignment i and steps through its M/=/X runs; the runs that the lanes are at
    // become items of eight positions, which the wavefront's lanes share evenly whatever the runs'
    // lengths (the counts are integers, so the order does not matter).  A run longer than
    // kEcReadItems items takes several turns.
    const DRead* rp = P.reads + c0 + lane;
    bool live = false, count = false;   // more to come; its bases are counted
    int k = 0;                          // next CIGAR operation
    int cx = 0, cy = 0;                 // column and query position at it
    int x = 0, y = 0, len = 0, left = 0;   // the run, and how much of it is still to be counted
    if (c0 + lane < P.n_reads) {
      const DRead R = *rp;
      const int t = P.pos_target[R.gpos];
      live = t >= 0 && P.target_scored[t];
      count = live && R.x1 <= 1 && P.do_errors;
      if (count && (int)R.rfile >= S) {   // covariate read_set out of range: ASSERT in the reference
        err |= kErrReadSet;
        count = false;
      }
      cx = R.gpos;
      if (R.flags & kReadSimple) {
        k = -1;
        cy = R.y0;
      }
    }
    while (__any(live)) {
      bool fresh = false;
      int last_indel = 0;
      if (live && left == 0) {   // the next run
        if (k < 0) {
          x = cx;
          y = cy;
          len = rp->gend - x;
          fresh = true;
        } else {
          const int n = rp->n_cigar;
          const uint32_t* c = P.cigar + rp->cig_off;
          for (; k < n && !fresh; k++) {
            const uint32_t op = c[k] & 15u;
            const int l = (int)(c[k] >> 4);
            if (op == OP_M || op == OP_EQ || op == OP_X) {
              if (l > 0) {
                x = cx;
                y = cy;
                len = l;
                last_indel = run_end_indel(c, k, n);
                fresh = true;
              }
              cx += l;
              cy += l;
            } else if (op == OP_I || op == OP_S) {
              cy += l;
            } else if (op == OP_D || op == OP_N) {
              cx += l;
            }
          }
          if (!fresh) {
            live = false;
            if (cx != rp->gend) err |= kErrCigar;
          }
        }
        left = (fresh && count) ? len : 0;
      }
      const int py = y + len - left;   // query position of the part still to be counted
      const int items = min(((py & 7) + left + 7) >> 3, left > 0 ? kEcReadItems : 0);
      const int part = (items > 0) ? min(left, 8 * items - (py & 7)) : 0;
      const int incl = wave_incl_scan(items);
      const int total = __builtin_amdgcn_readlane(incl, 63);
      if (total > 0) {
        for (int i = lane; i < 2 * kEcSteps; i += 64) ec_first[wave][i] = 0;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        if (items > 0) {
          const int start = incl - items;
          const int at = __popcll(__ballot(true) & ((1ull << lane) - 1ull));
          const int begin = (py & 7) + 8 * start;
          ec_rec[wave][at] = make_uint4((uint32_t)rp->seq_off + (uint32_t)(py & ~7) - 8u * (uint32_t)start,
                                        (uint32_t)(x + (py - y) - begin), (uint32_t)(begin + part),
                                        ((uint32_t)begin << 1) | ((rp->flags & kReadReversed) ? 1u : 0u));
          ec_row[wave][at] = (uint32_t)rp->rfile * (uint32_t)Q;
          atomicOr(&ec_first[wave][start >> 5], 1u << (start & 31));
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        struct Item {
          uint2 b, q, r;
          int lo, hi;
          uint32_t rev, row;
        };
        int before = -1;   // runs whose items start before the step, less one
        auto fetch = [&](int i0) {
          Item it;
          const uint32_t f0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)ec_first[wave][i0 >> 5]);
          const uint32_t f1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)ec_first[wave][(i0 >> 5) + 1]);
          const uint64_t f = ((uint64_t)f1 << 32) | f0, g = f >> 1;
          const int id = before + (int)(f0 & 1u) +
                         (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(g >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)g, 0u));
          before += __popcll(f);
          const int i = i0 + lane;
          it.hi = 0;
          if (i < total) {
            const uint4 rec = ec_rec[wave][id];
            it.row = ec_row[wave][id];
            const uint32_t at = rec.x + 8u * (uint32_t)i;
            it.b = *(const uint2*)(P.bases + at);
            it.q = *(const uint2*)(P.quals + at);
            it.r = load8(P.ref_idx + ((int)rec.y + 8 * i));   // from 7 columns before the run on; ref_idx is padded
            it.lo = ((int)rec.w >> 1) - 8 * i;
            it.hi = (int)rec.z - 8 * i;
            it.rev = rec.w & 1u;
          }
          return it;
        };
        auto add = [&](const Item& it) {
          if (it.hi > 0) ec_eight(it.b, it.q, it.r, it.lo, it.hi, it.rev != 0u, it.row, (uint32_t)Q, T, err);
        };
        Item a = fetch(0);
        for (int i0 = 64; i0 < total; i0 += 64) {   // the next items' bytes are on the way while one is counted
          const Item b = fetch(i0);
          add(a);
          a = b;
        }
        add(a);
      }
      left -= part;
      // the difference array and the run's ends come last: the loads above would wait for these atomics
      const int array = (fresh && rp->x1 > 1) ? P.n_pos + 1 : 0;
      add_equal(P.cov_diff, fresh ? array + x : -1, 1);
      add_equal(P.cov_diff, fresh ? array + x + len : -1, -1);
      if (fresh && count) {
        const DRead R = *rp;
        const uint8_t* sq = P.bases + R.seq_off;
        const uint8_t* ql = P.quals + R.seq_off;
        const uint32_t row0 = (uint32_t)R.rfile * (uint32_t)Q;
        ec_run_pairs(P, sq, ql, (R.flags & kReadReversed) != 0, x, y, len, last_indel, (int)R.qe0, row0, T, err);
        ec_run_indel(P, sq, ql, R, x, y, len, last_indel, row0, T, err);
      }
      if (k < 0 && left == 0) live = false;   // a single run, counted
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  __syncthreads();
  // bin of (read set rs, reference class ri, observed class oi, quality q): rs + S*(ri + 5*oi + 25*q)
  for (int i = threadIdx.x; i < P.n_bins; i += blockDim.x) {
    const int row = i / (int)kEcRow, c = i - row * (int)kEcRow;
    const int rs = row / Q, q = row - rs * Q;
    long long v;
    if (c == 24) {
      v = T.pairs[row];
      for (int oi = 0; oi < 4; oi++)
        for (int ri = 0; ri < 4; ri++) v += T.bins[row * (int)kEcRow + ri + 5 * oi];
    } else {
      v = T.bins[i];
    }
    if (v) atomicAdd(&P.counts[rs + S * (c + 25 * q)], (unsigned long long)v);
  }
  if (err) atomicOr(P.err, err);
}

/* ------------------------------------------------------------------------------------------ */
/* Preprocess mode: where qualifying reads start                                               */

// One thread per alignment: a unique alignment of a scored target whose first query base is
// aligned (nothing but deletions, skips, hard clips or pads before its first M/=/X run) marks its
// strand's bit at that column when its stranded aligned end (query_stranded_end_1 over
// query_bounds_1: soft clips, hard clips and skips at either end excluded; alignment.cpp:120-239)
// reaches required_junction_read_end_min_coordinate(read length) (settings.h:345-354).  The
// pileup entry there has query_position_1 == 1 (error_count.cpp:159-166).
__global__ void __launch_bounds__(256) k_read_starts(EcParams P) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.n_reads) return;
  const DRead R = P.reads[i];
  const int t = P.pos_target[R.gpos];
  if (t < 0 || !P.target_scored[t] || R.x1 > 1) return;
  const uint32_t* c = P.cigar + R.cig_off;
  const int n = R.n_cigar;
  int x = R.gpos, col = -1;
  for (int k = 0; k < n; k++) {
    const uint32_t op = c[k] & 15u;
    const int l = (int)(c[k] >> 4);
    if (op == OP_M || op == OP_EQ || op == OP_X) {
      if (l > 0) col = x;
      break;
    }
    if (op == OP_I || op == OP_S) break;   // a query base comes first
    if (op == OP_D || op == OP_N) x += l;
  }
  if (col < 0) return;
  uint32_t start1 = 1, qlen = 0;
  for (int k = 0; k < n; k++) {
    const uint32_t op = c[k] & 15u;
    if (op == OP_M || op == OP_I || op == OP_S || op == OP_EQ || op == OP_X) qlen += c[k] >> 4;
  }
  for (int k = 0; k < n; k++) {
    const uint32_t op = c[k] & 15u;
    if (op != OP_S && op != OP_H && op != OP_N) break;
    if (op == OP_S) start1 += c[k] >> 4;
  }
  uint32_t end1 = qlen;
  for (int k = n - 1; k > 0; k--) {
    const uint32_t op = c[k] & 15u;
    if (op != OP_S && op != OP_H && op != OP_N) break;
    if (op == OP_S) end1 -= c[k] >> 4;
  }
  const bool rev = (R.flags & kReadReversed) != 0;
  const uint32_t rl = R.l_qseq;
  const uint32_t stranded_end = rev ? rl - start1 + 1u : end1;
  const int32_t m = (int32_t)floor((double)((int32_t)rl - (int32_t)P.end_min_len) * P.end_factor);
  const uint32_t need = (m <= 0) ? rl : rl - (uint32_t)m;
  if (stranded_end >= need) atomicOr(&P.start_bits[col >> 4], 1u << ((col & 15) * 2 + (rev ? 1 : 0)));
}

/* ------------------------------------------------------------------------------------------ */
/* Coverage histogram: prefix scan of the difference arrays                                    */

__global__ void __launch_bounds__(256) k_cov_tile_sums(CovParams C) {
  __shared__ int red[2][4];
  const int64_t n = (int64_t)C.n_pos + 1;
  const int64_t base = (int64_t)blockIdx.x * kCovTile;
  const int32_t* du = C.cov_diff;
  const int32_t* dr = C.cov_diff + n;
  int su = 0, sr = 0;
#pragma unroll 4
  for (int i = 0; i < kCovTile / 256; i++) {
    const int64_t idx = base + i * 256 + threadIdx.x;
    if (idx < n) {
      su += du[idx];
      sr += dr[idx];
    }
  }
  su = wave_sum(su);
  sr = wave_sum(sr);
  const int wv = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[0][wv] = su;
    red[1][wv] = sr;
  }
  __syncthreads();
  if (threadIdx.x == 0) C.tile_sum[blockIdx.x] = make_int2(red[0][0] + red[0][1] + red[0][2] + red[0][3],
                                                           red[1][0] + red[1][1] + red[1][2] + red[1][3]);
}

// One block of 1024 threads: tile_sum becomes the exclusive prefix of the tile sums.
__global__ void __launch_bounds__(1024) k_cov_tile_scan(CovParams C) {
  __shared__ int wsum[2][16];
  __shared__ int carry[2];
  if (threadIdx.x == 0) carry[0] = carry[1] = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int b0 = 0; b0 < C.n_tiles; b0 += 1024) {
    const int b = b0 + threadIdx.x;
    const int2 v = (b < C.n_tiles) ? C.tile_sum[b] : make_int2(0, 0);
    const int iu = wave_incl_scan(v.x), ir = wave_incl_scan(v.y);
    if (lane == 63) {
      wsum[0][wv] = iu;
      wsum[1][wv] = ir;
    }
    __syncthreads();
    int ou = carry[0], orr = carry[1];
    for (int k = 0; k < wv; k++) {
      ou += wsum[0][k];
      orr += wsum[1][k];
    }
    if (b < C.n_tiles) C.tile_sum[b] = make_int2(ou + iu - v.x, orr + ir - v.y);
    __syncthreads();
    if (threadIdx.x == 1023) {
      carry[0] = ou + iu;
      carry[1] = orr + ir;
    }
    __syncthreads();
  }
}

__global__ void __launch_bounds__(256) k_cov_hist(CovParams C) {
  extern __shared__ uint32_t hist[];   // n_groups_lds * hist_lds
  __shared__ int wtot[2][4];
  __shared__ int st_block;                 // preprocess mode: the target whose counts the block adds up
  __shared__ uint32_t st_sum[2];
  if (threadIdx.x == 0) {
    st_block = -1;
    st_sum[0] = st_sum[1] = 0;
  }
  const int nh = C.n_groups_lds * C.hist_lds;
  for (int i = threadIdx.x; i < nh; i += blockDim.x) hist[i] = 0;
  const int64_t n = (int64_t)C.n_pos + 1;
  const int64_t c0 = (int64_t)blockIdx.x * kCovTile + (int64_t)threadIdx.x * 16;
  const int32_t* du = C.cov_diff;
  const int32_t* dr = C.cov_diff + n;
  int pu[16], pr[16];
  int su = 0, sr = 0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int64_t idx = c0 + i;
    const int a = (idx < n) ? du[idx] : 0;
    const int b = (idx < n) ? dr[idx] : 0;
    su += a;
    sr += b;
    pu[i] = su;
    pr[i] = sr;
  }
  // exclusive prefix of the thread totals within the block
  const int iu = wave_incl_scan(su), ir = wave_incl_scan(sr);
  const int wv = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 63) {
    wtot[0][wv] = iu;
    wtot[1][wv] = ir;
  }
  __syncthreads();
  const int2 tile = C.tile_sum[blockIdx.x];
  int ou = tile.x + iu - su, orr = tile.y + ir - sr;
  for (int k = 0; k < wv; k++) {
    ou += wtot[0][k];
    orr += wtot[1][k];
  }
  uint32_t err = 0;
  // preprocess mode: (position, strand) pairs without / with a qualifying start, per target
  int st_t = -1;
  uint32_t st_none = 0, st_some = 0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int64_t col = c0 + i;
    if (col >= C.n_pos) break;
    const int t = C.pos_target[col];
    if (t < 0 || !C.target_scored[t]) continue;
    const int cu = ou + pu[i], cr = orr + pr[i];
    if (cr != 0) continue;   // a redundant read covers the column (error_count.cpp:172-175)
    const int g = C.target_group[t];
    if (g < C.n_groups_lds && cu < C.hist_lds) atomicAdd(&hist[g * C.hist_lds + cu], 1u);
    else if (cu >= 0 && cu < C.hist_len) atomicAdd(&C.hist[(int64_t)g * C.hist_len + cu], 1ull);
    else err |= kErrCapacity;
    if (C.start_bits) {
      if (t != st_t) {
        if (st_t >= 0) {
          atomicAdd(&C.start_counts[2 * st_t], (unsigned long long)st_none);
          atomicAdd(&C.start_counts[2 * st_t + 1], (unsigned long long)st_some);
        }
        st_t = t;
        st_none = st_some = 0;
      }
      const uint32_t b = (C.start_bits[col >> 4] >> ((col & 15) * 2)) & 3u;
      const uint32_t some = (b & 1u) + (b >> 1);
      st_some += some;
      st_none += 2u - some;
    }
  }
  if (C.start_bits) {
    // The counts of all threads go to two words per target.  One 64-bit atomic per thread on them
    // serialized the kernel (2.47 ms on a 2.3 Mb target against 0.03 ms): the block adds up the
    // highest target among its threads' last ones in LDS first, by wavefronts, and adds it once.
    // Threads of other targets (a block of many short targets) add their own.
    if (st_t >= 0) atomicMax(&st_block, st_t);
    __syncthreads();
    const bool mine = st_t >= 0 && st_t == st_block;
    const int none = wave_sum(mine ? (int)st_none : 0), some = wave_sum(mine ? (int)st_some : 0);
    if ((threadIdx.x & 63) == 0) {
      atomicAdd(&st_sum[0], (uint32_t)none);
      atomicAdd(&st_sum[1], (uint32_t)some);
    }
    if (st_t >= 0 && !mine) {
      atomicAdd(&C.start_counts[2 * st_t], (unsigned long long)st_none);
      atomicAdd(&C.start_counts[2 * st_t + 1], (unsigned long long)st_some);
    }
  }
  __syncthreads();
  if (C.start_bits && threadIdx.x < 2 && st_block >= 0)
    atomicAdd(&C.start_counts[2 * st_block + threadIdx.x], (unsigned long long)st_sum[threadIdx.x]);
  for (int i = threadIdx.x; i < nh; i += blockDim.x) {
    if (hist[i]) {
      const int g = i / C.hist_lds, c = i % C.hist_lds;
      atomicAdd(&C.hist[(int64_t)g * C.hist_len + c], (unsigned long long)hist[i]);
    }
  }
  if (err) atomicOr(C.err, err);
}

}  // namespace bsq
