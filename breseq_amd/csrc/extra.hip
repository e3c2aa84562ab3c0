// extra.hip -- per-position reference trims on the GPU (SequenceTrims, calculate_trims.cpp:67-138).
//
// The reference scans each position for perfect tandem repeats of unit 1..18 and max-scatters the
// resulting trim lengths forward.  Here a block takes kTrimTile positions and turns the scatter into a
// prefix maximum: with m[p] the maximal repeat extent at p (at most 255) and M[x] the maximum of p + m[p]
// over p <= x,
//   left[x]  = max over p <= x of (m[p] - (x - p)) = M[x] - x
//   right[x] = max over p <= x with p + m[p] > x of (x - p + 1), whose p is the first with M[p] > x.
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>
#include <vector>

#include "device_common.h"
#include "engine.h"
#include "host_util.h"
#include "kernels.h"

namespace bsq {

// Device memory of bsq_sequence_trims_static, for callers that cannot allocate: the sequence and the
// two trim rows of a sequence of up to kStaticTrimsMax bases (3 bytes per base, 24 MiB).  Every GPU the library runs this entry point on holds its own copy until the
// process ends.  Host code never uses the array's name as an address: each device's copy is found
// once with hipGetSymbolAddress (scratch_on_device) and only that pointer reaches kernels and copies.
constexpr int64_t kStaticTrimsMax = (int64_t)8 << 20;
static __device__ __align__(256) uint8_t scratch[3 * kStaticTrimsMax];

static std::mutex g_scratch_mu;
static std::vector<uint8_t*> g_scratch_ptr;   // per device id

// Address of `scratch` on the current device, looked up on the first call on that device.
static uint8_t* scratch_on_device() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) throw BsqError(BSQ_ERR_DEVICE, "no current HIP device");
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if ((int)g_scratch_ptr.size() <= dev) g_scratch_ptr.resize((size_t)dev + 1, nullptr);
  if (!g_scratch_ptr[(size_t)dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      throw BsqError(BSQ_ERR_DEVICE, std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
    g_scratch_ptr[(size_t)dev] = (uint8_t*)p;
  }
  return g_scratch_ptr[(size_t)dev];
}

constexpr int kTrimBack = 256;                  // positions before them whose extents reach them (m <= 255)
constexpr int kTrimUnits = 18;                  // longest repeat unit
constexpr int kTrimWords = (kTrimBack + kTrimTile + 256) / 64;
constexpr int kTrimBytes = kTrimWords * 64 + kTrimUnits;

// The trims of the sequence s[0, len).  A repeat of unit u at p is a run of positions with
// s[i] == s[i + u] from p on: the comparisons of 64 positions make a 64-bit word (a ballot), and the run
// is the word's trailing ones, for most positions without a look at the next word.  A thread per
// position that compared bytes, and one that looked back over 255 extents, took 735 and 425 us for
// 4.6 Mb; this takes 104 us, bound by the 18 units' vector work a position.
__global__ void __launch_bounds__(256) k_sequence_trims(const char* __restrict__ s, int64_t len,
                                                        uint8_t* __restrict__ left_out, uint8_t* __restrict__ right_out) {
  __shared__ char seq[kTrimBytes];
  __shared__ uint64_t same[kTrimUnits][kTrimWords];   // bit i of word w: s[i] == s[i + unit], position 64 w + i
  __shared__ int reach[kTrimBack + kTrimTile];        // p + m[p], then its prefix maximum
  __shared__ int wave_max[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t g0 = (int64_t)blockIdx.x * kTrimTile - kTrimBack;   // position of index 0
  const int begin = (g0 < 0) ? (int)-g0 : 0;                        // indices [begin, end) are in the sequence
  const int end = (int)min<int64_t>(len - g0, kTrimBytes);
  for (int i = tid; i < kTrimBytes; i += 256) seq[i] = (i >= begin && i < end) ? s[g0 + i] : 0;
  __syncthreads();
  for (int w = wave; w < kTrimWords; w += 4) {
    const int i = 64 * w + lane;
    const char c = seq[i];
    uint64_t mine = 0;
#pragma unroll
    for (int u = 1; u <= kTrimUnits; u++) {
      const uint64_t eq = __ballot(c == seq[i + u] && i >= begin && i + u < end);
      if (lane == u - 1) mine = eq;
    }
    if (lane < kTrimUnits) same[lane][w] = mine;
  }
  __syncthreads();
  for (int i = tid; i < kTrimBack + kTrimTile; i += 256) {
    int m = 0;
    if (i >= begin && i < end) {
      m = 1;
      const int w = i >> 6, b = i & 63;
#pragma unroll
      for (int u = 1; u <= kTrimUnits; u++) {
        const uint64_t x = ~(same[u - 1][w] >> b);
        int run = x ? __builtin_ctzll(x) : 64;
        if (run >= 64 - b) {   // to the word's end
          run = 64 - b;
          for (int v = w + 1; run < 256 && v < kTrimWords; v++) {
            const uint64_t y = ~same[u - 1][v];
            run += y ? __builtin_ctzll(y) : 64;
            if (y) break;
          }
        }
        if (run >= u) m = max(m, (run / u + 1) * u);
      }
      m = min(m, 255);
    }
    reach[i] = i + m;
  }
  __syncthreads();
  // prefix maximum: five consecutive positions a thread
  constexpr int kEach = (kTrimBack + kTrimTile) / 256;
  int v[kEach], top = 0;
#pragma unroll
  for (int k = 0; k < kEach; k++) {
    top = max(top, reach[tid * kEach + k]);
    v[k] = top;
  }
  int incl = top;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(incl, o, 64);
    if (lane >= o) incl = max(incl, y);
  }
  if (lane == 63) wave_max[wave] = incl;
  int before = __shfl_up(incl, 1, 64);
  if (lane == 0) before = 0;
  __syncthreads();
  for (int k = 0; k < wave; k++) before = max(before, wave_max[k]);
#pragma unroll
  for (int k = 0; k < kEach; k++) reach[tid * kEach + k] = max(before, v[k]);
  __syncthreads();
  for (int x = kTrimBack + tid; x < min(end, kTrimBack + kTrimTile); x += 256) {
    int lo = x - 255, hi = x;   // the first index with reach > x lies in (lo, hi]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (reach[mid] > x) hi = mid;
      else lo = mid;
    }
    left_out[g0 + x] = (uint8_t)(reach[x] - x);
    right_out[g0 + x] = (uint8_t)(x - hi + 1);
  }
}

// BAM code -> the character breseq compares (basebam2char, common.h:263-275): A C G T, else N
__device__ __forceinline__ char trim_char(uint8_t b) {
  switch (b) {
    case 1: return 'A';
    case 2: return 'C';
    case 4: return 'G';
    case 8: return 'T';
    default: return 'N';
  }
}

// Eight bases from `s` on in read direction (or backwards from s[7] on), four bits each.
template <bool kBack>
__device__ __forceinline__ uint32_t eight_bases(const uint8_t* s, uint32_t& odd) {
  uint64_t w;
  __builtin_memcpy(&w, s, 8);   // one load; the hardware takes any alignment
  if (kBack) w = __builtin_bswap64(w);
  const uint32_t a = (uint32_t)w, b = (uint32_t)(w >> 32);
  odd |= not_bases(a) | not_bases(b);
  const uint32_t x = (a | (a >> 4)) & 0x00FF00FFu, y = (b | (b >> 4)) & 0x00FF00FFu;
  return ((x | (x >> 8)) & 0xFFFFu) | ((y | (y >> 8)) << 16);
}

// The longest perfect tandem repeat of unit 1..18 at the start of s[0, len) (kBack: of the reversed
// sequence), at least 1: repeat_match(seq, 0, unit, num) (calculate_trims.cpp:44-56).  A repeat of unit u is a
// run of positions i with s[i] == s[i + u] from 0 on, found for all units in the first 32 bases, four
// bits each, as the trailing zeros of the words XORed with themselves shifted; a run that reaches the
// words' end, and bases beyond A, C, G, T and N, are compared one by one.  400,000 alignments take
// 23 us, where comparing bytes one by one took 226.
template <bool kBack>
__device__ __forceinline__ uint32_t edge_trim(const uint8_t* s, int len) {
  uint32_t odd = (len < 32) ? 1u : 0u, n[4];
  if (!odd) {
#pragma unroll
    for (int k = 0; k < 4; k++) n[k] = eight_bases<kBack>(kBack ? s + len - 8 - 8 * k : s + 8 * k, odd);
  }
  uint32_t best = 1;
  if (!odd) {
    const uint64_t lo = ((uint64_t)n[1] << 32) | n[0], hi = ((uint64_t)n[3] << 32) | n[2];
    const unsigned __int128 w = ((unsigned __int128)hi << 64) | lo;
#pragma unroll
    for (int u = 1; u <= 18; u++) {
      const unsigned __int128 x = w ^ (w >> (4 * u));
      const uint64_t x0 = (uint64_t)x, x1 = (uint64_t)(x >> 64);
      const int run = (x0 ? __builtin_ctzll(x0) : x1 ? 64 + __builtin_ctzll(x1) : 128) >> 2;
      if (run >= 32 - u) odd = 1u;   // it may go on
      else if (run >= u) best = max(best, (uint32_t)((run / u + 1) * u));
    }
  }
  if (odd) {
    best = 1;
    for (int u = 1; u <= 18; u++) {
      int run = 0;
      while (run + u < len && trim_char(kBack ? s[len - 1 - run] : s[run]) ==
                                  trim_char(kBack ? s[len - 1 - run - u] : s[run + u]))
        run++;
      if (run >= u) best = max(best, (uint32_t)((run / u + 1) * u));
    }
  }
  return best;
}

// get_alignment_trims (calculate_trims.cpp:239-285) of every packed alignment, one thread each:
//   the genomic trims at the alignment's first and last reference positions, the read-edge trims
//   of its aligned sequence (edge_trims_for_sequence, :183-230: the longest perfect tandem repeat of
//   unit 1..18 starting at either end, at least 1), the larger of each pair, plus the bases outside
//   the match (query_start_0 on the left, read length - query_end_1 on the right; soft clips only,
//   alignment.cpp:248-289).  A repeat compared on the reverse complement matches exactly where the
//   reversed sequence does (complementing is a bijection on A, C, G, T, N), so the right edge reads
//   the sequence backwards.  left/right: the sample's per-column trims (global columns).
__global__ void __launch_bounds__(256) k_alignment_trims(const DRead* __restrict__ reads, int64_t n,
                                                         const uint32_t* __restrict__ cigar,
                                                         const uint8_t* __restrict__ bases,
                                                         const uint8_t* __restrict__ left, const uint8_t* __restrict__ right,
                                                         int32_t* __restrict__ xl, int32_t* __restrict__ xr) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const DRead R = reads[i];
  const uint32_t* c = cigar + R.cig_off;
  const int nc = R.n_cigar;
  uint32_t qs1 = 1, qlen = 0;
  for (int k = 0; k < nc; k++) {
    if ((c[k] & 15u) != 4u) break;
    qs1 += c[k] >> 4;
  }
  for (int k = 0; k < nc; k++) {
    const uint32_t op = c[k] & 15u;
    if (op == 0 || op == 1 || op == 4 || op == 7 || op == 8) qlen += c[k] >> 4;
  }
  uint32_t qe1 = qlen;
  for (int k = nc - 1; k > 0; k--) {
    if ((c[k] & 15u) != 4u) break;
    qe1 -= c[k] >> 4;
  }
  const uint8_t* s = bases + R.seq_off + (qs1 - 1);
  const int len = (qe1 >= qs1) ? (int)(qe1 - qs1 + 1) : 0;
  const uint32_t eL = edge_trim<false>(s, len), eR = edge_trim<true>(s, len);
  const uint32_t gL = left[R.gpos], gR = right[R.gend - 1];
  xl[i] = (int32_t)(max(gL, eL) + (qs1 - 1));
  xr[i] = (int32_t)(max(gR, eR) + (R.l_qseq - qe1));
}

}  // namespace bsq

using namespace bsq;

extern "C" int bsq_sequence_trims(const char* seq, int64_t len, uint8_t* out, bsq_status* status) {
  char* d_s = nullptr;
  uint8_t* d_o = nullptr;
  auto cleanup = [&]() {
    if (d_s) (void)hipFree(d_s);
    if (d_o) (void)hipFree(d_o);
  };
  try {
    if (!seq || !out || len < 0) throw BsqError(BSQ_ERR_ARG, "bad arguments");
    if (len == 0) {
      set_status(status, BSQ_OK, "");
      return BSQ_OK;
    }
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) throw BsqError(BSQ_ERR_DEVICE, "no HIP device available");
    if (hipMalloc((void**)&d_s, (size_t)len) != hipSuccess || hipMalloc((void**)&d_o, 2 * (size_t)len) != hipSuccess)
      throw BsqError(BSQ_ERR_DEVICE, "hipMalloc failed");
    if (hipMemcpy(d_s, seq, (size_t)len, hipMemcpyHostToDevice) != hipSuccess) throw BsqError(BSQ_ERR_DEVICE, "copy failed");
    hipLaunchKernelGGL(k_sequence_trims, dim3((unsigned)((len + kTrimTile - 1) / kTrimTile)), dim3(256), 0, 0, d_s, len, d_o,
                       d_o + len);
    if (hipGetLastError() != hipSuccess) throw BsqError(BSQ_ERR_DEVICE, "kernel launch failed");
    if (hipMemcpy(out, d_o, 2 * (size_t)len, hipMemcpyDeviceToHost) != hipSuccess) throw BsqError(BSQ_ERR_DEVICE, "copy failed");
    cleanup();
    set_status(status, BSQ_OK, "");
    return BSQ_OK;
  } catch (const BsqError& e) {
    cleanup();
    set_status(status, e.code, e.what());
    return e.code;
  }
}

// The trims of bsq_sequence_trims with no device allocation: input and output live in this device's
// `scratch` (sequences of at most kStaticTrimsMax bases).  Every byte read was written before, so
// nothing needs clearing between calls.  Calls that overlap on one
// GPU share the array and race.
extern "C" int bsq_sequence_trims_static(const char* seq, int64_t len, uint8_t* out, bsq_status* status) {
  try {
    if ((!seq || !out) && len > 0) throw BsqError(BSQ_ERR_ARG, "bad arguments");
    if (len < 0) throw BsqError(BSQ_ERR_ARG, "negative length");
    if (len > kStaticTrimsMax)
      throw BsqError(BSQ_ERR_LIMIT, "sequence of " + std::to_string(len) + " bases exceeds the " +
                                        std::to_string(kStaticTrimsMax) + "-base capacity of the allocation-free trims");
    if (len == 0) {
      set_status(status, BSQ_OK, "");
      return BSQ_OK;
    }
    uint8_t* base = scratch_on_device();
    char* d_s = (char*)base;
    uint8_t* d_o = base + kStaticTrimsMax;   // 2 * len bytes: left row, then right row
    if (hipMemcpy(d_s, seq, (size_t)len, hipMemcpyHostToDevice) != hipSuccess) throw BsqError(BSQ_ERR_DEVICE, "copy failed");
    hipLaunchKernelGGL(k_sequence_trims, dim3((unsigned)((len + kTrimTile - 1) / kTrimTile)), dim3(256), 0, 0, d_s, len, d_o,
                       d_o + len);
    if (hipGetLastError() != hipSuccess) throw BsqError(BSQ_ERR_DEVICE, "kernel launch failed");
    if (hipMemcpy(out, d_o, 2 * (size_t)len, hipMemcpyDeviceToHost) != hipSuccess) throw BsqError(BSQ_ERR_DEVICE, "copy failed");
    set_status(status, BSQ_OK, "");
    return BSQ_OK;
  } catch (const BsqError& e) {
    set_status(status, e.code, e.what());
    return e.code;
  }
}
