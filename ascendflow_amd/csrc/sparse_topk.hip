// Top-k index selection for sparse MLA on gfx950: the step that produces
// cmp_sparse_indices from per-token index scores over compressed positions.
//
// The reference takes cmp_sparse_indices as an input and leaves its producer
// (the top-k indexer) to the caller (docs/operators/sparse-mla.md:8,266). Its
// contract for the tensor is fixed, though: token t of request b may select
// compressed positions in [0, cutoff), cutoff = max(0, C_b R + r_b - n + j + 1)
// / R, at most min(TOPK, C_b, cutoff) of them, ascending, -1 after
// (docs/operators/sparse-mla.md:41-51,79; examples/sparse_attention/attention.py:339-341).
// These kernels take a score per (token, compressed position) and write, for
// every token, the min(TOPK, C_b, cutoff) positions of largest score among
// [0, cutoff), ties to the lower position, in ascending order.
//
// The selection works on a monotonic 32-bit key of each score. Three kernels:
// sparse_topk_row keeps a row in registers (calls of few tokens, rows up to 32K
// positions; longer ones split into segments and merged), described at its
// definition; the other two stream a row per workgroup. sparse_topk_filter (rows up
// to 256K positions; 256 threads up to 32K positions, 1024 beyond):
//   1. sample: four keys per thread (two in the 1024-thread form: 2048
//      keys), in blocks of 16 consecutive positions
//      evenly spaced over the row (issued with the request lookup, over the
//      whole allocated row, and kept when the token's candidates cover at
//      least half of it; shorter rows are sampled again over their
//      candidates); one histogram of the sample, linear in the score over its
//      range, or a two-digit radix selection (the 1024-thread form, and
//      samples with no usable range), gives an estimate of the threshold, taken at 1.25x the expected rank plus 8 (256 threads) or
//      twice it plus 16 (1024), so that somewhat more than `take` keys reach
//      it;
//   2. filter: one streaming pass over the row (16-byte loads, several in
//      flight per thread) appends every key >= estimate, with its position,
//      to an LDS buffer (wave ballots, one LDS atomic per wave and step);
//   3. exact selection over the buffer: one linear histogram and a ranking of
//      the few keys in the bin of the take-th, or a radix selection (digits of
//      11, 11 and 10 bits; the 1024-thread form, and fuller bins), giving the
//      threshold key and how many keys equal to it are taken (linear instead
//      of radix: 4096 rows of 16391 83.5 -> 78.6 us, 8192 of 16K 133.9 ->
//      127.4, 4096 of 4K 35.2 -> 32.7); if fewer than `take` keys reached the estimate,
//      or the buffer overflowed, the row is filtered again at another sample
//      rank (binary search, up to four passes), and failing that the same
//      selection runs over the whole row, re-reading it per digit (same
//      result, slower);
//   4. output: keys above the threshold, and keys equal to it, set bits in two
//      LDS bitmaps over the row's positions; one scan of the bitmaps writes
//      the positions in ascending order, taking the first `need` equal keys.
// The row is read once from HBM on the common path. sparse_topk_stream
// serves longer rows: every digit, and the output, re-read the row.
#include <algorithm>

#include "common.h"
#include "../../include/ascendflow_amd.h"

namespace afa {

constexpr int TK_BINS = 2048;  // widest digit: 11 bits
constexpr int TK_UNROLL = 4;    // 4-position groups in flight per thread in a streaming pass
constexpr int TK_FILTER_ROUNDS = 4;  // filter passes before the whole-row selection
// Sample keys per thread for the threshold estimate: 4 x 256 = 1024 keys in
// the 256-thread form, whose buffer of 2 TOPK entries needs the closer
// estimate; 2 x 1024 = 2048 in the 1024-thread form (4096 entries), where
// the sample's histogram atomics, crowded into the few bins that the leading
// digit of similar scores falls into, had made the estimate a tenth of the
// kernel (decode 38.4 -> 36.3 µs against 4096 keys).
template <int THREADS> constexpr int TK_SAMPLES = THREADS <= 256 ? 4 : 2;
constexpr int TK_WIDE_CAP = 4096;    // filter buffer entries of the 1024-thread form
constexpr int64_t TK_FILTER_MAX_C = 262144;  // two LDS bitmaps of C bits each
// Word 3 of a raw buffer resource on gfx9-family GPUs (32-bit data format,
// no swizzle): with stride 0, a load at byte offset >= num_records returns 0.
constexpr int BUFFER_WORD3 = 0x00020000;
constexpr int TK_STREAM_THREADS = 256;

// Order-preserving map of a float to an unsigned key: larger float, larger
// key; -0 and +0 share a key; every NaN takes the largest key (NaN ranks
// above +inf, as torch.topk ranks it). No score maps to 0 (the smallest key,
// that of -inf, is 0x007fffff): key 0 marks a position outside the row.
__device__ __forceinline__ uint32_t score_key(float v) {
  const uint32_t b = __float_as_uint(v), mag = b & 0x7fffffffu;
  if (mag > 0x7f800000u) return 0xffffffffu;  // NaN
  if (mag == 0u) return 0x80000000u;          // -0 as +0
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

struct TopkArgs {
  const float* scores;      // [T][C]
  const int32_t* cu;        // [B + 1]
  const int32_t* seq_cmp;   // [B]
  const int32_t* residual;  // [B]
  int32_t* indices;         // [T][1][TOPK]
  int64_t C;                // score columns per token
  int32_t B, T, TOPK, RATIO;
  int32_t cap;              // filter buffer entries (dynamic LDS)
  int32_t words;            // bitmap words per row in dynamic LDS: ceil(C / 32)
  int32_t first_token;      // token of workgroup 0 (sparse_topk_row)
  int32_t segments;         // of a split row (sparse_topk_row)
  int32_t seg_keep;         // entries kept per segment: min(TOPK, segment) rounded up to 4
  uint32_t* seg_key;        // workspace: [tokens][segments][seg_keep] keys, 0 for none
  int32_t* seg_pos;         // workspace: [tokens][segments][seg_keep] positions
};

// Candidates [0, cand) of a token and how many of them it takes, after the
// request lookup: the last b with cu[b] <= token (empty requests have
// cu[b] == cu[b + 1] and are passed over), as gather.py:10-21.
struct TokenBounds {
  int cand, take;
};

// Bounds of a token of the request holding cu[b] = begin, cu[b + 1] = next,
// seq_cmp[b] = available, residual[b] = residual.
__device__ __forceinline__ TokenBounds bounds_of(const TopkArgs& a, int token, int begin, int next, int available,
                                                 int residual) {
  const int count_q = next - begin, offset = token - begin;
  const int end = available * a.RATIO + residual;
  const int cutoff = max(0, end - count_q + offset + 1) / a.RATIO;
  TokenBounds tb;
  tb.cand = (int)min<int64_t>(cutoff, a.C);
  tb.take = min(max(0, min(a.TOPK, min(available, cutoff))), tb.cand);
  return tb;
}

__device__ __forceinline__ TokenBounds token_bounds(const TopkArgs& a, int token) {
  int lo = 0, n = a.B;
  while (n > 1) {
    const int half = n >> 1;
    if (a.cu[lo + half] <= token) {
      lo += half;
      n -= half;
    } else {
      n = half;
    }
  }
  return bounds_of(a, token, a.cu[lo], a.cu[lo + 1], a.seq_cmp[lo], a.residual[lo]);
}

// Writes the -1 tail and the trivial selections; true when nothing is left.
template <int THREADS>
__device__ __forceinline__ bool trivial_selection(const TopkArgs& a, TokenBounds tb, int32_t* out) {
  for (int i = tb.take + (int)threadIdx.x; i < a.TOPK; i += THREADS) out[i] = -1;
  if (tb.take == 0) return true;
  if (tb.take == tb.cand) {  // every candidate is selected
    for (int i = threadIdx.x; i < tb.take; i += THREADS) out[i] = i;
    return true;
  }
  return false;
}

// Exclusive prefix sums of two values over the workgroup, sharing barriers;
// totals in total[0..1]. scratch: 2 THREADS / 64 ints of LDS.
template <int THREADS>
__device__ __forceinline__ void block_exclusive_scan2(int& a, int& b, int* scratch, int* total) {
  constexpr int WAVES = THREADS / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ia = wave_inclusive_scan(a), ib = wave_inclusive_scan(b);
  __syncthreads();
  if (lane == 63) {
    scratch[wave] = ia;
    scratch[WAVES + wave] = ib;
  }
  __syncthreads();
  int before_a = 0, before_b = 0, sum_a = 0, sum_b = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    const int ca = scratch[w], cb = scratch[WAVES + w];
    before_a += w < wave ? ca : 0;
    before_b += w < wave ? cb : 0;
    sum_a += ca;
    sum_b += cb;
  }
  total[0] = sum_a;
  total[1] = sum_b;
  a = before_a + ia - a;
  b = before_b + ib - b;
}

constexpr int DIGIT_SHIFT[3] = {21, 10, 0};
constexpr int DIGIT_WIDTH[3] = {11, 11, 10};

// LDS of the radix selections: two histograms, used alternately, so the one
// for the next digit is cleared while a digit is chosen from the other.
// PACKED: 16-bit counts, two bins per word, for selections over fewer than
// 2^16 keys (a count never carries into its neighbour).
template <bool PACKED>
struct RadixLds {
  static constexpr int WORDS = PACKED ? TK_BINS / 2 : TK_BINS;
  alignas(16) uint32_t hist[2][WORDS];
  int choice[3];  // bin of the digit, keys in the bins above it, keys in it (pick_bin)
  __device__ __forceinline__ void add(int parity, int bin, int n) {
    if constexpr (PACKED)
      atomicAdd(&hist[parity][bin >> 1], (uint32_t)n << ((bin & 1) * 16));
    else
      atomicAdd(&hist[parity][bin], (uint32_t)n);
  }
  __device__ __forceinline__ int get(int parity, int bin) const {
    if constexpr (PACKED)
      return (int)((hist[parity][bin >> 1] >> ((bin & 1) * 16)) & 0xffffu);
    else
      return (int)hist[parity][bin];
  }
};

// One wave: the bin of histogram lds.hist[cur] holding the need-th largest
// entry, into lds.choice (bin, entries in the bins above it). ROW: also the
// entries in it, and where there are fewer than `need` the lowest bin.
template <bool PACKED, bool ROW = false>
__device__ __forceinline__ void pick_bin(RadixLds<PACKED>& lds, int cur, int bins, int need, int lane) {
  // Lane l sums bins [bins - (l + 1) per, bins - l per): U = 2, 4 or 8
  // aligned 16-byte units of whole words, read in the order c, c + 1, ...
  // (mod U) with c chosen so that the 16 lanes one ds_read_b128 pass
  // serves (four quads whose (lane >> 3) & 3 differ) touch 16 distinct
  // bank groups. Packed words are summed whole: no half-word sum reaches
  // 2^16. The lane whose bins hold the need-th key is found by a scan over
  // the lanes, then its bins are read one per lane and scanned the same way.
  const int per = bins / 64;
  const int W = PACKED ? per / 2 : per, U = W / 4;
  const int quad = (lane >> 3) & 3;
  const int c = U == 2 ? (quad & 1) : U == 4 ? quad : (((lane >> 1) & 1) | (quad << 1));
  const uint32_t* words = lds.hist[cur] + (bins - (lane + 1) * per) / (PACKED ? 2 : 1);
  uint32_t sum = 0;
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    if (it < U) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(words + 4 * ((c + it) & (U - 1)));
      sum += (v[0] + v[1]) + (v[2] + v[3]);
    }
  }
  const int local = PACKED ? (int)((sum & 0xffffu) + (sum >> 16)) : (int)sum;
  const int incl = wave_inclusive_scan(local);
  const uint64_t holds = __ballot(incl - local < need && incl >= need);
  if (ROW && holds == 0) {
    if (lane == 0) {
      lds.choice[0] = 0;
      lds.choice[1] = 0;
      lds.choice[2] = need;
    }
    return;
  }
  const int owner = (int)__builtin_ctzll(holds);
  const int above = __builtin_amdgcn_readlane(incl - local, owner);  // owner is wave-uniform
  const int count = lane < per ? lds.get(cur, bins - 1 - (owner * per + lane)) : 0;
  const int incl2 = wave_inclusive_scan(count);
  const int q = (int)__builtin_ctzll(__ballot(lane < per && above + incl2 >= need));
  if (lane == q) {
    lds.choice[0] = bins - 1 - (owner * per + q);
    lds.choice[1] = above + incl2 - count;
    if constexpr (ROW) lds.choice[2] = count;
  }
}

// Radix selection of the rank-th largest key among those a key source
// yields: for_each_key(f) calls f(key) for every key of the source held by
// this thread. Returns that key, with *need_out = how many keys equal to it
// are among the rank largest; with PASSES < 3 digits, the key's leading
// DIGIT_SHIFT[PASSES - 1] bits (the rest zero) and the count for that prefix.
// Per digit: LDS histogram atomics, one barrier, wave 0 finds the digit's bin
// (a scan over lanes from the top bin) while the other waves clear the other
// histogram, one barrier. Expects hist[parity] cleared and leaves
// hist[parity] (flipped) cleared.
template <int THREADS, bool PACKED, int PASSES = 3, typename ForEachKey>
__device__ __forceinline__ uint32_t radix_select(ForEachKey for_each_key, int rank, RadixLds<PACKED>& lds, int& parity,
                                                 int* need_out) {
  static_assert(PASSES >= 1 && PASSES <= 3, "one to three digits");
  static_assert(THREADS > 64, "the histogram is cleared by the waves other than wave 0");
  const int tid = threadIdx.x, lane = tid & 63;
  uint32_t prefix = 0, prefix_mask = 0;
  int need = rank;
#pragma unroll
  for (int pass = 0; pass < PASSES; ++pass) {
    const int shift = DIGIT_SHIFT[pass], bins = 1 << DIGIT_WIDTH[pass];
    const int cur = parity;
    for_each_key([&](uint32_t k) {
      // Lanes whose key falls in the same bin as the first counting lane's add
      // together in one atomic (keys often share their leading digit); the
      // others add their own.
      const bool counts = (k & prefix_mask) == prefix;
      const uint64_t active = __ballot(counts);
      if (active == 0) return;  // uniform
      const int bin = (int)((k >> shift) & (uint32_t)(bins - 1));
      const int leader = (int)__builtin_ctzll(active);
      const int lead_bin = __builtin_amdgcn_readlane(bin, leader);  // leader is wave-uniform
      const uint64_t same = __ballot(counts && bin == lead_bin);
      if (lane == leader) lds.add(cur, lead_bin, __popcll(same));
      else if (counts && bin != lead_bin) lds.add(cur, bin, 1);
    });
    __syncthreads();
    if (tid < 64) {
      pick_bin<PACKED>(lds, cur, bins, need, lane);
    } else {
      uint32_t* spare = lds.hist[parity ^ 1];
      for (int i = 4 * (tid - 64); i < RadixLds<PACKED>::WORDS; i += 4 * (THREADS - 64))
        *reinterpret_cast<u32x4*>(spare + i) = u32x4{0u, 0u, 0u, 0u};
    }
    __syncthreads();
    need -= lds.choice[1];
    prefix |= (uint32_t)lds.choice[0] << shift;
    prefix_mask |= (uint32_t)(bins - 1) << shift;
    parity ^= 1;
  }
  *need_out = need;
  return prefix;
}

// One streaming pass over the candidates [0, cand) of a row read through a
// buffer resource of range cand * 4 bytes (loads past it return zeros without
// touching memory): f(key, position) is called by every thread of the wave
// together, TK_UNROLL * 4 times per step, with key 0 for a position past the
// candidates (no score maps to key 0). 16-byte loads of 4 consecutive
// positions: a buffer load of any width needs dword alignment, which every f32
// row has, whatever C; against 4-byte loads for rows that are no multiple of 16
// bytes 4096 rows of 16391 take 76.9 us instead of 78.6 (both with the linear histograms).
template <int THREADS>
__device__ __forceinline__ int stream_position(int base, int j) {
  const int tid = threadIdx.x;
  return base + ((j >> 2) * THREADS + tid) * 4 + (j & 3);
}

// The same pass handing each step's UNROLL * 4 keys to f at once:
// f(keys, base), keys[j] being the key of position stream_position(base, j).
template <int THREADS, int UNROLL, typename F>
__device__ __forceinline__ void stream_row_steps(__amdgpu_buffer_rsrc_t rsrc, int cand, F f) {
  constexpr int STEP = THREADS * 4 * UNROLL;
  for (int base = 0; base < cand; base += STEP) {
    uint32_t w[UNROLL * 4];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const u32x4 x = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, stream_position<THREADS>(base, 4 * u) * 4, 0, 0));
#pragma unroll
      for (int e = 0; e < 4; ++e) w[4 * u + e] = x[e];
    }
    uint32_t keys[UNROLL * 4];
#pragma unroll
    for (int j = 0; j < UNROLL * 4; ++j)
      keys[j] = stream_position<THREADS>(base, j) < cand ? score_key(__uint_as_float(w[j])) : 0u;
    f(keys, base);
  }
}

template <int THREADS, typename F>
__device__ __forceinline__ void stream_row(__amdgpu_buffer_rsrc_t rsrc, int cand, F f) {
  constexpr int STEP = THREADS * 4 * TK_UNROLL;
  for (int base = 0; base < cand; base += STEP) {
    uint32_t w[TK_UNROLL * 4];
#pragma unroll
    for (int u = 0; u < TK_UNROLL; ++u) {
      const u32x4 x = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, stream_position<THREADS>(base, 4 * u) * 4, 0, 0));
#pragma unroll
      for (int e = 0; e < 4; ++e) w[4 * u + e] = x[e];
    }
#pragma unroll
    for (int j = 0; j < TK_UNROLL * 4; ++j) {
      const int p = stream_position<THREADS>(base, j);
      f(p < cand ? score_key(__uint_as_float(w[j])) : 0u, p);
    }
  }
}

__device__ __forceinline__ int lane_rank(uint64_t mask) {  // set bits of mask below this lane
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

constexpr uint32_t KEY_LOWEST = 0x00800000u, KEY_HIGHEST = 0xff7fffffu;  // keys of -FLT_MAX and FLT_MAX

__device__ __forceinline__ float key_score(uint32_t k) {  // inverse of score_key, of the nearest finite key
  k = min(max(k, KEY_LOWEST), KEY_HIGHEST);
  return __uint_as_float(k ^ ((uint32_t)((int32_t)~k >> 31) | 0x80000000u));
}

// Maximum over the 64 lanes of a wave (every lane active), in DPP moves as
// wave_inclusive_scan; lanes shifted in from outside a row keep `v`'s own.
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x111, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x112, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x114, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x118, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xa, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x143, 0xc, 0xf, false));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Histogram bins linear in the score over [base, base + span]: non-decreasing
// in the key; infinities, NaN and keys outside take the end bins.
struct LinearBins {
  float base, per_bin;
  // Over the scores of two keys; false where they span no usable range (none
  // finite, equal, or too far apart).
  __device__ __forceinline__ bool set(uint32_t low, uint32_t high) {
    base = key_score(low);
    const float span = key_score(high) - base;
    const bool usable = low <= high && high >= KEY_LOWEST && span > 1e-30f && span < 3e38f;
    base = usable ? base : 0.f;
    per_bin = usable ? (TK_BINS - 1) / span : 0.f;  // 0: one bin
    return usable;
  }
  __device__ __forceinline__ void to_scalar() {  // of uniform bins: out of the vector registers
    base = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(base)));
    per_bin = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(per_bin)));
  }
  __device__ __forceinline__ int of(uint32_t k) const {
    return (int)fminf(fmaxf((key_score(k) - base) * per_bin, 0.f), (float)(TK_BINS - 1));
  }
  // A key that no key of a bin >= b is below (a hundredth of a bin and one
  // step of the float against the rounding of either direction).
  __device__ __forceinline__ uint32_t lower_bound(int b) const {
    if (b <= 0) return 1u;
    return score_key(base + ((float)b - 0.01f) / per_bin) - 1u;
  }
};

// The need-th largest of the `inside` (1..64) keys in LDS, found by every wave of
// the workgroup for itself; *need becomes how many keys equal to it are taken.
// Lane l's key is the one when fewer than `need` keys are larger and, with
// those equal to it, at least `need`.
__device__ __forceinline__ uint32_t rank_small(const uint32_t* keys, int inside, int lane, int* need) {
  const uint32_t mine = lane < inside ? keys[lane] : 0u;
  int larger = 0, equal = 0;
  for (int i = 0; i < inside; ++i) {
    const uint32_t other = (uint32_t)__builtin_amdgcn_readlane((int)mine, i);
    larger += other > mine ? 1 : 0;
    equal += other == mine ? 1 : 0;
  }
  const int owner = (int)__builtin_ctzll(__ballot(lane < inside && larger < *need && larger + equal >= *need));
  const uint32_t key = (uint32_t)__builtin_amdgcn_readlane((int)mine, owner);
  *need -= __builtin_amdgcn_readlane(larger, owner);
  return key;
}
constexpr int TK_SMALL = 64;  // keys of a histogram bin that rank_small takes

template <bool COMPACT> struct BufferPosition { typedef int type; };
template <> struct BufferPosition<true> { typedef uint16_t type; };

// COMPACT (rows up to 32K positions, 256 threads): 16-bit histogram counts
// and buffer positions, so that more workgroups fit in a CU's LDS.
// Eight waves per SIMD (at most 64 VGPRs): two 1024-thread or eight 256-thread
// workgroups per CU, as many as the LDS holds.
template <int THREADS>
__global__ __launch_bounds__(THREADS, 8) void sparse_topk_filter(TopkArgs a) {
  constexpr bool COMPACT = THREADS <= 256;
  // Linear histograms (below); the 1024-thread form, at its register budget,
  // keeps the radix digits (384 rows of 64K 32.8 us, with them 33.6).
  constexpr bool LINEAR = COMPACT;
  // 4-position groups per thread and step of the filter pass.
  constexpr int FILTER_UNROLL = THREADS <= 256 ? TK_UNROLL : TK_UNROLL / 2;
  typedef typename BufferPosition<COMPACT>::type Position;
  // Dynamic LDS: two bitmaps of a.words words (keys above the threshold, keys
  // equal to it), then (COMPACT) the buffer of a.cap keys and positions; the
  // 1024-thread form keeps a static buffer of TK_WIDE_CAP entries.
  extern __shared__ uint32_t dynamic_lds[];
  __shared__ uint32_t wide_key[COMPACT ? 1 : TK_WIDE_CAP];
  __shared__ int wide_pos[COMPACT ? 1 : TK_WIDE_CAP];
  const int CAP = COMPACT ? a.cap : TK_WIDE_CAP;
  uint32_t* const bitmaps = dynamic_lds;
  uint32_t* const buf_key = COMPACT ? dynamic_lds + 2 * a.words : wide_key;
  Position* const buf_pos =
      COMPACT ? reinterpret_cast<Position*>(dynamic_lds + 2 * a.words + a.cap) : reinterpret_cast<Position*>(wide_pos);
  __shared__ RadixLds<COMPACT> radix;
  __shared__ int scan_scratch[2 * THREADS / 64];
  __shared__ int reached;
  __shared__ int request_lds[4];
  // Uses of LDS that is idle then (292 bytes more and rows of about 24K fit
  // seven workgroups per CU instead of eight): each wave's range of sample keys
  // in the buffer, the count of rank_small's keys in the request's place.
  uint32_t* const range_lds = buf_key;
  int* const small_count = request_lds;
  constexpr int WAVES = THREADS / 64;
  const int token = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  // 1. Sample: S keys in blocks of 16 consecutive positions (64 bytes), the
  // S / 16 blocks evenly spaced over a range of n positions (block b from
  // position floor(b n / (S / 16))), so the sample touches few cache lines;
  // thread t holds samples SPT t .. SPT t + SPT - 1. The first sample, S =
  // min(SPT THREADS, C) over the whole allocated row (n = C), goes out before
  // the request lookup; its keys at positions past the token's candidates are
  // left out, and when the candidates cover less than half of the row (or C
  // < SPT THREADS) the row is sampled again over them (n = cand,
  // S = min(SPT THREADS, cand), a row shorter than that whole).
  // A sample shorter than SPT THREADS is the whole range (block
  // positions i); otherwise it has SAMPLE_BLOCKS blocks, a power of two, so
  // floor(b n / SAMPLE_BLOCKS) is a shift. The loads are unconditional
  // (positions past the buffer's range read 0) and their words are turned
  // into keys only where they are used, so that the four go out together
  // with the request lookup's and share its round trip.
  constexpr int SPT = TK_SAMPLES<THREADS>;
  constexpr int SAMPLE_BLOCKS = SPT * THREADS / 16;
  constexpr int SAMPLE_SHIFT = __builtin_ctz(SAMPLE_BLOCKS);
  static_assert((SAMPLE_BLOCKS & (SAMPLE_BLOCKS - 1)) == 0, "sample blocks must be a power of two");
  auto sample_position = [&](int i, int64_t n, int s) {
    return s < SPT * THREADS ? i : (int)(((int64_t)(i >> 4) * n) >> SAMPLE_SHIFT) + (i & 15);
  };
  const int samples_c = (int)min<int64_t>(SPT * THREADS, a.C);
  const __amdgpu_buffer_rsrc_t rsrc_row = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(a.scores + (size_t)token * a.C), (short)0, (int)(a.C * 4), BUFFER_WORD3);
  uint32_t sample[SPT];  // the score words, then their keys
  int sample_pos[SPT];
#pragma unroll
  for (int j = 0; j < SPT; ++j) {
    sample_pos[j] = sample_position(tid * SPT + j, a.C, samples_c);
    sample[j] = __builtin_amdgcn_raw_buffer_load_b32(rsrc_row, sample_pos[j] * 4, 0, 0);
  }
  // Request lookup. B <= THREADS: one round trip, thread b loading request
  // b's cu[b], cu[b + 1], seq_cmp[b] and residual[b]; the token's request is
  // #{b: cu[b] <= token} - 1 (as in token_bounds), whose thread hands its
  // values to the others through LDS. Larger B: the binary search.
  TokenBounds tb;
  if (a.B <= THREADS) {
    int begin = 0, next = 0, available = 0, residual = 0;
    if (tid < a.B) {
      begin = a.cu[tid];
      next = a.cu[tid + 1];
      available = a.seq_cmp[tid];
      residual = a.residual[tid];
    }
    const int below = __popcll(__ballot(tid < a.B && begin <= token));
    if (lane == 0) scan_scratch[wave] = below;
    __syncthreads();
    int requests = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) requests += scan_scratch[w];
    if (tid == max(requests - 1, 0)) {  // request 0 at least (cu[0] = 0 <= token)
      request_lds[0] = begin;
      request_lds[1] = next;
      request_lds[2] = available;
      request_lds[3] = residual;
    }
    __syncthreads();
    tb = bounds_of(a, token, request_lds[0], request_lds[1], request_lds[2], request_lds[3]);
  } else {
    tb = token_bounds(a, token);
  }
  int32_t* out = a.indices + (size_t)token * a.TOPK;
  if (trivial_selection<THREADS>(a, tb, out)) return;
  const int cand = tb.cand, take = tb.take, words = (cand + 31) >> 5;
  uint32_t* above_bits = bitmaps;
  uint32_t* equal_bits = bitmaps + words;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(a.scores + (size_t)token * a.C), (short)0, cand * 4, BUFFER_WORD3);
  const bool whole_row_sample = samples_c == SPT * THREADS && 2 * (int64_t)cand >= a.C;  // uniform
  int samples = 0;           // keys in the sample
  uint32_t sample_mask = 0;  // bit j: sample[j] is one of them
  if (whole_row_sample) {
    int mine = 0;
#pragma unroll
    for (int j = 0; j < SPT; ++j) {
      sample[j] = score_key(__uint_as_float(sample[j]));  // every sample is in [0, C) here
      const bool in_row = sample_pos[j] < cand;
      sample_mask |= in_row ? 1u << j : 0u;
      mine += in_row ? 1 : 0;
    }
    mine = __builtin_amdgcn_readlane(wave_inclusive_scan(mine), 63);
    if (lane == 0) scan_scratch[WAVES + wave] = mine;  // summed after the barrier below
  } else {
    samples = min(SPT * THREADS, cand);
#pragma unroll
    for (int j = 0; j < SPT; ++j)
      sample[j] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, sample_position(tid * SPT + j, cand, samples) * 4, 0, 0);
#pragma unroll
    for (int j = 0; j < SPT; ++j) {
      const int i = tid * SPT + j;
      sample[j] = i < samples ? score_key(__uint_as_float(sample[j])) : 0u;
      sample_mask |= i < samples ? 1u << j : 0u;
    }
  }
  // Range of the sample's finite keys.
  uint32_t low = 0xffffffffu, high = 0u;
  if constexpr (LINEAR) {
#pragma unroll
    for (int j = 0; j < SPT; ++j)
      if ((sample_mask >> j) & 1u) {
        if (sample[j] >= KEY_LOWEST) low = min(low, sample[j]);
        if (sample[j] <= KEY_HIGHEST) high = max(high, sample[j]);
      }
    low = ~wave_max(~low);
    high = wave_max(high);
    if (lane == 0) {
      range_lds[wave] = low;
      range_lds[WAVES + wave] = high;
    }
  }
  for (int i = tid; i < 2 * words; i += THREADS) bitmaps[i] = 0u;
  for (int i = tid; i < RadixLds<COMPACT>::WORDS; i += THREADS) radix.hist[0][i] = 0u;
  if (tid == 0) reached = 0;
  __syncthreads();
  if (LINEAR && tid == 0) *small_count = 0;  // every thread has read the request
  LinearBins bins{0.f, 0.f};
  bool linear = false;  // uniform
  if constexpr (LINEAR) {
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      low = min(low, range_lds[w]);
      high = max(high, range_lds[WAVES + w]);
    }
    low = (uint32_t)__builtin_amdgcn_readfirstlane((int)low);
    high = (uint32_t)__builtin_amdgcn_readfirstlane((int)high);
    linear = bins.set(low, high) && take <= CAP;
    bins.to_scalar();
  }
  if (linear) {
#pragma unroll
    for (int j = 0; j < SPT; ++j)
      if ((sample_mask >> j) & 1u) radix.add(0, bins.of(sample[j]), 1);
    __syncthreads();
  }
  if (whole_row_sample) {
#pragma unroll
    for (int w = 0; w < WAVES; ++w) samples += scan_scratch[WAVES + w];
  }
  auto clear_histogram = [&](int which) {  // by the waves other than wave 0
    for (int i = 4 * (tid - 64); i < RadixLds<COMPACT>::WORDS; i += 4 * (THREADS - 64))
      *reinterpret_cast<u32x4*>(&radix.hist[which][i]) = u32x4{0u, 0u, 0u, 0u};
  };
  int parity = linear ? 1 : 0, unused = 0;  // hist[parity] is clear (hist[1]: from the first round on)

  // 2. Filter: keys >= estimate (>= 1, so never a position past the row),
  // the estimate being the rank-th largest sample. A rank whose estimate lets
  // fewer than `take` keys through, or more than the buffer holds, is
  // replaced by binary search between the ranks known to be too small and
  // too large, and the row filtered again; when no rank is left (a row of
  // many equal keys) the selection runs over the whole row below.
  // Sample rank: about 1.25x (256 threads: a buffer of 2 TOPK entries) or 2x
  // (4096 entries) the expected count of samples above the threshold, plus a
  // margin.
  int rank = THREADS <= 256 ? min(samples, (int)((5 * (int64_t)take * samples) / (4 * (int64_t)cand)) + 8)
                            : min(samples, (int)((2 * (int64_t)take * samples) / cand) + 16);
  int too_few = 0, too_many = samples + 1, n = 0;
  bool buffered = false;
  uint32_t filter_estimate = 0;
  // A filter pass succeeds only when take <= n <= CAP: with take above the
  // buffer's capacity no pass can, so the row goes straight to the whole-row
  // selection below instead of being streamed by every filter round first.
  for (int round = 0; take <= CAP && round < TK_FILTER_ROUNDS; ++round) {
    // From the linear histogram of the sample, unless its bin holds so many
    // samples (an outlier's range, or many equal scores) that it says little.
    uint32_t estimate = 0;
    if (linear) {
      if (wave == 0) pick_bin<COMPACT, true>(radix, 0, TK_BINS, rank, lane);
      else if (round == 0) clear_histogram(1);
      __syncthreads();
      linear = radix.choice[2] <= 8 + rank / 4;
      estimate = (uint32_t)__builtin_amdgcn_readfirstlane((int)bins.lower_bound(radix.choice[0]));
    }
    if (!linear) {
      if (LINEAR && parity == 1) __syncthreads();  // every wave has read the choice
      estimate = radix_select<THREADS, COMPACT, 2>(
          [&](auto f) {
#pragma unroll
            for (int j = 0; j < SPT; ++j)
              if ((sample_mask >> j) & 1u) f(sample[j]);
          },
          rank, radix, parity, &unused);  // ends with a barrier: every read of `reached` is done
    }
    if (!LINEAR || round > 0) {
      if (tid == 0) reached = 0;
      __syncthreads();
    }
    // Appends: per step, each lane counts its keys that reach the estimate, a
    // wave scan gives each lane its first slot, and ONE LDS atomic per wave
    // reserves the wave's slots (an atomic with a returned value per key
    // position and wave serialises the pass: prefill 217 -> 192 µs).
    stream_row_steps<THREADS, FILTER_UNROLL>(
        rsrc, cand, [&](const uint32_t (&keys)[FILTER_UNROLL * 4], int base) {
          int hits = 0;
#pragma unroll
          for (int j = 0; j < FILTER_UNROLL * 4; ++j) hits += keys[j] >= estimate ? 1 : 0;
          const int before = wave_inclusive_scan(hits) - hits;
          const int total = __builtin_amdgcn_readlane(before + hits, 63);
          if (total == 0) return;  // uniform
          int first = 0;
          if (lane == 0) first = atomicAdd(&reached, total);
          int slot = __builtin_amdgcn_readfirstlane(first) + before;
#pragma unroll
          for (int j = 0; j < FILTER_UNROLL * 4; ++j) {
            if (keys[j] >= estimate) {
              if (slot < CAP) {
                buf_key[slot] = keys[j];
                buf_pos[slot] = (Position)stream_position<THREADS>(base, j);
              }
              ++slot;
            }
          }
        });
    __syncthreads();
    n = reached;
    if (n >= take && n <= CAP) {
      buffered = true;
      filter_estimate = estimate;
      break;
    }
    if (n < take)
      too_few = rank;
    else
      too_many = rank;
    rank = too_many > samples ? min(samples, 2 * rank) : (too_few + too_many) / 2;
    if (rank <= too_few || rank >= too_many) break;  // no rank left to try
  }

  // 3. Exact selection, from the buffer when it holds every key that can be
  // taken, else from the row; then the selected keys are marked.
  int need = 0;
  uint32_t threshold = 0;
  if (buffered) {
    int bin = -1, inside = TK_SMALL + 1, rest = take;
    if (linear) {
      // One histogram, linear between the estimate and the largest sample:
      // keys above that share the top bin.
      bins.set(max(filter_estimate, low), high);
      bins.to_scalar();
      for (int i = tid; i < n; i += THREADS) radix.add(parity, bins.of(buf_key[i]), 1);
      __syncthreads();
      if (wave == 0) pick_bin<COMPACT, true>(radix, parity, TK_BINS, take, lane);
      else clear_histogram(parity ^ 1);
      __syncthreads();
      parity ^= 1;
      bin = radix.choice[0];
      inside = radix.choice[2];
      rest = take - radix.choice[1];
    }
    if (LINEAR && inside <= TK_SMALL) {  // uniform
      uint32_t* const small_key = radix.hist[parity ^ 1];  // the histogram just read
      for (int i = tid; i < n; i += THREADS) {
        const uint32_t k = buf_key[i];
        if (bins.of(k) == bin) small_key[atomicAdd(small_count, 1)] = k;
      }
      __syncthreads();
      threshold = rank_small(small_key, inside, lane, &rest);
      need = rest;
    } else {
      if (LINEAR) __syncthreads();  // every wave has read the choice
      threshold = radix_select<THREADS>(
          [&](auto f) {
            for (int i = tid; i < n; i += THREADS) {
              const uint32_t k = buf_key[i];
              if (bin < 0 || bins.of(k) == bin) f(k);
            }
          },
          rest, radix, parity, &need);
    }
    for (int i = tid; i < n; i += THREADS) {
      const uint32_t k = buf_key[i];
      const int p = buf_pos[i];
      if (k > threshold) atomicOr(&above_bits[p >> 5], 1u << (p & 31));
      else if (k == threshold) atomicOr(&equal_bits[p >> 5], 1u << (p & 31));
    }
  } else {
    threshold = radix_select<THREADS>(
        [&](auto f) {
          stream_row<THREADS>(rsrc, cand, [&](uint32_t k, int) {
            if (k != 0u) f(k);
          });
        },
        take, radix, parity, &need);
    stream_row<THREADS>(rsrc, cand, [&](uint32_t k, int p) {
      if (k > threshold) atomicOr(&above_bits[p >> 5], 1u << (p & 31));
      else if (k == threshold) atomicOr(&equal_bits[p >> 5], 1u << (p & 31));
    });
  }
  __syncthreads();

  // 4. Output in position order: thread t owns words [t per, (t + 1) per).
  // Slot of a selected position = keys above the threshold before it +
  // min(equal keys before it, need).
  const int per = (words + THREADS - 1) / THREADS, w0 = min(words, tid * per), w1 = min(words, w0 + per);
  int above_before = 0, equal_before = 0;
  for (int w = w0; w < w1; ++w) {
    above_before += __popc(above_bits[w]);
    equal_before += __popc(equal_bits[w]);
  }
  int totals[2];
  block_exclusive_scan2<THREADS>(above_before, equal_before, scan_scratch, totals);
  for (int w = w0; w < w1; ++w) {
    const uint32_t g = above_bits[w], q = equal_bits[w];
    uint32_t bits = g | q;
    while (bits) {
      const int b = __builtin_ctz(bits);
      bits &= bits - 1;
      const int p = w * 32 + b;
      if ((g >> b) & 1u) {
        const int at = above_before + min(equal_before, need);
        if (at < take) out[at] = p;
        ++above_before;
      } else {
        if (equal_before < need && above_before + equal_before < take) out[above_before + equal_before] = p;
        ++equal_before;
      }
    }
  }
}

// ---- rows held in registers --------------------------------------------------
//
// sparse_topk_row: one workgroup selects from up to THREADS * ITEMS positions
// that it keeps in registers: one 16-byte load per group of four positions, all
// in flight at once and in one round trip with the request lookup's. What bounds
// it is the chain of dependent steps of one row (calls of few tokens) and the
// vector operations per score (many): a score costs its key, a maximum, a
// comparison and a count.
//   1. bound: at least `take` scores are no smaller than the take-th largest
//      group maximum, so that is a lower bound of the threshold, and a close one
//      while groups outnumber `take` (512 of 16K: about 540 scores reach it). No
//      sample can miss it, so no row is filtered twice. It is taken to the
//      resolution of one histogram, linear in the score between the smallest
//      and largest finite maximum: the leading digit of the float key, which
//      crowds most of a row into a few bins, would take two.
//   2. keys that reach the bound go to LDS with their positions, in position
//      order (counts per group and wave, one scan);
//   3. the threshold among them: one linear histogram, whose bin of the
//      take-th key holds few; those are ranked against each other (more than
//      SMALL of them: radix selection);
//   4. the entries that are taken, compacted in order, are the output.
// A row with no usable range (its finite maxima all equal, or none finite) or
// with more entries than LDS holds (many equal scores) takes the radix selection
// over the whole row, read again.
// The scores buffer may be far wider than a token's candidates (short contexts
// among long ones, a buffer of the largest size). BOUNDED: the request is looked
// up first, and loads and work end at the candidates; one round trip more, which
// several workgroups per CU hide and which the registers of a wide row save
// anyway. Rows up to 16K of a workgroup that has a CU to itself keep both loads
// in one round trip. Measured with a quarter of the row as candidates, reading
// the whole row -> its candidates (us, TOPK 512): 500 rows of 30K 23.5 -> 13.1,
// 1000 of 16K 21.3 -> 15.3, 256 of 30K 14.9 -> 9.2; full rows 27.1 -> 26.3, 24.3
// -> 25.0, 16.8 -> 16.5.
// Measured, GPU time (us, against the streaming form of before): 64 rows of 16K
// 26.8 -> 9.7, 350 36.5 -> 15.2, 1500 46.3 -> 32.5; 256 rows of 30K 71 -> 16.5; split, 1
// row of 256K 52 -> 17.5, of 420K 1760 -> 17.7. One 16K row in a
// 1024-thread workgroup takes 8.2 us: row and lookup 3.3, bound 1.3, entries 1.6,
// threshold 1.6, output 0.4.
//
// ROW: scores to indices. SEGMENT: blockIdx.y is a segment of a longer row;
// its min(TOPK, candidates) largest go to the workspace as keys and positions
// in ascending position order, then key 0 up to a.seg_keep entries. A token with
// no candidates past the first segment gets its indices from that segment.
// MERGE: the segments' entries of any other token, in order, are the row (their
// order is the position order, so ties resolve alike), and give the indices.
enum { TK_ROW = 0, TK_SEGMENT = 1, TK_MERGE = 2 };
constexpr int TK_ENTRIES = 2048;  // keys that reach the bound, at most
constexpr int TK_SEGMENT_ITEMS = 16;
constexpr int64_t TK_SEGMENT_SIZE = 1024 * TK_SEGMENT_ITEMS;

template <int THREADS, int ITEMS, int MODE>
__global__ __launch_bounds__(THREADS, ITEMS <= 16 ? 8 : THREADS * ITEMS <= 16384 ? 6 : 4) void sparse_topk_row(TopkArgs a) {
  constexpr bool BOUNDED = MODE == TK_SEGMENT || (MODE == TK_ROW && (THREADS == 512 || ITEMS > 16));
  constexpr int WAVES = THREADS / 64, GROUPS = ITEMS / 4;
  constexpr int CELLS = GROUPS * WAVES;            // (group, wave) cells, in position order
  constexpr int PER_LANE = (CELLS + 63) / 64;
  constexpr int PER_THREAD = TK_ENTRIES / THREADS;  // entries per thread
  static_assert(ITEMS % 4 == 0 && (PER_LANE == 1 || WAVES % PER_LANE == 0), "cells of a lane stay in one group");
  static_assert(PER_THREAD * THREADS == TK_ENTRIES, "entries split evenly");
  __shared__ RadixLds<false> radix;
  __shared__ __attribute__((aligned(16))) uint32_t entry_key[TK_ENTRIES];
  __shared__ __attribute__((aligned(16))) int entry_pos[TK_ENTRIES];
  __shared__ int request_lds[4];
  __shared__ uint32_t range_lds[2][WAVES];
  __shared__ uint32_t small_key[TK_SMALL];
  __shared__ int small_count;
  __shared__ uint32_t cells[PER_LANE * 64];
  const int token = a.first_token + (int)blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- the request (thread b holds request b) and the row: in one round trip, or
  // (BOUNDED) the row's candidates alone once the request is known ---------------
  int begin = 0, next = 0, available = 0, residual = 0;
  const bool early = a.B <= THREADS;  // uniform
  if (early && tid < a.B) {
    begin = a.cu[tid];
    next = a.cu[tid + 1];
    available = a.seq_cmp[tid];
    residual = a.residual[tid];
  }
  const int64_t first = MODE == TK_SEGMENT ? (int64_t)blockIdx.y * (THREADS * ITEMS) : 0;
  const int held = MODE == TK_MERGE ? a.segments * a.seg_keep : (int)min<int64_t>(a.C - first, THREADS * ITEMS);
  const uint32_t* source = MODE == TK_MERGE ? a.seg_key + (size_t)blockIdx.x * held
                                            : reinterpret_cast<const uint32_t*>(a.scores) + (size_t)token * a.C + first;
  int reach = held;  // positions that are read
  auto load_group = [&](int u) {  // past the reach: zeros, with no memory traffic
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(source), (short)0, reach * 4, BUFFER_WORD3);
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (u * THREADS + tid) * 16, 0, 0));
  };
  uint32_t key[ITEMS];  // the score words, then their keys (0: not a candidate)
  auto load_row = [&]() {
#pragma unroll
    for (int u = 0; u < GROUPS; ++u) {
      const u32x4 x = load_group(u);
#pragma unroll
      for (int j = 0; j < 4; ++j) key[4 * u + j] = x[j];
    }
  };
  if constexpr (!BOUNDED) load_row();
  for (int i = 4 * tid; i < 2 * TK_BINS; i += 4 * THREADS)
    *reinterpret_cast<u32x4*>(&radix.hist[0][0] + i) = u32x4{0u, 0u, 0u, 0u};
  if (tid == 0) small_count = 0;
  TokenBounds tb;
  if (early) {
    // The last b with cu[b] <= token, request 0 at least (as token_bounds).
    if (tid < a.B && (begin <= token || tid == 0) && (tid == a.B - 1 || next > token)) {
      request_lds[0] = begin;
      request_lds[1] = next;
      request_lds[2] = available;
      request_lds[3] = residual;
    }
    block_barrier();
    tb = bounds_of(a, token, request_lds[0], request_lds[1], request_lds[2], request_lds[3]);
  } else {
    tb = token_bounds(a, token);
    block_barrier();
  }
  int32_t* out = a.indices + (size_t)token * a.TOPK;
  uint32_t* seg_key = nullptr;
  int32_t* seg_pos = nullptr;
  int cand = tb.cand, take = tb.take;
  if constexpr (MODE == TK_SEGMENT) {
    const size_t at = ((size_t)blockIdx.x * a.segments + blockIdx.y) * a.seg_keep;
    seg_key = a.seg_key + at;
    seg_pos = a.seg_pos + at;
    cand = (int)max<int64_t>(0, min<int64_t>(tb.cand - first, held));
    if (tb.cand <= THREADS * ITEMS) {  // the first segment is the row: its indices are the result
      if (blockIdx.y != 0 || trivial_selection<THREADS>(a, tb, out)) return;
    } else {
      take = min(take, cand);
      for (int i = take + tid; i < a.seg_keep; i += THREADS) seg_key[i] = 0u;
      if (take == 0) return;
    }
  } else {
    if (MODE == TK_MERGE && tb.cand <= TK_SEGMENT_SIZE) return;  // written by its segment
    if (trivial_selection<THREADS>(a, tb, out)) return;
  }
  if constexpr (BOUNDED) {
    reach = __builtin_amdgcn_readfirstlane(cand);
    load_row();
  }
  // What `key` holds that can be nonzero: the candidates, or the entries of the segments with any.
  const int members = MODE == TK_MERGE ? (cand + (int)TK_SEGMENT_SIZE - 1) / (int)TK_SEGMENT_SIZE * a.seg_keep : cand;
  auto used = [&](int u) { return !BOUNDED || u * THREADS * 4 < reach; };  // group u holds candidates (uniform)
  auto position = [&](int i) { return ((i >> 2) * THREADS + tid) * 4 + (i & 3); };  // of key[i]
  auto emit = [&](int slot, uint32_t k, int p) {
    if constexpr (MODE == TK_SEGMENT) {
      if (tb.cand <= THREADS * ITEMS) {
        out[slot] = p;
      } else {
        seg_key[slot] = k;
        seg_pos[slot] = (int)first + p;
      }
    } else if constexpr (MODE == TK_MERGE) {
      out[slot] = a.seg_pos[(size_t)blockIdx.x * held + p];
    } else {
      out[slot] = p;
    }
  };

  // ---- 1. bound ------------------------------------------------------------------
  uint32_t top[GROUPS];  // group maxima, 0 for a group with no candidate
  uint32_t low = 0xffffffffu, high = 0u;  // finite ones
#pragma unroll
  for (int u = 0; u < GROUPS; ++u) {
    uint32_t m = 0u;
    if (used(u)) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = 4 * u + j;
        if constexpr (MODE != TK_MERGE) key[i] = position(i) < cand ? score_key(__uint_as_float(key[i])) : 0u;
        key[i] = opaque(key[i]);  // no comparison is kept in scalar registers for the steps below
        m = max(m, key[i]);
      }
      if (m >= KEY_LOWEST) low = min(low, m);
      if (m <= KEY_HIGHEST) high = max(high, m);
    }
    top[u] = m;
  }
  low = ~wave_max(~low);
  high = wave_max(high);
  if (lane == 0) {
    range_lds[0][wave] = low;
    range_lds[1][wave] = high;
  }
  block_barrier();
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    low = min(low, range_lds[0][w]);
    high = max(high, range_lds[1][w]);
  }
  LinearBins bins;
  const bool linear = bins.set(low, high);
  uint32_t bound = 0u;
  int n = TK_ENTRIES + 1;  // keys that reach the bound
  uint32_t before[GROUPS];
  auto scan_cells = [&](auto count) {  // count(u): this thread's (packed) count of group u, at most 4 in each half
#pragma unroll
    for (int u = 0; u < GROUPS; ++u) {
      int c = 0, incl = 0;
      if (used(u)) {
        c = count(u);
        incl = wave_inclusive_scan(c);
      }
      before[u] = (uint32_t)(incl - c);
      if (lane == 63) cells[u * WAVES + wave] = (uint32_t)incl;
    }
    if (CELLS < 64 && tid >= CELLS && tid < 64) cells[tid] = 0u;
    block_barrier();
  };
  // Sums of the cells before (u, wave) and their total, low and high halves.
  uint32_t cell[PER_LANE];
  int lo_excl = 0, hi_excl = 0, lo_total = 0;
  auto read_cells = [&]() {
    int lo_sum = 0, hi_sum = 0;
#pragma unroll
    for (int i = 0; i < PER_LANE; ++i) {
      cell[i] = cells[lane * PER_LANE + i];
      lo_sum += (int)(cell[i] & 0xffffu);
      hi_sum += (int)(cell[i] >> 16);
    }
    const int lo_incl = wave_inclusive_scan(lo_sum);
    lo_excl = lo_incl - lo_sum;
    lo_total = __builtin_amdgcn_readlane(lo_incl, 63);
    hi_excl = wave_inclusive_scan(hi_sum) - hi_sum;
  };
  auto cell_base = [&](int u, int& lo, int& hi) {
    const int at = u * WAVES + wave, owner = at / PER_LANE;  // uniform
    lo = __builtin_amdgcn_readlane(lo_excl, owner);
    hi = __builtin_amdgcn_readlane(hi_excl, owner);
#pragma unroll
    for (int i = 0; i + 1 < PER_LANE; ++i)
      if (i < at % PER_LANE) {
        const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)cell[i], owner);
        lo += (int)(c & 0xffffu);
        hi += (int)(c >> 16);
      }
  };
  if (linear) {  // uniform
    // By group maxima, m `take` members leave 1.66 `take` keys at the bound for m
    // = 5 and 1.27 for m = 8, and with fewer groups than `take` all of them; where
    // that could overflow the entries, the histogram takes every key: little more
    // than `take` reach the bound (500 rows of 30K with 3.7K candidates and TOPK
    // 1024 16.6 us, by a radix selection over the row, -> 12.1).
    if (take > TK_ENTRIES / 4 && members > TK_ENTRIES &&
        members < (take <= TK_ENTRIES / 2 ? 5 : 8) * (int64_t)take) {  // uniform
#pragma unroll
      for (int u = 0; u < GROUPS; ++u) {
        if (u * THREADS * 4 >= members) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t k = opaque(key[4 * u + j]);
          if (k != 0u) atomicAdd(&radix.hist[0][bins.of(k)], 1u);
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < GROUPS; ++u)
        if (top[u] != 0u) atomicAdd(&radix.hist[0][bins.of(top[u])], 1u);
    }
    block_barrier();
    if (wave == 0) pick_bin<false, true>(radix, 0, TK_BINS, take, lane);
    block_barrier();
    bound = bins.lower_bound(radix.choice[0]);  // fewer groups than `take`: bin 0, every key

    // ---- 2. the keys that reach it, in position order ---------------------------
    scan_cells([&](int u) {
      int c = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) c += key[4 * u + j] >= bound ? 1 : 0;
      return c;
    });
    read_cells();
    n = lo_total;
  }
  if (n <= TK_ENTRIES) {  // uniform
#pragma unroll
    for (int u = 0; u < GROUPS; ++u) {
      if (!used(u)) continue;
      int slot, unused;
      cell_base(u, slot, unused);
      slot += (int)before[u];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t k = opaque(key[4 * u + j]);
        if (k >= bound) {
          entry_key[slot] = k;
          entry_pos[slot] = position(4 * u + j);
          ++slot;
        }
      }
    }
    block_barrier();

    // ---- 3. the threshold among them: thread t holds entries PER_THREAD t + e ----
    uint32_t k[PER_THREAD];
    int p[PER_THREAD];
#pragma unroll
    for (int e = 0; e < PER_THREAD; ++e) {
      const int i = tid * PER_THREAD + e;
      k[e] = i < n ? entry_key[i] : 0u;
      p[e] = entry_pos[i];
    }
    bins.set(max(bound, low), high);
#pragma unroll
    for (int e = 0; e < PER_THREAD; ++e)
      if (k[e] != 0u) atomicAdd(&radix.hist[1][bins.of(k[e])], 1u);
    block_barrier();
    if (wave == 0)
      pick_bin<false, true>(radix, 1, TK_BINS, take, lane);
    else
      for (int i = tid - 64; i < TK_BINS; i += THREADS - 64) radix.hist[0][i] = 0u;
    block_barrier();
    const int bin = radix.choice[0], inside = radix.choice[2];
    int need = take - radix.choice[1];
    uint32_t threshold;
    if (inside <= TK_SMALL) {  // uniform
#pragma unroll
      for (int e = 0; e < PER_THREAD; ++e)
        if (k[e] != 0u && bins.of(k[e]) == bin) small_key[atomicAdd(&small_count, 1)] = k[e];
      block_barrier();
      threshold = rank_small(small_key, inside, lane, &need);
    } else {
      int parity = 0;
      threshold = radix_select<THREADS, false>(
          [&](auto f) {
#pragma unroll
            for (int e = 0; e < PER_THREAD; ++e)
              if (k[e] != 0u && bins.of(k[e]) == bin) f(k[e]);
          },
          need, radix, parity, &need);
    }

    // ---- 4. the taken entries, in order --------------------------------------
    int c = 0;
#pragma unroll
    for (int e = 0; e < PER_THREAD; ++e) c += k[e] > threshold ? 1 : (k[e] == threshold ? 0x10000 : 0);
    const int incl = wave_inclusive_scan(c);
    if (lane == 63) cells[wave] = (uint32_t)incl;
    block_barrier();
    int above = 0, equal = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
      if (w < wave) {
        above += (int)(cells[w] & 0xffffu);
        equal += (int)(cells[w] >> 16);
      }
    above += (incl - c) & 0xffff;
    equal += (int)((uint32_t)(incl - c) >> 16);
#pragma unroll
    for (int e = 0; e < PER_THREAD; ++e) {
      const bool gt = k[e] > threshold, eq = k[e] == threshold;
      const int slot = above + min(equal, need);
      if ((gt || (eq && equal < need)) && slot < take) emit(slot, k[e], p[e]);
      above += gt ? 1 : 0;
      equal += eq ? 1 : 0;
    }
    return;
  }

  // ---- the whole row: radix selection (its keys formed again from memory, a
  // loop over the registers would be unrolled three times), then the same
  // counts and slots over the registers.
  block_barrier();  // every wave has read the cells and the choice
  for (int i = tid; i < TK_BINS; i += THREADS) radix.hist[0][i] = 0u;
  block_barrier();
  int parity = 0, need = 0;
  const uint32_t threshold = radix_select<THREADS, false>(
      [&](auto f) {
        for (int u = 0; u < GROUPS && u * THREADS * 4 < members; ++u) {
          const u32x4 x = load_group(u);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t k = MODE == TK_MERGE                 ? x[j]
                               : position(4 * u + j) < cand ? score_key(__uint_as_float(x[j]))
                                                                : 0u;
            if (k != 0u) f(k);
          }
        }
      },
      take, radix, parity, &need);
  scan_cells([&](int u) {
    int c = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) c += key[4 * u + j] > threshold ? 1 : (key[4 * u + j] == threshold ? 0x10000 : 0);
    return c;
  });
  read_cells();
#pragma unroll
  for (int u = 0; u < GROUPS; ++u) {
    if (!used(u)) continue;
    int above, equal;
    cell_base(u, above, equal);
    above += (int)(before[u] & 0xffffu);
    equal += (int)(before[u] >> 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t k = opaque(key[4 * u + j]);
      const bool gt = k > threshold, eq = k == threshold;
      const int slot = above + min(equal, need);
      if ((gt || (eq && equal < need)) && slot < take) emit(slot, k, position(4 * u + j));
      above += gt ? 1 : 0;
      equal += eq ? 1 : 0;
    }
  }
}

// Streaming form, for rows of any length: every digit re-reads the row, and
// the output is written chunk by chunk in position order (one scan per chunk
// of THREADS positions, counting keys equal to the threshold in the high
// half-word and keys above it in the low one).
__global__ __launch_bounds__(TK_STREAM_THREADS) void sparse_topk_stream(TopkArgs a) {
  constexpr int THREADS = TK_STREAM_THREADS;
  __shared__ RadixLds<false> radix;
  __shared__ int scan_scratch[2 * THREADS / 64];
  const int token = blockIdx.x, tid = threadIdx.x;
  const TokenBounds tb = token_bounds(a, token);
  int32_t* out = a.indices + (size_t)token * a.TOPK;
  if (trivial_selection<THREADS>(a, tb, out)) return;
  const float* row = a.scores + (size_t)token * a.C;
  const int cand = tb.cand;
  for (int i = tid; i < TK_BINS; i += THREADS) radix.hist[0][i] = 0u;
  __syncthreads();
  int parity = 0, need = 0;
  const uint32_t threshold = radix_select<THREADS>(
      [&](auto f) {
        for (int i = tid; i < cand; i += THREADS) f(score_key(row[i]));
      },
      tb.take, radix, parity, &need);

  int written = 0, equal_seen = 0;
  for (int base = 0; base < cand; base += THREADS) {
    const int i = base + tid;
    const uint32_t k = i < cand ? score_key(row[i]) : 0u;
    const bool gt = k > threshold, eq = k == threshold;  // k == 0 past the row
    int above = gt ? 1 : 0, equal = eq ? 1 : 0, both[2];
    block_exclusive_scan2<THREADS>(above, equal, scan_scratch, both);
    const int eq_left = max(0, need - equal_seen);  // equal keys still to take
    const int at = written + above + min(equal, eq_left);
    if ((gt || (eq && equal < eq_left)) && at < tb.take) out[at] = i;
    written += both[0] + min(both[1], eq_left);
    equal_seen += both[1];
    if (written >= tb.take) break;  // uniform: every thread sees the same totals
  }
}

}  // namespace afa

using namespace afa;

// Form of a call. ROW and SPLIT are the register forms (sparse_topk_row), for
// calls of few enough tokens that a row's chain of steps, not the scores'
// bytes, sets the time; FILTER and STREAM the streaming ones.
enum TopkForm { TK_FORM_ROW, TK_FORM_SPLIT, TK_FORM_FILTER, TK_FORM_STREAM };
struct TopkPlan {
  TopkForm form;
  int threads, items;  // ROW
  int segments, keep;  // SPLIT: segments of TK_SEGMENT_SIZE positions, entries kept of each
  int64_t tokens;      // SPLIT: tokens per pair of launches
};
constexpr int64_t TK_MERGE_MAX = 1024 * 32;  // entries of all segments of a row
constexpr int64_t TK_SPLIT_WORKGROUPS = 2048;
constexpr int64_t TK_SPLIT_BYTES = int64_t(64) << 20;  // workspace of a call, at most (one token at least)

// Lines of the form. A buffer's columns say little of its tokens' candidates, and
// the streaming form's time follows those more closely; the register form is
// taken up to where it is faster with half of the columns as candidates and at
// most about a tenth slower with a quarter, at every share for calls of up to 512
// tokens (decode, in buffers of its largest context). Measured either side (us,
// register form / streaming form; all, half, a quarter, an eighth of the columns;
// TOPK 512 unless stated): 500 rows of 30K 26 / 69, 18 / 37, 13 / 16, 11.3 / 13.2; 1000
// 45 / 74, 31 / 45, 24 / 22, 20 / 17; 1000 of 20K 0.72x, 0.72x, 1.15x, 1.25x, with TOPK 256
// 0.98x, 0.98x, 1.07x, 1.34x; 2000 of 16K 40 / 54, 30 / 32, 25 / 23, 24 / 23, 3000 0.82x,
// 1.00x, 1.10x, 1.11x, 5000 0.86x, 1.08x, 1.18x, 1.20x, with TOPK 1024
// 0.84x, 0.98x, 0.96x, 0.87x; 1300 of 16K with TOPK 256 0.93x, 0.93x, 1.04x, 0.95x, 2000
// 0.93x, 1.05x, 1.14x, 1.05x; 2000 of 8K 0.79x, 0.92x, 0.90x, 0.79x; of 700 with TOPK
// 256 0.91x, 1.16x.
// Split rows, 64 tokens: of 66K 20.2 / 22.0, 17.1 / 16.0, 16.5 / 12.6; of 100K 22.5 / 28.6,
// 17 / 19, 16 / 14; of 256K 36 / 98, 25 / 54, 19.3 / 21.1, 17.8 / 15.2; 96 tokens: of 181K
// 0.93x, 1.03x, 1.16x, of 215K 0.65x, 0.97x, 1.15x; 128 tokens: of 128K 34.7 / 33.6; of
// 200K 48.7 / 47.8, 32.9 / 29.9, 26.3 / 20.6; of 256K 58 / 99, 37 / 56, 28 / 22.
// Candidates past one segment and up to about 40K lose 1 to 5 us to the second
// launch; up to one segment there is nothing to merge (11.5 / 11.8).
static TopkPlan choose_topk(const SparseTopkParams* p, bool with_workspace) {
  TopkPlan plan{};
  const int64_t C = p->C, T = p->T;
  const bool fits = p->TOPK <= 1408;  // entries, whatever the candidates (see the bound)
  const int64_t most = C > 24576   ? 1024
                       : C > 16384 ? (p->TOPK > 256 ? 1024 : 512)
                       : C > 8192  ? (p->TOPK > 512 ? 5120 : p->TOPK > 256 ? 3072 : 1300)
                       : C > 1024  ? 2048
                                   : 1024;
  if (C <= 32768 && T <= most && fits) {
    plan.form = TK_FORM_ROW;
    // One 1024-thread workgroup per CU while every token gets a CU of its own,
    // smaller workgroups, more of which share a CU, beyond.
    plan.threads = T <= 256 ? 1024 : 512;
    plan.items = 4;
    while ((int64_t)plan.threads * plan.items < C) plan.items *= 2;
    if (plan.threads == 512) plan.items = std::max(plan.items, 8);
    return plan;
  }
  const int64_t segments = (C + TK_SEGMENT_SIZE - 1) / TK_SEGMENT_SIZE;
  const int64_t keep = (std::min<int64_t>(p->TOPK, TK_SEGMENT_SIZE) + 3) / 4 * 4;
  const bool few = T <= 64 || (segments >= (T <= 96 ? 13 : 15) && T * segments <= TK_SPLIT_WORKGROUPS);
  if (with_workspace && segments * keep <= TK_MERGE_MAX &&
      (C > TK_FILTER_MAX_C || (segments >= 6 && few && fits))) {
    plan.form = TK_FORM_SPLIT;
    plan.segments = (int)segments;
    plan.keep = (int)keep;
    plan.tokens = std::min(T, std::max<int64_t>(1, TK_SPLIT_BYTES / (segments * keep * 8)));
    return plan;
  }
  plan.form = C <= TK_FILTER_MAX_C ? TK_FORM_FILTER : TK_FORM_STREAM;
  return plan;
}

static uint64_t topk_split_bytes(const SparseTopkParams* p, const TopkPlan& plan) {
  return plan.form == TK_FORM_SPLIT ? (uint64_t)plan.tokens * plan.segments * plan.keep * 8 : 0;
}

static int check_topk(const SparseTopkParams* params) {
  if (!params) return AFA_E_NULL;
  if (params->B <= 0 || params->T <= 0 || params->TOPK <= 0 || params->C <= 0) return AFA_E_SHAPE;
  if (params->RATIO != 1 && params->RATIO != 2) return AFA_E_SHAPE;
  if (params->C > 0x7fffffffLL) return AFA_E_SHAPE;
  return AFA_OK;
}

template <int THREADS, int ITEMS, int MODE>
static void launch_row(const TopkArgs& a, dim3 grid, hipStream_t s) {
  hipLaunchKernelGGL((sparse_topk_row<THREADS, ITEMS, MODE>), grid, dim3(THREADS), 0, s, a);
}

static int launch_topk(hipStream_t s, const float* scores, const int32_t* cu_seqlens_q, const int32_t* seqused_cmp_kv,
                       const int32_t* cmp_residual_kv, int32_t* cmp_sparse_indices, void* workspace,
                       const SparseTopkParams* params, const TopkPlan& plan) {
  TopkArgs a;
  a.scores = scores;
  a.cu = cu_seqlens_q;
  a.seq_cmp = seqused_cmp_kv;
  a.residual = cmp_residual_kv;
  a.indices = cmp_sparse_indices;
  a.C = params->C;
  a.B = params->B;
  a.T = params->T;
  a.TOPK = params->TOPK;
  a.RATIO = params->RATIO;
  a.cap = a.words = a.first_token = a.segments = a.seg_keep = 0;
  a.seg_key = nullptr;
  a.seg_pos = nullptr;
  const dim3 grid((unsigned)a.T);
  switch (plan.form) {
    case TK_FORM_ROW:
      switch (plan.threads * 100 + plan.items) {
        case 102404: launch_row<1024, 4, TK_ROW>(a, grid, s); break;
        case 102408: launch_row<1024, 8, TK_ROW>(a, grid, s); break;
        case 102416: launch_row<1024, 16, TK_ROW>(a, grid, s); break;
        case 102432: launch_row<1024, 32, TK_ROW>(a, grid, s); break;
        case 51208: launch_row<512, 8, TK_ROW>(a, grid, s); break;
        case 51216: launch_row<512, 16, TK_ROW>(a, grid, s); break;
        case 51232: launch_row<512, 32, TK_ROW>(a, grid, s); break;
        default: launch_row<512, 64, TK_ROW>(a, grid, s); break;
      }
      break;
    case TK_FORM_SPLIT: {
      a.segments = plan.segments;
      a.seg_keep = plan.keep;
      a.seg_key = (uint32_t*)workspace;
      a.seg_pos = (int32_t*)workspace + (size_t)plan.tokens * a.segments * a.seg_keep;
      const int entries = a.segments * a.seg_keep;
      for (int64_t t = 0; t < a.T; t += plan.tokens) {
        a.first_token = (int32_t)t;
        const unsigned n = (unsigned)std::min<int64_t>(plan.tokens, a.T - t);
        launch_row<1024, TK_SEGMENT_ITEMS, TK_SEGMENT>(a, dim3(n, (unsigned)a.segments), s);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return (int)e;
        if (entries <= 1024 * 4)
          launch_row<1024, 4, TK_MERGE>(a, dim3(n), s);
        else if (entries <= 1024 * 16)
          launch_row<1024, 16, TK_MERGE>(a, dim3(n), s);
        else
          launch_row<1024, 32, TK_MERGE>(a, dim3(n), s);
        const hipError_t m = hipGetLastError();
        if (m != hipSuccess) return (int)m;
      }
      break;
    }
    case TK_FORM_FILTER: {
      a.words = (int32_t)((a.C + 31) / 32);
      // Buffer: rows up to 32K positions (16-bit positions) hold 2 TOPK entries,
      // between 1024 and 8192, so that little of a CU's LDS is spent on it at the
      // usual TOPK; longer rows hold TK_WIDE_CAP.
      a.cap = a.C <= 32768
                  ? (int32_t)std::min<int64_t>(8192, std::max<int64_t>(1024, ((int64_t)a.TOPK * 2 + 255) / 256 * 256))
                  : TK_WIDE_CAP;
      const size_t dynamic_bytes = 2 * 4 * (size_t)a.words + (a.C <= 32768 ? (size_t)a.cap * 6 : 0);
      // Rows up to 32K positions: 256 threads, more workgroups per CU; longer
      // rows: 1024 threads, more loads in flight per row.
      if (a.C <= 32768) {
        hipLaunchKernelGGL(sparse_topk_filter<256>, grid, dim3(256), dynamic_bytes, s, a);
      } else {
        hipLaunchKernelGGL(sparse_topk_filter<1024>, grid, dim3(1024), dynamic_bytes, s, a);
      }
      break;
    }
    default: hipLaunchKernelGGL(sparse_topk_stream, grid, dim3(TK_STREAM_THREADS), 0, s, a); break;
  }
  return (int)hipGetLastError();
}

extern "C" int launch_sparse_topk_indices(void* stream, const float* scores, const int32_t* cu_seqlens_q,
                                          const int32_t* seqused_cmp_kv, const int32_t* cmp_residual_kv,
                                          int32_t* cmp_sparse_indices, const SparseTopkParams* params) {
  const int status = check_topk(params);
  if (status) return status;
  if (!scores || !cu_seqlens_q || !seqused_cmp_kv || !cmp_residual_kv || !cmp_sparse_indices) return AFA_E_NULL;
  return launch_topk((hipStream_t)stream, scores, cu_seqlens_q, seqused_cmp_kv, cmp_residual_kv, cmp_sparse_indices,
                     nullptr, params, choose_topk(params, false));
}

extern "C" int workspace_size_sparse_topk_indices_split(uint64_t* bytes, const SparseTopkParams* params) {
  if (!bytes) return -1;
  const int status = check_topk(params);
  if (status) return status;
  *bytes = topk_split_bytes(params, choose_topk(params, true));
  return AFA_OK;
}

extern "C" int launch_sparse_topk_indices_split(void* stream, const float* scores, const int32_t* cu_seqlens_q,
                                                const int32_t* seqused_cmp_kv, const int32_t* cmp_residual_kv,
                                                int32_t* cmp_sparse_indices, void* workspace, uint64_t workspace_bytes,
                                                const SparseTopkParams* params) {
  const int status = check_topk(params);
  if (status) return status;
  if (!scores || !cu_seqlens_q || !seqused_cmp_kv || !cmp_residual_kv || !cmp_sparse_indices) return AFA_E_NULL;
  const TopkPlan plan = choose_topk(params, true);
  const uint64_t need = topk_split_bytes(params, plan);
  if (need > 0 && (!workspace || workspace_bytes < need)) return AFA_E_WORKSPACE;
  return launch_topk((hipStream_t)stream, scores, cu_seqlens_q, seqused_cmp_kv, cmp_residual_kv, cmp_sparse_indices,
                     workspace, params, plan);
}

extern "C" int form_sparse_topk_indices(int64_t form[3], const SparseTopkParams* params, int with_workspace) {
  if (!form) return AFA_E_NULL;
  const int status = check_topk(params);
  if (status) return status;
  const TopkPlan plan = choose_topk(params, with_workspace != 0);
  form[0] = plan.form;
  form[1] = plan.form == TK_FORM_ROW ? plan.threads : plan.form == TK_FORM_SPLIT ? plan.segments : 0;
  form[2] = plan.form == TK_FORM_ROW ? plan.items : plan.form == TK_FORM_SPLIT ? plan.tokens : 0;
  return AFA_OK;
}
