// Flash attention forward (BNSD) and the teaching single-tile attention for
// gfx950.
//
// attention_target: examples/flash_attention/attention.py:243-417. The
// reference's Cube/Vector stages (QK -> Score GM -> online softmax -> P GM ->
// PV -> PV GM -> rescale/update) collapse into one kernel per (batch, head,
// query tile): K and V chunks stream through double-buffered, XOR-swizzled
// LDS; each wave owns QT*16 query rows with Q resident in registers;
// S^T[keys, queries] = K * Q^T and O^T[d, queries] += V^T * P^T run on
// v_mfma_f32_16x16x32_{f16,bf16}; the online softmax (attention.py:73-139:
// m' = max(m, rowmax s), alpha = e^(m-m'), l = l*alpha + sum p, O = O*alpha +
// b16(p) V) stays in FP32 registers; V^T fragments come through
// ds_read_b64_tr_b16. Causal masking is top-left (key j visible to query i iff
// j <= i, attention.py:96-110); keys >= Sk and queries >= Sq are masked.
//
// simple_attention: examples/flash_attention/simple.py:60-141. One 128-key
// tile per head: S = Q K^T * 128^-1/2, P = f16(softmax(S)) normalised BEFORE
// the cast, O = f16(P V) (simple.py:25-57).
#include <algorithm>
#include <cmath>

#include "common.h"
#include "../../include/ascendflow_amd.h"

namespace afa {

constexpr float FA_LOG2E = 1.4426950408889634f;

struct FaArgs {
  const void* q;
  const void* k;
  const void* v;
  void* o;
  int64_t Sq, Sk;
  int32_t B, HQ, HKV, causal;
  int32_t level_order;  // causal forward kernel: the longest tiles of all heads first
  float scale;
};


// Flash-attention forward for D = 128. One workgroup of NW waves owns BQ =
// NW * QT * 16 query rows of one (batch, head); each wave owns QT 16-row query
// tiles with Q resident in registers. K and V stream in KC-key chunks through
// an LDS ring filled by the load-to-LDS path (rows XOR-swizzled on the global
// side, unit u of row r at u ^ (r & 15)): three slots each for NW = 8, K and V
// two chunks ahead; two for NW = 4, K two chunks ahead and V one, so that two
// workgroups fit a CU (128- or 64-row tiles: less of a ragged, short or causal
// problem is padding, and one workgroup's start and barriers run under the
// other's work; per row of a long one K and V are loaded two or four times as
// often, and 8192 x 8192 takes 990 / 1062 / 1350 us at 256 / 128 / 64 rows).
// S^T[keys, queries] = K * Q^T and O^T[d, queries] += V^T * P^T run on
// v_mfma_f32_16x16x32_{f16,bf16}; V^T fragments come through
// ds_read_b64_tr_b16. Per chunk c the QK MFMAs of chunk c + 1 are issued
// ahead of the softmax of chunk c, so they run under its VALU work.
//
// Online softmax (attention.py:73-139) in FP32 registers, exp2 domain: the
// chunk max is taken on raw scores (the scale is positive) and the scale goes
// into the exponent's FMA; the running max is raised, with O and l rescaled
// by alpha = 2^(m - m'), only when some query's max exceeds it by more than
// fa_tau, so P <= 2^fa_tau; O / l is independent of the reference point. The
// lazy reference point rounds the P of the key holding the running max to the
// storage dtype, where the reference's recurrence has P = 1 exactly: a
// relative error of at most 2^-12 in f16 (within its contract; eager rescaling
// measured 5% slower on FA C2) but 2^-9 in bf16, which with sharp scores moved
// outputs by 2 ulps, so bf16 raises the max whenever it grows (fa_tau = 0).
// Masks (attention.py:96-110): keys >= Sk, and for causal attention key j is
// visible to query i iff j <= i (top-left); they are applied only in chunks
// that reach the tail or the diagonal.
template <int DT> __device__ constexpr float fa_tau() { return DT == DT_F16 ? 8.0f : 0.0f; }
// Progress-ordered wave priorities: a wave starts each chunk at priority 3
// and steps down at half of QK, after QK and at half of PV, so of the two waves
// sharing a SIMD the one behind wins the MFMA arbitration (otherwise the older
// wave always wins, finishes first and waits at the barrier while the other
// runs alone).
constexpr bool FA_PROGRESS_PRIO = true;

template <int DT, int NW, int QT>
__global__ __launch_bounds__(NW * 64, NW == 8 ? 1 : 2) void fa_forward_kernel(FaArgs a) {
  typedef typename B16<DT>::scalar scalar;
  typedef typename B16<DT>::x8 x8;
  typedef typename B16<DT>::x4 x4;
  constexpr int D = 128, ROW_BYTES = 2 * D, UNITS = D / 8;
  constexpr int KC = 64;                       // keys per chunk
  constexpr int KT = KC / 16;                  // key tiles per chunk
  constexpr int TILE = KC * ROW_BYTES;         // bytes of one K or V tile
  constexpr int BQ = NW * QT * 16;
  constexpr int NS = NW == 8 ? 3 : 2;          // ring slots per tensor
  constexpr int ROWS_PER_LOAD = 64 / UNITS;    // rows one wave load covers
  constexpr int LOADS = KC / ROWS_PER_LOAD / NW;  // wave loads per tensor per chunk
  static_assert(LOADS * ROWS_PER_LOAD * NW == KC, "a chunk must split evenly over the waves");

  __shared__ __attribute__((aligned(16))) uint8_t kv_lds[NS][2][TILE];  // [slot][K, V]

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = lane >> 4, i16 = lane & 15;
  const int64_t q_tiles = (a.Sq + BQ - 1) / BQ;
  int64_t qtile, bh;
  if (a.level_order) {
    // Tiles of all heads from the longest down. The dispatcher deals workgroups
    // to an XCD's shader engines in turn, so with a head's tiles in a row and
    // an even number of them, engine 0 got the long ones of every head (B2
    // HQ32 HKV8 S1987 126 -> 80 us with this and 128-row tiles; 256-row tiles, B1
    // HQ32 S4096 211 -> 147). Heads that share a KV head stay on one XCD (blocks
    // go to XCD blockIdx % 8). All heads' keys are read again at every level:
    // only while they stay in the Infinity Cache (FA_LEVEL_BYTES).
    const uint32_t heads = (uint32_t)a.B * (uint32_t)a.HQ;
    const uint32_t level = blockIdx.x / heads, i = blockIdx.x % heads;
    qtile = q_tiles - 1 - level;
    bh = (heads & 7u) ? i : (i & 7u) * (heads >> 3) + (i >> 3);
  } else {
    const uint32_t logical = xcd_contiguous(blockIdx.x, gridDim.x);
    qtile = (int64_t)(logical % q_tiles);
    if (a.causal) qtile = q_tiles - 1 - qtile;
    bh = logical / q_tiles;
  }
  const int head = (int)(bh % a.HQ), batch = (int)(bh / a.HQ);
  const int kv_head = head / (a.HQ / a.HKV);
  const int64_t q0 = qtile * BQ;

  const scalar* Q = (const scalar*)a.q + ((int64_t)batch * a.HQ + head) * a.Sq * D;
  const char* K = (const char*)a.k + ((int64_t)batch * a.HKV + kv_head) * a.Sk * ROW_BYTES;
  const char* V = (const char*)a.v + ((int64_t)batch * a.HKV + kv_head) * a.Sk * ROW_BYTES;
  scalar* O = (scalar*)a.o + ((int64_t)batch * a.HQ + head) * a.Sq * D;

  // Q fragments: B operand of S^T = K * Q^T; query of tile qt: q0 + (wave*QT + qt)*16 + i16.
  x8 qf[QT][D / 32];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int64_t row = q0 + (wave * QT + qt) * 16 + i16;
#pragma unroll
    for (int j = 0; j < D / 32; ++j)
      qf[qt][j] = row < a.Sq ? *(const x8*)(Q + row * D + 32 * j + 8 * g) : __builtin_bit_cast(x8, u32x4{0u, 0u, 0u, 0u});
  }

  int64_t kv_end = a.Sk;
  if (a.causal) kv_end = min(a.Sk, q0 + BQ);  // keys past the tile's last query are masked
  const int chunks = (int)((kv_end + KC - 1) / KC);
  // First chunk that needs masking: it reaches Sk or (causal) the tile's first query.
  int64_t clean_end = a.Sk;
  if (a.causal) clean_end = min(clean_end, q0 + 1);
  const int clean_chunks = (int)(clean_end / KC);

  // ---- KV movement ---------------------------------------------------------
  const uint32_t kv_base = lds_address(kv_lds[0][0]);
  auto tile_address = [&](int chunk, int tensor) {
    return opaque_uniform(kv_base + (uint32_t)((chunk % NS) * 2 + tensor) * TILE);
  };
  // Wave load p of a chunk covers rows [(wave*LOADS + p)*ROWS_PER_LOAD, +ROWS_PER_LOAD);
  // this lane lands on unit (lane % UNITS) of row lane / UNITS and loads unit
  // (lane % UNITS) ^ (row & 15) of that row. Two loads per wave (NW = 8) keep
  // their offsets in registers; of four, whose registers would spill, loads 1-3
  // are load 0 with the swizzle's bits 4p flipped, 4p rows on (a wave's rows
  // then start at a multiple of 16, so the row bits add without carry).
  constexpr int OFFSETS = LOADS == 2 ? 2 : 1;
  static_assert(ROWS_PER_LOAD == 4 && (LOADS == 2 || LOADS == 4), "loads of a wave");
  uint32_t load_offset[OFFSETS];
#pragma unroll
  for (int p = 0; p < OFFSETS; ++p) {
    const int r = (wave * LOADS + p) * ROWS_PER_LOAD + lane / UNITS;
    load_offset[p] = (uint32_t)(r * ROW_BYTES + (((lane % UNITS) ^ (r & 15)) << 4));
  }
  // Rows past Sk read the last key instead (masked later).
  auto tail_offset = [&](int64_t key0, int p) {
    const int r = (wave * LOADS + p) * ROWS_PER_LOAD + lane / UNITS;
    const int rr = (int)min((int64_t)r, a.Sk - 1 - key0);
    return (uint32_t)(rr * ROW_BYTES + (((lane % UNITS) ^ (r & 15)) << 4));
  };
  auto fetch = [&](int chunk) {  // K and V (three slots)
    const int64_t key0 = (int64_t)chunk * KC;
    const char* kbase = K + key0 * ROW_BYTES;
    const char* vbase = V + key0 * ROW_BYTES;
    const bool tail = key0 + KC > a.Sk;
#pragma unroll
    for (int p = 0; p < LOADS; ++p) {
      uint32_t off = load_offset[p < OFFSETS ? p : 0];
      if (tail) off = tail_offset(key0, p);
      const uint32_t row0 = (uint32_t)((wave * LOADS + p) * ROWS_PER_LOAD * ROW_BYTES);
      const uint32_t kd = tile_address(chunk, 0) + row0, vd = tile_address(chunk, 1) + row0;
      __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                       :: "s"(kd), "v"(off), "s"(kbase) : "memory");
      __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                       :: "s"(vd), "v"(off), "s"(vbase) : "memory");
    }
  };
  auto fetch_one = [&](int chunk, int tensor) {  // two slots
    const int64_t key0 = (int64_t)chunk * KC;
    const char* base = (tensor ? V : K) + key0 * ROW_BYTES;
    const uint32_t tile = tile_address(chunk, tensor);
    const bool tail = key0 + KC > a.Sk;
#pragma unroll
    for (int p = 0; p < LOADS; ++p) {
      uint32_t off =
          p < OFFSETS ? load_offset[p] : (load_offset[0] ^ (uint32_t)(p << 6)) + (uint32_t)(p * 4 * ROW_BYTES);
      if (tail) off = tail_offset(key0, p);
      __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                       :: "s"(tile + (uint32_t)((wave * LOADS + p) * ROWS_PER_LOAD * ROW_BYTES)), "v"(off), "s"(base)
                       : "memory");
    }
  };

  // ---- fragment addressing ---------------------------------------------------
  const int ra = sigma(i16);                 // K fragment row inside a 16-key tile
  const int rt = sigma(4 * g + (i16 >> 2));  // transposing-read row inside a tile
  uint32_t qk_base[D / 32], tr_base[D / 16];
#pragma unroll
  for (int j = 0; j < D / 32; ++j) qk_base[j] = (uint32_t)(ra * ROW_BYTES + (((4 * j + g) ^ (ra & 15)) << 4));
#pragma unroll
  for (int t = 0; t < D / 16; ++t)
    tr_base[t] = (uint32_t)(rt * ROW_BYTES + (((2 * t + ((i16 & 3) >> 1)) ^ (rt & 15)) << 4) + (i16 & 1) * 8);

  f32x4 o[QT][D / 16];
  float m_run[QT], l_run[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    m_run[qt] = -1e30f;  // finite: a fully masked chunk then gives p = 0, never NaN
    l_run[qt] = 0.f;
#pragma unroll
    for (int t = 0; t < D / 16; ++t) o[qt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float scale_log2 = a.scale * FA_LOG2E;

  // S^T of one chunk: K fragments LOOK steps ahead of their MFMAs. After the
  // MFMAs of fragment f, between(f) issues independent VALU work (the softmax
  // of the previous chunk), which runs in the shadow of the MFMA pipe.
  constexpr int QK_FRAGS = (D / 32) * KT;  // 16 fragments, each feeds QT MFMAs
  constexpr int LOOK = 6;
  auto qk_chunk = [&](int chunk, f32x4 (&s)[KT][QT], auto&& between) {
    const uint32_t tile = tile_address(chunk, 0);
    uint32_t base[D / 32];
#pragma unroll
    for (int j = 0; j < D / 32; ++j) base[j] = opaque(tile + qk_base[j]);
    x8 kf[QK_FRAGS];
    auto load = [&](int f) {  // fragment f = (j, t): k-step j, key tile t
      const int j = f / KT, t = f % KT;
      kf[f] = *(const AFA_LDS x8*)(lds_at<uint8_t>(base[j]) + t * 16 * ROW_BYTES);
    };
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) s[t][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int f = 0; f < LOOK && f < QK_FRAGS; ++f) load(f);
#pragma unroll
    for (int f = 0; f < QK_FRAGS; ++f) {
      if (f + LOOK < QK_FRAGS) load(f + LOOK);
      const int j = f / KT, t = f % KT;
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) s[t][qt] = B16<DT>::mfma(kf[f], qf[qt][j], s[t][qt]);
      between(f);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // O^T[d, q] += V^T[d, keys] * P^T[keys, q], with between(f) as in qk_chunk.
  constexpr int PV_FRAGS = (KC / 32) * (D / 16);  // 16 fragments, each feeds QT MFMAs
  auto pv_chunk = [&](int chunk, x8 (&pf)[QT][KC / 32], auto&& between) {
    const uint32_t tile = tile_address(chunk, 1);
    uint32_t vb[D / 16];
#pragma unroll
    for (int t = 0; t < D / 16; ++t) vb[t] = opaque(tile + tr_base[t]);
    constexpr int VLOOK = 3;
    x4 vlo[PV_FRAGS], vhi[PV_FRAGS];
    auto vload = [&](int f) {  // f = (ks, t)
      const int ks = f / (D / 16), t = f % (D / 16);
      const AFA_LDS uint8_t* p = lds_at<uint8_t>(vb[t]) + ks * 32 * ROW_BYTES;
      vlo[f] = B16<DT>::read_tr((const AFA_LDS void*)p);
      vhi[f] = B16<DT>::read_tr((const AFA_LDS void*)(p + 16 * ROW_BYTES));
    };
#pragma unroll
    for (int f = 0; f < VLOOK; ++f) vload(f);
#pragma unroll
    for (int f = 0; f < PV_FRAGS; ++f) {
      if (f + VLOOK < PV_FRAGS) vload(f + VLOOK);
      const int ks = f / (D / 16), t = f % (D / 16);
      const x8 vf = {vlo[f][0], vlo[f][1], vlo[f][2], vlo[f][3], vhi[f][0], vhi[f][1], vhi[f][2], vhi[f][3]};
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) o[qt][t] = B16<DT>::mfma(vf, pf[qt][ks], o[qt][t]);
      between(f);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Scores of keys at or past a per-column limit (the tail chunk and the
  // causal diagonal) become -inf; 32-bit chunk-relative indices. This lane
  // holds query (column) i16 of each query tile and keys 16t + sigma(4g + i).
  auto mask = [&](int chunk, f32x4 (&s)[KT][QT]) {
    const int64_t key0 = (int64_t)chunk * KC;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const int64_t query = q0 + (wave * QT + qt) * 16 + i16;
      int64_t limit = a.Sk - key0;
      if (a.causal) limit = limit < query - key0 + 1 ? limit : query - key0 + 1;
      const int lim = limit < 0 ? 0 : (limit > KC ? KC : (int)limit);
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[t][qt][i] = 16 * t + sigma(4 * g + i) < lim ? s[t][qt][i] : -INFINITY;
    }
  };

  // ---- pipeline: chunk c+2 loads, QK(c+1) + softmax(c), PV(c) + softmax(c) --
  // Chunk c's scores are in cur (masked at the top of its iteration) and
  // QK(c+1) writes nxt; the loop is unrolled by two so the two score buffers
  // alternate without copies. The softmax of chunk c is spread over the MFMA
  // steps: the first QT steps of QK(c+1) take the column maxima, the next two
  // the cross-lane reduction and the (rare, uniform) rescale, the rest the
  // exponentials of key tiles 0-1; the first PV(c) steps, which use only
  // those, take the exponentials of key tiles 2-3.
  constexpr int HALF = QT * 8;                  // exponentials per key-tile pair
  constexpr int QK_EXP0 = QT + 2;               // first QK step with exponentials
  constexpr int PV_EXP_STEPS = PV_FRAGS / 2 - 1;  // PV steps with exponentials
  static_assert(QK_FRAGS > QK_EXP0, "no QK step left for exponentials");
  f32x4 s_a[KT][QT], s_b[KT][QT];
  // Three slots: K and V of chunk c+2 go out together. Two: K(c+2), in K(c)'s
  // place once QK(c) is over, and V(c+1), in V(c-1)'s; V runs one chunk later,
  // and two workgroups fit a CU.
  if (chunks > 0) {
    if constexpr (NS == 3) {
      fetch(0);
      if (chunks > 1) fetch(1);
    } else {
      fetch_one(0, 0);
      fetch_one(0, 1);
      if (chunks > 1) fetch_one(1, 0);
    }
    if (chunks > 1)
      wait_vmcnt<NS == 3 ? 2 * LOADS : LOADS>();  // chunk 0 landed, the rest may be in flight
    else
      wait_vmcnt<0>();
    block_barrier();
    qk_chunk(0, s_a, [](int) {});
  }
  auto iteration = [&](int c, f32x4 (&cur)[KT][QT], f32x4 (&nxt)[KT][QT]) {
    // K(c+1) and V(c) landed (their loads, with V(c+1)'s, are the only ones in
    // flight); after the barrier every wave is past QK(c) and PV(c-1), whose
    // slots are free.
    __builtin_amdgcn_s_waitcnt(0x0F70);
    block_barrier();
    if constexpr (NS == 3) {
      if (c + 2 < chunks) fetch(c + 2);
    } else {
      if (c + 2 < chunks) fetch_one(c + 2, 0);
      if (c + 1 < chunks) fetch_one(c + 1, 1);
    }
    if (c >= clean_chunks) mask(c, cur);

    x8 pf[QT][KC / 32];
    float cmax[QT], m_new[QT], psum[QT];
    auto exp_element = [&](int e) {  // e = (half, qt, t & 1, i)
      const int h = e / HALF, qt = (e / 8) % QT, t = 2 * h + (e / 4) % 2, i = e % 4;
      const float p = fast_exp2(__builtin_fmaf(cur[t][qt][i], scale_log2, -m_run[qt]));
      psum[qt] += p;
      pf[qt][h][(t & 1) * 4 + i] = (scalar)p;
    };
    auto qk_between = [&](int f) {
      if (FA_PROGRESS_PRIO && f == QK_FRAGS / 2 - 1) __builtin_amdgcn_s_setprio(2);
      if (f < QT) {
        float m = -INFINITY;
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) m = fmaxf(m, cur[t][f][i]);
        cmax[f] = m;
      } else if (f == QT) {
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
          m_new[qt] = fmaxf(m_run[qt], max_over_lane_groups(cmax[qt]) * scale_log2);
          psum[qt] = 0.f;
        }
      } else if (f == QT + 1) {
        bool grow = false;
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) grow |= m_new[qt] > m_run[qt] + fa_tau<DT>();
        if (__ballot(grow) != 0ull) {
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) {
            const float alpha = fast_exp2(m_run[qt] - m_new[qt]);
            l_run[qt] *= alpha;
#pragma unroll
            for (int t = 0; t < D / 16; ++t) o[qt][t] *= alpha;
            m_run[qt] = m_new[qt];
          }
        }
      } else {
        // Constant trip counts: the loop unrolls before f is known.
#pragma unroll
        for (int e = 0; e < HALF; ++e)
          if (QK_EXP0 + e * (QK_FRAGS - QK_EXP0) / HALF == f) exp_element(e);
      }
    };
    auto pv_between = [&](int f) {
      if (FA_PROGRESS_PRIO && f == PV_FRAGS / 2 - 1) __builtin_amdgcn_s_setprio(0);
      if (f < PV_EXP_STEPS) {
#pragma unroll
        for (int e = 0; e < HALF; ++e)
          if (e * PV_EXP_STEPS / HALF == f) exp_element(HALF + e);
      } else if (f == PV_EXP_STEPS + 1) {
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) l_run[qt] += psum[qt];
      }
    };

    // The last chunk also runs a QK, over the stale tile of its slot (no load
    // is in flight into it), so that the softmax has one code path; those
    // scores are never read.
    if (FA_PROGRESS_PRIO) __builtin_amdgcn_s_setprio(3);
    qk_chunk(c + 1, nxt, qk_between);
    if (FA_PROGRESS_PRIO) __builtin_amdgcn_s_setprio(1);
    pv_chunk(c, pf, pv_between);
  };
  for (int c = 0; c < chunks; c += 2) {
    iteration(c, s_a, s_b);
    if (c + 1 < chunks) iteration(c + 1, s_b, s_a);
  }

#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int64_t query = q0 + (wave * QT + qt) * 16 + i16;
    const float l = sum_over_lane_groups(l_run[qt]);
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    if (query < a.Sq) {
      scalar* orow = O + query * D + 4 * g;
#pragma unroll
      for (int t = 0; t < D / 16; ++t) {
        x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (scalar)(o[qt][t][i] * inv);
        *(x4*)(orow + 16 * t) = v;
      }
    }
  }
}

// Flash-attention forward of few query rows per KV head (decode, and prefill
// grids too small to fill the GPU). The query rows of the HQ / HKV heads that
// share a KV head are one contiguous block of group * Sq rows of Q and O, so
// they are packed into tiles of 16 * QT rows and every KV row is read once per
// tile instead of once per head. A workgroup owns one (batch, KV head, row
// tile, split): a contiguous range of 32-key tiles, dealt to its four waves in
// turn. Bound by HBM (each KV byte feeds at most 4 * QT * 16 FLOP per row tile),
// so the waves are four independent streams with no barrier in the loop: each
// keeps two K and two V tiles (32 KiB) in flight into an LDS ring of its own
// and waits on its own load counter only. Each wave holds its own running max,
// denominator and O over all its keys; they are combined through LDS at the
// end, and the splits' partial results (FP32) by fa_merge_kernel.
// STREAM: KV loads are non-temporal, for one or two row tiles whose KV is too
// large to stay in the 256 MiB Infinity Cache between calls (FD_STREAM_BYTES).
// Measured, B8 HQ32 HKV8 Sq1 Sk32768 bf16 (1.07 GB of KV), call: 823 -> 160 us
// (6.7 TB/s) against the forward kernel, whose 256 workgroups of 256 query
// rows each read their KV head once per query head; B1 HQ32 HKV8 Sq1 Sk16384
// 389 -> 22 us, B1 HQ32 HKV8 Sq64 Sk8192 207 -> 33 us.
constexpr int FD_KEYS = 32;                        // keys per tile
constexpr int FD_TILE = FD_KEYS * 256;             // bytes of one K or V tile
constexpr int FD_WAVES = 4, FD_SLOTS = 4;          // K, V, K, V of two tiles per wave
constexpr int FD_LOADS = FD_TILE / 1024;           // wave loads per tile
constexpr int FD_MAX_QT = 4;

struct FaSplitArgs {
  FaArgs fa;
  int32_t group;      // HQ / HKV
  int32_t row_tiles;  // tiles of 16 * QT rows per (batch, KV head)
  int32_t splits;
  float* partial_o;   // [splits][B * HQ * Sq][128], normalised by nothing (relative to its max)
  float* partial_ml;  // [splits][B * HQ * Sq][2]: running max (log2 units), denominator
};

template <int DT, int QT, bool STREAM>
__global__ __launch_bounds__(FD_WAVES * 64, 1) void fa_split_kernel(FaSplitArgs args) {
  typedef typename B16<DT>::scalar scalar;
  typedef typename B16<DT>::x8 x8;
  typedef typename B16<DT>::x4 x4;
  constexpr int D = 128, ROW_BYTES = 2 * D, UNITS = D / 8, KT = FD_KEYS / 16, ROWS = 16 * QT;
  const FaArgs& a = args.fa;
  __shared__ __attribute__((aligned(16))) uint8_t ring[FD_WAVES][FD_SLOTS][FD_TILE];
  __shared__ float wave_ml[2][FD_WAVES][ROWS];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = lane >> 4, i16 = lane & 15;
  // Row tiles of one split are neighbours (one XCD: they share its KV rows).
  const uint32_t logical = xcd_contiguous(blockIdx.x, gridDim.x);
  const int row_tile = (int)(logical % (uint32_t)args.row_tiles);
  const uint32_t rest = logical / (uint32_t)args.row_tiles;
  const int split = (int)(rest % (uint32_t)args.splits);
  const int64_t kv = rest / (uint32_t)args.splits;  // batch * HKV + KV head
  const int64_t rows = (int64_t)args.group * a.Sq;  // packed rows of this KV head
  const int64_t row0 = (int64_t)row_tile * ROWS;    // first one of this tile

  const scalar* Q = (const scalar*)a.q + kv * rows * D;
  const char* K = (const char*)a.k + kv * a.Sk * ROW_BYTES;
  const char* V = (const char*)a.v + kv * a.Sk * ROW_BYTES;

  // Keys of the whole tile (causal: up to its largest query), of this split,
  // and the per-column limit (top-left causal: key j visible to query i iff j <= i).
  int64_t kv_end = a.Sk, col_limit[QT], clean = a.Sk;
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) col_limit[qt] = a.Sk;
  if (a.causal) {
    const int64_t last = min(row0 + ROWS, rows) - 1;
    // Rows of one head only, in query order, or rows that cross heads (all queries possible).
    const bool one_head = row0 / a.Sq == last / a.Sq;
    kv_end = min(a.Sk, (one_head ? last % a.Sq : a.Sq - 1) + 1);
    clean = min(a.Sk, (one_head ? row0 % a.Sq : 0) + 1);
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) col_limit[qt] = min(a.Sk, (row0 + 16 * qt + i16) % a.Sq + 1);
  }
  const int tiles = (int)((kv_end + FD_KEYS - 1) / FD_KEYS);
  const int first = (int)((int64_t)tiles * split / args.splits), end = (int)((int64_t)tiles * (split + 1) / args.splits);
  const int n = end - first > wave ? (end - first - wave + FD_WAVES - 1) / FD_WAVES : 0;  // this wave's tiles
  auto tile_of = [&](int i) { return first + wave + i * FD_WAVES; };

  const uint32_t ring_base = lds_address(ring[wave][0]);
  auto slot_address = [&](int i, int tensor) {
    return opaque_uniform(ring_base + (uint32_t)((i & 1) * 2 + tensor) * FD_TILE);
  };
  // Wave load p covers rows 4p .. 4p + 3; this lane lands on unit lane % 16 of
  // row 4p + lane / 16 and loads unit (lane % 16) ^ (row & 15) of that row.
  uint32_t load_offset[FD_LOADS];
#pragma unroll
  for (int p = 0; p < FD_LOADS; ++p) {
    const int r = 4 * p + lane / UNITS;
    load_offset[p] = (uint32_t)(r * ROW_BYTES + (((lane % UNITS) ^ (r & 15)) << 4));
  }
  auto fetch = [&](int i, int tensor) {
    const int64_t key0 = (int64_t)tile_of(i) * FD_KEYS;
    const char* base = (tensor ? V : K) + key0 * ROW_BYTES;
    const uint32_t dst = slot_address(i, tensor);
    const bool tail = key0 + FD_KEYS > a.Sk;  // uniform; rows past Sk read the last key instead (masked later)
#pragma unroll
    for (int p = 0; p < FD_LOADS; ++p) {
      uint32_t off = load_offset[p];
      if (tail) {
        const int r = 4 * p + lane / UNITS;
        off = (uint32_t)((int)min((int64_t)r, a.Sk - 1 - key0) * ROW_BYTES + (((lane % UNITS) ^ (r & 15)) << 4));
      }
      if constexpr (STREAM)
        __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                         :: "s"(dst + (uint32_t)p * 1024u), "v"(off), "s"(base) : "memory");
      else
        __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                         :: "s"(dst + (uint32_t)p * 1024u), "v"(off), "s"(base) : "memory");
    }
  };

  x8 qf[QT][D / 32];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int64_t row = row0 + 16 * qt + i16;
#pragma unroll
    for (int j = 0; j < D / 32; ++j)
      qf[qt][j] = row < rows ? *(const x8*)(Q + row * D + 32 * j + 8 * g) : __builtin_bit_cast(x8, u32x4{0u, 0u, 0u, 0u});
  }
  // Q's loads are the wave's oldest and land before the first K tile.
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (i < n) {
      fetch(i, 0);
      fetch(i, 1);
    }

  const int ra = sigma(i16), rt = sigma(4 * g + (i16 >> 2));
  uint32_t qk_base[D / 32], tr_base[D / 16];
#pragma unroll
  for (int j = 0; j < D / 32; ++j) qk_base[j] = (uint32_t)(ra * ROW_BYTES + (((4 * j + g) ^ (ra & 15)) << 4));
#pragma unroll
  for (int t = 0; t < D / 16; ++t)
    tr_base[t] = (uint32_t)(rt * ROW_BYTES + (((2 * t + ((i16 & 3) >> 1)) ^ (rt & 15)) << 4) + (i16 & 1) * 8);

  f32x4 o[QT][D / 16];
  float m_run[QT], l_run[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    m_run[qt] = -1e30f;  // finite: a fully masked tile then gives p = 0, never NaN
    l_run[qt] = 0.f;
#pragma unroll
    for (int t = 0; t < D / 16; ++t) o[qt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float scale_log2 = a.scale * FA_LOG2E;

  // Before tile i the loads in flight are K(i), V(i), K(i+1), V(i+1) as far as
  // they exist, FD_LOADS each, in that order; K(i+2) replaces K(i) once its
  // fragments are in registers, then V(i+2) V(i). So K(i), and later V(i), has
  // landed once at most three younger batches are in flight; in the last two
  // tiles, which issue nothing, the wait is for everything.
  static_assert(4 * FD_LOADS < 64, "vmcnt holds 6 bits");
  for (int i = 0; i < n; ++i) {
    const bool more = i + 2 < n;
    if (more)
      wait_vmcnt<3 * FD_LOADS>();
    else
      wait_vmcnt<0>();
    __asm__ volatile("" ::: "memory");
    f32x4 s[KT][QT];
    {
      const uint32_t tile = slot_address(i, 0);
      x8 kf[D / 32][KT];
#pragma unroll
      for (int j = 0; j < D / 32; ++j)
#pragma unroll
        for (int t = 0; t < KT; ++t)
          kf[j][t] = *(const AFA_LDS x8*)(lds_at<uint8_t>(tile + qk_base[j]) + t * 16 * ROW_BYTES);
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) s[t][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < D / 32; ++j)
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) s[t][qt] = B16<DT>::mfma(kf[j][t], qf[qt][j], s[t][qt]);
    }
    if (more) {
      __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);  // K(i) is in registers
      __asm__ volatile("" ::: "memory");
      fetch(i + 2, 0);
    }
    const int64_t key0 = (int64_t)tile_of(i) * FD_KEYS;
    if (key0 + FD_KEYS > clean) {  // uniform
      __asm__ volatile("");
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        const int64_t limit = col_limit[qt] - key0;
        const int lim = limit < 0 ? 0 : (limit > FD_KEYS ? FD_KEYS : (int)limit);
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
          for (int k = 0; k < 4; ++k) s[t][qt][k] = 16 * t + sigma(4 * g + k) < lim ? s[t][qt][k] : -INFINITY;
      }
    }
    float m_new[QT];
    bool grow = false;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      float m = -INFINITY;
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int k = 0; k < 4; ++k) m = fmaxf(m, s[t][qt][k]);
      m_new[qt] = fmaxf(m_run[qt], max_over_lane_groups(m) * scale_log2);
      grow |= m_new[qt] > m_run[qt] + fa_tau<DT>();
    }
    if (__ballot(grow) != 0ull) {
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        const float alpha = fast_exp2(m_run[qt] - m_new[qt]);
        l_run[qt] *= alpha;
#pragma unroll
        for (int t = 0; t < D / 16; ++t) o[qt][t] *= alpha;
        m_run[qt] = m_new[qt];
      }
    }
    x8 pf[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float p = fast_exp2(__builtin_fmaf(s[t][qt][k], scale_log2, -m_run[qt]));
          sum += p;
          pf[qt][4 * t + k] = (scalar)p;
        }
      l_run[qt] += sum;
    }
    if (more) wait_vmcnt<3 * FD_LOADS>();  // else everything landed above
    __asm__ volatile("" ::: "memory");
    {
      const uint32_t tile = slot_address(i, 1);
      x4 vlo[D / 16], vhi[D / 16];
#pragma unroll
      for (int t = 0; t < D / 16; ++t) {
        const AFA_LDS uint8_t* p = lds_at<uint8_t>(tile + tr_base[t]);
        vlo[t] = B16<DT>::read_tr((const AFA_LDS void*)p);
        vhi[t] = B16<DT>::read_tr((const AFA_LDS void*)(p + 16 * ROW_BYTES));
      }
#pragma unroll
      for (int t = 0; t < D / 16; ++t) {
        const x8 vf = {vlo[t][0], vlo[t][1], vlo[t][2], vlo[t][3], vhi[t][0], vhi[t][1], vhi[t][2], vhi[t][3]};
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) o[qt][t] = B16<DT>::mfma(vf, pf[qt], o[qt][t]);
      }
    }
    if (more) {
      __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);  // V(i) is in registers
      __asm__ volatile("" ::: "memory");
      fetch(i + 2, 1);
    }
  }

  // ---- combine the four waves: each scales its O to the common max and lays
  // it out in its own (now idle) ring as [row][32 units of 4 features], unit u
  // of row r at u ^ (r & 15).
  static_assert(ROWS * D * 4 <= FD_SLOTS * FD_TILE, "a wave's O must fit its ring");
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const float l = sum_over_lane_groups(l_run[qt]);
    if (g == 0) {
      wave_ml[0][wave][16 * qt + i16] = m_run[qt];
      wave_ml[1][wave][16 * qt + i16] = l;
    }
  }
  __syncthreads();
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    float m = wave_ml[0][0][16 * qt + i16];
#pragma unroll
    for (int w = 1; w < FD_WAVES; ++w) m = fmaxf(m, wave_ml[0][w][16 * qt + i16]);
    const float weight = fast_exp2(m_run[qt] - m);
#pragma unroll
    for (int t = 0; t < D / 16; ++t)
      *(AFA_LDS f32x4*)(uintptr_t)(ring_base + (uint32_t)((16 * qt + i16) * 512 + (((4 * t + g) ^ i16) << 4))) =
          o[qt][t] * weight;
  }
  __syncthreads();
  // Thread tid takes unit tid % 32 of rows tid / 32, + 8, ...
  const int u = tid & 31;
#pragma unroll
  for (int r = tid >> 5; r < ROWS; r += FD_WAVES * 2) {
    const int64_t row = row0 + r;
    if (row >= rows) break;
    float m = wave_ml[0][0][r];
#pragma unroll
    for (int w = 1; w < FD_WAVES; ++w) m = fmaxf(m, wave_ml[0][w][r]);
    float l = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < FD_WAVES; ++w) {
      l += wave_ml[1][w][r] * fast_exp2(wave_ml[0][w][r] - m);
      acc += *lds_at<f32x4>(lds_address(ring[w][0]) + (uint32_t)(r * 512 + ((u ^ (r & 15)) << 4)));
    }
    const int64_t out_row = kv * rows + row;
    if (args.splits == 1) {
      const float inv = l > 0.f ? 1.0f / l : 0.f;
      x4 v;
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = (scalar)(acc[k] * inv);
      *(x4*)((scalar*)a.o + out_row * D + 4 * u) = v;
    } else {
      const int64_t at = (int64_t)split * (a.B * (int64_t)a.HQ * a.Sq) + out_row;
      *(f32x4*)(args.partial_o + at * D + 4 * u) = acc;
      if (u == 0) {
        args.partial_ml[2 * at] = m;
        args.partial_ml[2 * at + 1] = l;
      }
    }
  }
}

// Combines the splits of fa_split_kernel in split order (deterministic): with
// M = max_s m_s, O = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s. 32 threads
// per row, four features each.
constexpr int FM_ROWS = 8;  // rows per workgroup of 256 threads
template <int DT>
__global__ __launch_bounds__(256) void fa_merge_kernel(FaSplitArgs args) {
  typedef typename B16<DT>::scalar scalar;
  typedef typename B16<DT>::x4 x4;
  const FaArgs& a = args.fa;
  const int64_t total = a.B * (int64_t)a.HQ * a.Sq;
  const int64_t row = (int64_t)blockIdx.x * FM_ROWS + (threadIdx.x >> 5);
  const int u = threadIdx.x & 31;
  if (row >= total) return;
  // Thread u of the row holds the max and denominator of splits u and u + 32.
  float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 2; ++k)
    if (u + 32 * k < args.splits) {
      const float* ml = args.partial_ml + 2 * ((int64_t)(u + 32 * k) * total + row);
      m[k] = ml[0];
      l[k] = ml[1];
    }
  float M = fmaxf(m[0], m[1]);
#pragma unroll
  for (int d = 16; d > 0; d >>= 1) M = fmaxf(M, __shfl_xor(M, d, 32));
  float w[2], L = 0.f;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    w[k] = u + 32 * k < args.splits ? fast_exp2(m[k] - M) : 0.f;
    L += w[k] * l[k];
  }
#pragma unroll
  for (int d = 16; d > 0; d >>= 1) L += __shfl_xor(L, d, 32);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const float* src = args.partial_o + row * 128 + 4 * u;
#pragma unroll 8
  for (int s = 0; s < args.splits; ++s) {
    const float ws = __shfl(s < 32 ? w[0] : w[1], s & 31, 32);
    acc += *(const f32x4*)(src + (int64_t)s * total * 128) * ws;
  }
  const float inv = L > 0.f ? 1.0f / L : 0.f;
  x4 v;
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = (scalar)(acc[k] * inv);
  *(x4*)((scalar*)a.o + row * 128 + 4 * u) = v;
}

// Teaching attention: the whole 128-key tile of a head is resident in LDS, so
// the softmax is exact and P is normalised before its f16 cast
// (simple.py:25-41). A workgroup of four waves takes `steps` consecutive tiles
// of 64 query rows of one head, 16 rows per wave. Bound by HBM (Q read, O
// written once); what the split saves is the rest: K and V are loaded once per
// `steps` tiles instead of once per tile, the next tile's Q loads run under
// this tile's work, and O leaves through a wave-private LDS stage in whole
// 256-byte rows (straight from the accumulators a store instruction writes 16
// pieces of 32 bytes). Two workgroups share a CU (80 KiB of LDS each). Two row
// tiles per wave, which read each fragment for twice the MFMAs, measured the
// same. ONE: one tile per workgroup, a kernel of its own whose Q loads follow K's
// and V's: loads return in order, and Q's, in pieces of 64 bytes, would hold up
// the tile that all waves wait for (H4 S128 4.87 -> 4.44 us, H16 S1024 7.17 ->
// 6.90); over many tiles Q, which comes from HBM, goes first (H32 S8192 38.2, after
// them 39.4). GPU time of a call over inputs that no cache holds, one tile per
// workgroup with stores from the accumulators -> this (us): H4 S128 4.62 -> 4.44, H32
// S1024 11.8 -> 11.0, H64 S2048 37.2 -> 22.5, H32 S8192 65.0 -> 38.3 (3.5 TB/s), H64
// S8192 128 -> 64 (4.2 TB/s).
template <bool ONE>
__global__ __launch_bounds__(256, 2) void simple_attention_kernel(const _Float16* Qp, const _Float16* Kp,
                                                                  const _Float16* Vp, _Float16* Op, int64_t S,
                                                                  int32_t groups, int32_t tiles) {
  typedef B16<DT_F16> ops;
  constexpr int D = 128, SK = 128, ROW_BYTES = D * 2, KT = SK / 16, ROWS = 16;
  const int steps = ONE ? 1 : tiles;
  __shared__ __attribute__((aligned(16))) uint8_t k_lds[SK * ROW_BYTES];
  __shared__ __attribute__((aligned(16))) uint8_t v_lds[SK * ROW_BYTES];
  __shared__ __attribute__((aligned(16))) uint8_t o_lds[4][16 * ROW_BYTES];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int g = lane >> 4, i16 = lane & 15;
  const uint32_t logical = xcd_contiguous(blockIdx.x, gridDim.x);  // a head's groups share its K and V in one L2
  const int64_t head = logical / (uint32_t)groups, group = logical % (uint32_t)groups;
  const _Float16* Q = Qp + head * S * D;
  const _Float16* K = Kp + head * SK * D;
  const _Float16* V = Vp + head * SK * D;
  _Float16* O = Op + head * S * D;
  // This wave's first row of step s (S is a multiple of 64: a wave's rows are all in or all out).
  auto first_row = [&](int s) { return ((group * steps + s) * 4 + wave) * ROWS; };

  f16x8 qf[D / 32];
  auto load_q = [&](int s) {
    const int64_t row = first_row(s);
    if (row < S) {
#pragma unroll
      for (int j = 0; j < D / 32; ++j) qf[j] = *(const f16x8*)(Q + (row + i16) * D + 32 * j + 8 * g);
    }
  };
  if constexpr (!ONE) load_q(0);
  for (int flat = tid; flat < SK * (D / 8); flat += 256) {
    const int r = flat / (D / 8), u = flat % (D / 8);
    const int off = r * ROW_BYTES + (swz(r, u) << 4);
    *(u32x4*)(&k_lds[off]) = *(const u32x4*)(K + r * D + u * 8);
    *(u32x4*)(&v_lds[off]) = *(const u32x4*)(V + r * D + u * 8);
  }
  if constexpr (ONE) load_q(0);
  __syncthreads();

  const int ra = sigma(i16);
  const int rt = sigma(4 * g + (i16 >> 2));
  const int tr_half = (i16 & 1) * 8, tr_unit = (i16 & 3) >> 1;
  const float scale_log2 = 0.08838834764831845f * FA_LOG2E;
  for (int step = 0; step < steps; ++step) {
    const int64_t row0 = first_row(step);
    if (row0 >= S) break;
    f32x4 s[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < D / 32; ++j) {
      const int u = 4 * j + g;
#pragma unroll
      for (int t = 0; t < KT; ++t) {
        const int row = 16 * t + ra;
        const f16x8 kf = *(const f16x8*)(k_lds + row * ROW_BYTES + (swz(row, u) << 4));
        s[t] = ops::mfma(kf, qf[j], s[t]);
      }
    }
    if (step + 1 < steps) load_q(step + 1);  // lands during the softmax and PV
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[t][i] *= scale_log2;
        mx = fmaxf(mx, s[t][i]);
      }
    mx = max_over_lane_groups(mx);
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[t][i] = fast_exp2(s[t][i] - mx);
        sum += s[t][i];
      }
    const float inv = 1.0f / sum_over_lane_groups(sum);
    f16x8 pf[SK / 32];
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) pf[t >> 1][(t & 1) * 4 + i] = (_Float16)(s[t][i] * inv);
    f32x4 acc[D / 16];
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
      acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      const int u = 2 * t + tr_unit;
#pragma unroll
      for (int ks = 0; ks < SK / 32; ++ks) {
        const int r0 = 32 * ks + rt, r1 = 32 * ks + 16 + rt;
        const f16x4 lo = ops::read_tr((const AFA_LDS void*)(v_lds + r0 * ROW_BYTES + (swz(r0, u) << 4) + tr_half));
        const f16x4 hi = ops::read_tr((const AFA_LDS void*)(v_lds + r1 * ROW_BYTES + (swz(r1, u) << 4) + tr_half));
        const f16x8 vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        acc[t] = ops::mfma(vf, pf[ks], acc[t]);
      }
    }
    // This lane holds features 16t + 4g + 0..3 of row i16: staged as 16-byte
    // unit u of row r at u ^ r, read back four whole rows per access. Only this
    // wave touches the stage, and its LDS operations complete in order.
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
      f16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (_Float16)acc[t][i];
      *(f16x4*)(&o_lds[wave][i16 * ROW_BYTES + (((2 * t + (g >> 1)) ^ i16) << 4) + (g & 1) * 8]) = v;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = 4 * q + g;  // lane 16g + i16 takes unit i16 of it
      const u32x4 v = *(const u32x4*)(&o_lds[wave][r * ROW_BYTES + ((i16 ^ r) << 4)]);
      *(u32x4*)(O + (row0 + r) * D + 8 * i16) = v;
    }
  }
}

}  // namespace afa

using namespace afa;

namespace {
constexpr int FD_MAX_SPLITS = 64;  // fa_merge_kernel keeps two splits per thread of a row
constexpr int64_t FA_CUS = 256;
constexpr int64_t FD_STREAM_BYTES = int64_t(128) << 20;
// K and V of a causal call up to which the forward kernel takes the tiles of all
// heads by length; beyond, a head's tiles follow each other and read its keys
// from the L2. 128-row tiles by length / by head (us): 142 MiB 174 / 176, 219
// 372 / 380, 255 525 / 513, 266 388 / 364, 321 341 / 319, 445 849 / 711, 593 1017
// / 732 (256-row tiles by head: 771).
constexpr int64_t FA_LEVEL_BYTES = int64_t(240) << 20;

template <int DT, int NW, int QT>
int launch_forward(const FaArgs& a, hipStream_t s) {
  constexpr int BQ = NW * QT * 16;
  const int64_t blocks = (a.Sq + BQ - 1) / BQ * a.B * a.HQ;
  if (blocks > 0x7fffffffLL) return AFA_E_SHAPE;
  hipLaunchKernelGGL((fa_forward_kernel<DT, NW, QT>), dim3((unsigned)blocks), dim3(NW * 64), 0, s, a);
  return (int)hipGetLastError();
}

// Forms of the forward kernel, by query rows of a workgroup's tile: 256 rows in
// eight waves, one workgroup per CU; 128 and 64 in four waves, two per CU.
constexpr int FA_FORMS = 3;
constexpr int FA_ROWS[FA_FORMS] = {256, 128, 64};
template <int DT>
int launch_fa(const FaArgs& a, int form, hipStream_t s) {
  return form == 0 ? launch_forward<DT, 8, 2>(a, s)
                   : form == 1 ? launch_forward<DT, 4, 2>(a, s) : launch_forward<DT, 4, 1>(a, s);
}

// Form of a call: the packed split kernel (qt row tiles of 16 per workgroup,
// `splits` key ranges) or a forward kernel (qt = 0).
struct FaPlan {
  int qt, splits;
  int64_t row_tiles;
  int form;  // qt = 0
};

// Picks the cheaper form by a model of MI355X in microseconds (times measured
// on grids from 16 to 4096 workgroups, bf16), fixed at 256 CUs so that the
// workspace size depends on the sizes alone:
//  - forward kernel: per 64-key chunk ALONE while a CU runs one workgroup of it
//    (its longest tile then sets the time) and FULL while it runs all that
//    fit; FORWARD_START for a workgroup's Q, first loads and output; among its
//    tiles also PAIR_START for 128-row ones, two to a CU, that at most three
//    chunks follow (256 / 128 / 64 rows: B4 HQ64 S148 15.0 / 16.8 / 18.3; B8 HQ64 S156
//    27.4 / 29.9 / 26.3; B21 HQ32 Sq139 Sk101 30.9 / 33.6 / 28.2; causal B31 HQ32 S146
//    49.8 / 43.6 / 36.3);
//  - split kernel, one workgroup per CU: a step of four 32-key tiles costs the
//    larger of SPLIT_STEP[qt] (the latency of 64 KiB of loads, then the waves'
//    own chain of MFMAs and softmax) and KV_STEP, its 64 KiB when all CUs load
//    at once (6.9 TB/s), shared by the row tiles that read the same keys;
//    SPLIT_START for the first workgroup of a CU, ROUND + ROUND_QT * qt for
//    each later one (its first loads, and the waves' O through LDS), MERGE +
//    MERGE_SPLIT per split for the second kernel.
// A causal grid runs at least its longest tile and about half of a full one's
// work. Measured either side of the lines (us; forward kernel of 256 / 128 / 64
// rows, best split form): B1 HQ8 S1024 causal 37 / 27 / 19.1, 18.3; B1 HQ32 S700
// causal 27 / 20 / 16, 36; B1 HQ32 HKV8 Sq256 Sk8192 228 / 173 / 125, 93; B3 HQ28
// S1500 causal 77 / 68 / 82; B2 HQ32 S2048 139 / 146 / 179; B2 HQ32 S5401 causal
// 564 / 523 / 660; B6 HQ32 S429 42 / 35 / 37, 100; B2 HQ28 S158 11.6 / 9.9 / 6.9, 15.
// with_splits: there is a workspace for partial results.
FaPlan choose_fa(const FaArgs& a, bool with_splits) {
  constexpr int PER_CU[FA_FORMS] = {1, 2, 2};
  constexpr double ALONE[FA_FORMS] = {1.7, 1.25, 0.95}, FULL[FA_FORMS] = {1.8, 1.85, 1.3};
  constexpr double FORWARD_START[FA_FORMS] = {8.0, 6.5, 5.5}, PAIR_START = 2.5;
  constexpr double KV_STEP = 2.4, SPLIT_START = 8.0, ROUND = 3.0, ROUND_QT = 1.6, MERGE = 3.0, MERGE_SPLIT = 0.12;
  constexpr double SPLIT_STEP[FD_MAX_QT + 1] = {0, 1.4, 1.55, 2.0, 2.45};
  const int64_t group = a.HQ / a.HKV, kv_heads = (int64_t)a.B * a.HKV, rows = group * a.Sq;
  const int64_t keys = a.causal ? std::min(a.Sk, a.Sq) : a.Sk;
  // Mean tile length over the longest, with n row tiles per head.
  auto mean = [&](int64_t n) { return a.causal && n > 1 ? 0.5 * (1 + 1.0 / n) : 1.0; };
  FaPlan plan{0, 1, 0, 0};
  double best = 0, best_pair = 0;  // the cheapest tiles without and with PAIR_START
  for (int form = 0; form < FA_FORMS; ++form) {
    const int64_t tiles = (a.Sq + FA_ROWS[form] - 1) / FA_ROWS[form], blocks = tiles * a.B * a.HQ;
    const double chunks = std::ceil(keys / 64.0), slots = (double)FA_CUS * PER_CU[form];
    const double cost = FORWARD_START[form] * (0.5 + 0.5 * std::ceil(blocks / slots)) +
                        std::max(chunks * ALONE[form],
                                 (a.causal ? blocks / slots : std::ceil(blocks / slots)) * mean(tiles) * chunks * FULL[form] *
                                     std::min(1.0, std::max(blocks / slots, 1.0 / PER_CU[form])));
    const double with_pair = cost + (form == 1 && blocks > FA_CUS && chunks <= 3 ? PAIR_START : 0.0);
    if (form == 0 || with_pair < best_pair) {
      best_pair = with_pair;
      plan.form = form;
    }
    best = form == 0 ? cost : std::min(best, cost);
  }
  for (int qt = 1; qt <= FD_MAX_QT; ++qt) {
    const int64_t row_tiles = (rows + 16 * qt - 1) / (16 * qt);
    if (qt > 1 && rows <= 16 * (qt - 1)) break;  // no fewer tiles than with qt - 1
    const int64_t items = kv_heads * row_tiles;
    if (items * FD_MAX_SPLITS > 0x7fffffffLL) continue;
    // A causal row tile that crosses heads walks every key of both: only where those are few.
    if (a.causal && group > 1 && a.Sq > 256 && a.Sq % (16 * qt)) continue;
    const int64_t key_tiles = (keys + FD_KEYS - 1) / FD_KEYS;
    const int64_t most = with_splits ? std::min<int64_t>(FD_MAX_SPLITS, std::max<int64_t>(1, key_tiles / FD_WAVES)) : 1;
    const double tile_mean = mean((a.Sq + 16 * qt - 1) / (16 * qt));
    const double least = std::max(1.0, tile_mean * (double)items * (double)key_tiles / (FA_CUS * FD_WAVES));
    for (int64_t splits = 1; splits <= most; ++splits) {
      const int64_t blocks = items * splits;
      const double rounds = std::ceil((double)blocks / FA_CUS), active = std::min<double>(1.0, (double)blocks / FA_CUS);
      const double starts = SPLIT_START + (splits > 1 ? MERGE + MERGE_SPLIT * splits : 0.0) +
                            (rounds - 1) * (ROUND + ROUND_QT * qt);
      const double step = std::max(SPLIT_STEP[qt], KV_STEP * active / row_tiles);
      // More splits never make the starts or a step cheaper, and the steps of
      // all rounds together are at least `least`: none of them beats the best.
      if (starts + least * step >= best) break;
      const double steps = std::ceil((double)key_tiles / splits / FD_WAVES);
      const double cost = starts + std::max(1.0, rounds * tile_mean) * steps * step;
      if (cost < best) {
        best = cost;
        plan = FaPlan{qt, (int)splits, row_tiles, 0};
      }
    }
  }
  return plan;
}

int64_t fa_split_bytes(const FaArgs& a, const FaPlan& plan) {
  return plan.splits > 1 ? (int64_t)plan.splits * a.B * a.HQ * a.Sq * (128 + 2) * 4 : 0;
}

template <int DT>
int launch_split(const FaArgs& a, const FaPlan& plan, void* workspace, hipStream_t s) {
  FaSplitArgs args;
  args.fa = a;
  args.group = a.HQ / a.HKV;
  args.row_tiles = (int32_t)plan.row_tiles;
  args.splits = plan.splits;
  const int64_t total = (int64_t)a.B * a.HQ * a.Sq;
  args.partial_o = (float*)workspace;
  args.partial_ml = (float*)workspace + plan.splits * total * 128;
  const dim3 grid((unsigned)((int64_t)a.B * a.HKV * plan.row_tiles * plan.splits)), block(FD_WAVES * 64);
  // Non-temporal KV loads, measured with and without (us): 1.07 GB of KV 160 /
  // 182, 268 MB 46.8 / 52.8, 134 MB 27.9 / 31.2; but 67 MB, part of which stays
  // cached between calls, 24.0 / 21.7. Calls of three row tiles and more share
  // their KV through the L2 (262 MB 100.1 / 99.6) and keep ordinary loads.
  const bool stream = plan.row_tiles <= 2 && 2 * 256 * (int64_t)a.B * a.HKV * a.Sk >= FD_STREAM_BYTES;
  if (stream && plan.qt == 1)
    hipLaunchKernelGGL((fa_split_kernel<DT, 1, true>), grid, block, 0, s, args);
  else if (stream && plan.qt == 2)
    hipLaunchKernelGGL((fa_split_kernel<DT, 2, true>), grid, block, 0, s, args);
  else if (plan.qt == 1)
    hipLaunchKernelGGL((fa_split_kernel<DT, 1, false>), grid, block, 0, s, args);
  else if (plan.qt == 2)
    hipLaunchKernelGGL((fa_split_kernel<DT, 2, false>), grid, block, 0, s, args);
  else if (plan.qt == 3)
    hipLaunchKernelGGL((fa_split_kernel<DT, 3, false>), grid, block, 0, s, args);
  else
    hipLaunchKernelGGL((fa_split_kernel<DT, 4, false>), grid, block, 0, s, args);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || plan.splits == 1) return (int)e;
  hipLaunchKernelGGL(fa_merge_kernel<DT>, dim3((unsigned)((total + FM_ROWS - 1) / FM_ROWS)), dim3(256), 0, s, args);
  return (int)hipGetLastError();
}

int check_fa(int64_t Sq, int64_t Sk, const FaParams* p) {
  if (!p) return AFA_E_NULL;
  if (p->dtype != AFA_DTYPE_BF16 && p->dtype != AFA_DTYPE_F16) return AFA_E_DTYPE;
  if (p->D != 128 || p->B <= 0 || p->HQ <= 0 || p->HKV <= 0 || p->HQ % p->HKV) return AFA_E_SHAPE;
  if (Sq < 1 || Sk < 1 || !(p->scale > 0.0f)) return AFA_E_SHAPE;
  return AFA_OK;
}

FaArgs make_fa(const void* Q, const void* K, const void* V, void* O, int64_t Sq, int64_t Sk, const FaParams* p) {
  FaArgs a;
  a.q = Q;
  a.k = K;
  a.v = V;
  a.o = O;
  a.Sq = Sq;
  a.Sk = Sk;
  a.B = p->B;
  a.HQ = p->HQ;
  a.HKV = p->HKV;
  a.causal = p->causal ? 1 : 0;
  a.level_order = a.causal && 2 * 256 * (int64_t)p->B * p->HKV * std::min(Sq, Sk) <= FA_LEVEL_BYTES;
  a.scale = p->scale;
  return a;
}

int dispatch_fa(const FaArgs& a, const FaPlan& plan, void* workspace, int dtype, hipStream_t s) {
  if (plan.qt == 0) return dtype == AFA_DTYPE_F16 ? launch_fa<DT_F16>(a, plan.form, s) : launch_fa<DT_BF16>(a, plan.form, s);
  return dtype == AFA_DTYPE_F16 ? launch_split<DT_F16>(a, plan, workspace, s)
                                : launch_split<DT_BF16>(a, plan, workspace, s);
}
}  // namespace

extern "C" int launch_attention_target(void* stream, const void* Q, const void* K, const void* V,
                                       void* O, void* workspace, int64_t Sq, int64_t Sk,
                                       const FaParams* p) {
  (void)workspace;
  if (!p) return AFA_E_NULL;
  if (!Q || !K || !V || !O) return AFA_E_NULL;
  const int status = check_fa(Sq, Sk, p);
  if (status) return status;
  const FaArgs a = make_fa(Q, K, V, O, Sq, Sk, p);
  return dispatch_fa(a, choose_fa(a, false), nullptr, p->dtype, (hipStream_t)stream);
}

extern "C" int workspace_size_attention_target_split(uint64_t* bytes, int64_t Sq, int64_t Sk, const FaParams* p) {
  if (!bytes) return -1;
  const int status = check_fa(Sq, Sk, p);
  if (status) return status;
  const FaArgs a = make_fa(nullptr, nullptr, nullptr, nullptr, Sq, Sk, p);
  *bytes = (uint64_t)fa_split_bytes(a, choose_fa(a, true));
  return AFA_OK;
}

extern "C" int launch_attention_target_split(void* stream, const void* Q, const void* K, const void* V, void* O,
                                             void* workspace, uint64_t workspace_bytes, int64_t Sq, int64_t Sk,
                                             const FaParams* p) {
  if (!p) return AFA_E_NULL;
  if (!Q || !K || !V || !O) return AFA_E_NULL;
  const int status = check_fa(Sq, Sk, p);
  if (status) return status;
  const FaArgs a = make_fa(Q, K, V, O, Sq, Sk, p);
  const FaPlan plan = choose_fa(a, true);
  const int64_t need = fa_split_bytes(a, plan);
  if (need > 0 && (!workspace || workspace_bytes < (uint64_t)need)) return AFA_E_WORKSPACE;
  return dispatch_fa(a, plan, workspace, p->dtype, (hipStream_t)stream);
}

extern "C" int form_attention_target(int64_t form[3], int64_t Sq, int64_t Sk, const FaParams* p, int with_workspace) {
  if (!form) return AFA_E_NULL;
  const int status = check_fa(Sq, Sk, p);
  if (status) return status;
  const FaPlan plan = choose_fa(make_fa(nullptr, nullptr, nullptr, nullptr, Sq, Sk, p), with_workspace != 0);
  form[0] = plan.qt ? 1 : 0;
  form[1] = plan.qt ? 16 * plan.qt : FA_ROWS[plan.form];
  form[2] = plan.splits;
  return AFA_OK;
}

extern "C" int launch_simple_attention(void* stream, const void* Q, const void* K, const void* V,
                                       void* O, void* workspace, int64_t S, int64_t H) {
  (void)workspace;
  if (!Q || !K || !V || !O) return AFA_E_NULL;
  if (S <= 0 || S % 64 || H <= 0 || (S / 64) * H > 0x7fffffffLL) return AFA_E_SHAPE;
  // Tiles per workgroup that take the fewest rounds of two workgroups per CU,
  // each as long as its tiles and about one more for K and V (H36 S6912: 6 tiles
  // 33.1 us, 3 tiles, whose 1.3 rounds end with an idle GPU, 38.4).
  const int64_t slots = 2 * FA_CUS, tiles = S / 64;
  int64_t steps = 1, best = INT64_MAX;
  for (int64_t k = 1; k <= std::min<int64_t>(tiles, 16); ++k) {
    const int64_t cost = (((tiles + k - 1) / k * H + slots - 1) / slots) * (k + 1);
    if (cost < best) {
      best = cost;
      steps = k;
    }
  }
  const int64_t groups = (tiles + steps - 1) / steps;
  const auto kernel = steps == 1 ? simple_attention_kernel<true> : simple_attention_kernel<false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(groups * H)), dim3(256), 0, (hipStream_t)stream, (const _Float16*)Q,
                     (const _Float16*)K, (const _Float16*)V, (_Float16*)O, S, (int32_t)groups, (int32_t)steps);
  return (int)hipGetLastError();
}

extern "C" int kernel_config_attention_target(int64_t cfg[5]) {
  if (!cfg) return AFA_E_NULL;
  cfg[0] = 4;
  cfg[1] = 2;  // Sq, Sk
  cfg[2] = 0;
  cfg[3] = 256;
  cfg[4] = 4;
  return AFA_OK;
}

extern "C" int kernel_config_simple_attention(int64_t cfg[5]) {
  if (!cfg) return AFA_E_NULL;
  cfg[0] = 4;
  cfg[1] = 2;  // S, H
  cfg[2] = 0;
  cfg[3] = 256;
  cfg[4] = 4;
  return AFA_OK;
}

extern "C" int workspace_size_attention_target(uint64_t* bytes, int64_t Sq, int64_t Sk,
                                               const FaParams* p) {
  if (!bytes) return -1;
  (void)Sq;
  (void)Sk;
  (void)p;
  *bytes = 0;
  return AFA_OK;
}

extern "C" int workspace_size_simple_attention(uint64_t* bytes, int64_t S, int64_t H) {
  if (!bytes) return -1;
  (void)S;
  (void)H;
  *bytes = 0;
  return AFA_OK;
}

// Launch-ABI descriptions in the reference's metadata schema
// (src/backend/abi.py:19-59): tensors (dtype, shape with named axes, layout,
// access), runtime size parameters with minimum and multiple, workspace flag.
// The FA sizes the reference specialises at compile time (B, HQ, HKV, D,
// dtype, causal, scale) travel in FaParams ("params_struct"); "DTYPE" is one
// of "dtypes".
extern "C" const char* kernel_metadata_attention_target(void) {
  return "{\"version\":1,\"name\":\"attention_target\",\"target\":\"gfx950\",\"kind\":\"mixed\","
         "\"groups\":256,\"disjoint_external\":true,\"device_resources\":null,"
         "\"dtypes\":{\"DTYPE\":[\"f16\",\"bf16\"]},\"tensors\":["
         "{\"name\":\"Q\",\"dtype\":\"DTYPE\",\"shape\":[\"B\",\"HQ\",\"Sq\",\"D\"],"
         "\"layout\":\"linear\",\"access\":\"read\"},"
         "{\"name\":\"K\",\"dtype\":\"DTYPE\",\"shape\":[\"B\",\"HKV\",\"Sk\",\"D\"],"
         "\"layout\":\"linear\",\"access\":\"read\"},"
         "{\"name\":\"V\",\"dtype\":\"DTYPE\",\"shape\":[\"B\",\"HKV\",\"Sk\",\"D\"],"
         "\"layout\":\"linear\",\"access\":\"read\"},"
         "{\"name\":\"O\",\"dtype\":\"DTYPE\",\"shape\":[\"B\",\"HQ\",\"Sq\",\"D\"],"
         "\"layout\":\"linear\",\"access\":\"write\"}],"
         "\"parameters\":[{\"name\":\"Sq\",\"minimum\":1,\"multiple\":1},"
         "{\"name\":\"Sk\",\"minimum\":1,\"multiple\":1}],"
         "\"params_struct\":{\"name\":\"FaParams\",\"fields\":[\"B\",\"HQ\",\"HKV\",\"D\",\"dtype\","
         "\"causal\",\"scale\",\"reserved\"]},"
         "\"workspace\":false}";
}
extern "C" const char* kernel_metadata_simple_attention(void) {
  return "{\"version\":1,\"name\":\"simple_attention\",\"target\":\"gfx950\",\"kind\":\"mixed\","
         "\"groups\":256,\"disjoint_external\":true,\"device_resources\":null,\"tensors\":["
         "{\"name\":\"Q\",\"dtype\":\"f16\",\"shape\":[\"H\",\"S\",128],\"layout\":\"linear\","
         "\"access\":\"read\"},"
         "{\"name\":\"K\",\"dtype\":\"f16\",\"shape\":[\"H\",128,128],\"layout\":\"linear\","
         "\"access\":\"read\"},"
         "{\"name\":\"V\",\"dtype\":\"f16\",\"shape\":[\"H\",128,128],\"layout\":\"linear\","
         "\"access\":\"read\"},"
         "{\"name\":\"O\",\"dtype\":\"f16\",\"shape\":[\"H\",\"S\",128],\"layout\":\"linear\","
         "\"access\":\"write\"}],"
         "\"parameters\":[{\"name\":\"S\",\"minimum\":64,\"multiple\":64},"
         "{\"name\":\"H\",\"minimum\":1,\"multiple\":1}],\"workspace\":false}";
}
