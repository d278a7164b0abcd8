// Row-wise top-k of an fp32 score matrix (nrows, n) -> values (nrows, k) descending and
// int64 indices, the per-query top-100 the reference takes with torch.topk after scoring
// (src/cycle3_experiments.py:215).
//
// Each element becomes a 64-bit key: an order-preserving image of the float bits in the
// high word (NaN above +inf, as torch orders it) and the inverted index in the low word,
// so descending key order is "value descending, then index ascending" -- deterministic,
// and compared as integers (no float NaN semantics involved).
//
// Rows past one chunk at 8 <= k <= 512 go by group maxima (end of this file), the others by
// the tournament.
//
// Tournament: a workgroup selects the best k of a chunk of kChunk keys and each level
// shrinks a row by kChunk / k until one chunk holds it; the last level sorts its k keys
// (a last level of at most kShortRow keys runs a chunk of that size over four waves).
// Intermediate keys live in a caller-provided workspace. Levels that pass keys on first
// drop the keys below a bound on the chunk's k-th key taken from the threads' maxima
// (at k <= kFilterMaxK) and select among the survivors. Selection is a radix select on
// the 64-bit keys held in registers (4 or 16 per thread): one 256-bin LDS histogram per 8-bit
// digit, from the highest bit at which the chunk's real keys differ, narrowed to the
// keys that share the digits fixed so far, until the k-th largest key is known or a
// whole bin is needed (two or three passes for rows of similar scores). Padding keys are
// all 0 and a chunk's keys often share a digit, so the histogram updates would pile onto
// a few bins: each thread adds a run of equal bins with one atomic, and each wave counts
// into its own copy of the histogram.
#pragma once
#include "tms_common.h"
#include "tms_rules.h"

namespace tms {

// Threads per workgroup: a level that shrinks many chunks at once runs 4 waves per chunk
// (16 keys per thread); the last level, one chunk per row and nothing else running
// beside it, runs 16 waves (4 keys per thread, four waves per SIMD to overlap its serial
// steps). Measured on MaxSim-like and Gaussian rows, each is the faster of the two for
// its level.
constexpr int kLevelThreads = 256;
constexpr int kLastThreads = 1024;
constexpr int kMaxK = kChunk / 4;
// Rows (or last levels) of at most kShortRow keys: one chunk of that size over four
// waves, one per SIMD, so the serial steps (scans, reductions) are not repeated by four
// waves on every SIMD.
constexpr int kShortThreads = 256;
constexpr int kRankSortMaxK = 256;  // the last level orders up to this many keys by rank, more by a bitonic sort
// Levels that pass k keys on, at k <= kFilterMaxK, first drop the keys below a bound on
// the chunk's k-th key and select among the rest, gathered in LDS, when at most
// kCandCap of them remain.
constexpr int kCandCap = 1024;

// Order-preserving image of a float's bits, never 0 (0 is the padding key). Positive
// values map to b | 2^31 and negative ones to -b (mod 2^32), so -0.0 lands on +0.0's key
// (they compare equal, so they tie and go by index); every NaN, either sign, maps to the
// top key, above +inf, as torch ranks NaN.
__device__ __forceinline__ uint32_t order_key(float f) {
  const uint32_t b = __builtin_bit_cast(uint32_t, f);
  const uint32_t o = (int32_t)b < 0 ? 0u - b : (b | 0x80000000u);
  return (b & 0x7fffffffu) > 0x7f800000u ? 0xffffffffu : o;
}

// FIRST: input is fp32 scores (row stride in_stride), indices are positions in the row.
// Otherwise input is keys. LAST: write (value, index) pairs in descending order;
// otherwise write the best k keys of the chunk, in no particular order.
constexpr int kHistCopies = 4;  // wave w counts into copy w % 4; wave 0 scans four bins per lane

// Cross-lane steps without the LDS: DPP within 16-lane rows, row swaps across them.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ uint64_t dpp_u64(uint64_t v) {
  return ((uint64_t)dpp_u32<CTRL>((uint32_t)(v >> 32)) << 32) | dpp_u32<CTRL>((uint32_t)v);
}
// The value of lane l ^ 32 (permlane32_swap) or of the other row of the pair (row ^ 1,
// permlane16_swap), for a value every lane holds.
__device__ __forceinline__ uint32_t swap32_u32(uint32_t v, int lane) {
  const auto p = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return lane < 32 ? (uint32_t)p[1] : (uint32_t)p[0];
}
__device__ __forceinline__ uint32_t swap16_u32(uint32_t v, int lane) {
  const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return ((lane >> 4) & 1) ? (uint32_t)p[0] : (uint32_t)p[1];
}
__device__ __forceinline__ uint64_t swap32_u64(uint64_t v, int lane) {
  return ((uint64_t)swap32_u32((uint32_t)(v >> 32), lane) << 32) | swap32_u32((uint32_t)v, lane);
}
__device__ __forceinline__ uint64_t swap16_u64(uint64_t v, int lane) {
  return ((uint64_t)swap16_u32((uint32_t)(v >> 32), lane) << 32) | swap16_u32((uint32_t)v, lane);
}
// Wave-wide min and max of 64-bit values and sum of counts; every lane gets the result.
__device__ __forceinline__ void wave_minmax(uint64_t& lo, uint64_t& hi, uint32_t& n, int lane) {
  auto step = [&](uint64_t l2, uint64_t h2, uint32_t n2) {
    lo = l2 < lo ? l2 : lo;
    hi = h2 > hi ? h2 : hi;
    n += n2;
  };
  step(dpp_u64<0xB1>(lo), dpp_u64<0xB1>(hi), dpp_u32<0xB1>(n));     // quad_perm [1,0,3,2]
  step(dpp_u64<0x4E>(lo), dpp_u64<0x4E>(hi), dpp_u32<0x4E>(n));     // quad_perm [2,3,0,1]
  step(dpp_u64<0x141>(lo), dpp_u64<0x141>(hi), dpp_u32<0x141>(n));  // row_half_mirror
  step(dpp_u64<0x140>(lo), dpp_u64<0x140>(hi), dpp_u32<0x140>(n));  // row_mirror
  step(swap16_u64(lo, lane), swap16_u64(hi, lane), swap16_u32(n, lane));
  step(swap32_u64(lo, lane), swap32_u64(hi, lane), swap32_u32(n, lane));
}
// Wave-wide maximum of a 32-bit value; every lane gets it.
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x, int lane) {
  auto mx = [](uint32_t a, uint32_t b) { return a > b ? a : b; };
  x = mx(x, dpp_u32<0xB1>(x));   // quad_perm [1,0,3,2]
  x = mx(x, dpp_u32<0x4E>(x));   // quad_perm [2,3,0,1]
  x = mx(x, dpp_u32<0x141>(x));  // row_half_mirror
  x = mx(x, dpp_u32<0x140>(x));  // row_mirror
  x = mx(x, swap16_u32(x, lane));
  return mx(x, swap32_u32(x, lane));
}
// Inclusive prefix sum over the 64 lanes (lane order): row shifts, then row broadcasts.
__device__ __forceinline__ uint32_t wave_inclusive_sum(uint32_t x) {
  x += dpp_u32<0x111>(x);  // row_shr:1
  x += dpp_u32<0x112>(x);  // row_shr:2
  x += dpp_u32<0x114>(x);  // row_shr:4
  x += dpp_u32<0x118>(x);  // row_shr:8
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1, 3
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2, 3
  return x;
}

// The last level's ordering: each of the m distinct keys in sel[0, m) counts the keys
// above it among sel[0, m8) (m rounded up to a multiple of 8; slots [m, m8 + kRankPad)
// hold 0, below every real key), and a key of rank < k is written at its rank. S = 8, 4 or 2
// lanes share a key when the threads allow: lane part p counts among slots
// [p * m8 / S, (p + 1) * m8 / S), and DPP steps add the S counts.
constexpr int kRankPad = 48;  // zero slots past m8 that the one-lane-per-key loop may read
static_assert(kRankSortMaxK + kRankPad <= kMaxK, "the rank step's read ahead stays inside sel");
template <bool FIRST, int NT>
__device__ __forceinline__ void topk_rank_out(const uint64_t* sel, const uint32_t* sel_bits, int m, int m8,
                                              const float* __restrict__ vals, int64_t val_stride,
                                              float* __restrict__ out_vals, int64_t* __restrict__ out_idx, int k,
                                              int64_t row) {
  const int tid = threadIdx.x;
  const int lg = m * 8 <= NT ? 3 : (m * 4 <= NT ? 2 : (m * 2 <= NT ? 1 : 0));
  const int S = 1 << lg;
  const int per = m8 >> lg;
  for (int t = tid; t < (S > 1 ? S * m8 : m); t += NT) {
    const int i = t >> lg;
    const uint64_t me = sel[i];
    const int j0 = (t & (S - 1)) * per;
    uint32_t rank = 0u;
    int j = j0;
    const int end = j0 + per;
    if (S == 1) {
      // One lane per key, the whole range [0, m8) in steps of 32 with the next 16 keys
      // read ahead, so the LDS latency hides behind the compares (one wave per SIMD has
      // nothing else to run meanwhile). No exit between a read and its use, so the
      // compiler keeps the reads ahead. Reads run up to 40 slots past m8 and counts up
      // to 24, into slots that hold 0 (set with the keys): a 0 key is above nothing.
      uint64_t xa[16], xb[16];
      auto load16 = [&](uint64_t(&x)[16], int at) {
#pragma unroll
        for (int q = 0; q < 16; q++) x[q] = sel[at + q];
      };
      auto count16 = [&](const uint64_t(&x)[16]) {
#pragma unroll
        for (int q = 0; q < 16; q++) rank += x[q] > me ? 1u : 0u;
      };
      load16(xa, 0);
      for (j = 0; j < m8; j += 32) {
        load16(xb, j + 16);
        count16(xa);
        load16(xa, j + 32);
        count16(xb);
      }
      j = end;
    }
    for (; j + 8 <= end; j += 8) {  // eight reads in flight per step
      uint64_t x[8];
#pragma unroll
      for (int q = 0; q < 8; q++) x[q] = sel[j + q];
#pragma unroll
      for (int q = 0; q < 8; q++) rank += x[q] > me ? 1u : 0u;
    }
    for (; j < end; j++) rank += sel[j] > me ? 1u : 0u;
    if (S > 1) {
      rank += dpp_u32<0xB1>(rank);                 // quad_perm [1,0,3,2]: pairs
      if (S > 2) rank += dpp_u32<0x4E>(rank);      // quad_perm [2,3,0,1]: quads
      if (S > 4) rank += dpp_u32<0x141>(rank);     // row_half_mirror: the other quad of the eight
      if ((t & (S - 1)) != 0) continue;
    }
    if (i >= m || rank >= (uint32_t)k) continue;
    const int64_t idx = (int64_t)(0xffffffffu - (uint32_t)me);
    if constexpr (FIRST) out_vals[row * k + rank] = __builtin_bit_cast(float, sel_bits[i]);
    else out_vals[row * k + rank] = vals[row * val_stride + (idx < val_stride ? idx : val_stride - 1)];
    out_idx[row * k + rank] = idx;
  }
}

// One workgroup of NT threads selects the best k of its CH / NT keys a thread (0: padding).
// FIRST && LAST: v holds the keys' scores, whose own bits are written up to k =
// kRankSortMaxK; otherwise LAST reads the values back from the scores (vals, row stride
// val_stride) at the selected indices. Both keep the input's bits (-0.0, NaN payloads). Not LAST: the keys go to keys_out (memory
// or LDS). Every thread of the workgroup calls it (it synchronises the workgroup).
template <bool FIRST, bool LAST, int NT, int CH>
__device__ __forceinline__ void topk_core(uint64_t (&key)[CH / NT], const float (&v)[CH / NT],
                                          const float* __restrict__ vals, int64_t val_stride, int64_t n_in,
                                          uint64_t* keys_out, int64_t out_stride, float* __restrict__ out_vals,
                                          int64_t* __restrict__ out_idx, int k, int64_t row, int64_t chunk) {
  constexpr int kPerThread = CH / NT;
  constexpr int kTopkWaves = NT / 64;
  static_assert(NT % 256 == 0 && NT <= kHistCopies * 256, "histogram clearing and the per-wave copies");
  static_assert(kTopkWaves <= 64, "one lane per wave in the cross-wave reduction");
  // Three histogram buffers: pass p counts into buffer p % 3, and buffer (p + 2) % 3 is
  // cleared after pass p's barrier, when no wave can still be scanning it (its last
  // scan, in pass p - 1, ended before that barrier) -- one barrier per pass.
  __shared__ uint32_t hist[3][kHistCopies][256];
  __shared__ uint32_t n_gt, n_eq, n_cand;
  __shared__ uint64_t cand[LAST ? 1 : kCandCap];
  __shared__ uint32_t red_t[kTopkWaves], red_m[kTopkWaves];
  __shared__ uint64_t sel[LAST ? kMaxK : 1];
  // FIRST && LAST (a row that fits one chunk): the selected scores' own bits, kept from
  // the loads so the output needs no second read of the scores.
  __shared__ uint32_t sel_bits[(FIRST && LAST) ? kMaxK : 1];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  auto rank_out = [&](int m, int m8) {
    topk_rank_out<FIRST, NT>(sel, sel_bits, m, m8, vals, val_stride, out_vals, out_idx, k, row);
  };

  if constexpr (FIRST && LAST) {
    // A row of at most NT scores holds one key per thread (element tid), all real and
    // distinct (the index is in the low word): the top k are the keys of rank < k, with
    // no radix passes. n^2 / S compares per lane; at n = 256 about a quarter of the
    // passes' time.
    if (n_in <= NT && n_in <= kRankSortMaxK) {
      const int m8 = ((int)n_in + 7) & ~7;
      for (int t = tid; t < kRankSortMaxK + kRankPad; t += NT) sel[t] = t == tid ? key[0] : 0ull;  // 0 past the row
      if (tid < m8) sel_bits[tid] = __builtin_bit_cast(uint32_t, v[0]);
      __syncthreads();
      rank_out((int)n_in, m8);
      return;
    }
  }

  // Set-up that the first barrier below orders before its use: the first two histogram
  // buffers, the slot counters, and (last level) the padding slots of the rank sort.
  for (int i = tid; i < 2 * kHistCopies * 256; i += NT) (&hist[0][0][0])[i] = 0u;
  if (tid == 0) {
    n_gt = 0u;
    n_eq = 0u;
    n_cand = 0u;
  }
  if constexpr (LAST) {
    const int k8 = (k + 7) & ~7;
    if (k <= kRankSortMaxK)
      for (int t = k + tid; t < k8 + kRankPad; t += NT) sel[t] = 0ull;
  }
  auto below = [&](uint64_t m) -> uint32_t {  // set bits of m in lanes below this one
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  };

  // The selection below runs over key[0, E); key[E, kPerThread) are 0 (padding). After
  // the pre-filter, the candidates' high words lie in [fT, fM].
  int E = kPerThread;
  bool filtered = false;
  uint32_t fT = 0u, fM = 0u;
  if constexpr (!LAST) {
    // Pre-filter. Wave w finds T_w, the j-th largest of its 64 threads' maximum high words
    // (j = ceil(k / waves); padding counts as 0). Each of those j threads holds a key whose
    // high word is >= T_w, so the chunk has at least waves * j >= k keys whose high word
    // is >= T = min_w T_w, and every key below T is below all of them: the top k lie among
    // the keys with high word >= T. On continuous scores they are a few k; they are
    // gathered in LDS and selected from there, at most kCandCap / NT per thread. T = 0
    // (fewer than j real keys in some wave) or more than kCandCap candidates (ties at the
    // bound) keep the registers and the full selection.
    if (k <= kFilterMaxK) {
      static_assert(kFilterMaxK <= 64 * kTopkWaves, "j <= 64: the bound is taken within each wave");
      static_assert(kCandCap % NT == 0 && kCandCap / NT <= kPerThread, "candidates per thread");
      uint32_t tm = 0u;
#pragma unroll
      for (int e = 0; e < kPerThread; e++) {
        const uint32_t h = (uint32_t)(key[e] >> 32);
        tm = h > tm ? h : tm;
      }
      // the j-th largest of the wave's tm, one bit at a time from the top: the largest t
      // that at least j lanes reach
      const uint32_t j = (uint32_t)((k + kTopkWaves - 1) / kTopkWaves);
      uint32_t t = 0u;
#pragma unroll
      for (int b = 31; b >= 0; b--) {
        const uint32_t c = t | (1u << b);
        t = (uint32_t)__popcll(__ballot(tm >= c)) >= j ? c : t;
      }
      const uint32_t wm = wave_max_u32(tm, lane);
      if (lane == 0) {
        red_t[wid] = t;
        red_m[wid] = wm;
      }
      __syncthreads();
      uint32_t T = red_t[0], M = red_m[0];
#pragma unroll
      for (int w = 1; w < kTopkWaves; w++) {
        T = red_t[w] < T ? red_t[w] : T;
        M = red_m[w] > M ? red_m[w] : M;
      }
      if (T != 0u) {  // uniform
        uint64_t mc[kPerThread];
        uint32_t wave_n = 0u;
#pragma unroll
        for (int e = 0; e < kPerThread; e++) {
          mc[e] = __ballot((uint32_t)(key[e] >> 32) >= T);
          wave_n += (uint32_t)__popcll(mc[e]);
        }
        uint32_t base = 0u;
        if (lane == 0) base = atomicAdd(&n_cand, wave_n);
        base = (uint32_t)__builtin_amdgcn_readlane((int)base, 0);
#pragma unroll
        for (int e = 0; e < kPerThread; e++) {
          const uint32_t pos = base + below(mc[e]);
          if ((uint32_t)(key[e] >> 32) >= T && pos < (uint32_t)kCandCap) cand[pos] = key[e];
          base += (uint32_t)__popcll(mc[e]);
        }
        __syncthreads();
        const uint32_t nc = (uint32_t)__builtin_amdgcn_readfirstlane((int)n_cand);
        if (nc <= (uint32_t)kCandCap) {
          filtered = true;
          fT = T;
          fM = M;
          E = (int)((nc + NT - 1) / NT);
#pragma unroll
          for (int e = 0; e < kPerThread; e++) {
            const uint32_t p = (uint32_t)(e * NT + tid);
            key[e] = (e < kCandCap / NT && p < nc) ? cand[e < kCandCap / NT ? p : 0] : 0ull;
          }
        }
      }
    }
  }

  // Where the real keys differ: the radix passes start below the bits that every real
  // key shares (scores in one binade share sign, exponent and the top mantissa bits), so
  // a row of similar scores takes two or three passes instead of up to eight. Padding
  // keys (0) are not real; a chunk with fewer than k real keys starts from the top.
  __shared__ uint64_t red_lo[kTopkWaves], red_hi[kTopkWaves];
  __shared__ uint32_t red_n[kTopkWaves];
  uint64_t prefix = 0;  // the key bits fixed so far: candidates have key >> shift == prefix
  int shift = 64;
  if (filtered) {
    // At least k candidates, all with high words in [fT, fM]: they share the bits above
    // the highest bit at which fT and fM differ (all 32 if they are equal).
    const uint32_t diff = fT ^ fM;
    shift = diff == 0u ? 32 : 64 - __builtin_clz(diff);
    prefix = shift == 64 ? 0ull : ((uint64_t)fM << 32) >> shift;
  } else {
    uint64_t lo = ~0ull, hi = 0ull;
    uint32_t nr = 0u;
#pragma unroll
    for (int e = 0; e < kPerThread; e++) {
      if (e < E && key[e] != 0ull) {
        lo = key[e] < lo ? key[e] : lo;
        hi = key[e] > hi ? key[e] : hi;
        nr++;
      }
    }
    wave_minmax(lo, hi, nr, lane);
    if (lane == 0) {
      red_lo[wid] = lo;
      red_hi[wid] = hi;
      red_n[wid] = nr;
    }
    __syncthreads();
    // lane w brings wave w's partial results; every lane gets the chunk's
    lo = lane < kTopkWaves ? red_lo[lane] : ~0ull;
    hi = lane < kTopkWaves ? red_hi[lane] : 0ull;
    nr = lane < kTopkWaves ? red_n[lane] : 0u;
    wave_minmax(lo, hi, nr, lane);
    if (nr >= (uint32_t)k) {
      const uint64_t diff = hi ^ lo;
      shift = diff == 0ull ? 0 : 64 - __builtin_clzll(diff);
      prefix = shift == 64 ? 0ull : hi >> shift;
    }
  }

  // Radix select, 8-bit digits (narrower for the last one). After a pass, `need` is the
  // number of keys still to take among the keys that share the prefix.
  uint32_t need = (uint32_t)k;
  bool whole_bin = false;  // the selection is every key >= prefix << shift
  for (int pass = 0; shift > 0; pass++) {
    const int w = shift < 8 ? shift : 8;
    shift -= w;
    uint32_t(&hb)[kHistCopies][256] = hist[pass % 3];
    {
      uint32_t run_bin = 0u, run_n = 0u;  // a run of this thread's keys in one bin
      auto count = [&](uint32_t bin) {
        if (run_n != 0u && bin != run_bin) {
          atomicAdd(&hb[wid % kHistCopies][run_bin], run_n);
          run_n = 0u;
        }
        run_bin = bin;
        run_n++;
      };
      if (shift >= 32) {
        // The digit lies in the high word (the score's order bits, where rows of distinct
        // scores are decided): 32-bit shifts and one bit-field extract per key instead of
        // 64-bit shifts. top = shift + w - 32 <= 32; top == 32 is the first pass from the
        // top, which every key takes.
        const uint32_t sh = (uint32_t)(shift - 32), top = sh + (uint32_t)w, pre = (uint32_t)prefix;
#pragma unroll
        for (int e = 0; e < kPerThread; e++) {
          if (e >= E) break;
          const uint32_t hi = (uint32_t)(key[e] >> 32);
          if (top == 32u || (hi >> top) == pre) count(__builtin_amdgcn_ubfe(hi, sh, (uint32_t)w));
        }
      } else {
#pragma unroll
        for (int e = 0; e < kPerThread; e++) {
          if (e >= E) break;
          if (shift + w == 64 || (key[e] >> (shift + w)) == prefix)
            count((uint32_t)(key[e] >> shift) & ((1u << w) - 1u));
        }
      }
      if (run_n != 0u) atomicAdd(&hb[wid % kHistCopies][run_bin], run_n);
    }
    __syncthreads();
    for (int i = tid; i < kHistCopies * 256; i += NT) (&hist[(pass + 2) % 3][0][0])[i] = 0u;
    // Every wave scans the histogram itself (lane l: bins 255 - 4l .. 252 - 4l, high to
    // low) and finds the bin that holds the need-th key.
    uint32_t c[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int bin = 255 - 4 * lane - j;
      c[j] = hb[0][bin] + hb[1][bin] + hb[2][bin] + hb[3][bin];
    }
    const uint32_t own = c[0] + c[1] + c[2] + c[3];
    const uint32_t incl = wave_inclusive_sum(own);
    const uint32_t excl = incl - own;
    const bool mine = excl < need && need <= incl;  // exactly one lane
    uint32_t above = excl, j = 0;
    if (mine)
      while (above + c[j] < need) above += c[j++];
    const uint32_t cj = c[0] * (j == 0) + c[1] * (j == 1) + c[2] * (j == 2) + c[3] * (j == 3);
    const int src = (int)__builtin_ctzll(__ballot(mine)) & 63;
    const uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)(255 - 4 * lane - j), src);
    const uint32_t cnt = (uint32_t)__builtin_amdgcn_readlane((int)cj, src);
    above = (uint32_t)__builtin_amdgcn_readlane((int)above, src);
    need -= above;
    prefix = (prefix << w) | d;
    if (cnt == need && prefix != 0) {  // the whole bin is needed (keys are unique but padding)
      whole_bin = true;
      break;
    }
  }
  // Selection: every key > T, then `need` keys equal to T (only padding keys repeat).
  // Each wave reserves its slots with one atomic per 64 keys (ballot and lane count).
  const uint64_t T = whole_bin ? (prefix << shift) - 1 : prefix;
  const uint32_t need_eq = whole_bin ? 0u : need;
  auto put = [&](uint32_t pos, uint64_t kv, int e) {
    if constexpr (FIRST && LAST) sel_bits[pos] = __builtin_bit_cast(uint32_t, v[e]);
    if constexpr (LAST) sel[pos] = kv;
    else keys_out[row * out_stride + chunk * k + pos] = kv;
  };
  // The wave's selected keys in element order: ballots first, then one atomic per wave
  // for all of them (and one for the keys equal to T, which only padding can need).
  uint64_t mg[kPerThread];
  uint32_t wave_gt = 0u, wave_eq = 0u;
  uint64_t any_eq = 0ull;
#pragma unroll
  for (int e = 0; e < kPerThread; e++) {
    mg[e] = 0ull;
    if (e >= E) continue;
    mg[e] = __ballot(key[e] > T);
    wave_gt += (uint32_t)__popcll(mg[e]);
    if (need_eq > 0u) {
      const uint64_t me = __ballot(key[e] == T);
      any_eq |= me;
      wave_eq += (uint32_t)__popcll(me);
    }
  }
  uint32_t base_gt = 0u, base_eq = 0u;
  if (lane == 0 && wave_gt > 0u) base_gt = atomicAdd(&n_gt, wave_gt);
  if (lane == 0 && wave_eq > 0u) base_eq = atomicAdd(&n_eq, wave_eq);
  base_gt = (uint32_t)__builtin_amdgcn_readlane((int)base_gt, 0);
  base_eq = (uint32_t)__builtin_amdgcn_readlane((int)base_eq, 0);
#pragma unroll
  for (int e = 0; e < kPerThread; e++) {
    if (e >= E) break;
    if (mg[e] != 0ull) {
      const uint32_t pos = base_gt + below(mg[e]);
      if (key[e] > T && pos < (uint32_t)k - need_eq) put(pos, key[e], e);  // always below; bounds every write
      base_gt += (uint32_t)__popcll(mg[e]);
    }
    if (any_eq != 0ull) {
      const uint64_t me = __ballot(key[e] == T);
      const uint32_t j = base_eq + below(me);
      if (key[e] == T && j < need_eq) put((uint32_t)k - need_eq + j, key[e], e);
      base_eq += (uint32_t)__popcll(me);
    }
  }
  if constexpr (LAST) {
    __syncthreads();
    if (k <= kRankSortMaxK) {  // every selected key is real, so all are distinct: rank = keys above it
      rank_out(k, (k + 7) & ~7);  // the slots past k hold 0 (set at the start)
      return;
    }
    int P = 1;  // bitonic sort of the k survivors, padded to a power of two
    while (P < k) P <<= 1;
    for (int i = k + tid; i < P; i += NT) sel[i] = 0;
    __syncthreads();
    for (int size = 2; size <= P; size <<= 1) {
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        for (int i = tid; i < P / 2; i += NT) {
          const int pos = 2 * i - (i & (stride - 1));
          const int partner = pos + stride;
          const bool desc = (pos & size) == 0;
          const uint64_t a = sel[pos], b = sel[partner];
          if ((a < b) == desc) {
            sel[pos] = b;
            sel[partner] = a;
          }
        }
        __syncthreads();
      }
    }
    for (int i = tid; i < k; i += NT) {
      const int64_t idx = (int64_t)(0xffffffffu - (uint32_t)sel[i]);
      // a selected key is always a real element (k <= n); the clamp only bounds the read
      out_vals[row * k + i] = vals[row * val_stride + (idx < val_stride ? idx : val_stride - 1)];
      out_idx[row * k + i] = idx;
    }
  }
}


// topk_core over chunk `chunk` of row `row`.
template <bool FIRST, bool LAST, int NT, int CH = kChunk>
__device__ __forceinline__ void topk_chunk(const float* __restrict__ vals, int64_t val_stride,
                                           const uint64_t* __restrict__ keys_in, int64_t n_in, int64_t in_stride,
                                           uint64_t* __restrict__ keys_out, int64_t out_stride,
                                           float* __restrict__ out_vals, int64_t* __restrict__ out_idx, int k,
                                           int64_t row, int64_t chunk) {
  constexpr int kPerThread = CH / NT;
  const int tid = threadIdx.x;
  const int64_t c0 = chunk * CH;
  // All loads are issued before any key is formed (one memory round trip, not one per
  // element). A chunk inside the row reads from one uniform base at 32-bit offsets and
  // every key is real; in the row's last chunk, positions past the row read its last
  // element and become padding.
  uint64_t key[kPerThread];
  float v[kPerThread] = {};
  const bool inside = c0 + CH <= n_in;  // uniform
  if constexpr (FIRST) {
    if (inside) {
      const float* __restrict__ base = vals + row * val_stride + c0;
#pragma unroll
      for (int e = 0; e < kPerThread; e++) v[e] = base[e * NT + tid];
      const uint32_t inv = 0xffffffffu - (uint32_t)c0 - (uint32_t)tid;  // inverted index of element 0
#pragma unroll
      for (int e = 0; e < kPerThread; e++)
        key[e] = ((uint64_t)order_key(v[e]) << 32) | (uint64_t)(inv - (uint32_t)(e * NT));
    } else {
#pragma unroll
      for (int e = 0; e < kPerThread; e++) {
        const int64_t p = c0 + e * NT + tid;
        v[e] = vals[row * val_stride + (p < n_in ? p : n_in - 1)];
      }
#pragma unroll
      for (int e = 0; e < kPerThread; e++) {
        const int64_t p = c0 + e * NT + tid;
        key[e] = p < n_in ? ((uint64_t)order_key(v[e]) << 32) | (uint64_t)(0xffffffffu - (uint32_t)p)
                          : 0ull;  // below every real element
      }
    }
  } else {
    if (inside) {
      const uint64_t* __restrict__ base = keys_in + row * in_stride + c0;
#pragma unroll
      for (int e = 0; e < kPerThread; e++) key[e] = base[e * NT + tid];
    } else {
#pragma unroll
      for (int e = 0; e < kPerThread; e++) {
        const int64_t p = c0 + e * NT + tid;
        key[e] = keys_in[row * in_stride + (p < n_in ? p : n_in - 1)];
      }
#pragma unroll
      for (int e = 0; e < kPerThread; e++) {
        const int64_t p = c0 + e * NT + tid;
        key[e] = p < n_in ? key[e] : 0ull;
      }
    }
  }

  topk_core<FIRST, LAST, NT, CH>(key, v, vals, val_stride, n_in, keys_out, out_stride, out_vals, out_idx, k, row, chunk);
}

template <bool FIRST, bool LAST, int NT, int CH = kChunk>
__global__ void __launch_bounds__(NT) topk_level_kernel(const float* __restrict__ vals, int64_t val_stride,
                                                        const uint64_t* __restrict__ keys_in, int64_t n_in,
                                                        int64_t in_stride, uint64_t* __restrict__ keys_out,
                                                        int64_t out_stride, float* __restrict__ out_vals,
                                                        int64_t* __restrict__ out_idx, int k) {
  topk_chunk<FIRST, LAST, NT, CH>(vals, val_stride, keys_in, n_in, in_stride, keys_out, out_stride, out_vals, out_idx, k,
                                  blockIdx.y, blockIdx.x);
}

// Long rows by group maxima. One pass over the scores writes the largest key of every group
// of g = 4 << LG consecutive scores, and of every 1,024 (a span). The top k then lie in the
// k best groups, and those in the k best spans (compared by maximum, then by position): an
// element outside them has k maxima above it. So one workgroup a row selects spans, then
// their groups, then the scores of those groups, from at most CHS keys at a time, and reads
// g k scores again instead of sorting every chunk. The first pass is bound by the read of the
// scores; the tournament's first level was bound by its issue (VALUBusy 71-81 %).
constexpr int kGroupWaves = 4;  // waves per workgroup of the first pass

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // rows start at any score

// Largest key over the 1 << LG consecutive lanes of a group (every lane gets it).
template <int LG>
__device__ __forceinline__ uint32_t lanes_max_u32(uint32_t x, int lane) {
  auto mx = [](uint32_t a, uint32_t b) { return a > b ? a : b; };
  x = mx(x, dpp_u32<0xB1>(x));                       // quad_perm [1,0,3,2]
  x = mx(x, dpp_u32<0x4E>(x));                       // quad_perm [2,3,0,1]
  x = mx(x, dpp_u32<0x141>(x));                      // row_half_mirror
  if constexpr (LG >= 4) x = mx(x, dpp_u32<0x140>(x));  // row_mirror
  if constexpr (LG >= 5) x = mx(x, swap16_u32(x, lane));
  if constexpr (LG >= 6) x = mx(x, swap32_u32(x, lane));
  return x;
}

// LG = 3..6: 8 to 64 lanes of four scores a group (g = 32 to 256). Each wave walks spans of
// row blockIdx.y; lane l reads scores 256 j + 4 l .. + 4 of a span, j = 0..3. groups:
// (nrows, spans * kSpan / g), spans_out (or null): (nrows, spans); 0 for a group past the row.
template <int LG>
__global__ void __launch_bounds__(64 * kGroupWaves) topk_group_max_kernel(const float* __restrict__ vals, int64_t n,
                                                                          int64_t spans,
                                                                          uint32_t* __restrict__ groups,
                                                                          uint32_t* __restrict__ spans_out) {
  constexpr int LPG = 1 << LG;               // lanes per group
  constexpr int GPL = 64 / LPG;              // groups per 256 scores
  const int lane = threadIdx.x & 63;
  const int64_t stride = (int64_t)gridDim.x * kGroupWaves;
  const int64_t row = blockIdx.y;
  for (int64_t sp = (int64_t)blockIdx.x * kGroupWaves + (threadIdx.x >> 6); sp < spans; sp += stride) {
    const float* __restrict__ p = vals + row * n + sp * kSpan;
    const int64_t left = n - sp * kSpan;  // scores of the row from the span on
    uint32_t m[4];
    if (left >= kSpan) {  // uniform
      f32x4 x[4];
#pragma unroll
      for (int j = 0; j < 4; j++) x[j] = __builtin_nontemporal_load((const f32x4u*)(p + 256 * j + 4 * lane));
#pragma unroll
      for (int j = 0; j < 4; j++) {
        // the float maximum's key, or the NaN key when some score's bits (sign shifted out)
        // are a NaN's, about two operations a score
        const float f = fmaxf(fmaxf(x[j][0], x[j][1]), fmaxf(x[j][2], x[j][3]));
        uint32_t nan = 0u;
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const float xq = x[j][q];
          const uint32_t b = __builtin_bit_cast(uint32_t, xq) << 1;
          nan = b > nan ? b : nan;
        }
        const uint32_t fb = __builtin_bit_cast(uint32_t, f);
        const uint32_t o = (int32_t)fb < 0 ? 0u - fb : (fb | 0x80000000u);
        m[j] = nan > 0xff000000u ? 0xffffffffu : o;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        float x[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int64_t i = 256 * j + 4 * lane + q;
          x[q] = p[i < left ? i : left - 1];
        }
        m[j] = 0u;
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const uint32_t b = 256 * j + 4 * lane + q < left ? order_key(x[q]) : 0u;
          m[j] = b > m[j] ? b : m[j];
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) m[j] = lanes_max_u32<LG>(m[j], lane);
    // lane j of a group's lanes keeps the j-th 256 scores' maximum
    const int j = lane & (LPG - 1);
    const uint32_t mine = j == 0 ? m[0] : (j == 1 ? m[1] : (j == 2 ? m[2] : m[3]));
    if (j < 4) groups[(row * spans + sp) * (4 * GPL) + j * GPL + lane / LPG] = mine;
    if (spans_out) {
      uint32_t a = m[0] > m[1] ? m[0] : m[1], b = m[2] > m[3] ? m[2] : m[3];
      a = wave_max_u32(a > b ? a : b, lane);
      if (lane == 0) spans_out[row * spans + sp] = a;
    }
  }
}

// The selection of one row: spans (when spans_in is given: at most CH1 of them), their
// groups, their scores. lg: groups of 4 << lg scores, at most CHS / k of them in a span and
// at most CHS / k scores in a group; without spans_in, at most CHS groups a row.
//
// First the fast way: the k-th largest maximum T is a bound on the k-th largest score, so
// after one selection among the maxima only what reaches T is kept: the k best spans' groups,
// those groups' scores (on continuous scores a few more than k), and the scores kept are
// ordered by rank. Where more are kept than ranks are cheap for (sorted rows, ties) the last
// selection, or the last two, run over the groups or spans found so far: 1 row of 5,000 scores in
// sorted runs of 100, k = 100, 16 us (59 by ranks of up to 2,048), 64 sorted rows of 8,192 18
// (26 with all selections anew). 32 rows of 1M scores, k = 100: 32 us with the first pass,
// against 58 for the tournament and 41 selecting level by level throughout.
constexpr int kFastCap = 2048;
template <int CH1, int CHS>
__global__ void __launch_bounds__(kLastThreads) topk_group_last_kernel(const float* __restrict__ vals, int64_t n,
                                                                       int64_t spans, int lg,
                                                                       const uint32_t* __restrict__ groups,
                                                                       const uint32_t* __restrict__ spans_in,
                                                                       float* __restrict__ out_vals,
                                                                       int64_t* __restrict__ out_idx, int k) {
  constexpr int NT = kLastThreads, NW = NT / 64;
  constexpr int PER = CHS / NT;
  constexpr int kRankCap = CHS <= 4096 ? 768 : 1024;  // scores ordered by rank, within one turn of the threads
  __shared__ uint64_t picked[kMaxK];
  __shared__ uint32_t gsel[kFastCap];
  enum { NOTHING, FIRST_MAXIMA, GROUPS } have = NOTHING;  // selected so far: picked (of `top`), or gsel and total
  int total = 0;      // scores of the groups in gsel
  uint32_t at[PER];   // their indices (past the row: 2^32 - 1) and values
  float v[PER] = {};
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x;
  const int per = kSpan >> (lg + 2);  // groups per span
  const int glog = lg + 2;            // log2 of the scores per group
  const uint32_t* __restrict__ grow = groups + row * spans * per;
  const float* __restrict__ vrow = vals + row * n;
  auto load_scores = [&](int c0) {  // scores [c0, c0 + CHS) of the total
#pragma unroll
    for (int e = 0; e < PER; e++) {
      const int c = c0 + e * NT + tid;
      const bool in = c < total;
      const uint64_t i = ((uint64_t)gsel[in ? c >> glog : 0] << glog) + (uint64_t)(c & ((1 << glog) - 1));
      at[e] = in && i < (uint64_t)n ? (uint32_t)i : 0xffffffffu;
      v[e] = vrow[at[e] != 0xffffffffu ? at[e] : 0u];
    }
  };

  {
    __shared__ uint64_t list[kFastCap];
    __shared__ uint32_t wave_t[NW], n_list, n_groups, n_sel, bound;
    __shared__ uint64_t sel[kRankCap + kRankPad + 8];
    __shared__ uint32_t sel_bits[kRankCap];
    const int lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    // appends the lanes with `take` to a list; returns the lane's slot
    auto slot = [&](uint32_t* count, bool take) -> uint32_t {
      const uint64_t mask = __ballot(take);
      uint32_t base = 0u;
      if (mask != 0ull) {
        if (lane == 0) base = atomicAdd(count, (uint32_t)__popcll(mask));
        base = (uint32_t)__builtin_amdgcn_readlane((int)base, 0);
      }
      return base + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
    };
    // the maxima of the first level, spread over the waves (wave c % 16 holds maximum c)
    constexpr int P1 = (CH1 > CHS ? CH1 : CHS) / NT;
    const uint32_t* __restrict__ top = spans_in ? spans_in + row * spans : grow;
    const int count = (int)(spans_in ? spans : spans * per);
    uint32_t x[P1];
    uint32_t tm = 0u;
#pragma unroll
    for (int e = 0; e < P1; e++) {
      const int c = e * NT + lane * NW + wid;
      x[e] = c < count ? top[c] : 0u;
      tm = x[e] > tm ? x[e] : tm;
    }
    if (tid == 0) n_list = n_groups = n_sel = 0u;
    for (int i = tid; i < kRankCap + kRankPad + 8; i += NT) sel[i] = 0ull;
    // a lower bound on the k-th maximum, as in topk_core's pre-filter
    const uint32_t j = (uint32_t)((k + NW - 1) / NW);
    uint32_t t = 0u;
#pragma unroll
    for (int b = 31; b >= 0; b--) {
      const uint32_t c = t | (1u << b);
      t = (uint32_t)__popcll(__ballot(tm >= c)) >= j ? c : t;
    }
    if (lane == 0) wave_t[wid] = t;
    __syncthreads();
    uint32_t T = wave_t[0];
#pragma unroll
    for (int w = 1; w < NW; w++) T = wave_t[w] < T ? wave_t[w] : T;
    bool ok = T != 0u;  // uniform, as every decision below
    if (ok) {
#pragma unroll
      for (int e = 0; e < P1; e++) {
        if (e * NT >= count) break;
        const int c = e * NT + lane * NW + wid;
        const bool take = x[e] >= T;
        const uint32_t p = slot(&n_list, take);
        if (take && p < (uint32_t)kFastCap) list[p] = ((uint64_t)x[e] << 32) | (uint64_t)(0xffffffffu - (uint32_t)c);
      }
      __syncthreads();
      const int m = (int)n_list;
      ok = m <= kFastCap;
      if (ok) {
        // ranks by count, four or two lanes a key for a short list: the keys of rank < k are the k
        // best, in order, and the last of them is the bound
        const int lgS = m <= NT / 4 ? 2 : (m <= NT / 2 ? 1 : 0);
        const int part = tid & ((1 << lgS) - 1);
        for (int i = tid >> lgS; i < m; i += NT >> lgS) {  // one turn when lanes share keys
          const uint64_t me = list[i];
          uint32_t rank = 0u;
#pragma unroll 8
          for (int q = part; q < m; q += 1 << lgS) rank += list[q] > me ? 1u : 0u;
          if (lgS > 0) rank += dpp_u32<0xB1>(rank);  // a key's lanes take the turn together
          if (lgS > 1) rank += dpp_u32<0x4E>(rank);
          if (part == 0 && rank < (uint32_t)k) {
            picked[rank] = me;
            if (rank == (uint32_t)k - 1u) bound = (uint32_t)(me >> 32);
          }
        }
        __syncthreads();
        T = bound;
        have = FIRST_MAXIMA;
        uint32_t ng;
        if (spans_in) {
          uint32_t y[PER];
#pragma unroll
          for (int e = 0; e < PER; e++) {
            const int c = e * NT + tid;
            const uint32_t span = c < k * per ? 0xffffffffu - (uint32_t)picked[c / per] : 0u;
            at[e] = span * (uint32_t)per + (uint32_t)(c & (per - 1));
            y[e] = c < k * per ? grow[at[e]] : 0u;
          }
#pragma unroll
          for (int e = 0; e < PER; e++) {
            const bool take = y[e] >= T;  // T > 0
            const uint32_t p = slot(&n_groups, take);
            if (take && p < (uint32_t)kFastCap) gsel[p] = at[e];
          }
          __syncthreads();
          ng = n_groups;
        } else {
          if (tid < k) gsel[tid] = 0xffffffffu - (uint32_t)picked[tid];
          __syncthreads();
          ng = (uint32_t)k;
        }
        ok = ng <= (uint32_t)kFastCap && (int)(ng << glog) <= 4 * CHS;
        if (ok) {
          total = (int)(ng << glog);
          for (int c0 = 0; c0 < total; c0 += CHS) {
            load_scores(c0);
#pragma unroll
            for (int e = 0; e < PER; e++) {
              const uint32_t o = order_key(v[e]);
              const bool take = at[e] != 0xffffffffu && o >= T;
              const uint32_t p = slot(&n_sel, take);
              if (take && p < (uint32_t)kRankCap) {
                sel[p] = ((uint64_t)o << 32) | (uint64_t)(0xffffffffu - at[e]);
                sel_bits[p] = __builtin_bit_cast(uint32_t, v[e]);
              }
            }
          }
          if (total <= CHS) have = GROUPS;
          __syncthreads();
          const int ms = (int)n_sel;  // >= k: each of the k best maxima is one
          if (ms <= kRankCap) {
            topk_rank_out<true, NT>(sel, sel_bits, ms, (ms + 7) & ~7, nullptr, 0, out_vals, out_idx, k, row);
            return;
          }
        }
      }
    }
    __syncthreads();
  }

  uint64_t key[PER];
  if (have != GROUPS) {
    if (spans_in) {
      if (have == NOTHING) {
        uint64_t k1[CH1 / NT];
        const float none[CH1 / NT] = {};
#pragma unroll
        for (int e = 0; e < CH1 / NT; e++) {
          const int64_t c = e * NT + tid;
          k1[e] = c < spans ? ((uint64_t)spans_in[row * spans + c] << 32) | (uint64_t)(0xffffffffu - (uint32_t)c) : 0ull;
        }
        topk_core<false, false, NT, CH1>(k1, none, nullptr, 0, spans, picked, 0, nullptr, nullptr, k, 0, 0);
        __syncthreads();
      }
#pragma unroll
      for (int e = 0; e < PER; e++) {
        const int c = e * NT + tid;
        const uint32_t span = c < k * per ? 0xffffffffu - (uint32_t)picked[c / per] : 0u;
        at[e] = span * (uint32_t)per + (uint32_t)(c & (per - 1));
        key[e] = c < k * per ? (uint64_t)grow[at[e]] : 0ull;
      }
#pragma unroll
      for (int e = 0; e < PER; e++) key[e] = key[e] != 0ull ? (key[e] << 32) | (uint64_t)(0xffffffffu - at[e]) : 0ull;
      __syncthreads();  // picked is read; the next selection writes it
    } else {
#pragma unroll
      for (int e = 0; e < PER; e++) {
        const int64_t c = e * NT + tid;
        const uint32_t x = c < spans * per ? grow[c] : 0u;
        key[e] = x != 0u ? ((uint64_t)x << 32) | (uint64_t)(0xffffffffu - (uint32_t)c) : 0ull;
      }
    }
    topk_core<false, false, NT, CHS>(key, v, nullptr, 0, CHS, picked, 0, nullptr, nullptr, k, 0, 0);
    __syncthreads();
    // a padding key (fewer than k groups) names no group: its first score lies past the row
    if (tid < k) gsel[tid] = picked[tid] != 0ull ? 0xffffffffu - (uint32_t)picked[tid] : 0xffffffffu;
    __syncthreads();
    total = k << glog;
    load_scores(0);
  } else if (PER > 4) {  // too many to have been kept in registers
    load_scores(0);
  }
#pragma unroll
  for (int e = 0; e < PER; e++)
    key[e] = at[e] != 0xffffffffu ? ((uint64_t)order_key(v[e]) << 32) | (uint64_t)(0xffffffffu - at[e]) : 0ull;
  topk_core<true, true, NT, CHS>(key, v, vals, n, n, nullptr, 0, out_vals, out_idx, k, row, 0);
}

}  // namespace tms
