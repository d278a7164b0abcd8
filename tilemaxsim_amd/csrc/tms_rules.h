// Rules that pick a kernel's form from a call's sizes alone, in plain C++ so that they build
// and are tested without a GPU. Figures are microseconds a call on one MI355X.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace tms {

constexpr size_t kLdsPerCu = 160 * 1024;

// Waves that each fixed-length document of `tiles` tiles is split over in a small call of the
// general dense kernel: 1, 2 or 4, at most one a tile. A small call is bound by each wave's walk
// of its tiles, so a split helps while all the waves it makes run at once and each gets as
// far as it would alone.
//  * Query in LDS (ks_reg = 0; `lds` bytes of it): up to two waves a SIMD, one where a
//    workgroup's LDS leaves no room for a second one. fp16, 180 tokens, whole / in two / in
//    four: d = 512, 300 documents 32 / 21 / 19, 600 33 / 28; d = 1280 (80 KiB) 300 75 / 45 /
//    63, 600 78 / 88.
//  * Query in registers (fp32, or an fp32 query; ks_reg = d / 32 k-steps, nqb blocks): its
//    several MFMAs a product and the splitting keep one wave a SIMD busy, so 1,024 waves.
//    d = 128, two blocks, 33 tokens: 300 documents 10.3 whole and 9.5 in two, 600 10.4 and
//    17.3. Up to 1,536 where a tile is little work (one block of d = 64, 400 tokens: 600
//    documents 23 whole, 17 in two) or a walk is long (d = 96, 1,000 tokens, two blocks: 76, 64).
inline int dense_split_waves(int64_t B, int64_t tiles, size_t lds, int nqb, int ks_reg) {
  int64_t most;
  if (ks_reg > 0) {
    const int work = ks_reg * nqb;
    most = work <= 2 || (work <= 6 && tiles >= (work <= 3 ? 12 : 24)) ? 1536 : 1024;
  } else {
    const size_t fixed = 256 + 512 * (size_t)nqb;  // the kernel's static LDS
    most = 2 * (lds + fixed) <= kLdsPerCu ? 2048 : 1024;
  }
  int w = 1;
  while (w < 4 && 2 * w <= tiles && 2 * w * B <= most) w *= 2;
  return w;
}

// Whether batched queries over B documents spread their blocks over eight waves, one or two
// blocks each (tms_batched_kernel.h), rather than over four of up to four. Up to one document
// a CU, each workgroup has a CU to itself and walks its document as fast as one wave's step
// goes; above, two to four workgroups of four waves a CU do more than one of eight. d = 128,
// 1,000 tokens, 6 queries, over four / eight waves: 50 documents fp16 1 / 0.80, fp32 1 / 0.74; 256
// documents 1 / 0.85 and 0.80; 300 documents 1 / 1.37 and 1.20.
inline bool batched_spread(int64_t B) { return B <= 256; }

// Whether a batched PQ call (nQ queries of nbq blocks, `tokens` of them, M codes of dsub
// dimensions a token, a codebook of `lds` bytes) goes query by query. One pass of the
// shared-tile workgroups waits on each tile's gathers whatever the queries are, so a few
// queries over many tokens are faster one at a time, in their own kernel. With fewer tokens the
// launches and each workgroup's codebook copy weigh more: blocks^2 x 131,072 tokens are enough for
// two queries, or for five of a codebook that leaves a CU room for two shared-tile workgroups
// (above 37 KiB, codewords of 8 to 32 bytes: `wide`), else twice that. A shared pass takes the
// time of 5 to 6 queries there, of 3 to 4 where a query's own kernel gathers many short or few
// long codewords (dsub = 2 of M = 32 or 64, dsub = 32), else of 4 to 5. 25.6M tokens, 2, 4 and
// 6 queries, shared / one at a time: M = 16, K = 256, dsub = 8 1182 / 425, 1184 / 846, 1418 /
// 1272; M = 16, K = 64, dsub = 4 467 / 268, 502 / 544, 692 / 815; M = 64, K = 256, dsub = 2 1418 /
// 770, 1425 / 1547, 1676 / 2310.
inline bool pq_per_query(int64_t nQ, int64_t nbq, int64_t tokens, int64_t M, int64_t dsub, int64_t lds) {
  const int64_t blocks = nQ * nbq;
  const bool wide = lds > 37 * 1024 && dsub >= 4 && dsub <= 16;
  const int64_t unit = (int64_t)(nQ == 2 || (wide && nQ <= 5) ? 1 : 2) << 17;
  if (blocks > 6 || tokens < unit * blocks * blocks) return false;
  if (nQ <= 3) return true;
  if (dsub == 2 && M > 16) return false;
  return nQ <= (dsub > 16 ? 4 : 5) || wide;
}

// ---- top-k of fp32 rows (tms_topk_kernel.h) -----------------------------------------
constexpr int kChunk = 4096;      // keys a tournament workgroup selects from
constexpr int kFilterMaxK = 128;  // the largest k with a bound on the k-th key taken first
constexpr int kShortRow = 1024;   // the largest last level of four waves
constexpr int kSpan = 1024;       // scores a span
constexpr int64_t kGroupMaxSpans = 16384;

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Keys per row after each tournament level, starting from n; stops when a row fits one chunk.
inline int64_t topk_level_sizes(int64_t n, int k, int64_t* sizes, int max_levels) {
  int64_t lv = 0;
  while (n > kChunk && lv < max_levels) {
    n = ceil_div(n, kChunk) * k;
    sizes[lv++] = n;
  }
  return lv;
}

// Bytes of the tournament's keys, two buffers in turn; group maxima take no more.
inline int64_t topk_workspace(int64_t nrows, int64_t n, int k) {
  int64_t sizes[64];
  const int64_t lv = topk_level_sizes(n, k, sizes, 64);
  int64_t a = 0, b = 0;  // even levels in a, odd in b
  for (int64_t i = 0; i < lv; i++) {
    if (i % 2 == 0) a = sizes[i] > a ? sizes[i] : a;
    else b = sizes[i] > b ? sizes[i] : b;
  }
  return (a + b) * nrows * (int64_t)sizeof(uint64_t);
}

// Keys that the group maxima's selections work on.
inline int64_t topk_group_keys(int k) { return k <= kFilterMaxK ? 4096 : 16384; }

// log2 of the lanes a group (of 4 scores each) of the group maxima, or 0 where the tournament
// takes the rows. k groups of a span's or of g scores have to fit the selection's keys, the
// spans its first stage, and the maxima the tournament's workspace (k < 8 and a few k above a
// power of two do not). Then, tournament / group maxima over Gaussian scores in replayed graphs:
//  * a row is one selection of 16 waves and up to 112 KiB of LDS, so 256 rows run at once.
//    More take turns and need longer rows, which the tournament spends more on: k = 10, 512 rows
//    x 5,000 17 / 15, 1,024 x 16,384 30 / 31, x 24,000 41 / 37, 4,096 x 8,192 55 / 98; k = 100,
//    512 x 8,192 20 / 24, x 16,384 28 / 24, 1,024 x 30,000 63 / 54, 4,096 x 8,192 75 / 162. Up to
//    256 rows of 5,000 to 40,000 scores: 10-30 / 8-17;
//  * the tournament is slow where its last chunk holds few scores, fewer than k above all: 1
//    row x 4,200, k = 10 16 / 8, k = 128 34 / 15; 512 x 8,300, k = 112 43 / 22;
//  * of few groups for their k the k-th maximum bounds little: 64 rows x 5,000, k = 128 15.8 /
//    17.3, x 6,500 16.0 / 14.1; 1 x 5,000, k = 200 17 / 51;
//  * above k = 128 the last selection has 16 keys a thread. The tournament's level of four waves
//    (chunks * k <= 1,024) is the better one but for a row a CU (k = 200: 16 x 16,384 21 / 23, 256 x
//    16,384 32 / 25, 16 x 24,000 24 / 19; k = 160, 1,024 x 16,384 62 / 68), above k = 320 any
//    single level on short rows (k = 360: 16 x 40,000 32 / 35, x 60,000 42 / 34), and above
//    400 there has to be much to save (k = 460: 16 x 100,000 44 / 47; k = 512: 64 x 100,000 61 /
//    52, 1 x 300,000 48 / 53, 1 x 1M 55 / 46).
// Sorted rows are the other way round up to about 100,000 scores (64 rows x 8,192, k = 100:
// 14 / 18): every score of the k best groups reaches the bound.
inline int topk_group_lanes(int64_t nrows, int64_t n, int k) {
  const int64_t keys = topk_group_keys(k);
  if (n <= kChunk || k > keys / 32) return 0;
  const int64_t chunks = ceil_div(n, kChunk), tail = n % kChunk;
  if (k <= kFilterMaxK) {
    const bool thin = tail > 0 && (tail < k || (tail < 256 && (nrows <= 512 || k <= 64)));
    if (!thin) {
      if (k > 120 && n < (int64_t)47 * k) return 0;
      if (nrows > 512 && n < (k <= 64 && nrows <= 1024 ? 20000 : 28672)) return 0;
      if (nrows > 256 && k > 64 && n < (k <= 104 ? 16384 : 20000)) return 0;
    }
  } else {
    const bool round = nrows > 128 && nrows <= 256;  // about one row a CU
    if (n < (int64_t)64 * k) return 0;
    if (k > 176 ? !round && chunks * k <= kShortRow : nrows > 512 && chunks * k <= 640) return 0;
    if (k > 320 && !round && chunks * k <= kChunk && n < (int64_t)110 * k) return 0;
    const bool thin = chunks * k > kChunk && chunks * k % kChunk < k;
    if (k > 400 && !thin && n < (1 << 19) && nrows * n < ((int64_t)1 << 22)) return 0;
  }
  int lg = 3;
  // the largest group of which k fit, with twice k groups in the row
  while (lg < 6 && ((int64_t)8 << lg) * k <= keys && n >= 2 * ((int64_t)8 << lg) * k) lg++;
  const int64_t spans = ceil_div(n, kSpan), per = kSpan >> (lg + 2);
  const bool direct = spans * per <= keys;
  if (!direct && (spans > kGroupMaxSpans || per * k > keys || spans < k)) return 0;
  const int64_t need = nrows * spans * (per + (direct ? 0 : 1)) * (int64_t)sizeof(uint32_t);
  return need <= topk_workspace(nrows, n, k) ? lg : 0;
}

}  // namespace tms
