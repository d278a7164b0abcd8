// Dense MaxSim, d <= 128, query fragments in VGPRs, over fixed-length documents or
// documents at offsets: the streaming kernel with a control-flow shape the compiler's
// memory-counter tracking follows exactly.
//
// The general kernel (tms_dense.hip) walks documents with a cursor whose branches make
// the compiler drain every outstanding load before each tile. Here:
//  * a wave's tiles are a flat sequence; each document is padded to a multiple of
//    R = PFD + 1 tiles with clamped duplicates of its last token (a duplicate cannot
//    change a max), so every document starts at ring slot 0; with offsets, lane j holds
//    document j's first row and length and the walk reads them with readlane;
//  * the inner loop body is straight-line and unrolled R times: it issues the loads of
//    tile g + PFD (index clamped to the last tile, so the count never varies) and scores
//    tile g from the ring; the per-document reduction sits between inner loops;
//  * scores are staged in registers (lane i holds document i of the wave's run) and
//    stored once, coalesced, after the loop.
// Every wave streams its own documents with the same (one or two) query blocks. Batched
// queries use batched_tile_kernel (tms_batched_kernel.h), whose workgroups share tiles
// through LDS.
//
// Semantics as tms_dense.hip: fp32 accumulation, query rows past nq contribute 0, an
// empty document scores -inf.
#include <string.h>

#include "tms_common.h"

namespace tms {

struct StreamArgs {
  const uint8_t* Q;          // (nQ * nq, d)
  const uint8_t* D;          // fixed length: (B, nd, d); variable length: (T, d)
  const int64_t* offsets;    // variable length: (B + 1)
  const uint8_t* mask;       // masked: (B, nd), non-zero = real token
  float* out;                // (nQ, B)
  int64_t B, nd, T;
  PadLen pad;                // > 0 (variable length): score as if zero-padded to it
  int32_t nq, nbq;           // tokens per query, 32-token blocks per query
  int32_t blk0;              // first global query block of this launch
  int32_t blk_end;           // one past the last block of this launch
  int32_t nblk;              // blocks per wave
  int32_t d;                 // 32 * KS
  int32_t docs_per_wave;     // documents per wave; <= 64 (masked: times tiles per document <= 64)
  int32_t mask4;             // masked: nd % 4 == 0 and a 4-byte aligned mask (word loads)
};

// Validity bits of the 16 mask bytes of one tile (bit i: byte i non-zero), `n` >= 1 of them
// inside the document; the loads stay inside it. WORDS: n is a multiple of 4 and p is
// 4-byte aligned.
__device__ __forceinline__ uint32_t tile_mask_bits(const uint8_t* p, int32_t n, bool words) {
  uint32_t bits = 0;
  if (words) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = ((const uint32_t*)p)[4 * i < n ? i : 0];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      // 0x80 in every non-zero byte, then bits 0, 8, 16, 24 gathered into bits 24..27 of the
      // product (the sixteen partial products land on distinct bits)
      const uint32_t nz = ((((w[i] & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w[i]) & 0x80808080u) >> 7;
      bits |= ((nz * 0x01020408u) >> 24 & 0xfu) << (4 * i);
    }
  } else {
    uint8_t b[16];
#pragma unroll
    for (int i = 0; i < 16; i++) b[i] = p[i < n ? i : 0];
#pragma unroll
    for (int i = 0; i < 16; i++) bits |= (b[i] != 0 ? 1u : 0u) << i;
  }
  return n < 16 ? bits & ((1u << n) - 1u) : bits;
}

enum { ST_FIXED = 0, ST_VARLEN = 1, ST_MASKED = 2 };

// ST_MASKED: lane j * tiles + t holds the validity bits of tile t of document j, read once
// when the wave starts. The walk visits only tiles with a real token, and a masked-out row
// of such a tile reads the tile's first real row instead (a duplicate cannot change a max):
// masked tokens are neither fetched nor scored. A document without a real token takes R
// tiles of row 0 whose maxima are dropped. Bound by HBM on the real tokens: 20,000 x 180
// with a mean of 106 real tokens (0.55 GB) takes 91 us (6.0 TB/s of them), against 183 us
// for the general kernel, which fetches every token and drains its loads at each tile.
//
// ST_VARLEN: documents at offsets (T >= 1 rows). Lane j of a wave holds its document j's first
// row and length, which the walk reads with readlane, so the tile sequence stays
// straight-line as for fixed lengths. An empty document, or one with invalid offsets,
// takes R tiles of row 0 whose maxima are dropped: its score is -inf (0 when padded),
// or NaN for invalid offsets.
template <int DT, int KS, int NB, int PFD, int MODE>
__global__ void __launch_bounds__(256, 1) stream_maxsim_kernel(StreamArgs a) {
  constexpr bool VARLEN = MODE == ST_VARLEN, MASKED = MODE == ST_MASKED;
  constexpr int R = PFD + 1;
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int wid = threadIdx.x >> 6;
  const float NEG_INF = -__builtin_inff();

  const int my_blk0 = a.blk0;
  int my_nblk = a.blk_end - my_blk0;
  if (my_nblk > a.nblk) my_nblk = a.nblk;
  if (my_nblk <= 0) return;

  const int64_t unit = (int64_t)blockIdx.x * 4 + wid;
  const int64_t b_begin = unit * a.docs_per_wave;
  if (b_begin >= a.B) return;
  const int64_t b_end = (b_begin + a.docs_per_wave < a.B) ? b_begin + a.docs_per_wave : a.B;
  const int64_t ndocs = b_end - b_begin;

  // query fragments: block j, half h, step s -> token 16h + r of the block, chunk 4s + g
  auto q_valid = [&](int j, int h, int64_t& row) -> bool {
    const int jb = my_blk0 + j;
    const int qi = jb / a.nbq;
    const int tok = (jb - qi * a.nbq) * 32 + 16 * h + r;
    row = (int64_t)qi * a.nq + tok;
    return j < my_nblk && tok < a.nq;
  };
  u32x4 qf[NB][KS][2];
#pragma unroll
  for (int j = 0; j < NB; j++)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      int64_t row;
      const bool v = q_valid(j, h, row);
#pragma unroll
      for (int s = 0; s < KS; s++)
        qf[j][s][h] = v ? *(const u32x4*)(a.Q + (row * a.d + 8 * (4 * s + g)) * 2) : u32x4{0u, 0u, 0u, 0u};
    }

  // VARLEN: lane j holds document b_begin + j's first row (0 if it has no rows) and its
  // length (-1: invalid offsets).
  int64_t dbase = 0;
  int32_t dlen = 0;
  const int64_t pad = VARLEN ? pad_part(a.pad, lane) : 0;
  if constexpr (VARLEN) {
    dlen = -1;
    if (lane < ndocs) {
      const int64_t b = b_begin + lane;
      const int64_t s0 = a.offsets[b], e0 = a.offsets[b + 1];
      if (s0 >= 0 && e0 >= s0 && e0 <= a.T && e0 - s0 <= 0x7fffffff) {
        dlen = (int32_t)(e0 - s0);
        dbase = dlen > 0 ? s0 : 0;
      }
    }
    if (refused(pad)) {
      dlen = -1;
      dbase = 0;
    }
  }
  // MASKED: the bits of the lane's tile, and which of the wave's tiles hold a real token
  const int32_t mtiles = MASKED ? (int32_t)((a.nd + 15) / 16) : 0;  // tiles per document
  uint32_t mbits = 0;
  uint64_t mlive = 0;
  if constexpr (MASKED) {
    const int32_t t = lane % (mtiles > 0 ? mtiles : 1);
    if (lane < ndocs * mtiles)
      mbits = tile_mask_bits(a.mask + (b_begin + lane / mtiles) * a.nd + 16 * t, (int32_t)a.nd - 16 * t, a.mask4);
    mlive = __ballot(mbits != 0);
  }
  auto doc_live = [&](int64_t dd) -> uint64_t {  // MASKED: bit t: tile t holds a real token
    return (mlive >> (dd * mtiles)) & (~0ull >> (64 - mtiles));
  };
  const int64_t pad_len = VARLEN ? pad_length(a.pad, pad) : 0;
  auto doc_len = [&](int64_t dd) -> int64_t {
    if constexpr (VARLEN) return (int32_t)__builtin_amdgcn_readlane((uint32_t)dlen, (int)dd);
    else return a.nd;
  };
  auto doc_base = [&](int64_t dd) -> int64_t {
    if constexpr (VARLEN) {
      const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)dbase, (int)dd);
      const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)((uint64_t)dbase >> 32), (int)dd);
      return (int64_t)(((uint64_t)hi << 32) | lo);
    } else {
      return (b_begin + dd) * a.nd;
    }
  };
  // tiles of a document of `len` rows, padded to a multiple of R (at least R)
  auto doc_tiles = [&](int64_t len) -> int64_t {
    const int64_t t = len > 0 ? (len + 15) / 16 : 1;
    return (t + R - 1) / R * R;
  };
  auto live_tiles = [&](uint64_t live) -> int64_t {  // MASKED: the same of a document's tiles with a real token
    const int t = live != 0 ? __builtin_popcountll(live) : 1;
    return (t + R - 1) / R * R;
  };

  float pend[NB];
#pragma unroll
  for (int j = 0; j < NB; j++) pend[j] = NEG_INF;

  if (VARLEN || a.nd > 0) {
    const int64_t tpd = doc_tiles(a.nd);  // fixed length: tiles per document
    int64_t total;                        // tiles of the wave's documents
    if constexpr (VARLEN) {  // 64-bit: documents may overlap, each up to 2^31 rows
      int64_t n = lane < ndocs ? doc_tiles(dlen) : 0;
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) n += __shfl_xor(n, o);
      const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)n);
      const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)n >> 32));
      total = (int64_t)(((uint64_t)hi << 32) | lo);
    } else if constexpr (MASKED) {
      total = 0;
      for (int64_t dd = 0; dd < ndocs; dd++) total += live_tiles(doc_live(dd));
    } else {
      total = ndocs * tpd;
    }
    const int64_t row_bytes = (int64_t)a.d * 2;
    // LINES (rows of 128 or 256 bytes): each load covers whole 128-byte lines of eight rows
    // (line_frags); lane 16 g + 8 s + t reads bytes 64 s + 16 g of a line of row t or 8 + t.
    // Otherwise lane (r, g) reads chunk 4 s + g of row r, a quarter line per load.
    constexpr bool LINES = KS % 2 == 0;
    const int t8 = lane & 7;
    const uint8_t* base = a.D + (LINES ? (int64_t)(64 * ((lane >> 3) & 1) + 16 * g) : (int64_t)(8 * g) * 2);

    // Address of a token row of tile (document dd of the wave, tile t): row i of the
    // tile, clamped to the document's last row (row 0 for a document without rows).
    int64_t c_base = doc_base(0), c_len = doc_len(0);  // the prefetch cursor's document
    uint64_t c_rem = 0;  // MASKED: its tiles with a real token past the cursor
    uint32_t c_bits = 0;  // MASKED: the validity bits of the cursor's tile
    auto tile_ptr = [&](int64_t t, int i) -> const uint8_t* {
      if constexpr (MASKED) {
        const int first = __builtin_ctz(c_bits | 0x10000u) & 15;
        return base + (c_base + t * 16 + ((c_bits >> i) & 1u ? i : first)) * row_bytes;
      }
      int64_t tok = t * 16 + i;
      const int64_t last = c_len > 0 ? c_len - 1 : 0;
      if (tok > last) tok = last;
      return base + (c_base + tok) * row_bytes;
    };
    // Prefetch cursor: tile index pf (tile pt of document pd), saturating at the last tile
    // (the prefetches past the end re-read it, so each iteration issues KS loads).
    int64_t pd = 0, pt = 0, pf = 0, c_tiles = VARLEN ? doc_tiles(c_len) : tpd;
    int64_t c_left = 0;  // MASKED: tiles of the document from the cursor on, repeats included
    auto masked_doc = [&](uint64_t live) {
      c_left = live_tiles(live);
      pt = live != 0 ? __builtin_ctzll(live) : 0;
      c_rem = live & (live - 1);
    };
    auto masked_bits = [&]() { c_bits = __builtin_amdgcn_readlane(mbits, (int)(pd * mtiles + pt)); };
    if constexpr (MASKED) {
      masked_doc(doc_live(0));
      masked_bits();
    }
    auto pf_next = [&]() {
      const bool more = pf < total - 1;
      if constexpr (MASKED) {
        if (more) {  // uniform, and no load inside
          pf++;
          if (--c_left == 0) {
            pd++;
            masked_doc(doc_live(pd));
          } else if (c_rem != 0) {  // else: the last such tile again
            pt = __builtin_ctzll(c_rem);
            c_rem &= c_rem - 1;
          }
          c_base = (b_begin + pd) * a.nd;
          masked_bits();
        }
        return;
      }
      pf += more ? 1 : 0;
      pt += more ? 1 : 0;
      const bool wrap = pt == c_tiles;
      pt = wrap ? 0 : pt;
      pd += wrap ? 1 : 0;
      if constexpr (VARLEN) {  // pd < ndocs: the cursor stops at the last tile
        c_base = doc_base(pd);
        c_len = doc_len(pd);
        c_tiles = doc_tiles(c_len);
      } else {
        c_base = (b_begin + pd) * a.nd;
      }
    };

    u32x4 ring[R][KS];
    auto load = [&](u32x4 (&buf)[KS]) {
      if constexpr (LINES) {  // buf[2i], buf[2i+1]: line i of rows t and 8 + t
        const uint8_t* p0 = tile_ptr(pt, t8);
        const uint8_t* p1 = tile_ptr(pt, 8 + t8);
#pragma unroll
        for (int i = 0; i < KS / 2; i++) {
          buf[2 * i] = ld_stream<u32x4, true>(p0 + 128 * i);
          buf[2 * i + 1] = ld_stream<u32x4, true>(p1 + 128 * i);
        }
      } else {
        const uint8_t* p = tile_ptr(pt, r);
#pragma unroll
        for (int s = 0; s < KS; s++) buf[s] = ld_stream<u32x4, false>(p + 64 * s);
      }
    };
#pragma unroll
    for (int k = 0; k < PFD; k++) {
      load(ring[k]);
      pf_next();
    }

    float rmax[NB][2];
    auto score = [&](const u32x4 (&raw)[KS]) {
      u32x4 buf[KS];  // A-operand fragments: chunk 4 s + g of row r
      if constexpr (LINES) {
#pragma unroll
        for (int i = 0; i < KS / 2; i++) line_frags(raw[2 * i], raw[2 * i + 1], buf[2 * i], buf[2 * i + 1]);
      } else {
#pragma unroll
        for (int s = 0; s < KS; s++) buf[s] = raw[s];
      }
      f32x4 acc[NB][2];
#pragma unroll
      for (int j = 0; j < NB; j++) acc[j][0] = acc[j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; s++)
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
          for (int h = 0; h < 2; h++) acc[j][h] = mfma16x16x32<DT>(buf[s], qf[j][s][h], acc[j][h]);
#pragma unroll
      for (int j = 0; j < NB; j++)
#pragma unroll
        for (int h = 0; h < 2; h++)
          rmax[j][h] = fmaxf(rmax[j][h], fmaxf(fmaxf(acc[j][h][0], acc[j][h][1]), fmaxf(acc[j][h][2], acc[j][h][3])));
    };

    for (int64_t dd = 0; dd < ndocs; dd++) {
#pragma unroll
      for (int j = 0; j < NB; j++) rmax[j][0] = rmax[j][1] = NEG_INF;
      const int64_t len = doc_len(dd);
      const int64_t nt = VARLEN ? doc_tiles(len) : (MASKED ? live_tiles(doc_live(dd)) : tpd);
      for (int64_t t = 0; t < nt; t += R) {
#pragma unroll
        for (int k = 0; k < R; k++) {
          load(ring[(k + PFD) % R]);
          pf_next();
          score(ring[k]);
        }
      }
      // document done: max over the 64 rows of each column, sum over query tokens
      const bool padded = VARLEN && len < pad_len;  // zero padding adds dot products of 0
      float blk[NB];
#pragma unroll
      for (int j = 0; j < NB; j++) {
        float s = 0.f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
          float m = rmax[j][h];
          m = fmaxf(m, __shfl_xor(m, 16));
          m = fmaxf(m, __shfl_xor(m, 32));
          if (padded) m = fmaxf(m, 0.f);
          int64_t row;
          s += q_valid(j, h, row) ? m : 0.f;
        }
        s += __shfl_xor(s, 8);
        s += __shfl_xor(s, 4);
        s += __shfl_xor(s, 2);
        s += __shfl_xor(s, 1);
        if (MASKED && doc_live(dd) == 0) s = NEG_INF;  // no real token (the tiles read row 0)
        if (VARLEN && len <= 0) s = pad_len > 0 ? 0.f : NEG_INF;  // no rows (the tiles read row 0)
        blk[j] = s;
      }
      const bool mine = lane == (int)dd;
#pragma unroll
      for (int j = 0; j < NB; j++) pend[j] = mine ? blk[j] : pend[j];
    }
  }

  // coalesced store: lane i writes document b_begin + i, per query (blocks of one query
  // summed in order; a query that began in an earlier launch accumulates)
  if (lane < ndocs) {
    const int64_t b = b_begin + lane;
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < NB; j++) {
      if (j >= my_nblk) break;
      const int jb = my_blk0 + j;
      const int qi = jb / a.nbq;
      s += pend[j];
      if (j == my_nblk - 1 || (jb + 1) / a.nbq != qi) {
        float* o = a.out + (int64_t)qi * a.B + b;
        if (VARLEN && dlen < 0) store_nan_score(o);  // invalid offsets
        else *o = (qi * a.nbq < my_blk0) ? *o + s : s;
        s = 0.f;
      }
    }
  }
}

#ifndef TMS_STREAM_PFD
#define TMS_STREAM_PFD 2  // tiles in flight ahead of the one being scored (single-query path)
#endif
// Masked: one. A document's tiles with a real token are padded to a multiple of ahead + 1, and
// those repeats cost more than the second load in flight gains (20,000 x 180, 106 real: 91.3
// us a call against 93.1; 5,000, replayed: 32.9 against 34.7).
constexpr int kMaskedPFD = 1;
#ifndef TMS_STREAM_MIN_WAVES
#define TMS_STREAM_MIN_WAVES (256 * 16 * 2)  // fewer documents per wave below this many waves
#endif
#ifndef TMS_STREAM_TOKENS_PER_WAVE
#define TMS_STREAM_TOKENS_PER_WAVE 768  // document tokens one wave streams (rounded to whole documents)
#endif

template <int DT, int KS, int NB>
static int stream_launch(const StreamArgs& a, int64_t grid, hipStream_t st) {
  if (a.mask)
    hipLaunchKernelGGL((stream_maxsim_kernel<DT, KS, NB, kMaskedPFD, ST_MASKED>), dim3((unsigned)grid), dim3(256),
                       0, st, a);
  else if (a.offsets)
    hipLaunchKernelGGL((stream_maxsim_kernel<DT, KS, NB, TMS_STREAM_PFD, ST_VARLEN>), dim3((unsigned)grid), dim3(256),
                       0, st, a);
  else
    hipLaunchKernelGGL((stream_maxsim_kernel<DT, KS, NB, TMS_STREAM_PFD, ST_FIXED>), dim3((unsigned)grid), dim3(256),
                       0, st, a);
  return check_launch("stream_maxsim_kernel");
}

template <int DT, int NB>
static int stream_ks(const StreamArgs& a, int64_t grid, hipStream_t st) {
  switch (a.d / 32) {
    case 1: return stream_launch<DT, 1, NB>(a, grid, st);
    case 2: return stream_launch<DT, 2, NB>(a, grid, st);
    case 3: return stream_launch<DT, 3, NB>(a, grid, st);
    default: return stream_launch<DT, 4, NB>(a, grid, st);
  }
}

// Batched queries (tms_batched.hip).
int run_varlen_batched(const void* Q, int64_t nQ, int64_t nq, int64_t d, const void* D, int64_t T,
                       const int64_t* offsets, int64_t nd, int64_t B, PadLen pad, int dtype, float* out,
                       hipStream_t st, bool q32);

// Entry used by tms_dense.hip for d in {32, 64, 96, 128}, 16-byte aligned Q and D:
// fixed-length documents (offsets and mask null), padded ones with a (B, nd) token mask
// (1 <= nd <= kMaskedStreamMaxTokens), or documents at offsets into T >= 1 rows
// (pad > 0: scored as if zero-padded to that many tokens). nQ queries of nq tokens;
// out is (nQ, B).
int run_stream(const void* Q, int64_t nQ, int64_t nq, int64_t d, const void* D, int64_t B, int64_t nd,
               const int64_t* offsets, const uint8_t* mask, int64_t T, PadLen pad, int dtype, float* out,
               hipStream_t st) {
  StreamArgs a;
  memset(&a, 0, sizeof(a));
  a.Q = (const uint8_t*)Q;
  a.D = (const uint8_t*)D;
  a.offsets = offsets;
  a.mask = mask;
  a.mask4 = (nd % 4 == 0 && ((uintptr_t)mask & 3) == 0) ? 1 : 0;
  a.out = out;
  a.B = B;
  a.nd = offsets ? 0 : nd;
  a.T = T;
  a.pad = pad;
  a.nq = (int32_t)nq;
  a.nbq = (int32_t)((nq + 31) / 32);
  a.d = (int32_t)d;
  const int64_t nblocks = nQ * (int64_t)a.nbq;
  if (!offsets && !mask && a.nbq <= 4 && (nblocks >= 4 || nQ == 3))  // batched: documents at implicit offsets b * nd
    return run_varlen_batched(Q, nQ, nq, d, D, B * nd, nullptr, nd, B, PadLen{0, nullptr, 0, 0}, dtype, out, st, false);
  const int64_t hint = offsets ? (B > 0 ? T / B : 1) : nd;  // tokens per document
  int64_t dpw = hint > 0 ? TMS_STREAM_TOKENS_PER_WAVE / hint : 1;
  const int64_t min_waves = TMS_STREAM_MIN_WAVES;
  if (dpw > 1 && B / dpw < min_waves) dpw = B / min_waves;
  if (dpw < 1) dpw = 1;
  if (dpw > 64) dpw = 64;
  if (mask && nd > 0 && dpw > 64 / ((nd + 15) / 16)) dpw = 64 / ((nd + 15) / 16);  // one lane per tile
  a.docs_per_wave = (int32_t)dpw;
  const int64_t waves = (B + dpw - 1) / dpw;
  const int64_t grid = (waves + 3) / 4;
  for (int64_t b0 = 0; b0 < nblocks; b0 += 2) {  // two query blocks per pass over D
    a.blk0 = (int32_t)b0;
    a.blk_end = (int32_t)(nblocks - b0 < 2 ? nblocks : b0 + 2);
    a.nblk = a.blk_end - a.blk0;
    int rc;
    if (a.nblk == 2) {
      rc = dtype == TMS_DTYPE_F16 ? stream_ks<TMS_DTYPE_F16, 2>(a, grid, st)
                                  : stream_ks<TMS_DTYPE_BF16, 2>(a, grid, st);
    } else {
      rc = dtype == TMS_DTYPE_F16 ? stream_ks<TMS_DTYPE_F16, 1>(a, grid, st)
                                  : stream_ks<TMS_DTYPE_BF16, 1>(a, grid, st);
    }
    if (rc) return rc;
  }
  return TMS_OK;
}

}  // namespace tms
