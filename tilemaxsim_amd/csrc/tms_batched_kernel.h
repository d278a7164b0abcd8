// Batched queries: many query blocks share each document tile through LDS. A workgroup
// walks a run of at most 64 documents (document b is rows [offsets[b], offsets[b+1]) of D,
// or [b nd, (b+1) nd) for fixed-length documents) in 16-token tiles, every wave the same
// tiles; the last tile of a document repeats its last token, which cannot change a max. A
// wave holds NB query blocks (whole queries) in VGPRs and computes all NB, used or not.
// Wave w < KS loads k-step w of each tile (lane (r, g): chunk 4 w + g of token r, the MFMA
// A-operand layout) NS tiles ahead; step i writes tile i+1 to the LDS ring, passes one
// LDS-only barrier (the loads in flight are not waited for), reads tile i+1's fragments and
// scores tile i. The MFMA cluster runs at raised wave priority, so a wave that has its
// operands keeps the matrix pipe fed ahead of the other wave's bookkeeping; the running
// max takes two v_max3 per fragment and each document's reduction uses the row swaps and
// DPP. pad > 0 gives the zero-padding semantics of tms_maxsim_varlen_padded; invalid
// offsets score NaN.
//
// Workgroup forms. Bound by the matrix cores (a step's MFMA time is the blocks a SIMD's
// waves hold), so a pass should hold few unused blocks and keep two waves on each SIMD:
//  * W = 4 waves of NB = 1..4 blocks, two to four workgroups per CU, for up to 4 NB blocks;
//  * W = 8 waves, one workgroup per CU, above that: NBL blocks in each of waves 0-3 and NBX
//    in each of waves 4-7 (waves w and w + 4 share a SIMD), up to 4 (NBL + NBX) blocks.
// Calls of few documents take W = 8 for 5 to 16 blocks as well (batched_spread).
// 50,000 x 180 tokens, d = 128 fp16, for 4, 8, 16, 20, 24, 32 and 34 queries: 418, 583, 918,
// 1250, 1408, 1761 and 2160 us (1.34 PFLOP/s at 32), against 605, 656, 1136, 1670, 1750, 1848
// and 3523 with 8 waves of 1, 2 or 4 blocks for every pass.
#pragma once
#include <string.h>

#include "tms_common.h"
#include "tms_rules.h"

namespace tms {

template <int K>
struct RingSlotS {
  static constexpr int value = K;
};

constexpr int kMaxBlocksPerWave = 4;  // query blocks held in VGPRs per wave: 1 to 4

struct BatchedArgs {
  const uint8_t* Q;         // (nQ * nq, d)
  const uint8_t* D;         // (T, d) tokens, or (T, M) PQ codes
  const int64_t* offsets;   // (B + 1), or null: document b is rows [b * nd, (b + 1) * nd)
  const uint8_t* codebook;  // PQ: (M, K, dsub) elements of the input dtype
  float* out;               // (nQ, B)
  int64_t B, T, nd;
  PadLen pad;
  int32_t nq, nbq, blk0, blk_end, d, docs_per_wg, M, K;
  int32_t nblk_l, nblk_x;  // blocks of each wave 0-3 and of each wave 4-7 (whole queries)
};

// Tile sources. A loading wave fetches, per tile, the raw data of its lane's 8-dimension
// chunk c of token `row`; the source turns it into the MFMA A-operand fragment.
// Each tile chunk goes to the LDS ring as kParts 16-byte MFMA fragments: the fragment
// itself, or (fp32 rows) its bf16 hi and lo terms.
struct DenseTiles {  // fp16 / bf16 rows, stored to the ring as loaded
  static constexpr bool kDirect = true;
  static constexpr int kParts = 1;
  static constexpr bool kQ32 = false;  // queries of the rows' type
  typedef u32x4 Raw;
  __device__ static Raw load(const BatchedArgs& a, int64_t row, int c) {
    return *(const u32x4*)(a.D + row * a.d * 2 + 16 * c);
  }
  __device__ static u32x4 decode(const u32x4*, int, Raw raw, int) { return raw; }
  __device__ static void parts(const Raw& raw, u32x4 (&out)[1]) { out[0] = raw; }
};
// fp16 / bf16 rows scored against fp32 queries: each query element is split into hi + lo
// terms of the rows' type (fp16 after the token's power-of-two scale, split_f16) and a
// product takes two MFMAs, d*q_lo + d*q_hi, as in the per-query kernels: the query is
// never rounded to 16 bits.
struct DenseTilesQ32 : DenseTiles {
  static constexpr bool kQ32 = true;
};
// fp32 rows (and fp32 queries): every element split into bf16 hi + lo terms as it goes
// to the ring, a product formed from three bf16 MFMAs (lo*q_hi + hi*q_lo + hi*q_hi, the
// per-query fp32 kernel's order), as in tms_dense_kernel.h.
struct F32Tiles {
  static constexpr bool kDirect = true;
  static constexpr int kParts = 2;
  static constexpr bool kQ32 = true;
  typedef u32x8 Raw;
  __device__ static Raw load(const BatchedArgs& a, int64_t row, int c) {
    const u32x4* p = (const u32x4*)(a.D + row * a.d * 4 + 32 * c);
    const u32x4 x0 = p[0], x1 = p[1];
    return Raw{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
  }
  __device__ static void parts(const Raw& raw, u32x4 (&out)[2]) { split_bf16(raw, out[0], out[1]); }
};
// uint8 PQ codes (M per token), decoded through the codebook held in LDS: chunk c covers
// subspaces 8c / DSUB .. (8c + 7) / DSUB. Codes >= K are clamped into the table.
template <int DSUB>
struct PqTiles {
  static constexpr bool kDirect = false;
  static constexpr int kParts = 1;
  static constexpr bool kQ32 = false;
  typedef uint32_t Raw;
  __device__ static Raw load(const BatchedArgs& a, int64_t row, int c) {
    const uint8_t* p = a.D + row * a.M;
    if constexpr (DSUB == 8) return p[c];
    else if constexpr (DSUB == 4) return *(const uint16_t*)(p + 2 * c);
    else if constexpr (DSUB == 2) return *(const uint32_t*)(p + 4 * c);
    else return p[c / (DSUB / 8)];
  }
  __device__ static u32x4 decode(const u32x4* cb, int K, Raw raw, int c) {
    auto code = [&](int i) -> uint32_t {
      const uint32_t x = (raw >> (8 * i)) & 0xffu;
      return x < (uint32_t)K ? x : (uint32_t)K - 1u;
    };
    if constexpr (DSUB >= 8) {
      constexpr int P = DSUB / 8;  // 16-byte pieces per codeword
      return cb[((int64_t)(c / P) * K + code(0)) * P + c % P];
    } else if constexpr (DSUB == 4) {
      const uint2* cb8 = (const uint2*)cb;
      u32x4 v;
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const uint2 x = cb8[(int64_t)(2 * c + i) * K + code(i)];
        v[2 * i] = x.x;
        v[2 * i + 1] = x.y;
      }
      return v;
    } else {
      const uint32_t* cb4 = (const uint32_t*)cb;
      u32x4 v;
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = cb4[(int64_t)(4 * c + i) * K + code(i)];
      return v;
    }
  }
};

constexpr int kBatchedRing = 4;  // LDS ring slots and load lead, in tiles

template <class SRC>
using BatchedRing = u32x4[kBatchedRing][SRC::kParts][4][64];

// One wave's share of the workgroup: NB query blocks from my_blk0 on; LD waves also load.
template <int DT, int KS, int NB, bool LD, class SRC>
__device__ __forceinline__ void batched_body(const BatchedArgs& a, BatchedRing<SRC>& ring, const u32x4* cb,
                                             int wid, int my_blk0, int my_nblk) {
  constexpr int NS = kBatchedRing;
  constexpr int NP = SRC::kParts;
  constexpr bool SPLIT = NP == 2;        // fp32 rows and queries: DT is the MFMA type, bf16
  constexpr bool QLO = SRC::kQ32;        // fp32 queries: every query fragment has a lo term
  constexpr bool QSCALE = QLO && !SPLIT && DT == TMS_DTYPE_F16;  // fp16 terms of a scaled token
  static_assert(!SPLIT || DT == TMS_DTYPE_BF16, "split fp32 terms are bf16");
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const float NEG_INF = -__builtin_inff();
  const int64_t b_begin = wave_uniform((int64_t)blockIdx.x * a.docs_per_wg);
  const int64_t b_end = (b_begin + a.docs_per_wg < a.B) ? b_begin + a.docs_per_wg : a.B;
  const int64_t ndocs = b_end - b_begin;  // >= 1: the host launches no empty workgroup

  u32x4 qf[NB][KS][2];
  u32x4 qfl[QLO ? NB : 1][QLO ? KS : 1][2];  // fp32 queries: the lo terms
  float qinv[QSCALE ? NB : 1][2];           // QSCALE: 1 / the token's scale (a power of two)
  bool qv[NB][2];
#pragma unroll
  for (int j = 0; j < NB; j++)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int jb = my_blk0 + j;
      const int qi = jb / a.nbq;
      const int tok = (jb - qi * a.nbq) * 32 + 16 * h + r;
      qv[j][h] = j < my_nblk && tok < a.nq;
      const int64_t row = qv[j][h] ? (int64_t)qi * a.nq + tok : 0;
      if constexpr (QLO) {
        u32x8 raw[KS];
        float am = 0.f;
#pragma unroll
        for (int s = 0; s < KS; s++) {
          const u32x4* p = (const u32x4*)(a.Q + (row * a.d + 8 * (4 * s + g)) * 4);
          const u32x4 x0 = p[0], x1 = p[1];
          raw[s] = qv[j][h] ? u32x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]}
                            : u32x8{0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
          if constexpr (QSCALE) am = fmaxf(am, absmax8(raw[s]));
        }
        float sc = 1.f;
        if constexpr (QSCALE) {  // the token's chunks sit in lanes r, r+16, r+32, r+48
          am = fmaxf(am, __shfl_xor(am, 16));
          am = fmaxf(am, __shfl_xor(am, 32));
          sc = pow2_scale(am, qinv[j][h]);
        }
#pragma unroll
        for (int s = 0; s < KS; s++) {
          if constexpr (QSCALE) split_f16(raw[s], sc, qf[j][s][h], qfl[j][s][h]);
          else split_bf16(raw[s], qf[j][s][h], qfl[j][s][h]);
        }
      } else {
#pragma unroll
        for (int s = 0; s < KS; s++) {
          const u32x4 v = *(const u32x4*)(a.Q + (row * a.d + 8 * (4 * s + g)) * 2);
          qf[j][s][h] = qv[j][h] ? v : u32x4{0u, 0u, 0u, 0u};
        }
      }
    }

  // lane j holds document b_begin + j's first row and length (-1: invalid offsets)
  const int64_t pad = pad_part(a.pad, lane);
  int64_t dbase = 0;
  int32_t dlen = -1;
  if (lane < ndocs) {
    const int64_t b = b_begin + lane;
    const int64_t s0 = a.offsets ? a.offsets[b] : b * a.nd, e0 = a.offsets ? a.offsets[b + 1] : (b + 1) * a.nd;
    if (s0 >= 0 && e0 >= s0 && e0 <= a.T && e0 - s0 <= 0x7fffffff) {
      dbase = s0;
      dlen = (int32_t)(e0 - s0);
    }
  }
  if (refused(pad)) dlen = -1;
  const int64_t pad_len = pad_length(a.pad, pad);
  float pend[NB];  // lane j: scores of document b_begin + j
#pragma unroll
  for (int j = 0; j < NB; j++) pend[j] = NEG_INF;

  struct Cur {
    int64_t b, base;
    int32_t len, t0;
  };
  auto bounds = [&](int64_t b, int64_t& base) -> int32_t {
    const int j = (int)(b - b_begin);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)dbase, j);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)((uint64_t)dbase >> 32), j);
    base = (int64_t)(((uint64_t)hi << 32) | lo);
    return __builtin_amdgcn_readlane(dlen, j);
  };
  // First document at or after b with a token; with `record`, the empty or invalid ones
  // passed on the way get their scores. Past the end the cursor keeps its last tile.
  auto seek = [&](Cur& c, int64_t b, bool record) {
    for (; b < b_end; b++) {
      int64_t base = 0;
      const int32_t len = bounds(b, base);
      if (len > 0) {
        c.b = b;
        c.base = base;
        c.len = len;
        c.t0 = 0;
        return;
      }
      if (record) {  // invalid offsets (len < 0): the final store writes NaN for the lane
        const float v = pad_len > 0 ? 0.f : NEG_INF;
#pragma unroll
        for (int j = 0; j < NB; j++) pend[j] = lane == (int)(b - b_begin) ? v : pend[j];
      }
    }
    c.b = b_end;
  };
  auto advance = [&](Cur& c, bool record) {
    if (c.b >= b_end) return;
    c.t0 += 16;
    if (c.t0 >= c.len) seek(c, c.b + 1, record);
  };

  Cur wc, wl;  // scoring (tile i), loads (tile i + NS)
  wc.b = b_end;
  wc.base = 0;
  wc.len = 1;
  wc.t0 = 0;
  seek(wc, b_begin, true);

  // Loading and non-loading waves are separate instantiations, so each copy's loads are
  // straight-line code whose outstanding count the compiler tracks exactly.
  auto pipeline = [&]() {
    wl = wc;
    const int chunk = 4 * (LD ? wid : 0) + g;
    typedef typename SRC::Raw Raw;
    auto load = [&]() -> Raw {
      Raw v{};
      if constexpr (LD) {
        int32_t t = wl.t0 + r;
        if (t > wl.len - 1) t = wl.len - 1;
        v = SRC::load(a, wl.base + t, chunk);
      }
      advance(wl, false);
      return v;
    };
    auto sync = [&]() {  // LDS-only fence: the loads in flight are not waited for
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    // Direct sources store tile i+1 from its load slot at step i; decoding sources decode
    // tile i+2 at step i into `ahead` (the LDS gathers overlap the step) and store it a
    // step later.
    Raw stg[NS];
    u32x4 ahead = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int t = 0; t < NS; t++) stg[t] = load();
    auto put = [&](int slot, const Raw& raw) {  // a direct source's tile to a ring slot
      u32x4 pv[NP];
      if constexpr (SRC::kDirect) SRC::parts(raw, pv);
#pragma unroll
      for (int p = 0; p < NP; p++) ring[slot][p][wid][lane] = pv[p];
    };
    if constexpr (LD) {
      if constexpr (SRC::kDirect) {
        put(0, stg[0]);
      } else {
        ring[0][0][wid][lane] = SRC::decode(cb, a.K, stg[0], chunk);
        ahead = SRC::decode(cb, a.K, stg[1], chunk);
      }
    }
    sync();
    u32x4 frag[2][NP][KS];
#pragma unroll
    for (int p = 0; p < NP; p++)
#pragma unroll
      for (int s = 0; s < KS; s++) frag[0][p][s] = ring[0][p][s][lane];
    float rmax[NB][2];
#pragma unroll
    for (int j = 0; j < NB; j++) rmax[j][0] = rmax[j][1] = NEG_INF;

    DocEnd<NB, QSCALE> doc_end;
    doc_end.init(qv, qinv, lane);

    auto step = [&](auto slot) -> bool {
      constexpr int i = decltype(slot)::value;  // step index mod NS
      constexpr int s1 = (i + 1) % NS;
      constexpr int f = i & 1;
      stg[i] = load();  // tile i + NS (stg[i] was tile i, in the ring since the last step)
      if constexpr (LD) {
        if constexpr (SRC::kDirect) {
          put(s1, stg[s1]);  // tile i+1
        } else {
          ring[s1][0][wid][lane] = ahead;                            // tile i+1
          ahead = SRC::decode(cb, a.K, stg[(i + 2) % NS], chunk);  // tile i+2
        }
      }
      sync();
#pragma unroll
      for (int p = 0; p < NP; p++)
#pragma unroll
        for (int s = 0; s < KS; s++) frag[f ^ 1][p][s] = ring[s1][p][s][lane];
      const u32x4(&t)[KS] = frag[f][0];
      const u32x4(&tl)[KS] = frag[f][NP - 1];  // SPLIT: the lo terms
      f32x4 acc[NB][2];
#pragma unroll
      for (int j = 0; j < NB; j++) acc[j][0] = acc[j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int s = 0; s < KS; s++)
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
          for (int h = 0; h < 2; h++) {
            if constexpr (SPLIT) acc[j][h] = mfma16x16x32<DT>(tl[s], qf[j][s][h], acc[j][h]);
            if constexpr (QLO) acc[j][h] = mfma16x16x32<DT>(t[s], qfl[j][s][h], acc[j][h]);
            acc[j][h] = mfma16x16x32<DT>(t[s], qf[j][s][h], acc[j][h]);
          }
      __builtin_amdgcn_s_setprio(0);
#pragma unroll
      for (int j = 0; j < NB; j++)
#pragma unroll
        for (int h = 0; h < 2; h++)
          rmax[j][h] = fmaxf(fmaxf(fmaxf(fmaxf(rmax[j][h], acc[j][h][0]), acc[j][h][1]), acc[j][h][2]), acc[j][h][3]);
      if (wc.t0 + 16 >= wc.len) {  // document wc.b ends with this tile
        const bool padded = wc.len < pad_len;
        doc_end.finish(rmax, padded, lane, (int)(wc.b - b_begin), pend);
      }
      advance(wc, true);
      return wc.b >= b_end;
    };
    while (true) {
      if (step(RingSlotS<0>{})) break;
      if (step(RingSlotS<1>{})) break;
      if (step(RingSlotS<2>{})) break;
      if (step(RingSlotS<3>{})) break;
    }
  };
  if (wc.b < b_end) pipeline();

  // coalesced store: lane i writes document b_begin + i for each of the wave's queries
  if (my_nblk > 0 && lane < ndocs) {
    const int64_t b = b_begin + lane;
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < NB; j++) {
      if (j >= my_nblk) break;
      const int jb = my_blk0 + j;
      const int qi = jb / a.nbq;
      s += pend[j];
      if (j == my_nblk - 1 || (jb + 1) / a.nbq != qi) {  // the query's last block
        float* o = a.out + (int64_t)qi * a.B + b;
        if (dlen < 0) store_nan_score(o);  // invalid offsets
        else *o = s;
        s = 0.f;
      }
    }
  }
}

// Waves per SIMD the registers are budgeted for: four, three or two at one, two or more
// blocks per wave (at d = 128 98, 142 and 184-230 VGPRs), fewer with lo terms.
template <class SRC>
constexpr int batched_min_waves(int W, int NB) {
  if (W == 8 || SRC::kParts == 2) return 2;
  const int n = NB + (SRC::kQ32 ? NB : 0);
  return n == 1 ? 4 : (n == 2 ? 3 : 2);
}

template <int DT, int KS, int NBL, int NBX, int W, class SRC>
__global__ void __launch_bounds__(64 * W, batched_min_waves<SRC>(W, NBX)) batched_tile_kernel(BatchedArgs a) {
  static_assert(W == 8 || NBL == NBX, "waves 0-3 only");
  __shared__ BatchedRing<SRC> ring;
  extern __shared__ u32x4 cb[];  // PQ codebook
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if constexpr (!SRC::kDirect) {  // codebook -> LDS (d * K elements, a multiple of 16 bytes)
    const int n16 = a.d * a.K * 2 / 16;
    for (int i = threadIdx.x; i < n16; i += 64 * W) cb[i] = ((const u32x4*)a.codebook)[i];
    __syncthreads();
  }
  const int my_blk0 = a.blk0 + (wid < 4 ? wid * a.nblk_l : 4 * a.nblk_l + (wid - 4) * a.nblk_x);
  int my_nblk = a.blk_end - my_blk0;  // <= 0 for a wave with no query
  const int most = wid < 4 ? a.nblk_l : a.nblk_x;
  if (my_nblk > most) my_nblk = most;
  if (wid < KS) batched_body<DT, KS, NBL, true, SRC>(a, ring, cb, wid, my_blk0, my_nblk);
  else if (W == 4 || wid < 4) batched_body<DT, KS, NBL, false, SRC>(a, ring, cb, wid, my_blk0, my_nblk);
  else batched_body<DT, KS, NBX, false, SRC>(a, ring, cb, wid, my_blk0, my_nblk);
}

// The workgroup forms, in the order of their step time; the host takes the first that
// holds a pass's blocks. NBL, NBX: blocks per wave of waves 0-3 and 4-7 (W = 4: equal).
struct BatchedForm {
  int W, NBL, NBX;
};
constexpr BatchedForm kBatchedForms[] = {{4, 1, 1}, {4, 2, 2}, {4, 3, 3}, {4, 4, 4}, {8, 2, 3}, {8, 3, 3}, {8, 3, 4}, {8, 4, 4}};
constexpr BatchedForm kBatchedFormsQ32[] = {{4, 1, 1}, {4, 2, 2}, {8, 1, 2}, {8, 2, 2}};  // twice the registers a block
// For calls of few documents (batched_spread), the passes of 5 to 16 blocks.
constexpr BatchedForm kBatchedSpreadForms[] = {{8, 1, 1}, {8, 2, 2}};

// Blocks a form holds when every query takes nbq blocks (a wave holds whole queries).
static inline int64_t form_blocks(const BatchedForm& f, int nbq) {
  return 4 * (int64_t)(f.NBL / nbq * nbq) + (f.W == 8 ? 4 * (int64_t)(f.NBX / nbq * nbq) : 0);
}

template <int DT, int NBL, int NBX, int W, class SRC>
static int batched_ks(const BatchedArgs& a, int64_t grid, size_t lds, hipStream_t st) {
  const dim3 blk(64 * W), g((unsigned)grid);
  switch (a.d / 32) {
    case 1: hipLaunchKernelGGL((batched_tile_kernel<DT, 1, NBL, NBX, W, SRC>), g, blk, lds, st, a); break;
    case 2: hipLaunchKernelGGL((batched_tile_kernel<DT, 2, NBL, NBX, W, SRC>), g, blk, lds, st, a); break;
    case 3: hipLaunchKernelGGL((batched_tile_kernel<DT, 3, NBL, NBX, W, SRC>), g, blk, lds, st, a); break;
    default: hipLaunchKernelGGL((batched_tile_kernel<DT, 4, NBL, NBX, W, SRC>), g, blk, lds, st, a); break;
  }
  return check_launch("batched_tile_kernel");
}
// Form f of the list (Q32's for fp32 queries), or spread form -1 - f.
template <int DT, class SRC>
static int batched_form(int f, const BatchedArgs& a, int64_t grid, size_t lds, hipStream_t st) {
  if constexpr (SRC::kDirect) {
    if (f == -1) return batched_ks<DT, 1, 1, 8, SRC>(a, grid, lds, st);
    if (f == -2) return batched_ks<DT, 2, 2, 8, SRC>(a, grid, lds, st);
  }
  if constexpr (SRC::kQ32) {
    switch (f) {
      case 0: return batched_ks<DT, 1, 1, 4, SRC>(a, grid, lds, st);
      case 1: return batched_ks<DT, 2, 2, 4, SRC>(a, grid, lds, st);
      case 2: return batched_ks<DT, 1, 2, 8, SRC>(a, grid, lds, st);
      default: return batched_ks<DT, 2, 2, 8, SRC>(a, grid, lds, st);
    }
  } else {
    switch (f) {
      case 0: return batched_ks<DT, 1, 1, 4, SRC>(a, grid, lds, st);
      case 1: return batched_ks<DT, 2, 2, 4, SRC>(a, grid, lds, st);
      case 2: return batched_ks<DT, 3, 3, 4, SRC>(a, grid, lds, st);
      case 3: return batched_ks<DT, 4, 4, 4, SRC>(a, grid, lds, st);
      case 4: return batched_ks<DT, 2, 3, 8, SRC>(a, grid, lds, st);
      case 5: return batched_ks<DT, 3, 3, 8, SRC>(a, grid, lds, st);
      case 6: return batched_ks<DT, 3, 4, 8, SRC>(a, grid, lds, st);
      default: return batched_ks<DT, 4, 4, 8, SRC>(a, grid, lds, st);
    }
  }
}

// Documents per workgroup (at most 64, one lane each). `slots` workgroups run at once; a
// workgroup's start-up (its queries from L2, the pipeline's fill) costs about
// kBatchedStartSteps tile steps. Fixed lengths: the count whose rounds of workgroups take
// the fewest steps. Variable lengths: the last workgroup to finish starts late by up to
// one workgroup's work, so the count balances that against the start-ups.
// (32 queries over 1,700 x 71 tokens: 34 us at 7 documents a workgroup, 90 at one.)
constexpr double kBatchedStartSteps = 8;
static inline int64_t batched_docs_per_wg(int64_t B, int64_t tokens_per_doc, bool varlen, int64_t slots) {
  const double tiles = (double)((tokens_per_doc + 15) / 16 > 0 ? (tokens_per_doc + 15) / 16 : 1);
  int64_t best = 1;
  double least = 0;
  for (int64_t n = 1; n <= 64; n++) {
    const double wgs = (double)((B + n - 1) / n), work = n * tiles;
    const double rounds = varlen ? wgs / slots : (double)(((int64_t)wgs + slots - 1) / slots);
    const double steps = rounds * (work + kBatchedStartSteps) + (varlen ? work : 0.0);
    if (n == 1 || steps < least) {
      best = n;
      least = steps;
    }
  }
  return best;
}

// The launches of one call: passes of the largest form while they fill it, then the rest in
// the smallest form that holds it (a pass of 32 blocks costs 1.0, of 16 0.52, of 4 0.24: 48
// queries measured 2.9 ms as 24 + 24 and 34 queries 2.5 as 17 + 17, above 32 + 16 and 32 + 2).
template <class SRC>
static int batched_run(BatchedArgs a, int64_t nQ, int64_t tokens_per_doc, int dtype, size_t lds, hipStream_t st) {
  const BatchedForm* forms = SRC::kQ32 ? kBatchedFormsQ32 : kBatchedForms;
  constexpr int nf = SRC::kQ32 ? (int)(sizeof(kBatchedFormsQ32) / sizeof(BatchedForm)) : (int)(sizeof(kBatchedForms) / sizeof(BatchedForm));
  const int64_t most = form_blocks(forms[nf - 1], a.nbq) / a.nbq;  // queries per pass
  for (int64_t q0 = 0; q0 < nQ; q0 += most) {
    const int64_t q1 = q0 + most < nQ ? q0 + most : nQ;
    const int64_t blocks = (q1 - q0) * a.nbq;
    int f = 0;
    while (f < nf - 1 && form_blocks(forms[f], a.nbq) < blocks) f++;
    BatchedForm form = forms[f];
    if (SRC::kDirect && batched_spread(a.B)) {
      for (int i = 0; i < 2; i++)
        if (form_blocks(kBatchedSpreadForms[i], a.nbq) >= blocks && kBatchedSpreadForms[i].NBX < form.NBX) {
          form = kBatchedSpreadForms[i];
          f = -1 - i;
          break;
        }
    }
    a.blk0 = (int32_t)(q0 * a.nbq);
    a.blk_end = (int32_t)(q1 * a.nbq);
    a.nblk_l = form.NBL / a.nbq * a.nbq;
    a.nblk_x = form.NBX / a.nbq * a.nbq;
    int64_t per_cu = form.W == 8 ? 1 : batched_min_waves<SRC>(4, form.NBX);
    const int64_t fit = (160 * 1024) / (int64_t)(sizeof(BatchedRing<SRC>) + lds);
    if (per_cu > fit) per_cu = fit;
    a.docs_per_wg = (int32_t)batched_docs_per_wg(a.B, tokens_per_doc, a.offsets != nullptr, 256 * per_cu);
    const int64_t grid = (a.B + a.docs_per_wg - 1) / a.docs_per_wg;
    if (grid > 0x7fffffff) return fail(TMS_ERR_UNSUPPORTED, "batched MaxSim: too many documents");
    int rc;
    if constexpr (SRC::kParts == 2) rc = batched_form<TMS_DTYPE_BF16, SRC>(f, a, grid, lds, st);  // fp32
    else if (dtype == TMS_DTYPE_F16) rc = batched_form<TMS_DTYPE_F16, SRC>(f, a, grid, lds, st);
    else rc = batched_form<TMS_DTYPE_BF16, SRC>(f, a, grid, lds, st);
    if (rc) return rc;
  }
  return TMS_OK;
}

}  // namespace tms
