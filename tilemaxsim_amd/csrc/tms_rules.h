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

}  // namespace tms
