// Row-wise top-k: host entry points tms_topk and tms_topk_workspace_size, and the level
// launches that tms_topk_noalloc (tms_topk_noalloc.hip) shares; the selection kernel is in
// tms_topk_kernel.h.
#include <string.h>

#include "tms_topk_host.h"
#include "tms_topk_kernel.h"

namespace tms {

int64_t topk_workspace_bytes(int64_t nrows, int64_t n, int k) { return topk_workspace(nrows, n, k); }

}  // namespace tms

using namespace tms;

extern "C" {

int64_t tms_topk_workspace_size(int64_t nrows, int64_t n, int64_t k) {
  if (nrows <= 0 || n <= 0 || k <= 0 || k > kMaxK || k > n) return 0;
  return topk_workspace_bytes(nrows, n, (int)k);
}

int tms_topk(const float* scores, int64_t nrows, int64_t n, int64_t k, void* workspace, int64_t workspace_bytes_,
             float* out_values, int64_t* out_indices, void* stream) {
  const char* fn = "tms_topk";
  int rc = topk_checks(fn, scores, nrows, n, k, out_values, out_indices);
  if (rc != TMS_OK || nrows == 0 || k == 0) return rc;
  const int64_t need = topk_workspace_bytes(nrows, n, (int)k);
  if (need > 0 && (!workspace || workspace_bytes_ < need))
    return fail(TMS_ERR_INVALID, "%s: workspace of %lld bytes needed, got %lld", fn, (long long)need,
                (long long)workspace_bytes_);
  return topk_run(scores, nrows, n, k, workspace, out_values, out_indices, (hipStream_t)stream);
}

}  // extern "C"

namespace tms {

int topk_checks(const char* fn, const float* scores, int64_t nrows, int64_t n, int64_t k, const float* out_values,
                const int64_t* out_indices) {
  if (nrows < 0 || n < 0 || k < 0) return fail(TMS_ERR_INVALID, "%s: negative size", fn);
  if (k > n) return fail(TMS_ERR_INVALID, "%s: k=%lld exceeds the row length %lld", fn, (long long)k, (long long)n);
  if (k > kMaxK) return fail(TMS_ERR_UNSUPPORTED, "%s: k=%lld > %d is not supported", fn, (long long)k, kMaxK);
  if (n > 0xffffffffLL) return fail(TMS_ERR_UNSUPPORTED, "%s: rows longer than 2^32 - 1 are not supported", fn);
  if (nrows > 65535) return fail(TMS_ERR_UNSUPPORTED, "%s: more than 65535 rows per call", fn);
  if (nrows == 0 || k == 0) return TMS_OK;
  if (!scores || !out_values || !out_indices) return fail(TMS_ERR_INVALID, "%s: NULL pointer", fn);
  return TMS_OK;
}

template <int CH1, int CHS>
static void group_last(int64_t nrows, hipStream_t st, const float* scores, int64_t n, int64_t spans, int lg,
                       const uint32_t* groups, const uint32_t* spans_in, float* out_values, int64_t* out_indices, int k) {
  hipLaunchKernelGGL((topk_group_last_kernel<CH1, CHS>), dim3((unsigned)nrows), dim3(kLastThreads), 0, st, scores, n,
                     spans, lg, groups, spans_in, out_values, out_indices, k);
}

static int group_run(const float* scores, int64_t nrows, int64_t n, int k, int lg, uint32_t* ws, float* out_values,
                     int64_t* out_indices, hipStream_t st) {
  const int64_t keys = topk_group_keys(k);
  const int64_t spans = ceil_div(n, kSpan), per = kSpan >> (lg + 2), total = nrows * spans;
  uint32_t* groups = ws;
  uint32_t* spans_out = spans * per <= keys ? nullptr : ws + total * per;
  // one span a wave while that leaves the chip room (2,048 workgroups), else up to four
  int64_t per_row = ceil_div(spans, kGroupWaves);
  if (per_row * nrows > 2048) per_row = ceil_div(spans, kGroupWaves * (per_row * nrows > 8192 ? 4 : 2));
  const dim3 grid((unsigned)per_row, (unsigned)nrows);
  switch (lg) {
    case 3: hipLaunchKernelGGL(topk_group_max_kernel<3>, grid, dim3(64 * kGroupWaves), 0, st, scores, n, spans, groups, spans_out); break;
    case 4: hipLaunchKernelGGL(topk_group_max_kernel<4>, grid, dim3(64 * kGroupWaves), 0, st, scores, n, spans, groups, spans_out); break;
    case 5: hipLaunchKernelGGL(topk_group_max_kernel<5>, grid, dim3(64 * kGroupWaves), 0, st, scores, n, spans, groups, spans_out); break;
    default: hipLaunchKernelGGL(topk_group_max_kernel<6>, grid, dim3(64 * kGroupWaves), 0, st, scores, n, spans, groups, spans_out); break;
  }
  int rc = check_launch("topk_group_max_kernel");
  if (rc) return rc;
  const bool big = spans_out && spans > 4096, mid = spans_out && spans > 1024;
  if (keys == 4096) {
    if (big) group_last<16384, 4096>(nrows, st, scores, n, spans, lg, groups, spans_out, out_values, out_indices, k);
    else if (mid) group_last<4096, 4096>(nrows, st, scores, n, spans, lg, groups, spans_out, out_values, out_indices, k);
    else group_last<1024, 4096>(nrows, st, scores, n, spans, lg, groups, spans_out, out_values, out_indices, k);
  } else {
    if (big) group_last<16384, 16384>(nrows, st, scores, n, spans, lg, groups, spans_out, out_values, out_indices, k);
    else if (mid) group_last<4096, 16384>(nrows, st, scores, n, spans, lg, groups, spans_out, out_values, out_indices, k);
    else group_last<1024, 16384>(nrows, st, scores, n, spans, lg, groups, spans_out, out_values, out_indices, k);
  }
  return check_launch("topk_group_last_kernel");
}

// The levels of one call; `workspace` holds topk_workspace_bytes(nrows, n, k) bytes.
int topk_run(const float* scores, int64_t nrows, int64_t n, int64_t k, void* workspace, float* out_values,
             int64_t* out_indices, hipStream_t st) {
  if (const int lg = topk_group_lanes(nrows, n, (int)k))
    return group_run(scores, nrows, n, (int)k, lg, (uint32_t*)workspace, out_values, out_indices, st);
  int64_t sizes[64];
  const int64_t lv = topk_level_sizes(n, (int)k, sizes, 64);
  int64_t amax = 0;
  for (int64_t i = 0; i < lv; i += 2) amax = sizes[i] > amax ? sizes[i] : amax;
  uint64_t* bufs[2] = {(uint64_t*)workspace, (uint64_t*)workspace + amax * nrows};
  int64_t strides[2] = {amax, 0};
  for (int64_t i = 1; i < lv; i += 2) strides[1] = sizes[i] > strides[1] ? sizes[i] : strides[1];

  const dim3 last_block(kLastThreads), level_block(kLevelThreads);
  if (lv == 0) {
    if (n <= kShortRow)
      hipLaunchKernelGGL((topk_level_kernel<true, true, kShortThreads, kShortRow>), dim3(1, (unsigned)nrows),
                         dim3(kShortThreads), 0, st, scores, n, nullptr, n, n, nullptr, 0, out_values, out_indices,
                         (int)k);
    else
      hipLaunchKernelGGL((topk_level_kernel<true, true, kLastThreads>), dim3(1, (unsigned)nrows), last_block, 0, st,
                         scores, n, nullptr, n, n, nullptr, 0, out_values, out_indices, (int)k);
    return check_launch("topk_level_kernel");
  }
  // level 0: scores -> keys
  hipLaunchKernelGGL((topk_level_kernel<true, false, kLevelThreads>), dim3((unsigned)ceil_div(n, kChunk), (unsigned)nrows),
                     level_block, 0, st, scores, n, nullptr, n, n, bufs[0], strides[0], nullptr, nullptr, (int)k);
  int rc = check_launch("topk_level_kernel");
  if (rc) return rc;
  for (int64_t i = 1; i <= lv; i++) {
    const int64_t n_in = sizes[i - 1];
    const uint64_t* in = bufs[(i - 1) % 2];
    const int64_t in_stride = strides[(i - 1) % 2];
    if (i == lv && n_in <= kShortRow) {
      hipLaunchKernelGGL((topk_level_kernel<false, true, kShortThreads, kShortRow>), dim3(1, (unsigned)nrows),
                         dim3(kShortThreads), 0, st, scores, n, in, n_in, in_stride, nullptr, 0, out_values,
                         out_indices, (int)k);
    } else if (i == lv) {
      hipLaunchKernelGGL((topk_level_kernel<false, true, kLastThreads>), dim3(1, (unsigned)nrows), last_block, 0, st,
                         scores, n, in, n_in, in_stride, nullptr, 0, out_values, out_indices, (int)k);
    } else {
      hipLaunchKernelGGL((topk_level_kernel<false, false, kLevelThreads>),
                         dim3((unsigned)ceil_div(n_in, kChunk), (unsigned)nrows), level_block, 0, st, scores, n, in,
                         n_in, in_stride, bufs[i % 2], strides[i % 2], nullptr, nullptr, (int)k);
    }
    rc = check_launch("topk_level_kernel");
    if (rc) return rc;
  }
  return TMS_OK;
}

}  // namespace tms
