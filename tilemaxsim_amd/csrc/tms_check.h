// What the checked entry points (tms_check.hip) share with the scoring ones.
#pragma once
#include "tms_common.h"

namespace tms {

// Variable-length scores of nQ queries (tms_dense.hip); out is (nQ, B).
int varlen_scores(const char* fn, const void* Qs, int64_t nQ, int64_t nq, int64_t d, const void* D_flat, int64_t T,
                  const int64_t* offsets, int64_t B, PadLen pad, int dtype, float* out, void* stream);
// Residual-compressed documents (tms_residual.hip): one query, or `batched`.
int residual_scores(const char* fn, const void* Qs, int64_t nQ, int64_t nq, int64_t d, const void* centroids,
                    int64_t ncent, const void* bucket_weights, int nbits, const int32_t* codes,
                    const uint8_t* residuals, int64_t total_tokens, const int64_t* offsets, int64_t ndocs,
                    const int64_t* pids, int64_t B, PadLen pad, bool batched, float* out, void* stream);
// Copies the thread's last error text.
void keep_error(char* to, int n);

}  // namespace tms
