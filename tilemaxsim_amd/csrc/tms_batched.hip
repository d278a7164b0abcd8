// Batched queries over fp16 / bf16 documents: the shared-tile kernel (tms_batched_kernel.h)
// with the rows as they are as its tile source, and the entry of every dense batched call.
#include "tms_batched_kernel.h"

namespace tms {

int run_batched_f32(const BatchedArgs& a, int64_t nQ, int64_t tokens_per_doc, hipStream_t st);  // tms_batched_f32.hip
int run_batched_q32(const BatchedArgs& a, int64_t nQ, int64_t tokens_per_doc, int dtype, hipStream_t st);

// Entry used by tms_dense.hip and run_stream: d in {32, 64, 96, 128}, 16-byte aligned Q and
// D, queries of at most 4 blocks (2 for fp32 queries; q32: fp32 queries against 16-bit
// rows). offsets null: documents of nd tokens back to back.
int run_varlen_batched(const void* Q, int64_t nQ, int64_t nq, int64_t d, const void* D, int64_t T,
                       const int64_t* offsets, int64_t nd, int64_t B, PadLen pad, int dtype, float* out,
                       hipStream_t st, bool q32) {
  BatchedArgs a;
  memset(&a, 0, sizeof(a));
  a.Q = (const uint8_t*)Q;
  a.D = (const uint8_t*)D;
  a.offsets = offsets;
  a.out = out;
  a.B = B;
  a.T = T;
  a.pad = pad;
  a.nd = nd;
  a.nq = (int32_t)nq;
  a.nbq = (int32_t)((nq + 31) / 32);
  a.d = (int32_t)d;
  const int64_t per_doc = B > 0 ? T / B : 1;
  if (dtype == TMS_DTYPE_F32) return run_batched_f32(a, nQ, per_doc, st);
  if (q32) return run_batched_q32(a, nQ, per_doc, dtype, st);
  return batched_run<DenseTiles>(a, nQ, per_doc, dtype, 0, st);
}

}  // namespace tms
