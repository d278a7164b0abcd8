// Batched fp32 queries through the shared-tile kernel: against fp32 documents (every
// product from three bf16 MFMAs) and against fp16 / bf16 ones (two). Its own translation
// unit, so these instantiations build in parallel.
#include "tms_batched_kernel.h"

namespace tms {

int run_batched_f32(const BatchedArgs& a, int64_t nQ, int64_t tokens_per_doc, hipStream_t st) {
  return batched_run<F32Tiles>(a, nQ, tokens_per_doc, TMS_DTYPE_F32, 0, st);
}
int run_batched_q32(const BatchedArgs& a, int64_t nQ, int64_t tokens_per_doc, int dtype, hipStream_t st) {
  return batched_run<DenseTilesQ32>(a, nQ, tokens_per_doc, dtype, 0, st);
}

}  // namespace tms
