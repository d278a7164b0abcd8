// Batched queries over PQ codes with subvectors of 2 and 4 dimensions: its own translation
// unit, so these instantiations build in parallel with tms_batched_pq.hip.
#include "tms_batched_kernel.h"

namespace tms {

int run_pq_batched_small(const BatchedArgs& a, int64_t nQ, int64_t dsub, int dtype, size_t lds, hipStream_t st) {
  if (dsub == 2) return batched_run<PqTiles<2>>(a, nQ, a.nd, dtype, lds, st);
  return batched_run<PqTiles<4>>(a, nQ, a.nd, dtype, lds, st);
}

}  // namespace tms
