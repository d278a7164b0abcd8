// Batched queries over PQ codes: the shared-tile kernel with the codebook gather as its
// tile source (subvectors of 8 dimensions and more; tms_batched_pq_small.hip: 2 and 4).
#include "tms_batched_kernel.h"

namespace tms {

int run_pq_batched_small(const BatchedArgs& a, int64_t nQ, int64_t dsub, int dtype, size_t lds, hipStream_t st);

// Entry used by tms_pq.hip: fixed-length documents of uint8 codes, the codebook (d * K
// elements, at most 64 KiB) copied to LDS by each workgroup. Shapes as the single-query
// MFMA PQ kernel's.
int run_pq_batched(const void* Q, int64_t nQ, int64_t nq, const void* codebook, int64_t M, int64_t K, int64_t dsub,
                   int dtype, const uint8_t* codes, int64_t B, int64_t nd, float* out, hipStream_t st) {
  BatchedArgs a;
  memset(&a, 0, sizeof(a));
  a.Q = (const uint8_t*)Q;
  a.D = codes;
  a.codebook = (const uint8_t*)codebook;
  a.out = out;
  a.B = B;
  a.T = B * nd;
  a.nd = nd;
  a.nq = (int32_t)nq;
  a.nbq = (int32_t)((nq + 31) / 32);
  a.d = (int32_t)(M * dsub);
  a.M = (int32_t)M;
  a.K = (int32_t)K;
  const size_t lds = (size_t)a.d * K * 2;
  switch (dsub) {
    case 8: return batched_run<PqTiles<8>>(a, nQ, nd, dtype, lds, st);
    case 16: return batched_run<PqTiles<16>>(a, nQ, nd, dtype, lds, st);
    case 32: return batched_run<PqTiles<32>>(a, nQ, nd, dtype, lds, st);
    default: return run_pq_batched_small(a, nQ, dsub, dtype, lds, st);
  }
}

}  // namespace tms
