// C names for the rules of tms_rules.h (tests/rules.py).
#include "tms_rules.h"

extern "C" int dense_split_waves(int64_t B, int64_t tiles, size_t lds, int nqb, int ks_reg) {
  return tms::dense_split_waves(B, tiles, lds, nqb, ks_reg);
}
extern "C" int topk_group_lanes(int64_t nrows, int64_t n, int k) { return tms::topk_group_lanes(nrows, n, k); }
extern "C" int64_t topk_workspace(int64_t nrows, int64_t n, int k) { return tms::topk_workspace(nrows, n, k); }
extern "C" int pq_per_query(int64_t nQ, int64_t nbq, int64_t tokens, int64_t M, int64_t dsub, int64_t lds) {
  return tms::pq_per_query(nQ, nbq, tokens, M, dsub, lds);
}
