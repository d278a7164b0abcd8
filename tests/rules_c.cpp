// C names for the rules of tms_rules.h (tests/rules.py).
#include "tms_rules.h"

extern "C" int dense_split_waves(int64_t B, int64_t tiles, size_t lds, int nqb, int ks_reg) {
  return tms::dense_split_waves(B, tiles, lds, nqb, ks_reg);
}
