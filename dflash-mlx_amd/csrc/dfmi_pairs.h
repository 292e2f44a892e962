// (scale, bias) pair tables: the one layout the streaming, matrix-core and
// routed-expert kernels read scales and biases from.
#pragma once

#include "dfmi_host.h"

namespace dfmi {

constexpr int kPairSegs = 4;

// One matrix: scales and biases [E][N][G] (16-bit values of either dtype) into
// t [E][G][N] = scale | bias << 16, or with a second set (s2, b2) into
// [E][G][2N], the sets 32 columns at a time (table column 64 (n / 32) + 32 set
// + n % 32).
struct PairSeg {
  const uint16_t *s, *b, *s2, *b2;
  uint32_t* t;
  int N, blk0;  // blk0: set by pairs_launch
};
struct PairArgs {
  PairSeg seg[kPairSegs];
  int nseg, G;
};
// All matrices (same G) in one launch.
int pairs_launch(PairArgs& a, int64_t E, hipStream_t st, const char* what);

}  // namespace dfmi
