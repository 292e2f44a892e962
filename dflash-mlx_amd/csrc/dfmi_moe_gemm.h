// Expert sort and the many-pairs gather (dfmi_moe_gemm.hip), called by the
// entry points of dfmi_moe.hip.
#pragma once

#include "dfmi_host.h"

namespace dfmi {

constexpr int kMoeSortMaxExperts = 1023;
constexpr int kMoeSegRows = 32;  // pairs per segment: the tile's rows

// Stable sort of pairs by expert (ids outside [0, E) last): order[i] = the
// pair at sorted position i, rhs[i] its expert id, and the segment table of
// the sorted pairs: segs[0] = count, segs[1 ..] their first positions, then P.
int moe_sort_launch(const void* inds, int inds_bytes, int P, int E, int32_t* order, int32_t* rhs,
                    int32_t* segs, hipStream_t st);
// The segment table of pairs in any order: runs of one expert id, cut every
// kMoeSegRows pairs.
int moe_segments_launch(const int32_t* rhs, int P, int32_t* segs, hipStream_t st);

struct MoeGemmArgs {
  const uint16_t* x;
  const uint32_t* w[2];  // the matmul's (or gate) weights, up weights (SwiGLU)
  const uint32_t* t;     // pair tables [E][K/GS][N], or [E][K/GS][2N] interleaved (SwiGLU)
  const int32_t *lhs, *rhs, *segs;
  uint16_t* y;
  int64_t x_rows;
  int P, K, N, E;
  int div;  // GatherArgs::div
  int vec;  // y rows start on 16-byte boundaries
};
bool moe_gemm_eligible(int64_t x_rows, int64_t P, int64_t K, int64_t N, int64_t E, int gs,
                       bool glu);
int moe_gemm_launch(const MoeGemmArgs& a, int x_dtype, int gs, bool glu, hipStream_t st);

}  // namespace dfmi
