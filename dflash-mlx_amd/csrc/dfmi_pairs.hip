// Builds the pair tables (dfmi_pairs.h): dfmi_sb_pairs, dfmi_moe_pairs, and
// the tables the matrix-core kernel reads, in every call beyond 32 rows.
#include <algorithm>

#include "dfmi_core.h"
#include "dfmi_pairs.h"

namespace dfmi {

// A workgroup transposes 256 / P table columns x 8 P groups through LDS: a
// lane reads 8 groups of one row (16 bytes of each array), and writes four
// columns of a group's row (16 bytes) where VEC says that every row starts on
// a 16-byte boundary; else element by element.  Bound by memory, small tables
// by the launch: 34816 rows x 80 groups (22 MB read and written) 7.3 us, 5120
// x 80 2.8 us, 256 experts of 2 x 512 x 32 15.9 us (67 MB) and 2048 x 8 8.8 us.
template <int P, bool VEC>
__global__ __launch_bounds__(256) void pairs_kernel(PairArgs a) {
  constexpr int COLS = 256 / P, LD = COLS + 4;
  __shared__ __align__(16) uint32_t tile[8 * P * LD];
  const int nb = blockIdx.x, tid = threadIdx.x, G = a.G;
  int i = 0;
#pragma unroll
  for (int k = 1; k < kPairSegs; ++k)
    if (k < a.nseg && nb >= a.seg[k].blk0) i = k;
  const PairSeg g = a.seg[i];
  const bool two = g.s2 != nullptr;
  const int ntc = two ? 2 * g.N : g.N;
  const int c0 = (nb - g.blk0) * COLS, g0 = blockIdx.y * 8 * P;
  const int64_t e = blockIdx.z;
  {
    const int r = tid / P, p = tid % P, c = c0 + r, gr = g0 + 8 * p;
    uint32_t v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = 0;
    if (c < ntc && gr < G) {
      const bool up = two && (c & 32);
      const int n = two ? 32 * (c >> 6) + (c & 31) : c;
      const uint16_t* s = (up ? g.s2 : g.s) + (e * g.N + n) * G + gr;
      const uint16_t* b = (up ? g.b2 : g.b) + (e * g.N + n) * G + gr;
      if constexpr (VEC) {
        const u32x4 sv = *reinterpret_cast<const u32x4*>(s), bv = *reinterpret_cast<const u32x4*>(b);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[2 * j] = __builtin_amdgcn_perm(bv[j], sv[j], 0x05040100u);
          v[2 * j + 1] = __builtin_amdgcn_perm(bv[j], sv[j], 0x07060302u);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (gr + j < G) v[j] = (uint32_t)s[j] | ((uint32_t)b[j] << 16);
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) tile[(8 * p + j) * LD + r] = v[j];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int q = tid + 256 * k, gi = q / (COLS / 4), c = q % (COLS / 4) * 4;
    if (g0 + gi >= G || c0 + c >= ntc) continue;
    const u32x4 v = *reinterpret_cast<const u32x4*>(&tile[gi * LD + c]);
    uint32_t* out = g.t + (e * G + g0 + gi) * ntc + c0 + c;
    if constexpr (VEC) {
      *reinterpret_cast<u32x4*>(out) = v;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (c0 + c + j < ntc) out[j] = v[j];
    }
  }
}

template <int P>
static void pairs_launch_p(PairArgs& a, int64_t E, bool vec, hipStream_t st) {
  int64_t blocks = 0;
  for (int i = 0; i < a.nseg; ++i) {
    a.seg[i].blk0 = (int)blocks;
    const int64_t ntc = (a.seg[i].s2 ? 2 : 1) * (int64_t)a.seg[i].N;
    blocks += (ntc + 256 / P - 1) / (256 / P);
  }
  const dim3 grid((unsigned)blocks, (unsigned)((a.G + 8 * P - 1) / (8 * P)), (unsigned)E);
  if (vec) hipLaunchKernelGGL((pairs_kernel<P, true>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((pairs_kernel<P, false>), grid, dim3(256), 0, st, a);
}

int pairs_launch(PairArgs& a, int64_t E, hipStream_t st, const char* what) {
  bool vec = a.G % 8 == 0;
  for (int i = 0; i < a.nseg; ++i) {
    const PairSeg& g = a.seg[i];
    vec = vec && aligned16(g.s) && aligned16(g.b) && aligned16(g.s2) && aligned16(g.b2) &&
          aligned16(g.t) && g.N % 4 == 0;
  }
  // as many groups per workgroup as there are, at most 64 bytes of a row (256
  // x 2048 rows of 8 groups: P = 1 8.8 us, 4 10.3; 34816 rows of 80 groups: P
  // = 1 8.8, 4 7.3, 8 7.6)
  if (a.G <= 8) pairs_launch_p<1>(a, E, vec, st);
  else if (a.G <= 16) pairs_launch_p<2>(a, E, vec, st);
  else pairs_launch_p<4>(a, E, vec, st);
  return check_launch(what);
}

}  // namespace dfmi
