// Planning and launch of qmm_gemm_kernel (dfmi_gemm.h).
#include "dfmi_gemm.h"
#include "dfmi_pairs.h"

#include <algorithm>

namespace dfmi {

// The tiles, and what the plan chooses by, in us per 128-k step: `full`, a
// workgroup's share of a CU's time while whole rounds of 256 * slots of them
// follow each other (the next workgroups already run on the CU), and `alone`,
// the step of the last, partly filled round.  slots says how many workgroups
// a round puts on a CU, not how many the CU holds.
struct GemmCfg {
  int bm, bn, slots;
  double alone, full;
};
constexpr GemmCfg kGemmCfgs[] = {
    {64, 256, 1, 1.22, 0.80},
    {96, 128, 2, 1.74, 0.90},
    {32, 128, 1, 0.59, 0.365},
};
constexpr int kNumGemmCfgs = 3;
constexpr size_t kGemmWsOffset = 65536;  // the streaming kernels' counters come first
constexpr size_t kGemmMaxPartials = (size_t)64 << 20;

struct GemmPlan {
  int cfg, kp, tiles_m, tiles_n;
  size_t partials;  // bytes
};

// The tile and K split with the least estimated time: whole rounds of the CUs'
// slots at the full rate, the last round at the rate of its fill; a split adds
// the sum's launch (1.3 us) and 0.57 us per MB of partial tiles.  The figures
// were fitted to 3748 measured launches (six tiles, 1..12 splits, M 33..2000,
// eight K x N from 1024 x 512 to 17408 x 5120, MI355X, gs 64, 4-bit, bf16):
// what the rule picks is 1.2 % slower in the mean than the best of them all,
// 14 % at worst; 64 x 128, 32 x 256 and 128 x 256 tiles would add 0.9 %.
// Known limits: a single whole round is priced at `full` although its
// workgroups have no successors, so 256 of them are estimated below 255; and
// 8-bit weights, groups of 32 (which spill) and f16 take the same figures.
static GemmPlan gemm_plan(int64_t M, int64_t K, const int64_t* Ns, int nseg,
                          size_t max_partials) {
  const int steps = (int)((K + kGemmK - 1) / kGemmK);
  GemmPlan best{};
  double best_t = 0;
  for (int c = 0; c < kNumGemmCfgs; ++c) {
    const GemmCfg& g = kGemmCfgs[c];
    int64_t tm = (M + g.bm - 1) / g.bm, tn = 0;
    for (int i = 0; i < nseg; ++i) tn += (Ns[i] + g.bn - 1) / g.bn;
    const int64_t tiles = tm * tn;
    for (int kp = 1; kp <= 16 && 2 * kp <= std::max(steps, 2); ++kp) {
      const size_t bytes = kp > 1 ? (size_t)tiles * kp * g.bm * g.bn * 4u : 0;
      if (bytes > max_partials) break;
      const int64_t groups = tiles * kp, round = 256 * g.slots;
      double t = (double)(groups / round) * g.full * g.slots;
      const int64_t rem = groups % round;
      if (rem > 0)
        t += rem <= 256 ? g.alone
                        : g.alone + (g.full * g.slots - g.alone) * (double)(rem - 256) /
                                        (double)(round - 256);
      t *= (steps + kp - 1) / kp;
      if (kp > 1) t += 1.3 + 0.57e-6 * (double)bytes;
      if (best_t == 0 || t < best_t) {
        best_t = t;
        best = GemmPlan{c, kp, (int)tm, (int)tn, bytes};
      }
    }
  }
  return best;
}

static size_t table_bytes(int64_t K, int64_t N, int gs) {
  return round_up((size_t)(K / gs) * (size_t)N * 4u, 256);
}

// Bytes of a pair table a DMA may step through: lanes without a row read at
// kNoRow plus the step's offset, which stays past the table's end and below
// 2^32 only if the table is below 2^31.
static bool table_fits(int64_t K, int64_t cols, int gs) {
  return (K / gs) * cols * 4 < (1ll << 31);
}

// More rows than the streaming kernels take; 32-bit byte offsets within a
// tile's rows and the pair table.
bool gemm_shape(int64_t M, int64_t K, int64_t N, int gs) {
  return M > 32 && K < (1ll << 23) && table_fits(K, N, gs) &&
         ((M + 31) / 32) * ((N + 127) / 128) < (1ll << 24);
}

size_t gemm_workspace_bytes(int64_t M, int64_t K, int64_t N, int gs) {
  return kGemmWsOffset + table_bytes(K, N, gs) +
         gemm_plan(M, K, &N, 1, kGemmMaxPartials).partials;
}

size_t gemm_multi_workspace_bytes(int64_t M, int64_t K, const int64_t* Ns, int nseg, int gs) {
  size_t tables = 0;
  for (int i = 0; i < nseg; ++i) tables += table_bytes(K, Ns[i], gs);
  return kGemmWsOffset + tables + gemm_plan(M, K, Ns, nseg, kGemmMaxPartials).partials;
}

void gemm_plan_query(int64_t M, int64_t K, const int64_t* Ns, int nseg, int* rows, int* cols,
                     int* splits) {
  const GemmPlan p = gemm_plan(M, K, Ns, nseg, kGemmMaxPartials);
  *rows = kGemmCfgs[p.cfg].bm;
  *cols = kGemmCfgs[p.cfg].bn;
  *splits = p.kp;
}

// the planned launch of a whose matrices, table and rows are set
static int gemm_run(GemmArgs& a, int x_dtype, int gs, int bits, char* ws, size_t left,
                    hipStream_t st) {
  int64_t Ns[kGemmMaxSeg];
  bool vec = true;
  for (int i = 0; i < a.nseg; ++i) {
    Ns[i] = a.N[i];
    vec = vec && aligned16(a.y[i]) && a.N[i] % 8 == 0;
  }
  const GemmPlan p = gemm_plan(a.M, a.K, Ns, a.nseg, std::min(left, kGemmMaxPartials));
  const int bn = kGemmCfgs[p.cfg].bn;
  int tile = 0;
  for (int i = 0; i < a.nseg; ++i) {
    a.tile0[i] = tile;
    tile += (a.N[i] + bn - 1) / bn;
  }
  a.partials = reinterpret_cast<float*>(ws);
  a.steps = (a.K + kGemmK - 1) / kGemmK;
  a.tiles_m = p.tiles_m;
  a.tiles_n = p.tiles_n;
  a.kp = p.kp;
  a.vec = vec;
  if (x_dtype == DFMI_BF16)
    bits == 4 ? gemm_launch_bf16_4(p.cfg, gs, a, st) : gemm_launch_bf16_8(p.cfg, gs, a, st);
  else
    bits == 4 ? gemm_launch_f16_4(p.cfg, gs, a, st) : gemm_launch_f16_8(p.cfg, gs, a, st);
  return check_launch("dfmi_qmm_affine (gemm)");
}

// what of a caller's workspace is free for the tables and partial tiles
static size_t gemm_space(void* workspace, size_t bytes, char*& ws) {
  ws = static_cast<char*>(workspace) + kGemmWsOffset;
  return workspace && aligned16(workspace) && bytes > kGemmWsOffset ? bytes - kGemmWsOffset : 0;
}

int gemm_launch(const void* x, int x_dtype, const dfmi_qmm_segment* segs, int nseg,
                const uint32_t* fused, int64_t pair_stride, int64_t M, int64_t K, int gs,
                int bits, void* workspace, size_t workspace_bytes, hipStream_t st) {
  if (pair_stride && !table_fits(K, pair_stride, gs)) return kGemmNotTaken;
  // (tables, product and split sum pass data through the workspace)
  std::lock_guard<std::mutex> order(launch_order());
  char* ws;
  size_t left = gemm_space(workspace, workspace_bytes, ws);
  // matrices without a table: theirs into the workspace, for this call
  size_t need = 0;
  int64_t cols = 0;
  for (int i = 0; i < nseg; ++i) {
    if (!fused && !segs[i].sb_pairs) need += table_bytes(K, segs[i].N, gs);
    cols += segs[i].N;
  }
  if (left < need) return kGemmNotTaken;
  GemmArgs a{};
  a.x = static_cast<const uint16_t*>(x);
  a.nseg = nseg;
  a.M = (int)M;
  a.K = (int)K;
  PairArgs build{};
  build.G = (int)(K / gs);
  for (int i = 0; i < nseg; ++i) {
    const int64_t N = segs[i].N;
    a.w[i] = segs[i].w_q;
    a.y[i] = static_cast<uint16_t*>(segs[i].y);
    a.N[i] = (int)N;
    if (fused) {
      a.t[i] = fused;
      a.tn[i] = (uint32_t)cols;
      fused += N;
    } else if (segs[i].sb_pairs) {
      a.t[i] = segs[i].sb_pairs;
      a.tn[i] = (uint32_t)(pair_stride ? pair_stride : N);
    } else {
      uint32_t* t = reinterpret_cast<uint32_t*>(ws);
      build.seg[build.nseg++] = PairSeg{static_cast<const uint16_t*>(segs[i].scales),
                                        static_cast<const uint16_t*>(segs[i].biases),
                                        nullptr, nullptr, t, (int)N, 0};
      a.t[i] = t;
      a.tn[i] = (uint32_t)N;
      ws += table_bytes(K, N, gs);
      left -= table_bytes(K, N, gs);
    }
  }
  if (build.nseg > 0) {
    const int rc = pairs_launch(build, 1, st, "dfmi_qmm_affine (pair tables)");
    if (rc != DFMI_OK) return rc;
  }
  return gemm_run(a, x_dtype, gs, bits, ws, left, st);
}

}  // namespace dfmi
