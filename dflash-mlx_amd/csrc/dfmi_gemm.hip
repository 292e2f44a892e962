// Planning and launch of qmm_gemm_kernel (dfmi_gemm.h).
#include "dfmi_gemm.h"

#include <algorithm>

namespace dfmi {

// The tiles, and the time of one 128-k step of a workgroup, alone on its CU
// and per workgroup with the CU full (us, measured on MI355X at gs 64, 4-bit,
// bf16): what the plan chooses by.
struct GemmCfg {
  int bm, bn;
  double alone, full;
};
constexpr GemmCfg kGemmCfgs[] = {
    {64, 256, 1.20, 1.25},
    {96, 128, 1.15, 0.90},
    {32, 128, 0.59, 0.45},
};
constexpr int kNumGemmCfgs = 3;
constexpr size_t kGemmWsOffset = 65536;  // the streaming kernels' counters come first
constexpr size_t kGemmMaxPartials = (size_t)64 << 20;

struct GemmPlan {
  int cfg, kp, tiles_m, tiles_n;
  size_t partials;  // bytes
};

// The tile and K split with the least estimated time.  A launch costs about
// 4.5 us before and after its steps; a split writes and reads its partial
// tiles (about 3.5 TB/s) and launches the sum (2.5 us).  M = 77 on 5120 x
// 17408: 96 x 128 in 3 splits 37 us, unsplit 51; M = 512 on 5120 x 5120: 64 x
// 256 in 3 splits 45.6 us, unsplit 55.
static GemmPlan gemm_plan(int64_t M, int64_t K, int64_t N, size_t max_partials) {
  const int steps = (int)((K + kGemmK - 1) / kGemmK);
  GemmPlan best{};
  double best_t = 0;
  for (int c = 0; c < kNumGemmCfgs; ++c) {
    const GemmCfg& g = kGemmCfgs[c];
    const int64_t tm = (M + g.bm - 1) / g.bm, tn = (N + g.bn - 1) / g.bn, tiles = tm * tn;
    if (tiles >= (1ll << 31) / 64) continue;
    for (int kp = 1; kp <= 16 && 2 * kp <= std::max(steps, 2); ++kp) {
      const size_t bytes = kp > 1 ? (size_t)tiles * kp * g.bm * g.bn * 4u : 0;
      if (bytes > max_partials) break;
      const int64_t per_cu = (tiles * kp + 255) / 256;
      const int s = (steps + kp - 1) / kp;
      double t = 4.5 + s * (per_cu == 1 ? g.alone : per_cu * g.full);
      if (kp > 1) t += 2.5 + 2.0 * (double)bytes / 3.5e6;
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

// More rows than the streaming kernels take; 32-bit byte offsets within a
// tile's rows and the pair table.
bool gemm_shape(int64_t M, int64_t K, int64_t N, int gs) {
  return M > 32 && K < (1ll << 23) && (K / gs) * N * 4 <= 0xFFFFFFFFll &&
         ((M + 31) / 32) * ((N + 127) / 128) < (1ll << 24);
}

size_t gemm_workspace_bytes(int64_t M, int64_t K, int64_t N, int gs) {
  return kGemmWsOffset + table_bytes(K, N, gs) + gemm_plan(M, K, N, kGemmMaxPartials).partials;
}

int gemm_launch(const void* x, int x_dtype, const uint32_t* w, const void* scales,
                const void* biases, const uint32_t* pairs, int64_t pair_stride, void* y,
                int64_t M, int64_t K, int64_t N, int gs, int bits, void* workspace,
                size_t workspace_bytes, hipStream_t st) {
  char* ws = static_cast<char*>(workspace);
  size_t left = ws && workspace_bytes > kGemmWsOffset && aligned16(ws)
                    ? workspace_bytes - kGemmWsOffset : 0;
  ws += kGemmWsOffset;
  if (!pairs) {
    // the table into the workspace, for this call
    const size_t need = table_bytes(K, N, gs);
    if (left < need) return kGemmNotTaken;
    uint32_t* t = reinterpret_cast<uint32_t*>(ws);
    const int rc = dfmi_sb_pairs(scales, biases, x_dtype, N, K / gs, t, st);
    if (rc != DFMI_OK) return rc;
    pairs = t;
    pair_stride = N;
    ws += need;
    left -= need;
  }
  const GemmPlan p = gemm_plan(M, K, N, std::min(left, kGemmMaxPartials));
  GemmArgs a{};
  a.x = static_cast<const uint16_t*>(x);
  a.w = w;
  a.t = pairs;
  a.y = static_cast<uint16_t*>(y);
  a.partials = reinterpret_cast<float*>(ws);
  a.M = (int)M;
  a.K = (int)K;
  a.N = (int)N;
  a.tn = (uint32_t)(pair_stride ? pair_stride : N);
  a.steps = (int)((K + kGemmK - 1) / kGemmK);
  a.tiles_m = p.tiles_m;
  a.tiles_n = p.tiles_n;
  a.kp = p.kp;
  a.vec = aligned16(y) && N % 8 == 0;
  if (x_dtype == DFMI_BF16)
    bits == 4 ? gemm_launch_bf16_4(p.cfg, gs, a, st) : gemm_launch_bf16_8(p.cfg, gs, a, st);
  else
    bits == 4 ? gemm_launch_f16_4(p.cfg, gs, a, st) : gemm_launch_f16_8(p.cfg, gs, a, st);
  return check_launch("dfmi_qmm_affine (gemm)");
}

}  // namespace dfmi
