// Routed experts with many pairs (prefill): the expert sort, the segment
// table, and moe_gemm_kernel, the 32 x 128 tile of qmm_gemm_kernel's main
// loop over gathered activation rows.
#include <algorithm>

#include "dfmi_gemm.h"
#include "dfmi_moe_gemm.h"

namespace dfmi {

// One workgroup: every wavefront counts the experts of its own stretch of
// pairs, the counts are summed over experts and wavefronts, and every
// wavefront places its stretch 64 pairs at a time, ranking equal experts
// among the lanes by ballots over the id's bits.  Bound by the latency of its
// few passes over LDS: 128 pairs and 4000 pairs of 256 experts take 4.5 and 9
// us, against the eight launches (argsort 19 and 38 us) they replace.
constexpr int kSortWaves = 8;

template <typename Id>
__global__ __launch_bounds__(64 * kSortWaves) void moe_sort_kernel(const Id* inds, int P, int E,
                                                                   int32_t* order, int32_t* rhs,
                                                                   int32_t* segs) {
  __shared__ uint32_t cnt[kSortWaves][kMoeSortMaxExperts + 1];
  __shared__ uint32_t wsum[kSortWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int per = ((P + kSortWaves - 1) / kSortWaves + 63) / 64 * 64;
  const int p0 = min(wave * per, P), p1 = min(p0 + per, P);
  for (int i = tid; i < kSortWaves * (kMoeSortMaxExperts + 1); i += 64 * kSortWaves)
    (&cnt[0][0])[i] = 0;
  __syncthreads();
  // bucket E: ids outside [0, E)
  auto bucket = [&](Id e) { return e >= 0 && e < (Id)E ? (int)e : E; };
  for (int p = p0 + lane; p < p1; p += 64) atomicAdd(&cnt[wave][bucket(inds[p])], 1u);
  __syncthreads();
  // two buckets per thread: pairs (low half) and segments (high half) of each
  uint32_t tot[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    uint32_t n = 0;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) n += cnt[w][2 * tid + b];
    tot[b] = n | ((n + kMoeSegRows - 1) / kMoeSegRows) << 16;
  }
  uint32_t scan = tot[0] + tot[1];
  const uint32_t own = scan;
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const uint32_t v = __shfl_up(scan, d);
    if (lane >= d) scan += v;
  }
  if (lane == 63) wsum[wave] = scan;
  __syncthreads();
  uint32_t base = scan - own;
  for (int w = 0; w < wave; ++w) base += wsum[w];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    uint32_t run = base & 0xFFFFu;
    int s = (int)(base >> 16);
    const uint32_t end = run + (tot[b] & 0xFFFFu);
    for (uint32_t q = run; q < end; q += kMoeSegRows) segs[1 + s++] = (int32_t)q;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
      const uint32_t n = cnt[w][2 * tid + b];
      cnt[w][2 * tid + b] = run;
      run += n;
    }
    base += tot[b];
    if (2 * tid + b == kMoeSortMaxExperts) {  // the last bucket: the totals
      segs[0] = (int32_t)(base >> 16);
      segs[1 + (base >> 16)] = P;
    }
  }
  __syncthreads();
  const int bits = 32 - __clz(E);  // bucket ids 0 .. E
  for (int g = p0; g < p1; g += 64) {
    const int p = g + lane;
    const bool in = p < p1;
    const Id raw = in ? inds[p] : 0;
    const int e = in ? bucket(raw) : 0;
    uint64_t same = __ballot(in);
    for (int b = 0; b < bits; ++b) {
      const uint64_t m = __ballot(in && ((e >> b) & 1));
      same &= ((e >> b) & 1) ? m : ~m;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    uint32_t at = 0;
    if (in) at = cnt[wave][e];
    __builtin_amdgcn_wave_barrier();
    if (in) {
      order[at + rank] = p;
      rhs[at + rank] = raw >= (Id)INT32_MIN && raw <= (Id)INT32_MAX ? (int32_t)raw : -1;
      if ((same >> lane) == 1ull) cnt[wave][e] = at + rank + 1;  // its highest lane
    }
    __builtin_amdgcn_wave_barrier();
  }
}

int moe_sort_launch(const void* inds, int inds_bytes, int P, int E, int32_t* order, int32_t* rhs,
                    int32_t* segs, hipStream_t st) {
  if (inds_bytes == 8)
    hipLaunchKernelGGL(moe_sort_kernel<int64_t>, dim3(1), dim3(64 * kSortWaves), 0, st,
                       static_cast<const int64_t*>(inds), P, E, order, rhs, segs);
  else
    hipLaunchKernelGGL(moe_sort_kernel<int32_t>, dim3(1), dim3(64 * kSortWaves), 0, st,
                       static_cast<const int32_t*>(inds), P, E, order, rhs, segs);
  return check_launch("dfmi_switch_glu (sort)");
}

// One workgroup, 1024 pairs at a time: where each pair's run began (a maximum
// scan of run starts), whether a segment starts there, and its number (a sum
// scan).
__global__ __launch_bounds__(1024) void moe_segments_kernel(const int32_t* rhs, int P,
                                                            int32_t* segs) {
  __shared__ int wmax[16], wsum[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int carry = 0, count = 0;  // start of the last run so far, segments so far
  for (int p0 = 0; p0 < P; p0 += 1024) {
    const int p = p0 + tid;
    const bool in = p < P;
    int run = in && (p == 0 || rhs[p] != rhs[p - 1]) ? p : 0;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
      const int v = __shfl_up(run, d);
      if (lane >= d) run = max(run, v);
    }
    if (lane == 63) wmax[wave] = run;
    __syncthreads();
    int before = carry, all = carry;
    for (int w = 0; w < 16; ++w) {
      if (w < wave) before = max(before, wmax[w]);
      all = max(all, wmax[w]);
    }
    run = max(run, before);
    const bool seg = in && (p - run) % kMoeSegRows == 0;
    const uint64_t m = __ballot(seg);
    if (lane == 0) wsum[wave] = __popcll(m);
    __syncthreads();
    int base = count;
    for (int w = 0; w < 16; ++w) {
      if (w < wave) base += wsum[w];
      count += wsum[w];
    }
    if (seg) segs[1 + base + __popcll(m & ((1ull << lane) - 1ull))] = p;
    carry = all;
    __syncthreads();
  }
  if (tid == 0) {
    segs[0] = count;
    segs[1 + count] = P;
  }
}

int moe_segments_launch(const int32_t* rhs, int P, int32_t* segs, hipStream_t st) {
  hipLaunchKernelGGL(moe_segments_kernel, dim3(1), dim3(1024), 0, st, rhs, P, segs);
  return check_launch("dfmi_gather_qmm (segments)");
}

// Units of (segment, 128 table columns): 128 weight rows of the expert, or
// for the SwiGLU 64 output columns, whose gate and up rows alternate 32 at a
// time, as the interleaved table does: wavefront w takes gate (even w) or up
// rows.  kGroups workgroups (three per CU: 37 KB of LDS, at most 168 VGPRs)
// take the units of a contiguous eighth each XCD, so a segment's units share
// its activations, and an expert's segments its weights, in one L2.
constexpr int kMoeGemmGroups = 768;

template <typename Tag, int GS, bool GLU>
__global__ __launch_bounds__(256, 3) void moe_gemm_kernel(MoeGemmArgs a) {
  using G = Gemm<Tag, GS, 4, 1, 1, 1, 4, true>;
  constexpr int OUTC = GLU ? 64 : 128;
  const int ntc = GLU ? 2 * a.N : a.N, ncb = a.N / OUTC, groups = a.K / GS;
  const int units = a.segs[0] * ncb;
  const int xcd = blockIdx.x & 7, per = units >> 3, rest = units & 7;
  const int u0 = xcd * per + min(xcd, rest), u1 = u0 + per + (xcd < rest ? 1 : 0);
  typename G::Ctx cx;
  cx.x = buffer_rsrc(a.x, (uint32_t)(a.x_rows * a.K * 2));
  const int tid = threadIdx.x, lane = tid & 63;
  for (int u = u0 + (int)(blockIdx.x >> 3); u < u1; u += kMoeGemmGroups / 8) {
    const int s = u / ncb, cb = u - s * ncb;
    const int p0 = a.segs[1 + s], rows = a.segs[2 + s] - p0;
    const int e = __builtin_amdgcn_readfirstlane(a.rhs[p0]);
    const bool bad_e = e < 0 || e >= a.E;
    const int ee = bad_e ? 0 : e;
    G::setup(cx, a.K, (uint32_t)ntc, cb * 128, 128);
    const int sel = GLU ? cx.wave & 1 : 0;
    // this wavefront's 32 weight rows; its DMA offsets count from the tile's
    // row 32 wave
    const int n0 = GLU ? cb * 64 + 32 * (cx.wave >> 1) : cb * 128 + 32 * cx.wave;
    const uint32_t wrow = cx.wstride;
    cx.w = buffer_rsrc(a.w[sel] + ((int64_t)ee * a.N + n0) * (wrow / 4), 32 * wrow);
    cx.wg -= (uint32_t)(32 * cx.wave) * wrow;
    cx.t = buffer_rsrc(a.t + (int64_t)ee * groups * ntc, (uint32_t)ntc * (uint32_t)groups * 4u);
#pragma unroll
    for (int i = 0; i < G::X_DMA; ++i) {
      const int r = (cx.wave * G::X_DMA + i) * 4 + lane / 16;
      int xr = -1;
      if (r < rows) {
        const int l = a.lhs ? a.lhs[p0 + r] : p0 + r;
        xr = a.div > 1 ? l / a.div : l;
      }
      cx.xr[i] = xr >= 0 && xr < a.x_rows ? (uint32_t)xr * cx.xstride : kNoRow;
    }
    typename G::Acc acc;
    acc.v[0][0] = G::zero16();
    G::run(cx, 0, a.K / kGemmK, acc);
    // outputs through LDS, rounded as the separate products would be
    stage_barrier<0>();
    const int col = cx.wn * 32 + (lane & 31);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = 8 * (r >> 2) + 4 * cx.h + (r & 3);
      *reinterpret_cast<uint16_t*>(dfmi_smem + m * G::YROW + col * 2) =
          Num<Tag>::f2h(acc.v[0][0][r]);
    }
    stage_barrier<0>();
    constexpr int PPR = OUTC / 8;
    for (int q = tid; q < rows * PPR; q += 256) {
      const int m = q / PPR, c = (q % PPR) * 8;
      const int id = a.lhs ? a.lhs[p0 + m] : p0 + m;
      const int xr = a.div > 1 ? id / a.div : id;
      const char* row = dfmi_smem + m * G::YROW;
      u32x4 v;
      if (bad_e || xr < 0 || xr >= a.x_rows) {
        v = u32x4{0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu};  // NaN in both dtypes
      } else if constexpr (GLU) {
        // columns c .. c + 7 of 64: gate at table column 64 (c / 32) + c % 32, up 32 on
        const u32x4 g = *reinterpret_cast<const u32x4*>(row + (2 * (c & 32) + (c & 31)) * 2);
        const u32x4 p = *reinterpret_cast<const u32x4*>(row + (2 * (c & 32) + 32 + (c & 31)) * 2);
#pragma unroll
        for (int k = 0; k < 4; ++k)
          v[k] = (uint32_t)Num<Tag>::f2h(silu_mul<Tag>(Num<Tag>::lo(g[k]), Num<Tag>::lo(p[k]))) |
                 ((uint32_t)Num<Tag>::f2h(silu_mul<Tag>(Num<Tag>::hi(g[k]), Num<Tag>::hi(p[k])))
                  << 16);
      } else {
        v = *reinterpret_cast<const u32x4*>(row + c * 2);
      }
      uint16_t* out = a.y + (a.div > 0 ? id : p0 + m) * (int64_t)a.N + cb * OUTC + c;
      if (a.vec) {
        *reinterpret_cast<u32x4*>(out) = v;
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) out[k] = (uint16_t)(v[k / 2] >> (16 * (k & 1)));
      }
    }
    stage_barrier<0>();  // the next unit's DMA lands where these outputs lay
  }
}

// Shapes with a pair table, whole units, 32-bit buffer offsets; more pairs
// than moe_stream_kernel's tables hold are its callers' condition.
bool moe_gemm_eligible(int64_t x_rows, int64_t P, int64_t K, int64_t N, int64_t E, int gs,
                       bool glu) {
  const int64_t ntc = glu ? 2 * N : N;
  return (gs == 64 || gs == 128) && K >= 256 && K % 256 == 0 && N > 0 &&
         N % (glu ? 64 : 128) == 0 && P >= 1 && x_rows * K * 2 < (1ll << 31) &&
         K < (1ll << 23) && (K / gs) * ntc * 4 < (1ll << 31) &&
         (P + 1) * (N / (glu ? 64 : 128)) < (1ll << 31);
}

template <typename Tag, int GS, bool GLU>
static void moe_gemm_t(const MoeGemmArgs& a, hipStream_t st) {
  using G = Gemm<Tag, GS, 4, 1, 1, 1, 4, true>;
  hipLaunchKernelGGL((moe_gemm_kernel<Tag, GS, GLU>), dim3(kMoeGemmGroups), dim3(G::THREADS),
                     G::LDS_BYTES, st, a);
}

template <typename Tag>
static void moe_gemm_tag(const MoeGemmArgs& a, int gs, bool glu, hipStream_t st) {
  if (gs == 64) glu ? moe_gemm_t<Tag, 64, true>(a, st) : moe_gemm_t<Tag, 64, false>(a, st);
  else glu ? moe_gemm_t<Tag, 128, true>(a, st) : moe_gemm_t<Tag, 128, false>(a, st);
}

int moe_gemm_launch(const MoeGemmArgs& a, int x_dtype, int gs, bool glu, hipStream_t st) {
  if (x_dtype == DFMI_BF16) moe_gemm_tag<BF16>(a, gs, glu, st);
  else moe_gemm_tag<F16>(a, gs, glu, st);
  return check_launch(glu ? "dfmi_gather_qmm_swiglu" : "dfmi_gather_qmm_affine");
}

}  // namespace dfmi
