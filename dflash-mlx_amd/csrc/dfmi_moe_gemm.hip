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
// among the lanes by ballots over the id's bits.  Bound by latency, so the
// ids are read eight to a lane at once.  128 and 4000 pairs of 256 experts
// take 3.4 and 8.6 us, against eight launches (argsort 19 and 38 us) before.
constexpr int kSortWaves = 16, kSortIds = 8;

template <typename Id>
__global__ __launch_bounds__(64 * kSortWaves) void moe_sort_kernel(const Id* inds, int P, int E,
                                                                   int32_t* order, int32_t* rhs,
                                                                   int32_t* segs) {
  // [wavefront][bucket] counts, then first positions; bucket E: ids outside [0, E)
  uint32_t* cnt = reinterpret_cast<uint32_t*>(dfmi_smem);
  __shared__ uint32_t wsum[kSortWaves];
  const int nb = E + 1;  // <= 1024: one bucket per thread
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int per = ((P + kSortWaves - 1) / kSortWaves + 63) / 64 * 64;
  const int p0 = min(wave * per, P), p1 = min(p0 + per, P);
  uint32_t* mine = cnt + wave * nb;
  Id ids[kSortIds];
  auto load = [&](int q) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kSortIds; ++i) {
      const int p = q + 64 * i + lane;
      ids[i] = p < p1 ? inds[p] : (Id)-1;
    }
  };
  auto bucket = [&](Id e) __attribute__((always_inline)) {
    return e >= 0 && e < (Id)E ? (int)e : E;
  };
  load(p0);
  for (int i = tid; i < kSortWaves * nb; i += 64 * kSortWaves) cnt[i] = 0;
  __syncthreads();
  for (int q = p0; q < p1; q += 64 * kSortIds) {
    if (q > p0) load(q);
#pragma unroll
    for (int i = 0; i < kSortIds; ++i)
      if (q + 64 * i + lane < p1) atomicAdd(&mine[bucket(ids[i])], 1u);
  }
  const bool again = p1 - p0 > 64 * kSortIds;  // the ids are not all in registers
  __syncthreads();
  // this thread's bucket: pairs (low half) and segments (high half)
  uint32_t n = 0;
  if (tid < nb) {
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) n += cnt[w * nb + tid];
  }
  const uint32_t tot = n | ((n + kMoeSegRows - 1) / kMoeSegRows) << 16;
  uint32_t scan = tot;
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const uint32_t v = __shfl_up(scan, d);
    if (lane >= d) scan += v;
  }
  if (lane == 63) wsum[wave] = scan;
  __syncthreads();
  uint32_t base = scan - tot;
  for (int w = 0; w < wave; ++w) base += wsum[w];
  if (tid < nb) {
    uint32_t run = base & 0xFFFFu;
    int s = (int)(base >> 16);
    for (uint32_t q = run; q < run + n; q += kMoeSegRows) segs[1 + s++] = (int32_t)q;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
      const uint32_t c = cnt[w * nb + tid];
      cnt[w * nb + tid] = run;
      run += c;
    }
    if (tid == E) {  // the last bucket: the totals
      segs[0] = s;
      segs[1 + s] = P;
    }
  }
  __syncthreads();
  const int bits = 32 - __clz(E);  // bucket ids 0 .. E
  for (int q = p0; q < p1; q += 64 * kSortIds) {
    if (again) load(q);
#pragma unroll
    for (int i = 0; i < kSortIds; ++i) {
      if (q + 64 * i >= p1) break;  // uniform
      const int p = q + 64 * i + lane;
      const bool in = p < p1;
      const int e = bucket(ids[i]);
      uint64_t same = __ballot(in);
      for (int b = 0; b < bits; ++b) {
        const uint64_t m = __ballot(in && ((e >> b) & 1));
        same &= ((e >> b) & 1) ? m : ~m;
      }
      const int rank = __popcll(same & ((1ull << lane) - 1ull));
      uint32_t at = 0;
      if (in) at = mine[e];
      __builtin_amdgcn_wave_barrier();
      if (in) {
        order[at + rank] = p;
        rhs[at + rank] = e < E ? e : -1;
        if ((same >> lane) == 1ull) mine[e] = at + rank + 1;  // its highest lane
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

int moe_sort_launch(const void* inds, int inds_bytes, int P, int E, int32_t* order, int32_t* rhs,
                    int32_t* segs, hipStream_t st) {
  const size_t lds = (size_t)kSortWaves * (E + 1) * 4;  // at most 64 KiB
  static const bool allowed = [] {  // (and the static words beside them)
    const int most = kSortWaves * (kMoeSortMaxExperts + 1) * 4;
    return hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_sort_kernel<int64_t>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, most) == hipSuccess &&
           hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_sort_kernel<int32_t>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, most) == hipSuccess;
  }();
  (void)allowed;  // a refusal shows as the launch's own error
  const dim3 block(64 * kSortWaves);
  if (inds_bytes == 8)
    hipLaunchKernelGGL(moe_sort_kernel<int64_t>, dim3(1), block, lds, st,
                       static_cast<const int64_t*>(inds), P, E, order, rhs, segs);
  else
    hipLaunchKernelGGL(moe_sort_kernel<int32_t>, dim3(1), block, lds, st,
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
// rows.  Three workgroups per CU (45 KB of LDS, 168 VGPRs and 24 bytes of
// spills per lane) take
// consecutive units, those of an XCD a contiguous eighth, so a segment's units
// share its activations, and an expert's segments its weights, in one L2.
//
// Bound by the weight stream and, at the down projection's four steps per
// unit, by each unit's latencies: the next unit's first stages are therefore
// requested as soon as the last step's reads are done, under the outputs
// (which leave through LDS of their own), and a segment's ids are read only
// where it changes.  500 tokens, top-8 of 256 experts, 2048 x 512:
// SwiGLU 85 us, down 54 us (with every unit on its own 84 and 62; the gathers
// that stream an expert once per 16 of its rows 239 and 103).
constexpr int kMoeGemmGroups = 768;

template <typename Tag, int GS>
struct MoeGemmLayout {
  using G = Gemm<Tag, GS, 4, 1, 1, 1, 4, true>;
  static constexpr int OUT = G::LDS_LOOP;                // the output tile
  static constexpr int IDS = OUT + G::BM * G::YROW;      // int[32]: pair (or row) ids
  static constexpr int BYTES = IDS + 4 * kMoeSegRows;
  static_assert(3 * BYTES <= 160 * 1024 && G::BM == kMoeSegRows, "three workgroups per CU");
};

template <typename Tag, int GS, bool GLU>
__global__ __launch_bounds__(256, 3) void moe_gemm_kernel(MoeGemmArgs a) {
  using LY = MoeGemmLayout<Tag, GS>;
  using G = typename LY::G;
  constexpr int OUTC = GLU ? 64 : 128;
  const int ntc = GLU ? 2 * a.N : a.N, ncb = a.N / OUTC, groups = a.K / GS;
  const int steps = a.K / kGemmK;
  const int units = a.segs[0] * ncb;
  const int xcd = blockIdx.x & 7, x0 = (int)((int64_t)xcd * units / 8);
  const int xn = (int)((int64_t)(xcd + 1) * units / 8) - x0;
  constexpr int PER_XCD = kMoeGemmGroups / 8;
  int u = x0 + (int)((int64_t)(blockIdx.x >> 3) * xn / PER_XCD);
  const int u1 = x0 + (int)((int64_t)((blockIdx.x >> 3) + 1) * xn / PER_XCD);
  if (u >= u1) return;  // uniform
  const int tid = threadIdx.x, lane = tid & 63;
  int* s_ids = reinterpret_cast<int*>(dfmi_smem + LY::IDS);
  typename G::Ctx cx;
  G::setup(cx, a.K, (uint32_t)ntc, 0, 128);
  cx.x = buffer_rsrc(a.x, (uint32_t)(a.x_rows * a.K * 2));
  const uint32_t tg0 = cx.tg;
  cx.wg -= (uint32_t)(32 * cx.wave) * cx.wstride;  // counted from the wavefront's own rows
  int s = u / ncb, cb = u - s * ncb;
  // a segment's rows and expert
  int p0 = 0, rows = 0, e = 0;
  auto segment = [&]() __attribute__((always_inline)) {
    p0 = a.segs[1 + s];
    rows = a.segs[2 + s] - p0;
    e = __builtin_amdgcn_readfirstlane(a.rhs[p0]);
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
  };
  // the unit's weights and pairs
  auto unit_buffers = [&]() __attribute__((always_inline)) {
    const int ee = e < 0 || e >= a.E ? 0 : e;
    const int n0 = GLU ? cb * 64 + 32 * (cx.wave >> 1) : cb * 128 + 32 * cx.wave;
    cx.w = buffer_rsrc(a.w[GLU ? cx.wave & 1 : 0] + ((int64_t)ee * a.N + n0) * (cx.wstride / 4),
                       32 * cx.wstride);
    cx.t = buffer_rsrc(a.t + (int64_t)ee * groups * ntc, (uint32_t)ntc * (uint32_t)groups * 4u);
    cx.tg = tg0 == kNoRow ? kNoRow : tg0 + (uint32_t)cb * 512u;
  };
  segment();
  unit_buffers();
  G::start(cx, 0, steps);
  for (bool fresh = true;; fresh = false) {
    // this unit's place, as the next one's is set up before its outputs
    const int up0 = p0, urows = rows, ucb = cb;
    const bool bad_e = e < 0 || e >= a.E;
    const bool more = u + 1 < u1;
    if (fresh || cb == 0) {  // a new segment's ids (read after run()'s barriers)
      if (tid < rows) s_ids[tid] = a.lhs ? a.lhs[p0 + tid] : p0 + tid;
    }
    typename G::Acc acc;
    acc.v[0][0] = G::zero16();
    G::run(cx, 0, steps, acc, [&] {
      if (!more) return;
      ++u;
      if (++cb == ncb) {
        cb = 0;
        ++s;
        segment();
      }
      unit_buffers();
      G::start(cx, 0, steps);
    });
    // outputs through LDS, rounded as the separate products would be
    const int col = cx.wn * 32 + (lane & 31);
    char* tile = dfmi_smem + LY::OUT;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = 8 * (r >> 2) + 4 * cx.h + (r & 3);
      *reinterpret_cast<uint16_t*>(tile + m * G::YROW + col * 2) =
          Num<Tag>::f2h(acc.v[0][0][r]);
    }
    stage_barrier<15>();
    constexpr int PPR = OUTC / 8;
    for (int q = tid; q < urows * PPR; q += 256) {
      const int m = q / PPR, c = (q % PPR) * 8;
      const int id = s_ids[m];
      const int xr = a.div > 1 ? id / a.div : id;
      const char* row = tile + m * G::YROW;
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
      uint16_t* out = a.y + (a.div > 0 ? id : up0 + m) * (int64_t)a.N + ucb * OUTC + c;
      if (a.vec) {
        *reinterpret_cast<u32x4*>(out) = v;
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) out[k] = (uint16_t)(v[k / 2] >> (16 * (k & 1)));
      }
    }
    if (!more) return;  // uniform
    stage_barrier<15>();  // the ids and the output tile may be written again
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
  using LY = MoeGemmLayout<Tag, GS>;
  hipLaunchKernelGGL((moe_gemm_kernel<Tag, GS, GLU>), dim3(kMoeGemmGroups),
                     dim3(LY::G::THREADS), LY::BYTES, st, a);
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
