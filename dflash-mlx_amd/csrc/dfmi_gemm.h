// Affine quantised matmul for many activation rows (prefill and wide batches):
// y[M,N] = x[M,K] . dequant(W)^T on the 32x32x16 matrix instructions.
//
// A workgroup of WM x WN wavefronts owns a tile of BM = 32 MT WM activation
// rows and BN = 32 NT WN weight rows; a wavefront takes 32 MT rows and 32 NT
// columns of it.  K advances in steps of 128: activations, packed weights and
// (scale, bias) pairs go to LDS by DMA, DEPTH steps ahead, one barrier per
// step.
//
// Arithmetic, per quantisation group g of a weight row (exact products, fp32
// sums, the group's scale applied to its fp32 sum):
//     acc += s_g * sum_{k in g} x_k q_k  +  b_g * X_g,   X_g = sum_{k in g} x_k
// Codes become 16-bit floats without an offset: a nibble in a byte is the fp8
// (e4m3) number q / 512 (codes 0..7 are its subnormals, 8..15 its first
// binade, one spacing), and v_cvt_scalef32_pk_{bf16,f16}_fp8 with scale 512
// turns two of them into exact 16-bit values; 8-bit codes go through
// v_cvt_f32_ubyte.  X_g comes from MFMAs against ones, one row block per
// wavefront, is cut into three bf16 parts of 8 bits (24 bits: nothing of the
// fp32 sum is lost) and exchanged through LDS; the bias terms of two steps are
// then one bf16 MFMA per tile, its slots holding X's parts against b (an f16
// bias: against its two bf16 parts), again exact products.
//
// What bounds it: VALU issue and, with the chip full, the clock.  Per 32x32x16
// MFMA (32 cycles of the matrix core) a wavefront issues 4 scale FMAs and 9 /
// MT operations of dequantisation (a nibble word: three to split it, two byte
// permutes, four conversions), 8.3 VALU operations in all at MT = 2, of 4-5
// cycles each: 2000 x 4096 x 24576 keeps the VALU busy 63 % of the time and the
// matrix cores 52 %, at a clock of 2.0 GHz.  So the tile
// of the large sizes is 64 x 256 with two workgroups per CU (each one's waits
// are the other's work): 2000 x 4096 x 12288 256 us, 786 TFLOP/s, where 128 x
// 256 with one workgroup of 8 wavefronts per CU and three stages took 282 us,
// and 64 x 256 with three stages and one workgroup per CU 300 us (the
// general kernel of 32-row blocks, which this one replaces: 1.6 ms).
//
// Two workgroups share a CU's LDS (three of the 32 x 128 tile); with 8-bit
// weights the stages of the larger tiles take it for one.
//
// The loop is software-pipelined by hand (unit()): left to itself the
// compiler hoists reads and products until it spills, and a spill's reload
// waits for the DMA in flight.  What still spills (bytes per lane): the 96 x
// 128 tile 12..28, at group size 32 it and the 64 x 256 one 108..224.
#pragma once

#include "dfmi_device.h"
#include "dfmi_host.h"
#include "dfmi_stream.h"

namespace dfmi {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;

constexpr int kGemmK = 128;      // k per step

constexpr int kGemmMaxSeg = 3;   // matrices of one launch

// One or more matrices over the same activations; matrix i's column tiles are
// tile0 .. of the launch's tiles_n.
struct GemmArgs {
  const uint16_t* x;
  float* partials;    // split K: [tile][split][BM x BN] in register order
  const uint32_t* w[kGemmMaxSeg];
  const uint32_t* t[kGemmMaxSeg];  // (scale, bias) pairs [K/GS][tn], the matrix's column 0 first
  uint16_t* y[kGemmMaxSeg];
  int N[kGemmMaxSeg], tile0[kGemmMaxSeg];
  uint32_t tn[kGemmMaxSeg];
  int nseg, M, K;
  int steps;  // ceil(K / 128)
  int tiles_m, tiles_n, kp;
  int vec;    // every y's rows are 16-byte aligned: whole-piece stores
};

// the matrix of column tile nb
__device__ inline int gemm_seg(const GemmArgs& a, int nb) {
  return a.nseg > 2 && nb >= a.tile0[2] ? 2 : (a.nseg > 1 && nb >= a.tile0[1] ? 1 : 0);
}

// ROWS: the tile's activation rows are given one by one (xr), not consecutive.
template <typename Tag, int GS, int BITS, int MT, int NT, int WM, int WN, bool ROWS = false>
struct Gemm {
  static constexpr int WAVES = WM * WN, THREADS = 64 * WAVES;
  static constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN;
  static constexpr int SUB = GS == 32 ? 2 : 1;        // groups per 64-k unit
  static constexpr int TG = kGemmK / GS;              // groups per step: 4, 2, 1
  static constexpr int XROW = kGemmK * 2, XBUF = BM * XROW;
  static constexpr int WROW = kGemmK * BITS / 8, WBUF = BN * WROW;
  static constexpr int WPIECES = WROW / 16;
  static constexpr int TBUF = TG * BN * 4;
  static constexpr int STAGE = XBUF + WBUF + TBUF;
  // planes of the bias MFMA: a half wavefront holds 8 slots = two triples
  static constexpr int PLANES = std::is_same<Tag, BF16>::value ? SUB : 2 * SUB;
  // exchanged group sums: [parity of the batch][sub][row][parity of the step] 16 bytes
  static constexpr int XT = SUB * BM * 32;
  // Stages: two where two workgroups then share a CU's LDS, else three.
  static constexpr int DEPTH = 2 * (STAGE + XT) <= 80 * 1024   ? 2
                               : 3 * STAGE + 2 * XT <= 160 * 1024 ? 3
                                                                  : 2;
  static constexpr int XT_OFF = DEPTH * STAGE;
  static constexpr int LDS_LOOP = XT_OFF + 2 * XT;
  static constexpr int YROW = BN * 2 + 16;            // output tile row in LDS (epilogue)
  static constexpr int LDS_BYTES = LDS_LOOP > BM * YROW ? LDS_LOOP : BM * YROW;
  static_assert(LDS_BYTES <= 160 * 1024, "LDS");
  static constexpr int X_DMA = XBUF / 1024 / WAVES;
  // 16-row blocks of a wavefront's rows whose group sums it forms (the WN
  // wavefronts of a row share its 2 MT blocks)
  static constexpr int XB = (2 * MT + WN - 1) / WN;
  static constexpr int W_DMA = WBUF / 1024 / WAVES;
  static constexpr int TPB = TBUF / WAVES, TLANES = TPB / 16;
  static constexpr int STEP_DMA = X_DMA + W_DMA + 1;
  static_assert(TLANES >= 1 && TLANES <= 64 && X_DMA >= 1 && W_DMA >= 1, "DMA split");
  static_assert(BN <= THREADS, "one weight row per thread");

  __device__ static inline f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    if constexpr (std::is_same<Tag, BF16>::value)
      return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                     __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                    __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  __device__ static inline f32x16 mma_bf16(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  __device__ static inline f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.f;
    return z;
  }

  // two fp8 bytes (low or high half of v) -> two exact 16-bit values
  template <bool HI>
  __device__ static inline uint32_t cvt2(uint32_t v) {
    if constexpr (std::is_same<Tag, BF16>::value)
      return __builtin_bit_cast(uint32_t,
                                __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 512.f, HI));
    else
      return __builtin_bit_cast(uint32_t,
                                __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(v, 512.f, HI));
  }
  // 8 codes in k order: one 4-bit word ...
  __device__ static inline u32x4 dq4(uint32_t w) {
    const uint32_t ev = w & 0x0F0F0F0Fu, od = (w >> 4) & 0x0F0F0F0Fu;
    const uint32_t lo = __builtin_amdgcn_perm(od, ev, 0x05010400u);  // q0 q1 q2 q3
    const uint32_t hi = __builtin_amdgcn_perm(od, ev, 0x07030602u);  // q4 q5 q6 q7
    return u32x4{cvt2<false>(lo), cvt2<true>(lo), cvt2<false>(hi), cvt2<true>(hi)};
  }
  // ... or two 8-bit words (q < 256: 8 significant bits, exact in both types)
  __device__ static inline u32x4 dq8(uint32_t w0, uint32_t w1) {
    u32x4 r;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t w = h ? w1 : w0;
      const float f0 = (float)(w & 0xFFu), f1 = (float)((w >> 8) & 0xFFu);
      const float f2 = (float)((w >> 16) & 0xFFu), f3 = (float)(w >> 24);
      if constexpr (std::is_same<Tag, BF16>::value) {
        r[2 * h] = __builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
        r[2 * h + 1] = __builtin_amdgcn_perm(__float_as_uint(f3), __float_as_uint(f2), 0x07060302u);
      } else {
        r[2 * h] = __builtin_bit_cast(uint32_t, f16x2{(_Float16)f0, (_Float16)f1});
        r[2 * h + 1] = __builtin_bit_cast(uint32_t, f16x2{(_Float16)f2, (_Float16)f3});
      }
    }
    return r;
  }

  struct Ctx {
    __amdgpu_buffer_rsrc_t x, w, t;
    // DMA, first instruction, step 0: this lane's activation row and piece in
    // it, weight piece and pairs, as byte offsets
    uint32_t xg, xp, wg, tg;
    uint32_t xr[ROWS ? X_DMA : 1];  // ROWS: byte offset of each instruction's row
    uint32_t xo[4];             // activation fragment q of unit 0 in a stage, row block 0
    uint32_t xs[2];             // fragment (k half of unit 0) of 16-row blocks, the wavefront's first
    uint32_t wo[2];             // weight piece e of unit 0 in a stage, column tile 0
    uint32_t to;                // pair of group 0, column tile 0, in a stage
    uint32_t xstride, wstride;  // row bytes
    int K, groups, wave, wm, wn, lane, h;
    uint32_t tn;
    u32x4 ones;
  };

  // k piece (8 k, 16 bytes of activations) of a 64-k unit that half wavefront
  // h feeds MFMA q with: a half takes 32 consecutive k of the unit, or 16 of
  // each of its two groups at gs = 32
  __device__ static inline int piece_of(int h, int q) {
    return SUB == 1 ? 4 * h + q : 4 * (q >> 1) + 2 * h + (q & 1);
  }
  // swizzle key of a weight row in a stage
  __device__ static inline int wkey(int r) { return BITS == 4 ? (r >> 2) & 3 : r & 7; }

  // The lane's constants: K, the pair table's row length, and the first
  // column and number of columns of the tile in it.  The buffers are the
  // caller's.
  __device__ static inline void setup(Ctx& cx, int K, uint32_t tn, int n0, int cols) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    cx.lane = lane;
    cx.wave = wave;
    cx.wm = wave / WN;
    cx.wn = wave % WN;
    cx.h = lane >> 5;
    cx.K = K;
    cx.groups = K / GS;
    cx.tn = tn;
    cx.xstride = (uint32_t)K * 2u;
    cx.wstride = (uint32_t)(K / 8 * BITS);
    // activation DMA: one instruction brings 4 rows; slot s of row r holds
    // piece s ^ (r & 15).  Instruction i of a wavefront is 4 i rows on, which
    // flips bits 2 and 3 of the key
    {
      const int r = wave * X_DMA * 4 + lane / 16;
      cx.xg = (uint32_t)r * cx.xstride;
      cx.xp = (uint32_t)(((lane & 15) ^ (r & 15)) * 16);
    }
    // weight DMA: slot s of row r holds piece s ^ wkey(r); one instruction
    // brings 16 (4-bit) or 8 (8-bit) rows, a whole number of key periods
    constexpr int RPI = 64 / WPIECES;
    {
      const int r = wave * W_DMA * RPI + lane / WPIECES;
      cx.wg = (uint32_t)r * cx.wstride + (uint32_t)(((lane % WPIECES) ^ wkey(r)) * 16);
    }
    // pair DMA: wavefront w brings stage bytes w TPB .. of the [group][row] pairs
    {
      const int o = wave * TPB + 16 * lane;
      const int grp = o / (4 * BN), row = (o % (4 * BN)) / 4;
      cx.tg = (lane < TLANES && row < cols) ? ((uint32_t)grp * tn + (uint32_t)(n0 + row)) * 4u
                                            : kNoRow;
    }
    // fragments
    const int r = lane & 31, n = cx.wn * 32 * NT + r;
    const uint32_t xrow0 = (uint32_t)(cx.wm * 32 * MT * XROW);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      cx.xo[q] = xrow0 + (uint32_t)(r * XROW + ((piece_of(cx.h, q) ^ (r & 15)) * 16));
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
      cx.xs[kk] = xrow0 + (uint32_t)((lane & 15) * XROW +
                                     (((4 * kk + (lane >> 4)) ^ (lane & 15)) * 16));
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      // bytes of the unit: 4-bit, gs >= 64: 16 h .. 16 h + 15 (e unused); gs = 32: 16 e + 8 h
      // .. + 7; 8-bit: 32 h + 16 e .. or 32 e + 16 h .. + 15
      const int byte = BITS == 4 ? (SUB == 1 ? 16 * cx.h : 16 * e + 8 * cx.h)
                                 : (SUB == 1 ? 32 * cx.h + 16 * e : 32 * e + 16 * cx.h);
      cx.wo[e] = (uint32_t)(XBUF + n * WROW + (((byte >> 4) ^ wkey(n)) * 16) + (byte & 15));
    }
    cx.to = (uint32_t)(XBUF + WBUF + n * 4);
    u32x4 ones = u32x4{Num<Tag>::ONE2, Num<Tag>::ONE2, Num<Tag>::ONE2, Num<Tag>::ONE2};
    asm volatile("" : "+v"(ones));
    cx.ones = ones;
  }
  // unit U's fragments: 8 activation pieces (128 bytes), or 2 / 4 weight
  // pieces on, the swizzled slots' bits flipped
  template <int U>
  __device__ static inline uint32_t xu(uint32_t o, uint32_t st) { return (o ^ (U * 128u)) + st; }
  template <int U>
  __device__ static inline uint32_t wu(uint32_t o, uint32_t st) {
    return (o ^ (U * (BITS == 4 ? 32u : 64u))) + st;
  }

  __device__ static inline void issue(const Ctx& cx, int c, uint32_t st) {
    if (cx.K - c * kGemmK < kGemmK) issue_part<true>(cx, c, st);
    else issue_part<false>(cx, c, st);
  }
  // PART: the last step, of fewer than 128 k.  Activations past K come as
  // zeros, so every product and group sum there is zero; weights and pairs
  // past K are not read.
  template <bool PART>
  __device__ static inline void issue_part(const Ctx& cx, int c, uint32_t st) {
    char* base = dfmi_smem + st;
    constexpr int RPI = 64 / WPIECES;
    const int left = cx.K - c * kGemmK;
#pragma unroll
    for (int i = 0; i < X_DMA; ++i) {
      const uint32_t piece = cx.xp ^ (uint32_t)(64 * (i & 3));
      uint32_t off =
          piece + (ROWS ? cx.xr[ROWS ? i : 0] : cx.xg + (uint32_t)(4 * i) * cx.xstride);
      if (PART && (int)piece >= 2 * left) off = kNoRow;
      dma16(cx.x, off, (uint32_t)c * (uint32_t)XROW, base + (cx.wave * X_DMA + i) * 1024);
    }
    const bool wpast =
        PART && (int)((cx.lane % WPIECES) ^ wkey(cx.lane / WPIECES)) * 128 >= left * BITS;
#pragma unroll
    for (int i = 0; i < W_DMA; ++i)
      dma16(cx.w, wpast ? kNoRow : cx.wg + (uint32_t)(RPI * i) * cx.wstride,
            (uint32_t)c * (uint32_t)WROW, base + XBUF + (cx.wave * W_DMA + i) * 1024);
    if (cx.lane < TLANES) {
      const bool tpast = PART && c * TG + (cx.wave * TPB + 16 * cx.lane) / (4 * BN) >= cx.groups;
      dma16(cx.t, tpast ? kNoRow : cx.tg, (uint32_t)(c * TG) * cx.tn * 4u,
            base + XBUF + WBUF + cx.wave * TPB);
    }
  }

  struct Acc {
    f32x16 v[MT][NT];
  };

  // The bias terms of one batch (two steps): half wavefront h holds step
  // parity h.  rb[j][s]: this lane's column's biases of its step's two units.
  // zero_hi: only the first step of the batch exists.
  __device__ static inline void flush(const Ctx& cx, int bp, const uint32_t (&rb)[NT][SUB],
                                      Acc& acc, bool zero_hi) {
    const char* xt = dfmi_smem + XT_OFF + bp * XT + (cx.wm * 32 * MT + (cx.lane & 31)) * 32 +
                     cx.h * 16;
    const bool drop = zero_hi && cx.h;
#pragma unroll
    for (int s = 0; s < SUB; ++s) {
      u32x4 e[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        e[i] = *reinterpret_cast<const u32x4*>(xt + s * BM * 32 + i * 32 * 32);
        if (zero_hi) {
#pragma unroll
          for (int k = 0; k < 4; ++k) e[i][k] = drop ? 0u : e[i][k];
        }
      }
#pragma unroll
      for (int p = 0; p < PLANES / SUB; ++p) {
        u32x4 xa[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          if constexpr (std::is_same<Tag, BF16>::value) {
            // (X1 X2 | X3 of unit 0, X1 of unit 1 | X2 X3)
            xa[i] = u32x4{e[i].x, __builtin_amdgcn_perm(e[i].z, e[i].y, 0x05040100u),
                          __builtin_amdgcn_perm(e[i].w, e[i].z, 0x05040302u), 0u};
          } else {
            // unit p: (X1 X2 | X3 X1 | X2 X3)
            const uint32_t d0 = p ? e[i].z : e[i].x, d1 = p ? e[i].w : e[i].y;
            xa[i] = u32x4{d0, __builtin_amdgcn_perm(d0, d1, 0x05040100u),
                          __builtin_amdgcn_perm(d1, d0, 0x05040302u), 0u};
          }
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const uint32_t v = drop ? 0u : rb[j][s];
          u32x4 xb;
          if constexpr (std::is_same<Tag, BF16>::value) {
            xb = u32x4{__builtin_amdgcn_perm(v, v, 0x01000100u), v,
                       __builtin_amdgcn_perm(v, v, 0x03020302u), 0u};
          } else {
            const float f = p ? Num<F16>::hi(v) : Num<F16>::lo(v);
            const uint32_t b1 = __float_as_uint(f) & 0xFFFF0000u;
            const uint32_t b2 = __float_as_uint(f - __uint_as_float(b1));
            xb = u32x4{__builtin_amdgcn_perm(b1, b1, 0x07060302u),
                       __builtin_amdgcn_perm(b2, b1, 0x07060302u),
                       __builtin_amdgcn_perm(b2, b2, 0x07060302u), 0u};
          }
#pragma unroll
          for (int i = 0; i < MT; ++i) acc.v[i][j] = mma_bf16(xa[i], xb, acc.v[i][j]);
        }
      }
    }
  }

  // State of the software pipeline across regions.
  static constexpr int WN_ = BITS == 4 && SUB == 1 ? 1 : 2;  // weight reads per column tile
  static constexpr int AS = MT == 1 ? 2 : 1;                 // sets of activation fragments
  struct Pipe {
    u32x4 a[AS][MT][4];      // activations of the unit
    u32x4 xf[XB][2];         // and of the 16-row blocks to sum
    uint32_t w[NT][BITS];    // packed words of the next column tile to dequantise (by tile)
    uint32_t t[2][NT][SUB];  // (scale, bias) pairs, by unit
    u32x4 bq[2][4];          // dequantised column tile, by phase parity (unit, column tile)
    f32x16 p[SUB];           // the previous region's products, not yet scaled
    float ps[SUB];           // and their scales
    u32x4 e[XB][SUB];        // the step's group sums in parts
  };

  template <int U>
  __device__ static inline void load_a(const Ctx& cx, uint32_t st, int i, u32x4 (&a)[MT][4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      a[i][q] = *reinterpret_cast<const u32x4*>(dfmi_smem + xu<U>(cx.xo[q], st) + i * 32 * XROW);
  }
  template <int U>
  __device__ static inline void load_xf(const Ctx& cx, uint32_t st, Pipe& z) {
#pragma unroll
    for (int e = 0; e < XB; ++e)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
        z.xf[e][kk] = *reinterpret_cast<const u32x4*>(
            dfmi_smem + xu<U>(cx.xs[kk], st) + ((cx.wn + e * WN) % (2 * MT)) * 16 * XROW);
  }
  template <int U>
  __device__ static inline void load_w(const Ctx& cx, uint32_t st, int j, Pipe& z) {
#pragma unroll
    for (int e = 0; e < WN_; ++e) {
      const char* p = dfmi_smem + wu<U>(cx.wo[e], st) + j * 32 * WROW;
      if constexpr (BITS == 4 && SUB == 2) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(p);
        z.w[j][2 * e] = v.x;
        z.w[j][2 * e + 1] = v.y;
      } else {
        const u32x4 v = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
        for (int i = 0; i < 4; ++i) z.w[j][4 * e + i] = v[i];
      }
    }
  }
  template <int U>
  __device__ static inline void load_t(const Ctx& cx, uint32_t st, Pipe& z) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int s = 0; s < SUB; ++s) {
        const int g = GS == 32 ? 2 * U + s : (GS == 64 ? U : 0);
        z.t[U][j][s] =
            *reinterpret_cast<const uint32_t*>(dfmi_smem + (cx.to + st) + (g * BN + 32 * j) * 4);
      }
  }
  __device__ static inline u32x4 dq(const Pipe& z, int j, int q) {
    if constexpr (BITS == 4) return dq4(z.w[j][q]);
    else return dq8(z.w[j][2 * q], z.w[j][2 * q + 1]);
  }

  // the three bf16 parts of an fp32 sum: (first | second << 16), third
  __device__ static inline void parts(float v, uint32_t& d0, uint32_t& d1) {
    const uint32_t x1 = __float_as_uint(v) & 0xFFFF0000u;
    const float r1 = v - __uint_as_float(x1);
    const uint32_t x2 = __float_as_uint(r1) & 0xFFFF0000u;
    d0 = __builtin_amdgcn_perm(x2, x1, 0x07060302u);
    d1 = __float_as_uint(r1 - __uint_as_float(x2)) >> 16;
  }

  // Unit U of a step in MT NT regions.  Region (j, i): the products of row
  // block i and column tile j (4 MFMAs), while the VALU scales the previous
  // region's products and dequantises a share of the next column tile, and
  // the LDS brings what the next unit (stage nst, unit 1 - U) needs into the
  // registers that are done with.  The regions are fences for the scheduler,
  // which otherwise hoists reads and products until it spills.  Every read of
  // this unit's stage has been made before the unit starts, but for t.
  template <int U, int PAR>
  __device__ static inline void unit(const Ctx& cx, uint32_t nst, Acc& acc, Pipe& z,
                                     uint32_t (&rb)[NT][SUB]) {
    constexpr int R = MT * NT, V = 1 - U;
    constexpr int CUR = AS == 2 ? U : 0, NXT = AS == 2 ? V : 0;
    if constexpr (U == 1) {  // the step's biases (its first unit's pairs are about to go)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int s = 0; s < SUB; ++s) {
          const uint32_t v = __builtin_amdgcn_perm(z.t[1][j][s], z.t[0][j][s], 0x07060302u);
          rb[j][s] = cx.h == PAR ? v : rb[j][s];
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int j = r / MT, i = r % MT;
      const int ph = (U * NT + j) & 1;
      __builtin_amdgcn_sched_barrier(0);
      if (i == 0) load_w<V>(cx, nst, j, z);
      if (r == 0) load_t<V>(cx, nst, z);
      if (AS == 2 ? r == 0 : (j == NT - 1 && i > 0)) load_a<V>(cx, nst, AS == 2 ? 0 : i - 1, z.a[NXT]);
      // products
      f32x16 p[SUB];
      const u32x4(&av)[4] = z.a[CUR][i];
      if constexpr (SUB == 1) {
        p[0] = mma(av[0], z.bq[ph][0], zero16());
#pragma unroll
        for (int q = 1; q < 4; ++q) p[0] = mma(av[q], z.bq[ph][q], p[0]);
      } else {
#pragma unroll
        for (int s = 0; s < 2; ++s)
          p[s] = mma(av[2 * s + 1], z.bq[ph][2 * s + 1], mma(av[2 * s], z.bq[ph][2 * s], zero16()));
      }
      if (r == 0) {
        // group sums: ones as the rows, 16 activation rows as the columns, so
        // lane l ends with X[l % 16]
#pragma unroll
        for (int e = 0; e < XB; ++e) {
          float v[SUB];
          if constexpr (SUB == 1) {
            v[0] = Num<Tag>::mma(cx.ones, z.xf[e][1], Num<Tag>::mma(cx.ones, z.xf[e][0], zero4())).x;
          } else {
#pragma unroll
            for (int s = 0; s < 2; ++s) v[s] = Num<Tag>::mma(cx.ones, z.xf[e][s], zero4()).x;
          }
#pragma unroll
          for (int s = 0; s < SUB; ++s) {
            uint32_t d0, d1;
            parts(v[s], d0, d1);
            z.e[e][s][2 * U] = d0;
            z.e[e][s][2 * U + 1] = d1;
          }
        }
      }
      // the previous region's products, scaled
      const int pj = r ? (r - 1) / MT : NT - 1, pi = r ? (r - 1) % MT : MT - 1;
#pragma unroll
      for (int s = 0; s < SUB; ++s)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          acc.v[pi][pj][e] = __builtin_fmaf(z.ps[s], z.p[s][e], acc.v[pi][pj][e]);
      asm volatile("" : "+v"(acc.v[pi][pj]));  // here, not where it is next read
      // the next column tile (of this unit, or the next unit's first)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q * MT / 4 == i) {
          z.bq[ph ^ 1][q] = dq(z, (j + 1) % NT, q);
          asm volatile("" : "+v"(z.bq[ph ^ 1][q]));
        }
#pragma unroll
      for (int s = 0; s < SUB; ++s) {
        z.p[s] = p[s];
        z.ps[s] = Num<Tag>::lo(z.t[U][j][s]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (AS == 1) load_a<V>(cx, nst, MT - 1, z.a[NXT]);
    load_xf<V>(cx, nst, z);
  }

  // One step: unit 0; then the next step's stage is awaited, and this one's,
  // whose every read has been made, is refilled; unit 1.
  template <int PAR>
  __device__ static inline void step(const Ctx& cx, int c0, int n, int i, uint32_t& st, int bp,
                                     Acc& acc, Pipe& z, uint32_t (&rb)[NT][SUB]) {
    unit<0, PAR>(cx, st, acc, z, rb);
    const uint32_t nst = st == (DEPTH - 1) * STAGE ? 0 : st + STAGE;
    const bool one = DEPTH == 3 && i + 2 < n;  // step i + 2 may be in flight
    if (one) stage_barrier<STEP_DMA>();
    else stage_barrier<0>();
    if (i + DEPTH < n) issue(cx, c0 + i + DEPTH, st);
    // the bias terms of the batch before, whose sums this barrier published (the first: zeros)
    if constexpr (PAR == 0) flush(cx, bp ^ 1, rb, acc, false);
    unit<1, PAR>(cx, nst, acc, z, rb);
    if (cx.lane < 16) {
#pragma unroll
      for (int e = 0; e < XB; ++e)
        if (cx.wn + e * WN < 2 * MT)
#pragma unroll
          for (int s = 0; s < SUB; ++s)
            *reinterpret_cast<u32x4*>(
                dfmi_smem + XT_OFF + bp * XT + s * BM * 32 +
                (cx.wm * 32 * MT + (cx.wn + e * WN) * 16 + cx.lane) * 32 + PAR * 16) = z.e[e][s];
    }
    st = nst;
  }

  // Request the first stages of steps [c0, c1) (LDS stages free).
  __device__ static inline void start(const Ctx& cx, int c0, int c1) {
#pragma unroll
    for (int k = 0; k < DEPTH; ++k) {
      if (k < c1 - c0) issue(cx, c0 + k, k * STAGE);
    }
  }

  // Accumulate steps [c0, c1), whose first stages start() has requested.  On
  // return every wavefront is past its last read of the stages; the group
  // sums' exchange is read until the caller's next barrier.
  __device__ static inline void run(const Ctx& cx, int c0, int c1, Acc& acc) {
    run(cx, c0, c1, acc, [] {});
  }
  // between: called once the stages are free, before the last bias terms.
  template <typename F>
  __device__ static inline void run(const Ctx& cx, int c0, int c1, Acc& acc, F&& between) {
    const int n = c1 - c0;
    uint32_t rb[NT][SUB];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int s = 0; s < SUB; ++s) rb[j][s] = 0u;
    for (int o = threadIdx.x * 16; o < XT; o += THREADS * 16)  // what the first flush reads
      *reinterpret_cast<u32x4*>(dfmi_smem + XT_OFF + XT + o) = u32x4{0u, 0u, 0u, 0u};
    // step 0 in LDS: the later ones may be in flight
    if (n >= DEPTH) stage_barrier<(DEPTH - 1) * STEP_DMA>();
    else if (DEPTH == 3 && n == 2) stage_barrier<STEP_DMA>();
    else stage_barrier<0>();
    Pipe z;
#pragma unroll
    for (int j = 0; j < NT; ++j) load_w<0>(cx, 0, j, z);
    load_t<0>(cx, 0, z);
#pragma unroll
    for (int i = 0; i < MT; ++i) load_a<0>(cx, 0, i, z.a[0]);
    load_xf<0>(cx, 0, z);
#pragma unroll
    for (int q = 0; q < 4; ++q) z.bq[0][q] = dq(z, 0, q);
#pragma unroll
    for (int s = 0; s < SUB; ++s) {
      z.p[s] = zero16();
      z.ps[s] = 0.f;
    }
    uint32_t st = 0;
    int i = 0, bp = 0;
    for (; i + 2 <= n; i += 2) {
      step<0>(cx, c0, n, i, st, bp, acc, z, rb);
      step<1>(cx, c0, n, i + 1, st, bp, acc, z, rb);
      bp ^= 1;
    }
    const bool odd = i < n;
    if (odd) {
      step<0>(cx, c0, n, i, st, bp, acc, z, rb);
      bp ^= 1;
    }
#pragma unroll
    for (int s = 0; s < SUB; ++s)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        acc.v[MT - 1][NT - 1][e] = __builtin_fmaf(z.ps[s], z.p[s][e], acc.v[MT - 1][NT - 1][e]);
    stage_barrier<0>();
    between();
    flush(cx, bp ^ 1, rb, acc, odd);
  }
};

// workgroup -> tile: each XCD (workgroup id % 8 where dispatch goes round
// robin; a locality hint only) takes consecutive units, row blocks of one
// column block and split next to each other, so they share its weights in
// the XCD's L2
template <typename Tag, int GS, int BITS, int MT, int NT, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN, 2) void qmm_gemm_kernel(GemmArgs a) {
  using G = Gemm<Tag, GS, BITS, MT, NT, WM, WN>;
  const int total = gridDim.x, L = blockIdx.x;
  const int xcd = L & 7, q8 = total >> 3, r8 = total & 7;
  const int id = xcd * q8 + min(xcd, r8) + (L >> 3);
  const int nb = id / (a.kp * a.tiles_m);
  const int rest = id - nb * (a.kp * a.tiles_m);
  const int kpi = rest / a.tiles_m, mb = rest - kpi * a.tiles_m;
  const int g = gemm_seg(a, nb);
  const uint32_t* const w = g == 2 ? a.w[2] : (g == 1 ? a.w[1] : a.w[0]);
  uint16_t* const y = g == 2 ? a.y[2] : (g == 1 ? a.y[1] : a.y[0]);
  const int N = g == 2 ? a.N[2] : (g == 1 ? a.N[1] : a.N[0]);
  const int tile0 = g == 2 ? a.tile0[2] : (g == 1 ? a.tile0[1] : 0);
  const uint32_t* const t = g == 2 ? a.t[2] : (g == 1 ? a.t[1] : a.t[0]);
  const uint32_t tn = g == 2 ? a.tn[2] : (g == 1 ? a.tn[1] : a.tn[0]);
  const int m0 = mb * G::BM, n0 = (nb - tile0) * G::BN;
  const int c0 = (int)((int64_t)kpi * a.steps / a.kp);
  const int c1 = (int)((int64_t)(kpi + 1) * a.steps / a.kp);
  typename G::Ctx cx;
  const int rows = min(G::BM, a.M - m0), cols = min(G::BN, N - n0);
  G::setup(cx, a.K, tn, n0, cols);
  // the buffers end with the tile's last row: reads past it return zeros
  cx.x = buffer_rsrc(a.x + (int64_t)m0 * a.K, (uint32_t)rows * cx.xstride);
  cx.w = buffer_rsrc(w + (int64_t)n0 * (cx.wstride / 4), (uint32_t)cols * cx.wstride);
  cx.t = buffer_rsrc(t, (tn * (uint32_t)(cx.groups - 1) + (uint32_t)N) * 4u);
  typename G::Acc acc;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc.v[i][j] = G::zero16();
  G::start(cx, c0, c1);
  G::run(cx, c0, c1, acc);

  const int h = cx.h, col = cx.wn * 32 * NT + (cx.lane & 31), row = cx.wm * 32 * MT;
  if (a.kp > 1) {
    // fp32 partial tile in register order (256-byte rows); qmm_gemm_sum_kernel
    // adds the splits
    const int tile = nb * a.tiles_m + mb;
    float* mine = a.partials + ((int64_t)tile * a.kp + kpi) * (G::BM * G::BN) +
                  cx.wave * (MT * NT * 1024) + cx.lane;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[((i * NT + j) * 16 + r) * 64] = acc.v[i][j][r];
    return;
  }

  if (a.vec) {
    // through LDS, so that rows leave in whole 16-byte pieces
    stage_barrier<0>();
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = row + 32 * i + 8 * (r >> 2) + 4 * h + (r & 3);
          *reinterpret_cast<uint16_t*>(dfmi_smem + m * G::YROW + (col + 32 * j) * 2) =
              Num<Tag>::f2h(acc.v[i][j][r]);
        }
    stage_barrier<0>();
    constexpr int PPR = G::BN / 8;
#pragma unroll 4
    for (int p = threadIdx.x; p < G::BM * PPR; p += G::THREADS) {
      const int m = p / PPR, n = (p % PPR) * 8;
      const u32x4 v = *reinterpret_cast<const u32x4*>(dfmi_smem + m * G::YROW + n * 2);
      if (m0 + m < a.M && n0 + n < N)
        *reinterpret_cast<u32x4*>(y + (int64_t)(m0 + m) * N + n0 + n) = v;
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + row + 32 * i + 8 * (r >> 2) + 4 * h + (r & 3), n = n0 + col + 32 * j;
        if (m < a.M && n < N) y[(int64_t)m * N + n] = Num<Tag>::f2h(acc.v[i][j][r]);
      }
}

// Split K: the sum of every tile's splits, in split order, rounded into y.
// A thread takes four consecutive columns of one row; a workgroup 1024 values
// of a tile.  (The last split of a tile summing the others' inside the product
// kernel instead took 1.1 us per split on one CU: [77,5120] x [5120,5120] in 6
// splits 20.6 us.)
template <typename Tag, int MT, int NT, int WM, int WN>
__global__ __launch_bounds__(256) void qmm_gemm_sum_kernel(GemmArgs a) {
  constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN, TILE = BM * BN, PER = TILE / 1024;
  const int tile = blockIdx.x / PER, e = ((blockIdx.x % PER) * 256 + threadIdx.x) * 4;
  const int nb = tile / a.tiles_m, g = gemm_seg(a, nb), kp = a.kp;
  uint16_t* const y = g == 2 ? a.y[2] : (g == 1 ? a.y[1] : a.y[0]);
  const int N = g == 2 ? a.N[2] : (g == 1 ? a.N[1] : a.N[0]);
  const int tile0 = g == 2 ? a.tile0[2] : (g == 1 ? a.tile0[1] : 0);
  // e: wavefront, row block and column tile, register, lane
  const int wave = e / (MT * NT * 1024), ij = e / 1024 % (MT * NT), r = e / 64 % 16, lane = e % 64;
  const int m = (tile % a.tiles_m) * BM + (wave / WN) * 32 * MT + (ij / NT) * 32 + 8 * (r >> 2) +
                4 * (lane >> 5) + (r & 3);
  const int n = (nb - tile0) * BN + (wave % WN) * 32 * NT + (ij % NT) * 32 + (lane & 31);
  if (m >= a.M || n >= N) return;
  const float* p = a.partials + (int64_t)tile * kp * TILE + e;
  f32x4 sum = zero4();
  for (int k0 = 0; k0 < kp; k0 += 4) {
    f32x4 t[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      t[k] = *reinterpret_cast<const f32x4*>(p + (int64_t)min(k0 + k, kp - 1) * TILE);
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int c = 0; c < 4; ++c) sum[c] += k0 + k < kp ? t[k][c] : 0.f;
  }
  uint16_t* out = y + (int64_t)m * N + n;
  if (a.vec) {
    u32x2 v;
    v.x = (uint32_t)Num<Tag>::f2h(sum.x) | ((uint32_t)Num<Tag>::f2h(sum.y) << 16);
    v.y = (uint32_t)Num<Tag>::f2h(sum.z) | ((uint32_t)Num<Tag>::f2h(sum.w) << 16);
    *reinterpret_cast<u32x2*>(out) = v;
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (n + c < N) out[c] = Num<Tag>::f2h(sum[c]);
  }
}

// Host side of one configuration: the tile, and the launch of a planned call.
template <typename Tag, int GS, int BITS, int MT, int NT, int WM, int WN>
static void gemm_launch_cfg(const GemmArgs& a, hipStream_t st) {
  using G = Gemm<Tag, GS, BITS, MT, NT, WM, WN>;
  static const bool lds_allowed = [] {  // more than 64 KiB of dynamic LDS
    return hipFuncSetAttribute(
               reinterpret_cast<const void*>(&qmm_gemm_kernel<Tag, GS, BITS, MT, NT, WM, WN>),
               hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS_BYTES) == hipSuccess;
  }();
  (void)lds_allowed;  // a refusal shows as the launch's own error
  hipLaunchKernelGGL((qmm_gemm_kernel<Tag, GS, BITS, MT, NT, WM, WN>),
                     dim3(a.tiles_m * a.tiles_n * a.kp), dim3(G::THREADS), G::LDS_BYTES, st, a);
  if (a.kp > 1)
    hipLaunchKernelGGL((qmm_gemm_sum_kernel<Tag, MT, NT, WM, WN>),
                       dim3(a.tiles_m * a.tiles_n * (G::BM * G::BN / 1024)), dim3(256), 0, st, a);
}

// cfg: index into kGemmCfgs (dfmi_gemm.hip)
template <typename Tag, int GS, int BITS>
static void gemm_launch_gs(int cfg, const GemmArgs& a, hipStream_t st) {
  if (cfg == 0) gemm_launch_cfg<Tag, GS, BITS, 2, 2, 1, 4>(a, st);
  else if (cfg == 1) gemm_launch_cfg<Tag, GS, BITS, 3, 1, 1, 4>(a, st);
  else gemm_launch_cfg<Tag, GS, BITS, 1, 1, 1, 4>(a, st);
}

template <typename Tag, int BITS>
static void gemm_launch_bits(int cfg, int gs, const GemmArgs& a, hipStream_t st) {
  if (gs == 32) gemm_launch_gs<Tag, 32, BITS>(cfg, a, st);
  else if (gs == 64) gemm_launch_gs<Tag, 64, BITS>(cfg, a, st);
  else gemm_launch_gs<Tag, 128, BITS>(cfg, a, st);
}

// one per element type and weight width, each in a translation unit of its own
void gemm_launch_bf16_4(int cfg, int gs, const GemmArgs& a, hipStream_t st);
void gemm_launch_bf16_8(int cfg, int gs, const GemmArgs& a, hipStream_t st);
void gemm_launch_f16_4(int cfg, int gs, const GemmArgs& a, hipStream_t st);
void gemm_launch_f16_8(int cfg, int gs, const GemmArgs& a, hipStream_t st);

}  // namespace dfmi
