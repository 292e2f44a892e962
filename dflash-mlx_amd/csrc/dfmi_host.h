// Host-side helpers shared by the C-ABI translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstdarg>
#include <cstdio>
#include <mutex>

#include "../../include/dfmi.h"

namespace dfmi {

// Thread-local error message (dfmi_last_error).
void set_error(const char* fmt, ...) __attribute__((format(printf, 1, 2)));

// Held while a call enqueues several kernels that pass data through its
// workspace: another thread may use that workspace on the same stream, where
// the stream orders single kernels only.
std::mutex& launch_order();

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return DFMI_ELAUNCH;
  }
  return DFMI_OK;
}

inline size_t round_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Shapes the streaming main loop takes (int4 or 8-bit): M <= 32, whole 256-k steps and
// scale blocks of 8 groups; buffer offsets are 32-bit and the record count a
// signed int, so the packed weights stay under 2 GiB.
inline bool stream_eligible(int64_t M, int64_t K, int64_t N, int gs, int bits = 4) {
  return M <= 32 && K % 256 == 0 && K % (8 * gs) == 0 && K < (1ll << 24) &&
         N * (K / 8 * bits) < (1ll << 31);
}

// Many activation rows (dfmi_gemm.hip).  The workspace holds the streaming
// kernels' counters (untouched), the pair table of a call without one, and
// the partial tiles of a K split; with less of it (or none) the call runs
// unsplit, or, without a table either, is not taken.
constexpr int kGemmNotTaken = 1;
bool gemm_shape(int64_t M, int64_t K, int64_t N, int gs);
size_t gemm_workspace_bytes(int64_t M, int64_t K, int64_t N, int gs);
size_t gemm_multi_workspace_bytes(int64_t M, int64_t K, const int64_t* Ns, int nseg, int gs);
// tile and K splits of a launch with the whole workspace
void gemm_plan_query(int64_t M, int64_t K, const int64_t* Ns, int nseg, int* rows, int* cols,
                     int* splits);
// fused: the matrices' tables side by side, or null (their own sb_pairs, rows
// pair_stride apart if not 0).  More than one matrix: every N >= 1 and a
// multiple of 4.
int gemm_launch(const void* x, int x_dtype, const dfmi_qmm_segment* segs, int nseg,
                const uint32_t* fused, int64_t pair_stride, int64_t M, int64_t K, int gs,
                int bits, void* workspace, size_t workspace_bytes, hipStream_t st);

}  // namespace dfmi

// 8-bit affine qmm launch (dfmi_qmm8.hip), called by dfmi_qmm_affine_ex after
// its argument checks.
int dfmi_qmm8_launch(const void* x, int x_dtype, const uint32_t* w_q, const void* scales,
                     const void* biases, void* y, int64_t M, int64_t K, int64_t N, int gs,
                     void* stream);
