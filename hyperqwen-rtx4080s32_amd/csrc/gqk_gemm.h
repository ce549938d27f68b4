// gqk_gemm.h - the GEMM's tile geometries and the launch choice between them (host).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "gqk_internal.h"

namespace gqk {

// (MB, NR, WK): 32 MB tokens x 32 NR weight rows per workgroup, K split over WK groups of NR waves.
#define GQK_GEMM_GEOS(X) X(2, 2, 4) X(2, 4, 4) X(2, 5, 3) X(4, 4, 2) X(4, 5, 2) X(8, 8, 1)

// A launch of the GEMM: the geometry and its schedule.  MB < 8: one workgroup per (tile, token block,
// k-split of S); MB = 8: G persistent workgroups, the remainder tiles over gsk of them (stream-K).
struct GemmPick {
  int mb, nr, wk;
  int per;              // 32-row blocks per descriptor row
  int S, G, gsk, grid;
  int64_t slots, slot_bytes;   // fp32 partial slots of the launch
};

#define GQK_GEMM_DECL(MB)                                                                                       \
  int launch_gemm_mb##MB(const GemmPick& p, int only, int n_desc, int M, hipStream_t st, const uint8_t* packed, \
                         const int32_t* desc, const uint16_t* x, int64_t ldx, uint16_t* y, int64_t ldy,         \
                         const uint16_t* bias, float* part, int* ctr);
GQK_GEMM_DECL(2) GQK_GEMM_DECL(4) GQK_GEMM_DECL(8)
#undef GQK_GEMM_DECL

}  // namespace gqk
