// What the scans of a matrix state share (recurrent.hip, matrix_memory.hip).
#pragma once
#include "common.h"

#define TP_SCAN_AHEAD 4          // tokens whose loads are issued together

__device__ __forceinline__ float lane_value(float x, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// DK: key rows a lane keeps of its column (the head's key size rounded up to 16, 32 or a multiple of 64); NR registers
// hold a per-row vector, row (lane + 64 n) in register n.
template <typename T, int NR>
__device__ __forceinline__ void load_rows(float (&dst)[NR], const T* p, int rows, int lane, float scale) {
#pragma unroll
    for (int n = 0; n < NR; n++) {
        const int row = lane + 64 * n;
        dst[n] = row < rows ? ld_f32(p + row) * scale : 0.f;
    }
}

#define TP_SCAN_SIZES(LAUNCH, rows) do { \
    if ((rows) <= 16) LAUNCH(16); else if ((rows) <= 32) LAUNCH(32); else if ((rows) <= 64) LAUNCH(64); \
    else if ((rows) <= 128) LAUNCH(128); else LAUNCH(256); } while (0)
