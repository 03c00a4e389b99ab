// What the scans of a matrix state share (recurrent.hip, matrix_memory.hip).
#pragma once
#include "common.h"

#define TP_SCAN_AHEAD 4          // tokens whose loads are issued together

__device__ __forceinline__ int lane_value(int x, int lane) { return __builtin_amdgcn_readlane(x, lane); }
__device__ __forceinline__ float lane_value(float x, int lane) { return __int_as_float(lane_value(__float_as_int(x), lane)); }

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

// ---- a step of one row for each sequence: its state read and written once, by whole rows.  A thread holds four columns of every
// blockDim / (columns / 4)-th row, all of its loads asked for at once; what each row needs (its q, k, decay) reaches the threads
// through LDS while they travel, and the row parts of an output meet there once.
// threads for a state of rows x columns floats (0: sizes that it does not take): a thread holds at most 16 rows
static inline int tp_step_threads(int rows, int cols) {
    if (cols < 4 || cols > 256 || (cols & (cols - 1)) || rows > 256) return 0;
    return (long)rows * cols > 4096 ? 1024 : 256;
}
// four columns' sums of a thread, added over the wave's lanes of the same columns (Q column groups in turn), into the wave's part
__device__ __forceinline__ void step_parts(float4 o, int Q, int lane, float* part) {
    for (int x = Q; x < 64; x <<= 1) {
        o.x += __shfl_xor(o.x, x, 64);
        o.y += __shfl_xor(o.y, x, 64);
        o.z += __shfl_xor(o.z, x, 64);
        o.w += __shfl_xor(o.w, x, 64);
    }
    if (lane < Q) *reinterpret_cast<float4*>(part) = o;
}
