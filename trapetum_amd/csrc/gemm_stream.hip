// bf16 product for up to 64 rows (a decode step of many sequences): bound by reading W once, fp32 accumulation.
//
// A block owns BN = 32, 64, 96 or 128 rows of W and all rows of X (MB = 16, 32 or 64 of them), and walks K in steps of 64.  W and X
// come straight from global memory into LDS, S steps deep, so a CU has 72 to 128 KB of loads in flight without a register spent
// on them (the register-staged 64 x 64 tiles of gemm_mfma.hip hold one step each and wait for it; the 8-row kernel of
// gemm_rows8.hip holds eight loads a wave).  One barrier a step: behind it the step's tiles have arrived, and the place of the step
// before, which everyone has read, takes the tiles S - 1 steps on.  Waves of up to MB rows of X by 32 rows of W (a block of 96: by all)
// (v_mfma_f32_16x16x32_bf16 with W as the A operand: a lane ends up with four neighbours of a row of Y, and with gate and up column
// of a unit in two accumulators).  The 16-byte chunks of an LDS row (128 bytes) lie at chunk ^ (row % 8), the swizzle applied on
// the global side of the load.
//
// Measured on MI355X, cold weights, replayed graph, microseconds, before (the kernels named above) / here; down and o include
// the norm that adds their slices:
//             8 rows                                                    64 rows
//   2B        gate/up 19.3 / 18.2  down 16.0 / 14.8  qkv 6.3 / 5.7       gate/up 26.6 / 21.6  down 20.6 / 16.8  qkv 8.5 / 6.5
//             o 8.9 / 8.4    logits 209 / 202                            o 12.4 / 9.9   logits 258 / 243
//   9B        gate/up 40.3 / 38.0  down 27.5 / 24.0  qkv 14.4 / 12.4     gate/up 44.0 / 39.7  down 37.3 / 28.8  qkv 19.5 / 14.2
//             o 15.0 / 12.1                                              o 16.4 / 13.8
// (the 9B gate/up matrix of 205 MB in 38.0 us is 5.4 TB/s; a copy reaches 6.1.)
#include "gemm.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 st_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float st_f32x4;

namespace {
constexpr int BK = 64;
union StFrag { uint4 u; st_bf16x8 v; };
// until all but the N youngest loads, and every LDS read (whose place is filled again behind the barrier), are done
template <int N> __device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14)); }
}

template <int EPI, int MB, int BN, int WAVES, int S, int WN = BN / 32>
__global__ void __launch_bounds__(64 * WAVES)
gemm_stream_k(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W, void* __restrict__ Y, int M, int N, int K,
              int out_dtype, float4 epi, int units, int k_per_split) {
    constexpr int WM = WAVES / WN, ROWS = 8 * WAVES, LX = MB / ROWS, LW = BN / ROWS, L = LX + LW, STAGE = (MB + BN) * 128, TM = MB / 16 / WM, TN = BN / 16 / WN;
    static_assert(TM >= 1 && LX >= 1 && LW >= 1 && (S - 2) * L < 64, "tile");
    __shared__ __attribute__((aligned(16))) unsigned char lds[S * STAGE];
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave / WN, wn = wave % WN;
    const int n0 = blockIdx.x * BN;
    const int k_begin = blockIdx.y * k_per_split, k_end = min(K, k_begin + k_per_split);
    if (gridDim.y > 1) Y = (float*)Y + (size_t)blockIdx.y * M * N;
    const int steps = (k_end - k_begin) / BK;

    // loads: 8 rows of 128 bytes an instruction, lane l's place (row l / 8, place l % 8) holds chunk place ^ row; rows past the
    // edges read the last row (their products are not stored)
    const bf16_t* const wb = W + (size_t)n0 * K;
    const unsigned chunk = (unsigned)((lane & 7) ^ (lane >> 3)) * 16u;
    unsigned xo[LX], wo[LW];
#pragma unroll
    for (int i = 0; i < LX; i++) xo[i] = (unsigned)min(i * ROWS + wave * 8 + (lane >> 3), M - 1) * (unsigned)K * 2u + chunk;
#pragma unroll
    for (int i = 0; i < LW; i++) wo[i] = (unsigned)min(i * ROWS + wave * 8 + (lane >> 3), N - 1 - n0) * (unsigned)K * 2u + chunk;
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) void*)lds + wave * 1024;
    auto load = [&](const bf16_t* base, unsigned off, unsigned at) {
        // (written as the instruction: told of it, the compiler waits for every such load before any LDS read)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(off), "s"(base), "s"(lds0 + at) : "memory");
    };
    auto fill = [&](int step, unsigned stage) {
        const int k = k_begin + step * BK;
#pragma unroll
        for (int i = 0; i < LW; i++) load(wb + k, wo[i], stage + (MB + i * ROWS) * 128);
#pragma unroll
        for (int i = 0; i < LX; i++) load(X + k, xo[i], stage + i * ROWS * 128);
    };
    st_f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = (st_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < S - 1; t++)
        if (t < steps) fill(t, t * STAGE);
    unsigned cur = 0, free_ = (S - 1) * STAGE;
    for (int step = 0; step < steps; step++) {
        asm volatile("" ::: "memory");
        if (step + S - 2 < steps) wait_loads<(S - 2) * L>(); else wait_loads<0>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (step + S - 1 < steps) fill(step + S - 1, free_);
        const unsigned char* const xs = lds + cur + (wm * 16 * TM + r) * 128;
        const unsigned char* const ws = lds + cur + (MB + wn * 16 * TN + r) * 128;
        StFrag a[2][TM], b[2][TN];
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const int at = ((4 * s + g) ^ (r & 7)) * 16;
#pragma unroll
            for (int j = 0; j < TN; j++) b[s][j].u = *reinterpret_cast<const uint4*>(ws + j * 2048 + at);
#pragma unroll
            for (int i = 0; i < TM; i++) a[s][i].u = *reinterpret_cast<const uint4*>(xs + i * 2048 + at);
        }
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[s][j].v, a[s][i].v, acc[i][j], 0, 0, 0);
        free_ = cur;
        cur = cur + STAGE == S * STAGE ? 0 : cur + STAGE;
    }
    const int width = EPI == TP_EPI_GATED ? units : N;
    const bool wide = (width & 3) == 0 && ((uintptr_t)Y & 15) == 0;
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int m = wm * 16 * TM + i * 16 + r;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TN; j += EPI == TP_EPI_GATED ? 2 : 1) {
            const int at_n = n0 + (wn * TN + j) * 16, col = (EPI == TP_EPI_GATED ? at_n >> 1 : at_n) + g * 4;
            float o[4];
#pragma unroll
            for (int v = 0; v < 4; v++)
                o[v] = EPI == TP_EPI_GATED ? gated_unit_fast(acc[i][j][v], acc[i][j + 1 < TN ? j + 1 : j][v], epi) : plain_epilogue(EPI, acc[i][j][v], epi, col + v);
            if (col >= width) continue;
            const size_t at = (size_t)m * width + col;
            if (wide) {
                if (out_dtype == TP_F32) *reinterpret_cast<st_f32x4*>((float*)Y + at) = (st_f32x4){o[0], o[1], o[2], o[3]};
                else {
                    ushort4 pk;
                    pk.x = f32_to_bf16(o[0]); pk.y = f32_to_bf16(o[1]); pk.z = f32_to_bf16(o[2]); pk.w = f32_to_bf16(o[3]);
                    *reinterpret_cast<ushort4*>((bf16_t*)Y + at) = pk;
                }
            } else {
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    if (col + v >= width) break;
                    if (out_dtype == TP_F32) ((float*)Y)[at + v] = o[v];
                    else ((bf16_t*)Y)[at + v] = f32_to_bf16(o[v]);
                }
            }
        }
    }
}

bool gemm_stream_supports(const GemmArgs& a) {
    return a.in_dtype == TP_BF16 && a.M <= 64 && a.K % BK == 0 && 128L * a.K * 2 < (1L << 32);
}

struct StreamPlan { int rows, splits, kps; };   // rows of W a block owns, K slices, K of a slice

// What decides is how many steps the busiest CU walks.  K slices, where the consumer adds them: as many as leave the blocks
// within one a CU, none shorter than 512 (2B down, 36 blocks of 64 rows: 4 slices 15.1 us, 7 slices, 252 blocks, 14.8, 8 slices,
// 288 blocks, 17.1; 9B down, 56 blocks: 3 slices 25.0, 4 24.0, 5 30.5).  Without slices 32 rows a block where that gives the
// busiest CU fewer rows and all blocks run at once, three a CU (2B gate/up, 288 blocks of 64 rows or 576 of 32: 21.5 / 18.7 us; 9B,
// 448 or 896, beyond three a CU: 38.0 / 47.1).  128 rows a block from 33 rows of X on, where X's tile costs what W's costs, if
// the busiest CU gets no more rows by it (64 rows of X, logits 262 / 243 us, 9B gate/up 45.6 / 39.7) - but not where rows of W
// lie a multiple of 8 KB apart, when 128 of them meet in the same memory channels (N 32768, K 4096: 58.0 / 65.1).  Where 32 rows a block
// would be three blocks on the fullest CU, one block of 96 gives it the same rows of W and reads X once instead of three times:
// always from 33 rows of X on (32 / 96 rows of W a block, K 2304, 64 rows: N 16512 24.6 / 20.3 us, 17408 26.1 / 22.7, 18432 25.5 / 21.6, 24576 29.0 / 24.5; K 4096,
// N 16896 42.3 / 36.8), below where the CUs have two and a half on average at most (8 rows: N 18432 19.4 / 18.8, 24576 22.6 / 22.9;
// 32 rows, N 18432 20.8 / 19.6).  Its ring is four steps deep, and shorter K keeps the blocks of 32: three and five are slower (8 rows 21.5 and 18.9, 64 rows 22.0 and 22.3).
static StreamPlan stream_plan(const GemmArgs& a) {
    constexpr int CUS = 256, MAX_SPLITS = 16;
    const int blocks = tp_cdiv(a.N, 64), narrow = tp_cdiv(a.N, 32), wide = tp_cdiv(a.N, 128);
    StreamPlan p{64, 1, 0};
    if (a.defer && a.epilogue == TP_EPI_NONE) {
        p.splits = CUS / blocks;
        if (p.splits > a.K / 512) p.splits = a.K / 512;
        if (p.splits > MAX_SPLITS) p.splits = MAX_SPLITS;
        if (p.splits < 1) p.splits = 1;
    }
    p.kps = tp_cdiv(tp_cdiv(a.K, p.splits), BK) * BK;
    p.splits = tp_cdiv(a.K, p.kps);
    if (p.splits == 1) {
        if (a.K >= 4 * BK && narrow > 2 * CUS && tp_cdiv(a.N, 96) <= CUS && (a.M > 32 || 2 * narrow <= 5 * CUS)) p.rows = 96;
        else if (narrow <= 3 * CUS && tp_cdiv(narrow, CUS) < 2 * tp_cdiv(blocks, CUS)) p.rows = 32;
        else if (a.M > 32 && blocks > CUS && a.K % 4096 && 2 * tp_cdiv(wide, CUS) <= tp_cdiv(blocks, CUS)) p.rows = 128;
    }
    return p;
}

int gemm_stream_splits(const GemmArgs& a) { return stream_plan(a).splits; }
// rows of W a block of this kernel owns in a product (0: it is not one of its products)
extern "C" int tp_linear_stream_rows(int M, int N, int K, int epilogue, int defer) {
    GemmArgs a{};
    a.in_dtype = TP_BF16; a.M = M; a.N = N; a.K = K; a.epilogue = epilogue; a.defer = defer;
    return gemm_stream_supports(a) ? stream_plan(a).rows : 0;
}
// One slice is left as float32, too, where the choice of kernel is the library's: a product of so many rows of W that it has
// one slice here had several by the kernels before it, and its sums stay float32 (N 9216, K 2304, 64 rows: error against 64
// bits 1.7e-3 rounded to bf16, 2.9e-7 so).
int gemm_stream_slices_left(const GemmArgs& a) {
    const int s = stream_plan(a).splits;
    return a.defer && (s > 1 || a.algo == 0) ? s : 0;
}

template <int EPI, int MB, int BN, int WAVES, int S, int WN = BN / 32>
static void stream_tile(const GemmArgs& a, void* y, int out_dtype, const StreamPlan& p) {
    gemm_stream_k<EPI, MB, BN, WAVES, S, WN><<<dim3((unsigned)tp_cdiv(a.N, BN), p.splits), 64 * WAVES, 0, a.stream>>>(
        (const bf16_t*)a.x, (const bf16_t*)a.w, y, a.M, a.N, a.K, out_dtype, epi_constants(a), a.units, p.kps);
}

// depths: two blocks a CU (72 to 80 KB of LDS each) but three for 32 rows of W (48 KB); blocks of 96 rows are one a CU by their number
template <int EPI>
static void stream_launch(const GemmArgs& a, void* y, int out_dtype, const StreamPlan& p) {
    if (p.rows == 96) {
        if (a.M <= 32) stream_tile<EPI, 32, 96, 2, 4, 1>(a, y, out_dtype, p);
        else stream_tile<EPI, 64, 96, 4, 4, 1>(a, y, out_dtype, p);
    } else if (p.rows == 32) {
        if (a.M <= 16) stream_tile<EPI, 16, 32, 1, 8>(a, y, out_dtype, p);
        else if (a.M <= 32) stream_tile<EPI, 32, 32, 1, 6>(a, y, out_dtype, p);
        else stream_tile<EPI, 64, 32, 1, 4>(a, y, out_dtype, p);
    } else if (a.M <= 32) stream_tile<EPI, 32, 64, 4, 6>(a, y, out_dtype, p);
    else if (p.rows == 64) stream_tile<EPI, 64, 64, 4, 5>(a, y, out_dtype, p);
    else stream_tile<EPI, 64, 128, 8, 3>(a, y, out_dtype, p);
}

int gemm_stream_launch(const GemmArgs& a) {
    TP_REQUIRE(gemm_stream_supports(a), "product of up to 64 rows: needs bf16 and K a multiple of 64 (M=%d N=%d K=%d)", a.M, a.N, a.K);
    TP_REQUIRE(((uintptr_t)a.x % 16 == 0) && ((uintptr_t)a.w % 16 == 0), "product of up to 64 rows: operands must be 16-byte aligned");
    const StreamPlan p = stream_plan(a);
    const bool slices = gemm_stream_slices_left(a) > 0;
    const size_t need = (size_t)p.splits * a.M * a.N * sizeof(float);
    TP_REQUIRE(!slices || (a.workspace && a.workspace_bytes >= need), "product of up to 64 rows: workspace of %zu bytes, %zu needed", a.workspace_bytes, need);
    void* const y = slices ? a.workspace : a.y;
    const int out_dtype = slices ? TP_F32 : a.out_dtype;
    switch (a.epilogue) {
        case TP_EPI_GATED: stream_launch<TP_EPI_GATED>(a, y, out_dtype, p); break;
        case TP_EPI_SOFTCAP: stream_launch<TP_EPI_SOFTCAP>(a, y, out_dtype, p); break;
        case TP_EPI_RELU2: stream_launch<TP_EPI_RELU2>(a, y, out_dtype, p); break;
        case TP_EPI_SILU: stream_launch<TP_EPI_SILU>(a, y, out_dtype, p); break;
        default: stream_launch<TP_EPI_NONE>(a, y, out_dtype, p);
    }
    return tp_check_launch("linear (up to 64 rows)");
}
