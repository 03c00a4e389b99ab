// float32 products on the matrix cores (v_mfma_f32_16x16x4_f32: float32 operands, products and sums), for few and many rows.
//
// Every output element is formed in one order whatever the batch is, so that a row alone gives the bits it gives among
// others: K is cut into 16 parts of whole blocks of 16 k, a part is one chain of matrix instructions over its blocks (four
// a block: instruction t takes the block's k = t, 4 + t, 8 + t, 12 + t), four neighbouring parts are added in order to a
// group, and the four groups in order.  (Its error against 64 bits is smaller than that of one chain over K.)
//
// Up to 32 rows (a decode step) are bound by reading W.  A block of four waves owns 16 rows of W; a wave takes a group (or, where
// the groups are left to the consumer as slices, a part) and streams W and X through a ring of its own in LDS, three steps of
// 32 k deep, so that three blocks a CU keep 72 KB of W in flight and no wave waits for another before the sums.  Microseconds at
// 3 rows, cold weights, blocks of 16 waves that each asked for six blocks of 16 k in registers (one block a CU, so that its start
// and end were nobody's work) / here: 2B gate/up 53.2 / 35-37 (4.6-4.9 TB/s), down 29.3 / 20.4, o 10.7 / 6.9, qkv 11.8 / 10.3,
// logits 575 / 395 (6.0 TB/s); at 20 rows 74 / 48, 46 / 27, -, 18.7 / 13.9, 783 / 498.  Rings of four to eight steps and fewer
// blocks a CU are slower (gate/up 38-44, qkv 10.9-11.8).
// Operands off 16 bytes, which loads into LDS do not take, keep those blocks of 16 waves for any number of rows: a wave one part,
// six blocks of 16 k of W and X asked for together, the parts added in LDS.
// Many rows are bound by the matrix cores, 157 TFLOP/s in float32: a block of four waves owns 64 x 128 outputs (32 x 64 a
// wave, 32 matrix instructions of 32 cycles for six 16-byte fragment reads), or fewer columns where that leaves the fullest CU
// less, k steps of 32 straight from global memory into one of two LDS buffers, three blocks a CU.  Where the outputs alone leave
// CUs idle and the consumer adds slices, the four groups are four slices.  Microseconds, cold weights, before (accumulators moved
// between register files every 16 k, which also kept the third block out; 128 columns always) / here: 2B at 309 rows gate/up
// 286 / 246, qkv 113 / 73, o 46 / 34, down 172 / 126; at 2,048 rows 1,569 / 1,329 (131 TFLOP/s), 355 / 310, 251 / 158, 1,067 / 654.
#include "gemm.h"

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f3_f32x4;
typedef f3_f32x4 f3_anywhere __attribute__((aligned(4)));        // (the same load: a global one needs no more)

namespace {
constexpr int PARTS = 16, GROUP = 4;
constexpr int TM = 64, TN = 128;                 // of many rows: the outputs a block owns, at most

// until every load, and every LDS read (whose buffer is filled again behind the barrier), is done
__device__ __forceinline__ void wait_all() { __builtin_amdgcn_s_waitcnt(0x0070); }
// until all but the N youngest loads are done; until every LDS read is done
template <int N> __device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14)); }
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07f); }

__device__ __forceinline__ float epilogue_f32(int epilogue, float o, float4 epi, int n) {
    if (epilogue == TP_EPI_SILU) return (float)n < epi.z ? gate_act_exact(o, TP_ACT_SILU) : o;
    return plain_epilogue(epilogue, o, epi, n);
}
}

// NT, MT: tiles of 16 rows of W and of X.  Gated: NT = 2, the gate rows and the up rows of 16 units.
template <int NT, int MT, bool GATED>
__global__ void __launch_bounds__(1024)
gemm_f32_few_k(const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int M, int N, int K, int part_blocks,
               int epilogue, float4 epi, int units, int act) {
    constexpr int AHEAD = NT * MT > 2 ? 4 : 6;             // blocks of 16 k asked for together (the wave's registers hold no more of four tiles)
    __shared__ f3_f32x4 sums[PARTS][NT * MT][64];
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = blockIdx.x * 16 * NT, m0 = blockIdx.y * 16 * MT;
    const int k_blocks = (K + 15) >> 4, from = part * part_blocks, to = min(k_blocks, from + part_blocks);
    const float *wr[NT], *xr[MT];
#pragma unroll
    for (int j = 0; j < NT; j++) wr[j] = W + (size_t)min(n0 + 16 * j + r, N - 1) * K;
#pragma unroll
    for (int i = 0; i < MT; i++) xr[i] = X + (size_t)min(m0 + 16 * i + r, M - 1) * K;
    f3_f32x4 acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[j][i] = (f3_f32x4){0.f, 0.f, 0.f, 0.f};
    for (int b = from; b < to; b += AHEAD) {
        f3_f32x4 w[AHEAD][NT], x[AHEAD][MT];
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            const int k = min(min(b + u, to - 1) * 16 + 4 * g, K - 4);       // past the end: elements that exist, zeroed or unused below
#pragma unroll
            for (int j = 0; j < NT; j++) w[u][j] = *reinterpret_cast<const f3_anywhere*>(wr[j] + k);
#pragma unroll
            for (int i = 0; i < MT; i++) x[u][i] = *reinterpret_cast<const f3_anywhere*>(xr[i] + k);
        }
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            if (b + u >= to) break;
            if ((b + u) * 16 + 16 > K) {                                     // the last, partial block
                const bool in = (b + u) * 16 + 4 * g < K;
#pragma unroll
                for (int v = 0; v < 4; v++) {
#pragma unroll
                    for (int j = 0; j < NT; j++) w[u][j][v] = in ? w[u][j][v] : 0.f;
#pragma unroll
                    for (int i = 0; i < MT; i++) x[u][i][v] = in ? x[u][i][v] : 0.f;
                }
            }
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int i = 0; i < MT; i++)
                        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u][j][t], x[u][i][t], acc[j][i], 0, 0, 0);
        }
    }
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) sums[part][j * MT + i][lane] = acc[j][i];
    __syncthreads();
    // element e of a tile: lane e / 4, register e % 4 of the accumulators: row of X lane % 16, row of W 4 (lane / 16) + register
    auto total = [&](int tile, int e) {
        float t = 0.f;
#pragma unroll
        for (int q = 0; q < PARTS / GROUP; q++) {
            float s = 0.f;
#pragma unroll
            for (int p = 0; p < GROUP; p++) s += reinterpret_cast<const float*>(&sums[q * GROUP + p][tile][0])[e];
            t += s;
        }
        return t;
    };
    for (int idx = threadIdx.x; idx < (GATED ? 1 : NT) * MT * 256; idx += 1024) {
        const int tile = idx >> 8, e = idx & 255, l = e >> 2;
        const int j = GATED ? 0 : tile / MT, i = GATED ? tile : tile % MT;
        const int m = m0 + 16 * i + (l & 15), row = 16 * j + 4 * (l >> 4) + (e & 3);
        if (m >= M) continue;
        if (GATED) {
            const int unit = (n0 >> 1) + row;
            if (unit < units) Y[(size_t)m * units + unit] = gated_unit_exact(total(i, e), total(MT + i, e), act, epi.z, epi.w);
        } else if (n0 + row < N) Y[(size_t)m * N + n0 + row] = epilogue_f32(epilogue, total(tile, e), epi, n0 + row);
    }
}

// Up to 32 rows of operands on 16 bytes.  A wave walks PPW neighbouring parts of K of 16 NT rows of W and 16 MT of X through a
// ring of D steps of 32 k in LDS that it alone fills and reads, so that no wave waits for another before the end: whole lines of
// 128 bytes straight from global memory, a step read into registers and its place asked for again before its products.
// PPW = 4: the four waves' groups are added in LDS; PPW = 1: a block holds one group, its four parts are added in LDS, and
// the groups (blockIdx.y) are the consumer's slices.
// Gated: NT = 1, eight gate rows and the eight up rows of the same units.
template <int NT, int MT, bool GATED, int PPW, int D>
__global__ void __launch_bounds__(256)
gemm_f32_ring_k(const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int M, int N, int K, int part_blocks,
                int epilogue, float4 epi, int units, int act) {
    static_assert(!GATED || NT == 1, "a tile of 16 rows holds gate and up rows of eight units");
    constexpr int STEP = (NT + MT) * 2048, L = (NT + MT) * 2, OUT = NT * MT;
    static_assert(D >= 2 && (D - 1) * L < 64 && OUT <= 4 && D * STEP >= OUT * 1024, "ring");
    __shared__ __attribute__((aligned(16))) unsigned char lds[4 * D * STEP];
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = GATED ? (blockIdx.x >> 1) * 32 : blockIdx.x * 16 * NT;         // the first row of W; gated: of the 32 that the tile's 16 are among
    const int k_blocks = (K + 15) >> 4, part = blockIdx.y * GROUP + wave * PPW;
    const int from = part * part_blocks, to = min(k_blocks, from + PPW * part_blocks), steps = max(0, (to - from + 1) >> 1);

    // loads: 8 rows of 128 bytes an instruction; the place p of row `row` holds chunk p ^ (row / 2), so that the 16 rows of a
    // fragment read lie on all banks; rows past the edge of Y read the last row, chunks past the end of K its last one
    const float* const wb = W + (size_t)n0 * K;
    unsigned wo[NT][2], xo[MT][2];
    int chunk[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int row = h * 8 + (lane >> 3);
        chunk[h] = ((lane & 7) ^ (row >> 1)) * 4;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const int at = GATED ? (blockIdx.x & 1) * 8 + (row & 7) + (row >> 3) * 16 : 16 * j + row;
            wo[j][h] = (unsigned)min(at, N - 1 - n0) * (unsigned)K;
        }
#pragma unroll
        for (int i = 0; i < MT; i++) xo[i][h] = (unsigned)min(16 * i + row, M - 1) * (unsigned)K;
    }
    unsigned char* const ring = lds + wave * D * STEP;
    const unsigned ring0 = (unsigned)(size_t)(__attribute__((address_space(3))) void*)ring;
    auto fill = [&](int step, unsigned place) {
        // (written as the instruction: told of it, the compiler waits for every such load before any LDS read)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const unsigned k = (unsigned)min((from + 2 * step) * 16 + chunk[h], K - 4);
#pragma unroll
            for (int j = 0; j < NT; j++)
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"((wo[j][h] + k) * 4u), "s"(wb), "s"(ring0 + place + j * 2048 + h * 1024) : "memory");
#pragma unroll
            for (int i = 0; i < MT; i++)
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"((xo[i][h] + k) * 4u), "s"(X), "s"(ring0 + place + (NT + i) * 2048 + h * 1024) : "memory");
        }
    };
    f3_f32x4 acc[NT][MT], grp[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[j][i] = grp[j][i] = (f3_f32x4){0.f, 0.f, 0.f, 0.f};
    int part_end = from + part_blocks;
#pragma unroll
    for (int t = 0; t < D; t++)
        if (t < steps) fill(t, t * STEP);
    unsigned place = 0;
    for (int step = 0; step < steps; step++) {
        const int left = steps - 1 - step;                     // steps asked for behind this one, D - 1 at most
        asm volatile("" ::: "memory");
        if (left >= D - 1) wait_loads<(D - 1) * L>();
        else if (left >= D / 2) wait_loads<(D / 2) * L>();
        else wait_loads<0>();
        asm volatile("" ::: "memory");
        f3_f32x4 w[2][NT], x[2][MT];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const unsigned char* const at = ring + place + r * 128 + ((4 * h + g) ^ (r >> 1)) * 16;
#pragma unroll
            for (int j = 0; j < NT; j++) w[h][j] = *reinterpret_cast<const f3_f32x4*>(at + j * 2048);
#pragma unroll
            for (int i = 0; i < MT; i++) x[h][i] = *reinterpret_cast<const f3_f32x4*>(at + (NT + i) * 2048);
        }
        asm volatile("" ::: "memory");
        wait_lds();                                            // the step is in registers: its place may be filled again
        asm volatile("" ::: "memory");
        if (left >= D) fill(step + D, place);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int b = from + 2 * step + h;
            if (b >= to) break;
            if (b * 16 + 16 > K) {                             // the last, partial block
                const bool in = b * 16 + 4 * g < K;
#pragma unroll
                for (int v = 0; v < 4; v++) {
#pragma unroll
                    for (int j = 0; j < NT; j++) w[h][j][v] = in ? w[h][j][v] : 0.f;
#pragma unroll
                    for (int i = 0; i < MT; i++) x[h][i][v] = in ? x[h][i][v] : 0.f;
                }
            }
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int i = 0; i < MT; i++)
                        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[h][j][t], x[h][i][t], acc[j][i], 0, 0, 0);
            if (PPW > 1 && (b + 1 == part_end || b + 1 == to)) {
                part_end += part_blocks;
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int i = 0; i < MT; i++) {
                        grp[j][i] += acc[j][i];
                        acc[j][i] = (f3_f32x4){0.f, 0.f, 0.f, 0.f};
                    }
            }
        }
        place = place + STEP == D * STEP ? 0 : place + STEP;
    }
    // the waves' sums, each in its own ring, which it has read to the end
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) *reinterpret_cast<f3_f32x4*>(ring + (j * MT + i) * 1024 + lane * 16) = PPW > 1 ? grp[j][i] : acc[j][i];
    __syncthreads();
    if (wave >= OUT) return;
    auto total = [&](int l) {
        f3_f32x4 t = (f3_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; q++) t += *reinterpret_cast<const f3_f32x4*>(lds + q * D * STEP + wave * 1024 + l * 16);
        return t;
    };
    const int j = wave / MT, i = wave % MT, m = 16 * i + r, width = GATED ? units : N;
    const int c = GATED ? (n0 >> 1) + (blockIdx.x & 1) * 8 + 4 * g : n0 + 16 * j + 4 * g;
    if (m >= M || c >= width || (GATED && g >= 2)) return;
    f3_f32x4 o = total(lane);
    if (GATED) {
        const f3_f32x4 up = total(lane + 32);
#pragma unroll
        for (int v = 0; v < 4; v++) o[v] = gated_unit_exact(o[v], up[v], act, epi.z, epi.w);
    } else {
#pragma unroll
        for (int v = 0; v < 4; v++) o[v] = epilogue_f32(epilogue, o[v], epi, c + v);
    }
    float* const y = Y + (size_t)blockIdx.y * M * N + (size_t)m * width + c;
    if ((width & 3) == 0 && ((uintptr_t)Y & 15) == 0) *reinterpret_cast<f3_f32x4*>(y) = o;
    else {
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (c + v < width) y[v] = o[v];
    }
}

// NJ: tiles of 16 rows of W a wave holds (32 rows of X by 16 NJ of W); gated: an even number, gate rows and up rows in turn.
template <bool GATED, int NJ>
__global__ void __launch_bounds__(256, 3)
gemm_f32_many_k(const float* __restrict__ X, const float* __restrict__ W, float* __restrict__ Y, int M, int N, int K, int part_blocks,
                int m_tiles, int epilogue, float4 epi, int units, int act) {
    static_assert(!GATED || NJ % 2 == 0, "gate and up rows of a unit lie in two tiles of one wave");
    constexpr int TN = 32 * NJ, BUF = (TM + TN) * 128;
    __shared__ __attribute__((aligned(16))) unsigned char lds[2 * BUF];
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave >> 1, wn = wave & 1;
    const int m0 = (blockIdx.x % m_tiles) * TM, n0 = (blockIdx.x / m_tiles) * TN;
    const bool sliced = gridDim.y > 1;
    const int k_blocks = (K + 15) >> 4;
    const int from = sliced ? blockIdx.y * GROUP * part_blocks : 0, to = sliced ? min(k_blocks, from + GROUP * part_blocks) : k_blocks;
    if (sliced) Y += (size_t)blockIdx.y * M * N;

    // loads: 8 rows of 128 bytes an instruction, lane l's place (row l / 8, place l % 8) holds chunk place ^ (row / 2) of the 16
    // rows that a fragment read takes; rows past the edge of Y read the last row, chunks past the end of K its last one
    const float* const xb = X + (size_t)m0 * K;
    const float* const wb = W + (size_t)n0 * K;
    const int chunk = (lane & 7) ^ ((wave & 1) * 4 + (lane >> 4));
    unsigned xo[2], wo[NJ];
#pragma unroll
    for (int i = 0; i < 2; i++) xo[i] = (unsigned)min(i * 32 + wave * 8 + (lane >> 3), M - 1 - m0) * (unsigned)K;
#pragma unroll
    for (int i = 0; i < NJ; i++) wo[i] = (unsigned)min(i * 32 + wave * 8 + (lane >> 3), N - 1 - n0) * (unsigned)K;
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) void*)lds + wave * 1024;
    auto fill = [&](int b, unsigned buf) {
        const unsigned k = (unsigned)min(b * 16 + chunk * 4, K - 4), to_ = lds0 + buf;
        // (written as the instruction: told of it, the compiler waits for every such load before any LDS read)
#pragma unroll
        for (int i = 0; i < 2; i++)
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"((xo[i] + k) * 4u), "s"(xb), "s"(to_ + i * 4096) : "memory");
#pragma unroll
        for (int i = 0; i < NJ; i++)
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"((wo[i] + k) * 4u), "s"(wb), "s"(to_ + TM * 128 + i * 4096) : "memory");
    };
    f3_f32x4 acc[NJ][2], grp[NJ][2], tot[NJ][2];
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int i = 0; i < 2; i++) grp[j][i] = tot[j][i] = (f3_f32x4){0.f, 0.f, 0.f, 0.f};
    unsigned buf = 0;
    if (from < to) fill(from, 0);
    // One loop body, entered a part at a time: with the parts' ends as branches inside a loop over steps the compiler moved all
    // accumulators between register files every 16 k, and kept a third block from the CU.
    int b = from;
    for (int parts = 1; b < to; parts++) {
        const int part_end = min(to, b + part_blocks);
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int i = 0; i < 2; i++) acc[j][i] = (f3_f32x4){0.f, 0.f, 0.f, 0.f};
        for (; b < part_end; b++) {
            const int h = (b - from) & 1;            // a step of 32 k holds two blocks
            if (h == 0) {
                asm volatile("" ::: "memory");
                wait_all();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();        // the step's tiles are there, and the other buffer has been read by everyone
                asm volatile("" ::: "memory");
                if (b + 2 < to) fill(b + 2, BUF - buf);
            }
            const unsigned at = ((4 * h + g) ^ (r >> 1)) * 16;
            const unsigned char* const xs = lds + buf + (wm * 32 + r) * 128 + at;
            const unsigned char* const ws = lds + buf + TM * 128 + (wn * 16 * NJ + r) * 128 + at;
            f3_f32x4 w[NJ], x[2];
#pragma unroll
            for (int i = 0; i < 2; i++) x[i] = *reinterpret_cast<const f3_f32x4*>(xs + i * 2048);
#pragma unroll
            for (int j = 0; j < NJ; j++) w[j] = *reinterpret_cast<const f3_f32x4*>(ws + j * 2048);
            if (b * 16 + 16 > K) {                   // the last, partial block
                const bool in = b * 16 + 4 * g < K;
#pragma unroll
                for (int v = 0; v < 4; v++) {
#pragma unroll
                    for (int i = 0; i < 2; i++) x[i][v] = in ? x[i][v] : 0.f;
#pragma unroll
                    for (int j = 0; j < NJ; j++) w[j][v] = in ? w[j][v] : 0.f;
                }
            }
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int j = 0; j < NJ; j++)
#pragma unroll
                    for (int i = 0; i < 2; i++) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j][t], x[i][t], acc[j][i], 0, 0, 0);
            if (h) buf = BUF - buf;
        }
        const bool whole = parts % GROUP == 0 || b >= to;
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                grp[j][i] += acc[j][i];
                if (whole) {
                    tot[j][i] += grp[j][i];
                    grp[j][i] = (f3_f32x4){0.f, 0.f, 0.f, 0.f};
                }
            }
    }
    const int width = GATED ? units : N;
    const bool wide = (width & 3) == 0 && ((uintptr_t)Y & 15) == 0;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int m = m0 + wm * 32 + 16 * i + r;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < NJ; j += GATED ? 2 : 1) {
            const int n = n0 + wn * 16 * NJ + 16 * j;
            const int c = (GATED ? n >> 1 : n) + 4 * g;
            f3_f32x4 o;
#pragma unroll
            for (int v = 0; v < 4; v++)
                o[v] = GATED ? gated_unit_exact(tot[j][i][v], tot[j + 1 < NJ ? j + 1 : j][i][v], act, epi.z, epi.w) : epilogue_f32(epilogue, tot[j][i][v], epi, c + v);
            if (c >= width) continue;
            float* const to_ = Y + (size_t)m * width + c;
            if (wide) *reinterpret_cast<f3_f32x4*>(to_) = o;
            else {
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (c + v < width) to_[v] = o[v];
            }
        }
    }
}

// rows read in pieces of four; a tile's rows within 32-bit offsets
bool gemm_f32_supports(const GemmArgs& a) { return a.in_dtype == TP_F32 && a.out_dtype == TP_F32 && a.K % 4 == 0 && a.K < (1 << 23); }

// Up to 32 rows the ring kernel reads W once and its matrix instructions fit into that time; from 33 on whole tiles do the same
// work.  Loads into LDS want operands on 16 bytes: off them any number of rows goes to the blocks of 16 waves, in tiles of 32, so
// that a product's bits do not depend on where its operands lie.
static bool aligned(const GemmArgs& a) { return (uintptr_t)a.x % 16 == 0 && (uintptr_t)a.w % 16 == 0; }
static bool few(const GemmArgs& a) { return a.M <= 32 || !aligned(a); }

// Slices for the consumer: the four groups, where the outputs alone leave CUs idle (up to 32 rows: fewer than two blocks a CU,
// three rows, N 2304: K 2048 9.1 us as one, 7.0 as slices, K 9216 30.0 and 20.4).
int gemm_f32_splits(const GemmArgs& a) {
    if (!a.defer || a.epilogue != TP_EPI_NONE || a.K < 1024) return 1;
    if (a.M <= 32) return aligned(a) && tp_cdiv(a.N, 16) < 512 ? PARTS / GROUP : 1;
    return !few(a) && (long)tp_cdiv(a.M, TM) * tp_cdiv(a.N, TN) < 256 ? PARTS / GROUP : 1;
}

template <int NT, bool GATED>
static void few_launch(const GemmArgs& a, int part_blocks, float4 epi) {
    const dim3 blocks(tp_cdiv(a.N, 16 * NT), tp_cdiv(a.M, a.M <= 16 ? 16 : 32));
    if (a.M <= 16) gemm_f32_few_k<NT, 1, GATED><<<blocks, 1024, 0, a.stream>>>((const float*)a.x, (const float*)a.w, (float*)a.y, a.M, a.N, a.K, part_blocks, a.epilogue, epi, a.units, a.act);
    else gemm_f32_few_k<NT, 2, GATED><<<blocks, 1024, 0, a.stream>>>((const float*)a.x, (const float*)a.w, (float*)a.y, a.M, a.N, a.K, part_blocks, a.epilogue, epi, a.units, a.act);
}

template <int NT, int MT, bool GATED, int PPW, int D>
static void ring_launch(const GemmArgs& a, float* y, int part_blocks, float4 epi) {
    gemm_f32_ring_k<NT, MT, GATED, PPW, D><<<dim3(tp_cdiv(a.N, 16 * NT), PPW == 1 ? PARTS / GROUP : 1), 256, 0, a.stream>>>(
        (const float*)a.x, (const float*)a.w, y, a.M, a.N, a.K, part_blocks, a.epilogue, epi, a.units, a.act);
}

int gemm_f32_launch(const GemmArgs& a) {
    const int part_blocks = tp_cdiv(tp_cdiv(a.K, 16), PARTS), splits = gemm_f32_splits(a);
    const bool gated = a.epilogue == TP_EPI_GATED;
    const float4 epi = gated ? make_float4(0.f, 0.f, a.limit, a.shift) : make_float4(a.cap, 0.f, (float)a.units, 0.f);
    const size_t need = (size_t)splits * a.M * a.N * sizeof(float);
    TP_REQUIRE(splits == 1 || (a.workspace && a.workspace_bytes >= need), "float32 product: workspace of %zu bytes, %zu needed", a.workspace_bytes, need);
    float* const y = (float*)(splits > 1 ? a.workspace : a.y);
    if (a.M <= 32 && aligned(a)) {
        // depths: three blocks a CU (48 KB of LDS each, two where two tiles of each are held)
        if (a.M <= 16) {
            if (gated) ring_launch<1, 1, true, 4, 3>(a, y, part_blocks, epi);
            else if (splits > 1) ring_launch<1, 1, false, 1, 3>(a, y, part_blocks, epi);
            else ring_launch<1, 1, false, 4, 3>(a, y, part_blocks, epi);
        } else if (gated) ring_launch<1, 2, true, 4, 2>(a, y, part_blocks, epi);
        else if (splits > 1) ring_launch<1, 2, false, 1, 2>(a, y, part_blocks, epi);
        // two tiles of W share X's where that leaves two blocks a CU (20 rows, N 256000 K 2304: 540 us with one, 498; N 4096: 13.9, 18.8)
        else if (a.N >= 32 * 512) ring_launch<2, 2, false, 4, 2>(a, y, part_blocks, epi);
        else ring_launch<1, 2, false, 4, 2>(a, y, part_blocks, epi);
        return tp_check_launch("linear (float32, up to 32 rows)");
    }
    if (few(a)) {                                              // off 16 bytes
        TP_REQUIRE(a.y, "float32 product: K slices are left of operands on 16 bytes only");
        constexpr long MOST = 65535L * 32;                 // rows that one launch takes
        for (long m = 0; m < a.M; m += MOST) {
            GemmArgs rows = a;
            rows.M = (int)(a.M - m < MOST ? a.M - m : MOST);
            rows.x = (const float*)a.x + (size_t)m * a.K;
            rows.y = (float*)a.y + (size_t)m * (gated ? a.units : a.N);
            // two tiles of W share the block's X where that leaves two blocks a CU
            if (gated) few_launch<2, true>(rows, part_blocks, epi);
            else if (a.N >= 32 * 512) few_launch<2, false>(rows, part_blocks, epi);
            else few_launch<1, false>(rows, part_blocks, epi);
        }
        return tp_check_launch("linear (float32, few rows)");
    }
    const int m_tiles = tp_cdiv(a.M, TM);
    TP_REQUIRE((long)m_tiles * tp_cdiv(a.N, TN) < (1L << 31), "float32 product: too many tiles for one launch (M=%d N=%d)", a.M, a.N);
    // The matrix cores of the CU with the most outputs decide: 128 rows of W a block, or 96 (gated: 64) where the fullest CU gets
    // less by it.  Blocks of 128 tie.
    const int narrow = gated ? 2 : 3;
    auto most = [&](int nj) { return (long)tp_cdiv((long)m_tiles * tp_cdiv(a.N, 32 * nj) * splits, 256) * nj; };
    const int nj = most(narrow) < most(4) ? narrow : 4;
    const dim3 grid((unsigned)(m_tiles * tp_cdiv(a.N, 32 * nj)), splits);
#define TP_MANY(GATED, NJ) gemm_f32_many_k<GATED, NJ><<<grid, 256, 0, a.stream>>>((const float*)a.x, (const float*)a.w, y, a.M, a.N, a.K, part_blocks, m_tiles, a.epilogue, epi, a.units, a.act)
    if (gated) { if (nj == 4) TP_MANY(true, 4); else TP_MANY(true, 2); }
    else { if (nj == 4) TP_MANY(false, 4); else TP_MANY(false, 3); }
#undef TP_MANY
    return tp_check_launch("linear (float32)");
}
