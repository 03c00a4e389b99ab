// bf16 product for many rows on blocks of 8 waves, one block a CU: tiles of up to 256 x 256 outputs, fp32 accumulation.
//
// What bounds it.  A tile of 128 x 128 (gemm_mfma.hip) needs 62 bytes a clock from L2 at the matrix peak, and a CU's path
// takes 64; one of 256 x 256 needs half of that.  Its 2,048 matrix cycles a k step of 64 then have to cover 64 loads of a
// kilobyte into LDS (about 20 cycles each in the path), 192 KB of fragment reads and a barrier.  Measured on an 8,192^3
// product, cycles a step: matrix instructions alone 2,140, with fragment reads 2,220, with loads bunched in half of the step
// 2,780, spread over all of it 2,450.  The clock is a second bound: under this load the chip's power holds it at 1.7 - 1.9 GHz
// (2.4 without), so on random numbers the matrix instructions alone reach 1.65 to 1.70 PFLOP/s here.
// Hence the layout:
// * Eight waves, two a SIMD, in WM x 8/WM, each MT x NT tiles of v_mfma_f32_32x32x16_bf16 with W as the A operand: a lane ends
//   up with four neighbours of a row of Y, and with gate and up column of a unit in one accumulator.  Fragments of the next
//   16 k are read between the matrix instructions of this 16 k, one after each.
// * The loads are asked for evenly over the step (waves of odd number half a slot later), because the path takes one about
//   every 20 cycles and a wave that finds it busy cannot issue its matrix instructions either.  That needs places free over the
//   whole step: three for W's tile, two (256 rows of X) or three for X's.
// * One barrier a step, set between the matrix instructions of its last 16 k, when the fragments that it waits for have long
//   been asked for: at it a step's places become free, and the next step's tiles have arrived.
// * Outputs leave through LDS in whole 16-byte pieces of rows.  As the accumulators lie (8 bytes of 32 rows a store) the stores
//   alone took 13,000 cycles of a 256 x 256 tile, a tenth of a product with K = 2,304.
// Two groups of four waves that take turns at the matrix cores (a barrier a phase) reached 1,230 TFLOP/s where this loop reaches
// 1,305 (9B gate/up at 8,191 rows); four waves of 128 x 128 with one a SIMD 1,170; k steps of 32 in five places 1,170.
//
// Microseconds, cold weights, gemm_mfma.hip / here / the vendor library's plain product (measured beside, never called):
//   2B   2,048 rows: gate/up 180 / 154 / -    qkv 50 / 38 / 41    o 35 / 27 / 26    down (K slices, with their sum) 115 / 102 / -
//   9B   8,191 rows: gate/up 1,455 / 1,290 / -    qkv 433 / 368 / 315    o 233 / 192 / 165    down 875 / 670 / 665
//   2B logits, 1,716 rows, float32: 2,130 / 1,880 / -
// The library is 1.17 times faster at 9B qkv and o, and only a little of that is known: the fixed part of a tile (its first loads, its
// outputs) is 4 of the 92 us of each of qkv's four rounds, and o's second round fills 192 of the 256 CUs.
#include "gemm.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 wd_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 wd_bf16x4;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float wd_f32x16;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float wd_f32x4;

namespace {
constexpr int BK = 64, KSUB = BK / 16;                    // k step; an LDS row is one step long, 128 bytes
union WdFrag { uint4 u; wd_bf16x8 v; };

// s_waitcnt with the counters that are not named left alone
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07f); }
template <int N> __device__ __forceinline__ void wait_vm() { __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14)); }
__device__ __forceinline__ void block_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// 32 rows of a wave's outputs: out of the accumulators into the wave's own stretch of LDS (rows of PITCH bytes), and from
// there to Y in whole 16-byte pieces, neighbouring lanes writing neighbouring pieces of a row.
template <int EPI, int NT, bool F32>
__device__ __forceinline__ void store_rows(const wd_f32x16 (&acc)[NT], unsigned char* mine, void* __restrict__ Y, int m_first, int c_first,
                                           int M, int width, int lane, float4 epi) {
    constexpr int COLS = EPI == TP_EPI_GATED ? NT * 16 : NT * 32, SIZE = F32 ? 4 : 2, PER = 16 / SIZE, PIECES = COLS / PER, PITCH = COLS * SIZE + 16;
    const int l32 = lane & 31, hi = lane >> 5;
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int q = 0; q < (EPI == TP_EPI_GATED ? 2 : 4); q++) {
            wd_f32x4 o;
            const int c = (EPI == TP_EPI_GATED ? j * 16 : j * 32) + 8 * q + 4 * hi;
#pragma unroll
            for (int v = 0; v < 4; v++)
                o[v] = EPI == TP_EPI_GATED ? gated_unit_fast(acc[j][4 * q + v], acc[j][(4 * q + v + 8) & 15], epi)
                                           : plain_epilogue(EPI, acc[j][4 * q + v], epi, c_first + c + v);
            if (F32) *reinterpret_cast<wd_f32x4*>(mine + l32 * PITCH + c * 4) = o;
            else *reinterpret_cast<wd_bf16x4*>(mine + l32 * PITCH + c * 2) = __builtin_convertvector(o, wd_bf16x4);
        }
    const bool whole = width % PER == 0 && ((uintptr_t)Y & 15) == 0;      // an output may start anywhere
#pragma unroll
    for (int t = 0; t < PIECES / 2; t++) {
        const int idx = t * 64 + lane, row = idx / PIECES, piece = idx % PIECES, m = m_first + row, c = c_first + piece * PER;
        const uint4 v = *reinterpret_cast<const uint4*>(mine + row * PITCH + piece * 16);
        if (m >= M || c >= width) continue;
        unsigned char* const to = (unsigned char*)Y + ((size_t)m * width + c) * SIZE;
        if (whole) *reinterpret_cast<uint4*>(to) = v;
        else {
            const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < PER; e++) {
                if (c + e >= width) break;
                if (F32) ((unsigned*)to)[e] = w[e & 3];
                else ((bf16_t*)to)[e] = (bf16_t)(w[e >> 1] >> (16 * (e & 1)));
            }
        }
    }
}
// the slot (between matrix instructions) in which a wave asks for load q of P in a sub-step of SL slots
__device__ constexpr int slot_of(int q, int P, int SL, int odd) { return q * SL / P + (odd ? SL / P / 2 : 0); }
}

template <int EPI, int MT, int NT, int WM, int NX>
__global__ void __launch_bounds__(512, 2)
gemm_wide_k(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W, void* __restrict__ Y, int M, int N, int K,
            int m_tiles, int out_dtype, float4 epi, int units, int k_per_split, int panel) {
    constexpr int WN = 8 / WM, BM = 32 * MT * WM, BN = 32 * NT * WN, PX = BM * 128, PW = BN * 128, NW = 3;
    constexpr int LX = BM / 64, LW = BN / 64, SL = MT * NT;   // loads of a wave a step (64 rows each over the waves); slots of a sub-step
    static_assert(NX * PX + NW * PW <= 160 * 1024, "the places fit the LDS of a CU");
    __shared__ __attribute__((aligned(16))) unsigned char lds[NX * PX + NW * PW];
    const int lane = threadIdx.x & 63, l32 = lane & 31, hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave % WM, wn = wave / WM;

    // an XCD takes a contiguous range of the tiles, walked in panels of `panel` N tiles, N fastest
    int mt, nt;
    {
        const int total = gridDim.x, base = total >> 3, rem = total & 7, xcd = blockIdx.x & 7;
        const int vb = xcd * base + min(xcd, rem) + (blockIdx.x >> 3);
        const int n_tiles = total / m_tiles, per_panel = panel * m_tiles, p = vb / per_panel, q = vb - p * per_panel;
        const int width = min(panel, n_tiles - p * panel);
        nt = p * panel + q % width;
        mt = q / width;
    }
    const int m0 = mt * BM, n0 = nt * BN;
    const int k_begin = blockIdx.y * k_per_split, k_end = min(K, k_begin + k_per_split);
    if (gridDim.y > 1) Y = (float*)Y + (size_t)blockIdx.y * M * N;
    const int steps = (k_end - k_begin) / BK;

    // ---- loads: one instruction of a wave brings 8 rows of 128 bytes straight into LDS; lane l's place is (row l / 8, place
    // l % 8), and the chunk that belongs there is place ^ (row / 2) % 8: the 16 rows of 128 bytes that a fragment read takes at a time
    // then lie on all banks (place ^ row % 8 has two on each: 9B at 8,191 rows, gate/up 1,358 / 1,345 us, down 730 / 721).  Rows past
    // the edge of Y read the last row (their products are not stored).
    unsigned xo[LX], wo[LW];
    const unsigned chunk = (unsigned)((lane & 7) ^ ((wave & 1) * 4 + (lane >> 4))) * 16u;
#pragma unroll
    for (int i = 0; i < LX; i++) xo[i] = (unsigned)min(m0 + i * 64 + wave * 8 + (lane >> 3), M - 1) * (unsigned)K * 2u + chunk;
#pragma unroll
    for (int i = 0; i < LW; i++) wo[i] = (unsigned)min(n0 + i * 64 + wave * 8 + (lane >> 3), N - 1) * (unsigned)K * 2u + chunk;
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) void*)lds + wave * 1024;
    auto load = [&](const bf16_t* base, unsigned off, unsigned place, int i) {
        // (written as the instruction: told of it, the compiler waits for every such load before any LDS read)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(off), "s"(base), "s"(lds0 + place + i * 8192) : "memory");
    };
    auto load_x = [&](int step, unsigned place, int i) { load(X + k_begin + step * BK, xo[i], place, i); };
    auto load_w = [&](int step, unsigned place, int i) { load(W + k_begin + step * BK, wo[i], place, i); };
    // ---- fragments: row l % 32 of 32 rows, k chunk 2 s + l / 32 of the step; in the order they are used
    int at[KSUB];
#pragma unroll
    for (int s = 0; s < KSUB; s++) at[s] = l32 * 128 + (((2 * s + hi) ^ ((l32 >> 1) & 7)) << 4);
    WdFrag fa[2][MT], fb[2][NT];
    auto read = [&](unsigned px, unsigned pw, int s, int i) {
        const bool w = i == 0 || (i >= 2 && i <= NT);
        const int ix = w ? (i == 0 ? 0 : i - 1) : (i == 1 ? 0 : i - NT);
        if (w) fb[s & 1][ix].u = *reinterpret_cast<const uint4*>(lds + pw + (wn * 32 * NT + ix * 32) * 128 + at[s]);
        else fa[s & 1][ix].u = *reinterpret_cast<const uint4*>(lds + px + (wm * 32 * MT + ix * 32) * 128 + at[s]);
    };
    wd_f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;

    // a step's tile of X has one of NX places, its tile of W one of NW, in turn: px, pw this step's, x1, w1 the next one's;
    // xl, wl the last ones', which are those of the step before
    unsigned px = 0, x1 = PX, xl = (NX - 1) * PX, pw = NX * PX, w1 = pw + PW, wl = pw + 2 * PW;
    constexpr int HX = LX / 2, HW = LW / 2, BS = SL * 3 / 8;
#pragma unroll
    for (int i = 0; i < LX; i++) load_x(0, px, i);
#pragma unroll
    for (int i = 0; i < LW; i++) load_w(0, pw, i);
    if (steps > 1) {
#pragma unroll
        for (int i = 0; i < LW; i++) load_w(1, w1, i);
        if (NX == 3) {
#pragma unroll
            for (int i = 0; i < LX; i++) load_x(1, x1, i);
        }
    }
    if (NX - 1 < steps) {
#pragma unroll
        for (int i = 0; i < HX; i++) load_x(NX - 1, xl, i);
        wait_vm<LW + (NX - 2) * LX + HX>();
    } else wait_vm<0>();
    block_barrier();
#pragma unroll
    for (int i = 0; i < MT + NT; i++) read(px, pw, 0, i);
    for (int step = 0; step < steps; step++) {
        const bool more2 = step + 2 < steps;
#pragma unroll
        for (int s = 0; s < KSUB; s++) {
            // the loads of this sub-step: into the place of X that the step frees, in two parts, then into that of W
            const int first = s == KSUB - 1 ? 0 : s == 0 ? HX : s == 1 ? 0 : HW;
            const int last = s == KSUB - 1 ? HX : s == 0 ? LX : s == 1 ? HW : LW;
            const int from = s == KSUB - 1 ? BS : 0;
            const bool on = s == KSUB - 1 ? step + NX < steps : s == 0 ? step + NX - 1 < steps : more2;
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    const int n = i * NT + j;
                    if (s + 1 < KSUB) {
                        if (n < MT + NT) read(px, pw, s + 1, n);
                    } else if (n >= BS) {
                        if (n == BS) {
                            if (more2) wait_vm<LW + (NX - 2) * LX>(); else wait_vm<0>();   // the next step's tiles have arrived ...
                            wait_lds();                        // ... and this step's last fragments are in registers,
                            block_barrier();                   // everyone's: the step's places may be refilled
                        }
                        if (2 * (n - BS) < MT + NT) read(x1, w1, 0, 2 * (n - BS));
                        if (2 * (n - BS) + 1 < MT + NT) read(x1, w1, 0, 2 * (n - BS) + 1);
                    }
                    if (on)
#pragma unroll
                        for (int q = first; q < last; q++)
                            if (n == from + ((wave & 1) ? slot_of(q - first, last - first, SL - from, 1) : slot_of(q - first, last - first, SL - from, 0))) {
                                if (s == KSUB - 1) load_x(step + NX, px, q);
                                else if (s == 0) load_x(step + NX - 1, xl, q);
                                else load_w(step + NW - 1, wl, q);
                            }
                    __builtin_amdgcn_sched_barrier(0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[s & 1][j].v, fa[s & 1][i].v, acc[i][j], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
        const unsigned ox = px, ow = pw;
        px = x1; x1 = NX == 3 ? xl : ox; xl = ox;
        pw = w1; w1 = wl; wl = ow;
    }
    wait_lds();
    block_barrier();                                           // the places become the waves' stretches for the outputs
    constexpr int STRETCH = 32 * (NT * 32 * 4 + 16);
    static_assert(8 * STRETCH <= NX * PX + NW * PW, "the waves' stretches fit the places");
    const int width = EPI == TP_EPI_GATED ? units : N;
    const int c_first = EPI == TP_EPI_GATED ? (n0 + wn * 32 * NT) >> 1 : n0 + wn * 32 * NT;
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int m_first = m0 + wm * 32 * MT + 32 * i;
        if (out_dtype == TP_F32) store_rows<EPI, NT, true>(acc[i], lds + wave * STRETCH, Y, m_first, c_first, M, width, lane, epi);
        else store_rows<EPI, NT, false>(acc[i], lds + wave * STRETCH, Y, m_first, c_first, M, width, lane, epi);
    }
}

template <int EPI, int MT, int NT, int WM, int NX>
static void wide_launch(const GemmArgs& a, void* y, int out_dtype, int splits, int kps) {
    const int m_tiles = tp_cdiv(a.M, 32 * MT * WM), n_tiles = tp_cdiv(a.N, 32 * NT * (8 / WM));
    gemm_wide_k<EPI, MT, NT, WM, NX><<<dim3((unsigned)(m_tiles * n_tiles), splits), 512, 0, a.stream>>>(
        (const bf16_t*)a.x, (const bf16_t*)a.w, y, a.M, a.N, a.K, m_tiles, out_dtype, epi_constants(a), a.units, kps, 4);
}

int gemm_wide_launch(const GemmArgs& a, int shape, bool slices, int splits, int kps) {
    void* y = slices ? a.workspace : a.y;
    const int out_dtype = slices ? TP_F32 : a.out_dtype;
#define TP_WIDE(EPI) do { \
        if (shape == TP_WIDE_256x256) wide_launch<EPI, 4, 2, 2, 2>(a, y, out_dtype, splits, kps); \
        else if (shape == TP_WIDE_256x192) wide_launch<EPI, 2, 3, 4, 2>(a, y, out_dtype, splits, kps); \
        else if (shape == TP_WIDE_192x256) wide_launch<EPI, 3, 2, 2, 2>(a, y, out_dtype, splits, kps); \
        else wide_launch<EPI, 2, 2, 4, 3>(a, y, out_dtype, splits, kps); } while (0)
    switch (a.epilogue) {
        case TP_EPI_GATED: TP_WIDE(TP_EPI_GATED); break;
        case TP_EPI_SOFTCAP: TP_WIDE(TP_EPI_SOFTCAP); break;
        case TP_EPI_RELU2: TP_WIDE(TP_EPI_RELU2); break;
        case TP_EPI_SILU: TP_WIDE(TP_EPI_SILU); break;
        default: TP_WIDE(TP_EPI_NONE);
    }
#undef TP_WIDE
    return tp_check_launch("linear (wide tiles)");
}
