// Entry points of the matrix products and the plain tiled kernel.
//
// The plain kernel (every output element summed over k in index order whatever the batch is) is the fallback of both paths for
// shapes that the matrix-core kernels refuse: a K that is no multiple of 4 (float32) or 8 (bf16).  The reference's products are 4-bit codebook GEMVs
// (runtime/cuda/codebook_gemv.cu:86-114); its only dense one is gemv_fp16_warp_k (cu:496-517).
#include "gemm.h"

// A block of 16 x 16 threads owns a tile of 16 R x 16 R outputs, R x R per thread, and walks K in steps of BK
// through LDS.  Every output is one chain acc = fma(x, w, acc) over k = 0, 1, 2, ...: the same bits for every R,
// BK and batch.  R = 4 for many rows; R = 1 (sixteen times the blocks, whole 256-byte pieces of a row per load)
// for the few rows of a decode step, where a narrow product would otherwise run on a few dozen blocks.
template <typename TI, typename TO, int R, int BK>
__global__ void __launch_bounds__(256)
gemm_simple_k(const TI* __restrict__ X, const TI* __restrict__ W, TO* __restrict__ Y, int M, int N, int K, int epilogue, float4 epi) {
    constexpr int T = 16 * R;
    __shared__ float xs[BK][T + 1];
    __shared__ float ws[BK][T + 1];
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
    float acc[R][R] = {};
    for (int k0 = 0; k0 < K; k0 += BK) {
#pragma unroll
        for (int i = 0; i < T * BK / 256; i++) {
            const int idx = tid + i * 256, r = idx / BK, kk = idx % BK;
            const int k = k0 + kk;
            xs[kk][r] = (m0 + r < M && k < K) ? ld_f32(X + (size_t)(m0 + r) * K + k) : 0.f;
            ws[kk][r] = (n0 + r < N && k < K) ? ld_f32(W + (size_t)(n0 + r) * K + k) : 0.f;
        }
        __syncthreads();
#pragma unroll 16
        for (int kk = 0; kk < BK; kk++) {
            float a[R], b[R];
#pragma unroll
            for (int i = 0; i < R; i++) { a[i] = xs[kk][ty * R + i]; b[i] = ws[kk][tx * R + i]; }
#pragma unroll
            for (int i = 0; i < R; i++)
#pragma unroll
                for (int j = 0; j < R; j++) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < R; i++) {
        const int m = m0 + ty * R + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < R; j++) {
            const int n = n0 + tx * R + j;
            if (n >= N) continue;
            st_f32(Y + (size_t)m * N + n, epilogue == TP_EPI_SILU ? ((float)n < epi.z ? gate_act_exact(acc[i][j], TP_ACT_SILU) : acc[i][j])
                                                                      : plain_epilogue(epilogue, acc[i][j], epi, n));
        }
    }
}

extern "C" int tp_gated_act(const float* y, void* out, int dtype, int M, int I, int act, float limit, float shift, void* stream);

template <typename TI>
static int simple_typed(const GemmArgs& a, void* y, int out_dtype, int epilogue) {
    const float4 epi = make_float4(a.cap, 0.f, (float)a.units, 0.f);
    if (a.M <= 16) {
        dim3 grid(tp_cdiv(a.N, 16), 1);
        if (out_dtype == TP_F32)
            gemm_simple_k<TI, float, 1, 64><<<grid, 256, 0, a.stream>>>((const TI*)a.x, (const TI*)a.w, (float*)y, a.M, a.N, a.K, epilogue, epi);
        else
            gemm_simple_k<TI, bf16_t, 1, 64><<<grid, 256, 0, a.stream>>>((const TI*)a.x, (const TI*)a.w, (bf16_t*)y, a.M, a.N, a.K, epilogue, epi);
        return tp_check_launch("linear (plain kernel, few rows)");
    }
    dim3 grid(tp_cdiv(a.N, 64), tp_cdiv(a.M, 64));
    if (out_dtype == TP_F32)
        gemm_simple_k<TI, float, 4, 16><<<grid, 256, 0, a.stream>>>((const TI*)a.x, (const TI*)a.w, (float*)y, a.M, a.N, a.K, epilogue, epi);
    else
        gemm_simple_k<TI, bf16_t, 4, 16><<<grid, 256, 0, a.stream>>>((const TI*)a.x, (const TI*)a.w, (bf16_t*)y, a.M, a.N, a.K, epilogue, epi);
    return tp_check_launch("linear (plain kernel)");
}

int gemm_simple_launch(const GemmArgs& a) {
    void* y = a.y;
    int out_dtype = a.out_dtype;
    if (a.epilogue == TP_EPI_GATED) {
        TP_REQUIRE(a.workspace && a.workspace_bytes >= (size_t)a.M * a.N * 4, "gated product: workspace of %zu bytes is too small", a.workspace_bytes);
        y = a.workspace;
        out_dtype = TP_F32;
    }
    const int epilogue = a.epilogue == TP_EPI_GATED ? TP_EPI_NONE : a.epilogue;     // the activation of a gated product is a launch of its own here
    int rc = a.in_dtype == TP_BF16 ? simple_typed<bf16_t>(a, y, out_dtype, epilogue) : simple_typed<float>(a, y, out_dtype, epilogue);
    if (rc) return rc;
    if (a.epilogue == TP_EPI_GATED) return tp_gated_act((const float*)y, a.y, a.out_dtype, a.M, a.units, a.act, a.limit, a.shift, a.stream);
    return 0;
}

static int check_args(const GemmArgs& a) {
    TP_REQUIRE(a.M > 0 && a.N > 0 && a.K > 0, "linear: empty shape M=%d N=%d K=%d", a.M, a.N, a.K);
    TP_REQUIRE(a.in_dtype == TP_F32 || a.in_dtype == TP_BF16, "linear: unknown input dtype %d", a.in_dtype);
    TP_REQUIRE(a.out_dtype == TP_F32 || a.out_dtype == TP_BF16, "linear: unknown output dtype %d", a.out_dtype);
    TP_REQUIRE(!(a.in_dtype == TP_F32 && a.out_dtype == TP_BF16), "linear: float32 rows give float32 output");
    TP_REQUIRE(a.epilogue != TP_EPI_SOFTCAP || a.cap > 0.f, "linear: a soft cap must be positive");
    TP_REQUIRE(a.epilogue != TP_EPI_SILU || (a.units > 0 && a.units <= a.N && a.N < (1 << 24)), "linear: SiLU on the first %d of %d columns", a.units, a.N);
    TP_REQUIRE(!a.defer || a.epilogue == TP_EPI_NONE, "linear: K slices can be left to the consumer only without an epilogue (found %d)", a.epilogue);
    if (a.epilogue == TP_EPI_GATED) {
        const int padded = 2 * ((a.units + 15) / 16) * 16;
        TP_REQUIRE(a.units > 0 && a.N == padded, "gated product: %d units need a packed matrix of %d rows, found %d", a.units, padded, a.N);
        float c1, c3;
        TP_REQUIRE(tp_gate_constants(a.act, &c1, &c3), "gated product: activation %d is none of gelu-tanh (%d), SiLU (%d), ReLU (%d), g sigmoid(1.702 g) (%d)", a.act, TP_ACT_GELU_TANH, TP_ACT_SILU, TP_ACT_RELU, TP_ACT_QUICK_GELU);
        TP_REQUIRE(a.limit > 0.f, "gated product: the limit of the sums must be positive (infinity for none), found %g", (double)a.limit);
    }
    return 0;
}

// algo: 0 = choose, 1 = plain, 2 = skinny matrix-core, 3 = tiled matrix-core (6: with its wide tile, 7: with its 128 x 96 tile,
// 8, 9: with its loop that loads straight into LDS, 128 x 128 and 128 x 96; 10, 11: its 64 x 32 and 64 x 64 tiles with two k
// steps asked for ahead; 12 - 15: with the wide tiles of TP_WIDE_*), 16 = its own kernel for
// up to 64 rows that streams W through LDS, 4 = multiply-adds for one or two rows, 5 = matrix-core kernel for up to eight rows.  (float32: 1, or chosen.)
static int pick(const GemmArgs& a, int algo) {
    if (algo == 1) return 1;
    if (algo == 4) return gemv_supports(a) ? 4 : -4;
    if (algo == 5) return gemm_rows8_supports(a) ? 5 : -5;
    if (algo == 16) return gemm_stream_supports(a) ? 16 : -16;
    if (algo == 2) return gemm_skinny_supports(a) ? 2 : -2;
    if (algo == 3 || (algo >= 6 && algo <= 15)) return gemm_mfma_supports(a) ? 3 : -3;
    if (a.in_dtype == TP_F32) return gemm_f32_supports(a) ? 20 : 1;
    // Two to 64 rows, K a multiple of 64: the kernel that streams W through LDS, wherever enough blocks of it read at once
    // (its figures beside its plan).  With K slices for the consumer that is nearly always (2 rows, against the multiply-adds: 9B
    // down 27.6 / 23.8 us, qkv 15.3 / 12.8, 2B down 16.1 / 14.5).  Up to eight rows of a small matrix are the exception: its blocks
    // of 64 rows and slices of 512 k are too few to fetch it, and the kernels that start a wave every 2 or 8 rows of W are faster,
    // up to FEW_N rows of W at any K but the longest, beyond up to SMALL_NK elements (with the norm that adds the slices, stream /
    // 8-row kernel at 3 rows: N 256 K 2304 7.5 / 6.0 us, N 1024 K 4608 12.7 / 11.1, N 1536 K 2048 8.0 / 7.5; N 2304 K 2048 8.3 / 8.3,
    // N 1024 K 14336 18.1 / 23.2, N 2304 K 4608 11.5 / 12.0).  Two rows stay with the multiply-adds where those cut K as well,
    // up to SMALL_TWO_NK elements (N 384 K 9216 10.3 / 8.2, N 2048 K 3072 9.5 / 9.1, N 2560 K 3584 11.0 / 11.0); where they would
    // not, their one slice would be rounded to bf16, and the 8-row kernel takes the same time.
    // Without slices this kernel is the choice from 128 blocks of 64 rows of W on (8 rows, N 9216 K 2304: 13.2 / 11.8; 16 rows 21.4 / 13.0; but 8 rows, N 4096: 6.5 / 9.1).  A single row stays with the multiply-adds (2B down
    // 14.4 / 14.3, gate/up 16.6 / 18.6), and products without slices with the multiply-adds for two rows (2B gate/up 17.5 / 18.7)
    // and the 8-row kernel for three to seven where that reads K in one round, gates, or has the logits' many rows (2B gate/up
    // 17.2 / 18.7 at 4 rows, 18.2 / 18.7 at 6; logits 189 / 199).
    constexpr int ONE_ROUND_K = TP_R8_MAX_STEPS * 256, WIDE_N = 64 * 512, STREAM_N = 64 * 127;
    constexpr int FEW_N = 1024, FEW_N_K = 9216;
    constexpr long SMALL_NK = 1L << 22, SMALL_TWO_NK = 8000000;
    const bool sliced = a.defer && a.epilogue == TP_EPI_NONE;
    if (gemm_stream_supports(a) && a.M > 1) {
        const bool rows8 = a.M < 8 && gemm_rows8_supports(a) && (a.epilogue == TP_EPI_GATED || a.K <= ONE_ROUND_K || a.N >= WIDE_N);
        const bool slices = sliced && gemm_stream_splits(a) > 1;
        if (slices && a.M <= 8) {
            const long elements = (long)a.N * a.K;
            if (gemv_supports(a) && gemv_workspace(a) && (a.N <= FEW_N || elements <= SMALL_TWO_NK)) return 4;
            if (gemm_rows8_supports(a) && ((a.N <= FEW_N && a.K <= FEW_N_K) || elements <= SMALL_NK)) return 5;
        }
        if (slices || (a.N > STREAM_N && (a.M > 2 || !gemv_supports(a)) && !rows8)) return 16;
    }
    if (gemv_supports(a)) return 4;          // one or two rows: 2B gate/up 16.8 against 22.6 us on the skinny kernel
    // What is left: few rows of W, or K no multiple of 64.  Three to eight rows: the kernel whose blocks read 8 rows of W in one
    // go, where it was measured faster than the choice below.  The bounds in the kernels' own terms:
    //   ONE_ROUND_K  the K a block of the 8-row kernel reads in one round of loads (TP_R8_MAX_STEPS steps of 64 k by four
    //                waves): beyond it the kernel loops, and a slice of K left to the consumer keeps it within one round;
    //   WIDE_N       from here on a product is the logits' kind: so many rows of W that the tiled kernel's 64 x 64 tiles
    //                fill every CU several times over (512 tiles = two a CU) and its larger k steps win;
    //   LARGE_NK     elements of W from which the tiled kernel's streaming wins at 8 rows and more, measured between 21 M (the
    //                8-row kernel wins) and 42 M (the tiled kernel wins);
    //   R8_SLICED_NK elements of W up to which the 8-row kernel, its K in slices for the consumer, beat the tiled kernel
    //                in a whole step.
    constexpr long LARGE_NK = 24000000, R8_SLICED_NK = 32000000;
    if (a.M <= 8 && gemm_rows8_supports(a)) {
        if (sliced) {
            if ((long)a.N * a.K <= R8_SLICED_NK) return 5;
        } else if (a.M < 8) {
            if (a.epilogue == TP_EPI_GATED || a.K <= ONE_ROUND_K || a.N >= WIDE_N) return 5;
        } else if (a.K <= ONE_ROUND_K && a.N < WIDE_N) {
            return 5;
        }
    }
    if (gemm_mfma_supports(a)) {
        // (a single sequence is faster on the skinny kernel throughout)
        if (a.M >= 8 && (a.epilogue == TP_EPI_GATED || (long)a.N * a.K >= LARGE_NK)) return 3;
        if (a.M >= 8 && a.N >= WIDE_N) return 3;
        // from 9 rows on the tiled kernel wins every product of a layer against the skinny one (2B, 16 rows, cold
        // weights: qkv 6.4 / 8.0 us, o 5.1 / 5.3, down 11.5 / 18.6)
        if (a.M > 8 && (sliced || a.N >= 8192)) return 3;
    }
    if (gemm_skinny_supports(a)) return 2;
    if (gemm_mfma_supports(a)) return 3;
    return 1;
}

// bytes of workspace a product needs; with defer, a positive multiple of M * N * 4 means the product comes back as that
// many float32 K slices (one of them, where its sums are not to be rounded), 0 that the call is to be made again without defer
extern "C" long tp_linear_workspace_bytes(int in_dtype, int out_dtype, int M, int N, int K, int epilogue, int units,
                                          int defer, int algo) {
    GemmArgs a{nullptr, nullptr, nullptr, in_dtype, out_dtype, M, N, K, epilogue, 1.f, units, 0, INFINITY, 0.f, nullptr, 0, defer, algo, nullptr};
    const int p = pick(a, algo);
    if (p == 2) return (long)gemm_skinny_workspace(a);
    if (p == 4) return (long)gemv_workspace(a);
    if (p == 5) return (long)gemm_rows8_workspace(a);
    if (p == 16) return (long)gemm_stream_slices_left(a) * M * N * 4;
    if (p == 3) return (long)gemm_mfma_slices_left(a) * M * N * 4;
    if (p == 20) { const int s = gemm_f32_splits(a); return s > 1 ? (long)s * M * N * 4 : 0; }
    if (p == 1 && epilogue == TP_EPI_GATED) return (long)M * N * 4;
    return 0;
}

extern "C" int tp_linear(const void* x, const void* w, void* y, int in_dtype, int out_dtype, int M, int N, int K,
                         int epilogue, float cap, int units, int act, float limit, float shift, void* workspace, long workspace_bytes,
                         int defer, int algo, void* stream) {
    GemmArgs a{x, w, y, in_dtype, out_dtype, M, N, K, epilogue, cap, units, act, limit, shift, workspace, (size_t)workspace_bytes, defer,
               algo, (hipStream_t)stream};
    if (int rc = check_args(a)) return rc;
    const int p = pick(a, algo);
    TP_REQUIRE(p > 0, "linear: the requested kernel (%d) does not take M=%d N=%d K=%d dtype %d", algo, M, N, K, in_dtype);
    if (p == 2) return gemm_skinny_launch(a);
    if (p == 4) return gemv_launch(a);
    if (p == 5) return gemm_rows8_launch(a);
    if (p == 3) return gemm_mfma_launch(a);
    if (p == 16) return gemm_stream_launch(a);
    if (p == 20) return gemm_f32_launch(a);
    return gemm_simple_launch(a);
}
