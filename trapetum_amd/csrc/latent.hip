// Attention through a cached latent: what stands between the input projection and the attention kernels, and the
// per-head products that carry queries into the latent's space and weighted latents out of it.
#include "common.h"
#include "tile.h"
#include "tile_mfma.h"

// ---- a step's projections -> rotated query parts, and the rows [rope(key part) | rmsnorm(latent) * gain] ----------
// proj row: H heads of [dr rotated | dn unrotated] query elements, then (own) [dr key part | R latent].
// q row: H heads of [dr | R]; this kernel fills the first dr of each (the rest is a product's output).
// The first `rot` of the dr elements turn in pairs (f, f + rot / 2) by pos * inv_freq[f]; the others pass.
// grid (rows, [the latent] + heads by HPT * at_once).  All of it is waiting: the position, then what is read, then what is
// stored.  So a row is shared out: one block for the latent's norm, the others for the heads (the key part counts as one more),
// each thread keeping its pair f (its angle is its own, no table and no barrier) for HPT heads whose elements are asked for
// before the angle is worked out.  A block for the whole row, its angles in a table in LDS, took (bf16; 16 heads, 64 turning,
// latent of 192: rows 8 / 128 / 1300 / 4096) 5.2 / 5.3 / 8.0 / 17.8 us, this 2.9 / 3.1 / 7.6 / 17.3; with 128 heads and a latent
// of 512 15.5 / 16.0 / 36.9 / 81.3 us, this 3.1 / 4.1 / 18.7 / 52.0.
template <typename T, int HPT>
__global__ void __launch_bounds__(256)
latent_prepare_k(const T* __restrict__ proj, long proj_stride, int H, int dn, int dr, int R,
                 const float* __restrict__ gain, float eps, const float* __restrict__ inv_freq, int rot,
                 const int* __restrict__ row_seq, const int* __restrict__ row_pos, const int* __restrict__ new_len,
                 const int* __restrict__ table, int table_w, T* __restrict__ pool, int page, int rows_cap,
                 T* __restrict__ q, T* __restrict__ mine, int own, const T* __restrict__ tail_rows, long tail_stride,
                 int per_head, int at_once) {
    __shared__ float red[4];
    const int r = blockIdx.x, pos = row_pos[r], half = rot / 2, row = dr + R, tid = threadIdx.x;
    const T* pr = proj + (size_t)r * proj_stride;
    const T* tail = tail_rows ? tail_rows + (size_t)r * tail_stride : pr + (size_t)H * (dr + dn);     // a product of its own, or the row's end
    const int h_block = ((int)blockIdx.y - own) * at_once * HPT;          // below 0: the latent
    T* mr = nullptr;
    T* dst = nullptr;                                    // the row's place in the cache
    if (own && (h_block < 0 || h_block + at_once * HPT > H)) {
        mr = mine + (size_t)r * row;
        if (table) {
            const int seq = row_seq[r];
            int at = pos;
            bool keep = true;
            if (rows_cap > 0) {
                keep = pos + rows_cap >= new_len[seq];   // else a later row of this step takes the same ring row
                at = pos % rows_cap;
            }
            const int pg = keep && at / page < table_w ? table[(size_t)seq * table_w + at / page] : -1;     // a table too narrow for the position caches nothing
            if (pg >= 0) dst = pool + ((size_t)pg * page + at % page) * row;
        }
    }
    if (h_block < 0) {
        constexpr int NR = 4;                            // elements a thread keeps; a longer latent is read again
        float v[NR], w[NR], ss = 0.f;
#pragma unroll
        for (int i = 0; i < NR; i++) {
            const int e = tid + i * 256;
            v[i] = e < R ? ld_f32(tail + dr + e) : 0.f;
            w[i] = e < R ? gain[e] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < NR; i++) ss += v[i] * v[i];
        for (int e = tid + NR * 256; e < R; e += 256) { const float x = ld_f32(tail + dr + e); ss += x * x; }
        ss = block_sum_once<256>(ss, red);
        const float scale = rsqrtf(ss / (float)R + eps);
#pragma unroll
        for (int i = 0; i < NR; i++) {
            const int e = tid + i * 256;
            if (e >= R) continue;
            const float y = (v[i] * scale) * w[i];
            st_f32(mr + dr + e, y);
            if (dst) st_f32(dst + dr + e, y);
        }
        for (int e = tid + NR * 256; e < R; e += 256) {
            const float y = (ld_f32(tail + dr + e) * scale) * gain[e];
            st_f32(mr + dr + e, y);
            if (dst) st_f32(dst + dr + e, y);
        }
        return;
    }
    const int heads = H + own;
    const int h0 = h_block + tid / per_head;             // per_head: threads a head takes (its pairs and its elements that pass, at most 256)
    if (h0 >= h_block + at_once) return;
    for (int f = tid % per_head; f < dr - half; f += per_head) {
        const int lo = f < half ? f : f + half, hi = f + half;            // a pair, or twice an element that passes
        float a[HPT], b[HPT];
#pragma unroll
        for (int i = 0; i < HPT; i++) {
            const int h = min(h0 + i * at_once, heads - 1);
            const T* src = h < H ? pr + (size_t)h * (dr + dn) : tail;
            a[i] = ld_f32(src + lo);
            b[i] = ld_f32(src + hi);
        }
        float co = 1.f, si = 0.f;
        if (f < half) {
            const float ang = (float)pos * inv_freq[f];
            co = cosf(ang);
            si = sinf(ang);
        }
#pragma unroll
        for (int i = 0; i < HPT; i++) {
            const int h = h0 + i * at_once;
            if (h >= heads) continue;
            const float x = f < half ? a[i] * co - b[i] * si : a[i], y = f < half ? b[i] * co + a[i] * si : b[i];
            T* o = h < H ? q + ((size_t)r * H + h) * row : mr;
            st_f32(o + lo, x);
            if (f < half) st_f32(o + hi, y);
            if (h == H && dst) {
                st_f32(dst + lo, x);
                if (f < half) st_f32(dst + hi, y);
            }
        }
    }
}

extern "C" int tp_latent_prepare(const void* proj, long proj_stride, int dtype, int M, int H, int dn, int dr, int R,
                                 const float* gain, float eps, const float* inv_freq, int rot,
                                 const int* row_seq, const int* row_pos, const int* new_len,
                                 const int* table, int table_w, void* pool, int page, int rows_cap,
                                 void* q, void* mine, int own, const void* tail, long tail_stride, void* stream) {
    TP_REQUIRE(M > 0 && H > 0 && dn >= 0 && dr >= 0 && R > 0, "latent_prepare: empty shape M=%d H=%d dn=%d dr=%d R=%d", M, H, dn, dr, R);
    TP_REQUIRE(proj && q && row_pos, "latent_prepare: a null operand");
    TP_REQUIRE(rot >= 0 && rot <= dr && rot % 2 == 0, "latent_prepare: %d turning elements must be even and at most the rotated part's %d", rot, dr);
    TP_REQUIRE(rot == 0 || inv_freq, "latent_prepare: a rotation needs its frequency table");
    TP_REQUIRE(proj_stride >= (long)H * (dr + dn) + (own && !tail ? dr + R : 0), "latent_prepare: rows of %ld elements are too short", proj_stride);
    TP_REQUIRE(!tail || (own && tail_stride >= dr + R), "latent_prepare: the key part and latent as rows of their own need %d elements a row", dr + R);
    TP_REQUIRE(!own || (mine && gain && row_seq && new_len), "latent_prepare: a layer with a latent of its own needs its gain and the rows' output");
    TP_REQUIRE(!table || (pool && page > 0 && table_w > 0), "latent_prepare: a page table without a cache pool");
    if (!table) { page = 1; rows_cap = 0; }
    TP_REQUIRE(rows_cap >= 0 && (rows_cap == 0 || rows_cap % page == 0), "latent_prepare: ring of %d rows is no multiple of the page size %d", rows_cap, page);
    TP_REQUIRE(rot <= 8192, "latent_prepare: %d turning elements are more than a head may have (8192)", rot);
    hipStream_t s = (hipStream_t)stream;
    const int items = dr - rot / 2, per_head = items > 256 ? 256 : items > 0 ? items : 1, at_once = 256 / per_head, heads = items ? H + !!own : 0;
    // Four heads a thread once that many still fill the chip: one angle then serves four heads.  Below, more blocks with one
    // head a thread end sooner.  One / four heads a thread, 16 heads:
    // 8 rows 3.1 / 3.7 us, 256 rows 3.5 / 3.7, 512 rows 4.7 / 4.6, 4096 rows 21.6 / 17.3; 128 heads: 32 rows 3.2 / 3.4, 64 rows
    // 3.7 / 3.6, 4096 rows 74.3 / 51.5.
    const bool many = (long)M * heads > 8192;
    const int per_block = at_once * (many ? 4 : 1), blocks = !!own + tp_cdiv(heads, per_block);
    if (blocks == 0) return 0;                           // nothing turns and nothing is cached
    TP_REQUIRE(blocks <= 65535, "latent_prepare: %d heads exceed one launch", H);
    dim3 grid(M, blocks);
#define TP_LATENT_PREPARE(T, HPT) latent_prepare_k<T, HPT><<<grid, 256, 0, s>>>((const T*)proj, proj_stride, H, dn, dr, R, gain, eps, inv_freq, rot, row_seq, row_pos, \
        new_len, table, table_w, (T*)pool, page, rows_cap, (T*)q, (T*)mine, !!own, (const T*)tail, tail_stride, per_head, at_once)
    if (dtype == TP_BF16) { if (many) TP_LATENT_PREPARE(bf16_t, 4); else TP_LATENT_PREPARE(bf16_t, 1); }
    else if (dtype == TP_F32) { if (many) TP_LATENT_PREPARE(float, 4); else TP_LATENT_PREPARE(float, 1); }
    else return tp_fail("latent_prepare: unknown dtype %d", dtype);
#undef TP_LATENT_PREPARE
    return tp_check_launch("latent_prepare");
}

// ---- per-head products: out[m, h, n] = sum_k x[m, h, k] * w[h, n, k] ----------------------------------------------
// x and out are views of wider rows (strides in elements: row, head; elements of a head contiguous); w is contiguous.
// gate (or null): rows of H N elements of the same type; out[m, h, n] is multiplied by sigmoid(gate[m][h N + n]) before it is
// rounded.
__device__ __forceinline__ float gated_by(float x, float g) { return x / (1.f + expf(-g)); }

// grid (column tiles, row tiles, heads)
template <typename T, int TM>
__global__ void __launch_bounds__(256)
head_linear_k(const T* __restrict__ x, long x_row, long x_head, const T* __restrict__ w, T* __restrict__ out, long o_row, long o_head,
              int M, int N, int K, const T* __restrict__ gate, long gate_row) {
    constexpr int TN = 64, BK = 16;
    __shared__ TileShared<TM, TN, BK> sh;
    const int h = blockIdx.z, m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    const T* xh = x + (size_t)h * x_head;
    const T* wh = w + (size_t)h * N * K;
    float acc[TM / 16][TN / 16];
    tile_product<TM, TN, BK>(acc, K,
        [&](int m, int k) { return m0 + m < M ? ld_f32(xh + (size_t)(m0 + m) * x_row + k) : 0.f; },
        [&](int n, int k) { return n0 + n < N ? ld_f32(wh + (size_t)(n0 + n) * K + k) : 0.f; }, sh);
    const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
#pragma unroll
    for (int i = 0; i < TM / 16; i++)
#pragma unroll
        for (int j = 0; j < TN / 16; j++) {
            const int m = m0 + ty + 16 * i, n = n0 + tx + 16 * j;
            if (m < M && n < N) st_f32(out + (size_t)m * o_row + (size_t)h * o_head + n, gate ? gated_by(acc[i][j], ld_f32(gate + (size_t)m * gate_row + (size_t)h * N + n)) : acc[i][j]);
        }
}

// the same on the matrix cores: bf16, K a multiple of 8, every head's rows starting on 16 bytes
template <int TM>
__global__ void __launch_bounds__(256)
head_linear_mfma_k(const bf16_t* __restrict__ x, long x_row, long x_head, const bf16_t* __restrict__ w, bf16_t* __restrict__ out,
                   long o_row, long o_head, int M, int N, int K, const bf16_t* __restrict__ gate, long gate_row) {
    using Tile = MfmaTile<TM, false>;
    __shared__ typename Tile::Shared sh;
    const int h = blockIdx.z, m0 = blockIdx.y * TM, n0 = blockIdx.x * 64;
    const bf16_t* xh = x + (size_t)h * x_head;
    const bf16_t* wh = w + (size_t)h * N * K;
    const uint4 zero = make_uint4(0, 0, 0, 0);
    const bool quads = gate && gate_row % 4 == 0 && N % 4 == 0 && (uintptr_t)gate % 8 == 0;
    const bool wide = o_row % 4 == 0 && o_head % 4 == 0 && (uintptr_t)out % 8 == 0;
    Tile t;
    t.run(K,
        [&](int m, int k) { return m0 + m < M ? *reinterpret_cast<const uint4*>(xh + (size_t)(m0 + m) * x_row + k) : zero; },
        [&](int n, int k) { return n0 + n < N ? *reinterpret_cast<const uint4*>(wh + (size_t)(n0 + n) * K + k) : zero; }, sh);
#pragma unroll
    for (int i = 0; i < Tile::MI; i++)
#pragma unroll
        for (int j = 0; j < Tile::NJ; j++) {
            const int m = m0 + Tile::m_of(i), n = n0 + Tile::n_of(j);
            if (m >= M || n >= N) continue;
            bf16_t* dst = out + (size_t)m * o_row + (size_t)h * o_head + n;
            if (gate) {
                const bf16_t* gp = gate + (size_t)m * gate_row + (size_t)h * N + n;
                union { uint2 u; bf16_t h[4]; } g4;
                if (quads) g4.u = *reinterpret_cast<const uint2*>(gp);
                else for (int v = 0; v < 4; v++) g4.h[v] = gp[n + v < N ? v : 0];
#pragma unroll
                for (int v = 0; v < 4; v++) t.acc[0][i][j][v] = gated_by(t.acc[0][i][j][v], bf16_to_f32(g4.h[v]));
            }
            if (wide && n + 3 < N) {                      // the lane's four neighbours in one store
                uint2 o;
                o.x = (uint32_t)f32_to_bf16(t.acc[0][i][j][0]) | ((uint32_t)f32_to_bf16(t.acc[0][i][j][1]) << 16);
                o.y = (uint32_t)f32_to_bf16(t.acc[0][i][j][2]) | ((uint32_t)f32_to_bf16(t.acc[0][i][j][3]) << 16);
                *reinterpret_cast<uint2*>(dst) = o;
                continue;
            }
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (n + v < N) dst[v] = f32_to_bf16(t.acc[0][i][j][v]);
        }
}

// A few rows (up to 16), K a multiple of 32: such a product reads its matrices once and is over, so what counts is how soon
// they are asked for.  A wave has 16 of a head's outputs and all of K, by itself: operands go from memory straight to the
// registers that the matrix instruction reads (lane r + 16 g: row r, elements 8 g on of each 32), every step's at once, up to
// STEPS of them; no LDS, no barrier, four times the blocks.  The sums are formed in the order of the tile above.  (16 heads of
// 128 x 512, 4 rows: 7.0 us a launch through the tile, 3.9 so; 512 x 128: 4.2 and 2.9; 192 x 128: 3.8 and 2.3.)
// grid (column tiles of 16, 1, heads)
__global__ void __launch_bounds__(64)
head_linear_few_k(const bf16_t* __restrict__ x, long x_row, long x_head, const bf16_t* __restrict__ w, bf16_t* __restrict__ out,
                  long o_row, long o_head, int M, int N, int K, const bf16_t* __restrict__ gate, long gate_row) {
    constexpr int STEPS = 8;
    const int lane = threadIdx.x, r = lane & 15, g = lane >> 4, h = blockIdx.z, n0 = blockIdx.x * 16;
    const int xm = r < M ? r : M - 1, wn = n0 + r < N ? n0 + r : N - 1;           // (rows past the end: not stored)
    const bf16_t* xp = x + (size_t)h * x_head + (size_t)xm * x_row + 8 * g;
    const bf16_t* wp = w + ((size_t)h * N + wn) * K + 8 * g;
    tm_f32x4 acc{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += 32 * STEPS) {
        union { uint4 u; tm_bf16x8 v; } fx[STEPS], fw[STEPS];
#pragma unroll
        for (int s = 0; s < STEPS; s++)
            if (k0 + 32 * s < K) {
                fw[s].u = *reinterpret_cast<const uint4*>(wp + k0 + 32 * s);
                fx[s].u = *reinterpret_cast<const uint4*>(xp + k0 + 32 * s);
            }
#pragma unroll
        for (int s = 0; s < STEPS; s++)
            if (k0 + 32 * s < K) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[s].v, fx[s].v, acc, 0, 0, 0);
    }
    const int n = n0 + 4 * g;
    if (r >= M || n >= N) return;
    bf16_t* dst = out + (size_t)r * o_row + (size_t)h * o_head + n;
    if (gate) {
        const bf16_t* gp = gate + (size_t)r * gate_row + (size_t)h * N;
#pragma unroll
        for (int v = 0; v < 4; v++) acc[v] = gated_by(acc[v], bf16_to_f32(gp[n + v < N ? n + v : N - 1]));
    }
    if (o_row % 4 == 0 && o_head % 4 == 0 && (uintptr_t)out % 8 == 0 && n + 3 < N) {
        uint2 o;
        o.x = (uint32_t)f32_to_bf16(acc[0]) | ((uint32_t)f32_to_bf16(acc[1]) << 16);
        o.y = (uint32_t)f32_to_bf16(acc[2]) | ((uint32_t)f32_to_bf16(acc[3]) << 16);
        *reinterpret_cast<uint2*>(dst) = o;
    } else {
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (n + v < N) dst[v] = f32_to_bf16(acc[v]);
    }
}

extern "C" int tp_head_linear(const void* x, long x_row, long x_head, const void* w, void* out, long o_row, long o_head,
                              int dtype, int M, int H, int N, int K, const void* gate, long gate_row, int plain, void* stream) {
    TP_REQUIRE(!gate || gate_row >= (long)H * N, "head_linear: gates of %ld elements a row do not cover %d heads of %d", gate_row, H, N);
    TP_REQUIRE(M > 0 && H > 0 && N > 0 && K > 0, "head_linear: empty shape M=%d H=%d N=%d K=%d", M, H, N, K);
    TP_REQUIRE(x && w && out, "head_linear: a null operand");
    TP_REQUIRE(x_head >= K && o_head >= N && x_row >= (long)(H - 1) * x_head + K && o_row >= (long)(H - 1) * o_head + N,
               "head_linear: strides (%ld, %ld) -> (%ld, %ld) do not hold %d heads of %d -> %d elements", x_row, x_head, o_row, o_head, H, K, N);
    TP_REQUIRE(H <= 65535, "head_linear: %d heads exceed one launch", H);
    hipStream_t s = (hipStream_t)stream;
    const bool few = M <= 16;
    const int TM = few ? 16 : 64;
    dim3 grid(tp_cdiv(N, 64), tp_cdiv(M, TM), H);
    TP_REQUIRE(grid.y <= 65535, "head_linear: %d rows exceed one launch", M);
    if (dtype == TP_BF16 && !plain && M >= 512 && K % 8 == 0 && x_row % 8 == 0 && x_head % 8 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0) {
        grid.y = tp_cdiv(M, 128);
        head_linear_mfma_k<128><<<grid, 256, 0, s>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)w, (bf16_t*)out, o_row, o_head, M, N, K, (const bf16_t*)gate, gate_row);
        return tp_check_launch("head_linear (matrix cores)");
    }
    if (dtype == TP_BF16 && !plain && K % 8 == 0 && x_row % 8 == 0 && x_head % 8 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0) {
        if (few && K % 32 == 0) {
            grid.x = tp_cdiv(N, 16);
            head_linear_few_k<<<grid, 64, 0, s>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)w, (bf16_t*)out, o_row, o_head, M, N, K, (const bf16_t*)gate, gate_row);
        } else if (few) head_linear_mfma_k<16><<<grid, 256, 0, s>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)w, (bf16_t*)out, o_row, o_head, M, N, K, (const bf16_t*)gate, gate_row);
        else head_linear_mfma_k<64><<<grid, 256, 0, s>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)w, (bf16_t*)out, o_row, o_head, M, N, K, (const bf16_t*)gate, gate_row);
        return tp_check_launch("head_linear (matrix cores)");
    }
#define TP_HEAD_LINEAR(T, TMv) head_linear_k<T, TMv><<<grid, 256, 0, s>>>((const T*)x, x_row, x_head, (const T*)w, (T*)out, o_row, o_head, M, N, K, (const T*)gate, gate_row)
    if (dtype == TP_BF16) { if (few) TP_HEAD_LINEAR(bf16_t, 16); else TP_HEAD_LINEAR(bf16_t, 64); }
    else if (dtype == TP_F32) { if (few) TP_HEAD_LINEAR(float, 16); else TP_HEAD_LINEAR(float, 64); }
    else return tp_fail("head_linear: unknown dtype %d", dtype);
#undef TP_HEAD_LINEAR
    return tp_check_launch("head_linear");
}
