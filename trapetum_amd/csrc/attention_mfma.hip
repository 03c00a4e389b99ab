// bf16 attention of decode steps on the matrix cores for one head size (compiled with -DTP_HD=<head_dim>, a
// multiple of 16 up to 256): one query per sequence and head over the paged cache.  (Steps of many queries:
// attention_prefill.hip, in the same library.)
//
// Formula as the reference's attn_k (runtime/cuda/codebook_gemv.cu:240-270): score = (q . k) * scale, then
// cap * tanh(score / cap) if a cap is set, softmax over the visible keys in fp32, weighted sum of v, query head
// h reading kv head h / (heads / kv_heads).  The scale is an argument (rsqrt(head_dim) in the reference), and a
// window W hides keys with p - t >= W (the reference has none: runtime/src/lib.rs:4455).
//
// Scores are computed transposed, S^T = K . Q^T with v_mfma_f32_16x16x32_bf16: key rows are the A operand (a
// lane holds 8 consecutive elements of one key: one 16-byte load), queries the B operand, and a lane ends up
// with 4 keys of ONE query, so the softmax statistics are per-lane scalars.
//
// Compiled with -DTP_BY_POSITION=1 the scores may depend on positions (TpPositional in common.h): the query's temperature is a
// factor on its scale, and a lane fetches its four keys' biases with the round's keys; a gate per head multiplies the output
// where it is normalised.
#include "common.h"
#include <type_traits>
#include "error_channel.h"

#ifndef TP_HD
#error "compile with -DTP_HD=<head_dim>"
#endif

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

#ifndef TP_BY_POSITION
#define TP_BY_POSITION 0
#endif

namespace {
constexpr bool BY_POSITION = TP_BY_POSITION != 0;
constexpr int HD = TP_HD;
constexpr int HDP = (HD + 31) / 32 * 32;       // head size padded to the product's k step
constexpr int KSTEPS = HDP / 32;
constexpr int NCH = HD / 8;                     // 16-byte chunks of a row
static_assert(HD % 16 == 0 && HD >= 16 && HD <= 256, "head_dim must be a multiple of 16 up to 256");

union Frag { uint4 u; bf16x8 v; bf16_t h[8]; };

__device__ __forceinline__ bf16x8 ld_frag(const bf16_t* p, bool ok) {
    Frag f;
    if (ok) f.u = *reinterpret_cast<const uint4*>(p);
    else f.u = make_uint4(0, 0, 0, 0);
    return f.v;
}
// tanh through one exponential and one reciprocal: 1 - 2 / (1 + e^(2x)); exact at both ends, relative error of a
// few 1e-7 elsewhere (the scores are rounded to bf16 probabilities afterwards)
__device__ __forceinline__ float tanh_fast(float x) {
    return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __expf(2.f * x));
}
// scale_over_cap = scale / cap, so that a capped score costs two multiplications around the tanh
__device__ __forceinline__ float score_of(float dot, float scale, float cap, float scale_over_cap) {
    return cap > 0.f ? cap * tanh_fast(dot * scale_over_cap) : dot * scale;
}
// n / d of 0 <= n < 4096, 0 < d <= 256: (n + 1/2) / d lies 1/512 or more from every whole number, far more than the reciprocal's
// error (an integer division is some thirty instructions)
__device__ __forceinline__ int quotient(int n, int d) { return (int)(((float)n + 0.5f) * __builtin_amdgcn_rcpf((float)d)); }
}  // namespace

// =====================================================================================================
// decode: one query per sequence and head, keys and values in the paged cache.  A block owns one
// (sequence, kv head, slice of the keys) and all the query heads of that kv head, so K and V are read once
// for the group.  Scores by MFMA with key rows loaded straight from global memory; probabilities through
// a wave's LDS; the weighted sum of V with plain FMAs (V's rows are contiguous along the head, not along the
// keys), each lane owning one 16-byte chunk of the head for a subset of the wave's 16 keys.  A wave keeps its
// own running softmax over the keys it sees, so the waves of a block meet only once, at the end; a round's value
// chunks are fetched together with its key rows, before the scores are known, so the two latencies overlap.  Slices of the keys
// (flash-decoding) write (max, sum, unnormalised output) to a workspace that a second kernel combines in
// slice order.
// Few keys (nsplit 0): a block of eight waves has all of them and writes the result itself.  What such a step waits for is
// launches and trips to memory, not keys: the combination was a launch of 3 us for slices most of which were empty (chats of 1 / 64 up to
// 60 keys: 9.8 / 11.8 us a layer in slices, 6.8 / 8.4 so; up to where: HipOps._decode_slices), and the new token's key and value, which the block
// has just made, come from LDS instead of back from the cache.
// =====================================================================================================
struct DecodeArgs {
    const bf16_t* q; long q_stride; int H, KV; const int* new_len; const int* table; int table_w;
    bf16_t* k_pool; bf16_t* v_pool; int page, rows_cap; float scale, cap; int window;
    bf16_t* out; float* ws_o; float* ws_ml; int nsplit;
    // the step's projections, when the kernel rotates and caches them itself (else null): rows of
    // [heads | kv heads (keys) | kv heads (values)] x head size, bf16, or float32 in K slices that are added here
    const void* qkv; int qkv_f32, n_slices; long slice_stride, row_stride;
    const float* inv_freq; int rot, write_kv;
    // kv heads the pools really have (0: KV).  Fewer than KV: the grid's kv heads are groups of query heads that share
    // pool head `kvh % pool_kv` (a cache with one row per token for all heads is read by every group)
    int pool_kv;
    // chunk C > 0: the query sees keys from floor(p / C) C on only.  head_scale, sink ([H] or null): a factor on every
    // head's scores; a score without key or value that joins every head's softmax sum once
    int chunk; const float* head_scale; const float* sink;
    // the first `keep` positions stay visible behind the window; in a ring they live in the `pin` rows in front of it
    int keep, pin;
    TpPositional by_position;
    int G;                                           // query heads a kv head (set by the launch)
};

namespace {
// In the decode kernel a lane's two loads of a pair of product steps are adjacent 16-byte pieces, so the four lanes
// of a key row fetch a whole 128-byte line per pair: step ks, lane group g -> head elements dofs .. dofs + 7.
constexpr int DSTEPS = 2 * ((HD + 63) / 64);
__device__ __forceinline__ int dofs(int ks, int g) { return (ks >> 1) * 64 + g * 16 + (ks & 1) * 8; }
constexpr int DWAVES = 4;                        // waves of a block that works on a slice; each scores and sums its own 16 keys of a round
constexpr int WHOLE_WAVES = 8;                   // waves of a block that has all keys of its kv head (a launch without slices)
constexpr int KGW = 64 / NCH > 16 ? 16 : 64 / NCH;   // key groups of a wave: lanes with one chunk index walk the keys KGW apart
constexpr int VPT = (16 + KGW - 1) / KGW;        // value chunks a lane fetches per round
}

template <int QT, int WAVES = DWAVES>
__global__ void __launch_bounds__(64 * WAVES)
attn_decode_k(DecodeArgs a) {
    constexpr int DTH = 64 * WAVES, ROUND = 16 * WAVES;        // threads; keys a block takes per round
    constexpr bool WHOLE = WAVES > DWAVES;           // no slices: the block has all keys, one round of them or two
    constexpr int RQ = WHOLE && QT > 1 ? 2 : 1;      // heads whose parts are added at a time
    __shared__ float p_lds[WAVES][QT][16];           // a wave's probabilities of its 16 keys
    __shared__ float alpha_lds[WAVES][QT];
    __shared__ __attribute__((aligned(16))) float m_w[WHOLE ? QT : WAVES][WHOLE ? WAVES : QT], l_w[WHOLE ? QT : WAVES][WHOLE ? WAVES : QT];
    __shared__ float red[RQ * WAVES * KGW * HD];
    __shared__ __attribute__((aligned(16))) bf16_t q_lds[QT * HD], new_lds[WHOLE ? 2 * HD : 8];      // queries; the new key and value
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
    const int kvh = blockIdx.x, seq = blockIdx.y, split = blockIdx.z;
    const int G = a.G;
    const int held = a.new_len[seq];
    // ---- the projections' columns of this thread's first pair are asked for before anything is known of the sequence: they wait for
    // the kernel that has just written them, the keys for the sequence's length and page table, one after the other
    constexpr int NE = 6;                            // the pair of a query head, and the new key's and value's
    const int half = a.rot >> 1;
    unsigned early[NE][4];                           // float32 of four slices, or bf16 in the first
    float freq = 0.f;
    auto ask = [&](int idx) {
        const int qi = quotient(idx, half), f = idx - qi * half;
        const unsigned q0 = (unsigned)(kvh * G + qi) * HD + f, k0 = a.write_kv ? (unsigned)(a.H + kvh) * HD + f : q0, v0 = a.write_kv ? k0 + (unsigned)a.KV * HD : q0;
        const unsigned cols[6] = {q0, q0 + half, k0, k0 + half, v0, v0 + half};
        if (a.qkv_f32) {
            const char* slice = (const char*)a.qkv + (size_t)seq * a.row_stride * 4;
#pragma unroll
            for (int u = 0; u < 4; u++) {
#pragma unroll
                for (int c = 0; c < NE; c++) early[c][u] = *reinterpret_cast<const unsigned*>(slice + cols[c] * 4u);
                slice += u + 1 < a.n_slices ? a.slice_stride * 4 : 0;
            }
        } else {
#pragma unroll
            for (int c = 0; c < NE; c++) early[c][0] = *reinterpret_cast<const bf16_t*>((const char*)a.qkv + (size_t)seq * a.row_stride * 2 + cols[c] * 2u);
        }
        freq = a.inv_freq[f];
    };
    if constexpr (WHOLE) {
        if (a.qkv && half > 0) ask(min(tid, G * half - 1));
        __builtin_amdgcn_sched_barrier(0);
    }
    const int p = held - 1;
    int lo = a.window > 0 ? max(0, p - a.window + 1) : 0;
    if (a.chunk > 0) lo = max(lo, p / a.chunk * a.chunk);
    const int lo_al = lo & ~15;
    // The positions a block walks are counted without the gap between the kept ones (rounded up to a tile) and the
    // window: place u stands for position u below kept_al and for u + gap from there on.  Without kept positions (or where
    // the window reaches them) there is no gap.
    const int kept_al = (a.keep + 15) & ~15;
    const int first = a.keep > 0 ? 0 : lo_al, gap = a.keep > 0 && lo_al > kept_al ? lo_al - kept_al : 0;
    const int places = p + 1 - gap;
    int chunk = places - first;
    if constexpr (!WHOLE) chunk = (chunk + a.nsplit - 1) / a.nsplit;
    chunk = (chunk + ROUND - 1) / ROUND * ROUND;
    const int t_begin = first + split * chunk;           // in places
    const int t_end = min(places, t_begin + chunk);
    if (t_begin >= places) {                               // this slice has no keys (only when there are several)
        if (tid < G) {
            float* ml = a.ws_ml + (((size_t)seq * a.H + kvh * G + tid) * a.nsplit + split) * 2;
            ml[0] = -INFINITY;
            ml[1] = 0.f;
        }
        return;
    }
    const int* table = a.table + (size_t)seq * a.table_w;
    // Where the 16 keys of a tile live.  Tiles start at multiples of 16 positions; position t is row t, or row
    // t % rows_cap of a ring (rows_cap a multiple of the page size, the page size a power of two >= 16), so a tile
    // lies in one page, in 16 consecutive rows: one page-table entry per tile, looked up once for the wave.
    const int page_shift = __ffs(a.page) - 1, page_mask = a.page - 1;
    // (pin rows, whole pages, stand before the ring and keep the first positions)
    const int ring = a.rows_cap - a.pin, ring_from = max(lo_al, a.pin), ring_lo = a.rows_cap > 0 ? (ring_from - a.pin) % ring : 0;
    auto tile_offset = [&](int tb) -> size_t {                     // element offset of the tile's first row in a pool
        int row = tb;
        if (a.rows_cap > 0 && tb >= a.pin) {
            row = ring_lo + (tb - ring_from);
            row = a.pin + (row >= ring ? row - ring : row);
        }
        const int pg = table[row >> page_shift];
        return (((size_t)pg * a.pool_kv + (a.pool_kv == a.KV ? kvh : kvh % a.pool_kv)) * a.page + (row & page_mask)) * HD;
    };

    // the lane's part in the weighted sum: chunk ch of the head, keys kgw, kgw + KGW, ... of the wave's 16
    const int ch = lane % NCH, kgw = lane / NCH;
    const bool pv_lane = kgw < KGW;
    // ---- loads of a round: the key row of lane c for the scores, value chunks for the sum.  Unconditional loads of
    // rows that exist: a hidden or surplus key gets probability 0 (or is skipped) in the sum ---------------------
    auto row_in_tile = [&](int tb, int t) {                        // a row of the tile that exists, for position t of it
        const int m = min(t, p), low = min(max(lo, tb), tb + 15);
        return m < a.keep ? m : max(m, low);
    };
    const float* bias = nullptr;                                   // of query head c of the group
    if constexpr (BY_POSITION)
        if (a.by_position.bias) bias = a.by_position.bias + (size_t)(kvh * G + (c < G ? c : 0)) * (a.by_position.reach + 1);
    float bs[4] = {0.f, 0.f, 0.f, 0.f};                            // the round's biases of the lane's keys
    auto load_round = [&](int ub, bf16x8 (&kf)[DSTEPS], Frag (&vf)[VPT]) {
        const int tb = ub < kept_al ? ub : ub + gap;
        const size_t tile = tile_offset(__builtin_amdgcn_readfirstlane(tb));
        const int tk = row_in_tile(tb, tb + c);
        // (a row's address is the tile's plus 32 bits of the lane's: one instruction a load)
        const char* const kt = reinterpret_cast<const char*>(a.k_pool + tile);
        const char* const vt = reinterpret_cast<const char*>(a.v_pool + tile);
        const unsigned kr = (unsigned)(tk - tb) * (HD * 2);
        if constexpr (BY_POSITION)
            if (bias)
#pragma unroll
                for (int i = 0; i < 4; i++) bs[i] = bias[min(max(p - (tb + g * 4 + i), 0), (int)a.by_position.reach)];
#pragma unroll
        for (int ks = 0; ks < DSTEPS; ks++) {
            const int d0 = dofs(ks, g);
            kf[ks] = ld_frag(reinterpret_cast<const bf16_t*>(kt + (kr + (d0 < HD ? d0 : 0) * 2u)), d0 < HD);
        }
#pragma unroll
        for (int j = 0; j < VPT; j++) {
            int kk = kgw + j * KGW;
            kk = kk > 15 ? 15 : kk;
            const int tv = row_in_tile(tb, tb + kk);
            vf[j].u = *reinterpret_cast<const uint4*>(vt + ((unsigned)(tv - tb) * (HD * 2) + ch * 16u));
        }
    };
    // The wave's first round is fetched while the queries are prepared, unless its tile holds the row that this
    // block is about to write.
    bf16x8 kf[DSTEPS];
    Frag vf[VPT];
    const int tb0 = t_begin + wave * 16;
    const bool holds_new = a.qkv && a.write_kv && tb0 < places && places - 1 < tb0 + 16, late = !WHOLE && holds_new;
    if (tb0 < t_end && !late) load_round(tb0, kf, vf);

    // ---- the group's queries into LDS; in the fused form from the step's projections: K slices added, queries and
    // the new key rotated (pair (f, f + rot/2), angle p * inv_freq[f], in float32), and the slice that holds position
    // p writes the key and the value into the cache before anyone in the block reads that row ---------------------
    if (a.qkv) {
        const int rest = HD - a.rot;
        // NC columns of the sequence's row at once: their loads are asked for together (of float32 slices four slices
        // at a time, added in slice order), so that a thread pays one trip to memory for all it needs, not one a column
        // (a column's address is the block's row plus 32 bits of the lane's: one instruction a load)
        auto vals = [&](auto ncol, const unsigned* cols, float* out) {
            constexpr int NC = decltype(ncol)::value;
            if (a.qkv_f32) {
                const char* src = (const char*)a.qkv + (size_t)seq * a.row_stride * 4;
#pragma unroll
                for (int c = 0; c < NC; c++) out[c] = 0.f;
#pragma unroll 1
                for (int s0 = 0; s0 < a.n_slices; s0 += 4) {
                    float part[NC][4];
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const char* slice = src + (size_t)(s0 + u < a.n_slices ? s0 + u : a.n_slices - 1) * a.slice_stride * 4;
#pragma unroll
                        for (int c = 0; c < NC; c++) part[c][u] = *reinterpret_cast<const float*>(slice + cols[c] * 4u);
                    }
#pragma unroll
                    for (int c = 0; c < NC; c++)
#pragma unroll
                        for (int u = 0; u < 4; u++) out[c] += s0 + u < a.n_slices ? part[c][u] : 0.f;
                }
            } else {
                const char* src = (const char*)a.qkv + (size_t)seq * a.row_stride * 2;
#pragma unroll
                for (int c = 0; c < NC; c++) out[c] = bf16_to_f32(*reinterpret_cast<const bf16_t*>(src + cols[c] * 2u));
            }
        };
        // the slice that holds position p (t_begin < places holds here) also rotates the new key and writes it and the value
        // into the cache: thread f < rot/2 does that beside its pair of the first query head, whose angle is the same
        const bool writer = a.write_kv && places - 1 < t_begin + chunk;
        bf16_t* kdst = nullptr;
        bf16_t* vdst = nullptr;
        if (writer) {
            const int row = a.rows_cap > 0 && p >= a.pin ? a.pin + (p - a.pin) % ring : p;
            const int pg = table[row >> page_shift];
            const size_t at = (((size_t)pg * a.KV + kvh) * a.page + (row & page_mask)) * HD;
            kdst = a.k_pool + at;
            vdst = a.v_pool + at;
        }
        const unsigned kcol = (unsigned)(a.H + kvh) * HD, vcol = (unsigned)(a.H + a.KV + kvh) * HD;
        for (int idx = tid; idx < G * half; idx += DTH) {
            const int qi = quotient(idx, half), f = idx - qi * half;
            const bool kv = writer && idx < half;                 // then qi == 0 and f == idx
            const unsigned col = (unsigned)(kvh * G + qi) * HD;
            const unsigned cols[6] = {col + f, col + f + half, kcol + f, kcol + f + half, vcol + f, vcol + f + half};
            float x[6];
            if constexpr (WHOLE) {
                if (idx != tid) ask(idx);
#pragma unroll
                for (int c = 0; c < NE; c++) {
                    x[c] = 0.f;
                    if (a.qkv_f32) {
#pragma unroll
                        for (int u = 0; u < 4; u++) x[c] += u < a.n_slices ? __uint_as_float(early[c][u]) : 0.f;
                    } else x[c] = __uint_as_float(early[c][0] << 16);
                }
                for (int sl = 4; sl < a.n_slices; sl++) {
                    const char* slice = (const char*)a.qkv + ((size_t)seq * a.row_stride + (size_t)sl * a.slice_stride) * 4;
                    float more[NE];
#pragma unroll
                    for (int c = 0; c < NE; c++) more[c] = *reinterpret_cast<const float*>(slice + (c < 2 || a.write_kv ? cols[c] : col) * 4u);
#pragma unroll
                    for (int c = 0; c < NE; c++) x[c] += more[c];
                }
            } else {
                if (writer) vals(std::integral_constant<int, 6>(), cols, x);     // (the whole block takes this branch or the other)
                else vals(std::integral_constant<int, 2>(), cols, x);
                freq = a.inv_freq[f];
            }
            const float ang = (float)p * freq;
            float cs, sn;
            sincosf(ang, &sn, &cs);
            q_lds[qi * HD + f] = f32_to_bf16(x[0] * cs - x[1] * sn);
            q_lds[qi * HD + f + half] = f32_to_bf16(x[1] * cs + x[0] * sn);
            if (kv) {
                const bf16_t k0 = f32_to_bf16(x[2] * cs - x[3] * sn), k1 = f32_to_bf16(x[3] * cs + x[2] * sn);
                const bf16_t v0 = f32_to_bf16(x[4]), v1 = f32_to_bf16(x[5]);
                kdst[f] = k0; kdst[f + half] = k1;
                vdst[f] = v0; vdst[f + half] = v1;
                if constexpr (WHOLE) { new_lds[f] = k0; new_lds[f + half] = k1; new_lds[HD + f] = v0; new_lds[HD + f + half] = v1; }
            }
        }
        for (int idx = tid; idx < G * rest; idx += DTH) {         // elements outside the rotation
            const int qi = quotient(idx, rest), d = a.rot + idx - qi * rest;
            const bool kv = writer && idx < rest;                 // then qi == 0
            const unsigned cols[3] = {(unsigned)(kvh * G + qi) * HD + d, kcol + d, vcol + d};
            float x[3];
            if (writer) vals(std::integral_constant<int, 3>(), cols, x);     // (the whole block takes this branch or the other)
            else vals(std::integral_constant<int, 1>(), cols, x);
            q_lds[qi * HD + d] = f32_to_bf16(x[0]);
            if (kv) {
                const bf16_t k0 = f32_to_bf16(x[1]), v0 = f32_to_bf16(x[2]);
                kdst[d] = k0;
                vdst[d] = v0;
                if constexpr (WHOLE) { new_lds[d] = k0; new_lds[HD + d] = v0; }
            }
        }
        if (writer) __threadfence_block();
    } else {
        for (int idx = tid; idx < G * HD; idx += DTH)
            q_lds[idx] = a.q[(size_t)seq * a.q_stride + (size_t)kvh * G * HD + idx];
    }
    __syncthreads();
    bf16x8 qf[DSTEPS];
#pragma unroll
    for (int ks = 0; ks < DSTEPS; ks++) {
        const int d0 = dofs(ks, g);
        const bool ok = c < G && d0 < HD;
        Frag f;
        f.u = *reinterpret_cast<const uint4*>(q_lds + (ok ? c * HD + d0 : 0));
        const uint32_t keep = (uint32_t) - (int)ok;
        f.u.x &= keep; f.u.y &= keep; f.u.z &= keep; f.u.w &= keep;
        qf[ks] = f.v;
    }
    // (WHOLE: the row that this block is writing comes from LDS; the one trip to memory was on the way meanwhile, and what lay in its
    // place is not looked at: rows of the tile past it read the same row)
    auto take_new = [&](int tb) {
        if constexpr (WHOLE) {
            const int t0 = tb < kept_al ? tb : tb + gap;
            if (!(a.qkv && a.write_kv && tb < places && places - 1 < tb + 16)) return;
            if (row_in_tile(t0, t0 + c) == p)
#pragma unroll
                for (int ks = 0; ks < DSTEPS; ks++) {
                    const int d0 = dofs(ks, g);
                    kf[ks] = ld_frag(new_lds + (d0 < HD ? d0 : 0), d0 < HD);
                }
#pragma unroll
            for (int j = 0; j < VPT; j++) {
                const int kk = kgw + j * KGW > 15 ? 15 : kgw + j * KGW;
                if (row_in_tile(t0, t0 + kk) == p) vf[j].u = *reinterpret_cast<const uint4*>(new_lds + HD + ch * 8);
            }
        }
    };
    float acc[QT][8];
#pragma unroll
    for (int qi = 0; qi < QT; qi++)
#pragma unroll
        for (int e = 0; e < 8; e++) acc[qi][e] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;            // of query head c, over this wave's keys so far
    float scale_c = a.head_scale && c < G ? a.scale * a.head_scale[kvh * G + c] : a.scale;     // lane (c, g): query head c of the group
    if constexpr (BY_POSITION) scale_c *= query_temperature(a.by_position, p);
    const float soc = a.cap > 0.f ? scale_c / a.cap : 0.f;

    for (int tb = tb0; tb < t_end; tb += ROUND) {
        if (tb != tb0 || late) load_round(tb, kf, vf);
        take_new(tb);
        // ---- scores of 16 keys for the group's query heads: lane (c, g) gets keys g*4 .. g*4+3 of head c ----------
        f32x4 s = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < DSTEPS; ks++) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks], qf[ks], s, 0, 0, 0);
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int u = tb + g * 4 + i, t = u < kept_al ? u : u + gap;
            const bool ok = (t >= lo || t < a.keep) && u < t_end;
            float score = score_of(s[i], scale_c, a.cap, soc);
            if constexpr (BY_POSITION) score += bs[i];
            s[i] = ok ? score : -INFINITY;
            mx = fmaxf(mx, s[i]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m_run, mx);
        float alpha = 1.f, psum = 0.f;
        float pr[4] = {0.f, 0.f, 0.f, 0.f};
        if (m_new != -INFINITY) {
            alpha = __expf(m_run - m_new);
#pragma unroll
            for (int i = 0; i < 4; i++) { pr[i] = __expf(s[i] - m_new); psum += pr[i]; }
        }
        psum += __shfl_xor(psum, 16, 64);
        psum += __shfl_xor(psum, 32, 64);
        l_run = l_run * alpha + psum;
        m_run = m_new;
        if (c < QT) {
#pragma unroll
            for (int i = 0; i < 4; i++) p_lds[wave][c][g * 4 + i] = pr[i];
            if (g == 0) alpha_lds[wave][c] = alpha;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // ---- weighted sum of the round's values -----------------------------------------------------------------------
#pragma unroll
        for (int qi = 0; qi < QT; qi++) {
            const float al = alpha_lds[wave][qi];
#pragma unroll
            for (int e = 0; e < 8; e++) acc[qi][e] *= al;
        }
#pragma unroll
        for (int j = 0; j < VPT; j++) {
            const int kk = kgw + j * KGW;
            if (kk < 16) {
                float vv[8];
#pragma unroll
                for (int e = 0; e < 8; e++) vv[e] = bf16_to_f32(vf[j].h[e]);
#pragma unroll
                for (int qi = 0; qi < QT; qi++) {
                    const float w = p_lds[wave][qi][kk];
#pragma unroll
                    for (int e = 0; e < 8; e++) acc[qi][e] = fmaf(w, vv[e], acc[qi][e]);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    // ---- the waves' results: rescale to a common maximum, add in wave and key-group order, write -------------
    if constexpr (WHOLE) {
        const int used = min(WAVES, (t_end - t_begin + 15) >> 4);       // waves that had keys (the others leave -infinity and zeros)
        if (c < QT && g == 0) { m_w[c][wave] = m_run; l_w[c][wave] = l_run; }
#pragma unroll
        for (int q0 = 0; q0 < QT; q0 += RQ) {
            if (q0 >= G) continue;
            if (q0 > 0) __syncthreads();
            if (pv_lane)
#pragma unroll
                for (int u = 0; u < RQ; u++)
#pragma unroll
                    for (int e = 0; e < 8; e += 4)
                        *reinterpret_cast<float4*>(red + ((u * WAVES + wave) * KGW + kgw) * HD + ch * 8 + e) = make_float4(acc[q0 + u][e], acc[q0 + u][e + 1], acc[q0 + u][e + 2], acc[q0 + u][e + 3]);
            __syncthreads();
            for (int idx = tid; idx < RQ * HD; idx += DTH) {
                const int u = idx / HD, d = idx - u * HD, qi = q0 + u;
                if (qi >= G) break;
                float m[WAVES], l[WAVES], mx = -INFINITY, num = 0.f, den = 0.f;
#pragma unroll
                for (int w = 0; w < WAVES; w += 4) {
                    *reinterpret_cast<float4*>(m + w) = *reinterpret_cast<const float4*>(&m_w[qi][w]);
                    *reinterpret_cast<float4*>(l + w) = *reinterpret_cast<const float4*>(&l_w[qi][w]);
                }
#pragma unroll
                for (int w = 0; w < WAVES; w++) mx = fmaxf(mx, m[w]);
#pragma unroll
                for (int w0 = 0; w0 < WAVES; w0 += 4) {
                    if (w0 >= used) break;
                    float part[4][KGW];
#pragma unroll
                    for (int w = 0; w < 4; w++)
#pragma unroll
                        for (int k2 = 0; k2 < KGW; k2++) part[w][k2] = red[((u * WAVES + w0 + w) * KGW + k2) * HD + d];
#pragma unroll
                    for (int w = 0; w < 4; w++) {
                        const float f = __expf(m[w0 + w] - mx);
                        float sum = 0.f;
#pragma unroll
                        for (int k2 = 0; k2 < KGW; k2++) sum += part[w][k2];
                        num += f * sum;
                        den += f * l[w0 + w];
                    }
                }
                const int head = kvh * G + qi;
                if (a.sink) den += __expf(a.sink[head] - mx);                 // (the query's own key is among them: mx is finite)
                float o = num / den;
                if constexpr (BY_POSITION) if (a.by_position.gate) o *= head_gate(a.by_position, seq, head);
                a.out[((size_t)seq * a.H + head) * HD + d] = f32_to_bf16(o);
            }
        }
        return;
    } else {
    if (c < QT && g == 0) { m_w[wave][c] = m_run; l_w[wave][c] = l_run; }
#pragma unroll
    for (int qi = 0; qi < QT; qi++) {
        if (qi >= G) continue;                       // G is the same for the whole block; unrolled, so that acc stays in registers
        if (pv_lane) {
#pragma unroll
            for (int e = 0; e < 8; e++) red[(wave * KGW + kgw) * HD + ch * 8 + e] = acc[qi][e];
        }
        __syncthreads();
        if (tid < HD) {
            float mx = -INFINITY;
            for (int w = 0; w < 4; w++) mx = fmaxf(mx, m_w[w][qi]);
            float num = 0.f, den = 0.f;
            for (int w = 0; w < 4; w++) {
                const float mw = m_w[w][qi];
                if (mw == -INFINITY) continue;
                const float f = __expf(mw - mx);
                float part = 0.f;
                for (int k2 = 0; k2 < KGW; k2++) part += red[(w * KGW + k2) * HD + tid];
                num += f * part;
                den += f * l_w[w][qi];
            }
            const int head = kvh * G + qi;
            if (a.nsplit == 1) {
                if (a.sink) den += __expf(a.sink[head] - mx);                 // (the slice holds the query's own key: mx is finite)
                float o = num / den;
                if constexpr (BY_POSITION) if (a.by_position.gate) o *= head_gate(a.by_position, seq, head);
                a.out[((size_t)seq * a.H + head) * HD + tid] = f32_to_bf16(o);
            } else {
                const size_t at = ((size_t)seq * a.H + head) * a.nsplit + split;
                a.ws_o[at * HD + tid] = num;
                if (tid == 0) { a.ws_ml[at * 2] = mx; a.ws_ml[at * 2 + 1] = den; }
            }
        }
        __syncthreads();
    }
    }
}

// The slices of one (sequence, head): weights exp(m_s - max m) / sum, then every thread adds its head elements in slice
// order.  Loads are unconditional (a slice without keys left its sum unwritten: its weight is zero and the value is
// replaced by zero).  Little work, each part of which runs its code once and waits for it: a wave is a block and has 64 of
// the head's elements; it forms the weights for itself, slice s in lane s, and takes them lane by lane into scalar registers,
// without LDS or a barrier.  The attention's two launches, with 8 heads of 256 on 4 kv heads, by a block a head that forms its weights
// once through LDS, by a block of such waves, by a wave a block: 8 sequences of 700 keys 13.8, 13.0, 12.8 us; one 11.0, 9.9, 9.7; two of
// 7,000 in 128 slices 27.3, 26.2, 25.5.
__global__ void __launch_bounds__(64)
attn_decode_combine_k(const float* __restrict__ ws_o, const float* __restrict__ ws_ml, int nsplit,
                      bf16_t* __restrict__ out, const float* __restrict__ sink, int H, TpPositional by_position) {
    const unsigned at = blockIdx.x * (unsigned)nsplit;           // blockIdx.x = sequence * heads + head
    const int lane = threadIdx.x, tid = blockIdx.y * 64 + lane, last = nsplit - 1;
    // the first 16 slices' sums are asked for before the weights are known: both come from memory at the same time
    constexpr int FIRST = 16, GROUP = 8;
    const int d = tid < HD ? tid : HD - 1;                       // (a whole wave: every lane has a slice's weight)
    const float2* ml = reinterpret_cast<const float2*>(ws_ml) + at;
    const float* sums = ws_o + (size_t)at * HD;
    const float2 ml0 = ml[lane < last ? lane : last];
    float o0[FIRST];
#pragma unroll
    for (int j = 0; j < FIRST; j++) o0[j] = sums[(j < last ? j : last) * HD + d];
    float2 ml1 = ml0;
    if (nsplit > 64) ml1 = ml[lane + 64 < last ? lane + 64 : last];
    const float m0 = lane < nsplit ? ml0.x : -INFINITY, m1 = lane + 64 < nsplit ? ml1.x : -INFINITY;
    const float mx = wave_max(fmaxf(m0, m1));
    float w0 = m0 == -INFINITY ? 0.f : __expf(m0 - mx), w1 = m1 == -INFINITY ? 0.f : __expf(m1 - mx);
    // the sum in slice order, so that it does not depend on how lanes are paired (lanes from nsplit on add zero)
    const float l0 = w0 * ml0.y, l1 = w1 * ml1.y;
    auto of_lane = [](float v, int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l)); };
    float den = 0.f;
#pragma unroll
    for (int j = 0; j < FIRST; j++) den += of_lane(l0, j);
    for (int s0 = FIRST; s0 < nsplit; s0 += GROUP) {
        const float l = s0 < 64 ? l0 : l1;
#pragma unroll
        for (int j = 0; j < GROUP; j++) den += of_lane(l, (s0 + j) & 63);
    }
    if (sink) den += __expf(sink[blockIdx.x % H] - mx);           // (some slice holds the query's own key: mx is finite)
    if constexpr (BY_POSITION) if (by_position.gate) den /= head_gate(by_position, blockIdx.x / H, blockIdx.x % H);
    w0 /= den;
    w1 /= den;
    float num = 0.f;
#pragma unroll
    for (int j = 0; j < FIRST; j++) {
        const float w = of_lane(w0, j);
        num += w == 0.f ? 0.f : w * o0[j];
    }
    for (int s0 = FIRST; s0 < nsplit; s0 += GROUP) {
        float o[GROUP];
#pragma unroll
        for (int j = 0; j < GROUP; j++) o[j] = sums[(s0 + j < last ? s0 + j : last) * HD + d];
        const float v = s0 < 64 ? w0 : w1;
#pragma unroll
        for (int j = 0; j < GROUP; j++) {
            const float w = of_lane(v, (s0 + j) & 63);
            num += w == 0.f ? 0.f : w * o[j];
        }
    }
    if (tid < HD) out[(size_t)blockIdx.x * HD + tid] = f32_to_bf16(num);
}

extern "C" long tp_attn_decode_workspace_floats(int n_seq, int H, int nsplit) {
    return nsplit > 1 ? (long)n_seq * H * nsplit * (HD + 2) : 0;
}

static int decode_launch(DecodeArgs a, int n_seq, void* workspace, hipStream_t s) {
    TP_REQUIRE(n_seq > 0 && a.H > 0 && a.KV > 0, "attention decode: empty shape");
    TP_REQUIRE(a.H % a.KV == 0, "attention: %d query heads are no multiple of %d kv heads", a.H, a.KV);
    const int G = a.H / a.KV;
    TP_REQUIRE(G <= 16, "attention decode (matrix-core kernel): %d query heads per kv head exceed 16", G);
    a.G = G;
    if (a.pool_kv == 0) a.pool_kv = a.KV;
    TP_REQUIRE(a.pool_kv > 0 && a.KV % a.pool_kv == 0 && (a.pool_kv == a.KV || !a.qkv),
               "attention decode: %d groups of heads cannot share %d kv heads of the cache", a.KV, a.pool_kv);
    TP_REQUIRE(a.page >= 16 && (a.page & (a.page - 1)) == 0 && a.table_w > 0, "attention decode (matrix-core kernel): page size %d must be a power of two, at least 16", a.page);
    TP_REQUIRE(a.chunk >= 0, "attention decode: chunks of %d positions", a.chunk);
    TP_REQUIRE(a.keep >= 0 && a.pin >= 0 && a.pin % a.page == 0 && (a.keep == 0 || (a.window > 0 && a.chunk == 0)), "attention decode: %d kept positions (%d rows before the ring) stand beside a window, without chunks", a.keep, a.pin);
    TP_REQUIRE(a.rows_cap == 0 || (a.pin < a.rows_cap && a.keep <= a.pin), "attention decode: %d kept positions and %d rows before a ring do not fit a cache of %d rows", a.keep, a.pin, a.rows_cap);
    const int reach = a.window > 0 && a.chunk > 0 ? (a.window < a.chunk ? a.window : a.chunk) : (a.window > 0 ? a.window : a.chunk);
    TP_REQUIRE(a.rows_cap == 0 || (reach > 0 && reach <= a.rows_cap - a.pin), "attention decode: a reach of %d keys (window %d, chunk %d) does not fit a ring of %d rows", reach, a.window, a.chunk, a.rows_cap - a.pin);
    TP_REQUIRE(a.rows_cap >= 0 && a.rows_cap % a.page == 0, "attention decode: ring of %d rows is no multiple of the page size %d", a.rows_cap, a.page);
    const bool whole = a.nsplit == 0;
    if (whole) a.nsplit = 1;
    TP_REQUIRE(!whole || G <= 8, "attention decode: %d query heads per kv head exceed the 8 of a block with all keys", G);
    TP_REQUIRE(a.nsplit >= 1 && a.nsplit <= 128 && (a.nsplit == 1 || workspace), "attention decode: %d slices (at most 128) need a workspace", a.nsplit);
    TP_REQUIRE(a.KV <= 65535 && n_seq <= 65535, "attention decode: grid too large");
    if (a.nsplit > 1) {
        a.ws_o = (float*)workspace;
        a.ws_ml = a.ws_o + (size_t)n_seq * a.H * a.nsplit * HD;
    }
    dim3 grid(a.KV, n_seq, a.nsplit);
    if (whole) {
        if (G <= 1) attn_decode_k<1, WHOLE_WAVES><<<grid, 64 * WHOLE_WAVES, 0, s>>>(a);
        else if (G <= 2) attn_decode_k<2, WHOLE_WAVES><<<grid, 64 * WHOLE_WAVES, 0, s>>>(a);
        else if (G <= 4) attn_decode_k<4, WHOLE_WAVES><<<grid, 64 * WHOLE_WAVES, 0, s>>>(a);
        else attn_decode_k<8, WHOLE_WAVES><<<grid, 64 * WHOLE_WAVES, 0, s>>>(a);
        return tp_check_launch("attention decode (whole)");
    }
    constexpr int DTH = 64 * DWAVES;
    if (G <= 1) attn_decode_k<1><<<grid, DTH, 0, s>>>(a);
    else if (G <= 2) attn_decode_k<2><<<grid, DTH, 0, s>>>(a);
    else if (G <= 4) attn_decode_k<4><<<grid, DTH, 0, s>>>(a);
    else if (G <= 8) attn_decode_k<8><<<grid, DTH, 0, s>>>(a);
    else attn_decode_k<16><<<grid, DTH, 0, s>>>(a);
    if (int rc = tp_check_launch("attention decode")) return rc;
    if (a.nsplit > 1) {
        attn_decode_combine_k<<<dim3(n_seq * a.H, (HD + 63) / 64), 64, 0, s>>>(a.ws_o, a.ws_ml, a.nsplit, a.out, a.sink, a.H, a.by_position);
        return tp_check_launch("attention decode (combine)");
    }
    return 0;
}

static int take_positional(DecodeArgs& a, const TpPositional* by_position) {
    if (!by_position) return 0;
    TP_REQUIRE(BY_POSITION, "attention decode: this library's kernels know no scores by position");
    TP_REQUIRE(tp_positional_ok(by_position), "attention decode: a bias, a temperature or a gate that does not fit");
    a.by_position = *by_position;
    return 0;
}

extern "C" int tp_attn_decode(const void* q, long q_stride, int n_seq, int H, int KV, const int* new_len,
                              const int* table, int table_w, const void* k_pool, const void* v_pool, int page,
                              int rows_cap, float scale, float cap, int window, int chunk, const float* head_scale,
                              const float* sink, int keep, int pin, const TpPositional* by_position, void* out, void* workspace, int nsplit, void* stream) {
    TP_REQUIRE(q_stride % 8 == 0 && (uintptr_t)q % 16 == 0, "attention decode: query rows must be 16-byte aligned");
    DecodeArgs a{(const bf16_t*)q, q_stride, H, KV, new_len, table, table_w, (bf16_t*)k_pool, (bf16_t*)v_pool,
                 page, rows_cap, scale, cap, window, (bf16_t*)out, nullptr, nullptr, nsplit,
                 nullptr, 0, 1, 0, 0, nullptr, 0, 0, 0, chunk, head_scale, sink, keep, pin, TpPositional{}, 0};
    if (int rc = take_positional(a, by_position)) return rc;
    return decode_launch(a, n_seq, workspace, (hipStream_t)stream);
}

// The same over a cache with `pool_kv` kv heads read by `KV` groups of query heads (KV a multiple of pool_kv): group j
// reads pool head j % pool_kv.  With one row per token for all heads (pool_kv 1) the heads are cut into groups, each a
// block's worth of weighted sums, instead of one block forming all of them.
extern "C" int tp_attn_decode_shared(const void* q, long q_stride, int n_seq, int H, int KV, int pool_kv, const int* new_len,
                                     const int* table, int table_w, const void* k_pool, const void* v_pool, int page,
                                     int rows_cap, float scale, float cap, int window, const float* sink, void* out, void* workspace,
                                     int nsplit, void* stream) {
    TP_REQUIRE(q_stride % 8 == 0 && (uintptr_t)q % 16 == 0, "attention decode: query rows must be 16-byte aligned");
    DecodeArgs a{(const bf16_t*)q, q_stride, H, KV, new_len, table, table_w, (bf16_t*)k_pool, (bf16_t*)v_pool,
                 page, rows_cap, scale, cap, window, (bf16_t*)out, nullptr, nullptr, nsplit,
                 nullptr, 0, 1, 0, 0, nullptr, 0, 0, pool_kv, 0, nullptr, sink, 0, 0, TpPositional{}, 0};
    return decode_launch(a, n_seq, workspace, (hipStream_t)stream);
}

// One launch for a decode step's rotation, cache write and attention: `qkv` holds each sequence's projections
// [heads | kv heads (keys) | kv heads (values)] x head size (queries only when write_kv is 0) as bf16 rows, or as
// float32 rows in n_slices K slices `slice_stride` elements apart.  Sequence i's new token has position new_len[i] - 1.
extern "C" int tp_attn_decode_fused(const void* qkv, int qkv_dtype, int n_slices, long slice_stride, long row_stride,
                                    const float* inv_freq, int rot, int write_kv,
                                    int n_seq, int H, int KV, const int* new_len, const int* table, int table_w,
                                    void* k_pool, void* v_pool, int page, int rows_cap, float scale, float cap,
                                    int window, const float* sink, int keep, int pin, const TpPositional* by_position, void* out, void* workspace, int nsplit, void* stream) {
    TP_REQUIRE(qkv, "attention decode (fused): no projections");
    TP_REQUIRE(qkv_dtype == TP_BF16 || qkv_dtype == TP_F32, "attention decode (fused): projections of dtype %d", qkv_dtype);
    TP_REQUIRE(n_slices >= 1 && (n_slices == 1 || qkv_dtype == TP_F32), "attention decode (fused): %d slices must be float32", n_slices);
    TP_REQUIRE(rot >= 0 && rot <= HD && rot % 2 == 0, "attention decode (fused): rotary_dim %d must be even and at most head_dim %d", rot, HD);
    TP_REQUIRE(rot == 0 || inv_freq, "attention decode (fused): a rotation needs its frequency table");
    TP_REQUIRE(row_stride >= (long)(H + (write_kv ? 2 * KV : 0)) * HD, "attention decode (fused): rows of %ld elements are too short", row_stride);
    DecodeArgs a{nullptr, 0, H, KV, new_len, table, table_w, (bf16_t*)k_pool, (bf16_t*)v_pool,
                 page, rows_cap, scale, cap, window, (bf16_t*)out, nullptr, nullptr, nsplit,
                 qkv, qkv_dtype == TP_F32 ? 1 : 0, n_slices, slice_stride, row_stride, inv_freq, rot, write_kv, 0, 0, nullptr, sink, keep, pin, TpPositional{}, 0};
    if (int rc = take_positional(a, by_position)) return rc;
    return decode_launch(a, n_seq, workspace, (hipStream_t)stream);
}
