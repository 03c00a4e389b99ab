// Plain attention kernel for any dtype, head size up to 1024 and any grouping: a block of eight waves per (row, query head).
//
// The keys that the query sees are cut, from the first on, into groups of up to four; state w of eight takes the groups w, w + 8,
// .. with a running softmax of its own, and the eight states are joined in order at the end.  What bounds it is latency: a
// group's key and value rows are fetched while the group before is worked on, the dot products of its keys are summed over the
// wave together (seven exchanges instead of six a key, by lane moves), and eight waves, one a state, have their chains in flight.  (One wave, a
// key after the other, took 0.63 us a key: 132 us of a float32 decode step's layer at 200 keys and heads of 256, 11 us so.)
// Where a launch has many rows of few keys a wave takes a row and forms its eight states itself: the same bits (2,048 rows with a
// window of 3 and heads of 64: 91 us by blocks, 14 by waves).
//
// It is the float32 path's attention for prefill and decode alike (the groups and their order depend on what the query
// sees alone, so a token's result does not depend on how the prompt was cut), and the bf16 path's fallback for
// shapes the matrix-core kernels refuse.  Formula and order as the reference's attn_k
// (runtime/cuda/codebook_gemv.cu:240-270): score = dot * scale, cap * tanh(score / cap), softmax, weighted
// sum of v, kv head = head / (heads / kv_heads); the scale is an argument (rsqrt(head_dim) there), and a
// window W hides keys with p - t >= W (none there).  Beyond the reference: with chunks of C positions the query at p
// sees only keys from floor(p / C) C on; a head may have a temperature that multiplies its scores and a sink, a score
// without key or value whose exponential joins the denominator once, after the keys.  With `keep` the first keep positions
// of a sequence stay visible behind the window; in a ring they live in the `pin` rows in front of it.  A temperature of the
// query's position, a bias per distance and a gate per head come with TpPositional (common.h).
#include "common.h"

struct AttnSimpleArgs {
    const void* q; long q_stride;
    // keys and values of the step itself (prefill): rows of sequence s start at cu_rows[s] and stand at the
    // positions from new_len[s] - count on (from 0 without new_len); row_pos holds every row's position
    const void* k; long k_stride; const void* v; long v_stride;
    const int* cu_rows; const int* row_seq; const int* row_pos;
    // keys and values in the paged cache: all of them in a decode step (sequence i is row i, its last position
    // new_len[i] - 1), the positions before the step's own rows otherwise
    const int* new_len; const int* table; int table_w; const void* k_pool; const void* v_pool; int page; int rows_cap;
    void* out;
    int H, KV, hd; float scale, cap; int window; int paged;
    int chunk; const float* head_scale; const float* sink;        // 0 and null: none
    TpPositional by_position;
    int keep, pin;                                       // positions seen beside the window; rows of the cache in front of its ring
    int page_shift;                                      // the page size's power of two, -1 if it is none (set by the launch)
};

namespace {
constexpr int WAVES = 8;

// The maximum of a state that has seen no score: finite, so that a group of scores that are all -infinity, by a bias or an overflow,
// adds nothing to it (-infinity would give NaN).
constexpr float NONE = -3.4028235e38f;

// One query of one head: what a lane holds of it, and its keys in groups.  NJ: elements of a head a lane holds (head sizes up to
// 64 NJ); KEYS: keys of a group (4, 2 or 1: what the registers hold).
template <typename T, int NJ, int KEYS>
struct Query {
    const AttnSimpleArgs& a;
    int h, lane, g, seq, p, start, lo, kept, n_keys;
    float scale, q[NJ];
    const float* bias;

    __device__ __forceinline__ Query(const AttnSimpleArgs& args, int r, int head, int l) : a(args), h(head), lane(l), g(head / (args.H / args.KV)), start(0) {
        if (a.paged) { seq = r; p = a.new_len[r] - 1; start = p + 1; }      // start: the first position that is a row of the step
        else {
            seq = a.row_seq[r];
            p = a.row_pos[r];
            if (a.new_len) start = a.new_len[seq] - (a.cu_rows[seq + 1] - a.cu_rows[seq]);
        }
        lo = a.window > 0 ? max(0, p - a.window + 1) : 0;
        if (a.chunk > 0) lo = max(lo, p / a.chunk * a.chunk);
        scale = (a.head_scale ? a.scale * a.head_scale[h] : a.scale) * query_temperature(a.by_position, p);
        bias = a.by_position.bias ? a.by_position.bias + (size_t)h * (a.by_position.reach + 1) : nullptr;
        const T* row = (const T*)a.q + (size_t)r * a.q_stride + (size_t)h * a.hd;
#pragma unroll
        for (int j = 0; j < NJ; j++) q[j] = lane + 64 * j < a.hd ? ld_f32(row + lane + 64 * j) : 0.f;
        // the keys in order: the kept ones before the window, then the window's
        kept = min(a.keep, lo);
        n_keys = kept + p - lo + 1;
    }
    // where key i stands
    __device__ __forceinline__ int at(int i) const { return i < kept ? i : lo + i - kept; }

    // the key rows and the value rows of the group that starts at key `first`
    template <bool KEY, bool VALUE>
    __device__ __forceinline__ void fetch(int first, float (*kk)[NJ], float (*vv)[NJ]) const {
#pragma unroll
        for (int n = 0; n < KEYS; n++) {
            const int t = min(at(first + n), p);             // past the last key: a row that exists, without weight
            const T *kp, *vp;
            if (t < start) {
                // (a division is some thirty instructions, and a group has its keys' in a row before its loads)
                const int ring = a.rows_cap - a.pin, u = t - a.pin;
                const int row = a.rows_cap > 0 && u >= ring ? a.pin + u % ring : t;
                const int page = a.page_shift >= 0 ? row >> a.page_shift : row / a.page;
                const int pg = a.table[(size_t)seq * a.table_w + page];
                const size_t off = (((size_t)pg * a.KV + g) * a.page + (row - page * a.page)) * a.hd;
                kp = (const T*)a.k_pool + off;
                vp = (const T*)a.v_pool + off;
            } else {
                const size_t row = (size_t)(a.cu_rows[seq] + t - start);
                kp = (const T*)a.k + row * a.k_stride + (size_t)g * a.hd;
                vp = (const T*)a.v + row * a.v_stride + (size_t)g * a.hd;
            }
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const int d = lane + 64 * j;
                const unsigned dc = d < a.hd ? d : 0;
                const float kx = KEY ? ld_f32(kp + dc) : 0.f, vx = VALUE ? ld_f32(vp + dc) : 0.f;
                if (KEY) kk[n][j] = d < a.hd ? kx : 0.f;
                if (VALUE) vv[n][j] = d < a.hd ? vx : 0.f;
            }
        }
    }

    // no weight times a value of infinity: what stands in for keys past the last one becomes zero
    __device__ __forceinline__ void drop_past(int first, float (&vv)[KEYS][NJ]) const {
        if (first + KEYS <= n_keys) return;
#pragma unroll
        for (int n = 1; n < KEYS; n++)
            if (first + n >= n_keys)
#pragma unroll
                for (int j = 0; j < NJ; j++) vv[n][j] = 0.f;
    }

    // the scores of a group: a lane is left with that of its key lane % KEYS
    __device__ __forceinline__ float score(int first, const float (&kk)[KEYS][NJ]) const {
        float part[KEYS];
#pragma unroll
        for (int n = 0; n < KEYS; n++) {
            part[n] = 0.f;
#pragma unroll
            for (int j = 0; j < NJ; j++) part[n] = fmaf(q[j], kk[n][j], part[n]);
        }
        const int mine = lane & (KEYS - 1);
        float s = part[0];
        if constexpr (KEYS == 4) {
            const float s01 = ((lane & 1) ? part[1] : part[0]) + across_f<1>((lane & 1) ? part[0] : part[1], lane);
            const float s23 = ((lane & 1) ? part[3] : part[2]) + across_f<1>((lane & 1) ? part[2] : part[3], lane);
            s = ((lane & 2) ? s23 : s01) + across_f<2>((lane & 2) ? s01 : s23, lane);
        } else if constexpr (KEYS == 2) {
            s = ((lane & 1) ? part[1] : part[0]) + across_f<1>((lane & 1) ? part[0] : part[1], lane);
        }
        if constexpr (KEYS == 1) {                           // (heads of more than 512: 11.0 us by shuffles, 13.2 by lane moves, 40 keys)
#pragma unroll
            for (int x = 1; x < 64; x <<= 1) s += __shfl_xor(s, x, 64);
        } else {
            if constexpr (KEYS == 2) s += across_f<2>(s, lane);
            s += across_f<4>(s, lane);
            s += across_f<8>(s, lane);
            s += across_f<16>(s, lane);
            s += across_f<32>(s, lane);
        }
        s *= scale;
        if (a.cap > 0.f) s = softcap_f(s, a.cap);
        if (bias) s += bias[min(max(p - at(first + mine), 0), (int)a.by_position.reach)];
        return first + mine >= n_keys ? -INFINITY : s;
    }

    // the largest score of a group, in every lane
    __device__ __forceinline__ float top_of(float s) const {
        if constexpr (KEYS > 1) s = fmaxf(s, across_f<1>(s, lane));
        if constexpr (KEYS > 2) s = fmaxf(s, across_f<2>(s, lane));
        return s;
    }

    // a group into a running softmax (m, l, o)
    __device__ __forceinline__ void add(float s, const float (&vv)[KEYS][NJ], float& m, float& l, float (&o)[NJ]) const {
        const float m_new = fmaxf(m, top_of(s)), alpha = expf(m - m_new), pr = expf(s - m_new);
        float sum = pr;
        if constexpr (KEYS > 1) sum += across_f<1>(sum, lane);
        if constexpr (KEYS > 2) sum += across_f<2>(sum, lane);
        l = fmaf(l, alpha, sum);
        float w[KEYS];
#pragma unroll
        for (int n = 0; n < KEYS; n++) w[n] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(pr), n));
#pragma unroll
        for (int j = 0; j < NJ; j++) o[j] *= alpha;
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int n = 0; n < KEYS; n++) o[j] = fmaf(w[n], vv[n][j], o[j]);
        m = m_new;
    }

    // states that saw a key
    __device__ __forceinline__ int states() const { return min(WAVES, (n_keys + KEYS - 1) / KEYS); }
    __device__ __forceinline__ float with_sink(float top) const { return a.sink ? fmaxf(top, a.sink[h]) : top; }
    // what the states' sum is multiplied by
    __device__ __forceinline__ float inverse(float total, float top, int r) const {
        if (a.sink) total += expf(a.sink[h] - top);
        return (a.by_position.gate ? head_gate(a.by_position, r, h) : 1.f) / total;
    }
};
}

template <typename T, int NJ, int KEYS>
__global__ void __launch_bounds__(64 * WAVES)
attn_simple_k(AttnSimpleArgs a) {
    __shared__ float part_o[WAVES][64 * NJ], part_m[WAVES], part_l[WAVES];
    const int h = blockIdx.y, r = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Query<T, NJ, KEYS> query(a, r, h, lane);
    const int n_keys = query.n_keys;
    float m = NONE, l = 0.f, o[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) o[j] = 0.f;
    float k0[KEYS][NJ], v0[KEYS][NJ], k1[KEYS][NJ], v1[KEYS][NJ];
    int i = wave * KEYS;
    if (i < n_keys) {
        query.template fetch<true, true>(i, k0, v0);
        while (true) {
            const int i1 = i + WAVES * KEYS;
            if (i1 < n_keys) query.template fetch<true, true>(i1, k1, v1);
            query.drop_past(i, v0);
            query.add(query.score(i, k0), v0, m, l, o);
            if (i1 >= n_keys) break;
            i = i1 + WAVES * KEYS;
            if (i < n_keys) query.template fetch<true, true>(i, k0, v0);
            query.drop_past(i1, v1);
            query.add(query.score(i1, k1), v1, m, l, o);
            if (i >= n_keys) break;
        }
    }
#pragma unroll
    for (int j = 0; j < NJ; j++) part_o[wave][lane + 64 * j] = o[j];
    if (lane == 0) { part_m[wave] = m; part_l[wave] = l; }
    __syncthreads();
    const int used = query.states();
    float top = part_m[0];
    for (int w = 1; w < used; w++) top = fmaxf(top, part_m[w]);
    top = query.with_sink(top);
    float f[WAVES], total = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        f[w] = w < used ? expf(part_m[w] - top) : 0.f;
        if (w < used) total = fmaf(part_l[w], f[w], total);
    }
    const float inv = query.inverse(total, top, r);
    T* out = (T*)a.out + ((size_t)r * a.H + h) * a.hd;
    for (int d = threadIdx.x; d < a.hd; d += 64 * WAVES) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; w++)
            if (w < used) t = fmaf(part_o[w][d], f[w], t);
        st_f32(out + d, t * inv);
    }
}

// The same sums by one wave a (row, query head), for launches of many rows that see few keys, where most of a block's eight waves
// would be launched for a group or for none.  The wave takes the scores first, which gives the join's maximum and fills its
// stretch of LDS, and then forms the eight states one after the other (of keys beyond ROWS_KEYS, which the launch does not send
// here, the scores are formed again).
constexpr int ROWS_KEYS = 64;

template <typename T, int NJ, int KEYS>
__global__ void __launch_bounds__(64 * WAVES, NJ <= 4 ? 6 : NJ <= 8 ? 5 : 4)
attn_simple_rows_k(AttnSimpleArgs a, int M) {
    __shared__ float scores[WAVES][ROWS_KEYS];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = blockIdx.x * WAVES + wave;
    if (r >= M) return;
    const Query<T, NJ, KEYS> query(a, r, blockIdx.y, lane);
    const int n_keys = query.n_keys, mine = lane & (KEYS - 1);
    float x0[KEYS][NJ], x1[KEYS][NJ];                         // the keys' rows, then the values'
    float top = NONE, total = 0.f, t[NJ], m = NONE, l = 0.f, o[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) t[j] = o[j] = 0.f;
    auto fold = [&]() {                                       // a state that has seen its keys into the row's sum
        const float f = expf(m - top);
        total = fmaf(l, f, total);
#pragma unroll
        for (int j = 0; j < NJ; j++) { t[j] = fmaf(o[j], f, t[j]); o[j] = 0.f; }
        m = NONE;
        l = 0.f;
    };
    if (n_keys <= KEYS) {                                     // one group: its keys and values in one trip
        if (n_keys > 0) {
            query.template fetch<true, true>(0, x0, x1);
            const float s = query.score(0, x0);
            top = query.with_sink(fmaxf(top, query.top_of(s)));
            query.drop_past(0, x1);
            query.add(s, x1, m, l, o);
            fold();
        } else top = query.with_sink(top);
    } else {
        auto take = [&](int i, const float (&kk)[KEYS][NJ]) {
            const float s = query.score(i, kk);
            if (i < ROWS_KEYS) scores[wave][i + mine] = s;    // (the lanes of a key write the same)
            top = fmaxf(top, s);
        };
        query.template fetch<true, false>(0, x0, nullptr);
        for (int i = 0; i < n_keys; i += 2 * KEYS) {
            if (i + KEYS < n_keys) query.template fetch<true, false>(i + KEYS, x1, nullptr);
            take(i, x0);
            if (i + KEYS >= n_keys) break;
            if (i + 2 * KEYS < n_keys) query.template fetch<true, false>(i + 2 * KEYS, x0, nullptr);
            take(i + KEYS, x1);
        }
        top = query.with_sink(query.top_of(top));
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        int i = 0, w = 0;
        auto step = [&](float (&cur)[KEYS][NJ], float (&next)[KEYS][NJ]) {
            int to = i + WAVES * KEYS;
            const bool last = to >= n_keys;                   // of this state's groups
            if (last) to = ++w * KEYS;
            const bool more = w < WAVES && to < n_keys;
            if (more) query.template fetch<false, true>(to, nullptr, next);
            float s;
            if (i < ROWS_KEYS) s = scores[wave][i + mine];
            else {
                float kk[KEYS][NJ];
                query.template fetch<true, false>(i, kk, nullptr);
                s = query.score(i, kk);
            }
            query.drop_past(i, cur);
            query.add(s, cur, m, l, o);
            if (last) fold();
            i = to;
            return more;
        };
        query.template fetch<false, true>(0, nullptr, x0);
        while (step(x0, x1) && step(x1, x0)) {}
    }
    const float inv = query.inverse(total, top, r);
    T* out = (T*)a.out + ((size_t)r * a.H + query.h) * a.hd;
#pragma unroll
    for (int j = 0; j < NJ; j++)
        if (lane + 64 * j < a.hd) st_f32(out + lane + 64 * j, t[j] * inv);
}

static int launch(AttnSimpleArgs a, int dtype, int M, int most, hipStream_t s) {
    a.page_shift = a.page > 0 && (a.page & (a.page - 1)) == 0 ? __builtin_ctz((unsigned)a.page) : -1;
    TP_REQUIRE(a.keep >= 0 && a.pin >= 0 && (a.keep == 0 || (a.window > 0 && a.chunk == 0)), "attention: %d kept positions stand beside a window, without chunks", a.keep);
    TP_REQUIRE(a.rows_cap == 0 || (a.pin < a.rows_cap && a.keep <= a.pin), "attention: %d kept positions and %d rows before a ring do not fit a cache of %d rows", a.keep, a.pin, a.rows_cap);
    TP_REQUIRE(M > 0 && a.H > 0 && a.KV > 0 && a.hd > 0, "attention: empty shape rows=%d heads=%d kv=%d head_dim=%d", M, a.H, a.KV, a.hd);
    TP_REQUIRE(a.H % a.KV == 0, "attention: %d query heads are no multiple of %d kv heads", a.H, a.KV);
    TP_REQUIRE(a.hd <= 1024, "attention (plain kernel): head_dim %d exceeds 1024", a.hd);
    TP_REQUIRE(a.H <= 65535, "attention (plain kernel): %d heads exceed one launch (65535)", a.H);
    dim3 grid(M, a.H);
    if (dtype != TP_BF16 && dtype != TP_F32) return tp_fail("attention: unknown dtype %d", dtype);
    // Rows that see few keys, and so many of them that a wave's longer chain is hidden: 64 rows and heads a key of the most that
    // any sees (twice and four times that for heads of more than 256 and 512 elements, whose groups are two keys and one).
    // Float32, eight heads of 256, microseconds, blocks / waves: 16,384 rows and heads of prompts of 4 tokens 98.9 / 16.1, of 16
    // 118 / 41, of 64 179 / 127, of 128 232 / 236; 4,096 of 64 49.9 / 42.9; 1,024 of 8 9.9 / 8.0, of 32 13.5 / 18.5; 64 of 4 5.3 / 5.3.
    const int group = a.hd <= 256 ? 4 : a.hd <= 512 ? 2 : 1;
    const bool rows = most > 0 && most <= ROWS_KEYS && (long)M * a.H >= 256L / group * most;
    const dim3 grid_rows(tp_cdiv(M, WAVES), a.H);
#define TP_ATTN_SIMPLE_OF(T, NJ, KEYS) do { if (rows) attn_simple_rows_k<T, NJ, KEYS><<<grid_rows, 64 * WAVES, 0, s>>>(a, M); else attn_simple_k<T, NJ, KEYS><<<grid, 64 * WAVES, 0, s>>>(a); } while (0)
#define TP_ATTN_SIMPLE(NJ, KEYS) do { if (dtype == TP_BF16) TP_ATTN_SIMPLE_OF(bf16_t, NJ, KEYS); else TP_ATTN_SIMPLE_OF(float, NJ, KEYS); } while (0)
    if (a.hd <= 64) TP_ATTN_SIMPLE(1, 4);
    else if (a.hd <= 128) TP_ATTN_SIMPLE(2, 4);
    else if (a.hd <= 256) TP_ATTN_SIMPLE(4, 4);
    else if (a.hd <= 512) TP_ATTN_SIMPLE(8, 2);
    else TP_ATTN_SIMPLE(16, 1);
#undef TP_ATTN_SIMPLE
#undef TP_ATTN_SIMPLE_OF
    return tp_check_launch("attention (plain kernel)");
}

// most: a bound on the keys that a row sees, 0 for none (a choice between two ways to the same bits).
// new_len (or null): the sequences' lengths after the step; the positions before a sequence's first row of the step
// are read from the cache (pools [pages, kv_heads, page, head_dim] through `table`), as earlier steps left it
extern "C" int tp_attn_simple_prefill(const void* q, long q_stride, const void* k, long k_stride, const void* v, long v_stride,
                                      int dtype, int M, int H, int KV, int hd, const int* cu_rows, const int* row_seq,
                                      const int* row_pos, const int* new_len, const int* table, int table_w,
                                      const void* k_pool, const void* v_pool, int page, int rows_cap,
                                      float scale, float cap, int window, int chunk, const float* head_scale, const float* sink,
                                      int keep, int pin, const TpPositional* by_position, int most, void* out, void* stream) {
    TP_REQUIRE(chunk >= 0, "attention: chunks of %d positions", chunk);
    TP_REQUIRE(!new_len || (table && k_pool && v_pool && page > 0 && table_w > 0), "attention: cached positions need the page table and the pools");
    AttnSimpleArgs a{};
    a.q = q; a.q_stride = q_stride; a.k = k; a.k_stride = k_stride; a.v = v; a.v_stride = v_stride;
    a.cu_rows = cu_rows; a.row_seq = row_seq; a.row_pos = row_pos;
    a.new_len = new_len; a.table = table; a.table_w = table_w; a.k_pool = k_pool; a.v_pool = v_pool;
    a.page = new_len ? page : 1; a.rows_cap = new_len ? rows_cap : 0;
    a.out = out; a.H = H; a.KV = KV; a.hd = hd; a.scale = scale; a.cap = cap; a.window = window; a.paged = 0;
    a.chunk = chunk; a.head_scale = head_scale; a.sink = sink;
    a.keep = keep; a.pin = pin;
    TP_REQUIRE(tp_positional_ok(by_position), "attention: a bias, a temperature or a gate that does not fit");
    if (by_position) a.by_position = *by_position;
    return launch(a, dtype, M, most, (hipStream_t)stream);
}

extern "C" int tp_attn_simple_decode(const void* q, long q_stride, int dtype, int n_seq, int H, int KV, int hd,
                                     const int* new_len, const int* table, int table_w, const void* k_pool,
                                     const void* v_pool, int page, int rows_cap, float scale, float cap, int window,
                                     int chunk, const float* head_scale, const float* sink, int keep, int pin, const TpPositional* by_position, int most, void* out, void* stream) {
    TP_REQUIRE(chunk >= 0, "attention: chunks of %d positions", chunk);
    TP_REQUIRE(page > 0 && table_w > 0, "attention: page size %d, table width %d", page, table_w);
    AttnSimpleArgs a{};
    a.q = q; a.q_stride = q_stride; a.new_len = new_len; a.table = table; a.table_w = table_w;
    a.k_pool = k_pool; a.v_pool = v_pool; a.page = page; a.rows_cap = rows_cap;
    a.out = out; a.H = H; a.KV = KV; a.hd = hd; a.scale = scale; a.cap = cap; a.window = window; a.paged = 1;
    a.chunk = chunk; a.head_scale = head_scale; a.sink = sink;
    a.keep = keep; a.pin = pin;
    TP_REQUIRE(tp_positional_ok(by_position), "attention: a bias, a temperature or a gate that does not fit");
    if (by_position) a.by_position = *by_position;
    return launch(a, dtype, n_seq, most, (hipStream_t)stream);
}
