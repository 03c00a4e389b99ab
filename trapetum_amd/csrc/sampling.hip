// Token choice on the device: argmax, repetition penalty, temperature / top-k / top-p sampling.
#include "common.h"
#include "no_alloc.h"
#include <mutex>

// ---- argmax: the smallest index among the largest values (strict '>' scan in the reference:
// runtime/src/lib.rs:1376-1380; device twin runtime/cuda/codebook_gemv.cu:548-591).  One block per row. ----
__global__ void __launch_bounds__(1024)
argmax_k(const float* __restrict__ logits, int V, int* __restrict__ out) {
    __shared__ float sval[16];
    __shared__ int sidx[16];
    const float* z = logits + (size_t)blockIdx.x * V;
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    for (int i = threadIdx.x; i < V; i += blockDim.x) {
        const float v = z[i];
        if (v > bv || (v == bv && i < bi)) { bv = v; bi = i; }      // NaN never wins
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(bv, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) { sval[wave] = bv; sidx[wave] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); w++)
            if (sval[w] > bv || (sval[w] == bv && sidx[w] < bi)) { bv = sval[w]; bi = sidx[w]; }
        out[blockIdx.x] = bi == 0x7fffffff ? 0 : bi;
    }
}

// stage 1 of the two-stage form: grid (parts, rows), each block scans one contiguous part of a row
__global__ void __launch_bounds__(256)
argmax_part_k(const float* __restrict__ logits, int V, int per_part, float* __restrict__ pval, int* __restrict__ pidx) {
    __shared__ float sval[4];
    __shared__ int sidx[4];
    const float* z = logits + (size_t)blockIdx.y * V;
    const int lo = blockIdx.x * per_part, hi = min(V, lo + per_part);
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    for (int i = lo + threadIdx.x; i < hi; i += blockDim.x) {
        const float v = z[i];
        if (v > bv || (v == bv && i < bi)) { bv = v; bi = i; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(bv, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) { sval[wave] = bv; sidx[wave] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; w++)
            if (sval[w] > bv || (sval[w] == bv && sidx[w] < bi)) { bv = sval[w]; bi = sidx[w]; }
        pval[blockIdx.y * gridDim.x + blockIdx.x] = bv;
        pidx[blockIdx.y * gridDim.x + blockIdx.x] = bi;
    }
}

// stage 2: one wave per row over the parts' winners
__global__ void __launch_bounds__(64)
argmax_final_k(const float* __restrict__ pval, const int* __restrict__ pidx, int parts, int* __restrict__ out) {
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    for (int i = threadIdx.x; i < parts; i += 64) {
        const float v = pval[blockIdx.x * parts + i];
        const int id = pidx[blockIdx.x * parts + i];
        if (v > bv || (v == bv && id < bi)) { bv = v; bi = id; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(bv, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
    }
    if (threadIdx.x == 0) out[blockIdx.x] = bi == 0x7fffffff ? 0 : bi;
}

extern "C" long tp_argmax_workspace_bytes(int B, int V) {
    const int parts = V >= 16384 ? 64 : 1;
    return parts > 1 ? (long)B * parts * 8 : 0;
}

extern "C" int tp_argmax(const float* logits, int B, int V, int* out, void* workspace, void* stream) {
    TP_REQUIRE(B > 0 && V > 0, "argmax: empty shape B=%d V=%d", B, V);
    TP_REQUIRE(B <= 65535, "argmax: %d rows exceed one launch", B);
    const int parts = V >= 16384 ? 64 : 1;
    hipStream_t s = (hipStream_t)stream;
    if (parts == 1 || !workspace) {
        argmax_k<<<B, 1024, 0, s>>>(logits, V, out);
        return tp_check_launch("argmax");
    }
    float* pval = (float*)workspace;
    int* pidx = (int*)(pval + (size_t)B * parts);
    argmax_part_k<<<dim3(parts, B), 256, 0, s>>>(logits, V, tp_cdiv(V, parts), pval, pidx);
    if (int rc = tp_check_launch("argmax (parts)")) return rc;
    argmax_final_k<<<B, 64, 0, s>>>(pval, pidx, parts, out);
    return tp_check_launch("argmax (final)");
}

// ---- argmax for callers that cannot allocate (declared in no_alloc.h) -------------------------------------------
// The two-stage form above with the parts' winners in a file-scope device array instead of a caller's workspace.
// Every GPU the library runs on holds its own copy of the array (128 KiB) until the process ends; in host code the
// array's name is only a handle, so its device address is asked for once per device (hipGetSymbolAddress with that
// device current) and kept.  Nothing in the array has to start at zero: stage 2 reads exactly the B * parts pairs
// that stage 1 of the same call wrote.  All calls on one GPU share the array: calls that overlap there (two
// streams, two threads) race.
static __device__ __align__(256) unsigned char scratch[TP_ARGMAX_NO_ALLOC_SCRATCH_BYTES];

namespace {
constexpr int NO_ALLOC_MAX_DEVICES = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[NO_ALLOC_MAX_DEVICES];        // per device: where that GPU's copy of `scratch` lies

int scratch_address(void** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return tp_fail("argmax_no_alloc: no current device: %s", hipGetErrorString(e));
    TP_REQUIRE(dev >= 0 && dev < NO_ALLOC_MAX_DEVICES, "argmax_no_alloc: device %d is beyond the %d this library keeps track of", dev, NO_ALLOC_MAX_DEVICES);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return tp_fail("argmax_no_alloc: the scratch array's address on device %d is not available: %s", dev, hipGetErrorString(e));
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}
}  // namespace

extern "C" int tp_argmax_no_alloc_prepare(void) {
    void* base = nullptr;
    return scratch_address(&base);
}

extern "C" int tp_argmax_no_alloc(const float* logits, int B, int V, int* out, void* stream) {
    TP_REQUIRE(logits && out, "argmax_no_alloc: logits and output must be given");
    TP_REQUIRE(B > 0 && V > 0, "argmax_no_alloc: empty shape B=%d V=%d", B, V);
    TP_REQUIRE(B <= TP_ARGMAX_NO_ALLOC_MAX_ROWS, "argmax_no_alloc: %d rows exceed the %d that the fixed scratch array holds",
               B, TP_ARGMAX_NO_ALLOC_MAX_ROWS);
    static_assert((size_t)TP_ARGMAX_NO_ALLOC_MAX_ROWS * TP_ARGMAX_NO_ALLOC_PARTS * 8 <= TP_ARGMAX_NO_ALLOC_SCRATCH_BYTES,
                  "the scratch array must hold a (value, index) pair per row and part");
    void* base = nullptr;
    if (int rc = scratch_address(&base)) return rc;
    const int parts = TP_ARGMAX_NO_ALLOC_PARTS;
    float* pval = (float*)base;
    int* pidx = (int*)(pval + (size_t)B * parts);
    hipStream_t s = (hipStream_t)stream;
    argmax_part_k<<<dim3(parts, B), 256, 0, s>>>(logits, V, tp_cdiv(V, parts), pval, pidx);
    if (int rc = tp_check_launch("argmax_no_alloc (parts)")) return rc;
    argmax_final_k<<<B, 64, 0, s>>>(pval, pidx, parts, out);
    return tp_check_launch("argmax_no_alloc (final)");
}

// ---- repetition penalty: every distinct recent token once, z / penalty if z > 0 else z * penalty
// (runtime/src/bin/serve.rs:285-294; the reference keeps the last 128 tokens, prompt included, as a set). -----
__global__ void repetition_penalty_k(float* __restrict__ logits, int V, const int* __restrict__ recent, int R, float penalty) {
    float* z = logits + (size_t)blockIdx.x * V;
    const int* rec = recent + (size_t)blockIdx.x * R;
    for (int j = threadIdx.x; j < R; j += blockDim.x) {
        const int t = rec[j];
        if (t < 0 || t >= V) continue;
        bool first = true;
        for (int i = 0; i < j; i++) if (rec[i] == t) { first = false; break; }
        if (!first) continue;
        const float v = z[t];
        z[t] = v > 0.f ? v / penalty : v * penalty;
    }
}

extern "C" int tp_repetition_penalty(float* logits, int B, int V, const int* recent, int R, float penalty, void* stream) {
    TP_REQUIRE(B > 0 && V > 0 && R > 0, "repetition_penalty: empty shape B=%d V=%d R=%d", B, V, R);
    if (penalty <= 1.f) return 0;
    repetition_penalty_k<<<B, 128, 0, (hipStream_t)stream>>>(logits, V, recent, R, penalty);
    return tp_check_launch("repetition_penalty");
}

// The recent tokens of a row as a ring on the device, so that a captured decode graph can keep them by itself: the
// row's chosen id goes to the place its cursor names, and the cursor moves on (the oldest id is overwritten once
// the ring is full; the penalty reads the ring as a set, so the order inside it does not matter).
__global__ void recent_push_k(const int* __restrict__ tokens, int* __restrict__ recent, int* __restrict__ cursor, int B, int R) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B) return;
    int at = cursor[i];
    at = at < 0 || at >= R ? 0 : at;
    recent[(size_t)i * R + at] = tokens[i];
    cursor[i] = at + 1 == R ? 0 : at + 1;
}

extern "C" int tp_recent_push(const int* tokens, int* recent, int* cursor, int B, int R, void* stream) {
    TP_REQUIRE(tokens && recent && cursor && B > 0 && R > 0, "recent_push: empty shape B=%d R=%d", B, R);
    recent_push_k<<<tp_cdiv(B, 64), 64, 0, (hipStream_t)stream>>>(tokens, recent, cursor, B, R);
    return tp_check_launch("recent_push");
}

// ---- temperature sampling over the top_k largest logits with a top_p cut, as the reference's next_tok
// (runtime/src/bin/serve.rs:41-72): candidates sorted by logit descending (ties: smaller id first),
// p = exp((z - max) / T) / sum, the shortest prefix whose cumulative mass reaches top_p, then a walk with
// r = u * kept mass; falls back to the first candidate.  One block per row: a radix select over the value
// bits finds the k-th largest logit, an id select breaks ties at that value, the at most 1024 candidates are
// sorted in LDS, and the first wave does the short scans (sums in candidate order within a lane, then over the lanes). ---
__device__ __forceinline__ uint32_t value_key(float f) {           // larger float -> larger key; NaN lowest
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t k) {
    const uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
    return __uint_as_float(u);
}

// ---- the sampler's short scans, done by the block's first wave (a single thread walking LDS pays its latency per
// element: 45 us for 256 candidates) -----------------------------------------------------------------------------
__device__ __forceinline__ unsigned wave_scan_incl(unsigned v, int lane) {
    // within rows of 16 by moves (zeros come in from the left), then each row's last on to the rows behind it
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);
    const unsigned r0 = (unsigned)__builtin_amdgcn_readlane((int)v, 15), r1 = (unsigned)__builtin_amdgcn_readlane((int)v, 31), r2 = (unsigned)__builtin_amdgcn_readlane((int)v, 47);
    const int row = lane >> 4;
    return v + (row > 0 ? r0 : 0u) + (row > 1 ? r1 : 0u) + (row > 2 ? r2 : 0u);
}
__device__ __forceinline__ float wave_scan_incl(float v, int lane) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const float t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}
// Walks the 256 counters from the top (or from the bottom) until `rem` of them are covered: the bucket that holds the
// rem-th member, and how many of that bucket are still needed.  All 64 lanes of one wave call it.
__device__ __forceinline__ void pick_bucket(const unsigned* hist, bool from_top, unsigned rem, int lane, int& bucket, unsigned& rem_out) {
    unsigned c[4], local = 0u;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int o = lane * 4 + j;
        c[j] = hist[from_top ? 255 - o : o];
        local += c[j];
    }
    const unsigned incl = wave_scan_incl(local, lane);
    const unsigned long long hit = __ballot(incl >= rem);
    const int L = hit ? __ffsll((long long)hit) - 1 : 63;
    unsigned r = rem - (incl - local);
    int j = 0;
    for (; j < 3; j++) {
        if (c[j] >= r) break;
        r -= c[j];
    }
    const int o = L * 4 + __shfl(j, L, 64);
    bucket = from_top ? 255 - o : o;
    rem_out = (unsigned)__shfl((int)r, L, 64);
}

__device__ __forceinline__ int wave_least(int v, int lane) {
    v = min(v, (int)across<32>((uint32_t)v, lane));
    v = min(v, (int)across<16>((uint32_t)v, lane));
    v = min(v, (int)across<8>((uint32_t)v, lane));
    v = min(v, (int)across<4>((uint32_t)v, lane));
    v = min(v, (int)across<2>((uint32_t)v, lane));
    return min(v, (int)across<1>((uint32_t)v, lane));
}
// A candidate as one number, larger first: its value key, then the smaller id.
__device__ __forceinline__ unsigned long long packed(uint32_t key, int id) { return (unsigned long long)key << 32 | (uint32_t)~id; }

// lanes whose bit STRIDE is clear
__device__ constexpr unsigned long long lanes_below(int stride) {
    unsigned long long m = 0;
    for (int l = 0; l < 64; l++) if (!(l & stride)) m |= 1ull << l;
    return m;
}
// One exchange: lanes of the mask `firsts` keep the larger of their element and that of lane ^ STRIDE, the others the smaller.
template <int STRIDE>
__device__ __forceinline__ void sort_step(unsigned long long& e, int lane, unsigned long long firsts) {
    const unsigned long long o = (unsigned long long)across<STRIDE>((uint32_t)(e >> 32), lane) << 32 | across<STRIDE>((uint32_t)e, lane);
    if (__builtin_amdgcn_inverse_ballot_w64(__builtin_amdgcn_ballot_w64(e > o) ^ firsts)) e = o;
}
template <int SIZE, int STRIDE>
__device__ __forceinline__ void sort_within(unsigned long long& e, int lane) {       // stage SIZE (up to 32) of a wave, from STRIDE down
    constexpr unsigned long long firsts = ~(lanes_below(STRIDE) ^ lanes_below(SIZE));
    sort_step<STRIDE>(e, lane, firsts);
    if constexpr (STRIDE > 1) sort_within<SIZE, STRIDE / 2>(e, lane);
}
// the stages from `size` up to n of a bitonic network over the first n threads; those below 64 lie behind every wave already
__device__ __forceinline__ void sort_stages(unsigned long long& e, int size, int n, unsigned long long* lds) {
    const int tid = threadIdx.x, lane = tid & 63;
    int at = 0;                                                        // two places in turn: a round's reads are over before the next but one writes
    lds_barrier();
    for (; size <= n; size <<= 1) {
        for (int stride = size >> 1; stride >= 64; stride >>= 1) {
            lds[at + tid] = e;
            lds_barrier();
            const unsigned long long o = lds[at + (tid ^ stride)];
            at ^= 1024;
            if ((e > o) != (((tid & stride) == 0) == ((tid & size) == 0))) e = o;
        }
        if (tid >= n) continue;                                        // (whole waves: they would take the others' issue slots)
        const unsigned long long turn = __builtin_amdgcn_readfirstlane(tid & size) ? ~0ull : 0ull;
        sort_step<32>(e, lane, lanes_below(32) ^ turn);
        sort_step<16>(e, lane, lanes_below(16) ^ turn);
        sort_step<8>(e, lane, lanes_below(8) ^ turn);
        sort_step<4>(e, lane, lanes_below(4) ^ turn);
        sort_step<2>(e, lane, lanes_below(2) ^ turn);
        sort_step<1>(e, lane, lanes_below(1) ^ turn);
    }
}
// Sorts the block's elements, one a thread, larger first, over the first n threads (a power of two from 64 to 1024): exchanges
// within a wave stay in registers, so that only strides of 64 and more meet in LDS (10 of 55 rounds at 1,024 elements, 6 of 45 at
// 512).  Key and id compared as one number, and masks known when compiled: 45 rounds take 4.4 us less than compared one after the other.
__device__ __forceinline__ void block_sort(unsigned long long& e, int n, unsigned long long* lds) {
    const int lane = threadIdx.x & 63;
    if ((int)threadIdx.x < n) {
        sort_within<2, 1>(e, lane);
        sort_within<4, 2>(e, lane);
        sort_within<8, 4>(e, lane);
        sort_within<16, 8>(e, lane);
        sort_within<32, 16>(e, lane);
    }
    sort_stages(e, 64, n, lds);
}

// The rows' uniform numbers: an array on the device, or (null) up to TP_HOST_UNIFORMS of them that came with the launch, which saves a
// caller who draws them on the host a copy and the wait for it.
#define TP_HOST_UNIFORMS 64
struct Draws { const float* at; float v[TP_HOST_UNIFORMS]; };
__device__ __forceinline__ float draw_of(const Draws& d, int row) { return d.at ? d.at[row] : d.v[row]; }

// ---- groups: a row of many logits is read once, by many blocks, which leave the largest key of every group of 2^shift neighbours (at
// most GROUPS groups).  If t is the k-th largest of these, k logits are at least t, so the k largest all lie in groups whose
// largest is at least t: the sampler looks at little more than k groups and has hardly more than k candidates, whatever the logits'
// range.  (Before: a histogram of the top 12 key bits over many blocks, then everything from the bin of the k-th up copied to a list by many
// blocks, then the sampler.  Microseconds, 8 rows of 256,000, k 256: 5.9 + 10.2 + 10.0 so, 4.0 + 13.3 here; the call
// for 1 row of 32,000, which the sampler read by itself, 47.5 / 17.3.)
constexpr int GROUPS = 4096, GROUPS_MANY = 8192;                     // groups of a row at most; for more than MANY candidates, whose
constexpr int MANY = 512;                                            // groups are many to look at (k 1,024 of 256,000, 1 row: 29.1 / 25.8 us)
constexpr int GROUP_PART = 4096;                                     // logits of a block (1,024 a wave)
constexpr int GROUPS_FROM = 8192;                                    // rows of fewer logits: the sampler alone (1 row, k 256 / 1,024: 6,000 18.7 / 18.8 us against 15.0 / 20.0, 8,192 22.1 / 22.2 against 15.6 / 21.2)
constexpr int LIST = 8192;                                           // candidates that the sampler's LDS holds

static int group_shift(int V, int at_most) {
    int s = 0;
    while (((long)V + (1L << s) - 1) >> s > at_most) s++;
    return s;
}
static int groups_of(int V, int shift) { return (int)(((long)V + (1L << shift) - 1) >> shift); }

// the largest of a row of 16 lanes, in every lane (once lanes 8 apart agree, 4 on is as good as 4 across)
__device__ __forceinline__ uint32_t row_largest(uint32_t m) {
    m = max(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0x128, 0xf, 0xf, true));
    m = max(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0x124, 0xf, 0xf, true));
    m = max(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0x4e, 0xf, 0xf, true));
    return max(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0xb1, 0xf, 0xf, true));
}

__global__ void __launch_bounds__(256)
group_max_k(const float* __restrict__ logits, int V, int shift, int groups, uint32_t* __restrict__ largest) {
    const int lane = threadIdx.x & 63, begin = blockIdx.x * GROUP_PART + (threadIdx.x >> 6) * 1024 + lane, whole = shift > 6 ? (1 << (shift - 6)) - 1 : 0;
    const float* z = logits + (size_t)blockIdx.y * V;
    float v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) v[u] = z[min(begin + u * 64, V - 1)];
    uint32_t* const to = largest + (size_t)blockIdx.y * groups;
    uint32_t m[16];
#pragma unroll
    for (int u = 0; u < 16; u++) m[u] = begin + u * 64 < V ? value_key(v[u]) : 0u;
    if (shift == 6) {
        // 64 neighbours are the lanes of one load: halves and rows of lanes are folded by swapping them between two loads' registers,
        // which leaves four loads' largest in the four rows of 16 lanes
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const auto a = __builtin_amdgcn_permlane32_swap(m[4 * j], m[4 * j + 1], false, false), b = __builtin_amdgcn_permlane32_swap(m[4 * j + 2], m[4 * j + 3], false, false);
            const auto c = __builtin_amdgcn_permlane16_swap(max(a[0], a[1]), max(b[0], b[1]), false, false);
            const uint32_t largest_of = row_largest(max(c[0], c[1]));
            const int u = 4 * j + ((lane >> 5) & 1) + ((lane >> 4) & 1) * 2, group = (begin - lane + u * 64) >> 6;
            if ((lane & 15) == 0 && group < groups) to[group] = largest_of;
        }
        return;
    }
    if (shift == 5) {                                                // the same with rows of 16 lanes alone: two loads' in the four rows
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const auto c = __builtin_amdgcn_permlane16_swap(m[2 * j], m[2 * j + 1], false, false);
            const uint32_t largest_of = row_largest(max(c[0], c[1]));
            const int u = 2 * j + ((lane >> 4) & 1), group = (begin - lane + u * 64 + (lane & 32)) >> 5;
            if ((lane & 15) == 0 && group < groups) to[group] = largest_of;
        }
        return;
    }
    uint32_t run = 0u;
#pragma unroll
    for (int u = 0; u < 16; u++) {
        if (shift > 3) m[u] = row_largest(m[u]);
        else {
            if (shift > 0) m[u] = max(m[u], across<1>(m[u], lane));
            if (shift > 1) m[u] = max(m[u], across<2>(m[u], lane));
            if (shift > 2) m[u] = max(m[u], across<4>(m[u], lane));
        }
        if (shift > 5) m[u] = max(m[u], across<16>(m[u], lane));
        if (shift > 5) m[u] = max(m[u], across<32>(m[u], lane));
        run = (u & whole) == 0 ? m[u] : max(run, m[u]);
        const int group = (begin + u * 64) >> shift;
        if ((u & whole) == whole && (shift > 5 ? lane == 0 : (lane & ((1 << shift) - 1)) == 0) && group < groups) to[group] = run;
    }
}

// One block per row.  largest (or null): the keys of the row's groups; the sampler then works on the candidates they lead to, else,
// or where those are more than its list holds, on the whole row.
template <int AT_MOST>                                               // groups
__global__ void __launch_bounds__(1024)
sample_k(const float* __restrict__ logits, int V, float temperature, int top_k, float top_p, Draws draws, int* __restrict__ out,
         const uint32_t* __restrict__ largest, int groups, int shift) {
    __shared__ unsigned hist[256];
    constexpr int STAGE = 16384;                               // logits on their way into LDS at once; later the sort, keys, ids, weights
    __shared__ __attribute__((aligned(16))) float stage[STAGE];
    unsigned long long* const place = reinterpret_cast<unsigned long long*>(stage);
    uint32_t* const ckey = reinterpret_cast<uint32_t*>(stage + 4096);
    int* const cid = reinterpret_cast<int*>(stage + 5120);
    float* const prob = stage + 6144;
    __shared__ unsigned s_prefix, s_remaining, s_count, s_eq_total;
    __shared__ int s_id_limit;
    __shared__ __attribute__((aligned(16))) uint32_t list_val[LIST];      // (float bits; first the counters of the groups' keys)
    __shared__ int list_id[LIST];
    __shared__ unsigned short chosen[AT_MOST];
    __shared__ __attribute__((aligned(16))) unsigned s_wave[16];
    __shared__ unsigned s_above, s_inside, s_bucket, s_many;
    const float* const z = logits + (size_t)blockIdx.x * V;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int k = top_k < V ? top_k : V;                       // of the whole row, whichever source is read
    bool ids = false;                                          // the candidates are the list (else the row)
    constexpr int IN_ORDER = 2048;                             // candidates that are put in order as they are
    int sorted = 1024;
    if (largest) {
        constexpr int PER = AT_MOST / 1024;
        uint32_t key[PER];
#pragma unroll
        for (int j = 0; j < PER; j++) key[j] = largest[(size_t)blockIdx.x * groups + min(j * 1024 + tid, groups - 1)];
        // the k-th largest key of the groups: its top 12 bits, and 12 and 8 more while the groups from there up are many more than k
        uint32_t from = 0u;                                    // keys from here up lead to candidates
        unsigned need = (unsigned)k, counted = 0u;             // of the keys that share `from` above the level; groups beyond them
        for (int level = 20; level >= 0; level = level == 20 ? 8 : level - 8) {
            const int width = level == 0 ? 256 : 4096;
            for (int i = tid; i < width; i += 1024) list_val[i] = 0u;
            lds_barrier();
#pragma unroll
            for (int j = 0; j < PER; j++)
                if (j * 1024 + tid < groups && (level == 20 || (level == 8 ? key[j] >> 20 == from >> 20 : key[j] >> 8 == from >> 8)))
                    atomicAdd(&list_val[(key[j] >> level) & (unsigned)(width - 1)], 1u);
            lds_barrier();
            // four counters a thread, from the top
            const int top = width - 1 - tid * 4;
            const uint4 four = *reinterpret_cast<const uint4*>(list_val + max(top - 3, 0));
            const unsigned c[4] = {top >= 0 ? four.w : 0u, top >= 0 ? four.z : 0u, top >= 0 ? four.y : 0u, top >= 0 ? four.x : 0u};
            const unsigned mine = c[0] + c[1] + c[2] + c[3];
            const unsigned incl = wave_scan_incl(mine, lane);
            if (lane == 63) s_wave[wave] = incl;
            if (tid == 0) { s_bucket = 0u; s_above = 0u; s_inside = 0u; }
            lds_barrier();
            unsigned above = incl - mine;
#pragma unroll
            for (int w = 0; w < 15; w++) above += w < wave ? s_wave[w] : 0u;
            if (above < need && above + mine >= need) {        // exactly one thread
                int j = 0;
                for (; j < 3; j++) {
                    if (above + c[j] >= need) break;
                    above += c[j];
                }
                s_bucket = (unsigned)(top - j);
                s_above = above;
                s_inside = c[j];
            }
            lds_barrier();
            from |= s_bucket << level;
            counted += s_above;
            need -= s_above;
            if (counted + s_inside <= (unsigned)k + 64u) break;
            lds_barrier();                                     // (the counters are cleared for the next level)
        }
        // these groups, as pieces of at most 64 logits, and their logits from there up
        if (tid == 0) { s_count = 0u; s_many = 0u; }
        lds_barrier();
        const int parts = shift > 6 ? 1 << (shift - 6) : 1;
#pragma unroll
        for (int j = 0; j < PER; j++)
            if (j * 1024 + tid < groups && key[j] >= from) {
                const unsigned to = atomicAdd(&s_many, (unsigned)parts);
                for (int i = 0; i < parts; i++)
                    if (to + i < (unsigned)AT_MOST) chosen[to + i] = (unsigned short)((j * 1024 + tid) * parts + i);
            }
        lds_barrier();
        // The pieces come straight into LDS, 64 logits an instruction, all of up to 256 such on their way at once; then every thread
        // looks at sixteen of them.  (Code that runs once waits for its instructions: with the loads in registers, unrolled eight or
        // sixteen times, this part took two and a half times as long; 128 at a time, the next on their way, 1.4 times.)
        const int many = (int)s_many, piece = min(shift, 6), per = 64 >> piece, units = many <= AT_MOST ? (many + per - 1) / per : 0;
        const float least = from ? key_value(from) : -INFINITY;       // (NaN is not below it, and sinks)
        const unsigned stage0 = (unsigned)(size_t)(__attribute__((address_space(3))) void*)stage, last = (unsigned)(V - 1) * 4u;
        const unsigned within = (unsigned)(lane & ((1 << piece) - 1)) * 4u;
        if (units > 0 && tid < 64 && many + tid < AT_MOST) chosen[many + tid] = 0;      // what stands past the last piece in its load
        lds_barrier();
        for (int u0 = 0; u0 < units; u0 += STAGE / 64) {
            const int here = min(units - u0, STAGE / 64);
            int p = (u0 + wave) * per + (lane >> piece);
#pragma unroll 4
            for (int u = wave; u < here; u += 16, p += 16 * per) {
                const unsigned off = min(((unsigned)chosen[p & (AT_MOST - 1)] << (piece + 2)) + within, last);
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" :: "v"(off), "s"(z), "s"(stage0 + (unsigned)u * 256u) : "memory");
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0x0f70);
            lds_barrier();
            unsigned found = 0u;
#pragma unroll
            for (int j = 0; j < STAGE / 4096; j++) {
                const int e = (j * 1024 + tid) * 4;
                const float4 four = *reinterpret_cast<const float4*>(stage + e);
                if (e < here * 64)
                    found |= (!(four.x < least) ? 1u : 0u) << (4 * j) | (!(four.y < least) ? 2u : 0u) << (4 * j) | (!(four.z < least) ? 4u : 0u) << (4 * j) | (!(four.w < least) ? 8u : 0u) << (4 * j);
            }
            const unsigned own = (unsigned)__popc(found), incl = wave_scan_incl(own, lane);
            unsigned to = 0u;
            if (lane == 63) to = atomicAdd(&s_count, incl);            // one addition for all that a wave found
            to = (unsigned)__builtin_amdgcn_readlane((int)to, 63) + incl - own;
            for (; found; found &= found - 1u, to++) {
                const int bit = __ffs(found) - 1, e = ((bit >> 2) * 1024 + tid) * 4 + (bit & 3), p = (u0 + (e >> 6)) * per + ((e & 63) >> piece);
                const int id = ((int)chosen[min(p, many - 1)] << piece) + (e & ((1 << piece) - 1));
                const bool real = p < many && id < V;                  // (what stands past a row's or the last piece's end sinks)
                if (to < (unsigned)LIST) { list_val[to] = real ? __float_as_uint(stage[e]) : 0x7fffffffu; list_id[to] = real ? id : 0x7fffffff; }
            }
            lds_barrier();                                             // everyone has looked at them
        }
        if (many <= AT_MOST && s_count <= (unsigned)LIST) {     // (at least k: every group counted gave one)
            V = (int)s_count;
            ids = true;
        }
    }
    unsigned long long mine = packed(0u, 0x7fffffff);          // this thread's candidate; empty places sink
    const bool few = ids && V <= IN_ORDER;
    if (few) {
        if (tid < V) mine = packed(value_key(__uint_as_float(list_val[tid])), list_id[tid]);
        sorted = 64;
        while (sorted < V && sorted < 1024) sorted <<= 1;
    } else {

    auto at = [&](int i) { return ids ? __uint_as_float(list_val[i]) : z[i]; };
    // 1. the k-th largest value key, 8 bits at a time from the top
    if (tid == 0) { s_prefix = 0u; s_remaining = (unsigned)k; }
    for (int shift = 24; shift >= 0; shift -= 8) {
        if (tid < 256) hist[tid] = 0u;
        __syncthreads();
        const unsigned prefix = s_prefix;
        for (int i = tid; i < V; i += blockDim.x) {
            const uint32_t key = value_key(at(i));
            if (shift == 24 || (key >> (shift + 8)) == (prefix >> (shift + 8))) atomicAdd(&hist[(key >> shift) & 255u], 1u);
        }
        __syncthreads();
        if (tid < 64) {
            int b;
            unsigned rem;
            pick_bucket(hist, true, s_remaining, tid, b, rem);
            if (tid == 0) {
                s_prefix = prefix | ((unsigned)b << shift);
                s_remaining = rem;                   // how many of this bucket are still needed
                if (shift == 0) s_eq_total = hist[b];
            }
        }
        __syncthreads();
    }
    const uint32_t tkey = s_prefix;                  // value key of the k-th largest
    const unsigned need_eq = s_remaining;            // candidates to take among those equal to it
    // 2. ties at the threshold: the need_eq smallest ids among the equal ones
    if (tid == 0) s_id_limit = 0x7fffffff;
    __syncthreads();
    if (s_eq_total > need_eq) {
        if (tid == 0) { s_prefix = 0u; s_remaining = need_eq; }
        for (int shift = 24; shift >= 0; shift -= 8) {
            if (tid < 256) hist[tid] = 0u;
            __syncthreads();
            const unsigned prefix = s_prefix;
            for (int i = tid; i < V; i += blockDim.x) {
                if (value_key(at(i)) != tkey) continue;
                const unsigned id = (unsigned)(ids ? list_id[i] : i);
                if (shift == 24 || (id >> (shift + 8)) == (prefix >> (shift + 8))) atomicAdd(&hist[(id >> shift) & 255u], 1u);
            }
            __syncthreads();
            if (tid < 64) {
                int b;
                unsigned rem;
                pick_bucket(hist, false, s_remaining, tid, b, rem);
                if (tid == 0) {
                    s_prefix = prefix | ((unsigned)b << shift);
                    s_remaining = rem;
                }
            }
            __syncthreads();
        }
        if (tid == 0) s_id_limit = (int)s_prefix;    // the need_eq-th smallest id among the equal ones
        __syncthreads();
    }
    // 3. collect the k candidates
    if (tid == 0) s_count = 0u;
    ckey[tid] = 0u;
    cid[tid] = 0x7fffffff;
    __syncthreads();
    const int id_limit = s_id_limit;
    for (int i = tid; i < V; i += blockDim.x) {
        const uint32_t key = value_key(at(i));
        const int id = ids ? list_id[i] : i;
        if (key > tkey || (key == tkey && id <= id_limit)) {
            const unsigned at = atomicAdd(&s_count, 1u);
            if (at < 1024u) { ckey[at] = key; cid[at] = id; }
        }
    }
    __syncthreads();
    mine = packed(ckey[tid], cid[tid]);
    }
    // 4. in order; the first k are the candidates.  Of more than 1,024 the rest is put in order by itself, and of the two runs the
    // larger of first and last, second and last but one, ... are the 1,024 largest, a sequence that the last stage puts in order.
    block_sort(mine, sorted, place);
    if (few && V > 1024) {
        unsigned long long rest = packed(0u, 0x7fffffff);
        if (1024 + tid < V) rest = packed(value_key(__uint_as_float(list_val[1024 + tid])), list_id[1024 + tid]);
        int behind = 64;
        while (1024 + behind < V) behind <<= 1;
        block_sort(rest, behind, place);
        lds_barrier();
        place[1023 - tid] = rest;
        lds_barrier();
        rest = place[tid];
        if (rest > mine) mine = rest;
        sort_stages(mine, 1024, 1024, place);
    }
    lds_barrier();
    ckey[tid] = (uint32_t)(mine >> 32);
    cid[tid] = (int)~(uint32_t)mine;
    lds_barrier();
    // 5. probabilities, the nucleus and the draw: the first wave, each lane 16 consecutive candidates; sums run over a
    // lane's candidates in order, then over the lanes in order
    const float mx = key_value(ckey[0]);
    prob[tid] = tid < k ? expf((key_value((uint32_t)(mine >> 32)) - mx) / temperature) : 0.f;
    lds_barrier();
    if (tid < 64) {
        const int j0 = tid * 16;
        float p[16], c[16];
#pragma unroll
        for (int j = 0; j < 16; j += 4) *reinterpret_cast<float4*>(p + j) = *reinterpret_cast<const float4*>(prob + j0 + j);
        float local = 0.f;
#pragma unroll
        for (int j = 0; j < 16; j++) local += p[j];            // (zero beyond the k candidates)
        const float total = __shfl(wave_scan_incl(local, tid), 63, 64);
        float lsum = 0.f;
#pragma unroll
        for (int j = 0; j < 16; j++) { p[j] /= total; lsum += p[j]; }
        float run = wave_scan_incl(lsum, tid) - lsum;
#pragma unroll
        for (int j = 0; j < 16; j++) { run += p[j]; c[j] = run; }         // cumulative probabilities
        // the shortest prefix whose mass reaches top_p
        int first = k;
#pragma unroll
        for (int j = 15; j >= 0; j--)
            if (j0 + j < k && c[j] >= top_p) first = j0 + j;
        first = wave_least(first, tid);
        const int keep = first < k ? first + 1 : k;
        float last = 0.f;                                      // c of candidate keep - 1, in the lane that holds it
#pragma unroll
        for (int j = 0; j < 16; j++)
            if (j0 + j == keep - 1) last = c[j];
        const float kept = __shfl(last, (keep - 1) >> 4, 64);
        const float r = draw_of(draws, blockIdx.x) * kept;
        // the walk: the first candidate whose cumulative mass exceeds r; none (rounding at the end): the first candidate
        int hit = keep;
#pragma unroll
        for (int j = 15; j >= 0; j--)
            if (j0 + j < keep && r < c[j]) hit = j0 + j;
        hit = wave_least(hit, tid);
        if (tid == 0) out[blockIdx.x] = cid[hit < keep ? hit : 0];
    }
}

// ---- temperature sampling over the whole vocabulary (top_k 0, no nucleus; the reference always keeps 256): p_i =
// exp((z_i - max) / T), r = u * sum, the token whose cumulative mass in id order first exceeds r.  One block per
// row; thread t owns a contiguous range of ids, so sums run over ids in order within a thread, then over the threads
// in order. ----------------------------------------------------------------------------------------------------
// part: the sums of 1,024 threads' stretches -> what lies before each; returns the total
__device__ __forceinline__ float full_scan(float* part, float& total, int tid) {
    __syncthreads();
    if (tid < 64) {                                  // the first wave: totals of 16 threads per lane, then over the lanes
        float local = 0.f;
        for (int j = 0; j < 16; j++) local += part[tid * 16 + j];
        const float incl = wave_scan_incl(local, tid);
        float run = incl - local;
        for (int j = 0; j < 16; j++) { const float v = part[tid * 16 + j]; part[tid * 16 + j] = run; run += v; }   // exclusive sums
        if (tid == 63) total = incl;
    }
    __syncthreads();
    return total;
}

__global__ void __launch_bounds__(1024)
sample_full_k(const float* __restrict__ logits, int V, float temperature, Draws draws,
              int* __restrict__ out) {
    __shared__ float part[1024];
    __shared__ float s_total;
    __shared__ int s_winner;
    const float* z = logits + (size_t)blockIdx.x * V;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float mx = -INFINITY;
    for (int i = tid; i < V; i += 1024) { const float v = z[i]; mx = v > mx ? v : mx; }      // NaN never wins
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    if (lane == 0) part[wave] = mx;
    __syncthreads();
    mx = part[0];
    for (int w = 1; w < 16; w++) mx = fmaxf(mx, part[w]);
    __syncthreads();
    const int chunk = (V + 1023) / 1024, begin = tid * chunk, end = min(V, begin + chunk);
    float mine = 0.f;
    for (int i = begin; i < end; i++) { const float v = z[i]; mine += v == v ? expf((v - mx) / temperature) : 0.f; }
    part[tid] = mine;
    full_scan(part, s_total, tid);
    const float r = draw_of(draws, blockIdx.x) * s_total;
    const float before = part[tid];
    // the first thread whose range reaches past r walks it; rounding may leave r past every range: the last one
    if (tid == 0) s_winner = (V - 1) / chunk;
    __syncthreads();
    if (begin < end && r < before + mine) atomicMin(&s_winner, tid);
    __syncthreads();
    if (tid == s_winner) {
        float run = before;
        int pick = end - 1;
        for (int i = begin; i < end; i++) {
            const float v = z[i];
            run += v == v ? expf((v - mx) / temperature) : 0.f;
            if (r < run) { pick = i; break; }
        }
        out[blockIdx.x] = pick;
    }
}

// ---- the same on many blocks, to the same bits: a thread's stretch of ids above is a chunk here.  One launch leaves the groups'
// largest keys (above), one the chunks' sums (a block forms the exponentials of its chunks together, then a thread adds a chunk's in order),
// one finds the chunk and walks it.  Microseconds, 1 / 8 / 64 rows of 256,000: one block a row 156 / 179 / 337, here 20 / 26 / 52.
constexpr int FULL_CHUNKS = 1024;
constexpr int FULL_LDS = 16000;                                      // floats of LDS that a block's chunks take at most

template <int THREADS>
__device__ __forceinline__ float row_max(const uint32_t* __restrict__ largest, int groups, uint32_t* red) {
    uint32_t key[GROUPS / THREADS], m = 0u;
#pragma unroll
    for (int j = 0; j < GROUPS / THREADS; j++) key[j] = largest[min(j * THREADS + (int)threadIdx.x, groups - 1)];
#pragma unroll
    for (int j = 0; j < GROUPS / THREADS; j++) m = max(m, key[j]);
    const int lane = threadIdx.x & 63;
    m = max(m, across<32>(m, lane)); m = max(m, across<16>(m, lane)); m = max(m, across<8>(m, lane));
    m = max(m, across<4>(m, lane)); m = max(m, across<2>(m, lane)); m = max(m, across<1>(m, lane));
    if (lane == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = red[0];
#pragma unroll
    for (int w = 1; w < THREADS / 64; w++) m = max(m, red[w]);
    return m == 0u ? -INFINITY : key_value(m);                       // (NaN alone: as if there were nothing)
}

__global__ void __launch_bounds__(256)
full_sums_k(const float* __restrict__ logits, int V, float temperature, const uint32_t* __restrict__ largest, int groups, int chunk, int chunks,
            float* __restrict__ sums) {
    extern __shared__ float e[];
    __shared__ uint32_t red[4];
    const int tid = threadIdx.x, first = blockIdx.x * chunks, stride = chunk | 1;
    const float* z = logits + (size_t)blockIdx.y * V;
    const float mx = row_max<256>(largest + (size_t)blockIdx.y * groups, groups, red);
    const int begin = first * chunk, n = min(V - begin, chunks * chunk);           // (the last chunks may hold nothing)
    // sixteen lanes a chunk, eight logits of a lane at once
    const int mine = tid >> 4, own = min(chunk, n - mine * chunk);
    if (mine < chunks)
        for (int i0 = tid & 15; i0 < own; i0 += 128) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = z[begin + mine * chunk + min(i0 + 16 * j, own - 1)];
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (i0 + 16 * j < own) e[mine * stride + i0 + 16 * j] = v[j] == v[j] ? expf((v[j] - mx) / temperature) : 0.f;
        }
    __syncthreads();
    for (int c = tid; c < chunks && first + c < FULL_CHUNKS; c += 256) {
        const int len = max(0, min(chunk, n - c * chunk));
        float sum = 0.f;
#pragma unroll 8
        for (int i = 0; i < len; i++) sum += e[c * stride + i];
        sums[(size_t)blockIdx.y * FULL_CHUNKS + first + c] = sum;
    }
}

__global__ void __launch_bounds__(1024)
full_pick_k(const float* __restrict__ logits, int V, float temperature, const uint32_t* __restrict__ largest, int groups, int chunk,
            const float* __restrict__ sums, Draws draws, int* __restrict__ out) {
    __shared__ float part[FULL_CHUNKS], e[FULL_LDS];
    __shared__ uint32_t red[16];
    __shared__ float s_total;
    __shared__ int s_winner;
    const int tid = threadIdx.x;
    const float* z = logits + (size_t)blockIdx.x * V;
    const float mine = sums[(size_t)blockIdx.x * FULL_CHUNKS + tid];
    part[tid] = mine;
    const float mx = row_max<1024>(largest + (size_t)blockIdx.x * groups, groups, red);
    const float total = full_scan(part, s_total, tid);
    const float r = draw_of(draws, blockIdx.x) * total, before = part[tid];
    const int begin = tid * chunk, end = min(V, begin + chunk);
    if (tid == 0) s_winner = (V - 1) / chunk;
    __syncthreads();
    if (begin < end && r < before + mine) atomicMin(&s_winner, tid);
    __syncthreads();
    const int winner = s_winner, from = winner * chunk, n = min(V, from + chunk) - from;
    for (int i = tid; i < n; i += 1024) {
        const float v = z[from + i];
        e[i] = v == v ? expf((v - mx) / temperature) : 0.f;
    }
    __syncthreads();
    if (tid == 0) {
        float run = part[winner];
        int pick = n - 1;
        bool found = false;
        for (int i0 = 0; i0 < n && !found; i0 += 8) {            // eight at a time out of LDS; past the last they add nothing that counts
            float t[8];
#pragma unroll
            for (int j = 0; j < 8; j++) t[j] = e[min(i0 + j, n - 1)];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                run += t[j];
                if (!found && i0 + j < n && r < run) { pick = i0 + j; found = true; }
            }
        }
        out[blockIdx.x] = from + pick;
    }
}

static int full_chunk(int V) { return (V + FULL_CHUNKS - 1) / FULL_CHUNKS; }
// (1 row: 16,384 15.5 us by one block, 16.9 here; 32,000 25.8 / 17.8)
constexpr int FULL_FROM = 20480;
static bool full_on_many_blocks(int V) { return V >= FULL_FROM && full_chunk(V) < FULL_LDS; }

// bytes of the sampler's workspace for B rows (nothing has to lie in it)
extern "C" long tp_sample_workspace_bytes(int B, int V) {
    if (V < GROUPS_FROM) return 0;
    const long many = groups_of(V, group_shift(V, GROUPS_MANY)), full = groups_of(V, group_shift(V, GROUPS)) + (full_on_many_blocks(V) ? FULL_CHUNKS : 0);
    return (long)B * (many > full ? many : full) * 4;
}

static int sample_launch(const float* logits, int B, int V, float temperature, int top_k, float top_p, const Draws& draws, int* out,
                         void* workspace, void* stream) {
    TP_REQUIRE(B > 0 && V > 0, "sample: empty shape B=%d V=%d", B, V);
    TP_REQUIRE(temperature > 0.f, "sample: temperature %g must be positive (0 means argmax)", temperature);
    TP_REQUIRE(top_k >= 0 && top_k <= 1024, "sample: top_k %d must lie in 0..1024 (0: the whole vocabulary)", top_k);
    TP_REQUIRE(top_p > 0.f, "sample: top_p %g must be positive", top_p);
    TP_REQUIRE(top_k > 0 || top_p >= 1.f, "sample: a nucleus (top_p %g) needs top_k between 1 and 1024", top_p);
    TP_REQUIRE(B <= 65535, "sample: %d rows exceed one launch", B);
    hipStream_t s = (hipStream_t)stream;
    const bool many = top_k > MANY;
    const int shift = group_shift(V, many ? GROUPS_MANY : GROUPS), groups = groups_of(V, shift);
    const bool in_groups = workspace && V >= GROUPS_FROM && shift <= 10 && (top_k > 0 || full_on_many_blocks(V));
    uint32_t* const largest = in_groups ? (uint32_t*)workspace : nullptr;
    if (in_groups) {
        group_max_k<<<dim3(tp_cdiv(V, GROUP_PART), B), 256, 0, s>>>(logits, V, shift, groups, largest);
        if (int rc = tp_check_launch("sample (groups)")) return rc;
    }
    if (top_k > 0) {
        if (many) sample_k<GROUPS_MANY><<<B, 1024, 0, s>>>(logits, V, temperature, top_k, top_p, draws, out, largest, groups, shift);
        else sample_k<GROUPS><<<B, 1024, 0, s>>>(logits, V, temperature, top_k, top_p, draws, out, largest, groups, shift);
        return tp_check_launch("sample");
    }
    if (!in_groups) {
        sample_full_k<<<B, 1024, 0, s>>>(logits, V, temperature, draws, out);
        return tp_check_launch("sample (whole vocabulary)");
    }
    float* const sums = (float*)(largest + (size_t)B * groups);
    const int chunk = full_chunk(V);
    int chunks = FULL_LDS / (chunk | 1);                             // of a block
    if (chunks > 16) chunks = 16;
    full_sums_k<<<dim3(tp_cdiv(FULL_CHUNKS, chunks), B), 256, (size_t)chunks * (chunk | 1) * 4, s>>>(logits, V, temperature, largest, groups, chunk, chunks, sums);
    if (int rc = tp_check_launch("sample (sums)")) return rc;
    full_pick_k<<<B, 1024, 0, s>>>(logits, V, temperature, largest, groups, chunk, sums, draws, out);
    return tp_check_launch("sample (whole vocabulary)");
}

// uniforms: a float32 number per row, on the device
extern "C" int tp_sample(const float* logits, int B, int V, float temperature, int top_k, float top_p,
                         const float* uniforms, int* out, void* workspace, void* stream) {
    TP_REQUIRE(uniforms, "sample: no uniform numbers");
    Draws draws{};
    draws.at = uniforms;
    return sample_launch(logits, B, V, temperature, top_k, top_p, draws, out, workspace, stream);
}

// the same with the numbers in host memory, read before the call returns
extern "C" int tp_sample_host_uniforms(const float* logits, int B, int V, float temperature, int top_k, float top_p,
                                       const float* uniforms, int* out, void* workspace, void* stream) {
    TP_REQUIRE(uniforms && B <= TP_HOST_UNIFORMS, "sample: uniform numbers for %d rows (at most %d come from the host)", B, TP_HOST_UNIFORMS);
    Draws draws{};
    for (int i = 0; i < B; i++) draws.v[i] = uniforms[i];
    return sample_launch(logits, B, V, temperature, top_k, top_p, draws, out, workspace, stream);
}
