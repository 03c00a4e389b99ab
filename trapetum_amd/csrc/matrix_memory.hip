// The matrix memory of a head with exponential gates:
//   m' = max(f + m, i);  S <- e^(f + m - m') S + e^(i - m') k v^T, n likewise with k;
//   o = S^T q / (max(|n . q|, e^(-m')) + 1e-6), i and f capped by a tanh.
// S [dk, dv], n [dk] and m of a (sequence, head) are states, float32 like gates and sums.
//
// Three ways to the same rows:
// * a step of one row a sequence: matrix_memory_step_k;
// * up to 11 rows of the longest sequence: matrix_memory_scan_k, row after row, a lane keeping rows of one column of S in registers;
// * more: chunks of up to 64 rows side by side, as products on the float32 matrix instructions (float32 operands and sums; the
//   queries, keys and values are exact in them).  With b_t the sum of the log forget gates of a chunk's rows up to t, a_s = i_s - b_s
//   and m0 the maximum that the chunk starts from, M_t = max(m0, a_0 .. a_t) gives m_t = b_t + M_t, and
//     o_t = (e^(m0 - M_t) S0^T q_t + sum over s <= t of e^(a_s - M_t) (k_s . q_t) v_s) / den,
//   the normalizer's product likewise without v.  a and M are sums of up to 64 terms whose differences are what counts: they are
//   formed in float64.  First what every chunk adds to the state (mm_chunk_k, from nothing), then a walk over the chunks that
//   leaves each one's first state and the sequence's last (mm_carry_k), then the outputs (mm_outputs_k).  Row after row, which also in
//   chunks is a chain of a few hundred multiply-adds and reads a row, took 690 us for prompts of 700, 333, 64 and 1,025 rows, nine
//   heads, keys of 128 and values of 256; 125 so (43 + 24 + 58).  The two meet at about 12 rows a sequence (4 sequences of 8 rows
//   31 us row by row, 34 in chunks; of 16 48 and 35; one of 64 149 and 53).
// Error against 64 bits in chunks over that row after row, geometric means over twenty prompts of 12 to 699 rows and gates of three
// spreads: outputs 0.94 (the median row's 0.81), matrix 0.98, normalizer 0.97; outputs 1.3e-7 to 1.1e-6 (the denominator is a small
// difference now and then), states 3.5e-8 to 2.8e-7.
#include "recurrent.h"

struct MatrixMemoryArgs {
    const void* q; long q_stride; const void* k; long k_stride; const void* v; long v_stride;
    const float* gates; float cap, q_scale; float* memory; float* normalizer; float* maximum;
    const int* slot_ids; const int* cu_rows; float* y; int n_seq, H, dk, dv;
    // chunks of `chunk` rows, each in a place of its own (chunk_at).  ws_state [places, H, dk dv + dk]: a chunk's matrix,
    // then its normalizer, both in units of e^(its maximum); ws_aux [places, H, 8]: the maximum of a chunk run from
    // nothing, the sum of its log forget gates, the maximum it starts from, the maximum it leaves, what the sum was rounded by, and as
    // whole numbers its sequence, first row and rows (0: no chunk).  ws_first [n_seq]: a sequence's first place
    int chunk, places; float* ws_state; float* ws_aux; int* ws_first;
};

__device__ __forceinline__ float log_sigmoid_f(float z) { return -(log1pf(expf(-fabsf(z))) + fmaxf(-z, 0.f)); }

// ---- one row a sequence --------------------------------------------------------------------------------------------------------
// A block for each (sequence, head).  What bounds it is one CU's trip to memory for dk dv floats and their way back: 131 KB at keys of
// 128 and values of 256.  (The kernel of whole sequences, which reads columns in four waves' parts and prepares for rows that do
// not come, took 29.4 us for 4 sequences of 9 heads; 8.0 here.)  R: rows of S a thread holds.
template <typename T, int R>
__global__ void __launch_bounds__(1024)
matrix_memory_step_k(MatrixMemoryArgs a) {
    __shared__ __attribute__((aligned(16))) float parts[16][256];
    __shared__ float sq[256], sk[256], dots[4];
    const int seq = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, dk = a.dk, dv = a.dv, H = a.H;
    const int t = a.cu_rows[seq];
    if (a.cu_rows[seq + 1] <= t) return;
    const size_t slot = (size_t)a.slot_ids[seq];
    const int Q = dv >> 2, c4 = tid & (Q - 1), first = tid / Q, RG = blockDim.x / Q;
    float* const st = a.memory + (slot * H + h) * dk * dv + 4 * c4;
    float4 S[R];
#pragma unroll
    for (int i = 0; i < R; i++) S[i] = *reinterpret_cast<const float4*>(st + (size_t)min(first + RG * i, dk - 1) * dv);
    float* const sn = a.normalizer + (slot * H + h) * dk;
    const int row = min(tid, dk - 1);
    const float q = ld_f32((const T*)a.q + (size_t)t * a.q_stride + (size_t)h * dk + row) * a.q_scale;
    const float k = ld_f32((const T*)a.k + (size_t)t * a.k_stride + (size_t)h * dk + row);
    const float n = sn[row], m = a.maximum[slot * H + h];
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = ld_f32((const T*)a.v + (size_t)t * a.v_stride + (size_t)h * dv + 4 * c4 + e);
    const float gi = a.gates[(size_t)t * 2 * H + h], gf = a.gates[(size_t)t * 2 * H + H + h];
    const float li = a.cap * tanhf(gi / a.cap), lf = log_sigmoid_f(a.cap * tanhf(gf / a.cap));
    const float m_new = fmaxf(lf + m, li), keep = expf(lf + m - m_new), take = expf(li - m_new);
    if (wave < 4) {
        const float n_new = __builtin_fmaf(keep, n, take * k), dot = wave_sum(tid < dk ? n_new * q : 0.f);
        if (tid < dk) { sq[tid] = q; sk[tid] = k; sn[tid] = n_new; }
        if (lane == 0) dots[wave] = dot;
    }
    lds_barrier();
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] *= take;
#pragma unroll
    for (int i = 0; i < R; i++) {
        const int r = first + RG * i;
        if (r < dk) {
            const float kr = sk[r], qr = sq[r];
            S[i].x = __builtin_fmaf(keep, S[i].x, kr * v[0]);
            S[i].y = __builtin_fmaf(keep, S[i].y, kr * v[1]);
            S[i].z = __builtin_fmaf(keep, S[i].z, kr * v[2]);
            S[i].w = __builtin_fmaf(keep, S[i].w, kr * v[3]);
            o.x = __builtin_fmaf(qr, S[i].x, o.x);
            o.y = __builtin_fmaf(qr, S[i].y, o.y);
            o.z = __builtin_fmaf(qr, S[i].z, o.z);
            o.w = __builtin_fmaf(qr, S[i].w, o.w);
            *reinterpret_cast<float4*>(st + (size_t)r * dv) = S[i];
        }
    }
    step_parts(o, Q, lane, &parts[wave][4 * c4]);
    lds_barrier();                                       // everyone has worked with m, too
    if (tid == 0) a.maximum[slot * H + h] = m_new;
    if (tid < dv) {
        float sum = 0.f, dot = 0.f;
        for (int w = 0; w < (int)blockDim.x >> 6; w++) sum += parts[w][tid];
#pragma unroll
        for (int w = 0; w < 4; w++) dot += dots[w];
        a.y[((size_t)t * H + h) * dv + tid] = sum / (fmaxf(fabsf(dot), expf(-m_new)) + 1e-6f);
    }
}

// ---- row after row ---------------------------------------------------------------------------------------------------------------
// One block for a (sequence, head), a group of waves for every 64 value columns: every wave carries n and m along (they are the
// same in all), reads them before any wave writes them back, and the first wave stores them at the end.
// The matrix memory's split: a block holds up to four groups of 64 value columns, each in MM_SPLIT waves
#define TP_MM_SPLIT(DK) ((DK) >= 256 ? 2 : (DK) >= 64 ? 4 : 1)

template <typename T, int DK>
__global__ void __launch_bounds__(256 * TP_MM_SPLIT(DK))
matrix_memory_scan_k(MatrixMemoryArgs a) {
    constexpr int NR = (DK + 63) / 64, RS = TP_MM_SPLIT(DK), AH = RS > 1 ? 2 : TP_SCAN_AHEAD, DKW = DK / RS;
    const int h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, group = wave / RS, part = wave % RS;
    const int j = group * 64 + lane, row0 = part * DKW;
    const int seq = blockIdx.x;
    const int dk = a.dk, dv = a.dv, H = a.H;
    const bool col = j < dv;
    const int begin = a.cu_rows[seq], end = a.cu_rows[seq + 1];
    if (begin >= end) return;                               // no rows: what `fetch` would read past the end may lie before the first row
    const size_t slot = (size_t)a.slot_ids[seq];
    float* st = a.memory + (slot * H + h) * dk * dv;
    float* sn = a.normalizer + (slot * H + h) * dk;
    float S[DKW], nn[NR];                               // rows row0 .. row0 + DKW - 1 of column j; all of n, a row a lane
#pragma unroll
    for (int i = 0; i < DKW; i++) {                     // every lane reads an element that exists; what is none of S becomes zero
        const float x = st[min(row0 + i, dk - 1) * dv + min(j, dv - 1)];
        S[i] = (col && row0 + i < dk) ? x : 0.f;
    }
    load_rows<float, NR>(nn, sn, dk, lane, 1.f);
    float m = a.maximum[slot * H + h];
    __syncthreads();
    // lane p of a group of tokens forms token p's two gates; the others read them from it
    // the block's first wave forms q and k of the tokens in flight for all its waves, carries n and forms the denominators
    const bool stager = wave == 0;
    float qq[AH][NR] = {}, kk[AH][NR] = {}, vv[AH], gi, gf;
    auto fetch = [&](int t0, float (&Q)[AH][NR], float (&K)[AH][NR], float (&V)[AH], float& I, float& F) {
#pragma unroll
        for (int p = 0; p < AH; p++) {
            const int t = min(t0 + p, end - 1);
            if (stager) {
                load_rows<T, NR>(Q[p], (const T*)a.q + (size_t)t * a.q_stride + (size_t)h * dk, dk, lane, a.q_scale);
                load_rows<T, NR>(K[p], (const T*)a.k + (size_t)t * a.k_stride + (size_t)h * dk, dk, lane, 1.f);
            }
            V[p] = col ? ld_f32((const T*)a.v + (size_t)t * a.v_stride + (size_t)h * dv + j) : 0.f;
        }
        const int t = min(t0 + min(lane, AH - 1), end - 1);
        I = a.gates[(size_t)t * 2 * H + h];
        F = a.gates[(size_t)t * 2 * H + H + h];
    };
    // q and k of the tokens in flight, written a row a lane by the first wave and read back by every lane; for rounds in turn
    __shared__ __attribute__((aligned(16))) float stage_all[2][AH][2][DK];
    __shared__ float dens_all[2][AH];
    __shared__ float parts[2][4 * RS][AH][64];           // the waves' parts of the outputs, for rounds in turn
    int round = 0;
    fetch(begin, qq, kk, vv, gi, gf);
    for (int t0 = begin; t0 < end; t0 += AH, round ^= 1) {
        float (*stage)[2][DK] = stage_all[round];
        float qn[AH][NR] = {}, kn[AH][NR] = {}, vn[AH], gin, gfn;
        fetch(t0 + AH, qn, kn, vn, gin, gfn);
        const float li = a.cap * tanhf(gi / a.cap), lf = log_sigmoid_f(a.cap * tanhf(gf / a.cap));
        // what the gates make of m, token after token: every wave for itself
        float keeps[AH], takes[AH], floors[AH];
#pragma unroll
        for (int p = 0; p < AH; p++) {
            keeps[p] = 1.f; takes[p] = 0.f; floors[p] = 1.f;
            if (t0 + p < end) {
                const float i_t = lane_value(li, p), f_t = lane_value(lf, p);
                const float m_new = fmaxf(f_t + m, i_t);
                keeps[p] = expf(f_t + m - m_new);
                takes[p] = expf(i_t - m_new);
                m = m_new;
                floors[p] = expf(-m);
            }
        }
        if (stager)
#pragma unroll
            for (int p = 0; p < AH; p++) {
                float dot = 0.f;
#pragma unroll
                for (int n = 0; n < NR; n++) {
                    const int row = lane + 64 * n;
                    if (t0 + p < end) nn[n] = __builtin_fmaf(keeps[p], nn[n], takes[p] * kk[p][n]);
                    dot = __builtin_fmaf(nn[n], qq[p][n], dot);
                    if (row < DK) {
                        stage[p][0][row] = qq[p][n];
                        stage[p][1][row] = kk[p][n];
                    }
                }
                const float den = fmaxf(fabsf(wave_sum(dot)), floors[p]) + 1e-6f;
                if (lane == 0) dens_all[round][p] = den;
            }
        __syncthreads();
        float outs[AH], dens[AH];                        // stored together after the tokens: no branch of the lanes between them
#pragma unroll
        for (int p = 0; p < AH; p++) {
            outs[p] = 0.f;
            dens[p] = dens_all[round][p];
            if (t0 + p < end) {
                const float keep = keeps[p];
                const float tv = takes[p] * vv[p];
                const float4* Q4 = (const float4*)(stage[p][0] + row0);
                const float4* K4 = (const float4*)(stage[p][1] + row0);
                float o0 = 0.f, o1 = 0.f, o2 = 0.f, o3 = 0.f;                    // four sums: no FMA waits for the one before
#pragma unroll
                for (int i = 0; i < DKW; i += 4) {
                    if (i % 16 == 0) __builtin_amdgcn_sched_barrier(0);      // the reads of sixteen rows at a time, not of all
                    const float4 q4 = Q4[i / 4], k4 = K4[i / 4];
                    S[i] = __builtin_fmaf(keep, S[i], k4.x * tv);
                    o0 = __builtin_fmaf(q4.x, S[i], o0);
                    S[i + 1] = __builtin_fmaf(keep, S[i + 1], k4.y * tv);
                    o1 = __builtin_fmaf(q4.y, S[i + 1], o1);
                    S[i + 2] = __builtin_fmaf(keep, S[i + 2], k4.z * tv);
                    o2 = __builtin_fmaf(q4.z, S[i + 2], o2);
                    S[i + 3] = __builtin_fmaf(keep, S[i + 3], k4.w * tv);
                    o3 = __builtin_fmaf(q4.w, S[i + 3], o3);
                }
                outs[p] = (o0 + o1) + (o2 + o3);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (RS > 1) {                                // a group's first wave adds the parts of its waves
#pragma unroll
            for (int p = 0; p < AH; p++) parts[round][wave][p][lane] = outs[p];
            __syncthreads();
            if (part == 0)
#pragma unroll
                for (int p = 0; p < AH; p++) {
                    float sum = 0.f;
#pragma unroll
                    for (int w = 0; w < RS; w++) sum += parts[round][group * RS + w][p][lane];
                    outs[p] = sum;
                }
        }
        if (col && part == 0)
#pragma unroll
            for (int p = 0; p < AH; p++) if (t0 + p < end) a.y[((size_t)(t0 + p) * H + h) * dv + j] = outs[p] / dens[p];
        gi = gin; gf = gfn;
#pragma unroll
        for (int p = 0; p < AH; p++) {
            vv[p] = vn[p];
#pragma unroll
            for (int n = 0; n < NR; n++) { qq[p][n] = qn[p][n]; kk[p][n] = kn[p][n]; }
        }
    }
    if (col)
#pragma unroll
        for (int i = 0; i < DKW; i++) if (row0 + i < dk) st[(row0 + i) * dv + j] = S[i];
    if (wave == 0) {
#pragma unroll
        for (int n = 0; n < NR; n++) if (lane + 64 * n < dk) sn[lane + 64 * n] = nn[n];
        if (lane == 0) a.maximum[slot * H + h] = m;
    }
}

// ---- in chunks -------------------------------------------------------------------------------------------------------------------
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float mm_f32x4;

namespace {
constexpr int CHUNK = 64;                                // rows of a chunk, at most: a lane each where the gates are formed
constexpr int AUX = 8;                                   // floats of a chunk's ws_aux

// elements c .. c + 3 of a row of n, read inside of it (VEC: rows, their starts and n are whole pieces of four)
template <bool VEC>
__device__ __forceinline__ mm_f32x4 quad(const float* row, int c, int n) {
    if (VEC) return *reinterpret_cast<const mm_f32x4*>(row + min(c, n - 4));
    return (mm_f32x4){row[min(c, n - 1)], row[min(c + 1, n - 1)], row[min(c + 2, n - 1)], row[min(c + 3, n - 1)]};
}
template <bool VEC>
__device__ __forceinline__ mm_f32x4 quad(const bf16_t* row, int c, int n) {
    if (VEC) {
        const ushort4 u = *reinterpret_cast<const ushort4*>(row + min(c, n - 4));
        return (mm_f32x4){bf16_to_f32(u.x), bf16_to_f32(u.y), bf16_to_f32(u.z), bf16_to_f32(u.w)};
    }
    return (mm_f32x4){ld_f32(row + min(c, n - 1)), ld_f32(row + min(c + 1, n - 1)), ld_f32(row + min(c + 2, n - 1)), ld_f32(row + min(c + 3, n - 1))};
}
// the same with zeros past the end
template <bool VEC, typename P>
__device__ __forceinline__ mm_f32x4 quad_or_zero(const P* row, int c, int n) {
    mm_f32x4 x = quad<VEC>(row, c, n);
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = c + e < n ? x[e] : 0.f;
    return x;
}
template <bool VEC>
__device__ __forceinline__ void store_quad(float* row, int c, int n, mm_f32x4 x) {
    if (VEC) { if (c < n) *reinterpret_cast<mm_f32x4*>(row + c) = x; }
    else {
#pragma unroll
        for (int e = 0; e < 4; e++) if (c + e < n) row[c + e] = x[e];
    }
}
// (Every sum over more than 16 terms of one size is taken in pieces of 16 from zero: a chain over a whole head, let alone with the rows
// behind it, loses more than the four waves' parts of the kernel of whole sequences do.  Rows go in as they follow one another, 4 u + g of
// 16, and into a state in one chain: where gates forget, the last are the largest, and every sum after them is rounded at their size.)
__device__ __forceinline__ mm_f32x4 mm_mfma(float a, float b, mm_f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// e^x to float32's last place: the library's function of x rounded, corrected by what was rounded off
__device__ __forceinline__ float exp_of(double x) {
    const float hi = (float)x, e = expf(hi);
    return e > 0.f ? __builtin_fmaf(e, (float)(x - (double)hi), e) : e;
}

// The chunks lie in places one after the other, those of sequence 0 first, so that a launch has as many blocks as the step's rows fill and
// those of the sequences' last chunks, whatever the longest sequence has.  (With as many for every sequence as the longest needs, 2,048
// rows beside 63 single ones took 2.4 GB of workspace and 1,437 us, nearly all for chunks without rows; 0.13 GB and 289 us here.)
// The chunk at a place: its sequence, its number there, first row and rows.  False: there is none.  A lane counts a sequence's chunks,
// 64 sequences at a time.
__device__ __forceinline__ bool chunk_at(const MatrixMemoryArgs& a, int place, int lane, int& seq, int& number, int& begin, int& n) {
    for (int s0 = 0; s0 < a.n_seq; s0 += 64) {
        const int at = min(s0 + lane, a.n_seq - 1), row = a.cu_rows[at], rows = s0 + lane < a.n_seq ? a.cu_rows[at + 1] - row : 0;
        const int mine = (int)((unsigned)(rows + a.chunk - 1) / (unsigned)a.chunk);
        int up_to = mine;                                // the chunks up to and with the lane's sequence
        for (int o = 1; o < min(64, a.n_seq - s0); o <<= 1) {
            const int x = __shfl_up(up_to, o, 64);
            if (lane >= o) up_to += x;
        }
        const unsigned long long behind = __ballot(place < up_to);
        if (behind) {
            const int l = __ffsll((long long)behind) - 1;
            seq = s0 + l;
            number = place - (lane_value(up_to, l) - lane_value(mine, l));
            begin = lane_value(row, l) + number * a.chunk;
            n = min(lane_value(rows, l) - number * a.chunk, a.chunk);
            return true;
        }
        place -= lane_value(up_to, 63);
    }
    return false;
}

// A lane's row of a chunk of n rows: b, the sum of the log forget gates up to it, and a, its log input gate less b (-infinity past the
// chunk's end, where b stands still).
__device__ __forceinline__ void chunk_gates(const MatrixMemoryArgs& g, int begin, int n, int h, int lane, double& a, double& b) {
    const size_t t = (size_t)begin + min(lane, n - 1);
    const float li = g.cap * tanhf(g.gates[t * 2 * g.H + h] / g.cap), lf = log_sigmoid_f(g.cap * tanhf(g.gates[t * 2 * g.H + g.H + h] / g.cap));
    b = lane < n ? (double)lf : 0.0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double x = __shfl_up(b, o, 64);
        if (lane >= o) b += x;
    }
    a = lane < n ? (double)li - b : -INFINITY;
}
}

// What a chunk adds to the state, sum over its rows s of e^(a_s - M) k_s v_s^T with M about the largest a.  grid (places, heads,
// groups of 64 keys), a wave for every 64 values.  v is the A operand and the weighted k the B operand; a lane's four neighbours
// of a row of k or v belong to four tiles (element 4 r + tile of 64), so a lane ends up with four neighbours of a row of S.
template <typename T, bool VEC>
__global__ void __launch_bounds__(256)
mm_chunk_k(MatrixMemoryArgs a) {
    __shared__ float weights[4][CHUNK];
    const int h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4, H = a.H, dk = a.dk, dv = a.dv;
    float* const aux = a.ws_aux + ((size_t)blockIdx.x * H + h) * AUX;
    int seq = 0, number, begin = 0, n = 0;
    const bool any = chunk_at(a, blockIdx.x, lane, seq, number, begin, n);
    if (blockIdx.z == 0 && threadIdx.x == 0) {
        aux[5] = __int_as_float(seq); aux[6] = __int_as_float(begin); aux[7] = __int_as_float(n);
        if (any && number == 0 && h == 0) a.ws_first[seq] = blockIdx.x;
    }
    if (!any) return;
    double al, bl;
    chunk_gates(a, begin, n, h, lane, al, bl);
    double top = al;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top = fmax(top, __shfl_xor(top, o, 64));
    const double all = __shfl(bl, 63, 64);
    const float m = (float)(all + top);                  // the units of what is left are e^m as it is stored
    weights[wave][lane] = lane < n ? (float)exp(al - ((double)m - all)) : 0.f;
    if (blockIdx.z == 0 && threadIdx.x == 0) { aux[0] = m; aux[1] = (float)all; aux[4] = (float)(all - (double)(float)all); }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    const int i0 = blockIdx.z * 64, j0 = wave * 64, blocks = (n + 15) >> 4;
    const T* const kh = (const T*)a.k + (size_t)h * dk;
    const T* const vh = (const T*)a.v + (size_t)h * dv;
    mm_f32x4 acc[4][4];
#pragma unroll
    for (int x = 0; x < 4; x++)
#pragma unroll
        for (int y = 0; y < 4; y++) acc[x][y] = (mm_f32x4){0.f, 0.f, 0.f, 0.f};
    mm_f32x4 kq[2][4], vq[2][4];
    auto fetch = [&](int kb, int to) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const size_t t = (size_t)begin + min(16 * kb + 4 * u + g, n - 1);
            kq[to][u] = quad<VEC>(kh + t * a.k_stride, i0 + 4 * r, dk);
            vq[to][u] = quad<VEC>(vh + t * a.v_stride, j0 + 4 * r, dv);
        }
    };
    fetch(0, 0);
#pragma unroll
    for (int kb = 0; kb < 4; kb++) {
        if (kb >= blocks) break;
        if (kb + 1 < blocks) fetch(kb + 1, (kb + 1) & 1);
        float w[4];
#pragma unroll
        for (int u = 0; u < 4; u++) w[u] = weights[wave][16 * kb + 4 * u + g];
        if (16 * kb + 16 > n) {                          // rows past the chunk's end are its last again: no infinity of it may meet their weight of 0
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (16 * kb + 4 * u + g >= n) kq[kb & 1][u] = vq[kb & 1][u] = (mm_f32x4){0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int y = 0; y < 4; y++) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const float kw = kq[kb & 1][u][y] * w[u];
#pragma unroll
                for (int x = 0; x < 4; x++) acc[x][y] = mm_mfma(vq[kb & 1][u][x], kw, acc[x][y]);
            }
        }
    }
    float* const ws = a.ws_state + ((size_t)blockIdx.x * H + h) * ((size_t)dk * dv + dk);
#pragma unroll
    for (int y = 0; y < 4; y++) {
        const int i = i0 + 4 * r + y;
        if (i >= dk) continue;
#pragma unroll
        for (int v = 0; v < 4; v++)
            store_quad<VEC>(ws + (size_t)i * dv, j0 + 16 * g + 4 * v, dv, (mm_f32x4){acc[0][y][v], acc[1][y][v], acc[2][y][v], acc[3][y][v]});
    }
    if (wave == 0 && i0 + lane < dk) {
        float sum = 0.f;
#pragma unroll 8
        for (int s = 0; s < n; s++) sum = __builtin_fmaf(weights[0][s], ld_f32(kh + (size_t)(begin + s) * a.k_stride + i0 + lane), sum);
        ws[(size_t)dk * dv + i0 + lane] = sum;
    }
}

// Chunk after chunk of a sequence: the state that a chunk starts from takes the place of what it adds, and the sequence's last state goes
// to its slot.  A state x in units of e^m goes on over a chunk with F, the sum of its log forget gates, and M, the maximum it reaches
// from nothing, as m' = max(F + m, M), x' = e^(F + m - m') x + e^(M - m') (what the chunk adds).  grid (sequences, heads, blocks of
// 256 E elements of the matrix and the normalizer); the loads of eight chunks are in flight together.
template <int E>
__global__ void __launch_bounds__(256)
mm_carry_k(MatrixMemoryArgs a) {
    struct alignas(4 * E) Piece { float v[E]; };
    const int seq = blockIdx.x, h = blockIdx.y, e = (blockIdx.z * 256 + threadIdx.x) * E, H = a.H, dk = a.dk, dv = a.dv;
    const int n = (a.cu_rows[seq + 1] - a.cu_rows[seq] + a.chunk - 1) / a.chunk, per = dk * dv + dk;
    if (e >= per || n <= 0) return;
    const size_t slot = (size_t)a.slot_ids[seq];
    float* const home = e < dk * dv ? a.memory + (slot * H + h) * dk * dv + e : a.normalizer + (slot * H + h) * dk + e - dk * dv;
    Piece x = *reinterpret_cast<const Piece*>(home);
    float m = a.maximum[slot * H + h];
    const size_t g0 = (size_t)a.ws_first[seq];
    for (int c0 = 0; c0 < n; c0 += 8) {
        Piece L[8];
        float M[8];
        double F[8];
#pragma unroll
        for (int p = 0; p < 8; p++) {
            const size_t at = (g0 + min(c0 + p, n - 1)) * H + h;
            L[p] = *reinterpret_cast<const Piece*>(a.ws_state + at * per + e);
            M[p] = a.ws_aux[at * AUX];
            F[p] = (double)a.ws_aux[at * AUX + 1] + a.ws_aux[at * AUX + 4];
        }
#pragma unroll
        for (int p = 0; p < 8; p++) {
            const int c = c0 + p;
            if (c >= n) break;
            const size_t at = (g0 + c) * H + h;
            *reinterpret_cast<Piece*>(a.ws_state + at * per + e) = x;
            const double kept = F[p] + m;
            const float m_new = fmaxf((float)kept, M[p]), keep = exp_of(kept - m_new), take = exp_of((double)M[p] - m_new);
            if (e == 0) { a.ws_aux[at * AUX + 2] = m; a.ws_aux[at * AUX + 3] = m_new; }
#pragma unroll
            for (int i = 0; i < E; i++) x.v[i] = __builtin_fmaf(keep, x.v[i], take * L[p].v[i]);
            m = m_new;
        }
    }
    *reinterpret_cast<Piece*>(home) = x;
}

// A chunk's outputs from the state that it starts from.  grid (places, heads), a wave for every 64 values.  The chunk's
// weighted scores P[t, s] (k as the A operand, q as B) go to LDS, 16 rows t a wave; then every wave forms S0^T q and, its columns
// scaled, adds v^T P for its values, tiles of 16 rows t and 64 values whose A operand is four neighbours of a row of S0 or v.
template <typename T, bool VEC>
__global__ void __launch_bounds__(256)
mm_outputs_k(MatrixMemoryArgs a) {
    constexpr int PITCH = CHUNK + 4;
    __shared__ __attribute__((aligned(16))) float P[CHUNK][PITCH];
    __shared__ double as[4][CHUNK], tops[4][CHUNK];
    __shared__ float scales[4][CHUNK], floors[4][CHUNK], dens[CHUNK];
    const int h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4, H = a.H, dk = a.dk, dv = a.dv;
    const float* const aux = a.ws_aux + ((size_t)blockIdx.x * H + h) * AUX;
    const int seq = __float_as_int(aux[5]), begin = __float_as_int(aux[6]), n = __float_as_int(aux[7]);
    if (n <= 0) return;
    const float* const ws = a.ws_state + ((size_t)blockIdx.x * H + h) * ((size_t)dk * dv + dk);
    const T* const qh = (const T*)a.q + (size_t)h * dk;
    const T* const kh = (const T*)a.k + (size_t)h * dk;
    const T* const vh = (const T*)a.v + (size_t)h * dv;
    const int tiles = (n + 15) >> 4, blocks = (dk + 15) >> 4;
    {
        double al, bl;
        chunk_gates(a, begin, n, h, lane, al, bl);
        const float m0 = aux[2];
        double top = fmax(al, (double)m0);
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const double x = __shfl_up(top, o, 64);
            if (lane >= o) top = fmax(top, x);
        }
        as[wave][lane] = al;
        tops[wave][lane] = top;
        scales[wave][lane] = (float)exp((double)m0 - top);
        floors[wave][lane] = (float)exp(-(bl + top));
        if (threadIdx.x == 0 && begin + n == a.cu_rows[seq + 1]) a.maximum[(size_t)a.slot_ids[seq] * H + h] = aux[3];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    const int waves = blockDim.x >> 6;
    for (int tt = wave; tt < tiles; tt += waves) {
        const int t = 16 * tt + r;
        const T* const qt = qh + (size_t)(begin + min(t, n - 1)) * a.q_stride;
        mm_f32x4 s[4];
#pragma unroll
        for (int st = 0; st < 4; st++) s[st] = (mm_f32x4){0.f, 0.f, 0.f, 0.f};
        float sum = 0.f;
        for (int kb = 0; kb < blocks; kb++) {
            const int c = 16 * kb + 4 * g;
            const mm_f32x4 q = quad_or_zero<VEC>(qt, c, dk) * a.q_scale, nq = quad_or_zero<VEC>(ws + (size_t)dk * dv, c, dk);
            mm_f32x4 k[4];
#pragma unroll
            for (int st = 0; st < 4; st++)
                if (st <= tt) k[st] = quad_or_zero<VEC>(kh + (size_t)(begin + min(16 * st + r, n - 1)) * a.k_stride, c, dk);
            mm_f32x4 p[4] = {};
#pragma unroll
            for (int u = 0; u < 4; u++) {
                sum = __builtin_fmaf(nq[u], q[u], sum);
#pragma unroll
                for (int st = 0; st < 4; st++) if (st <= tt) p[st] = mm_mfma(k[st][u], q[u], p[st]);
            }
#pragma unroll
            for (int st = 0; st < 4; st++) if (st <= tt) s[st] += p[st];
        }
        sum *= scales[wave][t];
        const double top = tops[wave][t];
#pragma unroll
        for (int st = 0; st < 4; st++)
            if (st <= tt) {
                mm_f32x4 p;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int row = 16 * st + 4 * g + v;
                    p[v] = row <= t && row < n ? s[st][v] * exp_of(as[wave][row] - top) : 0.f;
                    sum += p[v];
                }
                *reinterpret_cast<mm_f32x4*>(&P[t][16 * st + 4 * g]) = p;
            }
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        if (g == 0) dens[t] = fmaxf(fabsf(sum), floors[wave][t]) + 1e-6f;
    }
    __syncthreads();

    const int j0 = wave * 64;
    mm_f32x4 acc[4][4];                                  // [value 4 r + x of the wave's 64][tile of rows t]
#pragma unroll
    for (int x = 0; x < 4; x++)
#pragma unroll
        for (int tt = 0; tt < 4; tt++) acc[x][tt] = (mm_f32x4){0.f, 0.f, 0.f, 0.f};
    mm_f32x4 sq[4], qq[4], sn[4], qn[4];
    auto fetch = [&](int kb, mm_f32x4 (&S)[4], mm_f32x4 (&Q)[4]) {
#pragma unroll
        for (int u = 0; u < 4; u++) S[u] = quad<VEC>(ws + (size_t)min(16 * kb + 4 * g + u, dk - 1) * dv, j0 + 4 * r, dv);
#pragma unroll
        for (int tt = 0; tt < 4; tt++) Q[tt] = quad<VEC>(qh + (size_t)(begin + min(16 * tt + r, n - 1)) * a.q_stride, 16 * kb + 4 * g, dk);
    };
    fetch(0, sq, qq);
    for (int kb = 0; kb < blocks; kb++) {
        if (kb + 1 < blocks) fetch(kb + 1, sn, qn);
        if (16 * kb + 16 > dk) {                         // keys past the end are the last again, as above
#pragma unroll
            for (int u = 0; u < 4; u++) if (16 * kb + 4 * g + u >= dk) sq[u] = (mm_f32x4){0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int tt = 0; tt < 4; tt++) {
            if (tt >= tiles) break;
            mm_f32x4 p[4] = {};
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const float q = 16 * kb + 4 * g + u < dk ? qq[tt][u] * a.q_scale : 0.f;
#pragma unroll
                for (int x = 0; x < 4; x++) p[x] = mm_mfma(sq[u][x], q, p[x]);
            }
#pragma unroll
            for (int x = 0; x < 4; x++) acc[x][tt] += p[x];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) { sq[u] = sn[u]; qq[u] = qn[u]; }
    }
    const float first = scales[wave][r];                 // of the first tile: goes into its one addition
#pragma unroll
    for (int tt = 1; tt < 4; tt++) {
        const float f = scales[wave][16 * tt + r];
#pragma unroll
        for (int x = 0; x < 4; x++) acc[x][tt] *= f;
    }
#pragma unroll
    for (int kb = 0; kb < 4; kb++) {
        if (kb >= tiles) break;
        mm_f32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = quad<VEC>(vh + (size_t)(begin + min(16 * kb + 4 * u + g, n - 1)) * a.v_stride, j0 + 4 * r, dv);
        // The tile's own rows t do not see the rows behind them: a weight of 0 keeps finite values out, but no infinity and no NaN.
        // Where a value is none, the tile is summed row after row without what is not seen.
        float none = 0.f;
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int x = 0; x < 4; x++) none = __builtin_fmaf(v[u][x], 0.f, none);
        const bool finite = !__any(none != 0.f);
#pragma unroll
        for (int tt = kb; tt < 4; tt++) {
            if (tt >= tiles) break;
            mm_f32x4 p[4] = {};
            if (tt == kb && !finite) {
                for (int s = 16 * kb; s < min(16 * kb + 16, n); s++) {
                    const float w = P[16 * kb + r][s];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const mm_f32x4 value = quad<VEC>(vh + (size_t)(begin + s) * a.v_stride, j0 + 16 * g + 4 * e, dv);
#pragma unroll
                        for (int x = 0; x < 4; x++) p[x][e] = s <= 16 * kb + r ? __builtin_fmaf(value[x], w, p[x][e]) : p[x][e];
                    }
                }
            } else {
                float w[4];
#pragma unroll
                for (int u = 0; u < 4; u++) w[u] = P[16 * tt + r][16 * kb + 4 * u + g];
#pragma unroll
                for (int u = 0; u < 4; u++)
#pragma unroll
                    for (int x = 0; x < 4; x++) p[x] = mm_mfma(v[u][x], w[u], p[x]);
            }
#pragma unroll
            for (int x = 0; x < 4; x++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[x][tt][e] = tt == 0 ? __builtin_fmaf(acc[x][tt][e], first, p[x][e]) : acc[x][tt][e] + p[x][e];
        }
    }
#pragma unroll
    for (int tt = 0; tt < 4; tt++) {
        const int t = 16 * tt + r;
        if (t >= n) continue;
        const float den = dens[t];
        float* const y = a.y + ((size_t)(begin + t) * H + h) * dv;
#pragma unroll
        for (int v = 0; v < 4; v++)
            store_quad<VEC>(y, j0 + 16 * g + 4 * v, dv, (mm_f32x4){acc[0][tt][v] / den, acc[1][tt][v] / den, acc[2][tt][v] / den, acc[3][tt][v] / den});
    }
}

extern "C" long tp_matrix_memory_scan_workspace_floats(int n_seq, int places, int H, int dk, int dv) {
    return (long)places * H * ((long)dk * dv + dk + AUX) + n_seq;
}

template <typename T>
static void chunks_launch(const MatrixMemoryArgs& a, bool vec, hipStream_t s) {
    const int threads = 64 * tp_cdiv(a.dv, 64), per = a.dk * a.dv + a.dk;
    const dim3 chunks(a.places, a.H), groups(a.places, a.H, tp_cdiv(a.dk, 64));
    if (vec) {
        mm_chunk_k<T, true><<<groups, threads, 0, s>>>(a);
        mm_carry_k<4><<<dim3(a.n_seq, a.H, tp_cdiv(per, 1024)), 256, 0, s>>>(a);
        mm_outputs_k<T, true><<<chunks, threads, 0, s>>>(a);
    } else {
        mm_chunk_k<T, false><<<groups, threads, 0, s>>>(a);
        mm_carry_k<1><<<dim3(a.n_seq, a.H, tp_cdiv(per, 256)), 256, 0, s>>>(a);
        mm_outputs_k<T, false><<<chunks, threads, 0, s>>>(a);
    }
}

// chunk 0: whole sequences, in pieces of one row where no sequence has more (one_row_each); otherwise chunks of up to 64 rows, `places`
// of them in all sequences or more.
// memory [slots, H, dk, dv], normalizer [slots, H, dk], maximum [slots, H], gates [M, 2 H] (input sums, then forget sums), all float32
extern "C" int tp_matrix_memory_scan(const void* q, long q_stride, const void* k, long k_stride, const void* v, long v_stride, int dtype,
                                     const float* gates, float cap, float q_scale, float* memory, float* normalizer, float* maximum,
                                     const int* slot_ids, const int* cu_rows, float* y, int n_seq, int H, int dk, int dv,
                                     int chunk, int places, float* workspace, int one_row_each, void* stream) {
    TP_REQUIRE(n_seq > 0 && H > 0 && dk > 0 && dv > 0, "matrix_memory_scan: empty shape sequences=%d heads=%d key=%d value=%d", n_seq, H, dk, dv);
    TP_REQUIRE(dk <= 256, "matrix_memory_scan: keys of %d elements exceed the 256 a lane keeps", dk);
    TP_REQUIRE(dv <= 256, "matrix_memory_scan: values of %d elements exceed the 256 columns of a block", dv);
    TP_REQUIRE(H <= 65535, "matrix_memory_scan: %d heads exceed one launch", H);
    TP_REQUIRE(cap > 0.f, "matrix_memory_scan: the gates' cap must be positive");
    TP_REQUIRE(q && k && v && gates && memory && normalizer && maximum && slot_ids && cu_rows && y, "matrix_memory_scan: null operand");
    TP_REQUIRE(chunk == 0 || (chunk > 0 && chunk <= CHUNK && places > 0 && workspace),
               "matrix_memory_scan: %d chunks of %d rows (at most %d) need a workspace", places, chunk, CHUNK);
    TP_REQUIRE(dtype == TP_BF16 || dtype == TP_F32, "matrix_memory_scan: unknown dtype %d", dtype);
    hipStream_t s = (hipStream_t)stream;
    float* ws_aux = workspace ? workspace + (size_t)places * H * ((size_t)dk * dv + dk) : nullptr;
    int* ws_first = workspace ? (int*)(ws_aux + (size_t)places * H * AUX) : nullptr;
    const MatrixMemoryArgs a{q, q_stride, k, k_stride, v, v_stride, gates, cap, q_scale, memory, normalizer, maximum, slot_ids, cu_rows, y, n_seq, H, dk, dv,
                             chunk, places, workspace, ws_aux, ws_first};
    const size_t piece = dtype == TP_BF16 ? 8 : 16;
    if (chunk > 0) {
        const bool vec = dk % 4 == 0 && dv % 4 == 0 && q_stride % 4 == 0 && k_stride % 4 == 0 && v_stride % 4 == 0 &&
                         ((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) % piece == 0 &&
                         ((uintptr_t)memory | (uintptr_t)normalizer | (uintptr_t)workspace | (uintptr_t)y) % 16 == 0;
        if (dtype == TP_BF16) chunks_launch<bf16_t>(a, vec, s);
        else chunks_launch<float>(a, vec, s);
        return tp_check_launch("matrix_memory_scan (chunks)");
    }
    const dim3 grid(n_seq, H);
    const int step_threads = one_row_each && (uintptr_t)memory % 16 == 0 ? tp_step_threads(dk, dv) : 0;
    if (step_threads) {
        const int rows = tp_cdiv((long)dk * dv, 4 * step_threads);
#define TP_STEP(R) do { if (dtype == TP_BF16) matrix_memory_step_k<bf16_t, R><<<grid, step_threads, 0, s>>>(a); else matrix_memory_step_k<float, R><<<grid, step_threads, 0, s>>>(a); } while (0)
        if (rows <= 2) TP_STEP(2); else if (rows <= 4) TP_STEP(4); else if (rows <= 8) TP_STEP(8); else TP_STEP(16);
#undef TP_STEP
        return tp_check_launch("matrix_memory_scan (one row)");
    }
    const int threads = 64 * tp_cdiv(dv, 64);            // times the waves a group of columns is split over
#define TP_LAUNCH(DK) do { if (dtype == TP_BF16) matrix_memory_scan_k<bf16_t, DK><<<grid, threads * TP_MM_SPLIT(DK), 0, s>>>(a); else matrix_memory_scan_k<float, DK><<<grid, threads * TP_MM_SPLIT(DK), 0, s>>>(a); } while (0)
    TP_SCAN_SIZES(TP_LAUNCH, dk);
#undef TP_LAUNCH
    return tp_check_launch("matrix_memory_scan");
}
