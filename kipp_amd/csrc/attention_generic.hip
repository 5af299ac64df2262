// Causal grouped-query attention over the paged cache for any mix of query
// tokens (prompt portions and single decoded tokens alike), any key size up
// to 1,024, values of their own width (`dv`; the value cache may be the key
// cache itself, a value then being the first dv numbers of its key's row of
// `v_row` numbers) and any storage type: the float32 path's kernel and the fallback of sizes the MFMA kernels refuse.
//
// For query position p of a sequence the keys are s in [max(0, p-window+1), p]
// (window 0: from 0; with `chunk` c > 0 from p - p % c, the start of p's chunk of c positions counted from 0), score = (q . k_s) * scale (with `softcap` c > 0: c tanh(score / c)), softmax with the maximum
// subtracted (with `sink` one more term e^0 joins the denominator: a key of score 0 without a value),
// out = sum p_s v_s  (/root/reference/src/kipp.c:2882-2922).
//
// Keys are taken in blocks of 64 aligned to absolute key index.  A block gives its maximum, its denominator and its sum
// of values by itself, and the blocks are merged in order, so the sequence of operations for one query depends on its own
// position only: not on what else is in the batch, and not on how many waves share the blocks.
//
// A workgroup takes (token, HPW query heads of one key/value head); its WAVES waves take the blocks in turn, and wave h
// merges head h's after every round (one wave alone merges where it stands).  A lane holds a key for the scores, so
// that a key is read once for HPW heads, and C columns of the values.
// Bound by the chain of loads of a block (a lane's key row, then 64 value rows), so by how many blocks are under way:
// one token behind 333 keys (32 heads over 8, float32) takes 19 us, 333 tokens 59 us.  One wave a (token, head) that
// walked its keys with sixteen predicated columns a key took 355 and 330 us.
#include "common.h"
#include <math.h>
#include <algorithm>

#define MAX_D 1024
#define BLOCK_KEYS KIPP_WAVE

__device__ __forceinline__ void load4(const float* p, float (&v)[4]) {
    const float4 u = *reinterpret_cast<const float4*>(p);
    v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
}
__device__ __forceinline__ void load4(const bf16_t* p, float (&v)[4]) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    v[0] = __uint_as_float(u.x << 16); v[1] = __uint_as_float(u.x & 0xffff0000u);
    v[2] = __uint_as_float(u.y << 16); v[3] = __uint_as_float(u.y & 0xffff0000u);
}

// HPW dots q . k over d numbers, each added in index order whatever the width of the loads.  q_s: [HPW][dp].
template <int HPW, typename TC>
__device__ __forceinline__ void dots(const float* __restrict__ q_s, int dp, const TC* __restrict__ k, int d, float (&dot)[HPW]) {
#pragma unroll
    for (int h = 0; h < HPW; ++h) dot[h] = 0.0f;
    int e = 0;
    if ((((uintptr_t)k) & (4 * sizeof(TC) - 1)) == 0) {
#pragma unroll 8
        for (; e + 4 <= d; e += 4) {
            float v[4];
            load4(k + e, v);
#pragma unroll
            for (int h = 0; h < HPW; ++h) {
                const float4 qv = *reinterpret_cast<const float4*>(q_s + h * dp + e);
                dot[h] = fmaf(qv.x, v[0], dot[h]);
                dot[h] = fmaf(qv.y, v[1], dot[h]);
                dot[h] = fmaf(qv.z, v[2], dot[h]);
                dot[h] = fmaf(qv.w, v[3], dot[h]);
            }
        }
    }
    for (; e < d; ++e) {
        const float v = load_f(k, e);
#pragma unroll
        for (int h = 0; h < HPW; ++h) dot[h] = fmaf(q_s[h * dp + e], v, dot[h]);
    }
}

// What the blocks so far have left of one head in a lane: the maximum, the denominator, C columns of the sum.
template <int C>
struct Merged {
    float m, l, acc[C];
    __device__ __forceinline__ void start() {
        m = -INFINITY;
        l = 0.0f;
#pragma unroll
        for (int c = 0; c < C; ++c) acc[c] = 0.0f;
    }
    // the scales of what is here and of the next block (a block whose scores are all -inf weighs nothing: mb = -inf, lb = 0)
    __device__ __forceinline__ void turn(float mb, float lb, float& a, float& b) {
        const float top = fmaxf(m, mb);
        a = m == top ? 1.0f : expf(m - top);
        b = mb == top ? 1.0f : expf(mb - top);
        m = top;
        l = fmaf(l, a, __fmul_rn(lb, b));
    }
    __device__ __forceinline__ void add(int c, float a, float b, float accb) { acc[c] = fmaf(acc[c], a, __fmul_rn(accb, b)); }
    template <typename TO>
    __device__ __forceinline__ void write(TO* __restrict__ row, int lane, int dv, int sink) {
        float under = l;
        if (sink) under += expf(-m);        // the term of score 0 (m is finite: a position sees itself)
        const float inv = 1.0f / under;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int e = lane + c * KIPP_WAVE;
            if (e < dv) store_f(row, e, __fmul_rn(acc[c], inv));
        }
    }
};

template <typename TQ, typename TC, typename TO, int HPW, int C, int WAVES>
__global__ void __launch_bounds__(WAVES * KIPP_WAVE) paged_attention_generic_kernel(
    const TQ* __restrict__ q, const TC* __restrict__ k_cache, const TC* __restrict__ v_cache, TO* __restrict__ out,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ seq_of_token,
    const int32_t* __restrict__ block_table, int max_blocks,
    int n_q, int n_kv, int d, int dv, int v_row, int page, float scale, int window, float softcap, int chunk, int sink) {
    static_assert(WAVES == 1 || WAVES >= HPW, "a wave a head merges");
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int dp = (d + 3) & ~3;
    float* q_s = lds;                                        // [HPW][dp]
    float* p_s = q_s + HPW * dp;                             // [WAVES][64][HPW]
    float* part_s = p_s + WAVES * BLOCK_KEYS * HPW;          // [WAVES][HPW][2 + C 64] (several waves): maximum, denominator, sum
    __shared__ unsigned long long off_all[WAVES][BLOCK_KEYS];
    constexpr int PART = 2 + C * KIPP_WAVE;
    const int wave = threadIdx.x / KIPP_WAVE;
    const int lane = threadIdx.x & (KIPP_WAVE - 1);
    const int t = blockIdx.y;
    const int head0 = blockIdx.x * HPW;
    const int g = head0 / (n_q / n_kv);
    const int pos = positions[t];
    const int32_t* table = block_table + (size_t)seq_of_token[t] * max_blocks;
    const int lo = chunk > 0 ? pos - pos % chunk : (window > 0 ? max(0, pos - window + 1) : 0);

    for (int i = threadIdx.x; i < HPW * dp; i += WAVES * KIPP_WAVE) {
        const int h = i / dp, e = i - h * dp;
        q_s[i] = e < d ? load_f(q + ((size_t)t * n_q + head0 + h) * d, e) : 0.0f;
    }
    __syncthreads();

    float* p_w = p_s + wave * BLOCK_KEYS * HPW;
    unsigned long long* off_s = off_all[wave];
    constexpr int RUNS = WAVES == 1 ? HPW : 1;
    Merged<C> run[RUNS];
#pragma unroll
    for (int r = 0; r < RUNS; ++r) run[r].start();
    const int first = lo / BLOCK_KEYS, last = pos / BLOCK_KEYS;
    for (int b0 = first; b0 <= last; b0 += WAVES) {
        const int s0 = (b0 + wave) * BLOCK_KEYS;
        float mb[HPW], lb[HPW], acc[HPW][C];
        if (s0 <= pos) {
            const int s = s0 + lane;
            const bool valid = s >= lo && s <= pos;
            float score[HPW];
#pragma unroll
            for (int h = 0; h < HPW; ++h) score[h] = -INFINITY;
            unsigned long long off = 0;
            if (valid) {
                off = ((unsigned long long)table[s / page] * n_kv + g) * page + s % page;
                dots<HPW>(q_s, dp, k_cache + off * d, d, score);
#pragma unroll
                for (int h = 0; h < HPW; ++h) {
                    score[h] = __fmul_rn(score[h], scale);
                    if (softcap > 0.0f) score[h] = softcap * tanhf(score[h] / softcap);
                }
            }
            off_s[lane] = off;
#pragma unroll
            for (int h = 0; h < HPW; ++h) {
                mb[h] = wave_max(score[h]);
                const float p = score[h] != -INFINITY ? expf(score[h] - mb[h]) : 0.0f;      // -inf: not seen, or of no weight
                lb[h] = wave_sum(p);
                p_w[lane * HPW + h] = p;
#pragma unroll
                for (int c = 0; c < C; ++c) acc[h][c] = 0.0f;
            }
            __builtin_amdgcn_wave_barrier();        // LDS is in order within a wave: the compiler keeps the order too
            // every column's sum runs over the keys in order; the keys are the outer loop so that the loads of several are on their way together
            const int j_lo = max(0, lo - s0), j_hi = min(BLOCK_KEYS, pos - s0 + 1);
#pragma unroll 8
            for (int j = j_lo; j < j_hi; ++j) {
                const TC* v_at = v_cache + off_s[j] * v_row;
                float p[HPW];
#pragma unroll
                for (int h = 0; h < HPW; ++h) p[h] = p_w[j * HPW + h];
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const int e = lane + c * KIPP_WAVE;
                    const float v = load_f(v_at, e < dv ? e : 0);       // a lane beyond the value's width reads its first number
#pragma unroll
                    for (int h = 0; h < HPW; ++h) acc[h][c] = fmaf(p[h], v, acc[h][c]);
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
        if constexpr (WAVES == 1) {
#pragma unroll
            for (int h = 0; h < HPW; ++h) {
                float a, b;
                run[h].turn(mb[h], lb[h], a, b);
#pragma unroll
                for (int c = 0; c < C; ++c) run[h].add(c, a, b, acc[h][c]);
            }
        } else {
            if (s0 <= pos) {
#pragma unroll
                for (int h = 0; h < HPW; ++h) {
                    float* part = part_s + (wave * HPW + h) * PART;
                    if (lane == 0) {
                        part[0] = mb[h];
                        part[1] = lb[h];
                    }
#pragma unroll
                    for (int c = 0; c < C; ++c) part[2 + c * KIPP_WAVE + lane] = acc[h][c];
                }
            }
            __syncthreads();
            if (wave < HPW) {
                const int n = min(WAVES, last - b0 + 1);
                for (int w = 0; w < n; ++w) {
                    const float* part = part_s + (w * HPW + wave) * PART;
                    float a, b;
                    run[0].turn(part[0], part[1], a, b);
#pragma unroll
                    for (int c = 0; c < C; ++c) run[0].add(c, a, b, part[2 + c * KIPP_WAVE + lane]);
                }
            }
            __syncthreads();
        }
    }
    if constexpr (WAVES == 1) {
#pragma unroll
        for (int h = 0; h < HPW; ++h) run[h].write(out + ((size_t)t * n_q + head0 + h) * dv, lane, dv, sink);
    } else if (wave < HPW) {
        run[0].write(out + ((size_t)t * n_q + head0 + wave) * dv, lane, dv, sink);
    }
}

struct GenericArgs {
    const void *q, *k, *v;
    void* out;
    const int32_t *positions, *seq_of_token, *block_table;
    int max_blocks, n_tokens, n_q, n_kv, d, dv, v_row, page;
    float scale;
    int window;
    float softcap;
    int chunk, sink;
    hipStream_t stream;
};

template <typename TQ, typename TC, typename TO, int HPW, int C, int WAVES>
static int launch_waves(const GenericArgs& a) {
    const int dp = (a.d + 3) & ~3;
    const size_t lds = sizeof(float) * ((size_t)HPW * dp + WAVES * BLOCK_KEYS * HPW + (WAVES > 1 ? WAVES * HPW * (2 + C * KIPP_WAVE) : 0));
    hipLaunchKernelGGL((paged_attention_generic_kernel<TQ, TC, TO, HPW, C, WAVES>), dim3(a.n_q / HPW, a.n_tokens), dim3(WAVES * KIPP_WAVE), lds,
                       a.stream, (const TQ*)a.q, (const TC*)a.k, (const TC*)a.v, (TO*)a.out, a.positions, a.seq_of_token, a.block_table,
                       a.max_blocks, a.n_q, a.n_kv, a.d, a.dv, a.v_row, a.page, a.scale, a.window, a.softcap, a.chunk, a.sink);
    return KIPP_LAUNCH_CHECK();
}

// How many waves share a token's blocks changes how long they take, never what comes out: enough of them to fill the chip
// (256 compute units of 16 waves each), no more than there are blocks.
template <typename TQ, typename TC, typename TO, int HPW, int C>
static int launch_heads(const GenericArgs& a) {
    const long long groups = (long long)a.n_tokens * (a.n_q / HPW);
    const long long table_keys = (long long)a.max_blocks * a.page;
    const long long keys = a.window > 0 ? std::min(table_keys, (long long)a.window + BLOCK_KEYS) : (a.chunk > 0 ? std::min(table_keys, (long long)a.chunk + BLOCK_KEYS) : table_keys);
    const long long blocks = (keys + BLOCK_KEYS - 1) / BLOCK_KEYS;
    if (groups >= 8192 || blocks <= 1) return launch_waves<TQ, TC, TO, HPW, C, 1>(a);
    if (groups >= 1024 || blocks <= 4) return launch_waves<TQ, TC, TO, HPW, C, 4>(a);
    return launch_waves<TQ, TC, TO, HPW, C, 8>(a);
}

template <typename TQ, typename TC, typename TO>
static int launch_types(const GenericArgs& a) {
    const int group = a.n_q / a.n_kv, columns = (a.dv + KIPP_WAVE - 1) / KIPP_WAVE;
    if (columns > 8) return launch_heads<TQ, TC, TO, 1, 16>(a);
    if (columns > 4) return launch_heads<TQ, TC, TO, 1, 8>(a);
    if (columns > 2) return group % 2 == 0 ? launch_heads<TQ, TC, TO, 2, 4>(a) : launch_heads<TQ, TC, TO, 1, 4>(a);
    if (group % 4 == 0) return launch_heads<TQ, TC, TO, 4, 2>(a);
    return group % 2 == 0 ? launch_heads<TQ, TC, TO, 2, 2>(a) : launch_heads<TQ, TC, TO, 1, 2>(a);
}

// Values of width dv in rows of v_row numbers (v_row = dv for a value cache of its own).
extern "C" int kipp_paged_attention_generic_masked(
    const void* q, int q_dtype, const void* k_cache, const void* v_cache, int cache_dtype, void* out, int out_dtype,
    const int32_t* positions, const int32_t* seq_of_token, const int32_t* block_table, int max_blocks,
    int n_tokens, int n_q, int n_kv, int d, int dv, int v_row, int page, float scale, int window, float softcap,
    int chunk, int sink, hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (chunk < 0 || (chunk > 0 && window > 0)) return -1;
    if (d > MAX_D || d <= 0 || dv > MAX_D || dv <= 0 || v_row < dv || n_kv <= 0 || n_q % n_kv) return -1;
    const GenericArgs a = {q, k_cache, v_cache, out, positions, seq_of_token, block_table, max_blocks, n_tokens, n_q, n_kv, d, dv, v_row, page,
                           scale, window, softcap, chunk, sink, stream};
    if (q_dtype == KIPP_F32 && cache_dtype == KIPP_F32 && out_dtype == KIPP_F32) return launch_types<float, float, float>(a);
    if (q_dtype == KIPP_BF16 && cache_dtype == KIPP_BF16 && out_dtype == KIPP_BF16) return launch_types<bf16_t, bf16_t, bf16_t>(a);
    return -2;
}

extern "C" int kipp_paged_attention_generic_capped(
    const void* q, int q_dtype, const void* k_cache, const void* v_cache, int cache_dtype, void* out, int out_dtype,
    const int32_t* positions, const int32_t* seq_of_token, const int32_t* block_table, int max_blocks,
    int n_tokens, int n_q, int n_kv, int d, int dv, int v_row, int page, float scale, int window, float softcap,
    hipStream_t stream) {
    return kipp_paged_attention_generic_masked(q, q_dtype, k_cache, v_cache, cache_dtype, out, out_dtype, positions, seq_of_token,
                                               block_table, max_blocks, n_tokens, n_q, n_kv, d, dv, v_row, page, scale, window, softcap,
                                               0, 0, stream);
}

extern "C" int kipp_paged_attention_generic_v(
    const void* q, int q_dtype, const void* k_cache, const void* v_cache, int cache_dtype, void* out, int out_dtype,
    const int32_t* positions, const int32_t* seq_of_token, const int32_t* block_table, int max_blocks,
    int n_tokens, int n_q, int n_kv, int d, int dv, int v_row, int page, float scale, int window, hipStream_t stream) {
    return kipp_paged_attention_generic_capped(q, q_dtype, k_cache, v_cache, cache_dtype, out, out_dtype, positions, seq_of_token,
                                               block_table, max_blocks, n_tokens, n_q, n_kv, d, dv, v_row, page, scale, window, 0.0f, stream);
}

extern "C" int kipp_paged_attention_generic(
    const void* q, int q_dtype, const void* k_cache, const void* v_cache, int cache_dtype, void* out, int out_dtype,
    const int32_t* positions, const int32_t* seq_of_token, const int32_t* block_table, int max_blocks,
    int n_tokens, int n_q, int n_kv, int d, int page, float scale, int window, hipStream_t stream) {
    if (d > 256) return -1;
    return kipp_paged_attention_generic_v(q, q_dtype, k_cache, v_cache, cache_dtype, out, out_dtype, positions, seq_of_token,
                                          block_table, max_blocks, n_tokens, n_q, n_kv, d, d, d, page, scale, window, stream);
}
