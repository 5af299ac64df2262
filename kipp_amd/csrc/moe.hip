// A routed feed-forward (mixture of experts): the router's choice, the tokens sorted by expert, the experts'
// two products over those runs of rows, and the weighted sum.
//
//     route    p = softmax(z) over all experts (float32); the `top` largest p (the lower index first among equals);
//              weight = p / (sum of the chosen p + eps)
//     route (grouped)  s = sigmoid(z), or softmax(z); choice scores c = s + correction; experts in equal groups of neighbours, a
//              group's score the sum of its two largest c, or its largest; only experts of the `keep` best groups can be chosen; the
//              `top` largest c among them; weight = s / (sum of the chosen s + eps) * scale, or s * scale (not renormalized)
//     sort     the (token, choice) pairs in runs of one expert each, cut into tiles of up to 16 (64, 128, 256) rows; the list of tiles
//              is made on the device, so the host never learns the counts and the launches have a fixed shape.  The router may
//              have more outputs than there are experts with matrices: those behind are identity experts, whose pairs get no
//              row (place -1)
//     expert   a tile's rows against its expert's matrix: out[row][n] = act(sum_k W_e[n][k] x[row][k]).  bfloat16 with K a
//              multiple of 32: on the matrix cores, in three forms.  Few rows an expert (tiles of up to 64): a workgroup 16 columns,
//              its eight waves every eighth 64 numbers of k each, whose sums are added in order.  Walking (tiles of
//              up to 64, 128 or 256): the walk of the prompt products, one chain of 16 x 16 x 32 products along k.  Staged (tiles of up to
//              128, for rows and matrices that begin at no multiple of 16 bytes): a workgroup
//              128 columns, 64 numbers of k a step through registers and LDS, the same chain.  Else (float32, other K): a
//              lane takes a column of a tile of 16 rows, one chain along k.
//              A form sums over k in one order for every row, whichever tile the row is in; the forms' orders differ, and the form
//              follows from the pairs of the whole step and the matrices' sizes: under bfloat16 a token's last bits depend on how
//              many tokens share its step
//     gated expert  the same against an expert's [gate; up] matrix with a weight s a row of x:
//              out[row][n] = act(s (W_gate x)[n]) * s (W_up x)[n], which is the expert applied to s x; on the matrix cores a wave's
//              two fragments of 16 columns are the gate's and the up's of the same 16 inner columns
//     combine  out[t] = sum_j weight[t][j] y[place of (t, j)], or weight[t][j] x[t] for an identity expert (+ the shared expert's
//              result, slabs added in order, maybe times the sigmoid of a logit of its own)
#include "line_walk.h"
#include <math.h>

#define ROUTE_WAVES 4
#define MAX_EXPERTS 1024
#define MAX_TOP 32
#define SORT_THREADS 1024
#define TILE_ROWS 16
#define EXPERT_COLS 256
#define EXPERT_KC 128
#define MFMA_ROWS 128       // rows of a tile of the matrix-core products for whole tiles: eight fragments of 16, or four of 32
#define MFMA_COLS 128       // columns of a workgroup of the staged one: four waves with two fragments each
#define MFMA_NF (MFMA_COLS / 64)
#define MFMA_KC 64          // numbers of k a step brings into LDS
#define MFMA_PITCH 72       // bfloat16 numbers from a row to the next in LDS
#define MFMA_THREADS 256
#define MANY_ROWS 256       // rows of a tile of the walking one where an expert has many
#define TILE_ACROSS 4       // waves of its workgroup across the columns, two down
#define TILE_COLS(GLU) (((GLU) ? 32 : 64) * TILE_ACROSS)     // output columns of its tile
#define ROWS_TILE 64        // rows of a tile of the product for few rows
#define ROWS_WAVES 8        // waves of its workgroup
#define ROWS_SHORT_K 1024   // K up to which a workgroup of it has two steps a wave at most, and is the slower one
#define ROWS_SHORT_GROUPS 2048      // in a launch of more workgroups than this
#define DIE_UNITS 32        // compute units of a die
#define XCDS 8              // dies of the chip; consecutive workgroups of a launch go to them in turn

enum { ACT_NONE = -1, ACT_SILU = 0, ACT_RELU = 1, ACT_GELU = 2, ACT_GELU_TANH = 3, ACT_RELU2 = 4 };

// exp(-a) for a >= 0 (beyond 150 that of 150: zero).  a / ln 2 in two parts, so that its fraction keeps its bits.
__device__ __forceinline__ float exp_minus(float a) {
    a = fminf(a, 150.0f);
    const float t = a * -1.44269502f, k = rintf(t);
    const float low = fmaf(a, -1.92596303e-8f, fmaf(a, -1.44269502f, -t));
    return ldexpf(__builtin_amdgcn_exp2f((t - k) + low), (int)k);
}

// z / (1 + exp(-by)): with E = exp(-|by|), 1 / (1 + E) or E / (1 + E), whose divisor lies between 1 and 2: a reciprocal and one step
// on it.  18 instructions where expf and a division take 27.
__device__ __forceinline__ float logistic_times(float z, float by) {
    const float e = exp_minus(fabsf(by)), d = 1.0f + e;
    float r = __builtin_amdgcn_rcpf(d);
    r = fmaf(fmaf(-d, r, 1.0f), r, r);
    return (by < 0.0f ? z * e : z) * r;
}

// z Phi(z), Phi(-|z|) = 2^-(1 + |z| Q(|z|)): Q of degree 7 by weighted least squares for the largest error of z Phi(z) on [0, 6], its
// leading coefficient above zero, so that Phi goes to zero beyond.  12 instructions where erff's two branches take 45.
__device__ __forceinline__ float gelu_of(float z) {
    const float a = fabsf(z);
    float q = 2.834737415e-06f;
    q = fmaf(q, a, -3.937564543e-05f);
    q = fmaf(q, a, 1.861709025e-04f);
    q = fmaf(q, a, 1.369577512e-04f);
    q = fmaf(q, a, -7.063446101e-03f);
    q = fmaf(q, a, 5.249619484e-02f);
    q = fmaf(q, a, 4.592081904e-01f);
    q = fmaf(q, a, 1.151105165e+00f);
    const float e = __builtin_amdgcn_exp2f(fmaf(-q, a, -1.0f));
    return z * (z < 0.0f ? e : 1.0f - e);
}

// For results that stay float32 (`ROUNDED` false) by expf, erff and tanhf; for those that are rounded to bfloat16 by the short forms above, whose
// errors against 64 bits are between 0.8 and 1.4 of those (by a model of the arithmetic 1.6 for silu of numbers below zero alone; 2e-8 to 1e-7 in the mean square, on N(0, 0.02^2) to N(0, 20^2)), a ten-thousandth of the rounding's:
// the rounded results have the same mean square error to nine digits.
template <bool ROUNDED>
__device__ __forceinline__ float activate(float z, int act) {
    switch (act) {
        case ACT_SILU: return ROUNDED ? logistic_times(z, z) : z / (1.0f + expf(-z));
        case ACT_RELU: return fmaxf(z, 0.0f);
        case ACT_GELU: return ROUNDED ? gelu_of(z) : 0.5f * z * (1.0f + erff(z * 0.70710678118654752440f));
        case ACT_GELU_TANH: {
            const float u = 0.79788456080286535588f * (z + 0.044715f * z * z * z);
            return ROUNDED ? logistic_times(z, 2.0f * u) : 0.5f * z * (1.0f + tanhf(u));       // 1 + tanh u = 2 / (1 + exp(-2 u))
        }
        case ACT_RELU2: { const float r = fmaxf(z, 0.0f); return r * r; }
        default: return z;
    }
}

// The same of several values: one look at `act` for all of them.
template <bool ROUNDED, int N>
__device__ __forceinline__ void activate_all(float (&z)[N], int act) {
#define KIPP_ACT(A)                                              \
    case A:                                                      \
        _Pragma("unroll") for (int i = 0; i < N; ++i) z[i] = activate<ROUNDED>(z[i], A); \
        break
    switch (act) {
        KIPP_ACT(ACT_SILU);
        KIPP_ACT(ACT_RELU);
        KIPP_ACT(ACT_GELU);
        KIPP_ACT(ACT_GELU_TANH);
        KIPP_ACT(ACT_RELU2);
        default: break;
    }
#undef KIPP_ACT
}

// What the sort of a step's pairs reads and leaves.  tiles: int32 [max_tiles][3] = (expert, first row, rows); rows 0 marks an unused tile.
// `row_weight` (or null) receives every sorted row's weight.  Choices from `experts` on are identity experts: no row, place -1.
struct Sort {
    int pairs, experts, top;
    int32_t *pair_token, *place_of_pair, *tiles;
    int max_tiles, tile_rows;
    float* row_weight;
};

// One workgroup sorts all pairs.  PER > 0: no more than PER pairs a thread, which keeps them in registers, asked for together; a pair's place
// within its expert's run is what its count returned.  PER 0: any number.
template <int PER>
__device__ __forceinline__ void sort_pairs(const Sort& sort, const int32_t* chosen, const float* weight) {
    const int pairs = sort.pairs, experts = sort.experts, top = sort.top, max_tiles = sort.max_tiles, tile_rows = sort.tile_rows;
    int32_t *pair_token = sort.pair_token, *place_of_pair = sort.place_of_pair, *tiles = sort.tiles;
    float* row_weight = sort.row_weight;
    __shared__ int count[MAX_EXPERTS];
    __shared__ int first[MAX_EXPERTS + 1];
    __shared__ int tile_first[MAX_EXPERTS + 1];
    for (int e = threadIdx.x; e < experts; e += blockDim.x) count[e] = 0;
    __syncthreads();
    int own_e[PER > 0 ? PER : 1], own_place[PER > 0 ? PER : 1];         // (PER) this thread's pairs
    if (PER > 0) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int p = threadIdx.x + i * blockDim.x;
            own_e[i] = chosen[min(p, pairs - 1)];
            own_place[i] = 0;
            if (p >= pairs) own_e[i] = experts;
        }
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (own_e[i] < experts) own_place[i] = atomicAdd(&count[own_e[i]], 1);
    } else {
        for (int p = threadIdx.x; p < pairs; p += blockDim.x) {
            const int e = chosen[p];
            if (e < experts) atomicAdd(&count[e], 1);
        }
    }
    __syncthreads();
    if (threadIdx.x < KIPP_WAVE) {          // where every expert's rows and tiles begin: running sums over 64 experts at a time
        int rows = 0, tl = 0;
        for (int e0 = 0; e0 < experts; e0 += KIPP_WAVE) {
            const int e = e0 + threadIdx.x;
            const int n = e < experts ? count[e] : 0, mine = (n + tile_rows - 1) / tile_rows;
            int up_rows = n, up_tl = mine;
            for (int off = 1; off < KIPP_WAVE; off <<= 1) {
                const int r = __shfl_up(up_rows, off, KIPP_WAVE), t = __shfl_up(up_tl, off, KIPP_WAVE);
                if ((int)threadIdx.x >= off) {
                    up_rows += r;
                    up_tl += t;
                }
            }
            if (e < experts) {
                first[e] = rows + up_rows - n;
                tile_first[e] = tl + up_tl - mine;
            }
            rows += __shfl(up_rows, KIPP_WAVE - 1, KIPP_WAVE);
            tl += __shfl(up_tl, KIPP_WAVE - 1, KIPP_WAVE);
        }
        if (threadIdx.x == 0) {
            first[experts] = rows;
            tile_first[experts] = tl;
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < experts; e += blockDim.x) {
        const int n = count[e], parts = (n + tile_rows - 1) / tile_rows;
        // whole tiles: an expert's rows shared out evenly.  The walk multiplies 64s; tiles of 128 are shared out in 32s, which keep two tiles of
        // an expert alike (in 64s 241 steps took the same in the mean, two experts of 130 rows each 8 % more)
        const int grain = tile_rows == MANY_ROWS ? 64 : 32;
        const int each = tile_rows >= MFMA_ROWS && parts > 0 ? ((n + parts - 1) / parts + grain - 1) / grain * grain : tile_rows;
        for (int j = 0; j < parts; ++j) {
            int32_t* tile = tiles + (size_t)(tile_first[e] + j) * 3;
            tile[0] = e;
            tile[1] = first[e] + j * each;
            tile[2] = min(each, n - j * each);
        }
    }
    for (int i = tile_first[experts] + threadIdx.x; i < max_tiles; i += blockDim.x) {
        tiles[(size_t)i * 3] = 0;
        tiles[(size_t)i * 3 + 1] = 0;
        tiles[(size_t)i * 3 + 2] = 0;
    }
    if (PER > 0) {
        float w[PER > 0 ? PER : 1];
#pragma unroll
        for (int i = 0; i < PER; ++i) w[i] = row_weight != nullptr ? weight[min((int)(threadIdx.x + i * blockDim.x), pairs - 1)] : 0.0f;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int p = threadIdx.x + i * blockDim.x;
            if (p >= pairs) break;
            const int at = own_e[i] < experts ? first[own_e[i]] + own_place[i] : -1;
            place_of_pair[p] = at;
            if (at < 0) continue;
            pair_token[at] = p / top;
            if (row_weight != nullptr) row_weight[at] = w[i];
        }
        return;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < experts; e += blockDim.x) count[e] = 0;     // now the next free place of a run
    __syncthreads();
    for (int p = threadIdx.x; p < pairs; p += blockDim.x) {
        const int e = chosen[p];
        if (e >= experts) {
            place_of_pair[p] = -1;
            continue;
        }
        const int at = first[e] + atomicAdd(&count[e], 1);
        pair_token[at] = p / top;
        place_of_pair[p] = at;
        if (row_weight != nullptr) row_weight[at] = weight[p];
    }
}

template <int PER>
__global__ void __launch_bounds__(SORT_THREADS) moe_sort_kernel(Sort sort, const int32_t* chosen, const float* weight) { sort_pairs<PER>(sort, chosen, weight); }

// The sum of a number's slabs in order, four asked for at once.
__device__ __forceinline__ float sum_of_slabs(const float* __restrict__ z, int parts, size_t part_stride) {
    float v = z[0];
    for (int q0 = 1; q0 < parts; q0 += 4) {
        float more[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) more[i] = z[min(q0 + i, parts - 1) * part_stride];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (q0 + i < parts) v += more[i];
    }
    return v;
}

// Few tokens (one workgroup's) are chosen for and sorted in one launch (`SORT`): one token's four of 32 experts 4.3 us by the sigmoid, 5.6 by the softmax.
#define ROUTE_SORT_TOKENS 16        // a wave each
// Choices by rank cost a step an expert (up to 64), one after the other a tree of exchanges each.  17 tokens, us, by trees / by rank: one of 32 experts 5.6 / 5.9,
// four 7.1 / 6.0, one of 64 5.5 / 6.7, two 6.1 / 6.7, eight 9.6 / 6.9.  A build each.
#define RANK_EXPERTS 24
// One wave a token, a lane REGS of the experts.  z: float32 [tokens][stride] (or slabs of it, added in order).
template <int REGS, int WAVES, bool SORT>
__global__ void __launch_bounds__(WAVES * KIPP_WAVE)
moe_route_kernel(const float* __restrict__ z, int parts, size_t part_stride, int stride, int32_t* chosen,
                 float* weight, int tokens, int experts, int top, float eps, Sort sort) {
    const int wave = threadIdx.x / KIPP_WAVE, lane = threadIdx.x & (KIPP_WAVE - 1);
    int t = blockIdx.x * WAVES + wave;
    const bool live = t < tokens;
    if (!live) t = tokens - 1;
    float p[REGS];
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < REGS; ++i) {
        const int e = lane + i * KIPP_WAVE;
        float v = -INFINITY;
        if (e < experts) {
            v = sum_of_slabs(z + (size_t)t * stride + e, parts, part_stride);
        }
        p[i] = v;
        m = fmaxf(m, v);
    }
    m = wave_max(m);
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < REGS; ++i) {
        p[i] = (lane + i * KIPP_WAVE < experts) ? expf(p[i] - m) : -1.0f;
        if (p[i] > 0.0f) sum += p[i];
    }
    sum = wave_sum(sum);
    float picked_sum = 0.0f;
    float mine = 0.0f;          // lane j keeps the j-th choice
    int mine_e = 0;
    for (int j = 0; j < top; ++j) {
        float best = -1.0f;
        int best_e = MAX_EXPERTS;
#pragma unroll
        for (int i = 0; i < REGS; ++i)
            if (p[i] > best) { best = p[i]; best_e = lane + i * KIPP_WAVE; }     // the lowest index of a lane's largest
        for (int off = 32; off > 0; off >>= 1) {
            const float ob = __shfl_xor(best, off, KIPP_WAVE);
            const int oe = __shfl_xor(best_e, off, KIPP_WAVE);
            if (ob > best || (ob == best && oe < best_e)) { best = ob; best_e = oe; }
        }
#pragma unroll
        for (int i = 0; i < REGS; ++i)
            if (lane + i * KIPP_WAVE == best_e) p[i] = -1.0f;
        const float s = best / sum;
        picked_sum += s;
        if (lane == j) { mine = s; mine_e = best_e; }
    }
    __shared__ int32_t chosen_s[SORT ? WAVES * MAX_TOP : 1];
    __shared__ float weight_s[SORT ? WAVES * MAX_TOP : 1];
    if (live && lane < top) {
        const float w = mine / (picked_sum + eps);
        chosen[(size_t)t * top + lane] = mine_e;
        weight[(size_t)t * top + lane] = w;
        if (SORT) {
            chosen_s[t * top + lane] = mine_e;
            weight_s[t * top + lane] = w;
        }
    }
    if (SORT) sort_pairs<1>(sort, chosen_s, weight_s);
}

// One wave a token: sigmoid scores (`softmax`: a softmax over all of them), a correction for the choice alone, groups of
// neighbouring experts of which the best stay (by the sum of their two largest, or, `by_largest`, by their largest).
template <int REGS, int WAVES, bool SORT, bool BY_RANK>
__global__ void __launch_bounds__(WAVES * KIPP_WAVE)
moe_route_grouped_kernel(const float* __restrict__ z, int parts, size_t part_stride, int stride, const float* __restrict__ correction,
                         int32_t* chosen, float* weight, int tokens, int experts, int top, float eps,
                         int group_count, int group_keep, float scale, int renormalize, int softmax, int by_largest, Sort sort) {
    __shared__ float c_s[WAVES][REGS * KIPP_WAVE];     // choice scores, then -inf for experts of groups that do not stay
    __shared__ float g_s[WAVES][REGS * KIPP_WAVE];     // group scores, -inf once a group is taken
    const int wave = threadIdx.x / KIPP_WAVE, lane = threadIdx.x & (KIPP_WAVE - 1);
    int t = blockIdx.x * WAVES + wave;
    const bool live = t < tokens;
    if (!live) t = tokens - 1;      // stay in step with the barriers
    const int size = experts / group_count;
    float s[REGS], correct[REGS];
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < REGS; ++i) correct[i] = correction != nullptr ? correction[min(lane + i * KIPP_WAVE, experts - 1)] : 0.0f;
#pragma unroll
    for (int i = 0; i < REGS; ++i) {
        const int e = lane + i * KIPP_WAVE;
        s[i] = 0.0f;
        if (e < experts) {
            const float v = sum_of_slabs(z + (size_t)t * stride + e, parts, part_stride);
            s[i] = softmax ? v : 1.0f / (1.0f + expf(-v));
            m = fmaxf(m, v);
        }
    }
    if (softmax) {
        m = wave_max(m);
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < REGS; ++i)
            if (lane + i * KIPP_WAVE < experts) {
                s[i] = expf(s[i] - m);
                sum += s[i];
            }
        sum = wave_sum(sum);
#pragma unroll
        for (int i = 0; i < REGS; ++i) s[i] = s[i] / sum;
    }
#pragma unroll
    for (int i = 0; i < REGS; ++i) {
        const int e = lane + i * KIPP_WAVE;
        if (e < experts) c_s[wave][e] = s[i] + correct[i];
    }
    __syncthreads();
    if (group_keep < group_count) {
        for (int g = lane; g < group_count; g += KIPP_WAVE) {
            float a = -INFINITY, b = -INFINITY;      // the two largest of the group
            for (int j = 0; j < size; ++j) {
                const float v = c_s[wave][g * size + j];
                if (v > a) { b = a; a = v; } else if (v > b) { b = v; }
            }
            g_s[wave][g] = size > 1 && !by_largest ? a + b : a;
        }
        __syncthreads();
        if (group_count <= KIPP_WAVE) {
            // a lane a group: it stays if fewer than `keep` groups come before it (a larger score, or as large with a lower index)
            const float mine_g = lane < group_count ? g_s[wave][lane] : 0.0f;
            int before = 0;
            for (int g = 0; g < group_count; ++g) {
                const float v = g_s[wave][g];
                before += v > mine_g || (v == mine_g && g < lane) ? 1 : 0;
            }
            __syncthreads();
            if (lane < group_count && before < group_keep) g_s[wave][lane] = -INFINITY;         // taken: it stays
            __syncthreads();
        } else {
            for (int round = 0; round < group_keep; ++round) {
                float best = -INFINITY;
                int best_g = MAX_EXPERTS;
                for (int g = lane; g < group_count; g += KIPP_WAVE) {
                    const float v = g_s[wave][g];
                    if (v > best || (best_g == MAX_EXPERTS && v != -INFINITY)) { best = v; best_g = g; }
                }
                for (int off = 32; off > 0; off >>= 1) {
                    const float ob = __shfl_xor(best, off, KIPP_WAVE);
                    const int og = __shfl_xor(best_g, off, KIPP_WAVE);
                    if (og != MAX_EXPERTS && (best_g == MAX_EXPERTS || ob > best || (ob == best && og < best_g))) { best = ob; best_g = og; }
                }
                __syncthreads();
                if (lane == 0 && best_g != MAX_EXPERTS) g_s[wave][best_g] = -INFINITY;      // taken: it stays
                __syncthreads();
            }
        }
        for (int e = lane; e < experts; e += KIPP_WAVE)
            if (g_s[wave][e / size] != -INFINITY) c_s[wave][e] = -INFINITY;             // its group was not taken
        __syncthreads();
    }
    __shared__ int32_t chosen_s[WAVES * MAX_TOP];
    __shared__ float weight_s[WAVES * MAX_TOP];
    float picked_sum = 0.0f, mine = 0.0f;       // lane j keeps the j-th choice
    int mine_e = 0;
    if constexpr (BY_RANK) {
        static_assert(REGS == 1, "a lane an expert");
        // a lane an expert: its place is the number of experts ahead of it (a larger score, or as large with a lower index)
        const float own = lane < experts ? c_s[wave][lane] : -INFINITY;
        int ahead = 0;
        for (int e = 0; e < experts; ++e) {
            const float v = c_s[wave][e];
            ahead += v > own || (v == own && e < lane) ? 1 : 0;
        }
        if (lane < top) {
            chosen_s[wave * top + lane] = 0;        // (where fewer can be chosen)
            weight_s[wave * top + lane] = 0.0f;
        }
        __syncthreads();
        if (own > -INFINITY && ahead < top) {
            chosen_s[wave * top + ahead] = lane;
            weight_s[wave * top + ahead] = s[0];
        }
        __syncthreads();
        for (int j = 0; j < top; ++j) picked_sum += weight_s[wave * top + j];
        if (lane < top) {
            mine = weight_s[wave * top + lane];
            mine_e = chosen_s[wave * top + lane];
        }
        __syncthreads();
    } else {
        float c[REGS];
#pragma unroll
        for (int i = 0; i < REGS; ++i) {
            const int e = lane + i * KIPP_WAVE;
            c[i] = e < experts ? c_s[wave][e] : -INFINITY;
        }
        for (int j = 0; j < top; ++j) {
            float best = -INFINITY, best_s = 0.0f;
            int best_e = MAX_EXPERTS;
#pragma unroll
            for (int i = 0; i < REGS; ++i)
                if (c[i] > best) { best = c[i]; best_e = lane + i * KIPP_WAVE; best_s = s[i]; }     // the lowest index of a lane's largest
            for (int off = 32; off > 0; off >>= 1) {
                const float ob = __shfl_xor(best, off, KIPP_WAVE), os = __shfl_xor(best_s, off, KIPP_WAVE);
                const int oe = __shfl_xor(best_e, off, KIPP_WAVE);
                if (ob > best || (ob == best && oe < best_e)) { best = ob; best_e = oe; best_s = os; }
            }
#pragma unroll
            for (int i = 0; i < REGS; ++i)
                if (lane + i * KIPP_WAVE == best_e) c[i] = -INFINITY;
            picked_sum += best_s;
            if (lane == j) { mine = best_s; mine_e = best_e < experts ? best_e : 0; }
        }
    }
    if (live && lane < top) {
        const float w = renormalize ? mine / (picked_sum + eps) * scale : mine * scale;
        chosen[(size_t)t * top + lane] = mine_e;
        weight[(size_t)t * top + lane] = w;
        if (SORT) {
            chosen_s[t * top + lane] = mine_e;
            weight_s[t * top + lane] = w;
        }
    }
    if (SORT) sort_pairs<1>(sort, chosen_s, weight_s);
}

// x rows are x[gather[row]] (gather null: x[row]); w: [experts][n_out][k]; out[row][n_out].  GLU: w is [experts][2 n_out][k] =
// [gate; up], `row_weight` (or null: one) a row's weight.
template <typename TX, typename TW, typename TO, bool GLU>
__global__ void __launch_bounds__(EXPERT_COLS)
moe_expert_kernel(const TX* __restrict__ x, const int32_t* __restrict__ gather, const float* __restrict__ row_weight,
                  const TW* __restrict__ w, const int32_t* __restrict__ tiles, TO* __restrict__ out, int n_out, int k, int act) {
    __shared__ float x_s[TILE_ROWS][EXPERT_KC];
    const int32_t* tile = tiles + (size_t)blockIdx.x * 3;
    const int rows = tile[2];
    if (rows == 0) return;      // uniform over the workgroup
    const int expert = tile[0], row0 = tile[1];
    const int col = blockIdx.y * EXPERT_COLS + threadIdx.x;
    const TW* w_row = w + ((size_t)expert * (GLU ? 2 : 1) * n_out + (col < n_out ? col : 0)) * k;
    const TW* up_row = w_row + (size_t)n_out * k;
    float acc[TILE_ROWS], up[GLU ? TILE_ROWS : 1];
#pragma unroll
    for (int r = 0; r < TILE_ROWS; ++r) {
        acc[r] = 0.0f;
        if (GLU) up[r] = 0.0f;
    }
    for (int k0 = 0; k0 < k; k0 += EXPERT_KC) {
        const int kc = min(EXPERT_KC, k - k0);
        __syncthreads();
        for (int i = threadIdx.x; i < TILE_ROWS * EXPERT_KC; i += EXPERT_COLS) {
            const int r = i / EXPERT_KC, e = i - r * EXPERT_KC;
            float v = 0.0f;
            if (r < rows && e < kc) {
                const size_t src_row = gather != nullptr ? (size_t)gather[row0 + r] : (size_t)(row0 + r);
                v = load_f(x + src_row * k, k0 + e);
            }
            x_s[r][e] = v;
        }
        __syncthreads();
        if (col < n_out) {
            for (int e = 0; e < kc; ++e) {
                const float wv = load_f(w_row, k0 + e);
#pragma unroll
                for (int r = 0; r < TILE_ROWS; ++r) acc[r] = fmaf(wv, x_s[r][e], acc[r]);
                if (GLU) {
                    const float uv = load_f(up_row, k0 + e);
#pragma unroll
                    for (int r = 0; r < TILE_ROWS; ++r) up[r] = fmaf(uv, x_s[r][e], up[r]);
                }
            }
        }
    }
    if (col >= n_out) return;
#pragma unroll
    for (int r = 0; r < TILE_ROWS; ++r)
        if (r < rows) {
            float y;
            if (GLU) {
                const float s = row_weight != nullptr ? row_weight[row0 + r] : 1.0f;
                y = activate<sizeof(TO) == 2>(s * acc[r], act) * (s * up[r]);
            } else {
                y = activate<sizeof(TO) == 2>(acc[r], act);
            }
            store_f(out + (size_t)(row0 + r) * n_out, col, y);
        }
}

// The same on the matrix cores: bfloat16 x and w, K a multiple of 32, tiles of up to MFMA_ROWS rows, a workgroup 128 columns,
// K staged through registers and LDS 64 numbers a step.  A 16 x 16 x 32
// product takes, from lane l, 8 numbers of row l % 16 at k = 8 (l / 16) .. + 7 of either operand, and leaves
// C[4 (l / 16) + v][l % 16] in its register v.
typedef __attribute__((ext_vector_type(4))) float f32x4;

template <typename TO, bool GLU>
__global__ void __launch_bounds__(MFMA_THREADS)
moe_expert_mfma_kernel(const bf16_t* __restrict__ x, const int32_t* __restrict__ gather, const float* __restrict__ row_weight,
                       const bf16_t* __restrict__ w, const int32_t* __restrict__ tiles, TO* __restrict__ out, int n_out, int k, int act) {
    // 64 numbers of k of every row of the tile and of every column of the workgroup, a row 144 bytes apart from the next
    // (the fragments' reads of 16 bytes a lane then spread over the banks)
    __shared__ __attribute__((aligned(16))) bf16_t a_s[MFMA_ROWS * MFMA_PITCH];
    __shared__ __attribute__((aligned(16))) bf16_t b_s[MFMA_COLS * MFMA_PITCH];
    // Workgroups go to the chip's 8 dies in turn, each with an L2 of its own: the launch's workgroups are renumbered so
    // that a die works on neighbouring tiles at a time, which are mostly row tiles of one expert and read the same
    // columns of its matrix.
    const unsigned launched = blockIdx.x + blockIdx.y * gridDim.x, total = gridDim.x * gridDim.y;
    const unsigned die = launched % XCDS, turn = launched / XCDS, each = total / XCDS, more = total % XCDS;
    const unsigned item = (die < more ? die * (each + 1) : more * (each + 1) + (die - more) * each) + turn;
    const int32_t* tile = tiles + (size_t)(item % gridDim.x) * 3;
    const int rows = tile[2];
    if (rows == 0) return;      // uniform over the workgroup
    const int expert = tile[0], row0 = tile[1];
    const int tid = threadIdx.x;
    const int wave = tid / KIPP_WAVE, lane = tid & (KIPP_WAVE - 1), l16 = lane & 15, h = lane >> 4;
    const int col_base = (item / gridDim.x) * (GLU ? MFMA_COLS / 2 : MFMA_COLS);
    const int mfrags = (rows + 15) >> 4;
    // from memory, 8 threads take the 128 bytes of a row's step: thread t rows t / 8 + 32 i, bytes 16 (t % 8) ..
    const int ld_row = tid >> 3, ld_ch = tid & 7;
    // where a lane's rows begin, in numbers from x and from the expert's matrix (the launcher has checked that 32 bits hold them)
    unsigned a_src[MFMA_ROWS / 32], b_src[MFMA_COLS / 32];
    const bf16_t* w_e = w + (size_t)expert * (GLU ? 2 : 1) * n_out * k;
#pragma unroll
    for (int i = 0; i < MFMA_ROWS / 32; ++i) {
        const int r = min(ld_row + 32 * i, rows - 1);       // rows beyond the tile's read its last one and are not stored
        const unsigned src = gather != nullptr ? (unsigned)gather[row0 + r] : (unsigned)(row0 + r);
        a_src[i] = src * (unsigned)k + 8 * ld_ch;
    }
#pragma unroll
    for (int i = 0; i < MFMA_COLS / 32; ++i) {
        const int at = ld_row + 32 * i;         // the staged column: a wave's 32 are 16 of the gate's, then 16 of the up's
        const int c = GLU ? min(col_base + 16 * (at >> 5) + (at & 15), n_out - 1) + (at & 16 ? n_out : 0) : min(col_base + at, n_out - 1);
        b_src[i] = (unsigned)c * (unsigned)k + 8 * ld_ch;
    }
    u32x4 a_r[MFMA_ROWS / 32], b_r[MFMA_COLS / 32];
    const u32x4 zero = (u32x4){0u, 0u, 0u, 0u};
    auto fetch = [&](int k0) {
        const bool there = k0 + 8 * ld_ch < k;              // k is a multiple of 32: the last step may be half a step
#pragma unroll
        for (int i = 0; i < MFMA_ROWS / 32; ++i)
            if (32 * i < 16 * mfrags) a_r[i] = there ? *(const u32x4*)(x + a_src[i] + k0) : zero;
#pragma unroll
        for (int i = 0; i < MFMA_COLS / 32; ++i) b_r[i] = there ? *(const u32x4*)(w_e + b_src[i] + k0) : zero;
    };
    f32x4 acc[MFMA_ROWS / 16][MFMA_NF];
#pragma unroll
    for (int i = 0; i < MFMA_ROWS / 16; ++i)
#pragma unroll
        for (int j = 0; j < MFMA_NF; ++j) acc[i][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    fetch(0);
    for (int k0 = 0; k0 < k; k0 += MFMA_KC) {
        __syncthreads();        // the step before has been multiplied
#pragma unroll
        for (int i = 0; i < MFMA_ROWS / 32; ++i)
            if (32 * i < 16 * mfrags) *(u32x4*)(a_s + (ld_row + 32 * i) * MFMA_PITCH + 8 * ld_ch) = a_r[i];
#pragma unroll
        for (int i = 0; i < MFMA_COLS / 32; ++i) *(u32x4*)(b_s + (ld_row + 32 * i) * MFMA_PITCH + 8 * ld_ch) = b_r[i];
        __syncthreads();
        if (k0 + MFMA_KC < k) fetch(k0 + MFMA_KC);      // on its way while this step is multiplied
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            Frag b[MFMA_NF];
#pragma unroll
            for (int j = 0; j < MFMA_NF; ++j) b[j].u = *(const u32x4*)(b_s + (wave * 16 * MFMA_NF + 16 * j + l16) * MFMA_PITCH + 32 * half + 8 * h);
            if (mfrags == MFMA_ROWS / 16) {          // a whole tile: nothing to ask between the fragments
#pragma unroll
                for (int i = 0; i < MFMA_ROWS / 16; ++i) {
                    Frag a;
                    a.u = *(const u32x4*)(a_s + (16 * i + l16) * MFMA_PITCH + 32 * half + 8 * h);
#pragma unroll
                    for (int j = 0; j < MFMA_NF; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b[j].v, acc[i][j], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int i = 0; i < MFMA_ROWS / 16 - 1; ++i) {
                    if (i < mfrags) {
                        Frag a;
                        a.u = *(const u32x4*)(a_s + (16 * i + l16) * MFMA_PITCH + 32 * half + 8 * h);
#pragma unroll
                        for (int j = 0; j < MFMA_NF; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b[j].v, acc[i][j], 0, 0, 0);
                    }
                }
            }
        }
    }
    if (GLU) {
        const int c = col_base + wave * 16 + l16;
#pragma unroll
        for (int i = 0; i < MFMA_ROWS / 16; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = 16 * i + 4 * h + v;
                if (r < rows && c < n_out) {
                    const float s = row_weight != nullptr ? row_weight[row0 + r] : 1.0f;
                    store_f(out + (size_t)(row0 + r) * n_out, c, activate<sizeof(TO) == 2>(s * acc[i][0][v], act) * (s * acc[i][1][v]));
                }
            }
        return;
    }
    const int col0 = col_base + wave * 16 * MFMA_NF;
#pragma unroll
    for (int i = 0; i < MFMA_ROWS / 16; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = 16 * i + 4 * h + v;
            if (r < rows) {
                TO* dst = out + (size_t)(row0 + r) * n_out;
#pragma unroll
                for (int j = 0; j < MFMA_NF; ++j) {
                    const int c = col0 + 16 * j + l16;
                    if (c < n_out) store_f(dst, c, activate<sizeof(TO) == 2>(acc[i][j][v], act));
                }
            }
        }
}

// The same by the walk of the products for prompt portions (`line_walk.h`), its rows of x taken through `gather`: eight waves take a tile's rows
// (up to 64 XF) and 128 WF rows of the expert's matrix (GLU: 64 WF of the gate's and the 64 WF of the up's that belong to them), two waves down and four
// across.  Bound by the experts' matrices, which arrive at 4.9 to 5.5 TB/s where an expert has up to 100 rows, and by whole rounds of
// workgroups.  32 experts, [gate; up] of 2 x 2,432 x 2,560, one such matrix, and back, us: the staged kernel or a walk in steps of half
// lines with tiles of 128 or 256, the best of them / now: 416 rows 161 / 148, 104 / 84, 94 / 82; 2,048 rows 195 / 154, 130 / 91, 119 / 89;
// 4,000 rows 225 / 175, 149 / 108, 132 / 106; 8,192 rows 345 / 264, 203 / 149, 176 / 143; 128 experts of 768, 3,968 rows 201 / 178, 124 / 94, 127 / 114.
template <typename TO, bool GLU, int XF, int WF>
__device__ __forceinline__ void expert_tile(const bf16_t* __restrict__ x, const int32_t* __restrict__ gather, const float* __restrict__ row_weight,
                                            const bf16_t* __restrict__ w_e, TO* __restrict__ out, int row0, int rows, int col0, int n_out, int k,
                                            int act, unsigned char* lds) {
    using Walk = LineWalk<XF, WF, 2, TILE_ACROSS>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, quarter = lane >> 4, across = wave % TILE_ACROSS, first = 32 * XF * (wave / TILE_ACROSS);     // this wave's columns and rows
    // a lane's rows begin at 32-bit offsets from x and from the expert's matrix (the launcher has checked that they fit)
    uint32_t x_src[2][Walk::X_MOST], w_src[2][Walk::W_MOST];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int n = 0; n < Walk::X_MOST; ++n) {
            const int p = Walk::x_row(n, wave, lane), r = row0 + min(Walk::x_tile_row(h, p), rows - 1);     // rows beyond the tile's read its last one and are not stored
            x_src[h][n] = (uint32_t)(((size_t)(gather != nullptr ? gather[r] : r) * k + line_col(lane, p, k / BK)) * 2);
        }
#pragma unroll
        for (int n = 0; n < Walk::W_MOST; ++n) {
            const int p = Walk::w_row(n, wave, lane);       // of the half; 16 WF of either half a wave multiplies: under GLU the gate's and the up's
            const int wr = GLU ? min(col0 + p, n_out - 1) + h * n_out : min(col0 + Walk::w_tile_row(h, p), n_out - 1);
            w_src[h][n] = (uint32_t)(((size_t)wr * k + line_col(lane, p, k / BK)) * 2);
        }
    }
    f32x4 acc[2 * XF][2 * WF];
    line_walk<XF, WF, 2, TILE_ACROSS>(lds, lane, wave, (const unsigned char*)x, (const unsigned char*)w_e, x_src, w_src, k / BK, acc);
    // Of fragment (i, j) a lane holds row l16 and columns 16 j + 4 quarter .. + 3.  Sums that are stored as they are go straight from there.
    if constexpr (!GLU && sizeof(TO) == 4) {
        if (act == ACT_NONE && (n_out & 7) == 0) {
#pragma unroll
            for (int i = 0; i < 2 * XF; ++i) {
                const int r = first + 16 * i + l16;
                if (r >= rows) continue;
#pragma unroll
                for (int j = 0; j < 2 * WF; ++j) {
                    const int c = col0 + 32 * WF * across + 16 * j + 4 * quarter;
                    if (c < n_out) *(f32x4*)(out + (size_t)(row0 + r) * n_out + c) = acc[i][j];
                }
            }
            return;
        }
    }
    // (Of an item's 70 us at 256 rows this end took 25 with erff, and takes 10.)  Others: 32 rows at a time go through the wave's own
    // corner of LDS (now free) as they are; a lane then takes 8 neighbouring columns of a row, activates and stores them (the
    // activations written out for every accumulator register were hundreds of KB of code that ran once).
    constexpr int WCOLS = (GLU ? 16 : 32) * WF, PITCH = 32 * WF + 4, LANES_PER_ROW = WCOLS / 8, ROWS_PER_PASS = 64 / LANES_PER_ROW;
    static_assert(32 * PITCH * 4 * Walk::WAVES <= Walk::LDS_BYTES, "a wave's staging fits its share of LDS");
    __syncthreads();                                               // every wave is done reading operands
    float* stage = (float*)lds + wave * 32 * PITCH;
    const int c_in = (lane % LANES_PER_ROW) * 8, c = col0 + WCOLS * across + c_in;
#pragma unroll
    for (int i = 0; i < XF; ++i) {
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int j = 0; j < 2 * WF; ++j) *(f32x4*)(stage + (16 * f + l16) * PITCH + 16 * j + 4 * quarter) = acc[2 * i + f][j];
        __builtin_amdgcn_s_waitcnt(0xC07F);                        // lgkmcnt(0): what the wave wrote it reads back
        __builtin_amdgcn_wave_barrier();
#pragma unroll 1
        for (int r = lane / LANES_PER_ROW; r < 32; r += ROWS_PER_PASS) {
            if (first + 32 * i + r >= rows || c >= n_out) continue;
            const float* at = stage + r * PITCH + c_in;
            float y[8], u[8];
#pragma unroll
            for (int q = 0; q < 8; q += 4) {
                *(f32x4*)(y + q) = *(const f32x4*)(at + q);
                if (GLU) *(f32x4*)(u + q) = *(const f32x4*)(at + 16 * WF + q);
            }
            const float s = GLU && row_weight != nullptr ? row_weight[row0 + first + 32 * i + r] : 1.0f;
#pragma unroll
            for (int q = 0; q < 8; ++q) y[q] = GLU ? s * y[q] : y[q];
            activate_all<sizeof(TO) == 2>(y, act);
            if (GLU) {
#pragma unroll
                for (int q = 0; q < 8; ++q) y[q] *= s * u[q];
            }
            TO* dst = out + (size_t)(row0 + first + 32 * i + r) * n_out + c;
            if (c + 8 <= n_out && (n_out & 7) == 0) {
                if constexpr (sizeof(TO) == 4) {
                    *(f32x4*)dst = *(const f32x4*)y;
                    *(f32x4*)(dst + 4) = *(const f32x4*)(y + 4);
                } else {
                    u32x4 packed;
#pragma unroll
                    for (int q = 0; q < 4; ++q) packed[q] = (uint32_t)f32_to_bf16(y[2 * q]) | ((uint32_t)f32_to_bf16(y[2 * q + 1]) << 16);
                    *(u32x4*)dst = packed;
                }
            } else {
                for (int q = 0; q < 8; ++q)
                    if (c + q < n_out) store_f(dst, q, y[q]);
            }
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_s_waitcnt(0xC07F);                        // the reads are done before the next 32 rows overwrite them
    }
}

// FEW: tiles of up to 64 rows alone.  Their 80 KB of LDS (128 KB where tiles of 256 may come) and 128 registers let two workgroups share a compute unit, one's
// start and end beside the other's walk: 256 experts of 2 rows each, gated 704 x 384 43 us, alone on a compute unit 59 (the staged kernel 48); 2,048 x 256 of
// 12 rows 55, 78 (71); 6,400 x 64 gated of 2 153, 226 (152); 102 such products of K from 32 to 1,024: 0.83 of the time in the mean.
template <typename TO, bool GLU, bool FEW>
__global__ void __launch_bounds__(512, FEW ? 4 : 2)
moe_expert_tiles_kernel(const bf16_t* __restrict__ x, const int32_t* __restrict__ gather, const float* __restrict__ row_weight,
                        const bf16_t* __restrict__ w, const int32_t* __restrict__ tiles, int max_tiles, int col_tiles, TO* __restrict__ out,
                        int n_out, int k, int act) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    constexpr int PLACES = DIE_UNITS * (FEW ? 2 : 1);       // of a die
    // Workgroups id, id + 8, .. run on one die of the chip, each with an L2 of its own: a die takes a run of (tiles of one expert that lie side by
    // side in the list, columns), those tiles fastest, so that workgroups which need the same rows of w walk over them at the same time.  (The sort
    // lists an expert's tiles side by side and the used ones first; any other order is as right.)
    const int lane = threadIdx.x & 63;
    int used = 0;                                       // up to the last tile with rows
    for (int at = 0; at < max_tiles; at += KIPP_WAVE) {
        const unsigned long long some = __ballot(at + lane < max_tiles && tiles[(size_t)(at + lane) * 3 + 2] > 0);
        if (some != 0) used = at + KIPP_WAVE - __clzll((long long)some);
    }
    const int items = used * col_tiles, per_die = (items + XCDS - 1) / XCDS, die = blockIdx.x % XCDS, turn = blockIdx.x / XCDS;
    // What a die has beyond whole rounds of its compute units goes in halves of the columns where those take one round of half the time
    // (7,204 rows of the experts above, 608 whole ones in three rounds / 512 and 192 halves: 238 and 223 us)
    const int mine = min(per_die, items - die * per_die), whole = mine / PLACES * PLACES, rest = mine - whole;
    const bool halved = turn >= whole && 2 * rest <= PLACES;
    const int at_die = halved ? whole + (turn - whole) / 2 : turn, half = halved ? (turn - whole) & 1 : 0;
    if (at_die >= mine) return;                         // uniform over the workgroup
    const int item = die * per_die + at_die;
    const int one = item / col_tiles, expert = __builtin_amdgcn_readfirstlane(tiles[(size_t)one * 3]);       // a tile of this item's expert
    int begin = 0, end = used;                          // the tiles of that expert which lie side by side with it
    for (int at = 0; at < used; at += KIPP_WAVE) {
        const unsigned long long others = __ballot(at + lane < used && tiles[(size_t)(at + lane) * 3] != expert);
        const unsigned long long ahead = one - at >= KIPP_WAVE ? others : (one > at ? others & ((1ull << (one - at)) - 1) : 0), behind = others ^ ahead;
        if (ahead != 0) begin = at + KIPP_WAVE - __clzll((long long)ahead);
        if (behind != 0 && end == used) end = at + __ffsll((long long)behind) - 1;
    }
    const int beside = end - begin, within = item - begin * col_tiles;
    const int32_t* tile = tiles + (size_t)(begin + within % beside) * 3;
    const int row0 = __builtin_amdgcn_readfirstlane(tile[1]), rows = __builtin_amdgcn_readfirstlane(tile[2]);
    const int col0 = within / beside * TILE_COLS(GLU) + half * TILE_COLS(GLU) / 2;
    if (col0 >= n_out) return;                          // the last columns may fill less than half a tile
    const bf16_t* w_e = w + (size_t)expert * (GLU ? 2 : 1) * n_out * k;
    // a wave's fragments: as many as the tile's rows ask for
#define KIPP_ET(N)                                                                                                                     \
    case N:                                                                                                                            \
        if (halved) expert_tile<TO, GLU, N, 1>(x, gather, row_weight, w_e, out, row0, rows, col0, n_out, k, act, lds);                  \
        else expert_tile<TO, GLU, N, 2>(x, gather, row_weight, w_e, out, row0, rows, col0, n_out, k, act, lds);                          \
        break
    if constexpr (FEW) {
        switch ((rows + 63) / 64) { KIPP_ET(1); }
        return;
    }
    switch ((rows + 63) / 64) {
        KIPP_ET(1);
        KIPP_ET(2);
        KIPP_ET(3);
        KIPP_ET(4);
    }
#undef KIPP_ET
}

// Tiles of few rows (single tokens): a workgroup (16 columns, tile), its waves a share of K each, the matrix straight from memory into the
// products' operands, 128 bytes a row and wave at a time; the waves' sums are added in order through LDS.  Bound by the read of the
// experts' matrices: four experts' [gate; up] of 2 x 2,432 x 2,560 (100 MB) 22.9 us, twelve's 54.7 (5.5 TB/s); four experts' 2,560 x
// 2,432 (50 MB) 11.1 us.  The kernel for whole tiles above stages 64 numbers of k a step behind two barriers with a workgroup for 128
// columns: 80 workgroups that walk 38 steps took 44 us for those 50 MB.  One step of 64 numbers ahead for two matrices, two for one: more
// of them in registers were slower (five: 25.4, 67.8 and 12.7 us), and so were four waves for two matrices.
template <typename TO, bool GLU, int MT>
__device__ __forceinline__ void expert_rows(const bf16_t* __restrict__ x, const int32_t* __restrict__ gather, const float* __restrict__ row_weight,
                                            const bf16_t* __restrict__ w_row, TO* __restrict__ out, int row0, int rows, int n0, int n_out, int k,
                                            int act, float (*part_s)[GLU ? 2 : 1][KIPP_WAVE][4]) {
    constexpr int NW = GLU ? 2 : 1, STEP = 64, AHEAD = GLU || MT > 2 ? 1 : 2;
    const int wave = threadIdx.x / KIPP_WAVE, lane = threadIdx.x & (KIPP_WAVE - 1), l16 = lane & 15, h8 = 8 * (lane >> 4);
    const bf16_t* x_row[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int r = row0 + min(16 * i + l16, rows - 1);           // rows beyond the last read it and are not stored
        x_row[i] = x + (size_t)(gather != nullptr ? gather[r] : r) * k + h8;
    }
    const u32x4 zero = (u32x4){0u, 0u, 0u, 0u};
    f32x4 acc[NW][MT];
#pragma unroll
    for (int g = 0; g < NW; ++g)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[g][i] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    Frag wf[AHEAD][2][NW], xf[AHEAD][2][MT];
    auto fetch = [&](int j, int at) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int kk = at + 32 * half;          // k is a multiple of 32: the last step may be half a step
#pragma unroll
            for (int g = 0; g < NW; ++g) wf[j][half][g].u = kk < k ? *(const u32x4*)(w_row + (size_t)g * n_out * k + kk + h8) : zero;
#pragma unroll
            for (int i = 0; i < MT; ++i) xf[j][half][i].u = kk < k ? *(const u32x4*)(x_row[i] + kk) : zero;
        }
    };
    for (int at = STEP * wave; at < k; at += STEP * ROWS_WAVES * AHEAD) {
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) fetch(j, at + STEP * ROWS_WAVES * j);
#pragma unroll
        for (int j = 0; j < AHEAD; ++j)
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
                for (int g = 0; g < NW; ++g)
#pragma unroll
                    for (int i = 0; i < MT; ++i)
                        acc[g][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j][half][g].v, xf[j][half][i].v, acc[g][i], 0, 0, 0);
    }
    // a lane holds columns 4 (l / 16) .. + 3 of row l % 16
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        if (i > 0) __syncthreads();
#pragma unroll
        for (int g = 0; g < NW; ++g) *(f32x4*)part_s[wave][g][lane] = acc[g][i];
        __syncthreads();
        const int c = threadIdx.x & 15, m = threadIdx.x >> 4;
        if (m < 16 && 16 * i + m < rows && n0 + c < n_out) {
            const int from = 16 * (c >> 2) + m;
            float total[NW];
#pragma unroll
            for (int g = 0; g < NW; ++g) {
                total[g] = 0.0f;
#pragma unroll
                for (int p = 0; p < ROWS_WAVES; ++p) total[g] += part_s[p][g][from][c & 3];
            }
            const int r = row0 + 16 * i + m;
            float y;
            if (GLU) {
                const float s = row_weight != nullptr ? row_weight[r] : 1.0f;
                y = activate<sizeof(TO) == 2>(s * total[0], act) * (s * total[NW - 1]);
            } else {
                y = activate<sizeof(TO) == 2>(total[0], act);
            }
            store_f(out + (size_t)r * n_out, n0 + c, y);
        }
    }
}

template <typename TO, bool GLU>
__global__ void __launch_bounds__(ROWS_WAVES * KIPP_WAVE)
moe_expert_rows_kernel(const bf16_t* __restrict__ x, const int32_t* __restrict__ gather, const float* __restrict__ row_weight,
                       const bf16_t* __restrict__ w, const int32_t* __restrict__ tiles, TO* __restrict__ out, int n_out, int k, int act) {
    __shared__ __attribute__((aligned(16))) float part_s[ROWS_WAVES][GLU ? 2 : 1][KIPP_WAVE][4];
    const int32_t* tile = tiles + (size_t)blockIdx.y * 3;
    const int rows = tile[2];
    if (rows == 0) return;      // uniform over the workgroup
    const int n0 = 16 * blockIdx.x, row0 = tile[1];
    const bf16_t* w_row = w + ((size_t)tile[0] * (GLU ? 2 : 1) * n_out + min(n0 + (int)(threadIdx.x & 15), n_out - 1)) * k;
    if (rows <= 16) expert_rows<TO, GLU, 1>(x, gather, row_weight, w_row, out, row0, rows, n0, n_out, k, act, part_s);
    else if (rows <= 32) expert_rows<TO, GLU, 2>(x, gather, row_weight, w_row, out, row0, rows, n0, n_out, k, act, part_s);
    else expert_rows<TO, GLU, 4>(x, gather, row_weight, w_row, out, row0, rows, n0, n_out, k, act, part_s);
}

// One matrix, steps of up to 16 tokens, whose tiles have no more rows than that (any number is taken, 16 after another): one fragment of rows fits 64
// registers, four workgroups share a compute unit where the form above has two, and the matrix is asked for before it is known which rows
// of x the tile has.  A wave's place along k is the same for all its lanes: whole branches, no masks around the loads.  Which K it is for: `few_pays`.
template <typename TO>
__global__ void __launch_bounds__(ROWS_WAVES * KIPP_WAVE, 8)
moe_expert_few_kernel(const bf16_t* __restrict__ x, const int32_t* __restrict__ gather, const bf16_t* __restrict__ w, const int32_t* __restrict__ tiles,
                      TO* __restrict__ out, int n_out, int k, int act) {
    constexpr int STEP = 64, AHEAD = 2;
    __shared__ __attribute__((aligned(16))) float part_s[ROWS_WAVES][KIPP_WAVE][4];
    const int32_t* tile = tiles + (size_t)blockIdx.y * 3;
    const int rows = tile[2];
    if (rows == 0) return;      // uniform over the workgroup
    const int n0 = 16 * blockIdx.x, row0 = tile[1];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KIPP_WAVE), lane = threadIdx.x & (KIPP_WAVE - 1), l16 = lane & 15, h8 = 8 * (lane >> 4);
    const bf16_t* w_row = w + ((size_t)tile[0] * n_out + min(n0 + l16, n_out - 1)) * k + h8;
    for (int r0 = 0; r0 < rows; r0 += 16) {
        if (r0 > 0) __syncthreads();
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        Frag wf[AHEAD][2], xf[AHEAD][2];
        auto fetch = [&](Frag (&to)[2], const bf16_t* row, int from) {          // k is a multiple of a step
            if (from >= k) return;
#pragma unroll
            for (int half = 0; half < 2; ++half) to[half].u = *(const u32x4*)(row + from + 32 * half);
        };
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) fetch(wf[j], w_row, STEP * (wave + ROWS_WAVES * j));
        const int r = row0 + min(r0 + l16, rows - 1);               // rows beyond the last read it and are not stored
        const bf16_t* x_row = x + (size_t)(gather != nullptr ? gather[r] : r) * k + h8;
        for (int at = STEP * wave; at < k; at += STEP * ROWS_WAVES * AHEAD) {
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) {
                if (at > STEP * wave) fetch(wf[j], w_row, at + STEP * ROWS_WAVES * j);
                fetch(xf[j], x_row, at + STEP * ROWS_WAVES * j);
            }
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) {
                if (at + STEP * ROWS_WAVES * j >= k) break;
#pragma unroll
                for (int half = 0; half < 2; ++half) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j][half].v, xf[j][half].v, acc, 0, 0, 0);
            }
        }
        *(f32x4*)part_s[wave][lane] = acc;          // a lane holds columns 4 (l / 16) .. + 3 of row l % 16
        __syncthreads();
        const int c = threadIdx.x & 15, m = threadIdx.x >> 4;
        if (m < 16 && r0 + m < rows && n0 + c < n_out) {
            float total = 0.0f;
#pragma unroll
            for (int p = 0; p < ROWS_WAVES; ++p) total += part_s[p][16 * (c >> 2) + m][c & 3];
            store_f(out + (size_t)(row0 + r0 + m) * n_out, n0 + c, activate<sizeof(TO) == 2>(total, act));
        }
    }
}

// A logit that weighs the shared expert's result, by its sigmoid: float32 at column `column` of rows of `stride` (slabs added in
// order); z null: none, the result as it is.
struct SharedGate {
    const float* z;
    int parts;
    size_t part_stride;
    int stride, column;
};

__device__ __forceinline__ float shared_weight(const SharedGate& g, int t) {
    if (g.z == nullptr) return 1.0f;
    const float* at = g.z + (size_t)t * g.stride + g.column;
    float v = at[0];
    for (int q = 1; q < g.parts; ++q) v += at[q * g.part_stride];
    return 1.0f / (1.0f + expf(-v));
}

// out[t][c] = sum_j weight[t][j] y[place[t top + j]][c] (weight null: every weight one; place below 0: x[t][c] in the place of
// y's row) + the shared gate's weight times the sum of the slabs of shared[t][c]
template <typename TX>
__global__ void moe_combine_kernel(const float* __restrict__ y, const int32_t* __restrict__ place, const float* __restrict__ weight,
                                   const float* __restrict__ shared, int shared_parts, size_t shared_stride, const TX* __restrict__ x,
                                   SharedGate gate, float* __restrict__ out, int tokens, int width, int top) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)tokens * width) return;
    const int t = (int)(i / width), c = (int)(i - (size_t)t * width);
    float acc = 0.0f;
    for (int j = 0; j < top; ++j) {
        const int at = place[(size_t)t * top + j];
        const float v = at >= 0 ? y[(size_t)at * width + c] : (x != nullptr ? load_f(x, i) : 0.0f);
        acc = fmaf(weight != nullptr ? weight[(size_t)t * top + j] : 1.0f, v, acc);
    }
    if (shared_parts > 0) {
        float a = 0.0f;
        for (int p = 0; p < shared_parts; ++p) a += shared[p * shared_stride + i];
        acc = fmaf(shared_weight(gate, t), a, acc);
    }
    out[i] = acc;
}

__device__ __forceinline__ float4 row4(const float* x, size_t i4) { return ((const float4*)x)[i4]; }
__device__ __forceinline__ float4 row4(const bf16_t* x, size_t i4) {
    const uint2 r = ((const uint2*)x)[i4];
    return make_float4(__uint_as_float(r.x << 16), __uint_as_float(r.x & 0xffff0000u), __uint_as_float(r.y << 16), __uint_as_float(r.y & 0xffff0000u));
}

// The same four columns a thread, for widths that are a multiple of 4: blockIdx.x a token, its rows of y asked for eight at a time.
template <typename TX>
__global__ void __launch_bounds__(256)
moe_combine4_kernel(const float* __restrict__ y, const int32_t* __restrict__ place, const float* __restrict__ weight,
                    const float* __restrict__ shared, int shared_parts, size_t shared_stride, const TX* __restrict__ x, SharedGate gate,
                    float* __restrict__ out, int width, int top) {
    const int t = blockIdx.x, c4 = blockIdx.y * 256 + threadIdx.x, w4 = width / 4;
    if (c4 >= w4) return;
    const size_t at = (size_t)t * w4 + c4;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float4 own = x != nullptr ? row4(x, at) : acc;
    for (int j0 = 0; j0 < top; j0 += 8) {
        float4 v[8];
        float by[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (j0 + j < top) {
                const size_t pair = (size_t)t * top + j0 + j;
                const int from = place[pair];
                by[j] = weight != nullptr ? weight[pair] : 1.0f;
                v[j] = from >= 0 ? ((const float4*)y)[(size_t)from * w4 + c4] : own;
            }
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (j0 + j < top) {
                acc.x = fmaf(by[j], v[j].x, acc.x);
                acc.y = fmaf(by[j], v[j].y, acc.y);
                acc.z = fmaf(by[j], v[j].z, acc.z);
                acc.w = fmaf(by[j], v[j].w, acc.w);
            }
    }
    if (shared_parts > 0) {
        float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (int p = 0; p < shared_parts; ++p) {
            const float4 s = ((const float4*)(shared + p * shared_stride))[at];
            a.x += s.x; a.y += s.y; a.z += s.z; a.w += s.w;
        }
        const float by = shared_weight(gate, t);
        acc.x = fmaf(by, a.x, acc.x);
        acc.y = fmaf(by, a.y, acc.y);
        acc.z = fmaf(by, a.z, acc.z);
        acc.w = fmaf(by, a.w, acc.w);
    }
    ((float4*)out)[at] = acc;
}

// Registers for twice the pairs at hand are asked for and masked: 8,192 pairs in 16 a thread 15.7 us with the routers' launch, in 8 12.6, without 14.5.
static void launch_sort(const Sort& sort, const int32_t* chosen, const float* weight, hipStream_t stream) {
#define KIPP_SORT(PER) hipLaunchKernelGGL(moe_sort_kernel<PER>, dim3(1), dim3(SORT_THREADS), 0, stream, sort, chosen, weight)
    if (sort.pairs <= 4 * SORT_THREADS) KIPP_SORT(4);
    else if (sort.pairs <= 8 * SORT_THREADS) KIPP_SORT(8);
    else if (sort.pairs <= 16 * SORT_THREADS) KIPP_SORT(16);
    else KIPP_SORT(0);
#undef KIPP_SORT
}

extern "C" int kipp_moe_route(const float* z, int parts, int stride, int32_t* chosen, float* weight, int tokens, int experts, int top,
                              float eps, int32_t* pair_token, int32_t* place_of_pair, int32_t* tiles, int max_tiles, int tile_rows,
                              float* row_weight, hipStream_t stream) {
    if (tokens <= 0) return 0;
    if (experts <= 0 || experts > MAX_EXPERTS || top <= 0 || top > MAX_TOP || top > experts || stride < experts || parts <= 0) return -1;
    const int pairs = tokens * top;
    if (tile_rows != TILE_ROWS && tile_rows != ROWS_TILE && tile_rows != MFMA_ROWS && tile_rows != MANY_ROWS) return -1;
    if (max_tiles < (pairs + tile_rows - 1) / tile_rows + (experts < pairs ? experts : pairs)) return -1;
    const Sort sort = {pairs, experts, top, pair_token, place_of_pair, tiles, max_tiles, tile_rows, row_weight};
#define KIPP_RT(REGS, WAVES, SORT)                                                                                                     \
    hipLaunchKernelGGL((moe_route_kernel<REGS, WAVES, SORT>), dim3((tokens + WAVES - 1) / WAVES), dim3(WAVES * KIPP_WAVE), 0, stream, z, \
                       parts, (size_t)tokens * stride, stride, chosen, weight, tokens, experts, top, eps, sort)
    if (tokens <= ROUTE_SORT_TOKENS && experts <= 4 * KIPP_WAVE) {
        if (tokens <= ROUTE_WAVES && experts <= KIPP_WAVE) KIPP_RT(1, ROUTE_WAVES, true);
        else if (experts <= KIPP_WAVE) KIPP_RT(1, ROUTE_SORT_TOKENS, true);
        else KIPP_RT(4, ROUTE_SORT_TOKENS, true);
        return KIPP_LAUNCH_CHECK();
    }
    if (experts <= KIPP_WAVE) KIPP_RT(1, ROUTE_WAVES, false);
    else if (experts <= 4 * KIPP_WAVE) KIPP_RT(4, ROUTE_WAVES, false);
    else KIPP_RT(MAX_EXPERTS / KIPP_WAVE, ROUTE_WAVES, false);
#undef KIPP_RT
    launch_sort(sort, chosen, weight, stream);
    return KIPP_LAUNCH_CHECK();
}

// The same with sigmoid scores (`softmax` 0) or a softmax, a correction of the choice (or none) and groups of which `group_keep` of
// `group_count` stay, by the sum of their two largest choice scores (`by_largest` 0) or their largest.  `experts` counts the
// router's outputs, the last `identity` of which are identity experts.
extern "C" int kipp_moe_route_grouped(const float* z, int parts, int stride, const float* correction, int32_t* chosen, float* weight,
                                      int tokens, int experts, int top, float eps, int group_count, int group_keep, float scale,
                                      int renormalize, int softmax, int by_largest, int identity, int32_t* pair_token, int32_t* place_of_pair,
                                      int32_t* tiles, int max_tiles, int tile_rows, float* row_weight, hipStream_t stream) {
    if (tokens <= 0) return 0;
    if (identity < 0 || identity >= experts || (identity > 0 && row_weight != nullptr)) return -1;
    if (experts <= 0 || experts > MAX_EXPERTS || top <= 0 || top > MAX_TOP || top > experts || stride < experts || parts <= 0) return -1;
    if (group_count <= 0 || experts % group_count || group_keep <= 0 || group_keep > group_count ||
        top > group_keep * (experts / group_count)) return -1;
    const int pairs = tokens * top, real = experts - identity;
    if (tile_rows != TILE_ROWS && tile_rows != ROWS_TILE && tile_rows != MFMA_ROWS && tile_rows != MANY_ROWS) return -1;
    if (max_tiles < (pairs + tile_rows - 1) / tile_rows + (real < pairs ? real : pairs)) return -1;
    const Sort sort = {pairs, real, top, pair_token, place_of_pair, tiles, max_tiles, tile_rows, row_weight};
#define KIPP_RG(REGS, WAVES, SORT, BY_RANK)                                                                                            \
    hipLaunchKernelGGL((moe_route_grouped_kernel<REGS, WAVES, SORT, BY_RANK>), dim3((tokens + WAVES - 1) / WAVES), dim3(WAVES * KIPP_WAVE), 0, stream, \
                       z, parts, (size_t)tokens * stride, stride, correction, chosen, weight, tokens, experts, top, eps, group_count, group_keep, \
                       scale, renormalize, softmax, by_largest, sort)
    const bool by_rank = experts <= KIPP_WAVE && experts <= RANK_EXPERTS * top;
    if (tokens <= ROUTE_SORT_TOKENS && experts <= 4 * KIPP_WAVE) {
        if (tokens <= ROUTE_WAVES && by_rank) KIPP_RG(1, ROUTE_WAVES, true, true);
        else if (by_rank) KIPP_RG(1, ROUTE_SORT_TOKENS, true, true);
        else if (tokens <= ROUTE_WAVES && experts <= KIPP_WAVE) KIPP_RG(1, ROUTE_WAVES, true, false);
        else if (experts <= KIPP_WAVE) KIPP_RG(1, ROUTE_SORT_TOKENS, true, false);
        else KIPP_RG(4, ROUTE_SORT_TOKENS, true, false);
        return KIPP_LAUNCH_CHECK();
    }
    if (by_rank) KIPP_RG(1, ROUTE_WAVES, false, true);
    else if (experts <= KIPP_WAVE) KIPP_RG(1, ROUTE_WAVES, false, false);
    else if (experts <= 4 * KIPP_WAVE) KIPP_RG(4, ROUTE_WAVES, false, false);
    else KIPP_RG(MAX_EXPERTS / KIPP_WAVE, ROUTE_WAVES, false, false);
#undef KIPP_RG
    launch_sort(sort, chosen, weight, stream);
    return KIPP_LAUNCH_CHECK();
}

template <typename TO, bool GLU, bool FEW>
static int launch_tiles(const void* x, const int32_t* gather, const float* row_weight, const void* w, const int32_t* tiles, int max_tiles,
                        void* out, int n_out, int k, int act, hipStream_t stream) {
    constexpr int lds_bytes = LineWalk<FEW ? 1 : MANY_ROWS / 64, 2, 2, TILE_ACROSS>::LDS_BYTES;
    static bool prepared = false;
    if (!prepared) {
        if (hipFuncSetAttribute((const void*)moe_expert_tiles_kernel<TO, GLU, FEW>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                lds_bytes) != hipSuccess)
            return -6;
        prepared = true;
    }
    const int col_tiles = (n_out + TILE_COLS(GLU) - 1) / TILE_COLS(GLU);
    const int grid = XCDS * ((max_tiles * col_tiles + XCDS - 1) / XCDS + DIE_UNITS / (FEW ? 1 : 2));        // halves: as many more
    hipLaunchKernelGGL((moe_expert_tiles_kernel<TO, GLU, FEW>), dim3(grid), dim3(512), lds_bytes, stream, (const bf16_t*)x,
                       gather, row_weight, (const bf16_t*)w, tiles, max_tiles, col_tiles, (TO*)out, n_out, k, act);
    return KIPP_LAUNCH_CHECK();
}

// Whether tiles of up to 16 rows of one matrix take the form that four workgroups a compute unit share: where there are two rounds of them (with less
// up to 3 % slower), in whole steps of k (with half a step at the end 1 to 6 % slower), of more than one turn of the waves (1,024 numbers; up to
// there the same within 1 %) and up to two and a half: what the rows are waited for is a smaller part of a longer walk.  Not where rows of the
// matrix lie 4 KiB apart: four workgroups' requests then crowd into the same parts of memory (60 experts of 2,048 x 2,048 88.9 / 98.4 us).
// The form for up to 64 rows / this, us: 28 experts of 2 rows, 2,432 x 2,560, gathered, 66.3 / 62.6, 2,560 x 2,432 62.5 / 61.1 (5.7 TB/s); 60 of one row,
// 1,536 x 1,408 51.7 / 45.0; 32 of 8 rows, 2,432 x 2,560 92.0 / 83.2.  1,640 products of 512 to 3,584 rows of W and 1 to 16 of x, two rounds and more:
// 6 to 13 % less in the mean, 1.3 % more at most.  A gated product gains nothing (11 experts 54.8, 54.9; 60 of 768 x 2,048 68.3, 69.7).
static bool few_pays(long long groups, int k) {
    const int step = 64, turn = 2 * step * ROWS_WAVES;
    return groups > 8 * 256 && k % step == 0 && k > turn && k <= 5 * turn / 2 && k % 2048 != 0;
}

template <bool GLU>
static int launch_expert(const void* x, int x_dtype, const int32_t* gather, const float* row_weight, const void* w, int w_dtype,
                         const int32_t* tiles, int max_tiles, void* out, int out_dtype, int n_out, int k, int act, int tile_rows,
                         int x_rows, int sorted_rows, int experts, int most_rows, hipStream_t stream) {
    if (max_tiles <= 0) return 0;
    if (n_out <= 0 || k <= 0 || act < ACT_NONE || act > ACT_RELU2) return -1;
    // a lane's offsets into x and into an expert's matrix are 32 bits wide in the kernels for whole tiles: numbers in the staged one, bytes
    // in the walk; rows of x that `gather` may name reach as far as x does
    const bool fits = (long long)max_tiles * tile_rows * k < (1ll << 31) && (long long)(GLU ? 2 : 1) * n_out * k < (1ll << 31) &&
                      (long long)x_rows * k < (1ll << 32);
    // Tiles of few rows whose workgroups would have little of K each, and be many, are the walk's: beside the staged kernel, in whose time the walk takes 0.78 here,
    // the one for few rows takes, 256 experts of 1,024 x 512 and 10 pairs an expert, 1.25 and 1.5 of the time (gated, and back); 64 of 2,048 x 704, up 0.8, back 1.35.
    const long long hit = sorted_rows < experts ? sorted_rows : experts;
    const bool short_k = k <= ROWS_SHORT_K && hit * ((n_out + 15) / 16) > ROWS_SHORT_GROUPS;
    if (tile_rows == ROWS_TILE && !(short_k && fits)) {
        if (x_dtype != KIPP_BF16 || w_dtype != KIPP_BF16 || k % 32 || (((uintptr_t)x | (uintptr_t)w) & 15)) return -2;
        dim3 grid((n_out + 15) / 16, max_tiles), block(ROWS_WAVES * KIPP_WAVE);
        const bool few = !GLU && most_rows > 0 && most_rows <= 16 && few_pays(hit * ((n_out + 15) / 16), k);
#define KIPP_ROWS(TO)                                                                                                                       \
    if (few)                                                                                                                                \
        hipLaunchKernelGGL(moe_expert_few_kernel<TO>, grid, block, 0, stream, (const bf16_t*)x, gather, (const bf16_t*)w, tiles, (TO*)out,    \
                           n_out, k, act);                                                                                                  \
    else                                                                                                                                    \
        hipLaunchKernelGGL((moe_expert_rows_kernel<TO, GLU>), grid, block, 0, stream, (const bf16_t*)x, gather, row_weight, (const bf16_t*)w, \
                           tiles, (TO*)out, n_out, k, act)
        if (out_dtype == KIPP_BF16) {
            KIPP_ROWS(bf16_t);
        } else if (out_dtype == KIPP_F32) {
            KIPP_ROWS(float);
        } else {
            return -2;
        }
#undef KIPP_ROWS
        return KIPP_LAUNCH_CHECK();
    }
    if (tile_rows == ROWS_TILE || tile_rows == MFMA_ROWS || tile_rows == MANY_ROWS) {
        if (x_dtype != KIPP_BF16 || w_dtype != KIPP_BF16 || k % 32 || !fits) return -2;
        // the walk brings 16 bytes a lane
        const bool walks = (((uintptr_t)x | (uintptr_t)w) & 15) == 0 && (long long)x_rows * k < (1ll << 31);
        if (!walks && tile_rows != MANY_ROWS) {
            const int cols = GLU ? MFMA_COLS / 2 : MFMA_COLS;
            dim3 grid(max_tiles, (n_out + cols - 1) / cols), block(MFMA_THREADS);
            if (out_dtype == KIPP_BF16)
                hipLaunchKernelGGL((moe_expert_mfma_kernel<bf16_t, GLU>), grid, block, 0, stream, (const bf16_t*)x, gather, row_weight,
                                   (const bf16_t*)w, tiles, (bf16_t*)out, n_out, k, act);
            else if (out_dtype == KIPP_F32)
                hipLaunchKernelGGL((moe_expert_mfma_kernel<float, GLU>), grid, block, 0, stream, (const bf16_t*)x, gather, row_weight,
                                   (const bf16_t*)w, tiles, (float*)out, n_out, k, act);
            else
                return -2;
            return KIPP_LAUNCH_CHECK();
        }
        if (!walks) return -2;
        if (out_dtype == KIPP_BF16) return tile_rows == ROWS_TILE ? launch_tiles<bf16_t, GLU, true>(x, gather, row_weight, w, tiles, max_tiles, out, n_out, k, act, stream)
                                       : launch_tiles<bf16_t, GLU, false>(x, gather, row_weight, w, tiles, max_tiles, out, n_out, k, act, stream);
        if (out_dtype == KIPP_F32) return tile_rows == ROWS_TILE ? launch_tiles<float, GLU, true>(x, gather, row_weight, w, tiles, max_tiles, out, n_out, k, act, stream)
                                       : launch_tiles<float, GLU, false>(x, gather, row_weight, w, tiles, max_tiles, out, n_out, k, act, stream);
        return -2;
    }
    if (tile_rows != TILE_ROWS) return -1;
    dim3 grid(max_tiles, (n_out + EXPERT_COLS - 1) / EXPERT_COLS), block(EXPERT_COLS);
#define KIPP_ME(TX, TW, TO)                                                                                                  \
    hipLaunchKernelGGL((moe_expert_kernel<TX, TW, TO, GLU>), grid, block, 0, stream, (const TX*)x, gather, row_weight,         \
                       (const TW*)w, tiles, (TO*)out, n_out, k, act)
    if (x_dtype == KIPP_F32 && w_dtype == KIPP_F32 && out_dtype == KIPP_F32) KIPP_ME(float, float, float);
    else if (x_dtype == KIPP_BF16 && w_dtype == KIPP_BF16 && out_dtype == KIPP_BF16) KIPP_ME(bf16_t, bf16_t, bf16_t);
    else if (x_dtype == KIPP_BF16 && w_dtype == KIPP_BF16 && out_dtype == KIPP_F32) KIPP_ME(bf16_t, bf16_t, float);
    else return -2;
#undef KIPP_ME
    return KIPP_LAUNCH_CHECK();
}

// `tile_rows`: the rows of the tiles that `kipp_moe_route` was asked for: 64, 128 and 256 take the matrix cores (bfloat16 x and w, K a
// multiple of 32), 16 the plain kernel.  `x_rows`: rows that x has.  `sorted_rows` of `experts` experts in all: which kernel for whole tiles is the faster.
// `most_rows`: the rows that a tile has at most, where the caller knows (else 0): which kernel for few rows is.
extern "C" int kipp_moe_expert(const void* x, int x_dtype, const int32_t* gather, const void* w, int w_dtype, const int32_t* tiles,
                               int max_tiles, void* out, int out_dtype, int n_out, int k, int act, int tile_rows, int x_rows, int sorted_rows,
                               int experts, int most_rows, hipStream_t stream) {
    return launch_expert<false>(x, x_dtype, gather, nullptr, w, w_dtype, tiles, max_tiles, out, out_dtype, n_out, k, act, tile_rows, x_rows, sorted_rows,
                                experts, most_rows, stream);
}

// The same against w [experts][2 n_out][k] = [gate; up] with a weight a sorted row (or null): out = act(s gate) * (s up).
extern "C" int kipp_moe_expert_gated(const void* x, int x_dtype, const int32_t* gather, const float* row_weight, const void* w, int w_dtype,
                                     const int32_t* tiles, int max_tiles, void* out, int out_dtype, int n_out, int k, int act,
                                     int tile_rows, int x_rows, int sorted_rows, int experts, hipStream_t stream) {
    return launch_expert<true>(x, x_dtype, gather, row_weight, w, w_dtype, tiles, max_tiles, out, out_dtype, n_out, k, act, tile_rows, x_rows, sorted_rows,
                               experts, 0, stream);
}

// `x` (or null): the rows that identity experts hand on.  `gate_z` (or null): rows whose column `gate_column` holds the logit that
// weighs `shared` (float32, or slabs of it).
extern "C" int kipp_moe_combine(const float* y, const int32_t* place, const float* weight, const float* shared, int shared_parts,
                                const void* x, int x_dtype, const float* gate_z, int gate_parts, int gate_stride, int gate_column,
                                float* out, int tokens, int width, int top, hipStream_t stream) {
    if (tokens <= 0) return 0;
    if (width <= 0 || top <= 0 || (x_dtype != KIPP_F32 && x_dtype != KIPP_BF16)) return -1;
    if (gate_z != nullptr && (gate_parts <= 0 || gate_column < 0 || gate_column >= gate_stride || shared == nullptr)) return -1;
    const size_t total = (size_t)tokens * width;
    const SharedGate gate = {gate_z, gate_parts, (size_t)tokens * gate_stride, gate_stride, gate_column};
    const int parts = shared != nullptr ? shared_parts : 0;
    if (width % 4 == 0 && (((uintptr_t)y | (uintptr_t)out | (uintptr_t)shared | (uintptr_t)x) & 15) == 0) {
        dim3 grid(tokens, (width / 4 + 255) / 256), block(256);
        if (x_dtype == KIPP_BF16)
            hipLaunchKernelGGL(moe_combine4_kernel<bf16_t>, grid, block, 0, stream, y, place, weight, shared, parts, total, (const bf16_t*)x, gate, out, width, top);
        else
            hipLaunchKernelGGL(moe_combine4_kernel<float>, grid, block, 0, stream, y, place, weight, shared, parts, total, (const float*)x, gate, out, width, top);
        return KIPP_LAUNCH_CHECK();
    }
    dim3 grid((unsigned)((total + 255) / 256)), block(256);
    if (x_dtype == KIPP_BF16)
        hipLaunchKernelGGL(moe_combine_kernel<bf16_t>, grid, block, 0, stream, y, place, weight, shared, parts, total, (const bf16_t*)x, gate, out, tokens, width, top);
    else
        hipLaunchKernelGGL(moe_combine_kernel<float>, grid, block, 0, stream, y, place, weight, shared, parts, total, (const float*)x, gate, out, tokens, width, top);
    return KIPP_LAUNCH_CHECK();
}

// out[r][i] = act(sum of the slabs of u[r][i]) [* sum of the slabs of u[r][inner + i] when `glu`]; with `bias` (over u's
// columns) each sum has its column's bias added first
// COLS neighbouring columns a thread: four where they lie together (gelu of 2,048 x 2,432 in one slab to bfloat16 9.2 us, 10.9 one by one with erff).
template <typename TO, int COLS>
__global__ void __launch_bounds__(256) activate_kernel(const float* __restrict__ u, int parts, size_t part_stride, TO* __restrict__ out, size_t total,
                                                       int inner, int glu, int act, const float* __restrict__ bias) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * COLS;
    if (i >= total) return;
    const size_t r = total <= 0xffffffffull ? (uint32_t)i / (uint32_t)inner : i / inner;
    const int c = (int)(i - r * inner);
    const size_t at = glu ? r * 2 * inner + c : i;
    typedef __attribute__((ext_vector_type(COLS))) float fN;
    fN a = *(const fN*)(u + at), b = {};
    if (glu) b = *(const fN*)(u + at + inner);
    for (int p = 1; p < parts; ++p) {
        a += *(const fN*)(u + p * part_stride + at);
        if (glu) b += *(const fN*)(u + p * part_stride + at + inner);
    }
    if (bias != nullptr) {
        a += *(const fN*)(bias + c);
        if (glu) b += *(const fN*)(bias + inner + c);
    }
    float y[COLS];
#pragma unroll
    for (int k = 0; k < COLS; ++k) y[k] = a[k];
    activate_all<sizeof(TO) == 2>(y, act);
    if (glu) {
#pragma unroll
        for (int k = 0; k < COLS; ++k) y[k] *= b[k];
    }
    if constexpr (COLS == 1) {
        store_f(out, i, y[0]);
    } else if constexpr (sizeof(TO) == 4) {
        *(f32x4*)(out + i) = (f32x4){y[0], y[1], y[2], y[3]};
    } else {
        *(uint2*)(out + i) = make_uint2((uint32_t)f32_to_bf16(y[0]) | ((uint32_t)f32_to_bf16(y[1]) << 16),
                                        (uint32_t)f32_to_bf16(y[2]) | ((uint32_t)f32_to_bf16(y[3]) << 16));
    }
}

template <typename TO>
static void launch_activate(const float* u, int parts, size_t part_stride, TO* out, size_t total, int inner, int glu, int act, const float* bias,
                            hipStream_t stream) {
    const bool four = inner % 4 == 0 && (((uintptr_t)u | (uintptr_t)out | (uintptr_t)bias) & 15) == 0;
    const dim3 grid((unsigned)((total / (four ? 4 : 1) + 255) / 256)), block(256);
    if (four)
        hipLaunchKernelGGL((activate_kernel<TO, 4>), grid, block, 0, stream, u, parts, part_stride, out, total, inner, glu, act, bias);
    else
        hipLaunchKernelGGL((activate_kernel<TO, 1>), grid, block, 0, stream, u, parts, part_stride, out, total, inner, glu, act, bias);
}

extern "C" int kipp_activate_biased(const float* u, int parts, void* out, int out_dtype, int rows, int inner, int glu, int act,
                                    const float* bias, hipStream_t stream) {
    if (rows <= 0) return 0;
    if (inner <= 0 || parts <= 0 || act < ACT_SILU || act > ACT_RELU2) return -1;
    const size_t total = (size_t)rows * inner;
    const size_t part_stride = total * (glu ? 2 : 1);
    if (out_dtype == KIPP_F32)
        launch_activate<float>(u, parts, part_stride, (float*)out, total, inner, glu, act, bias, stream);
    else if (out_dtype == KIPP_BF16)
        launch_activate<bf16_t>(u, parts, part_stride, (bf16_t*)out, total, inner, glu, act, bias, stream);
    else
        return -2;
    return KIPP_LAUNCH_CHECK();
}

extern "C" int kipp_activate(const float* u, int parts, void* out, int out_dtype, int rows, int inner, int glu, int act,
                             hipStream_t stream) {
    return kipp_activate_biased(u, parts, out, out_dtype, rows, inner, glu, act, nullptr, stream);
}
