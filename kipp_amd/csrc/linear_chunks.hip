// The matrix memories of `linear_scan` over prompt portions, 64 tokens at a time, on the matrix cores' float32 instruction
// (v_mfma_f32_16x16x4_f32: products and sums stay float32).
//
// Within a chunk, with g_t the token's decay, G_t = g_0 .. g_t, D[t][s] = g_(s+1) .. g_t for s <= t, and S the memory ahead of it:
//
//     U = V                                      (decay, gated)
//     U = (I + L)^-1 beta (V - G (K S))          (delta: L[t][s] = beta_t D[t][s] k_t . k_s for s < t)
//     o = G (Q S) + A U                          A[t][s] = D[t][s] q_t . k_s for s <= t
//     S <- G_last S + K^T (D[last][s] U)
//
// which is the walk's sums in another order.  D is made by running products (a decay of zero stays one), never by
// quotients.  Three launches:
//
//     ready    (decay only) silu of q and k, once
//     prepare  a workgroup (chunk, head, entry): A, T = (I + L)^-1 by forward substitution (a lane a column), G and
//              D[last]; every chunk of the launch at once
//     walk     a workgroup (16 columns of S, head, entry) takes its chunks in order.  S stays in registers as the
//              instruction leaves it (a wave a quarter of its rows) and is shown to all waves through LDS; a wave takes 16 of the
//              chunk's tokens for Q S, K S, T R and A U.  Q, K, T and A are operands straight from memory: a wave reads its own
//              rows only, and the next chunk's are asked for as soon as this one's have been multiplied.
//
// Bound by the walk's chain: at keys of 128 a chunk is 80 instructions of 32 cycles a wave (delta: 128), the sums in between
// and two or three barriers, 3.8 us a chunk with 160 workgroups on 256 compute units.  2,048 tokens of 8 heads, keys of 128,
// values of 320: 145 us (124 the walk) with a fixed decay, 193 (168) for the delta rule, where the walk token by token takes 772
// and 663; 1,801 tokens of 40 heads with a state of 128 x 64: 120 (99), was 560.
//
// A position's bits depend on its place in the chunk, so this is for activations that are rounded to bfloat16 behind it; the walk
// token by token keeps the float32 path, where a portion gives the bits of single tokens.
//
// Entries of fewer than `from` tokens are left to that walk: a request's single token costs the same whether another request's prompt
// is in the step or not.  (64 single tokens beside a prompt of 512: a step of 7 layers, five of them with keys of 128, takes 3,750 us;
// 4,180 with every entry through the chunks, 4,590 with every entry walked.)
//
// Rows beyond an entry's last token: g = 1, beta = 0, V = 0, and the last token's q and k in place of theirs.
#include "common.h"
#include <math.h>

#define CHUNK 64
#define THREADS 256
#define UP 68               // floats from a column to the next of U and R in LDS
#define COLS 16             // columns of S a workgroup of the walk

enum { MODE_DECAY = 0, MODE_DELTA = 1, MODE_GATED = 2 };

typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ float silu_f(float z) { return z / (1.0f + expf(-z)); }

// 16 numbers of the contraction: lane l holds those at 4 (l / 16) .. + 3 of row l % 16 of a and of column l % 16 of b; the
// sums lie in lane l as rows 4 (l / 16) .. + 3 of column l % 16.
__device__ __forceinline__ f32x4 mul16(f32x4 a, f32x4 b, f32x4 acc) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], acc, 0, 0, 0);
    return acc;
}

__device__ __forceinline__ f32x4 zero4() { return (f32x4){0.0f, 0.0f, 0.0f, 0.0f}; }

// The nth of the entries that bring `from` tokens or more (-1: there are fewer), and how many chunks those before it make:
// its own lie behind them in the work space.  The same in every lane.
struct Portion {
    int entry, base;
};
__device__ __forceinline__ Portion portion_of(const int32_t* __restrict__ q_len, int entries, int from, int nth) {
    Portion p = {-1, 0};
    for (int e0 = 0; e0 < entries; e0 += KIPP_WAVE) {
        const int lane = threadIdx.x & (KIPP_WAVE - 1);
        const int n = e0 + lane < entries ? q_len[e0 + lane] : 0;
        unsigned long long found = __ballot(n > 0 && n >= from);
        const int here = __popcll(found);
        int upto = KIPP_WAVE;
        if (nth < here) {
            for (int i = 0; i < nth; ++i) found &= found - 1;
            upto = __ffsll((long long)found) - 1;
        }
        int chunks = lane < upto && n > 0 && n >= from ? (n + CHUNK - 1) / CHUNK : 0;
#pragma unroll
        for (int off = KIPP_WAVE / 2; off > 0; off >>= 1) chunks += __shfl_xor(chunks, off, KIPP_WAVE);
        p.base += chunks;
        if (nth < here) {
            p.entry = e0 + upto;
            return p;
        }
        nth -= here;
    }
    return p;
}

struct ChunkArgs {
    const float* q;             // row t, head hh: q + t * qk_stride + hh * d
    const float* k;
    int qk_stride;
    const float* src;           // v, beta and g
    int stride, v_at, beta_at, g_at;
    const float* decays;
    float* state;
    size_t state_stride;
    const int32_t *q_start, *q_len, *slots;
    float* o_raw;
    float *a, *t, *vec;         // [chunk][head][64][64], the same (delta), [chunk][head][3][64]: G, D[last], beta
    int heads, qk_rep, dv, entries, from;
};

__global__ void __launch_bounds__(THREADS)
chunks_ready_kernel(const float* __restrict__ src, int stride, float* __restrict__ out, int width) {
    const int c = (blockIdx.x * THREADS + threadIdx.x) * 4;
    if (c >= width) return;
    f32x4 v = *reinterpret_cast<const f32x4*>(src + (size_t)blockIdx.y * stride + c);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = silu_f(v[i]);
    *reinterpret_cast<f32x4*>(out + (size_t)blockIdx.y * width + c) = v;
}

template <int MODE, int DT>
__global__ void __launch_bounds__(THREADS) chunks_prepare_kernel(const ChunkArgs p) {
    constexpr int D = 64 * DT;
    __shared__ float d_s[CHUNK][CHUNK + 1];
    __shared__ __attribute__((aligned(16))) float l_s[MODE == MODE_DELTA ? CHUNK : 1][UP];
    __shared__ float beta_s[CHUNK];
    const int head = blockIdx.y, chunk = blockIdx.x;
    const Portion portion = portion_of(p.q_len, p.entries, p.from, blockIdx.z);
    if (portion.entry < 0) return;          // uniform over the workgroup, as below
    const int entry = portion.entry;
    const int n = p.q_len[entry], first = p.q_start[entry];
    if (chunk * CHUNK >= n) return;
    const int m = min(CHUNK, n - chunk * CHUNK);
    const int t0 = first + chunk * CHUNK;
    const int tid = threadIdx.x, wave = tid / KIPP_WAVE, lane = tid & (KIPP_WAVE - 1), l16 = lane & 15, h4 = 4 * (lane >> 4);
    const size_t at = (size_t)(portion.base + chunk) * p.heads + head;
    float* a_out = p.a + at * CHUNK * CHUNK;
    float* vec = p.vec + at * 3 * CHUNK;
    if (wave == 0) {
        // the wave with the fewest products below: D column by column, a lane a column
        const float* row = p.src + (size_t)(t0 + min(lane, m - 1)) * p.stride;
        const float g = lane >= m ? 1.0f : (MODE == MODE_DECAY ? p.decays[head] : row[p.g_at + head]);
        if (MODE == MODE_DELTA) {
            const float b = lane < m ? row[p.beta_at + head] : 0.0f;
            beta_s[lane] = b;
            vec[2 * CHUNK + lane] = b;
        }
        float run = 0.0f, all = 1.0f, whole = 0.0f;
        for (int t = 0; t < CHUNK; ++t) {
            const float gt = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g), t));
            run = lane == t ? 1.0f : run * gt;          // zero until the lane's own token
            all *= gt;
            if (lane == t) whole = all;
            d_s[t][lane] = run;
        }
        vec[lane] = whole;
        vec[CHUNK + lane] = run;
    }
    const float* q = p.q + (size_t)(head / p.qk_rep) * D;
    const float* k = p.k + (size_t)(head / p.qk_rep) * D;
    f32x4 qk[4], kk[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) qk[s] = kk[s] = zero4();
    if (16 * wave < m) {
        const float* q_row = q + (size_t)(t0 + min(16 * wave + l16, m - 1)) * p.qk_stride + h4;
        const float* k_row = k + (size_t)(t0 + min(16 * wave + l16, m - 1)) * p.qk_stride + h4;
        const float* s_row[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) s_row[s] = k + (size_t)(t0 + min(16 * s + l16, m - 1)) * p.qk_stride + h4;
#pragma unroll 2
        for (int j = 0; j < D; j += 16) {
            const f32x4 qv = *reinterpret_cast<const f32x4*>(q_row + j);
            const f32x4 kv = MODE == MODE_DELTA ? *reinterpret_cast<const f32x4*>(k_row + j) : zero4();
#pragma unroll
            for (int s = 0; s < 4; ++s)
                if (s <= wave) {
                    const f32x4 sv = *reinterpret_cast<const f32x4*>(s_row[s] + j);
                    qk[s] = mul16(qv, sv, qk[s]);
                    if (MODE == MODE_DELTA) kk[s] = mul16(kv, sv, kk[s]);
                }
        }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (s > wave) continue;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int t = 16 * wave + h4 + v, c = 16 * s + l16;
            const float decay = c <= t && t < m ? d_s[t][c] : 0.0f;
            a_out[t * CHUNK + c] = decay != 0.0f ? qk[s][v] * decay : 0.0f;
            if (MODE == MODE_DELTA) l_s[t][c] = c < t && decay != 0.0f ? beta_s[t] * decay * kk[s][v] : 0.0f;
        }
    }
    if (MODE != MODE_DELTA) return;
    __syncthreads();
    if (wave != 0) return;
    // T column by column: T[t] = [t = column] - sum over s < t of L[t][s] T[s]
    float x[CHUNK];
#pragma unroll
    for (int t = 0; t < CHUNK; ++t) {
        float sum = 0.0f;
#pragma unroll
        for (int s = 0; s + 4 <= t; s += 4) {
            const f32x4 l = *reinterpret_cast<const f32x4*>(&l_s[t][s]);
#pragma unroll
            for (int i = 0; i < 4; ++i) sum = fmaf(l[i], x[s + i], sum);
        }
#pragma unroll
        for (int s = t & ~3; s < t; ++s) sum = fmaf(l_s[t][s], x[s], sum);
        x[t] = (t == lane ? 1.0f : 0.0f) - sum;
        p.t[at * CHUNK * CHUNK + t * CHUNK + lane] = x[t];
    }
}

// What a wave multiplies in a chunk: its own rows of q, k, T and A, its rows of K^T, the values of its tokens.
template <int MODE, int DT>
struct Operands {
    f32x4 q[4 * DT], k[MODE == MODE_DELTA ? 4 * DT : 1], a[4], t[MODE == MODE_DELTA ? 4 : 1], e[4], kt[DT][4], v, g, b;
    float g_last;
};

template <int MODE, int DT>
__global__ void __launch_bounds__(THREADS) chunks_walk_kernel(const ChunkArgs p) {
    constexpr int D = 64 * DT, SP = D + 4;
    __shared__ __attribute__((aligned(16))) float s_s[COLS * SP];           // [column][row]
    __shared__ __attribute__((aligned(16))) float u_s[COLS * UP];           // [column][token]
    __shared__ __attribute__((aligned(16))) float r_s[MODE == MODE_DELTA ? COLS * UP : 4];
    const int head = blockIdx.y;
    const Portion portion = portion_of(p.q_len, p.entries, p.from, blockIdx.z);
    if (portion.entry < 0) return;          // uniform over the workgroup
    const int entry = portion.entry;
    const int tid = threadIdx.x, wave = tid / KIPP_WAVE, lane = tid & (KIPP_WAVE - 1), l16 = lane & 15, h4 = 4 * (lane >> 4);
    const int n = p.q_len[entry], first = p.q_start[entry];
    const int col = blockIdx.x * COLS + l16;
    const bool live = col < p.dv;
    const int own = 16 * wave;              // the wave's tokens of a chunk
    const int row0 = D / 4 * wave;          // its rows of S
    float* S_col = p.state + (size_t)p.slots[entry] * p.state_stride + ((size_t)head * p.dv + (live ? col : 0)) * D + row0 + h4;
    const float* q = p.q + (size_t)(head / p.qk_rep) * D;
    const float* k = p.k + (size_t)(head / p.qk_rep) * D;
    const float* v_src = p.src + p.v_at + (size_t)head * p.dv + (live ? col : 0);

    f32x4 S[DT];
#pragma unroll
    for (int a = 0; a < DT; ++a) S[a] = live ? *reinterpret_cast<const f32x4*>(S_col + 16 * a) : zero4();

    // The next chunk's operands are asked for as soon as this one's have been used.  (A second set of registers, asked for
    // a whole chunk ahead, changed nothing and left a compute unit one workgroup instead of two.)
    Operands<MODE, DT> x;
    auto rows_of = [&](int c) {
        const int m = min(CHUNK, n - c * CHUNK);
        if (own >= m) return;
        const size_t row = (size_t)(first + c * CHUNK + min(own + l16, m - 1)) * p.qk_stride + h4;
#pragma unroll
        for (int j = 0; j < 4 * DT; ++j) {
            x.q[j] = *reinterpret_cast<const f32x4*>(q + row + 16 * j);
            if (MODE == MODE_DELTA) x.k[j] = *reinterpret_cast<const f32x4*>(k + row + 16 * j);
        }
    };
    auto rest_of = [&](int c) {
        const int m = min(CHUNK, n - c * CHUNK), t0 = first + c * CHUNK;
        const size_t at = (size_t)(portion.base + c) * p.heads + head;
        const float* vec = p.vec + at * 3 * CHUNK;
        if (own < m) {
            const float* a_row = p.a + at * CHUNK * CHUNK + (own + l16) * CHUNK + h4;
            const float* t_row = p.t + at * CHUNK * CHUNK + (own + l16) * CHUNK + h4;
#pragma unroll
            for (int i = 0; i < 4; ++i) x.v[i] = own + h4 + i < m ? v_src[(size_t)(t0 + own + h4 + i) * p.stride] : 0.0f;
            x.g = *reinterpret_cast<const f32x4*>(vec + own + h4);
            if (MODE == MODE_DELTA) x.b = *reinterpret_cast<const f32x4*>(vec + 2 * CHUNK + own + h4);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j <= wave) {
                    if (MODE == MODE_DELTA) x.t[j] = *reinterpret_cast<const f32x4*>(t_row + 16 * j);
                    x.a[j] = *reinterpret_cast<const f32x4*>(a_row + 16 * j);
                }
        }
        x.g_last = vec[CHUNK - 1];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (16 * j >= m) continue;
            x.e[j] = *reinterpret_cast<const f32x4*>(vec + CHUNK + 16 * j + h4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float* k_row = k + (size_t)(t0 + min(16 * j + h4 + i, m - 1)) * p.qk_stride + row0 + l16;
#pragma unroll
                for (int a = 0; a < DT; ++a) x.kt[a][j][i] = k_row[16 * a];
            }
        }
    };
    const int chunks = (n + CHUNK - 1) / CHUNK;
    rows_of(0);
    rest_of(0);
    for (int c = 0; c < chunks; ++c) {
        const int m = min(CHUNK, n - c * CHUNK);
        const bool mine = own < m, more = c + 1 < chunks;
#pragma unroll
        for (int a = 0; a < DT; ++a) *reinterpret_cast<f32x4*>(&s_s[l16 * SP + row0 + 16 * a + h4]) = S[a];
        __syncthreads();
        f32x4 inter = zero4(), read = zero4();
        if (mine) {
#pragma unroll
            for (int j = 0; j < 4 * DT; ++j) {
                const f32x4 sv = *reinterpret_cast<const f32x4*>(&s_s[l16 * SP + 16 * j + h4]);
                inter = mul16(x.q[j], sv, inter);
                if (MODE == MODE_DELTA) read = mul16(x.k[j], sv, read);
            }
            f32x4 u = x.v;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (MODE == MODE_DECAY) u[i] = silu_f(u[i]);        // silu(0) = 0
                if (MODE == MODE_DELTA) u[i] = own + h4 + i < m ? x.b[i] * (x.v[i] - x.g[i] * read[i]) : 0.0f;
            }
            *reinterpret_cast<f32x4*>((MODE == MODE_DELTA ? r_s : u_s) + l16 * UP + own + h4) = u;
        }
        if (more) rows_of(c + 1);
        __syncthreads();
        if (MODE == MODE_DELTA) {
            if (mine) {
                f32x4 u = zero4();
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (j <= wave) u = mul16(x.t[j], *reinterpret_cast<const f32x4*>(r_s + l16 * UP + 16 * j + h4), u);
                *reinterpret_cast<f32x4*>(u_s + l16 * UP + own + h4) = u;
            }
            __syncthreads();
        }
        f32x4 u[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (16 * j < m) u[j] = *reinterpret_cast<const f32x4*>(u_s + l16 * UP + 16 * j + h4);
        if (mine) {
            f32x4 o = inter * x.g;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j <= wave) o = mul16(x.a[j], u[j], o);
            if (live) {
                float* o_at = p.o_raw + (size_t)(first + c * CHUNK + own + h4) * p.heads * p.dv + (size_t)head * p.dv + col;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (own + h4 + i < m) o_at[(size_t)i * p.heads * p.dv] = o[i];
            }
        }
#pragma unroll
        for (int a = 0; a < DT; ++a) S[a] *= x.g_last;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (16 * j >= m) continue;
            const f32x4 eu = u[j] * x.e[j];
#pragma unroll
            for (int a = 0; a < DT; ++a) S[a] = mul16(x.kt[a][j], eu, S[a]);
        }
        if (more) rest_of(c + 1);
    }
    if (live) {
#pragma unroll
        for (int a = 0; a < DT; ++a) *reinterpret_cast<f32x4*>(S_col + 16 * a) = S[a];
    }
}

extern "C" {

// Chunks that `tokens` tokens of `portions` entries make at most, whatever their lengths.
static long long chunk_count(int tokens, int portions) { return (long long)tokens / CHUNK + portions; }

// Floats of work space, or 0 where this kernel does not take the sizes: keys of 64, 128, 192 or 256 numbers.
long long kipp_matrix_chunks_work(int mode, int tokens, int portions, int heads, int d) {
    if (mode < MODE_DECAY || mode > MODE_GATED || tokens <= 0 || portions <= 0 || heads <= 0 || d <= 0 || d % 64 || d > 256) return 0;
    const long long each = (mode == MODE_DELTA ? 2 : 1) * CHUNK * CHUNK + 3 * CHUNK;
    return chunk_count(tokens, portions) * heads * each + (mode == MODE_DECAY ? (long long)tokens * 2 * heads * d : 0);
}

// src: float32 [tokens][stride] with q, k, v (and beta, g) at the given columns, as `kipp_decay_scan`, `kipp_delta_scan` and `kipp_gated_scan` read it
// (mode 0, 1, 2); q and k of a head at q_at + (head / qk_rep) d.  Of the entries only those of `from` tokens and more, at most `portions` of
// them; `longest`: the most tokens an entry brings.
int kipp_matrix_chunks(int mode, const float* src, int stride, int q_at, int k_at, int v_at, int beta_at, int g_at, const float* decays,
                       float* state, size_t state_stride, const int32_t* q_start, const int32_t* q_len, const int32_t* slots, float* o_raw,
                       int tokens, int entries, int heads, int qk_rep, int d, int dv, int longest, int from, int portions, float* work,
                       long long work_floats,
                       hipStream_t stream) {
    if (entries <= 0 || tokens <= 0 || portions <= 0) return 0;
    const long long need = kipp_matrix_chunks_work(mode, tokens, portions, heads, d);
    if (need == 0 || work_floats < need || longest <= 0 || qk_rep <= 0 || heads % qk_rep || dv <= 0) return -1;
    if (state_stride < (size_t)heads * d * dv || (state_stride & 3) || (stride & 3) || (q_at & 3) || (k_at & 3)) return -1;
    if (((uintptr_t)src | (uintptr_t)state | (uintptr_t)work) & 15) return -1;
    ChunkArgs p;
    const long long slots_all = chunk_count(tokens, portions) * heads;
    p.a = work;
    p.t = mode == MODE_DELTA ? p.a + slots_all * CHUNK * CHUNK : p.a;
    p.vec = p.t + slots_all * CHUNK * CHUNK;
    p.q = src + q_at;
    p.k = src + k_at;
    p.qk_stride = stride;
    if (mode == MODE_DECAY) {
        if (q_at != 0 || k_at != heads * d || qk_rep != 1) return -1;
        float* ready = p.vec + slots_all * 3 * CHUNK;
        const int width = 2 * heads * d;
        hipLaunchKernelGGL(chunks_ready_kernel, dim3((width / 4 + THREADS - 1) / THREADS, tokens), dim3(THREADS), 0, stream, src, stride, ready, width);
        p.q = ready;
        p.k = ready + heads * d;
        p.qk_stride = width;
    }
    p.src = src;
    p.stride = stride;
    p.v_at = v_at;
    p.beta_at = beta_at;
    p.g_at = g_at;
    p.decays = decays;
    p.state = state;
    p.state_stride = state_stride;
    p.q_start = q_start;
    p.q_len = q_len;
    p.slots = slots;
    p.o_raw = o_raw;
    p.heads = heads;
    p.qk_rep = qk_rep;
    p.dv = dv;
    p.entries = entries;
    p.from = from;
    const dim3 prepare((longest + CHUNK - 1) / CHUNK, heads, portions), walk((dv + COLS - 1) / COLS, heads, portions), block(THREADS);
#define KIPP_CHUNKS(MODE, DT)                                                              \
    do {                                                                                   \
        hipLaunchKernelGGL((chunks_prepare_kernel<MODE, DT>), prepare, block, 0, stream, p); \
        hipLaunchKernelGGL((chunks_walk_kernel<MODE, DT>), walk, block, 0, stream, p);       \
    } while (0)
#define KIPP_CHUNKS_D(MODE)                     \
    do {                                        \
        if (d == 64) KIPP_CHUNKS(MODE, 1);      \
        else if (d == 128) KIPP_CHUNKS(MODE, 2); \
        else if (d == 192) KIPP_CHUNKS(MODE, 3); \
        else KIPP_CHUNKS(MODE, 4);              \
    } while (0)
    if (mode == MODE_DECAY) KIPP_CHUNKS_D(MODE_DECAY);
    else if (mode == MODE_DELTA) KIPP_CHUNKS_D(MODE_DELTA);
    else KIPP_CHUNKS_D(MODE_GATED);
#undef KIPP_CHUNKS_D
#undef KIPP_CHUNKS
    return KIPP_LAUNCH_CHECK();
}

}  // extern "C"
