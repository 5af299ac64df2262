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
// and an mLSTM is a decay a token and head, g = exp(lf + m - m'), with U = exp(li - m') V and one more column of S, of values of one: n, whose
// o is what the others are divided by.
//
// These are the walk's sums in another order.  D is made by running products (a decay of zero stays one), never by
// quotients.  Two or three launches:
//
//     ready    (decay only) silu of q and k, once
//     gates    (mLSTM only) m, and what follows from it
//     prepare  a workgroup (chunk, head, entry): A, T = (I + L)^-1 by forward substitution (a lane a column), G and
//              D[last]; every chunk of the launch at once
//     walk     a workgroup (16 columns of S, head, entry) takes its chunks in order.  Four waves keep S in registers as the
//              instruction leaves it (a wave a quarter of its rows), take it through the chunk (U first, for the delta rule) and show it
//              through LDS for the next one; four others sum o for 16 of the chunk's tokens each, Q S and A U, meanwhile: what S waits for
//              is a chain of 16 instructions a chunk (delta: 80), not of 80 (128).  One barrier a chunk (delta: three).  Q, K, T and A are operands
//              straight from memory, the next chunk's asked for as soon as this one's have been multiplied.
//
// Bound by the walk's chain and the latency of its operands: 2,048 tokens of 8 heads, keys of 128, values of 320, all launches, us, with four
// waves that do both / now: fixed decay 145 / 101, delta rule 185 / 154, an mLSTM 137 / 113; keys of 256, values of 512: 229 / 193, 293 / 250, 378 / 303;
// 40 heads with a state of 128 x 64 127 / 98.  Token by token they take 772, 663 and 751, and 560.  More workgroups than the chip has places for are
// the other way round (16 entries of 80 tokens, gated, 73 / 77): those keep the four waves.
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

#define VECS 4              // vectors of 64 numbers a chunk and head

enum { MODE_DECAY = 0, MODE_DELTA = 1, MODE_GATED = 2, MODE_MLSTM = 3 };

// Runs that a contraction over the key size is summed in, every RUNS-th 16 numbers one, then in pairs: an mLSTM divides by a sum that may
// almost cancel, so its sums are kept as short as the walk's (errors of its rows against 64 bits, median over 1,100 tokens of 128 x 320: 1.66e-7
// in one run, 1.44e-7 in two, 1.31e-7 in four, 1.52e-7 by the walk; 600 tokens of 256 x 64: 2.6e-7, 2.1e-7, 1.8e-7, 1.5e-7 in eight, 1.5e-7).
constexpr int runs_of(int mode, int dt) { return mode != MODE_MLSTM ? 1 : (dt == 4 ? 8 : 4); }

typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ float silu_f(float z) { return z / (1.0f + expf(-z)); }

// 16 numbers of the contraction: lane l holds those at 4 (l / 16) .. + 3 of row l % 16 of a and of column l % 16 of b; the
// sums lie in lane l as rows 4 (l / 16) .. + 3 of column l % 16.
__device__ __forceinline__ f32x4 mul16(f32x4 a, f32x4 b, f32x4 acc) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], acc, 0, 0, 0);
    return acc;
}

template <int RUNS, int N>
__device__ __forceinline__ f32x4 sum_runs(const f32x4 (&runs)[RUNS][N], int n) {
    f32x4 sum[RUNS];
#pragma unroll
    for (int h = 0; h < RUNS; ++h) sum[h] = runs[h][n];
#pragma unroll
    for (int w = 1; w < RUNS; w <<= 1)
#pragma unroll
        for (int h = 0; h + w < RUNS; h += 2 * w) sum[h] += sum[h + w];
    return sum[0];
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
    float *a, *t, *vec;         // [chunk][head][64][64], the same (delta), [chunk][head][4][64]: G, D[last], beta (mLSTM: the input gate), mLSTM's floor of a denominator
    int heads, qk_rep, d, dv, entries, from, portions;
    // mLSTM: the gates' columns and biases, their cap, where a slot's copies of n begin and how many there are, 1 / sqrt(d), and what a
    // token's sums are divided by, [token][head]
    const float *bias_i, *bias_f;
    int i_at, f_at, n_at, copies;
    float cap, q_scale;
    float* den;
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

__device__ __forceinline__ float log_sigmoid(float z) { return fminf(z, 0.0f) - log1pf(expf(-fabsf(z))); }

#define GATE_WAVES 16

// The gates of an mLSTM head: m' = max(lf + m, li) is an affine step of (max, +), so a wave scans 64 tokens in six exchanges and the
// waves' results are joined through LDS: 1,024 tokens a turn.  Leaves a token's decay (in G's place), input gate and floor.  For an entry
// that walks it writes the ones that its finished sums are divided by.
__global__ void __launch_bounds__(GATE_WAVES * KIPP_WAVE) chunks_gates_kernel(const ChunkArgs p) {
    __shared__ float a_s[GATE_WAVES], b_s[GATE_WAVES];
    const int head = blockIdx.x, entry = blockIdx.y, tid = threadIdx.x;
    const int wave = tid / KIPP_WAVE, lane = tid & (KIPP_WAVE - 1);
    const int n = p.q_len[entry], first = p.q_start[entry];
    if (n <= 0) return;
    if (n < p.from) {
        if (tid < n) p.den[(size_t)(first + tid) * p.heads + head] = 1.0f;      // `from` is less than the threads
        return;
    }
    int base = 0, ahead = 0;        // chunks of the entries ahead, as `portion_of` counts them, and how many entries those are
    for (int e0 = 0; e0 < entry; e0 += KIPP_WAVE) {
        const int len = e0 + lane < entry ? p.q_len[e0 + lane] : 0;
        const bool portion = len > 0 && len >= p.from;
        int chunks = portion ? (len + CHUNK - 1) / CHUNK : 0;
#pragma unroll
        for (int off = KIPP_WAVE / 2; off > 0; off >>= 1) chunks += __shfl_xor(chunks, off, KIPP_WAVE);
        base += chunks;
        ahead += __popcll(__ballot(portion));
    }
    if (ahead >= p.portions) return;        // beyond what the work space is laid out for and the other kernels take; uniform over the workgroup
    float* m_all = p.state + (size_t)p.slots[entry] * p.state_stride + p.n_at + (size_t)p.copies * p.heads * (p.d);
    float m = m_all[head];
    const float bi = p.bias_i[head], bf = p.bias_f[head];
    for (int t0 = 0; t0 < n; t0 += GATE_WAVES * CHUNK) {
        const int chunk = t0 / CHUNK + wave, t = chunk * CHUNK + lane;
        float lf = 0.0f, li = -INFINITY;        // beyond the last token: m stays
        if (t < n) {
            const float* row = p.src + (size_t)(first + t) * p.stride;
            li = p.cap * tanhf((row[p.i_at + head] + bi) / p.cap);
            lf = log_sigmoid(p.cap * tanhf((row[p.f_at + head] + bf) / p.cap));
        }
        float a = lf, b = li;                   // tokens up to this one: m -> max(a + m, b)
#pragma unroll
        for (int off = 1; off < KIPP_WAVE; off <<= 1) {
            const float a0 = __shfl_up(a, off, KIPP_WAVE), b0 = __shfl_up(b, off, KIPP_WAVE);
            if (lane >= off) {
                b = fmaxf(b0 + a, b);
                a += a0;
            }
        }
        __syncthreads();                        // the turn before has been read
        if (lane == KIPP_WAVE - 1) {
            a_s[wave] = a;
            b_s[wave] = b;
        }
        __syncthreads();
        float mine = m;
        for (int w = 0; w < GATE_WAVES; ++w) {
            if (w == wave) mine = m;
            m = fmaxf(a_s[w] + m, b_s[w]);
        }
        const float after = fmaxf(a + mine, b);
        float before = __shfl_up(after, 1, KIPP_WAVE);
        if (lane == 0) before = mine;
        if (chunk * CHUNK < n) {
            float* vec = p.vec + ((size_t)(base + chunk) * p.heads + head) * VECS * CHUNK;
            vec[lane] = t < n ? expf(lf + before - after) : 1.0f;
            vec[2 * CHUNK + lane] = t < n ? expf(li - after) : 0.0f;
            vec[3 * CHUNK + lane] = expf(-after);
        }
    }
    for (int c = tid; c < p.copies; c += GATE_WAVES * KIPP_WAVE) m_all[(size_t)c * p.heads + head] = m;
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
    float* vec = p.vec + at * VECS * CHUNK;
    if (wave == 0) {
        // the wave with the fewest products below: D column by column, a lane a column
        const float* row = p.src + (size_t)(t0 + min(lane, m - 1)) * p.stride;
        const float g = lane >= m ? 1.0f : (MODE == MODE_DECAY ? p.decays[head] : (MODE == MODE_MLSTM ? vec[lane] : row[p.g_at + head]));
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
    constexpr int RUNS = runs_of(MODE, DT);
    f32x4 qk[RUNS][4], kk[RUNS][4];
#pragma unroll
    for (int h = 0; h < RUNS; ++h)
#pragma unroll
        for (int s = 0; s < 4; ++s) qk[h][s] = kk[h][s] = zero4();
    if (16 * wave < m) {
        const float* q_row = q + (size_t)(t0 + min(16 * wave + l16, m - 1)) * p.qk_stride + h4;
        const float* k_row = k + (size_t)(t0 + min(16 * wave + l16, m - 1)) * p.qk_stride + h4;
        const float* s_row[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) s_row[s] = k + (size_t)(t0 + min(16 * s + l16, m - 1)) * p.qk_stride + h4;
#pragma unroll(RUNS == 1 ? 2 : 1)
        for (int j0 = 0; j0 < D; j0 += 16 * RUNS)
#pragma unroll
            for (int h = 0; h < RUNS; ++h) {
                const int j = j0 + 16 * h;
                const f32x4 qv = *reinterpret_cast<const f32x4*>(q_row + j);
                const f32x4 kv = MODE == MODE_DELTA ? *reinterpret_cast<const f32x4*>(k_row + j) : zero4();
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    if (s <= wave) {
                        const f32x4 sv = *reinterpret_cast<const f32x4*>(s_row[s] + j);
                        qk[h][s] = mul16(qv, sv, qk[h][s]);
                        if (MODE == MODE_DELTA) kk[h][s] = mul16(kv, sv, kk[h][s]);
                    }
            }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (s > wave) continue;
        qk[0][s] = sum_runs(qk, s);
        if (MODE == MODE_DELTA) kk[0][s] = sum_runs(kk, s);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int t = 16 * wave + h4 + v, c = 16 * s + l16;
            const float decay = c <= t && t < m ? d_s[t][c] : 0.0f;
            a_out[t * CHUNK + c] = decay != 0.0f ? (MODE == MODE_MLSTM ? qk[0][s][v] * p.q_scale : qk[0][s][v]) * decay : 0.0f;
            if (MODE == MODE_DELTA) l_s[t][c] = c < t && decay != 0.0f ? beta_s[t] * decay * kk[0][s][v] : 0.0f;
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

template <bool B>
struct Bool {
    static constexpr bool value = B;
};

// What a wave needs in a chunk to sum o for 16 of its tokens (q, a, g, f), or to keep 16 DT rows of S and, for the delta rule, make R and U of 16
// tokens.  The delta rule's two share their places, which a wave uses in one way only.
template <int MODE, int DT>
struct Operands {
    static constexpr bool SHARED = MODE == MODE_DELTA;
    f32x4 kt[4 * DT], k[SHARED ? 4 * DT : 1], t[SHARED ? 4 : 1], e[4], v, g, b, f;
    f32x4 q_own[SHARED ? 1 : 4 * DT], a_own[SHARED ? 1 : 4];
    float g_last;
    __device__ __forceinline__ f32x4* q() { return SHARED ? kt : q_own; }
    __device__ __forceinline__ f32x4* a() { return SHARED ? t : a_own; }
};

// Eight waves: four keep S, four sum o.
template <int MODE, int DT>
__global__ void __launch_bounds__(2 * THREADS, 2) chunks_walk_kernel(const ChunkArgs p) {
    constexpr int D = 64 * DT, SP = D + 4;
    __shared__ __attribute__((aligned(16))) float s_s[2][COLS * SP];        // [chunk's parity][column][row]
    __shared__ __attribute__((aligned(16))) float u_s[2][COLS * UP];        // [chunk's parity][column][token]
    __shared__ __attribute__((aligned(16))) float r_s[MODE == MODE_DELTA ? COLS * UP : 4];
    const int head = blockIdx.y;
    const Portion portion = portion_of(p.q_len, p.entries, p.from, blockIdx.z);
    if (portion.entry < 0) return;          // uniform over the workgroup
    const int entry = portion.entry;
    const int lane = threadIdx.x & (KIPP_WAVE - 1), l16 = lane & 15, h4 = 4 * (lane >> 4);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KIPP_WAVE) & 3;
    const bool keeps = __builtin_amdgcn_readfirstlane(threadIdx.x / KIPP_WAVE) < 4;
    const int n = p.q_len[entry], first = p.q_start[entry];
    const int col = blockIdx.x * COLS + l16;
    const bool norm = MODE == MODE_MLSTM && col == p.dv;        // n: one more column of S, of values of one
    const bool live = col < p.dv || norm;
    const int own = 16 * wave;              // the wave's tokens of a chunk
    const int row0 = D / 4 * wave;          // its rows of S
    float* S_col = p.state + (size_t)p.slots[entry] * p.state_stride + row0 + h4 +
                   (norm ? p.n_at + (size_t)head * D : ((size_t)head * p.dv + (live ? col : 0)) * D);
    const float* q = p.q + (size_t)(head / p.qk_rep) * D;
    const float* k = p.k + (size_t)(head / p.qk_rep) * D;
    const float* v_src = p.src + p.v_at + (size_t)head * p.dv + (live && !norm ? col : 0);
    const int chunks = (n + CHUNK - 1) / CHUNK;

    // A chunk's operands are asked for as soon as the one before has used its own; always all of them (rows beyond the last token are the last
    // one's): behind a branch the compiler waits for everything that is on its way, so the last chunk, which asks for none, is code of its own.
    Operands<MODE, DT> x;
    f32x4 S[DT];
    auto vec_of = [&](int c) { return p.vec + ((size_t)(portion.base + c) * p.heads + head) * VECS * CHUNK; };
    auto own_rows = [&](int c, const float* from, f32x4* to) {          // of q or k
        const int m = min(CHUNK, n - c * CHUNK);
        const size_t row = (size_t)(first + c * CHUNK + min(own + l16, m - 1)) * p.qk_stride + h4;
#pragma unroll
        for (int j = 0; j < 4 * DT; ++j) to[j] = *reinterpret_cast<const f32x4*>(from + row + 16 * j);
    };
    auto square_of = [&](int c, const float* from, f32x4* to) {         // of A or T
        const float* row = from + ((size_t)(portion.base + c) * p.heads + head) * CHUNK * CHUNK + (own + l16) * CHUNK + h4;
#pragma unroll
        for (int j = 0; j < 4; ++j) to[j] = *reinterpret_cast<const f32x4*>(row + 16 * min(j, wave));       // (none above the diagonal)
    };
    auto gates_of = [&](int c) {
        x.g = *reinterpret_cast<const f32x4*>(vec_of(c) + own + h4);
        if (MODE == MODE_MLSTM) x.f = *reinterpret_cast<const f32x4*>(vec_of(c) + 3 * CHUNK + own + h4);
    };
    auto values_of = [&](int c) {
        c = min(c, chunks - 1);
        const int m = min(CHUNK, n - c * CHUNK), t0 = first + c * CHUNK;
#pragma unroll
        for (int i = 0; i < 4; ++i) x.v[i] = v_src[(size_t)(t0 + min(own + h4 + i, m - 1)) * p.stride];
        if (MODE == MODE_DELTA) x.g = *reinterpret_cast<const f32x4*>(vec_of(c) + own + h4);
        if (MODE == MODE_DELTA || MODE == MODE_MLSTM) x.b = *reinterpret_cast<const f32x4*>(vec_of(c) + 2 * CHUNK + own + h4);
    };
    auto keys_of = [&](int c) {
        const int m = min(CHUNK, n - c * CHUNK), t0 = first + c * CHUNK;
        const float* vec = vec_of(c);
        x.g_last = vec[CHUNK - 1];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            x.e[j] = *reinterpret_cast<const f32x4*>(vec + CHUNK + 16 * j + h4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float* k_row = k + (size_t)(t0 + min(16 * j + h4 + i, m - 1)) * p.qk_stride + row0 + l16;
#pragma unroll
                for (int a = 0; a < DT; ++a) x.kt[4 * a + j][i] = k_row[16 * a];
            }
        }
    };
    auto show_state = [&](int c) {
#pragma unroll
        for (int a = 0; a < DT; ++a) *reinterpret_cast<f32x4*>(&s_s[c & 1][l16 * SP + row0 + 16 * a + h4]) = S[a];
    };
    auto show_values = [&](int c) {         // U of the wave's tokens, where it does not hang on S
        const int m = min(CHUNK, n - c * CHUNK);
        f32x4 u = x.v;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (own + h4 + i >= m) u[i] = 0.0f;
            if (MODE == MODE_DECAY) u[i] = silu_f(u[i]);        // silu(0) = 0
            if (MODE == MODE_MLSTM) u[i] = x.b[i] * (norm ? 1.0f : u[i]);       // a gate of zero beyond the last token
        }
        *reinterpret_cast<f32x4*>(&u_s[c & 1][l16 * UP + own + h4]) = u;
    };
    auto values_shown = [&](int c, int m, f32x4 (&u)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (16 * j < m) u[j] = *reinterpret_cast<const f32x4*>(&u_s[c & 1][l16 * UP + 16 * j + h4]);
    };
    // the 16 columns of S against the wave's rows of q or k
    auto with_state = [&](int c, const f32x4* rows) {
        constexpr int RUNS = runs_of(MODE, DT);
        f32x4 sum[RUNS][1];
#pragma unroll
        for (int h = 0; h < RUNS; ++h) sum[h][0] = zero4();
#pragma unroll
        for (int j = 0; j < 4 * DT; j += RUNS) {
            f32x4 sv[RUNS];
#pragma unroll
            for (int h = 0; h < RUNS; ++h) sv[h] = *reinterpret_cast<const f32x4*>(&s_s[c & 1][l16 * SP + 16 * (j + h) + h4]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int h = 0; h < RUNS; ++h) sum[h][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(rows[j + h][i], sv[h][i], sum[h][0], 0, 0, 0);
        }
        return sum_runs(sum, 0);
    };

    f32x4 u_all[4];         // (the delta rule's, in one place for both kinds of waves: 14 registers fewer, and next to no spills at keys of 256)
    // ---- S: through a chunk, and shown for the next one
    auto begin_keeping = [&]() {
#pragma unroll
        for (int a = 0; a < DT; ++a) S[a] = live ? *reinterpret_cast<const f32x4*>(S_col + 16 * a) : zero4();
        values_of(0);
        if (MODE == MODE_DELTA) {
            own_rows(0, k, x.k);
            square_of(0, p.t, x.t);
        }
        keys_of(0);
        show_state(0);
        if (MODE != MODE_DELTA) {
            show_values(0);
            values_of(1);
        }
    };
    auto keep = [&](int c, auto there_are_more) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(there_are_more)::value;
        const int m = min(CHUNK, n - c * CHUNK);
        if constexpr (MODE == MODE_DELTA) {
            const bool mine = own < m;
            if (mine) {
                const f32x4 read = with_state(c, x.k);
                f32x4 r;
#pragma unroll
                for (int i = 0; i < 4; ++i) r[i] = own + h4 + i < m ? x.b[i] * (x.v[i] - x.g[i] * read[i]) : 0.0f;
                *reinterpret_cast<f32x4*>(r_s + l16 * UP + own + h4) = r;
            }
            if (MORE) {
                own_rows(c + 1, k, x.k);
                values_of(c + 1);
            }
            __syncthreads();
            if (mine) {
                f32x4 w = zero4();
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (j <= wave) w = mul16(x.t[j], *reinterpret_cast<const f32x4*>(r_s + l16 * UP + 16 * j + h4), w);
                *reinterpret_cast<f32x4*>(&u_s[c & 1][l16 * UP + own + h4]) = w;
            }
            if (MORE) square_of(c + 1, p.t, x.t);
            __syncthreads();
        }
        f32x4 u_own[4];
        f32x4 (&u)[4] = MODE == MODE_DELTA ? u_all : u_own;
        values_shown(c, m, u);
#pragma unroll
        for (int a = 0; a < DT; ++a) S[a] *= x.g_last;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (16 * j >= m) continue;
            const f32x4 eu = u[j] * x.e[j];
#pragma unroll
            for (int a = 0; a < DT; ++a) S[a] = mul16(x.kt[4 * a + j], eu, S[a]);
        }
        if (MORE) {
            keys_of(c + 1);
            show_state(c + 1);
            if (MODE != MODE_DELTA) {
                show_values(c + 1);
                values_of(c + 2);
            }
        }
    };
    auto end_keeping = [&]() {
        if (!live) return;
        for (int c = 0; c < (norm ? p.copies : 1); ++c)         // every copy of n
#pragma unroll
            for (int a = 0; a < DT; ++a) *reinterpret_cast<f32x4*>(S_col + (size_t)c * p.heads * D + 16 * a) = S[a];
    };
    // ---- o of a chunk
    auto begin_summing = [&]() {
        own_rows(0, q, x.q());
        gates_of(0);
        square_of(0, p.a, x.a());
    };
    auto sum_up = [&](int c, auto there_are_more) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(there_are_more)::value;
        const int m = min(CHUNK, n - c * CHUNK);
        const bool mine = own < m;
        f32x4 inter = zero4();
        if (mine) inter = with_state(c, x.q());
        if (MORE) own_rows(c + 1, q, x.q());
        if (MODE == MODE_DELTA) {
            __syncthreads();
            __syncthreads();
        }
        f32x4 u_own[4];
        f32x4 (&u)[4] = MODE == MODE_DELTA ? u_all : u_own;
        values_shown(c, m, u);
        if (mine) {
            f32x4 o = MODE == MODE_MLSTM ? zero4() : inter * x.g;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j <= wave) o = mul16(x.a()[j], u[j], o);
            if (MODE == MODE_MLSTM) o += inter * (x.g * p.q_scale);
            if (norm) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (own + h4 + i < m) p.den[(size_t)(first + c * CHUNK + own + h4 + i) * p.heads + head] = fmaxf(fabsf(o[i]), x.f[i]) + 1e-6f;
            } else if (live) {
                float* o_at = p.o_raw + (size_t)(first + c * CHUNK + own + h4) * p.heads * p.dv + (size_t)head * p.dv + col;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (own + h4 + i < m) o_at[(size_t)i * p.heads * p.dv] = o[i];
            }
        }
        if (MORE) {
            gates_of(c + 1);
            square_of(c + 1, p.a, x.a());
        }
    };

    // All waves meet once a chunk (S ahead of it is shown, and U where that does not hang on S), and for the delta rule behind R and behind U.
    if (keeps) {
        begin_keeping();
        for (int c = 0; c + 1 < chunks; ++c) {
            __syncthreads();
            keep(c, Bool<true>{});
        }
        __syncthreads();
        keep(chunks - 1, Bool<false>{});
        end_keeping();
    } else {
        begin_summing();
        for (int c = 0; c + 1 < chunks; ++c) {
            __syncthreads();
            sum_up(c, Bool<true>{});
        }
        __syncthreads();
        sum_up(chunks - 1, Bool<false>{});
    }
}

// The walk of many short portions: four waves that do both, one behind the other (`walk_waves` says when).  Its workgroups are half as large, and more
// of them than the chip has places for run beside each other; where they do not, a chunk's chain is what counts, and the eight waves are faster.
// What one of four waves multiplies in a chunk: its own rows of q, k, T and A, its rows of K^T, the values of its tokens.
template <int MODE, int DT>
struct FourOperands {
    f32x4 q[4 * DT], k[MODE == MODE_DELTA ? 4 * DT : 1], a[4], t[MODE == MODE_DELTA ? 4 : 1], e[4], kt[DT][4], v, g, b, f;
    float g_last;
};

template <int MODE, int DT>
__global__ void __launch_bounds__(THREADS) chunks_walk_four_kernel(const ChunkArgs p) {
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
    const bool norm = MODE == MODE_MLSTM && col == p.dv;        // n: one more column of S, of values of one
    const bool live = col < p.dv || norm;
    const int own = 16 * wave;              // the wave's tokens of a chunk
    const int row0 = D / 4 * wave;          // its rows of S
    float* S_col = p.state + (size_t)p.slots[entry] * p.state_stride + row0 + h4 +
                   (norm ? p.n_at + (size_t)head * D : ((size_t)head * p.dv + (live ? col : 0)) * D);
    const float* q = p.q + (size_t)(head / p.qk_rep) * D;
    const float* k = p.k + (size_t)(head / p.qk_rep) * D;
    const float* v_src = p.src + p.v_at + (size_t)head * p.dv + (live && !norm ? col : 0);

    f32x4 S[DT];
#pragma unroll
    for (int a = 0; a < DT; ++a) S[a] = live ? *reinterpret_cast<const f32x4*>(S_col + 16 * a) : zero4();

    // The next chunk's operands are asked for as soon as this one's have been used.  (A second set of registers, asked for
    // a whole chunk ahead, changed nothing and left a compute unit one workgroup instead of two.)
    FourOperands<MODE, DT> x;
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
        const float* vec = p.vec + at * VECS * CHUNK;
        if (own < m) {
            const float* a_row = p.a + at * CHUNK * CHUNK + (own + l16) * CHUNK + h4;
            const float* t_row = p.t + at * CHUNK * CHUNK + (own + l16) * CHUNK + h4;
#pragma unroll
            for (int i = 0; i < 4; ++i) x.v[i] = own + h4 + i < m ? v_src[(size_t)(t0 + own + h4 + i) * p.stride] : 0.0f;
            x.g = *reinterpret_cast<const f32x4*>(vec + own + h4);
            if (MODE == MODE_DELTA || MODE == MODE_MLSTM) x.b = *reinterpret_cast<const f32x4*>(vec + 2 * CHUNK + own + h4);
            if (MODE == MODE_MLSTM) x.f = *reinterpret_cast<const f32x4*>(vec + 3 * CHUNK + own + h4);
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
            constexpr int RUNS = runs_of(MODE, DT);
            f32x4 in[RUNS][1], rd[RUNS][1];
#pragma unroll
            for (int h = 0; h < RUNS; ++h) in[h][0] = rd[h][0] = zero4();
#pragma unroll
            for (int j = 0; j < 4 * DT; j += RUNS) {
                f32x4 sv[RUNS];
#pragma unroll
                for (int h = 0; h < RUNS; ++h) sv[h] = *reinterpret_cast<const f32x4*>(&s_s[l16 * SP + 16 * (j + h) + h4]);
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int h = 0; h < RUNS; ++h) {
                        in[h][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[j + h][i], sv[h][i], in[h][0], 0, 0, 0);
                        if (MODE == MODE_DELTA) rd[h][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[j + h][i], sv[h][i], rd[h][0], 0, 0, 0);
                    }
            }
            inter = sum_runs(in, 0);
            if (MODE == MODE_DELTA) read = sum_runs(rd, 0);
            f32x4 u = x.v;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (MODE == MODE_DECAY) u[i] = silu_f(u[i]);        // silu(0) = 0
                if (MODE == MODE_MLSTM) u[i] = x.b[i] * (norm ? 1.0f : u[i]);       // a gate of zero beyond the last token
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
            f32x4 o = MODE == MODE_MLSTM ? zero4() : inter * x.g;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j <= wave) o = mul16(x.a[j], u[j], o);
            if (MODE == MODE_MLSTM) o += inter * (x.g * p.q_scale);
            if (norm) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (own + h4 + i < m) p.den[(size_t)(first + c * CHUNK + own + h4 + i) * p.heads + head] = fmaxf(fabsf(o[i]), x.f[i]) + 1e-6f;
            } else if (live) {
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
        for (int c = 0; c < (norm ? p.copies : 1); ++c)         // every copy of n
#pragma unroll
            for (int a = 0; a < DT; ++a) *reinterpret_cast<f32x4*>(S_col + (size_t)c * p.heads * D + 16 * a) = S[a];
    }
}

extern "C" {

// Chunks that `tokens` tokens of `portions` entries make at most, whatever their lengths.
static long long chunk_count(int tokens, int portions) { return (long long)tokens / CHUNK + portions; }

// Floats of work space, or 0 where this kernel does not take the sizes: keys of 64, 128, 192 or 256 numbers.
long long kipp_matrix_chunks_work(int mode, int tokens, int portions, int heads, int d) {
    if (mode < MODE_DECAY || mode > MODE_MLSTM || tokens <= 0 || portions <= 0 || heads <= 0 || d <= 0 || d % 64 || d > 256) return 0;
    const long long each = (mode == MODE_DELTA ? 2 : 1) * CHUNK * CHUNK + VECS * CHUNK;
    return chunk_count(tokens, portions) * heads * each + (mode == MODE_DECAY ? (long long)tokens * 2 * heads * d : 0);
}

}  // extern "C"

// The work space's parts, and the launches behind what a mode puts ahead of them.
static void lay_out(ChunkArgs& p, int mode, long long slots_all, float* work) {
    p.a = work;
    p.t = mode == MODE_DELTA ? p.a + slots_all * CHUNK * CHUNK : p.a;
    p.vec = p.t + slots_all * CHUNK * CHUNK;
}

// Eight waves a workgroup of the walk, or four.  Eight shorten the chain of a chunk; four start and end sooner and fit twice or more often on a
// compute unit (registers; from keys of 256 on, 128 for the delta rule, they fit once only and eight always win).  So four have many short
// portions: more workgroups than compute units (fixed decays of short keys, whose values are work ahead of the chain: three or four to a unit) and two
// chunks a portion ahead for every one a unit.  Calls of four / eight waves, us: 64 portions of 80 tokens, 16 heads of 192 x 128, a decay a token 225 / 307, an mLSTM 347 /
// 442; delta rule, 32 heads of 64 x 64, 64 portions of 64 176 / 235, 4 of 64 30.5 / 32.4; 4 of 80, 16 heads of 128 x 128, a decay a token 22 / 25; and the other
// way 16 heads of 128 x 128, 10 portions of 1,000 tokens 12 % and one of 2,048 26 % less with eight.  1,350 calls of both, from 16 to 12,800 workgroups and 64 to 2,048
// tokens: this choice is 0.2 % over the faster one in the mean, eight waves up to 1,024 workgroups (keys of 128) or always were 2.6.
static int walk_waves(int mode, int dt, long long groups, int chunks) {
    if (dt >= (mode == MODE_DELTA ? 2 : 4)) return 8;
    const int units = 256, places = dt == 1 && (mode == MODE_DECAY || mode == MODE_GATED) ? 2 * units : units;        // of eight waves: two fit where they have 128 registers
    const int always = mode != MODE_DECAY || dt > 2 ? units : (dt == 1 ? 4 * units : 3 * units);
    // (an mLSTM's eight waves have 130 registers with keys of 64: what is one round of four waves is two of eight)
    if (mode == MODE_MLSTM && dt == 1 && groups > units && groups <= 2 * units) return 4;
    return groups <= always || groups <= (long long)places * (chunks - 2) ? 8 : 4;
}

template <int MODE, int DT>
static void launch_chunks(const ChunkArgs& p, int longest, int portions, hipStream_t stream) {
    const int cols = p.dv + (MODE == MODE_MLSTM ? 1 : 0);
    const dim3 prepare((longest + CHUNK - 1) / CHUNK, p.heads, portions), walk((cols + COLS - 1) / COLS, p.heads, portions), block(THREADS);
    hipLaunchKernelGGL((chunks_prepare_kernel<MODE, DT>), prepare, block, 0, stream, p);
    if constexpr (DT < (MODE == MODE_DELTA ? 2 : 4)) {
        if (walk_waves(MODE, DT, (long long)walk.x * walk.y * walk.z, (longest + CHUNK - 1) / CHUNK) == 4) {
            hipLaunchKernelGGL((chunks_walk_four_kernel<MODE, DT>), walk, block, 0, stream, p);
            return;
        }
    }
    hipLaunchKernelGGL((chunks_walk_kernel<MODE, DT>), walk, dim3(2 * THREADS), 0, stream, p);
}

// Waves of a workgroup of the walk, 4 or 8, as a launch of these sizes has them; 0 where chunks do not take them.
extern "C" int kipp_matrix_chunks_waves(int mode, int heads, int d, int dv, int longest, int portions) {
    if (kipp_matrix_chunks_work(mode, 1, 1, heads, d) == 0 || dv <= 0 || longest <= 0 || portions <= 0) return 0;
    const int cols = dv + (mode == MODE_MLSTM ? 1 : 0);
    return walk_waves(mode, d / 64, (long long)((cols + COLS - 1) / COLS) * heads * portions, (longest + CHUNK - 1) / CHUNK);
}

template <int MODE>
static void launch_mode(const ChunkArgs& p, int longest, int portions, hipStream_t stream) {
    if (p.d == 64) launch_chunks<MODE, 1>(p, longest, portions, stream);
    else if (p.d == 128) launch_chunks<MODE, 2>(p, longest, portions, stream);
    else if (p.d == 192) launch_chunks<MODE, 3>(p, longest, portions, stream);
    else launch_chunks<MODE, 4>(p, longest, portions, stream);
}

extern "C" {

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
    if (mode == MODE_MLSTM || need == 0 || work_floats < need || longest <= 0 || qk_rep <= 0 || heads % qk_rep || dv <= 0) return -1;
    if (state_stride < (size_t)heads * d * dv || (state_stride & 3) || (stride & 3) || (q_at & 3) || (k_at & 3)) return -1;
    if (((uintptr_t)src | (uintptr_t)state | (uintptr_t)work) & 15) return -1;
    ChunkArgs p = {};
    const long long slots_all = chunk_count(tokens, portions) * heads;
    lay_out(p, mode, slots_all, work);
    p.q = src + q_at;
    p.k = src + k_at;
    p.qk_stride = stride;
    if (mode == MODE_DECAY) {
        if (q_at != 0 || k_at != heads * d || qk_rep != 1) return -1;
        float* ready = p.vec + slots_all * VECS * CHUNK;
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
    p.d = d;
    p.dv = dv;
    p.entries = entries;
    p.from = from;
    p.portions = portions;
    if (mode == MODE_DECAY) launch_mode<MODE_DECAY>(p, longest, portions, stream);
    else if (mode == MODE_DELTA) launch_mode<MODE_DELTA>(p, longest, portions, stream);
    else launch_mode<MODE_GATED>(p, longest, portions, stream);
    return KIPP_LAUNCH_CHECK();
}

// The same for an mLSTM: `proj` and `state` as `kipp_mlstm_scan` has them, `copies` of n and m in a slot.  o_raw receives the sums before they
// are divided, den [tokens][heads] what they are to be divided by (ones for the entries of fewer than `from` tokens, at most 1,024, which
// are left to the walk).
int kipp_mlstm_chunks(const float* proj, int stride, const float* bias_i, const float* bias_f, float cap, float* state, size_t state_stride,
                      int copies, const int32_t* q_start, const int32_t* q_len, const int32_t* slots, float* o_raw, float* den, int tokens, int entries,
                      int heads, int d, int dv, int longest, int from, int portions, float* work, long long work_floats, hipStream_t stream) {
    if (entries <= 0 || tokens <= 0 || portions <= 0) return 0;
    const long long need = kipp_matrix_chunks_work(MODE_MLSTM, tokens, portions, heads, d);
    if (need == 0 || work_floats < need || longest <= 0 || dv <= 0 || copies <= 0 || from > GATE_WAVES * KIPP_WAVE || !(cap > 0.0f)) return -1;
    if (stride < 2 * heads * d + 2 * heads * dv + 2 * heads || state_stride < (size_t)heads * d * dv + (size_t)copies * (heads * d + heads)) return -1;
    if ((state_stride & 3) || (stride & 3) || (((uintptr_t)proj | (uintptr_t)state | (uintptr_t)work) & 15)) return -1;
    ChunkArgs p = {};
    lay_out(p, MODE_MLSTM, chunk_count(tokens, portions) * heads, work);
    p.q = proj;
    p.k = proj + heads * d;
    p.qk_stride = stride;
    p.src = proj;
    p.stride = stride;
    p.v_at = 2 * heads * d;
    p.i_at = 2 * heads * d + 2 * heads * dv;
    p.f_at = p.i_at + heads;
    p.bias_i = bias_i;
    p.bias_f = bias_f;
    p.cap = cap;
    p.q_scale = 1.0f / sqrtf((float)d);
    p.state = state;
    p.state_stride = state_stride;
    p.n_at = heads * d * dv;
    p.copies = copies;
    p.q_start = q_start;
    p.q_len = q_len;
    p.slots = slots;
    p.o_raw = o_raw;
    p.den = den;
    p.heads = heads;
    p.qk_rep = 1;
    p.d = d;
    p.dv = dv;
    p.entries = entries;
    p.from = from;
    p.portions = portions;
    hipLaunchKernelGGL(chunks_gates_kernel, dim3(heads, entries), dim3(GATE_WAVES * KIPP_WAVE), 0, stream, p);
    launch_mode<MODE_MLSTM>(p, longest, portions, stream);
    return KIPP_LAUNCH_CHECK();
}

}  // extern "C"
