// Attention of single tokens over rows that are key and value at once: one row of D numbers a token in the paged cache, which every
// query head reads (a latent's cache), bfloat16.
//
//   scores   a workgroup takes (a run of the token's keys, token), keys 64 at a time: their rows go from memory through registers into
//            LDS, once, as keys and as values; a wave scores 16 keys against all heads on the matrix cores (the heads are the
//            product's columns), masks them and takes their weights against the run's maximum so far;
//   values   a wave multiplies the float32 weights with every fourth 32 columns of the rows on the float32 matrix instruction: the
//            weights are not rounded;
//   merge    a second kernel adds the runs in order.
//
// Bound by latencies (the pages, then the rows, then a chain of LDS exchanges), so a run is one tile of 64 keys until the runs fill the
// chip twice.  8 tokens behind about 200 keys, 16 heads, D = 256: 6.9 + 4.7 us (1,500 keys 17.8 in all); the kernel for grouped heads, which multiplies
// weights and values by plain FMA for 16 heads and takes 192 keys or more a workgroup, 42.6 us (44).  Error against 64 bits the
// same in both, 0.00165 of the result: its rounding.
#include "common.h"
#include <math.h>

#define SH_KEYS 64
#define SH_HEADS 16                 // columns of the products: query heads at most
#define SH_WAVES 4
#define SH_THREADS (SH_WAVES * KIPP_WAVE)
#define SH_MAX_RUNS 64

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

union Frag {
    u32x4 u;
    bf16x8 v;
};

// How the keys of the token at `pos` are cut: tiles of 64 (absolute index) from the first that it sees, in runs of `chunk` of them.
__device__ __forceinline__ void run_of(int pos, int window, int n_runs, int& lo, int& tile0, int& tiles, int& chunk) {
    lo = window > 0 ? max(0, pos - window + 1) : 0;
    tile0 = lo / SH_KEYS;
    tiles = pos / SH_KEYS - tile0 + 1;
    chunk = (tiles + n_runs - 1) / n_runs;
}

// STEPS: 32 columns each, of which a row has D (a multiple of 16).  part_acc: float32 [tokens][runs][16][D]; part_ml [tokens][runs][16][2].
template <int STEPS>
__global__ void __launch_bounds__(SH_THREADS) attention_shared_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ cache, float* __restrict__ part_acc, float* __restrict__ part_ml,
    const int32_t* __restrict__ rows, const int32_t* __restrict__ positions, const int32_t* __restrict__ seq_of_token,
    const int32_t* __restrict__ block_table, int max_blocks, int heads, int d, int page_shift, float scale_log2e, int window) {
    constexpr int PITCH = 32 * STEPS + 8;           // of a row in LDS (the pad spreads the banks)
    constexpr int CHUNKS = 4 * STEPS;               // 16-byte chunks of a row
    __shared__ __attribute__((aligned(16))) bf16_t s_rows[SH_KEYS * PITCH];
    __shared__ float s_p[SH_KEYS][SH_HEADS];
    __shared__ float s_top[SH_WAVES][SH_HEADS], s_sum[SH_WAVES][SH_HEADS], s_shrink[SH_HEADS];
    const int token = blockIdx.y, run = blockIdx.x, n_runs = gridDim.x;
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, quarter = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = rows[token], pos = positions[row];
    const int32_t* table = block_table + (size_t)seq_of_token[row] * max_blocks;
    int lo, tile0, tiles, chunk;
    run_of(pos, window, n_runs, lo, tile0, tiles, chunk);
    const int begin = min(tiles, run * chunk), end = min(tiles, begin + chunk);
    if (begin >= end) return;                       // the merge counts the runs by the same rule
    const int page_mask = (1 << page_shift) - 1;

    // this thread's chunks of a tile: row (tid + 256 j) / CHUNKS, chunk (tid + 256 j) % CHUNKS
    u32x4 held[STEPS];
    auto ask = [&](int tile) {
        int32_t page[STEPS];
#pragma unroll
        for (int j = 0; j < STEPS; ++j) page[j] = table[min(max((tile0 + tile) * SH_KEYS + (tid + SH_THREADS * j) / CHUNKS, lo), pos) >> page_shift];
#pragma unroll
        for (int j = 0; j < STEPS; ++j) {
            const int i = tid + SH_THREADS * j;
            const int key = min(max((tile0 + tile) * SH_KEYS + i / CHUNKS, lo), pos);       // keys that are not seen: one that is (masked below)
            const int col = 8 * (i % CHUNKS);
            held[j] = *(const u32x4*)(cache + (((size_t)page[j] << page_shift) + (key & page_mask)) * d + min(col, d - 8));
            if (col >= d) held[j] = (u32x4){0u, 0u, 0u, 0u};
        }
    };
    ask(begin);
    Frag qf[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        const int col = 32 * s + 8 * quarter;
        qf[s].u = *(const u32x4*)(q + ((size_t)row * heads + min(l16, heads - 1)) * d + min(col, d - 8));
        if (col >= d) qf[s].u = (u32x4){0u, 0u, 0u, 0u};
    }
    float top = -INFINITY, sum = 0.0f;              // of head l16; the sum over this lane's keys alone
    constexpr int BLOCKS = (STEPS + SH_WAVES - 1) / SH_WAVES;       // 32-column blocks of a wave: wave, wave + 4, ..
    f32x4 acc[BLOCKS][2];                           // [even, odd columns]: heads 4 quarter + v, column 32 block + 2 l16 (+ 1)
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) acc[b][0] = acc[b][1] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    for (int tile = begin; tile < end; ++tile) {
        if (tile > begin) __syncthreads();          // every wave is done with the tile before
#pragma unroll
        for (int j = 0; j < STEPS; ++j) {
            const int i = tid + SH_THREADS * j;
            *(u32x4*)(s_rows + (i / CHUNKS) * PITCH + 8 * (i % CHUNKS)) = held[j];
        }
        __syncthreads();
        if (tile + 1 < end) ask(tile + 1);
        f32x4 s4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            Frag kf;
            kf.u = *(const u32x4*)(s_rows + (16 * wave + l16) * PITCH + 32 * s + 8 * quarter);
            s4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf.v, qf[s].v, s4, 0, 0, 0);
        }
        float here = -INFINITY;
#pragma unroll
        for (int v = 0; v < 4; ++v) {               // s4[v]: key 16 wave + 4 quarter + v, head l16
            const int key = (tile0 + tile) * SH_KEYS + 16 * wave + 4 * quarter + v;
            s4[v] = key >= lo && key <= pos ? s4[v] * scale_log2e : -INFINITY;
            here = fmaxf(here, s4[v]);
        }
        here = fmaxf(here, __shfl_xor(here, 16, KIPP_WAVE));
        here = fmaxf(here, __shfl_xor(here, 32, KIPP_WAVE));
        if (quarter == 0) s_top[wave][l16] = here;
        __syncthreads();
        float next = top;
#pragma unroll
        for (int w = 0; w < SH_WAVES; ++w) next = fmaxf(next, s_top[w][l16]);
        const float shrink = top == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(top - next);
        sum *= shrink;
        top = next;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float p = s4[v] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(s4[v] - top);
            sum += p;
            s_p[16 * wave + 4 * quarter + v][l16] = p;
        }
        if (wave == 0 && quarter == 0) s_shrink[l16] = shrink;
        __syncthreads();
        float pf[SH_KEYS / 4];                      // weights of head l16, keys 4 s + quarter
#pragma unroll
        for (int s = 0; s < SH_KEYS / 4; ++s) pf[s] = s_p[4 * s + quarter][l16];
        f32x4 keep;
#pragma unroll
        for (int v = 0; v < 4; ++v) keep[v] = s_shrink[4 * quarter + v];
#pragma unroll
        for (int b = 0; b < BLOCKS; ++b) {
            const int block = wave + SH_WAVES * b;
            if (block >= STEPS) continue;           // uniform over the wave
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                acc[b][0][v] *= keep[v];
                acc[b][1][v] *= keep[v];
            }
#pragma unroll
            for (int s = 0; s < SH_KEYS / 4; ++s) {
                const uint32_t two = *(const uint32_t*)(s_rows + (4 * s + quarter) * PITCH + 32 * block + 2 * l16);
                acc[b][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(pf[s], __uint_as_float(two << 16), acc[b][0], 0, 0, 0);
                acc[b][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(pf[s], __uint_as_float(two & 0xffff0000u), acc[b][1], 0, 0, 0);
            }
        }
    }
    sum += __shfl_xor(sum, 16, KIPP_WAVE);
    sum += __shfl_xor(sum, 32, KIPP_WAVE);
    if (quarter == 0) s_sum[wave][l16] = sum;
    __syncthreads();
    const size_t slot = ((size_t)token * n_runs + run) * SH_HEADS;
    if (wave == 0 && quarter == 0) {
        float total = 0.0f;
#pragma unroll
        for (int w = 0; w < SH_WAVES; ++w) total += s_sum[w][l16];
        *(float2*)(part_ml + (slot + l16) * 2) = make_float2(top, total);
    }
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) {
        const int col = 32 * (wave + SH_WAVES * b) + 2 * l16;
        if (col >= d) continue;                     // d is even: both columns or none
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (4 * quarter + v < heads) *(float2*)(part_acc + (slot + 4 * quarter + v) * d + col) = make_float2(acc[b][0][v], acc[b][1][v]);
    }
}

// out[row][head][d] = the runs' sums, each times 2^(its maximum - the largest), added in order, over the same of their denominators.
__global__ void __launch_bounds__(KIPP_WAVE) attention_shared_merge_kernel(
    const float* __restrict__ part_acc, const float* __restrict__ part_ml, bf16_t* __restrict__ out, const int32_t* __restrict__ rows,
    const int32_t* __restrict__ positions, int heads, int d, int window, int n_runs) {
    const int head = blockIdx.x, token = blockIdx.y, lane = threadIdx.x;
    const int row = rows[token];
    int lo, tile0, tiles, chunk;
    run_of(positions[row], window, n_runs, lo, tile0, tiles, chunk);
    const int used = (tiles + chunk - 1) / chunk;
    const size_t slot0 = (size_t)token * n_runs * SH_HEADS + head;
    constexpr int COLS = 4, AT_ONCE = 4;            // of up to 256 columns a lane takes 4, side by side
    // (a lane holds one run's numbers: at most SH_MAX_RUNS = 64 of them)
    const float2 ml = lane < used ? *(const float2*)(part_ml + (slot0 + (size_t)lane * SH_HEADS) * 2) : make_float2(-INFINITY, 0.0f);
    const float m = wave_max(ml.x);
    const float w = lane < used ? __builtin_amdgcn_exp2f(ml.x - m) : 0.0f;
    const int col = COLS * lane, from = min(col, d - COLS);        // d is a multiple of 16; the loop is every lane's: its numbers are read across lanes
    float a[COLS] = {0.0f, 0.0f, 0.0f, 0.0f}, denom = 0.0f;
    for (int r0 = 0; r0 < used; r0 += AT_ONCE) {
        f32x4 v[AT_ONCE];
#pragma unroll
        for (int u = 0; u < AT_ONCE; ++u) v[u] = *(const f32x4*)(part_acc + (slot0 + (size_t)min(r0 + u, used - 1) * SH_HEADS) * d + from);
#pragma unroll
        for (int u = 0; u < AT_ONCE; ++u) {
            if (r0 + u >= used) break;
            const float wr = __shfl(w, r0 + u, KIPP_WAVE);
            denom += wr * __shfl(ml.y, r0 + u, KIPP_WAVE);
#pragma unroll
            for (int c = 0; c < COLS; ++c) a[c] += wr * v[u][c];
        }
    }
    if (col < d) {
        uint2 packed;
        packed.x = (uint32_t)f32_to_bf16(a[0] / denom) | ((uint32_t)f32_to_bf16(a[1] / denom) << 16);
        packed.y = (uint32_t)f32_to_bf16(a[2] / denom) | ((uint32_t)f32_to_bf16(a[3] / denom) << 16);
        *(uint2*)(out + ((size_t)row * heads + head) * d + col) = packed;
    }
}

extern "C" {

// Rows rows[i] of the batch, i < n_tokens: out [batch rows][heads][d] over cache [pages][1][page][d] (keys and values).  part_acc: float32
// [n_tokens][n_runs][16][d], part_ml: [n_tokens][n_runs][16][2].  d a multiple of 16 up to 256, at most 16 heads, pages of a power of two.
int kipp_attention_shared(const void* q, const void* cache, void* out, float* part_acc, float* part_ml, const int32_t* rows, int n_tokens,
                          const int32_t* positions, const int32_t* seq_of_token, const int32_t* block_table, int max_blocks, int heads, int d,
                          int page, float scale, int window, int n_runs, hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (d <= 0 || d % 16 || d > 256 || heads <= 0 || heads > SH_HEADS) return -1;
    if (page <= 0 || (page & (page - 1)) || n_runs < 1 || n_runs > SH_MAX_RUNS) return -2;
    const float scale_log2e = scale * 1.4426950408889634f;
    const int shift = __builtin_ctz(page);
#define KIPP_SHARED(STEPS)                                                                                                              \
    case STEPS:                                                                                                                        \
        hipLaunchKernelGGL(attention_shared_kernel<STEPS>, dim3(n_runs, n_tokens), dim3(SH_THREADS), 0, stream, (const bf16_t*)q,        \
                           (const bf16_t*)cache, part_acc, part_ml, rows, positions, seq_of_token, block_table, max_blocks, heads, d, shift, \
                           scale_log2e, window);                                                                                       \
        break
    switch ((d + 31) / 32) {
        KIPP_SHARED(1);
        KIPP_SHARED(2);
        KIPP_SHARED(3);
        KIPP_SHARED(4);
        KIPP_SHARED(5);
        KIPP_SHARED(6);
        KIPP_SHARED(7);
        KIPP_SHARED(8);
    }
#undef KIPP_SHARED
    hipLaunchKernelGGL(attention_shared_merge_kernel, dim3(heads, n_tokens), dim3(KIPP_WAVE), 0, stream, (const float*)part_acc,
                       (const float*)part_ml, (bf16_t*)out, rows, positions, heads, d, window, n_runs);
    return KIPP_LAUNCH_CHECK();
}

}  // extern "C"
