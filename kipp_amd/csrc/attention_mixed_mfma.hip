// Attention whose softmax weights are mixed across heads, on the matrix cores (bfloat16 storage, float32
// arithmetic around the products).  The formulas are those at the head of attention_mixed.hip; built for one key
// size HEAD_DIM (a multiple of 32), one value size V_DIM (a multiple of 16) and HPW heads a wave (up to 8 HPW heads);
// SHARED_KV says that a wave's heads all read one key/value head, whose keys and values it then loads once.
//
// Mixing the heads' weights needs every head's FINAL weight of a (query, key) pair in one place, so the softmax
// cannot be rescaled on the way as flash attention does.  The work is therefore cut into items (a tile of up to 16
// query rows of one entry, a run of its keys) and done in two walks over the keys:
//
//   mixed_stats_kernel    scores of all heads, each lane keeping a running maximum and sum of its own keys;
//                         an item leaves (maximum, sum) of every (head, row);
//   mixed_values_kernel   merges the items' statistics of its tile (the sink joins here), then, 32 keys at a time:
//                         1. scores again, weights p = exp(s - M) / L, final, into LDS as [row][key][head],
//                            split into two bfloat16 halves (hi + lo carries 16 bits of mantissa);
//                         2. p' = mix . p on the matrix cores, contraction over heads, into LDS as [head][row][key];
//                         3. O^T[dv][row] += V^T . p'^T, the values read as they lie in the cache: the cache keeps
//                            them transposed inside a page, [page][kv head][dv][slot], so eight keys of one value
//                            column are sixteen contiguous bytes.
//                         A tile whose keys are one run writes gate * O as bfloat16; otherwise float32 partial sums
//                         (weights are final, so runs simply add), which mixed_finish_kernel adds and gates.
//
// v_mfma_f32_16x16x32_bf16: A lane l holds row l % 16, k = 8 (l / 16) + j; B lane l holds column l % 16, same k;
// D lane l holds rows 4 (l / 16) + v of column l % 16.  Scores: A = 16 keys, B = 16 query rows.  Mixing: A = 16
// (row, key) pairs over heads, B = mix^T.  Values: A = V^T (16 value columns over 32 keys), B = p'.
//
// A single token has no use for a tile of 16 rows: its form is `mixed_single_scores_kernel` and `mixed_single_values_kernel` below, in which the
// heads are the products' columns.
//
// Everything a workgroup does follows from device-side lengths (ctx_len, q_len), so a recorded step whose item list
// was made for the longest context of its class still computes each sequence's own keys; an item whose run of keys
// is empty leaves neutral statistics and zeros.
#include "common.h"
#include <math.h>

#ifndef HEAD_DIM
#define HEAD_DIM 64
#endif
#ifndef V_DIM
#define V_DIM 64
#endif
#ifndef HPW
#define HPW 1
#endif
#ifndef SHARED_KV
#define SHARED_KV 1                     // the HPW heads of a wave read one key/value head (heads a kv head are a multiple of HPW)
#endif

#define MX_WAVES 8
#define MX_THREADS (MX_WAVES * KIPP_WAVE)
#define MX_ROWS 16
#define MX_KEYS 32
#define MX_HPAD 32                      // heads padded to one step of the mixing product
// LDS strides, in bfloat16 values, chosen so that the lanes of a wave fall into different banks: the weights as
// [row][key][head] with 40 values a key (32 heads and 8 unused) and 1,288 a row, which a lane writes two bytes at a
// time (16 rows x 4 keys of one head: 4 lanes a bank instead of 64 with the plain strides) and reads 16 bytes at a
// time (no conflict); the mixed weights as [head][row][key] with 40 values a row and 656 a head.
#define P_KEY 40
#define P_ROW 1288
#define M_ROW 40
#define M_HEAD 656
#define MX_LDS_BYTES ((2 * MX_ROWS * P_ROW + MX_HPAD * M_HEAD) * 2 + HEAD_BLOCKS * KIPP_WAVE * 16)
#define KSTEPS (HEAD_DIM / 32)
#ifndef V_SLICE
#define V_SLICE V_DIM                   // value columns a workgroup sums: V_DIM / V_SLICE workgroups share an item, each
#endif                                  // with its own columns (their sums then fit a wave's registers) and all of the weights
#define VBLOCKS (V_SLICE / 16)
#define HEAD_BLOCKS (MX_WAVES * HPW > 16 ? 2 : 1)       // blocks of 16 mixed heads: a build of more heads a wave has more than 16 in all

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

union Frag {
    u32x4 u;
    bf16x8 v;
    bf16_t h[8];
};

typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

__device__ __forceinline__ uint32_t to_bf16_pair(float a, float b) {
    const f32x2 f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}

#define LOG2E 1.4426950408889634f

template <bool V>
struct Const {
    static constexpr bool value = V;
};

struct MixedGeometry {
    const int32_t* item_entry;      // [items] entry of the batch
    const int32_t* item_row0;       // [items] first row of the tile within its entry
    const int32_t* item_split;      // [items] which run of the tile's keys
    const int32_t* item_nsplits;    // [items] runs of the tile (its items are consecutive)
    const int32_t* q_start;         // [entries]
    const int32_t* q_len;           // [entries]
    const int32_t* ctx_len;         // [entries] tokens of the sequence after this step
    const int32_t* block_table;     // [entries][max_blocks]
    int max_blocks, page, n_q, n_kv, window, keep_first;
    float scale;
    const float *r1, *r2;           // [n_q] or null
};

struct Tile {
    int entry, first_row, rows, pos0, last;     // rows of the batch first_row .. + rows - 1 at positions pos0 ..; last = pos0 + rows - 1
    int kept_tiles, window_tile0;               // key tiles 0 .. kept_tiles - 1, then window_tile0 ..
    int begin, end;                             // this item's run of tile indices
    const int32_t* table;
};

__device__ __forceinline__ Tile tile_of(const MixedGeometry& g, int item) {
    Tile t;
    t.entry = g.item_entry[item];
    const int row0 = g.item_row0[item], q_len = g.q_len[t.entry];
    t.rows = max(0, min(MX_ROWS, q_len - row0));
    t.first_row = g.q_start[t.entry] + row0;
    t.pos0 = g.ctx_len[t.entry] - q_len + row0;
    t.last = t.pos0 + t.rows - 1;
    t.table = g.block_table + (size_t)t.entry * g.max_blocks;
    const int lo = g.window > 0 ? max(0, t.pos0 - g.window + 1) : 0;
    const int kept = g.window > 0 ? min(g.keep_first, lo) : 0;
    t.kept_tiles = kept > 0 ? (kept - 1) / MX_KEYS + 1 : 0;
    t.window_tile0 = max(lo / MX_KEYS, t.kept_tiles);
    const int total = t.rows > 0 ? t.kept_tiles + (t.last / MX_KEYS - t.window_tile0 + 1) : 0;
    const int nsplits = g.item_nsplits[item], split = g.item_split[item];
    const int chunk = (total + nsplits - 1) / nsplits;
    t.begin = min(total, split * chunk);
    t.end = min(total, t.begin + chunk);
    return t;
}

__device__ __forceinline__ int key_tile(const Tile& t, int index) {
    return index < t.kept_tiles ? index : t.window_tile0 + index - t.kept_tiles;
}

// The 16 keys from a multiple of 16 on lie in one page (whose size is a multiple of 16): where, the same for every lane of a wave, so
// that the table is read through the scalar cache and a load's address is a scalar base and a lane's own 32-bit offset.
struct Block {
    int first;                  // the first of them; the last key of the tile where they all lie beyond it
    int page, slot;             // of `first`
};

__device__ __forceinline__ Block block_of(const MixedGeometry& g, const Tile& t, int key0) {
    Block b;
    b.first = __builtin_amdgcn_readfirstlane(min(key0, t.last));
    const int at = __builtin_amdgcn_readfirstlane((int)((uint32_t)b.first / (uint32_t)g.page));
    b.page = ((const __attribute__((address_space(4))) int32_t*)t.table)[at];
    b.slot = b.first - at * g.page;
    return b;
}

// A block's keys of key/value head `c` as A operands: lane l holds key l % 16, columns 32 s + 8 (l / 16) ..
__device__ __forceinline__ void load_keys(const MixedGeometry& g, const Tile& t, const bf16_t* __restrict__ k_cache, int c, const Block& b,
                                          int lane, Frag* kf) {
    const int l16 = lane & 15, quarter = lane >> 4;
    const bf16_t* base = k_cache + (((size_t)b.page * g.n_kv + c) * g.page + b.slot) * HEAD_DIM;
    // (rows beyond the context are masked later; their loads stay inside it)
    const uint32_t own = min(l16, t.last - b.first) * HEAD_DIM + 8 * quarter;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) kf[s].u = *(const u32x4*)(base + own + 32 * s);
}

// S^T[key][row] of one head for the 16 keys from `key0` on: lane l gets keys key0 + 4 (l / 16) + v of row l % 16,
// already scaled, biased by distance and masked (-inf), in base 2 (2^score is the weight: `scale2` is the scale times log2 e, and
// e^(-a ln u) is 2^(-a log2 u)).  `kf`: the keys as A operands, `qf`: the head's query rows as B operands.
template <bool INSIDE>
__device__ __forceinline__ void scores16(const MixedGeometry& g, const Tile& t, int key0, const Frag* kf, const Frag* qf,
                                         float a, float b, int lane, float sc[4]) {
    const int l16 = lane & 15, quarter = lane >> 4;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[s].v, qf[s].v, acc, 0, 0, 0);
    const int i = t.pos0 + l16, away = i - key0 - 4 * quarter;
    const float scale2 = g.scale * LOG2E, away0 = (float)away;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        // INSIDE: every row of the tile sees all 16 keys (rows that only fill the tile up compute unused numbers)
        const bool sees = INSIDE || (l16 < t.rows && away >= v && (g.window <= 0 || away - v < g.window || i - away + v < g.keep_first));
        const float s = fmaf(acc[v], scale2, -a * __builtin_amdgcn_logf(fmaf(b, away0 - (float)v, 1.0f)));
        sc[v] = sees ? s : -INFINITY;
    }
}

// Whether every row of the tile sees every key of the 32 from `key0` on: behind the first row, and inside the window of
// the last (or among the kept first keys).
__device__ __forceinline__ bool all_seen(const MixedGeometry& g, const Tile& t, int key0) {
    return key0 + MX_KEYS - 1 <= t.pos0 && (g.window <= 0 || t.pos0 + MX_ROWS - 1 - key0 < g.window || key0 + MX_KEYS <= g.keep_first);
}

// The query rows of head h as B operands: lane l holds row l % 16, columns 32 s + 8 (l / 16) ..
__device__ __forceinline__ void load_queries(const Tile& t, const bf16_t* __restrict__ q, int n_q, int h, Frag* qf) {
    const int lane = threadIdx.x & (KIPP_WAVE - 1), l16 = lane & 15, quarter = lane >> 4;
    const int row = t.first_row + min(l16, max(t.rows - 1, 0));
    const bf16_t* at = q + ((size_t)row * n_q + h) * HEAD_DIM + 8 * quarter;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) qf[s].u = *(const u32x4*)(at + 32 * s);
}

// stats [items][n_q][16][2]: (maximum, sum of 2^(score - maximum)) over the item's keys, without the sink.
// Bound by vector instructions (a logarithm and an exponential a score): 1,500 rows of 32 heads 41 us, as 414 items with a page looked up by
// every lane 51, in base e 68.
__global__ void __launch_bounds__(MX_THREADS) mixed_stats_kernel(MixedGeometry g, const bf16_t* __restrict__ q,
                                                                 const bf16_t* __restrict__ k_cache, float* __restrict__ stats) {
    const int item = blockIdx.x;
    const Tile t = tile_of(g, item);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KIPP_WAVE), lane = threadIdx.x & (KIPP_WAVE - 1);
    const int group = g.n_q / g.n_kv, h0 = wave * HPW;
    if (h0 >= g.n_q) return;
    constexpr bool shared = SHARED_KV != 0;                 // the wave's heads read one key/value head
    Frag qf[HPW][KSTEPS];
    float a[HPW], b[HPW], m[HPW], l[HPW];
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh) {
        const int h = min(h0 + hh, g.n_q - 1);
        load_queries(t, q, g.n_q, h, qf[hh]);
        a[hh] = g.r1 != nullptr ? g.r1[h] : 0.0f;
        b[hh] = g.r2 != nullptr ? g.r2[h] : 0.0f;
        m[hh] = -INFINITY;
        l[hh] = 0.0f;
    }
    Frag kf[MX_KEYS / 16][KSTEPS], next[MX_KEYS / 16][KSTEPS];
    Block at[MX_KEYS / 16], at_next[MX_KEYS / 16];          // of this tile's keys and of the next's: asked for a tile ahead of the keys
    if (t.begin < t.end) {
#pragma unroll
        for (int kb = 0; kb < MX_KEYS / 16; ++kb) {
            at[kb] = block_of(g, t, key_tile(t, t.begin) * MX_KEYS + 16 * kb);
            at_next[kb] = block_of(g, t, key_tile(t, min(t.begin + 1, t.end - 1)) * MX_KEYS + 16 * kb);
        }
#pragma unroll
        for (int kb = 0; kb < MX_KEYS / 16; ++kb) load_keys(g, t, k_cache, h0 / group, at[kb], lane, next[kb]);
    }
    for (int index = t.begin; index < t.end; ++index) {
        const int key0 = key_tile(t, index) * MX_KEYS;
#pragma unroll
        for (int kb = 0; kb < MX_KEYS / 16; ++kb)
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) kf[kb][s] = next[kb][s];
        const bool inside = all_seen(g, t, key0);
        Block own_at[MX_KEYS / 16];
#pragma unroll
        for (int kb = 0; kb < MX_KEYS / 16; ++kb) own_at[kb] = at[kb];
        if (index + 1 < t.end) {            // the next tile's keys are on their way while this one is scored
#pragma unroll
            for (int kb = 0; kb < MX_KEYS / 16; ++kb) {
                at[kb] = at_next[kb];
                load_keys(g, t, k_cache, h0 / group, at[kb], lane, next[kb]);
                at_next[kb] = block_of(g, t, key_tile(t, min(index + 2, t.end - 1)) * MX_KEYS + 16 * kb);
            }
        }
#pragma unroll
        for (int hh = 0; hh < HPW; ++hh) {
            if (h0 + hh >= g.n_q) break;
#pragma unroll
            for (int kb = 0; kb < MX_KEYS / 16; ++kb) {
                Frag own[KSTEPS];
                if (!shared && hh > 0) load_keys(g, t, k_cache, (h0 + hh) / group, own_at[kb], lane, own);
                float sc[4];
                if (inside) scores16<true>(g, t, key0 + 16 * kb, (!shared && hh > 0) ? own : kf[kb], qf[hh], a[hh], b[hh], lane, sc);
                else scores16<false>(g, t, key0 + 16 * kb, (!shared && hh > 0) ? own : kf[kb], qf[hh], a[hh], b[hh], lane, sc);
                const float m_new = fmaxf(m[hh], fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])));
                if (m_new != -INFINITY) {
                    float sum = 0.0f;
#pragma unroll
                    for (int v = 0; v < 4; ++v) sum += __builtin_amdgcn_exp2f(sc[v] - m_new);       // exp(-inf) = 0
                    l[hh] = l[hh] * __builtin_amdgcn_exp2f(m[hh] - m_new) + sum;
                    m[hh] = m_new;
                }
            }
        }
    }
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh) {
        if (h0 + hh >= g.n_q) break;
        float mm = m[hh], ll = l[hh];
        // the four lanes that share a row
#pragma unroll
        for (int off = 16; off <= 32; off <<= 1) {
            const float m_o = __shfl_xor(mm, off, KIPP_WAVE), l_o = __shfl_xor(ll, off, KIPP_WAVE);
            const float m_new = fmaxf(mm, m_o);
            if (m_new != -INFINITY) ll = ll * __builtin_amdgcn_exp2f(mm - m_new) + l_o * __builtin_amdgcn_exp2f(m_o - m_new);
            mm = m_new;
        }
        if (lane < 16) {
            float* out = stats + (((size_t)item * g.n_q + h0 + hh) * MX_ROWS + lane) * 2;
            out[0] = mm;
            out[1] = ll;
        }
    }
}

// Bound by vector instructions, LDS and two barriers a tile; a compute unit holds one workgroup, so its loads' latencies show: the table is read
// through the scalar cache a tile ahead, the values leave memory while the heads are mixed.  Registers (256 a wave) decide: sums and queries take 192, and with a
// lane's places in LDS kept over tiles, the mix in registers and all heads' scores at once in the scheduler's hands 73 to 175 spilled.  1,500 rows of 32
// heads of 128, us: 166 as it was (73 spilled, 414 items of up to eight tiles); 89 now (232 items of up to twelve, `ops.mixed_tile_runs`).
// The first keys of the next tile asked for as well: 75 spill where a workgroup sums all of 128 value columns; there they wait.
// LDS: p_hi, p_lo [16 rows][32 keys][32 heads] bfloat16, then p' [32 heads][16 rows][32 keys] bfloat16, with the padded strides above.
__global__ void __launch_bounds__(MX_THREADS) mixed_values_kernel(
    MixedGeometry g, const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const float* __restrict__ stats, const float* __restrict__ sink, const float* __restrict__ mix,
    const float* __restrict__ gate, int gate_stride, int gate_parts, size_t gate_part_stride,
    bf16_t* __restrict__ out, float* __restrict__ partial, size_t partial_stride) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    bf16_t* p_hi = (bf16_t*)lds_raw;
    bf16_t* p_lo = p_hi + MX_ROWS * P_ROW;
    bf16_t* p_mixed = p_lo + MX_ROWS * P_ROW;
    const int item = blockIdx.x, v0 = blockIdx.y * V_SLICE;        // this workgroup's value columns v0 .. v0 + V_SLICE - 1 of every head
    const Tile t = tile_of(g, item);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KIPP_WAVE), lane_of_wave = threadIdx.x & (KIPP_WAVE - 1), l16 = lane_of_wave & 15, quarter = lane_of_wave >> 4;
    const int nsplits = g.item_nsplits[item], split = g.item_split[item];
    const int n_q = g.n_q, group = g.n_q / g.n_kv;
    constexpr bool shared = SHARED_KV != 0;                 // the wave's heads read one key/value head

    // columns of heads that do not exist stay zero for the whole walk
    if (n_q < MX_HPAD)
        for (int e = threadIdx.x; e < 2 * MX_ROWS * P_ROW / 8; e += MX_THREADS) ((u32x4*)p_hi)[e] = (u32x4){0u, 0u, 0u, 0u};

    // mix^T as B operands: lane holds head (column) 16 nb + l % 16, contraction heads 8 (l / 16) ..  (asked for whatever the head, inside the
    // matrix: all loads beside each other)
    u32x4* mix_frags = (u32x4*)(p_mixed + MX_HPAD * M_HEAD);        // in LDS: in registers they would take the place of keys on their way
    if (wave < HEAD_BLOCKS) {
        const int h = 16 * wave + l16;
        float w[8];
        if (mix != nullptr) {
#pragma unroll
            for (int j = 0; j < 8; ++j) w[j] = mix[min(h, n_q - 1) * n_q + min(8 * quarter + j, n_q - 1)];
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) w[j] = h == 8 * quarter + j ? 1.0f : 0.0f;
        }
        Frag mf;
#pragma unroll
        for (int j = 0; j < 8; ++j) mf.h[j] = f32_to_bf16(h < n_q && 8 * quarter + j < n_q ? w[j] : 0.0f);
        mix_frags[64 * wave + lane_of_wave] = mf.u;
    }

    // this wave's heads: queries, bias numbers, and every row's maximum and denominator over ALL runs of the tile
    Frag qf[HPW][KSTEPS];
    float bias_a[HPW], bias_b[HPW], under[HPW];         // a weight is 2^(score + under)
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh) {
        // (heads that do not exist take the last one's queries, and weigh nothing)
        const int h = min(wave * HPW + hh, n_q - 1);
        load_queries(t, q, n_q, h, qf[hh]);
        bias_a[hh] = g.r1 != nullptr ? g.r1[h] : 0.0f;
        bias_b[hh] = g.r2 != nullptr ? g.r2[h] : 0.0f;
        const float sunk = sink != nullptr ? sink[h] * LOG2E : -INFINITY;
        // the runs' statistics: each quarter of the wave takes every fourth run (four asked for at once), the
        // quarters are then merged, the sink last; any order gives the same maximum, and the sums differ in rounding only
        float m = -INFINITY, l = 0.0f;
        for (int s0 = quarter; s0 < nsplits; s0 += 16) {
            float2 st[4];
#pragma unroll
            for (int s = 0; s < 4; ++s)
                st[s] = *(const float2*)(stats + (((size_t)(item - split + min(s0 + 4 * s, nsplits - 1)) * n_q + h) * MX_ROWS + l16) * 2);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                if (s0 + 4 * s >= nsplits) st[s] = make_float2(-INFINITY, 0.0f);
                const float m_new = fmaxf(m, st[s].x);
                if (m_new != -INFINITY) l = l * __builtin_amdgcn_exp2f(m - m_new) + st[s].y * __builtin_amdgcn_exp2f(st[s].x - m_new);
                m = m_new;
            }
        }
#pragma unroll
        for (int off = 16; off <= 32; off <<= 1) {
            const float m_o = __shfl_xor(m, off, KIPP_WAVE), l_o = __shfl_xor(l, off, KIPP_WAVE);
            const float m_new = fmaxf(m, m_o);
            if (m_new != -INFINITY) l = l * __builtin_amdgcn_exp2f(m - m_new) + l_o * __builtin_amdgcn_exp2f(m_o - m_new);
            m = m_new;
        }
        if (sink != nullptr) {
            const float m_new = fmaxf(m, sunk);
            l = (m == -INFINITY ? 0.0f : l * __builtin_amdgcn_exp2f(m - m_new)) + __builtin_amdgcn_exp2f(sunk - m_new);
            m = m_new;
        }
        under[hh] = wave * HPW + hh < n_q && l > 0.0f ? -m - __builtin_amdgcn_logf(l) : -INFINITY;
    }

    f32x4 acc[HPW][VBLOCKS];
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh)
#pragma unroll
        for (int mb = 0; mb < VBLOCKS; ++mb) acc[hh][mb] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    __syncthreads();

    Block at_next[MX_KEYS / 16];            // where the next tile's keys and values lie: asked for a tile ahead
    // where registers are left: the first half of a tile's keys, asked for while the tile before meets its values
    constexpr bool keys_ahead = shared && 4 * HPW * (VBLOCKS + KSTEPS) <= 128;
    Frag first_keys[KSTEPS];
    if (t.begin < t.end) {
#pragma unroll
        for (int kb = 0; kb < MX_KEYS / 16; ++kb) at_next[kb] = block_of(g, t, key_tile(t, t.begin) * MX_KEYS + 16 * kb);
        if (keys_ahead) load_keys(g, t, k_cache, min(wave * HPW, n_q - 1) / group, at_next[0], lane_of_wave, first_keys);
    }
    for (int index = t.begin; index < t.end; ++index) {
        const int key0 = key_tile(t, index) * MX_KEYS;
        const bool inside = all_seen(g, t, key0);
        // a lane's places in LDS and in the caches are made again for every tile: kept, they take registers that the sums need
        int lane = lane_of_wave;
        asm volatile("" : "+v"(lane));
        const int l16 = lane & 15, quarter = lane >> 4;
        Block at_key[MX_KEYS / 16];
#pragma unroll
        for (int kb = 0; kb < MX_KEYS / 16; ++kb) {
            at_key[kb] = at_next[kb];
            at_next[kb] = block_of(g, t, key_tile(t, min(index + 1, t.end - 1)) * MX_KEYS + 16 * kb);
        }
        // 1. the final weights of this wave's heads; 16 keys are loaded once for all heads that share them, and a lane
        //    writes the weights of its heads (they are neighbours in the [row][key][head] layout) with one store
        auto weights = [&](auto all) __attribute__((always_inline)) {
#pragma unroll
            for (int kb = 0; kb < MX_KEYS / 16; ++kb) {
                __builtin_amdgcn_sched_barrier(0);
                Frag kf[KSTEPS];
                if (keys_ahead && kb == 0) {
#pragma unroll
                    for (int s = 0; s < KSTEPS; ++s) kf[s] = first_keys[s];
                } else {
                    load_keys(g, t, k_cache, min(wave * HPW, n_q - 1) / group, at_key[kb], lane, kf);
                }
                float p[HPW][4];
#pragma unroll
                for (int hh = 0; hh < HPW; ++hh) {
                    if (!shared && hh > 0) load_keys(g, t, k_cache, min(wave * HPW + hh, n_q - 1) / group, at_key[kb], lane, kf);
                    __builtin_amdgcn_sched_barrier(0);      // one head after the other: mixed, their scores fill the registers that the sums need
                    float sc[4];
                    scores16<decltype(all)::value>(g, t, key0 + 16 * kb, kf, qf[hh], bias_a[hh], bias_b[hh], lane, sc);
#pragma unroll
                    for (int v = 0; v < 4; ++v) p[hh][v] = __builtin_amdgcn_exp2f(sc[v] + under[hh]);
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int at = l16 * P_ROW + (16 * kb + 4 * quarter + v) * P_KEY + wave * HPW;
                    if (HPW == 4 || HPW == 2) {
                        uint32_t hi[(HPW + 1) / 2], lo[(HPW + 1) / 2];
#pragma unroll
                        for (int two = 0; two < HPW / 2; ++two) {
                            const float a = p[2 * two % HPW][v], b = p[(2 * two + 1) % HPW][v];
                            hi[two] = to_bf16_pair(a, b);
                            lo[two] = to_bf16_pair(a - __uint_as_float(hi[two] << 16), b - __uint_as_float(hi[two] & 0xffff0000u));
                        }
                        if (HPW == 4) {
                            *(uint2*)(p_hi + at) = make_uint2(hi[0], hi[HPW / 2 - 1]);
                            *(uint2*)(p_lo + at) = make_uint2(lo[0], lo[HPW / 2 - 1]);
                        } else {
                            *(uint32_t*)(p_hi + at) = hi[0];
                            *(uint32_t*)(p_lo + at) = lo[0];
                        }
                    } else {
#pragma unroll
                        for (int hh = 0; hh < HPW; ++hh) {
                            const bf16_t hi = f32_to_bf16(p[hh][v]);
                            p_hi[at + hh] = hi;
                            p_lo[at + hh] = f32_to_bf16(p[hh][v] - bf16_to_f32(hi));
                        }
                    }
                }
            }
        };
        if (wave * HPW < n_q) {
            if (inside) weights(Const<true>{});
            else weights(Const<false>{});
        }
        // where the values lie, and the first of them asked for while the heads are mixed
        // (eight keys of one page: those of quarters 0 and 1 lie in the first block, of 2 and 3 in the second)
        const Block& low = at_key[0];
        const Block& high = at_key[MX_KEYS / 16 - 1];
        const size_t v_page = (size_t)(quarter < 2 ? low.page : high.page) * g.n_kv;
        const int v_slot = ((quarter < 2 ? low.slot : high.slot) & ~15) + 8 * (quarter & 1);
        constexpr int VB = VBLOCKS < 4 ? VBLOCKS : 4;                // value blocks asked for together
        constexpr int VGROUPS = (VBLOCKS + VB - 1) / VB;
        Frag vf[2][VB];
        const bf16_t* v_at = v_cache + ((v_page + min(wave * HPW, n_q - 1) / group) * V_DIM + v0 + l16) * g.page + v_slot;
        auto load_values = [&](int m0) __attribute__((always_inline)) {
#pragma unroll
            for (int mb = 0; mb < VB; ++mb)
                if (m0 + mb < VBLOCKS) vf[m0 / VB % 2][mb].u = *(const u32x4*)(v_at + (size_t)16 * (m0 + mb) * g.page);
        };
        if (shared) load_values(0);
        __syncthreads();
        // 2. the heads mixed: 32 blocks of 16 (row, key) pairs, four a wave
        Frag mf[HEAD_BLOCKS];
#pragma unroll
        for (int nb = 0; nb < HEAD_BLOCKS; ++nb) mf[nb].u = mix_frags[64 * nb + lane];
#pragma unroll
        for (int u = 0; u < (MX_ROWS * MX_KEYS / 16) / MX_WAVES; ++u) {
            const int block = wave + MX_WAVES * u;              // row = block / 2, keys 16 (block % 2) ..
            const int row = block >> 1, kb = block & 1;
            const int at = row * P_ROW + (16 * kb + l16) * P_KEY + 8 * quarter;
            Frag hi, lo;
            hi.u = *(const u32x4*)(p_hi + at);
            lo.u = *(const u32x4*)(p_lo + at);
#pragma unroll
            for (int nb = 0; nb < HEAD_BLOCKS; ++nb) {
                f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo.v, mf[nb].v, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi.v, mf[nb].v, d, 0, 0, 0);
                uint2 w;                            // d[v]: keys 16 kb + 4 quarter + v of `row`, head 16 nb + l16
                w.x = to_bf16_pair(d[0], d[1]);
                w.y = to_bf16_pair(d[2], d[3]);
                *(uint2*)(p_mixed + ((16 * nb + l16) * M_HEAD + row * M_ROW + 16 * kb + 4 * quarter)) = w;
            }
        }
        __syncthreads();
        if (shared && VGROUPS > 1) load_values(VB);
        // 3. times the values
        if (shared) {
            if (wave * HPW < n_q) {
#pragma unroll
                for (int m0 = 0; m0 < VBLOCKS; m0 += VB) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int hh = 0; hh < HPW; ++hh) {
                        __builtin_amdgcn_sched_barrier(0);
                        Frag pf;
                        pf.u = *(const u32x4*)(p_mixed + (min(wave * HPW + hh, n_q - 1) * M_HEAD + l16 * M_ROW + 8 * quarter));
#pragma unroll
                        for (int mb = 0; mb < VB; ++mb)
                            if (m0 + mb < VBLOCKS)
                                acc[hh][m0 + mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[m0 / VB % 2][mb].v, pf.v, acc[hh][m0 + mb], 0, 0, 0);
                    }
                    if (m0 + 2 * VB < VBLOCKS) load_values(m0 + 2 * VB);
                    // (behind the last group but one, whose registers are free)
                    if (keys_ahead && m0 / VB == (VGROUPS > 1 ? VGROUPS - 2 : 0))
                        load_keys(g, t, k_cache, min(wave * HPW, n_q - 1) / group, at_next[0], lane, first_keys);
                }
            }
        } else {
#pragma unroll
            for (int hh = 0; hh < HPW; ++hh) {
                const int h = wave * HPW + hh;
                if (h < n_q) {
                    Frag pf;
                    pf.u = *(const u32x4*)(p_mixed + (h * M_HEAD + l16 * M_ROW + 8 * quarter));
                    const bf16_t* v_at = v_cache + ((v_page + h / group) * V_DIM + v0 + l16) * g.page + v_slot;
#pragma unroll
                    for (int mb = 0; mb < VBLOCKS; ++mb) {
                        Frag vf;
                        vf.u = *(const u32x4*)(v_at + (size_t)16 * mb * g.page);
                        acc[hh][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, pf.v, acc[hh][mb], 0, 0, 0);
                    }
                }
            }
        }
        // the next tile's weights overwrite p only after every wave has passed the barrier behind step 2,
        // and p' only after the barrier behind the next step 1
    }

    // acc[hh][mb][v]: value column 16 mb + 4 quarter + v of row l16
    if (l16 >= t.rows) return;
    const size_t row = (size_t)t.first_row + l16;
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh) {
        const int h = wave * HPW + hh;
        if (h >= n_q) break;
#pragma unroll
        for (int mb = 0; mb < VBLOCKS; ++mb) {
            const int col = h * V_DIM + v0 + 16 * mb + 4 * quarter;
            if (nsplits > 1) {
                *(f32x4*)(partial + split * partial_stride + row * ((size_t)n_q * V_DIM) + col) = acc[hh][mb];
            } else {
                float o[4];
                if (gate != nullptr) {
                    float z[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                    for (int p = 0; p < gate_parts; ++p)
#pragma unroll
                        for (int v = 0; v < 4; ++v) z[v] += gate[p * gate_part_stride + row * gate_stride + col + v];
#pragma unroll
                    for (int v = 0; v < 4; ++v) o[v] = acc[hh][mb][v] * (1.0f / (1.0f + __expf(-z[v])));
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v) o[v] = acc[hh][mb][v];
                }
                uint2 w;
                w.x = (uint32_t)f32_to_bf16(o[0]) | ((uint32_t)f32_to_bf16(o[1]) << 16);
                w.y = (uint32_t)f32_to_bf16(o[2]) | ((uint32_t)f32_to_bf16(o[3]) << 16);
                *(uint2*)(out + row * ((size_t)n_q * V_DIM) + col) = w;
            }
        }
    }
}

// ---- single tokens ------------------------------------------------------------------------------------------------
//
// A workgroup takes (a run of the token's keys, token), keys 64 at a time; a wave takes key/value heads in turn.
//
//   mixed_single_scores_kernel   scores of a key/value head's query heads (16 keys x the heads a product), scaled, biased and masked, into
//                                memory as float32 [token][key][32 heads], and the run's (maximum, sum) of every head;
//   mixed_single_values_kernel   merges the runs' statistics and the sink; a lane takes 8 heads of a key, makes their final weights
//                                (two bfloat16 halves, as above) and mixes them on the matrix cores without a trip through LDS; the
//                                mixed weights through LDS to the waves of their key/value heads, which multiply the values, asked
//                                for before anything else.  Every run leaves float32 partial sums.
//
// Bound by its chains of loads (page, keys; statistics, scores), not by bytes: one token behind 1,500 keys of 8 heads (32 query
// heads of 128 over them) takes 8.8 us for the scores, 14.2 for the values (15.0 while their scores, the mix and the sink were asked for behind the
// statistics) and 5.0 for the sum of the 24 runs (5.5 with the gate asked for behind the sums).  The tiles of 16 rows
// took 21.5, 41.5 and 4.9 us for it (bias, mask, exponentials and exchanges for 16 rows, at most 16 runs of 128 keys and more).
#define SG_KEYS 64
#define SG_PITCH 72                     // bfloat16 values from a head to the next of the mixed weights in LDS
#define SG_PARTS (MX_THREADS / MX_HPAD)

struct SingleGeometry {
    const int32_t* rows;            // [tokens] row of the batch
    const int32_t* positions;       // [rows of the batch]
    const int32_t* seq_of_token;    // [rows of the batch] row of the block table
    const int32_t* block_table;
    int max_blocks, page, n_q, n_kv, window, keep_first, n_runs, max_tiles;
    float scale;
    const float *r1, *r2;           // [n_q] or null
};

struct Single {
    int row, pos, lo, kept;                         // it sees keys 0 .. kept - 1 and lo .. pos
    int kept_tiles, window_tile0, begin, end;       // tiles of 64 keys: 0 .. kept_tiles - 1, then window_tile0 ..; this run's indices
    const int32_t* table;
};

__device__ __forceinline__ Single single_of(const SingleGeometry& g, int token, int run) {
    Single t;
    t.row = g.rows[token];
    t.pos = g.positions[t.row];
    t.table = g.block_table + (size_t)g.seq_of_token[t.row] * g.max_blocks;
    t.lo = g.window > 0 ? max(0, t.pos - g.window + 1) : 0;
    t.kept = g.window > 0 ? min(g.keep_first, t.lo) : 0;
    t.kept_tiles = (t.kept + SG_KEYS - 1) / SG_KEYS;
    t.window_tile0 = max(t.lo / SG_KEYS, t.kept_tiles);
    const int total = min(g.max_tiles, t.kept_tiles + t.pos / SG_KEYS - t.window_tile0 + 1);
    const int chunk = (total + g.n_runs - 1) / g.n_runs;
    t.begin = min(total, run * chunk);
    t.end = min(total, t.begin + chunk);
    return t;
}

__device__ __forceinline__ int single_key0(const Single& t, int index) {
    return SG_KEYS * (index < t.kept_tiles ? index : t.window_tile0 + index - t.kept_tiles);
}

// scores: float32 [tokens][max_tiles][64][32]; stats: float32 [tokens][runs][32][2].
__global__ void __launch_bounds__(MX_THREADS) mixed_single_scores_kernel(SingleGeometry g, const bf16_t* __restrict__ q,
                                                                         const bf16_t* __restrict__ k_cache, float* __restrict__ scores,
                                                                         float* __restrict__ stats) {
    const int token = blockIdx.y, run = blockIdx.x;
    const Single t = single_of(g, token, run);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KIPP_WAVE), lane = threadIdx.x & (KIPP_WAVE - 1), l16 = lane & 15, quarter = lane >> 4;
    const int group = g.n_q / g.n_kv;
    for (int c = wave; c < g.n_kv; c += MX_WAVES) {
        const int h = c * group + min(l16, group - 1);      // lanes beyond the head's group compute what nobody reads
        Frag qf[KSTEPS];
        const bf16_t* q_at = q + ((size_t)t.row * g.n_q + h) * HEAD_DIM + 8 * quarter;
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) qf[s].u = *(const u32x4*)(q_at + 32 * s);
        const float a = g.r1 != nullptr ? g.r1[h] : 0.0f, b = g.r2 != nullptr ? g.r2[h] : 0.0f;
        float m = -INFINITY, l = 0.0f;
        for (int index = t.begin; index < t.end; ++index) {
            const int key0 = single_key0(t, index);
            Frag kf[SG_KEYS / 16][KSTEPS];
#pragma unroll
            for (int kb = 0; kb < SG_KEYS / 16; ++kb) {
                const int key = min(key0 + 16 * kb + l16, t.pos);       // masked below; its load stays inside the context
                const bf16_t* k_at = k_cache + (((size_t)t.table[key / g.page] * g.n_kv + c) * g.page + key % g.page) * HEAD_DIM + 8 * quarter;
#pragma unroll
                for (int s = 0; s < KSTEPS; ++s) kf[kb][s].u = *(const u32x4*)(k_at + 32 * s);
            }
            float sc[SG_KEYS / 16][4];
            float top = m;
#pragma unroll
            for (int kb = 0; kb < SG_KEYS / 16; ++kb) {
                f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int s = 0; s < KSTEPS; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kb][s].v, qf[s].v, acc, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int j = key0 + 16 * kb + 4 * quarter + v, away = t.pos - j;
                    sc[kb][v] = away >= 0 && (j >= t.lo || j < t.kept) ? acc[v] * g.scale - a * __logf(1.0f + b * (float)away) : -INFINITY;
                    top = fmaxf(top, sc[kb][v]);
                }
            }
            if (l16 < group) {
                float* at = scores + (((size_t)token * g.max_tiles + index) * SG_KEYS + 4 * quarter) * MX_HPAD + h;
#pragma unroll
                for (int kb = 0; kb < SG_KEYS / 16; ++kb)
#pragma unroll
                    for (int v = 0; v < 4; ++v) at[(16 * kb + v) * MX_HPAD] = sc[kb][v];
            }
            if (top != -INFINITY) {
                float sum = 0.0f;
#pragma unroll
                for (int kb = 0; kb < SG_KEYS / 16; ++kb)
#pragma unroll
                    for (int v = 0; v < 4; ++v) sum += __expf(sc[kb][v] - top);     // exp(-inf) = 0
                l = l * __expf(m - top) + sum;
                m = top;
            }
        }
#pragma unroll
        for (int off = 16; off <= 32; off <<= 1) {      // the four lanes that share a head
            const float m_o = __shfl_xor(m, off, KIPP_WAVE), l_o = __shfl_xor(l, off, KIPP_WAVE);
            const float m_new = fmaxf(m, m_o);
            if (m_new != -INFINITY) l = l * __expf(m - m_new) + l_o * __expf(m_o - m_new);
            m = m_new;
        }
        if (quarter == 0 && l16 < group) *(float2*)(stats + (((size_t)token * g.n_runs + run) * MX_HPAD + h) * 2) = make_float2(m, l);
    }
}

// partial: float32 [runs][tokens][n_q V_DIM].
__global__ void __launch_bounds__(MX_THREADS) mixed_single_values_kernel(SingleGeometry g, const bf16_t* __restrict__ v_cache,
                                                                         const float* __restrict__ scores, const float* __restrict__ stats,
                                                                         const float* __restrict__ sink, const float* __restrict__ mix,
                                                                         float* __restrict__ partial) {
    constexpr int BLOCKS = V_DIM / 16, KS = SG_KEYS / 32;
    __shared__ __attribute__((aligned(16))) bf16_t p_mixed[2][MX_HPAD * SG_PITCH];
    __shared__ float2 merged[MX_WAVES][MX_HPAD];
    __shared__ float2 weigh[MX_HPAD];       // a head's maximum and 1 / denominator
    const int token = blockIdx.y, run = blockIdx.x, n_tokens = gridDim.y;
    const Single t = single_of(g, token, run);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KIPP_WAVE), lane = threadIdx.x & (KIPP_WAVE - 1), l16 = lane & 15, quarter = lane >> 4;
    const int n_q = g.n_q, group = g.n_q / g.n_kv;
    auto load_values = [&](int c, int key0, Frag (&vf)[KS][BLOCKS]) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int key = key0 + 32 * ks + 8 * quarter;           // eight keys of one page (a page holds a multiple of 8)
            const bf16_t* v_at = v_cache + (((size_t)t.table[min(key, t.pos) / g.page] * g.n_kv + c) * V_DIM + l16) * g.page + key % g.page;
#pragma unroll
            for (int mb = 0; mb < BLOCKS; ++mb) vf[ks][mb].u = *(const u32x4*)(v_at + (size_t)16 * mb * g.page);
        }
    };
    Frag vf[KS][BLOCKS];
    if (t.begin < t.end && wave < g.n_kv) load_values(wave, single_key0(t, t.begin), vf);

    // this wave mixes 16 keys of a tile for 16 of the mixed heads; mix^T as B operand: column 16 nb + l % 16, contraction heads
    // 8 (l / 16) ..  The first tile's scores and the mix are on their way while the statistics are merged.
    const int kb = wave & 3, nb = wave >> 2;
    const int mixed_h = 16 * nb + l16;
    auto load_scores = [&](int index, float (&sc)[8]) {
        const float* at = scores + (((size_t)token * g.max_tiles + index) * SG_KEYS + 16 * kb + l16) * MX_HPAD + 8 * quarter;
        *(f32x4*)sc = *(const f32x4*)at;
        *(f32x4*)(sc + 4) = *(const f32x4*)(at + 4);
    };
    float first_sc[8], mix_w[8];
    if (t.begin < t.end && 16 * nb < n_q) load_scores(t.begin, first_sc);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int from = 8 * quarter + j;
        mix_w[j] = 0.0f;
        if (mixed_h < n_q && from < n_q) mix_w[j] = mix != nullptr ? mix[mixed_h * n_q + from] : (mixed_h == from ? 1.0f : 0.0f);
    }
    const float sunk = sink != nullptr && (int)(threadIdx.x & (MX_HPAD - 1)) < n_q ? sink[threadIdx.x & (MX_HPAD - 1)] : -INFINITY;

    // the weights' numbers a head: the runs' statistics, a thread a head and every SG_PARTS-th run; the sink last
    {
        const int h = threadIdx.x & (MX_HPAD - 1), part = threadIdx.x / MX_HPAD;
        float m = -INFINITY, l = 0.0f;
        if (h < n_q)
            for (int r0 = part; r0 < g.n_runs; r0 += 4 * SG_PARTS) {
                float2 st[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    st[i] = r0 + i * SG_PARTS < g.n_runs ? *(const float2*)(stats + (((size_t)token * g.n_runs + r0 + i * SG_PARTS) * MX_HPAD + h) * 2)
                                                         : make_float2(-INFINITY, 0.0f);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float m_new = fmaxf(m, st[i].x);
                    if (m_new != -INFINITY) l = l * __expf(m - m_new) + st[i].y * __expf(st[i].x - m_new);
                    m = m_new;
                }
            }
        {                                   // a wave's two parts
            const float m_o = __shfl_xor(m, MX_HPAD, KIPP_WAVE), l_o = __shfl_xor(l, MX_HPAD, KIPP_WAVE), m_new = fmaxf(m, m_o);
            if (m_new != -INFINITY) l = l * __expf(m - m_new) + l_o * __expf(m_o - m_new);
            m = m_new;
        }
        if (lane < MX_HPAD) merged[wave][h] = make_float2(m, l);
        __syncthreads();
        if (threadIdx.x < MX_HPAD) {
            float2 of_wave[MX_WAVES];
            float top = sunk;
#pragma unroll
            for (int i = 0; i < MX_WAVES; ++i) {
                of_wave[i] = merged[i][h];
                top = fmaxf(top, of_wave[i].x);
            }
            float sum = sunk != -INFINITY ? __expf(sunk - top) : 0.0f;
#pragma unroll
            for (int i = 0; i < MX_WAVES; ++i)
                if (of_wave[i].x != -INFINITY) sum += of_wave[i].y * __expf(of_wave[i].x - top);
            weigh[h] = make_float2(top, sum > 0.0f ? 1.0f / sum : 0.0f);
        }
        __syncthreads();
    }

    float2 of_head[8];
    Frag mf;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        of_head[j] = weigh[8 * quarter + j];
        mf.h[j] = f32_to_bf16(mix_w[j]);
    }
    for (int c0 = 0; c0 < g.n_kv; c0 += MX_WAVES) {         // (more than eight key/value heads: the weights are made again for each eight)
        const int c = c0 + wave;
        f32x4 acc[BLOCKS];
#pragma unroll
        for (int mb = 0; mb < BLOCKS; ++mb) acc[mb] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        for (int index = t.begin; index < t.end; ++index) {
            const int key0 = single_key0(t, index);
            bf16_t* pm = p_mixed[index & 1];                // the other half is read until every wave is past the barrier
            if ((c0 > 0 || index > t.begin) && c < g.n_kv) load_values(c, key0, vf);
            if (16 * nb < n_q) {
                float sc[8];
                if (c0 > 0 || index > t.begin) load_scores(index, sc);
                else
#pragma unroll
                    for (int j = 0; j < 8; ++j) sc[j] = first_sc[j];
                Frag hi, lo;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    // (heads that do not exist were never written)
                    const float p = 8 * quarter + j < n_q && sc[j] != -INFINITY ? __expf(sc[j] - of_head[j].x) * of_head[j].y : 0.0f;
                    hi.h[j] = f32_to_bf16(p);
                    lo.h[j] = f32_to_bf16(p - bf16_to_f32(hi.h[j]));
                }
                f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo.v, mf.v, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi.v, mf.v, d, 0, 0, 0);
                uint2 w;                                    // d[v]: key 16 kb + 4 quarter + v, head 16 nb + l16
                w.x = (uint32_t)f32_to_bf16(d[0]) | ((uint32_t)f32_to_bf16(d[1]) << 16);
                w.y = (uint32_t)f32_to_bf16(d[2]) | ((uint32_t)f32_to_bf16(d[3]) << 16);
                *(uint2*)(pm + (16 * nb + l16) * SG_PITCH + 16 * kb + 4 * quarter) = w;
            }
            __syncthreads();
            if (c < g.n_kv) {
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const int first = key0 + 32 * ks + 8 * quarter;
                    const bool whole = first + 7 <= t.pos && (first >= t.lo || first + 7 < t.kept);
                    Frag pf;
                    pf.u = *(const u32x4*)(pm + (c * group + min(l16, group - 1)) * SG_PITCH + 32 * ks + 8 * quarter);
#pragma unroll
                    for (int mb = 0; mb < BLOCKS; ++mb) {
                        Frag f = vf[ks][mb];
                        if (!whole) {           // what the token does not see weighs nothing, but its slots hold anything
#pragma unroll
                            for (int j = 0; j < 8; ++j)
                                if (first + j > t.pos || (first + j < t.lo && first + j >= t.kept)) f.h[j] = 0;
                        }
                        acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.v, pf.v, acc[mb], 0, 0, 0);
                    }
                }
            }
        }
        // acc[mb][v]: value column 16 mb + 4 quarter + v of the head's l16-th query head
        if (c < g.n_kv && l16 < group) {
            float* at = partial + ((size_t)run * n_tokens + token) * ((size_t)n_q * V_DIM) + (size_t)(c * group + l16) * V_DIM + 4 * quarter;
#pragma unroll
            for (int mb = 0; mb < BLOCKS; ++mb) *(f32x4*)(at + 16 * mb) = acc[mb];
        }
        if (c0 + MX_WAVES < g.n_kv) __syncthreads();
    }
}

// Rows whose keys were cut into runs: out = gate * (sum of the runs' partial sums, in order).  A thread takes four
// columns of a row and asks for every run's sums before it adds the first.  `rows` (or null: every row of the batch): the
// rows whose sums lie one after the other, all of `runs` runs; else a row's own number of them (one: it is written already).
__global__ void __launch_bounds__(256) mixed_finish_kernel(const float* __restrict__ partial, size_t partial_stride,
                                                           const int32_t* __restrict__ row_splits, const int32_t* __restrict__ rows, int runs,
                                                           const float* __restrict__ gate,
                                                           int gate_stride, int gate_parts, size_t gate_part_stride,
                                                           bf16_t* __restrict__ out, int width) {
    const size_t at_row = blockIdx.y, row = rows != nullptr ? rows[at_row] : at_row;
    const int n = rows != nullptr ? runs : row_splits[row];
    const int e = 4 * (blockIdx.x * 256 + threadIdx.x);
    if ((rows == nullptr && n <= 1) || e >= width) return;
    // the gate and eight runs' sums are asked for together, the next eight before those are added
    f32x4 part[8], next[8], z = {0.0f, 0.0f, 0.0f, 0.0f};
    auto ask = [&](int s0, f32x4 (&to)[8]) {
#pragma unroll
        for (int s = 0; s < 8; ++s)
            to[s] = s0 + s < n ? *(const f32x4*)(partial + (s0 + s) * partial_stride + at_row * width + e) : (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    };
    ask(0, next);
    if (gate != nullptr)
        for (int p = 0; p < gate_parts; ++p)
#pragma unroll
            for (int v = 0; v < 4; ++v) z[v] += gate[p * gate_part_stride + row * gate_stride + e + v];
    f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = 0; s0 < n; s0 += 8) {
#pragma unroll
        for (int s = 0; s < 8; ++s) part[s] = next[s];
        if (s0 + 8 < n) ask(s0 + 8, next);
#pragma unroll
        for (int s = 0; s < 8; ++s) o += part[s];
    }
    float r[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        r[v] = o[v];
        if (gate != nullptr) r[v] *= 1.0f / (1.0f + __expf(-z[v]));
    }
    uint2 w;
    w.x = (uint32_t)f32_to_bf16(r[0]) | ((uint32_t)f32_to_bf16(r[1]) << 16);
    w.y = (uint32_t)f32_to_bf16(r[2]) | ((uint32_t)f32_to_bf16(r[3]) << 16);
    *(uint2*)(out + row * width + e) = w;
}

extern "C" {

int kipp_mixed_mfma_sizes(int* head_dim, int* v_dim, int* heads_per_wave, int* lds_bytes) {
    *head_dim = HEAD_DIM;
    *v_dim = V_DIM;
    *heads_per_wave = HPW;
    *lds_bytes = MX_LDS_BYTES;
    return 0;
}

// stats: float32 [items][n_q][16][2]; partial: float32 [max_splits][n_rows][n_q V_DIM] (may be null when no tile is cut);
// row_splits: int32 [n_rows], the runs of each row's tile; out: bfloat16 [n_rows][n_q V_DIM].
int kipp_mixed_attention_mfma(const void* q, const void* k_cache, const void* v_cache, void* out,
                              const float* gate, int gate_stride, int gate_parts,
                              const int32_t* item_entry, const int32_t* item_row0, const int32_t* item_split,
                              const int32_t* item_nsplits, int n_items, const int32_t* row_splits, int max_splits,
                              const int32_t* q_start, const int32_t* q_len, const int32_t* ctx_len,
                              const int32_t* block_table, int max_blocks,
                              const float* r1, const float* r2, const float* sink, const float* mix,
                              float* stats, float* partial,
                              int n_rows, int n_q, int n_kv, int d, int dv, int page, float scale, int window, int keep_first,
                              hipStream_t stream) {
    if (n_items <= 0 || n_rows <= 0) return 0;
    if (V_DIM % V_SLICE || V_SLICE % 16) return -5;
    if (d != HEAD_DIM || dv != V_DIM || n_kv <= 0 || n_q % n_kv || n_q > MX_WAVES * HPW || n_q > MX_HPAD) return -1;
    if (SHARED_KV && HPW > 1 && (n_q / n_kv) % HPW) return -4;
    if (page <= 0 || page % 16 || max_splits < 1 || (max_splits > 1 && (partial == nullptr || row_splits == nullptr))) return -2;
    MixedGeometry g;
    g.item_entry = item_entry; g.item_row0 = item_row0; g.item_split = item_split; g.item_nsplits = item_nsplits;
    g.q_start = q_start; g.q_len = q_len; g.ctx_len = ctx_len; g.block_table = block_table;
    g.max_blocks = max_blocks; g.page = page; g.n_q = n_q; g.n_kv = n_kv; g.window = window; g.keep_first = keep_first;
    g.scale = scale; g.r1 = r1; g.r2 = r2;
    const int lds = MX_LDS_BYTES;
    static bool raised = false;
    if (!raised) {
        if (hipFuncSetAttribute((const void*)mixed_values_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return -3;
        raised = true;
    }
    const size_t gate_part_stride = (size_t)n_rows * gate_stride;
    const size_t partial_stride = (size_t)n_rows * n_q * V_DIM;
    hipLaunchKernelGGL(mixed_stats_kernel, dim3(n_items), dim3(MX_THREADS), 0, stream, g, (const bf16_t*)q, (const bf16_t*)k_cache, stats);
    hipLaunchKernelGGL(mixed_values_kernel, dim3(n_items, V_DIM / V_SLICE), dim3(MX_THREADS), lds, stream, g, (const bf16_t*)q,
                       (const bf16_t*)k_cache, (const bf16_t*)v_cache, stats, sink, mix, gate, gate_stride, gate_parts,
                       gate_part_stride, (bf16_t*)out, partial, partial_stride);
    if (max_splits > 1)
        hipLaunchKernelGGL(mixed_finish_kernel, dim3((n_q * V_DIM / 4 + 255) / 256, n_rows), dim3(256), 0, stream, partial, partial_stride, row_splits,
                           (const int32_t*)nullptr, 0, gate, gate_stride, gate_parts, gate_part_stride, (bf16_t*)out, n_q * V_DIM);
    return KIPP_LAUNCH_CHECK();
}

// Single tokens: rows[i] of the batch for i < n_tokens, `at_a_time` of them after another.  scores: float32
// [at_a_time][max_tiles][64][32]; stats: float32 [at_a_time][n_runs][32][2]; partial: float32 [n_runs][at_a_time][n_q V_DIM]; out: bfloat16 [n_rows][n_q V_DIM], the rows named.
// max_tiles: tiles of 64 keys that a token can see at most.
int kipp_mixed_attention_single(const void* q, const void* k_cache, const void* v_cache, void* out, const float* gate, int gate_stride,
                                int gate_parts, const int32_t* rows, int n_tokens, int at_a_time, const int32_t* positions, const int32_t* seq_of_token,
                                const int32_t* block_table, int max_blocks, const float* r1, const float* r2, const float* sink,
                                const float* mix, float* scores, float* stats, float* partial, int n_runs, int max_tiles, int n_rows, int n_q,
                                int n_kv, int d, int dv, int page, float scale, int window, int keep_first, hipStream_t stream) {
    if (n_tokens <= 0 || n_rows <= 0) return 0;
    if (d != HEAD_DIM || dv != V_DIM || n_kv <= 0 || n_q % n_kv || n_q > MX_HPAD || n_q / n_kv > 16) return -1;
    if (page <= 0 || page % 16 || n_runs < 1 || max_tiles < 1 || at_a_time < 1) return -2;
    SingleGeometry g;
    g.positions = positions; g.seq_of_token = seq_of_token; g.block_table = block_table;
    g.max_blocks = max_blocks; g.page = page; g.n_q = n_q; g.n_kv = n_kv; g.window = window; g.keep_first = keep_first;
    g.n_runs = n_runs; g.max_tiles = max_tiles; g.scale = scale; g.r1 = r1; g.r2 = r2;
    for (int from = 0; from < n_tokens; from += at_a_time) {
        const int n = n_tokens - from < at_a_time ? n_tokens - from : at_a_time;
        g.rows = rows + from;
        hipLaunchKernelGGL(mixed_single_scores_kernel, dim3(n_runs, n), dim3(MX_THREADS), 0, stream, g, (const bf16_t*)q, (const bf16_t*)k_cache,
                           scores, stats);
        hipLaunchKernelGGL(mixed_single_values_kernel, dim3(n_runs, n), dim3(MX_THREADS), 0, stream, g, (const bf16_t*)v_cache,
                           (const float*)scores, (const float*)stats, sink, mix, partial);
        hipLaunchKernelGGL(mixed_finish_kernel, dim3((n_q * V_DIM / 4 + 255) / 256, n), dim3(256), 0, stream, (const float*)partial,
                           (size_t)n * n_q * V_DIM, (const int32_t*)nullptr, g.rows, n_runs, gate, gate_stride, gate_parts,
                           (size_t)n_rows * gate_stride, (bf16_t*)out, n_q * V_DIM);
    }
    return KIPP_LAUNCH_CHECK();
}

}  // extern "C"
