// Matrix product for prompt portions (hundreds to thousands of rows):
// Y[M, N] = X[M, K] . W[N, K]^T, bfloat16 operands, float32 accumulation on
// v_mfma_f32_16x16x32_bf16, K a multiple of 32.
//
// A workgroup of eight waves, two a SIMD, owns a tile of 256 x 256 outputs (also 256 x 192, 256 x 128 and smaller ones, chosen by the
// launcher so that the tiles of a product fill the 256 compute units in whole rounds, or by the caller).  It walks K in steps of 64
// columns (`line_walk.h`), whose pieces of X and W go from global memory straight into LDS (global_load_lds_dwordx4: no
// registers, no waiting wave), two steps deep.  Why so, each measured:
//   whole lines   a step's 128 bytes of a row are one memory line.  Out of L2 a compute unit draws 64-byte halves at three quarters of the rate of whole
//                 lines (15.3 against 20.2 TB/s over all of them), and steps of 32 columns met every line twice;
//   16 x 16       with two waves a SIMD the 32 x 32 x 16 instruction is as fast until the chip meets its power limit, which prompt
//                 products do: on normal operands a kernel that only multiplies sustains 1.82 PFLOP/s with it and 2.03 with 16 x 16 x 32
//                 (`python -m kipp_amd.workloads mfma`), half of whose accumulator traffic it has (same sums in the same order: the same bits);
//   two a SIMD    a wave that issues a DMA instruction or a read cannot issue its next product; the other one does.  With four waves of
//                 128 x 128, one a SIMD, a step takes 3,840 cycles where its products take 2,048, with eight 2,220 (builds that read the shader
//                 clock around the walk, which are not in the tree);
//   64 x 128      outputs a wave, of the cuts of 256 x 256 into eight the one that a few per cent are won by (78 us of 128 x 64's 79 at
//                 2,048 x 2,560 x 9,728).
// What bounds it: by that count the matrix cores are busy 92 cycles of 100 inside the walk, at 1.75 to 1.9 GHz under the power limit, but
// over whole launches of a prefill 47 to 54.  A tile's start and end are 13 us by the fit over all cuts (kFixed), about a quarter of such a
// product's time (K of 2,560: 40 steps of 1.2 us a round): a compute unit holds one workgroup of the large tile, and nothing
// runs beside its first data and its stores.  The rest is the last round, which few tiles fill.  2,048 rows of the 4B
// shape, us, steps of 32 columns (32 x 32 x 16, best cut) / now: QKV 65 / 55, output 49 / 43, gate-up with its end 198 / 163, down 96 / 82;
// 49 sizes from 256 to 1,800 rows: 1.19 in the mean.
//
// An output element is summed over K in the same order whatever the tile: cuts with the same parts of K give the same bits.
//
// The result leaves through one of five ends:
//   slabs   float32 [parts, M, N]: K is split over `parts` workgroups (grid.z) where the tiles
//           alone would leave compute units idle, and the consumer adds the slabs in order
//           (the residual add, the rotary kernel: no atomics, the same bits every time);
//   swiglu  W = [gate; up] ([2 I, K]): a wave's halves of W are gate rows and the up rows that belong
//           to them, a lane holds both values of an output, and bfloat16(silu(gate) * up)
//           [M, I] is all that is written (/root/reference/src/kipp.c:2633-2653);
//   glu     the same with silu or relu, and maybe a bias on gate and up ahead of it;
//   bf16    bfloat16 [M, N];
//   relu2   bfloat16 [M, N] = bfloat16(relu(product)^2).
// W is the instruction's first operand, so that a lane holds neighbouring columns of one row: 16 bytes a store, straight from the
// accumulators.
//
// Tiles are handed to the 8 dies of the GPU in blocks: workgroups that run on one die (every
// eighth one) take tiles that share their rows of W and of X, which that die's L2 then serves.
#include "line_walk.h"

enum { END_SLABS = 0, END_SWIGLU = 1, END_BF16 = 2, END_RELU2 = 3, END_GLU = 4 };
constexpr bool pairs_columns(int end) { return end == END_SWIGLU || end == END_GLU; }      // W = [gate; up]

// silu(g) * u with the exponential of the hardware (base 2)
__device__ __forceinline__ float swiglu_of(float g, float u) {
    return g / (1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * g)) * u;
}

#define BAND 8              // tiles' rows of X that neighbouring tiles share out

// The part of K that part `part` of `parts` walks, in steps of BK columns: cut at whole lines of 64 columns where there are enough of them.
__device__ __forceinline__ void part_of_k(int K, int part, int parts, int& begin, int& steps) {
    const int all = K / BK, lines = (all + 1) / 2, grain = lines >= parts ? 2 : 1, units = grain == 2 ? lines : all;
    begin = (int)((long long)units * part / parts) * grain;
    steps = min((int)((long long)units * (part + 1) / parts) * grain, all) - begin;
}

// What the end END_GLU computes of gate + its bias and up + its bias: as swiglu_of, or with relu in silu's place.  (A product of
// 2,048 x 2,560 with 2 x 9,728 columns that ends in relu: 213 us; as slabs of float32 and an activation behind them it took 232 + 71.)
struct Glu {
    const float* bias;      // [2 inner]: the gate's, then the up's; or null
    int relu;
};

template <int XF, int WF, int GM, int GN, int END>
__global__ void __launch_bounds__(512, (LineWalk<XF, WF, GM, GN>::LDS_BYTES <= 65536 ? 4 : 2)) gemm_tiles_kernel(
    const bf16_t* __restrict__ X, const bf16_t* __restrict__ W, void* __restrict__ Y, int M, int N, int K,
    int tiles_m, int tiles_n, int parts, int inner, int col_begin, int col_end, Glu glu) {
    using Walk = LineWalk<XF, WF, GM, GN>;
    constexpr bool PAIRS = pairs_columns(END);
    constexpr int OUT_N = PAIRS ? Walk::TN / 2 : Walk::TN;         // output columns of a tile
    // The bfloat16 ends: rows 4 q .. + 3 of two neighbouring fragments are W's rows 8 q .. + 7 of the
    // pair's 32, so that a lane holds 8 neighbouring columns of its row.
    constexpr bool EIGHT = END != END_SLABS;
    static_assert(WF % 2 == 0 || !EIGHT, "pairs of fragments across for the bfloat16 ends");
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // ---- which tile: workgroups id, id + 8, id + 16, ... run on one die; each die takes a run of consecutive tiles, rows of X
    //      fastest within bands of up to eight tiles' rows, so that the 32 tiles a die works on share rows of W and of X
    const int n_tiles = tiles_m * tiles_n;
    const int id = blockIdx.x;
    const int per_die = (n_tiles + 7) / 8;
    const int tile = (id & 7) * per_die + (id >> 3);
    if ((id >> 3) >= per_die || tile >= n_tiles) return;          // the grid is rounded up to whole dies
    const int bands = (tiles_m + BAND - 1) / BAND, band_rows = (tiles_m + bands - 1) / bands;
    const int band = tile / (band_rows * tiles_n), in_band = tile % (band_rows * tiles_n), rows_here = min(band_rows, tiles_m - band * band_rows);
    const int tm = band * band_rows + in_band % rows_here, tn = in_band / rows_here;
    const int part = blockIdx.z;
    int s_begin, steps;
    part_of_k(K, part, parts, s_begin, steps);

    // ---- the DMA: an address is a base that all lanes share (it walks along K in scalar registers) plus a lane's own 32-bit
    //      offset, which never changes: no vector arithmetic for an address inside the walk (the launcher refuses
    //      operands of 4 GiB and more)
    uint32_t x_src[2][Walk::X_MOST], w_src[2][Walk::W_MOST];
    const unsigned char* x_base = (const unsigned char*)(X + (size_t)s_begin * BK);
    const unsigned char* w_base = (const unsigned char*)(W + (size_t)s_begin * BK);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int n = 0; n < Walk::X_MOST; ++n) {
            const int p = Walk::x_row(n, wave, lane), r = tm * Walk::TM + Walk::x_tile_row(h, p);
            x_src[h][n] = (uint32_t)(((size_t)min(r, M - 1) * K + line_col(lane, p, steps)) * 2);
        }
#pragma unroll
        for (int n = 0; n < Walk::W_MOST; ++n) {
            const int p = Walk::w_row(n, wave, lane);
            // row p of the half: of fragment f, its row e
            const int f = p / 16 % WF, e = p % 16, across = p / (16 * WF);
            const int within = EIGHT ? f / 2 * 32 + 8 * (e / 4) + 4 * (f % 2) + e % 4 : 16 * f + e;
            int wr;
            if (PAIRS)      // a wave's first half is gate rows, the second the up rows that belong to them
                wr = min(col_begin + tn * OUT_N + 16 * WF * across + within, col_end - 1) + h * inner;
            else
                wr = min(col_begin + tn * OUT_N + 32 * WF * across + 16 * WF * h + within, col_end - 1);
            w_src[h][n] = (uint32_t)(((size_t)wr * K + line_col(lane, p, steps)) * 2);
        }
    }
    f32x4 acc[2 * XF][2 * WF];
    line_walk<XF, WF, GM, GN>(lds, lane, wave, x_base, w_base, x_src, w_src, steps, acc);

    // ---- the ends.  Of fragment (i, j) a lane holds row lane % 16 of X and four rows of W, from 4 (lane / 16) on.
    const int l16 = lane & 15, quarter = lane >> 4;
    const int row0 = tm * Walk::TM + wave / GN * (32 * XF) + l16;
    if constexpr (END == END_SLABS) {
        float* out = (float*)Y + (size_t)part * M * N;
        const int col0 = col_begin + tn * OUT_N + wave % GN * (32 * WF) + 4 * quarter;
        // (a row begins at a multiple of 4 bytes only where N is no multiple of 4.  16 bytes a store there too: 1,923 x 15,473 x 64
        // 28 us, 73 one by one)
        typedef f32x4 __attribute__((aligned(4))) f32x4_any;
#pragma unroll
        for (int i = 0; i < 2 * XF; ++i) {
            const int row = row0 + 16 * i;
            if (row >= M) continue;
#pragma unroll
            for (int j = 0; j < 2 * WF; ++j) {
                const int col = col0 + 16 * j;
                float* at = out + (size_t)row * N + col;
                if (col + 4 <= col_end) {
                    *(f32x4_any*)at = acc[i][j];
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (col + v < col_end) at[v] = acc[i][j][v];
                }
            }
        }
    } else {
        constexpr int RUN = 8;                                     // neighbouring columns a lane holds
        constexpr int RUNS = (PAIRS ? 1 : 2) * 16 * WF / (4 * RUN);  // runs of columns of a row
        const int width = PAIRS ? inner : N;
        const int col0 = col_begin + tn * OUT_N + wave % GN * (PAIRS ? 16 * WF : 32 * WF) + RUN * quarter;
        bf16_t* out = (bf16_t*)Y;
        // (rows begin at any multiple of 2 bytes where the width is no multiple of 8: 16 bytes a store there too, as above.  1,016 x 12,980 x 32 with
        // relu^2 36 -> 13 us, 2,534 x 8,394 x 256 60 -> 23; 120 such sizes of all ends 0.76 of the time in the mean)
        typedef u32x4 __attribute__((aligned(2))) u32x4_any;
#pragma unroll
        for (int g = 0; g < RUNS; ++g) {
            const int col = col0 + 4 * RUN * g;
            float bias_gate[RUN] = {}, bias_up[RUN] = {};
            if (END == END_GLU && glu.bias != nullptr) {
#pragma unroll
                for (int c = 0; c < RUN; ++c) {
                    const int at = min(col + c, col_end - 1);
                    bias_gate[c] = glu.bias[at];
                    bias_up[c] = glu.bias[inner + at];
                }
            }
#pragma unroll
            for (int i = 0; i < 2 * XF; ++i) {
                const int row = row0 + 16 * i;
                bf16_t value_of[RUN];
#pragma unroll
                for (int c = 0; c < RUN; ++c) {
                    const int j = g * (RUN / 4) + c / 4;
                    float value = acc[i][j][c % 4];
                    if (END == END_SWIGLU) value = swiglu_of(value, acc[i][(j + WF) % (2 * WF)][c % 4]);
                    if (END == END_GLU) {
                        const float gate = value + bias_gate[c], up = acc[i][(j + WF) % (2 * WF)][c % 4] + bias_up[c];
                        value = glu.relu ? fmaxf(gate, 0.0f) * up : swiglu_of(gate, up);
                    }
                    if (END == END_RELU2) {
                        value = fmaxf(value, 0.0f);
                        value *= value;
                    }
                    value_of[c] = f32_to_bf16(value);
                }
                if (row >= M) continue;
                bf16_t* at = out + (size_t)row * width + col;
                if (col + RUN <= col_end) {
                    uint32_t packed[RUN / 2];
#pragma unroll
                    for (int c = 0; c < RUN / 2; ++c) packed[c] = (uint32_t)value_of[2 * c] | ((uint32_t)value_of[2 * c + 1] << 16);
                    *(u32x4_any*)at = (u32x4){packed[0], packed[1], packed[2], packed[3]};
                } else {
#pragma unroll
                    for (int c = 0; c < RUN; ++c)
                        if (col + c < col_end) at[c] = value_of[c];
                }
            }
        }
    }
}

// How a product is cut: the workgroup's tile (tm rows of X by tn rows of W) and the parts of K, for a range of output columns.
// The cost of a cut is what its slowest compute unit does: rounds of tiles over the 256 units, each a fixed cost
// (first data, the stores of the end) plus the steps of its part of K, and for every slab beyond the first what the kernel that adds them
// reads once more.  Microseconds, fitted to the times of all cuts of seven products (4B and 8B shapes) at 256 to 1,800 rows.
struct Cut {
    int tm, tn, parts;
    int col_begin, col_end;     // output columns
};

// Tiles 192 wide are there for the slabs alone (a gate's half would be 96).  128 x 192 fills the last round where 128 x 256 leaves 96
// units idle: 2,048 x 2,560 x 2,560 34.0 -> 30.6 us (214 tiles for 160), 1,024 x 5,120 x 2,560 34.2 -> 30.6, 600 x 7,168 x 2,560
// 33.5 -> 29.7.  129 sizes from 200 to 2,048 rows: the plan is 0.44 % over the fastest cut in the mean, without that tile 1.56.
#define N_SHAPES 6
static const int kShapes[N_SHAPES][2] = {{256, 256}, {256, 192}, {256, 128}, {128, 256}, {128, 192}, {128, 128}};
static const double kStep[N_SHAPES] = {0.581, 0.510, 0.339, 0.315, 0.269, 0.217};    // 32 columns of one tile
static const double kFixed[N_SHAPES] = {12.9, 9.7, 7.5, 9.9, 7.7, 4.6};              // start and end of a tile

static double cut_cost(int M, int cols, int steps, int end, int shape, int parts) {
    const int tm = kShapes[shape][0], tn = pairs_columns(end) ? kShapes[shape][1] / 2 : kShapes[shape][1];
    const long long tiles = (long long)((M + tm - 1) / tm) * ((cols + tn - 1) / tn);
    const long long rounds = (tiles * parts + 255) / 256;
    return rounds * (kFixed[shape] + kStep[shape] * ((steps + parts - 1) / parts)) + (1.27 + (double)M * cols * 4.0 / 5e6) * (parts - 1);
}

// The output columns of the whole rounds of 256 tiles of 256 x 256 (0 where there are none, or nothing is left beside them).  What is left
// would hold every compute unit for a round that few of them have a tile in, and goes in smaller tiles.
static int columns_of_whole_rounds(int M, int cols, int end) {
    const int tn = pairs_columns(end) ? 128 : 256;
    const int tiles_m = (M + 255) / 256;
    const long long whole = ((long long)tiles_m * (cols / tn)) / 256 * 256;
    const int first_cols = (int)(whole / tiles_m) * tn;
    return first_cols < cols ? first_cols : 0;
}

// Up to two cuts, side by side in the output's columns.  The float32 end takes one cut, whose parts of K may be
// more than one.  The bfloat16 ends cannot split K; where whole rounds of the largest tile leave a rest of tiles
// that would hold the 256 units for another whole round, the rest of the columns is cut into smaller tiles.
static int plan(int M, int N, int K, int end, int max_parts, Cut* cuts) {
    const int steps = K / BK;
    const int cols = pairs_columns(end) ? N / 2 : N;
    double best = 1e30;
    int n_cuts = 1;
    for (int s = 0; s < N_SHAPES; ++s) {
        if (kShapes[s][1] == 192 && end != END_SLABS) continue;
        for (int parts = 1; parts <= (end == END_SLABS ? max_parts : 1) && parts <= steps; ++parts) {
            const double cost = cut_cost(M, cols, steps, end, s, parts);
            if (cost < best - 1e-9) {
                best = cost;
                cuts[0] = {kShapes[s][0], kShapes[s][1], parts, 0, cols};
            }
        }
    }
    if (end != END_SLABS) {
        // whole rounds of the largest tile first, the rest of the columns in smaller tiles
        const int first_cols = columns_of_whole_rounds(M, cols, end);
        if (first_cols > 0) {
            for (int s = 2; s < N_SHAPES; ++s) {
                if (kShapes[s][1] == 192) continue;
                const double cost = cut_cost(M, first_cols, steps, end, 0, 1) + cut_cost(M, cols - first_cols, steps, end, s, 1);
                if (cost < best - 1e-9) {
                    best = cost;
                    n_cuts = 2;
                    cuts[0] = {256, 256, 1, 0, first_cols};
                    cuts[1] = {kShapes[s][0], kShapes[s][1], 1, first_cols, cols};
                }
            }
        }
    }
    return n_cuts;
}

// The cuts that a product is launched in: the planned ones, or those that `force` names (kipp_gemm_tiles).
static int cuts_of(int M, int N, int K, int end, int max_parts, int force, Cut* cuts) {
    if (!force) return plan(M, N, K, end, max_parts, cuts);
    const int cols = pairs_columns(end) ? N / 2 : N, rest = force / 10000, code = force % 10000;
    cuts[0] = {64 * (code / 100), 64 * (code / 10 % 10), code % 10, 0, cols};        // (tiles without a kernel are refused where they are launched)
    if (code != 2421) return 1;
    const int tile = rest == 0 ? 3 : rest == 1 ? 2 : rest == 3 ? 5 : -1;
    cuts[0] = {256, 256, tile < 0 ? 0 : 1, 0, cols};
    const int first_cols = end == END_SLABS ? 0 : columns_of_whole_rounds(M, cols, end);
    if (first_cols <= 0 || tile < 0) return 1;
    cuts[0].col_end = first_cols;
    cuts[1] = {kShapes[tile][0], kShapes[tile][1], 1, first_cols, cols};
    return 2;
}

template <int XF, int WF, int GM, int GN, int END>
static int launch_cut(const void* X, const void* W, void* Y, int M, int N, int K, const Cut& cut, hipStream_t stream, Glu glu) {
    using Walk = LineWalk<XF, WF, GM, GN>;
    static bool prepared = false;
    if (!prepared) {
        if (hipFuncSetAttribute((const void*)gemm_tiles_kernel<XF, WF, GM, GN, END>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                Walk::LDS_BYTES) != hipSuccess)
            return -6;
        prepared = true;
    }
    const int tn = pairs_columns(END) ? Walk::TN / 2 : Walk::TN;
    const int tiles_m = (M + Walk::TM - 1) / Walk::TM, tiles_n = (cut.col_end - cut.col_begin + tn - 1) / tn;
    const int per_die = (tiles_m * tiles_n + 7) / 8;
    hipLaunchKernelGGL((gemm_tiles_kernel<XF, WF, GM, GN, END>), dim3(per_die * 8, 1, cut.parts), dim3(512), Walk::LDS_BYTES, stream,
                       (const bf16_t*)X, (const bf16_t*)W, Y, M, N, K, tiles_m, tiles_n, cut.parts, N / 2, cut.col_begin,
                       cut.col_end, glu);
    return KIPP_LAUNCH_CHECK();
}

template <int END>
static int launch_end(const void* X, const void* W, void* Y, int M, int N, int K, const Cut& cut, hipStream_t stream, Glu glu) {
    switch (cut.tm * 1000 + cut.tn) {
        case 256256: return launch_cut<2, 4, 4, 2, END>(X, W, Y, M, N, K, cut, stream, glu);
        case 256128: return launch_cut<2, 2, 4, 2, END>(X, W, Y, M, N, K, cut, stream, glu);
        case 128256: return launch_cut<2, 2, 2, 4, END>(X, W, Y, M, N, K, cut, stream, glu);
        case 128128: return launch_cut<1, 2, 4, 2, END>(X, W, Y, M, N, K, cut, stream, glu);
    }
    if constexpr (END == END_SLABS) {
        if (cut.tm == 256 && cut.tn == 192) return launch_cut<2, 3, 4, 2, END>(X, W, Y, M, N, K, cut, stream, glu);
        if (cut.tm == 128 && cut.tn == 192) return launch_cut<1, 3, 4, 2, END>(X, W, Y, M, N, K, cut, stream, glu);
    }
    return -5;
}

static int launch_product(const void* X, const void* W, void* Y, int M, int N, int K, int end, int max_parts, int force, Glu glu,
                          hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || (K % BK) || max_parts <= 0) return -1;
    if (pairs_columns(end) && (N & 1)) return -4;
    // a lane's offset into an operand is 32 bits wide
    if ((unsigned long long)M * K * 2 >= (1ull << 32) || (unsigned long long)N * K * 2 >= (1ull << 32)) return -6;
    Cut cuts[2];
    const int n_cuts = cuts_of(M, N, K, end, max_parts, force, cuts);
    for (int c = 0; c < n_cuts; ++c) {
        const Cut& cut = cuts[c];
        if (cut.parts < 1 || cut.parts > K / BK || (end != END_SLABS && cut.parts != 1)) return -2;
        const int rc = end == END_SLABS ? launch_end<END_SLABS>(X, W, Y, M, N, K, cut, stream, glu)
                       : end == END_SWIGLU ? launch_end<END_SWIGLU>(X, W, Y, M, N, K, cut, stream, glu)
                       : end == END_GLU    ? launch_end<END_GLU>(X, W, Y, M, N, K, cut, stream, glu)
                       : end == END_RELU2  ? launch_end<END_RELU2>(X, W, Y, M, N, K, cut, stream, glu)
                                           : launch_end<END_BF16>(X, W, Y, M, N, K, cut, stream, glu);
        if (rc != 0) return rc;
    }
    return 0;
}

extern "C" {
// parts that kipp_gemm_tiles cuts K into for these sizes when it may use up to `max_parts` (1 for the ends that are not slabs)
int kipp_gemm_tiles_parts(int M, int N, int K, int end, int max_parts) {
    if (K <= 0 || (K % BK) || M <= 0 || N <= 0) return -1;
    Cut cuts[2];
    plan(M, N, K, end, max_parts, cuts);
    return cuts[0].parts;
}

// Microseconds that the plan's prices give for a product cut as planned, or as `force` says (kipp_gemm_tiles); -1 for a cut that these
// sizes do not take.
double kipp_gemm_tiles_cost(int M, int N, int K, int end, int max_parts, int force) {
    if (K <= 0 || (K % BK) || M <= 0 || N <= 0 || max_parts <= 0) return -1.0;
    Cut cuts[2];
    const int n_cuts = cuts_of(M, N, K, end, max_parts, force, cuts);
    double cost = 0.0;
    for (int c = 0; c < n_cuts; ++c) {
        int s = 0;
        while (s < N_SHAPES && (kShapes[s][0] != cuts[c].tm || kShapes[s][1] != cuts[c].tn)) ++s;
        if (s == N_SHAPES || cuts[c].parts < 1 || cuts[c].parts > K / BK || (end != END_SLABS && (cuts[c].parts != 1 || kShapes[s][1] == 192))) return -1.0;
        cost += cut_cost(M, cuts[c].col_end - cuts[c].col_begin, K / BK, end, s, cuts[c].parts);
    }
    return cost;
}

// Y: float32 [parts, M, N] with parts = kipp_gemm_tiles_parts(...) (end 0), bfloat16 [M, N / 2] = silu(gate) * up for
// W = [gate; up] (end 1), bfloat16 [M, N] (end 2), bfloat16 [M, N] = relu(product)^2 (end 3).  K a multiple of 32.  `force`: 0, or 100 a + 10 b + parts for tiles of 64 a x 64 b
// or 2421 (bfloat16 ends: 256 x 256 for whole rounds of tiles, the rest of the columns in 128 x 256; + 10000: the rest in 256 x 128,
// + 30000: in 128 x 128; the slabs' end: 256 x 256) to take that cut whatever the plan says (the runtime's timed choice, tests).
int kipp_gemm_tiles(const void* X, const void* W, void* Y, int M, int N, int K, int end, int max_parts, int force,
                    hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (end != END_SLABS && end != END_SWIGLU && end != END_BF16 && end != END_RELU2) return -3;
    return launch_product(X, W, Y, M, N, K, end, max_parts, force, Glu{}, stream);
}

// Y: bfloat16 [M, N / 2] = act(gate + its bias) * (up + its bias) for W = [gate; up], act relu (`relu` 1) or silu (0); `bias`: float32 [N],
// as W's rows, or null.  `force` as above.
int kipp_gemm_tiles_glu(const void* X, const void* W, void* Y, int M, int N, int K, int relu, const float* bias, int force,
                        hipStream_t stream) {
    return launch_product(X, W, Y, M, N, K, END_GLU, 1, force, Glu{bias, relu != 0}, stream);
}

}  // extern "C"
