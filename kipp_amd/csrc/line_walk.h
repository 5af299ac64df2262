// The walk over K that the matrix products for many rows share: bfloat16 operands, float32 accumulation on
// v_mfma_f32_16x16x32_bf16, X and W a step of 64 columns at a time from global memory straight into LDS
// (`gemm_tiles.hip` says why it is laid out as it is).
//
// A workgroup of eight waves, GM down and GN across; a wave 2 XF x 2 WF fragments of 16 x 16 outputs.  A step's 64 columns of a row
// are one whole memory line.  Its pieces are the two halves of the tile's rows of X and the two of W: a half holds, for every wave down
// (across), the first or the last 16 XF (16 WF) of that wave's rows.  A step is four phases, each the products of one half of X with one of W
// over all 64 columns, in the order (0, F) (0, S) (1, S) (1, F): a phase needs one new half only, whose operands leave LDS during the
// phase before, and F is 0 in even steps and 1 in odd ones, so that the half a step ends with makes room for the one the next begins with.
//
// LDS holds two steps.  A half's place is free as soon as every wave has its operands in registers, long before its step ends,
// and is filled for the step after the next one then: X 0 and W F from the barrier ahead of phase 0 on (group 0), X 1 and W S from the
// barrier ahead of phase 2 on (group 1).  They are wanted six phases later (3,000 cycles at 256 x 256 outputs).
#pragma once
#include "common.h"

#define BK 32                                      // K is a multiple of this: a last step may be half a one
#define LINE_ROWS 8                                // rows one DMA instruction of a wave brings: 128 bytes each

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

union Frag {
    u32x4 u;
    bf16x8 v;
};

#define LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))
#define GLOBAL_PTR(p) ((const __attribute__((address_space(1))) void*)(p))

template <int XF, int WF, int GM, int GN>
struct LineWalk {
    static constexpr int WAVES = GM * GN;
    static constexpr int TM = 32 * XF * GM, TN = 32 * WF * GN;                  // the workgroup's tile
    static constexpr int X_HALF = TM / 2 * 128, W_HALF = TN / 2 * 128;           // bytes of a half of a step
    static constexpr int X_ALL = TM / 2 / LINE_ROWS, W_ALL = TN / 2 / LINE_ROWS; // DMA instructions of a half
    // a wave's share of them; four that are left over go to waves 0 .. 3 for one half of a step and to waves 4 .. 7 for the other
    static constexpr int X_EACH = X_ALL / WAVES, X_LEFT = X_ALL % WAVES, W_EACH = W_ALL / WAVES, W_LEFT = W_ALL % WAVES;
    static constexpr int X_MOST = X_EACH + (X_LEFT > 0), W_MOST = W_EACH + (W_LEFT > 0);
    static constexpr int LDS_BYTES = 4 * X_HALF + 4 * W_HALF;
    static_assert(WAVES == 8 && (X_LEFT == 0 || X_LEFT == 4) && (W_LEFT == 0 || W_LEFT == 4), "shares of eight waves");
    static_assert(4 * X_HALF <= 65536 && 4 * W_HALF <= 65536, "a read's offset has 16 bits");

    // which row of a half DMA instruction `n` of this wave brings for this lane
    static __device__ __forceinline__ int x_row(int n, int wave, int lane) { return row_of(n, X_EACH, wave, lane); }
    static __device__ __forceinline__ int w_row(int n, int wave, int lane) { return row_of(n, W_EACH, wave, lane); }
    static __device__ __forceinline__ int slot_of(int n, int each, int wave) { return n < each ? wave * each + n : WAVES * each + (wave & 3); }
    static __device__ __forceinline__ int row_of(int n, int each, int wave, int lane) { return slot_of(n, each, wave) * LINE_ROWS + (lane >> 3); }
    // row `p` of half `h` as a row of the tile
    static __device__ __forceinline__ int x_tile_row(int h, int p) { return p / (16 * XF) * (32 * XF) + h * 16 * XF + p % (16 * XF); }
    static __device__ __forceinline__ int w_tile_row(int h, int p) { return p / (16 * WF) * (32 * WF) + h * 16 * WF + p % (16 * WF); }
};

// The columns (the first of eight) that this lane brings of row `p` of a half: in LDS a row is 128 bytes, its eight 16-byte chunks permuted by the
// row, so that the 16 lanes which read one operand column together meet sixteen different places (no bank conflict).  A walk of a single half
// step (`steps` of BK columns: 1) takes its 32 columns from both halves of the line.
__device__ __forceinline__ int line_col(int lane, int p, int steps) {
    const int chunk = (lane & 7) ^ ((p >> 1) & 7);
    return 8 * (steps == 1 ? chunk | 4 : chunk);
}

template <int N>
__device__ __forceinline__ void tie_operands(u32x4 (&f)[N]) {       // no product moves in front of the wait for its operands
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(f[i]));
}

template <int V>
struct Const {
    static constexpr int value = V;
};

// `steps` steps of BK columns into acc: acc[i][j] is the wave's fragment of rows 16 i of X and 16 j of W, transposed: lane l holds row
// l % 16 of X and rows 4 (l / 16) .. + 3 of W.  A lane's source for DMA instruction n of half h is base + step + src[h][n].  An output is summed
// over K in one order whatever the tile.  `lds` holds LDS_BYTES, which nobody reads or writes any more.
template <int XF, int WF, int GM, int GN>
__device__ __forceinline__ void line_walk(unsigned char* lds, int lane, int wave, const unsigned char* x_base, const unsigned char* w_base,
                                          uint32_t (&x_src)[2][LineWalk<XF, WF, GM, GN>::X_MOST],
                                          uint32_t (&w_src)[2][LineWalk<XF, WF, GM, GN>::W_MOST], int steps, f32x4 (&acc)[2 * XF][2 * WF]) {
    using C = LineWalk<XF, WF, GM, GN>;
    constexpr int X_HALF = C::X_HALF, W_HALF = C::W_HALF;
    constexpr int PRODUCTS = XF * WF * 2;                                // of a phase
    constexpr int X_READS = XF * 2, W_READS = WF * 2;                    // of a half
    constexpr int ITEMS = C::X_MOST + C::W_MOST;                         // DMA instructions of a group, at most
    constexpr int FEWEST = C::X_EACH + C::W_EACH;                        // ... at least
    constexpr int TWO_GROUPS = 2 * FEWEST + (C::X_LEFT > 0) + (C::W_LEFT > 0);      // of two groups behind one another, in every wave
    static_assert(TWO_GROUPS + FEWEST < 64, "the wait counts must fit the counter");
    const int l16 = lane & 15, quarter = lane >> 4;
    const bool low = wave < 4;
    const int odd = steps & 1, count = (steps + 1) >> 1;                 // the last of `count` steps of 64 columns may be half a one
    // a lane's place in the operands: row l16 of a fragment, chunk 4 t + quarter of its line
    uint32_t x_at[2], w_at[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const uint32_t at = (uint32_t)(uintptr_t)LDS_PTR(lds) + l16 * 128 + (((4 * t + quarter) ^ ((l16 >> 1) & 7)) << 4);
        x_at[t] = at + wave / GN * (16 * XF * 128);
        w_at[t] = at + 4 * X_HALF + wave % GN * (16 * WF * 128);
    }
#pragma unroll
    for (int i = 0; i < 2 * XF; ++i)
#pragma unroll
        for (int j = 0; j < 2 * WF; ++j) acc[i][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};

    // where a step begins, for every lane: pinned to scalar registers (left to itself the compiler adds the lane's offset
    // first and then walks a 64-bit vector address along K).  Steps beyond the last are asked for again from the last one,
    // so that the count of loads on their way is the same at every step.  A last half step ends where K does: its columns are
    // the second half of the line that is brought.
    auto step_base = [&](const unsigned char* base, int step) __attribute__((always_inline)) {
        const unsigned char* at = base + (ptrdiff_t)min(step, count - 1) * 128 - (step >= count - 1 ? 64 * odd : 0);
        asm volatile("" : "+s"(at));
        return at;
    };
    // a lane's offset passes through an empty asm, so that its widening to 64 bits stands beside the load: the compiler then
    // takes the form "scalar base + 32-bit vector offset" and adds nothing per load (in place: a copy could be handed to a
    // read out of LDS as its destination right behind the DMA instruction)
    auto bring = [&](const unsigned char* at, uint32_t& off, unsigned char* to) __attribute__((always_inline)) {
        asm volatile("" : "+v"(off));
        __builtin_amdgcn_global_load_lds(GLOBAL_PTR(at + off), LDS_PTR(to), 16, 0, 0);
    };
    // DMA instruction n of group G of a step into buffer BUF: X half G, then W half `w_half`
    auto dma = [&](auto group, const unsigned char* xa, const unsigned char* wa, int buf, int w_half, int n) __attribute__((always_inline)) {
        constexpr int G = decltype(group)::value;
        if (n < C::X_MOST) {
            unsigned char* to = lds + (2 * buf + G) * X_HALF + C::slot_of(n, C::X_EACH, wave) * 1024;
            if (n < C::X_EACH || low == (G == 0)) bring(xa, x_src[G][n < C::X_MOST ? n : 0], to);
        } else {
            const int i = n - C::X_MOST;
            unsigned char* to = lds + 4 * X_HALF + (2 * buf + w_half) * W_HALF + C::slot_of(i, C::W_EACH, wave) * 1024;
            // (where both operands leave four over, a wave brings one of them in either group)
            if (i < C::W_EACH || low == (C::X_LEFT > 0 ? G == 1 : G == 0)) bring(wa, w_src[w_half][i < 0 ? 0 : i], to);
        }
    };
    u32x4 x[2][X_READS], w[2][W_READS];                                 // the halves' operands
    // reads out of LDS written out by hand: through ordinary loads the compiler would make every one wait for all DMA
    // into LDS that is on its way
    auto read_x = [&](int buf, int h, int r) __attribute__((always_inline)) {
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(x[h][r]) : "v"(x_at[r / XF]), "i"((2 * buf + h) * X_HALF + r % XF * 2048));
    };
    auto read_w = [&](int buf, int h, int r) __attribute__((always_inline)) {
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(w[h][r]) : "v"(w_at[r / WF]), "i"((2 * buf + h) * W_HALF + r % WF * 2048));
    };
    auto product = [&](int hx, int hw, int m) __attribute__((always_inline)) {
        const int t = m / (XF * WF), i = m % (XF * WF) / WF, j = m % WF;
        Frag fx, fw;
        fx.u = x[hx][t * XF + i];
        fw.u = w[hw][t * WF + j];
        acc[hx * XF + i][hw * WF + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw.v, fx.v, acc[hx * XF + i][hw * WF + j], 0, 0, 0);
    };
#define KIPP_VMCNT(N) __builtin_amdgcn_s_waitcnt(0x0F70 | ((N) & 15) | (((N) >> 4) << 14))
#define KIPP_LGKM() asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory")
    // the bare barrier: __syncthreads() also fences, and the fence waits for EVERY load into LDS that is on its way (the
    // compiler writes vmcnt(0) for it), which would leave nothing in flight across a step
#define KIPP_BARRIER()                  \
    do {                                \
        asm volatile("" ::: "memory");  \
        __builtin_amdgcn_s_barrier();   \
        asm volatile("" ::: "memory");  \
    } while (0)
    // a phase: products of X half HX with W half HW, R reads and D DMA instructions spread behind them, the reads first
    // (the scheduler may not carry instructions over the marks: the order written here is the order meant)
#define KIPP_PHASE(HX, HW, R, READ, D, DMA)                                    \
    _Pragma("unroll") for (int m = 0; m < PRODUCTS; ++m) {                     \
        product(HX, HW, m);                                                    \
        _Pragma("unroll") for (int p_ = 0; p_ < (R) + (D); ++p_) {             \
            if (p_ * PRODUCTS / ((R) + (D)) != m) continue;                    \
            if (p_ < (R)) { READ(p_); } else { DMA(p_ - (R)); }                \
        }                                                                      \
        __builtin_amdgcn_sched_barrier(0);                                     \
    }

#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const unsigned char *xa = step_base(x_base, s), *wa = step_base(w_base, s);
#pragma unroll
        for (int n = 0; n < ITEMS; ++n) dma(Const<0>{}, xa, wa, s, s, n);
#pragma unroll
        for (int n = 0; n < ITEMS; ++n) dma(Const<1>{}, xa, wa, s, 1 - s, n);
    }
    KIPP_VMCNT(TWO_GROUPS + FEWEST);               // group 0 of step 0 is there; three groups may be on their way
    KIPP_BARRIER();
#pragma unroll
    for (int r = 0; r < X_READS; ++r) read_x(0, 0, r);
#pragma unroll
    for (int r = 0; r < W_READS; ++r) read_w(0, 0, r);

    auto step = [&](auto buffer, int kt) __attribute__((always_inline)) {
        constexpr int BUF = decltype(buffer)::value, F = BUF, S = 1 - F;
        const unsigned char *xa = step_base(x_base, kt + 2), *wa = step_base(w_base, kt + 2);
        // a group's instructions are shared out over its two phases by what those have to read
        constexpr int EARLY = ITEMS / 2 + (W_READS < X_READS ? (ITEMS + 1) / 4 : 0), LATE = ITEMS - EARLY;
#define KIPP_READ_WS(r) read_w(BUF, S, r)
#define KIPP_READ_X1(r) read_x(BUF, 1, r)
#define KIPP_READ_X0(r) read_x(1 - BUF, 0, r)
#define KIPP_READ_WF(r) read_w(1 - BUF, S, r)
#define KIPP_DMA_0(n) dma(Const<0>{}, xa, wa, BUF, F, n)
#define KIPP_DMA_1(n) dma(Const<0>{}, xa, wa, BUF, F, EARLY + (n))
#define KIPP_DMA_2(n) dma(Const<1>{}, xa, wa, BUF, S, n)
#define KIPP_DMA_3(n) dma(Const<1>{}, xa, wa, BUF, S, LATE + (n))
        // every wave has X 0 and W F in registers, and group 1 of this step has arrived
        KIPP_LGKM();
        tie_operands(x[0]);
        tie_operands(w[F]);
        KIPP_VMCNT(TWO_GROUPS);
        KIPP_BARRIER();
        __builtin_amdgcn_sched_barrier(0);
        KIPP_PHASE(0, F, W_READS, KIPP_READ_WS, EARLY, KIPP_DMA_0)
        KIPP_LGKM();
        tie_operands(w[S]);
        __builtin_amdgcn_sched_barrier(0);
        KIPP_PHASE(0, S, X_READS, KIPP_READ_X1, LATE, KIPP_DMA_1)
        // every wave has X 1 and W S in registers, and group 0 of the next step has arrived
        KIPP_LGKM();
        tie_operands(x[1]);
        KIPP_VMCNT(TWO_GROUPS);
        KIPP_BARRIER();
        __builtin_amdgcn_sched_barrier(0);
        KIPP_PHASE(1, S, X_READS, KIPP_READ_X0, LATE, KIPP_DMA_2)
        KIPP_PHASE(1, F, W_READS, KIPP_READ_WF, EARLY, KIPP_DMA_3)
#undef KIPP_READ_WS
#undef KIPP_READ_X1
#undef KIPP_READ_X0
#undef KIPP_READ_WF
#undef KIPP_DMA_0
#undef KIPP_DMA_1
#undef KIPP_DMA_2
#undef KIPP_DMA_3
    };
    const int whole = count - odd;
    int kt = 0;
    for (; kt + 1 < whole; kt += 2) {
        step(Const<0>{}, kt);
        step(Const<1>{}, kt + 1);
    }
    if (kt < whole) step(Const<0>{}, kt);
    KIPP_LGKM();
    tie_operands(x[0]);
    tie_operands(x[1]);
    tie_operands(w[0]);
    tie_operands(w[1]);
    KIPP_VMCNT(0);                               // nothing may still be on its way into LDS when it is used again
    if (odd) {
        // the last half step, whose columns are the second half of its line: read as a whole, then multiplied
        KIPP_BARRIER();
        x_at[1] += (whole & 1) * (2 * X_HALF);
        w_at[1] += (whole & 1) * (2 * W_HALF);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int r = XF; r < X_READS; ++r) read_x(0, h, r);
#pragma unroll
            for (int r = WF; r < W_READS; ++r) read_w(0, h, r);
        }
        KIPP_LGKM();
        tie_operands(x[0]);
        tie_operands(x[1]);
        tie_operands(w[0]);
        tie_operands(w[1]);
#pragma unroll
        for (int h = 0; h < 4; ++h)
#pragma unroll
            for (int m = PRODUCTS / 2; m < PRODUCTS; ++m) product(h >> 1, h & 1, m);
    }
#undef KIPP_PHASE
#undef KIPP_BARRIER
#undef KIPP_LGKM
#undef KIPP_VMCNT
}
