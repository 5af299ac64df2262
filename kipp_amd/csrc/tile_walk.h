// The walk over K that the matrix products for many rows share: bfloat16 operands, float32 accumulation on
// v_mfma_f32_32x32x16_bf16, X and W a step of 32 columns at a time from global memory straight into LDS
// (`gemm_tiles.hip` says why it is laid out as it is; `moe.hip` walks the same way over the rows of one expert).
#pragma once
#include "common.h"

#define BK 32                                      // columns of a step
#define CHUNKS (BK / 8)                            // 16-byte chunks of a row of a piece
#define GROUP_ROWS (16 / CHUNKS)                   // rows that share 256 bytes of LDS
#define INSTR_ROWS (4 * GROUP_ROWS)                // rows one DMA instruction of a wave brings (1 KB)

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

union Frag {
    u32x4 u;
    bf16x8 v;
};

#define LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))
#define GLOBAL_PTR(p) ((const __attribute__((address_space(1))) void*)(p))

// Every operand register of a set is tied to the wait for its reads, so that no product moves in front of it.
template <int WM, int WN>
__device__ __forceinline__ void wait_reads(u32x4 (&fa)[WM], u32x4 (&fb)[WN]) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < WM; ++i) asm volatile("" : "+v"(fa[i]));
#pragma unroll
    for (int j = 0; j < WN; ++j) asm volatile("" : "+v"(fb[j]));
}

// The DMA: an instruction of a wave brings INSTR_ROWS rows of a piece; a lane brings the 16 bytes that belong at its
// place of the KB: group g = 4 i + lane / 16 of GROUP_ROWS rows, slot s = lane % 16, which holds chunk s ^ (g % CHUNKS) of
// the group: row (that / CHUNKS) of the group, columns 8 (that % CHUNKS) .. + 7.
__device__ __forceinline__ void dma_place(int lane, int& row, int& col8) {
    const int q4 = lane >> 4, s16 = lane & 15;
    const int in_group = s16 ^ (q4 & (CHUNKS - 1));
    row = GROUP_ROWS * q4 + in_group / CHUNKS;
    col8 = (in_group % CHUNKS) * 8;
}

// nk steps of K into acc: WM x WN products of 32 x 32 a half step for this wave.  A step's buffer of STAGE_BYTES holds its
// piece of X, then (at X_PIECE) of W; this wave brings XI and WI KB of them, to x_dst and w_dst; a lane's source is
// base + step + its own 32-bit offset; this wave's operands begin at a_base and b_base of a step's buffer.
template <int WM, int WN, int XI, int WI, int STAGES, int STAGE_BYTES>
__device__ __forceinline__ void tile_walk(unsigned char* lds, int lane, const unsigned char* x_base, const unsigned char* w_base,
                                          uint32_t (&x_src)[XI], uint32_t (&w_src)[WI], int x_dst, int w_dst, int a_base, int b_base, int nk,
                                          f32x16 (&acc)[WM][WN]) {
    constexpr int LOADS = XI + WI;                                // DMA instructions a wave issues a step
    constexpr int NM = WM * WN;                                   // products of a half step
    constexpr int NR = WM + WN;                                   // operand reads of a half step
    static_assert((STAGES - 1) * LOADS < 64, "the wait counts below must fit the counter");
    const int l32 = lane & 31, hh = lane >> 5;
    // where step `step` of an operand begins, for every lane: pinned to scalar registers (left to itself the
    // compiler adds the lane's offset first and then walks a 64-bit vector address along K)
    auto step_base = [&](const unsigned char* base, int step) {
        const unsigned char* at = base + (size_t)step * (BK * 2);
        asm volatile("" : "+s"(at));
        return at;
    };
    auto issue_one = [&](const unsigned char* x_at, const unsigned char* w_at, int stage, int n) {   // DMA instruction n (0 .. LOADS - 1) of a step
        // the lane's offset passes through an empty asm here, so that its widening to 64 bits stands beside the
        // load: the compiler then takes the form "scalar base + 32-bit vector offset" and adds nothing per load
        // (widened once outside the walk, the offset would cost a 64-bit vector add for every load)
        // (in place: the offset keeps its own register for the whole walk.  A copy in a scratch register could be
        // handed to a read out of LDS as its destination right behind the DMA instruction, and nothing says how
        // long the memory pipeline takes to fetch an instruction's address registers)
        unsigned char* dst = lds + stage * STAGE_BYTES;
        if (n < XI) {
            uint32_t& off = x_src[n < XI ? n : 0];
            asm volatile("" : "+v"(off));
            __builtin_amdgcn_global_load_lds(GLOBAL_PTR(x_at + off), LDS_PTR(dst + x_dst + 1024 * n), 16, 0, 0);
        } else {
            uint32_t& off = w_src[n < XI ? 0 : n - XI];
            asm volatile("" : "+v"(off));
            __builtin_amdgcn_global_load_lds(GLOBAL_PTR(w_at + off), LDS_PTR(dst + w_dst + 1024 * (n - XI)), 16, 0, 0);
        }
    };

    // ---- a lane's place in the operands: row 32 j + l32 of the wave's rows, chunk 2 t + hh of the step
    int frag_at[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int group = l32 / GROUP_ROWS;
        frag_at[t] = group * 256 + (((CHUNKS * (l32 % GROUP_ROWS) + 2 * t + hh) ^ (group & (CHUNKS - 1))) << 4);
    }
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    // ---- the walk over K.  The operands of a product leave LDS through reads written out by hand (through
    //      ordinary loads the compiler would make every read wait for all DMA into LDS that is on its way), asked
    //      for one half step ahead.  Steps beyond the last are asked for again from the last one (into a buffer
    //      that nobody reads any more), so that the count of loads on their way is the same at every step.
    u32x4 a[2][WM], b[2][WN];
    // read R of a half step: the first row operand, every column operand, then the other row operands (the
    // order in which the products below want them)
#define KIPP_READ_ONE(T, STEP, KS, R)                                                                              \
    do {                                                                                                           \
        const uint32_t st_ = (uint32_t)(uintptr_t)LDS_PTR(lds + ((STEP) % STAGES) * STAGE_BYTES);                  \
        const uint32_t a_at_ = st_ + a_base + frag_at[KS], b_at_ = st_ + b_base + frag_at[KS];                     \
        if ((R) == 0) asm volatile("ds_read_b128 %0, %1" : "=v"(a[T][0]) : "v"(a_at_));                            \
        else if ((R) <= WN)                                                                                        \
            asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(b[T][(R) <= WN ? (R) - 1 : 0]) : "v"(b_at_), "i"(((R) - 1) * 32 * BK * 2)); \
        else                                                                                                       \
            asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(a[T][(R) > WN ? (R) - WN : 0]) : "v"(a_at_), "i"(((R) - WN) * 32 * BK * 2)); \
    } while (0)
#define KIPP_PRODUCT(T, M_)                                                                         \
    do {                                                                                            \
        Frag fa, fb;                                                                                \
        fa.u = a[T][(M_) / WN];                                                                     \
        fb.u = b[T][(M_) % WN];                                                                     \
        acc[(M_) / WN][(M_) % WN] =                                                                 \
            __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa.v, fb.v, acc[(M_) / WN][(M_) % WN], 0, 0, 0); \
    } while (0)

    // The DMA instructions of a step go out in two groups, half a step apart: the first LOADS_EARLY of step
    // kt + STAGES behind the products of the second half of step kt (into the buffer of step kt, which every wave
    // has left at the barrier in the middle of step kt), the others behind the products of the first half of
    // step kt + 1.  So a wave asks for 1 KB every third product and not every product for half of the time:
    // the four waves' requests together then stay under what the compute unit's path to memory takes, and no
    // wave waits to hand one in (measured: 20 cycles an instruction when they all came behind one another).
    constexpr int LOADS_EARLY = (LOADS + 1) / 2, LOADS_LATE = LOADS - LOADS_EARLY;
    // the items of a half step: NR reads of operands, one behind each of the first products, then D DMA
    // instructions spread over the products that are left (all spread evenly where there are more items than products)
#define KIPP_ITEMS(D, M_, READ, DMA)                                                          \
    do {                                                                                      \
        constexpr int T_ = NR + (D);                                                          \
        _Pragma("unroll") for (int p_ = 0; p_ < T_; ++p_) {                                   \
            const int behind_ = T_ > NM ? p_ * NM / T_ : (p_ < NR ? p_ : NR + (p_ - NR) * (NM - NR) / (D)); \
            if (behind_ != (M_)) continue;                                                    \
            if (p_ >= NR) { DMA(p_ - NR); }                                                   \
            else { READ(p_); }                                                                \
        }                                                                                     \
    } while (0)

#pragma unroll
    for (int s = 0; s < STAGES; ++s) {
        const unsigned char* x_at = step_base(x_base, min(s, nk - 1));
        const unsigned char* w_at = step_base(w_base, min(s, nk - 1));
#pragma unroll
        for (int n = 0; n < (s == STAGES - 1 ? LOADS_EARLY : LOADS); ++n) issue_one(x_at, w_at, s, n);
    }
    // step 0 has arrived when steps 1 .. STAGES - 2 and the early part of step STAGES - 1 may still be on their way
    constexpr int AFTER_FIRST = (STAGES - 2) * LOADS + LOADS_EARLY;
    static_assert(AFTER_FIRST < 64, "the wait counts must fit the counter");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (AFTER_FIRST & 15) | ((AFTER_FIRST >> 4) << 14));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();                                  // bare, as in the walk below
    asm volatile("" ::: "memory");
#pragma unroll
    for (int r = 0; r < NR; ++r) KIPP_READ_ONE(0, 0, 0, r);
    for (int kt = 0; kt < nk; ++kt) {
        // first half: products of columns 0 .. 15 of the step; the operands of the second half arrive meanwhile,
        // and the late DMA instructions of step kt + STAGES - 1 go out, into the buffer of step kt - 1
        // (the scheduler may not carry instructions over the marks: the order written here is the order meant)
        wait_reads<WM, WN>(a[0], b[0]);
        __builtin_amdgcn_sched_barrier(0);
        const int late = min(kt + STAGES - 1, nk - 1), late_stage = (kt + STAGES - 1) % STAGES;
        const unsigned char* x_late = step_base(x_base, late);
        const unsigned char* w_late = step_base(w_base, late);
#define KIPP_READ_A(R) KIPP_READ_ONE(1, kt, 1, R)
#define KIPP_DMA_A(N_) issue_one(x_late, w_late, late_stage, LOADS_EARLY + (N_))
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            KIPP_PRODUCT(0, m);
            KIPP_ITEMS(LOADS_LATE, m, KIPP_READ_A, KIPP_DMA_A);
            __builtin_amdgcn_sched_barrier(0);
        }
        // second half: every wave's part of the next step has arrived (what may still be on its way: the steps
        // behind it), and every wave is done with this step's buffer (its operands are in registers), into which
        // the early DMA instructions of step kt + STAGES now go
        wait_reads<WM, WN>(a[1], b[1]);
        __builtin_amdgcn_s_waitcnt(0x0F70 | (((STAGES - 2) * LOADS) & 15) | ((((STAGES - 2) * LOADS) >> 4) << 14));
        // the bare barrier: __syncthreads() also fences, and the fence waits for EVERY load into LDS that is on
        // its way (the compiler writes vmcnt(0) for it), which would leave nothing in flight across a step
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const int ahead = min(kt + STAGES, nk - 1);
        const unsigned char* x_ahead = step_base(x_base, ahead);
        const unsigned char* w_ahead = step_base(w_base, ahead);
#define KIPP_READ_B(R) KIPP_READ_ONE(0, kt + 1, 0, R)
#define KIPP_DMA_B(N_) issue_one(x_ahead, w_ahead, kt % STAGES, N_)
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            KIPP_PRODUCT(1, m);
            KIPP_ITEMS(LOADS_EARLY, m, KIPP_READ_B, KIPP_DMA_B);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#undef KIPP_READ_A
#undef KIPP_DMA_A
#undef KIPP_READ_B
#undef KIPP_DMA_B
#undef KIPP_ITEMS
    wait_reads<WM, WN>(a[0], b[0]);
    __builtin_amdgcn_s_waitcnt(0x0F70);      // nothing may still be on its way into LDS when the buffers are used again
#undef KIPP_READ_ONE
#undef KIPP_PRODUCT
}
