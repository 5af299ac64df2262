// True 32-bit matrix product for the float32 path: Y[M,N] = X[M,K] . W[N,K]^T
// with W stored [out][in] row-major like every projection of the model
// (/root/reference/src/kipp.c:2233-2244).  Products and sums are float32 throughout, on the
// matrix cores' float32 instruction (v_mfma_f32_16x16x4_f32: 155 TFLOP/s in a large product here, twice the plain FMA's rate).
//
// An output's bits depend on its two rows and K alone, not on M, on the tile it falls in or on what else is in the
// batch.  K is cut into KPARTS runs of `part_of(K)` numbers (the last ones shorter or empty); a run is one chain of
// instructions, four numbers of k each (16 j + i, + 4, + 8, + 12 for i = 0..3, j counting up from the run's start), and the runs' sums are added
// in order.  Both kernels below do exactly that, W always the instruction's first operand and X its second.
//
//   rows   up to 16 rows of X a workgroup: 16 rows of W, a wave a run of K, straight from memory into the instruction's
//          operands (16 bytes a lane), the runs' sums added through LDS.  Bound by the read of W.  A 16-column fragment of
//          X is multiplied whether its rows are there or not: at one row the matrix cores could feed 19 TB/s.
//   tiles  more rows: 64 or 32 rows of W times 64, 48 or 32 of X a workgroup, a wave a run of K here too, so that every wave of a
//          workgroup multiplies all of its outputs and none waits for another in the walk.  Bound by the instruction's rate (80 %
//          of it at 1,024 rows) and, below a few rounds of tiles, by what the last round leaves idle: the shape goes by that.
// Measured at the 4B shape, W in turn from three copies, us: one row against 19,456 x 2,560 46 (4.3 TB/s), 2,560 x 9,728 34, the head's
// 151,936 x 2,560 325 (4.8 TB/s).  The tiles, against 19,456 x 2,560 / 6,144 x 2,560 / 2,560 x 4,096 / 2,560 x 9,728, beside what these
// rows took before (up to 64 rows of X through the kernel for rows, 64 x 64 tiles of four waves that share a step of K beyond):
//      32 rows    56 / 16 / 20 / 49      106 / 36 / 28 / 73
//      64 rows    78 / 27 / 21 / 49      171 / 64 / 46 / 115
//     128 rows   125 / 45 / 31 / 68      156 / 71 / 92 / 219
//     333 rows   305 / 100 / 69 / 157    402 / 153 / 114 / 271     (110 TFLOP/s; 68 to 83)
//   1,024 rows   814 / 257 / 183 / 454   957 / 308 / 240 / 566
// Without the walk's requests for the next steps the same tiles reach 127 TFLOP/s, without its writes into LDS either 139; operands straight
// from memory into registers, 16 rows of 64 bytes a request, 65 to 85; all sixteen requests of a step behind one another 77 to 100.
#include "common.h"

#define KPARTS 8
#define STEP 32             // numbers of k a tile's wave asks for together; a run is a multiple of it
#define UNITS 256           // compute units
#define XCDS 8              // dies of the chip; consecutive workgroups of a launch go to them in turn
#define ROWS_THREADS (KPARTS * KIPP_WAVE)

typedef __attribute__((ext_vector_type(4))) float f32x4;

__host__ __device__ __forceinline__ int part_of(int K) {
    const int each = (K + KPARTS - 1) / KPARTS;
    return (each + STEP - 1) / STEP * STEP;
}

// Numbers k .. k + 3 of a row, zeros from K on.  VEC: K is a multiple of 4 and rows begin at multiples of four numbers.
template <bool VEC>
__device__ __forceinline__ f32x4 four(const float* __restrict__ row, int k, int K) {
    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (VEC) {
        if (k < K) v = *reinterpret_cast<const f32x4*>(row + k);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (k + i < K) v[i] = row[k + i];
    }
    return v;
}

template <bool VEC>
__device__ __forceinline__ f32x4 four(const bf16_t* __restrict__ row, int k, int K) {
    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (VEC) {
        if (k < K) {
            const uint2 u = *reinterpret_cast<const uint2*>(row + k);
            v[0] = __uint_as_float(u.x << 16);
            v[1] = __uint_as_float(u.x & 0xffff0000u);
            v[2] = __uint_as_float(u.y << 16);
            v[3] = __uint_as_float(u.y & 0xffff0000u);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (k + i < K) v[i] = bf16_to_f32(row[k + i]);
    }
    return v;
}

// The same where all four are inside the row.
template <bool VEC>
__device__ __forceinline__ f32x4 four_inside(const float* __restrict__ at) {
    if (VEC) return *reinterpret_cast<const f32x4*>(at);
    return (f32x4){at[0], at[1], at[2], at[3]};
}

template <bool VEC>
__device__ __forceinline__ f32x4 four_inside(const bf16_t* __restrict__ at) {
    if (!VEC) return (f32x4){bf16_to_f32(at[0]), bf16_to_f32(at[1]), bf16_to_f32(at[2]), bf16_to_f32(at[3])};
    const uint2 u = *reinterpret_cast<const uint2*>(at);
    return (f32x4){__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u)};
}

// 16 numbers of k: lane l holds those at 4 (l / 16) .. + 3 of row l % 16 of either operand.
__device__ __forceinline__ f32x4 mul16(f32x4 w, f32x4 x, f32x4 acc) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[i], acc, 0, 0, 0);
    return acc;
}

// The sums of a fragment lie in lane l as rows 4 (l / 16) .. + 3 (of W) of column l % 16 (a row of X).
template <typename TW, bool VEC>
__global__ void __launch_bounds__(ROWS_THREADS)
gemm_f32_rows_kernel(const float* __restrict__ X, const TW* __restrict__ W, float* __restrict__ Y, int M, int N, int K) {
    __shared__ __attribute__((aligned(16))) float part_s[KPARTS][KIPP_WAVE][4];
    const int wave = threadIdx.x / KIPP_WAVE, lane = threadIdx.x & (KIPP_WAVE - 1);
    const int l16 = lane & 15, h4 = 4 * (lane >> 4);
    const int blocks = (N + 15) / 16, n0 = blockIdx.x % blocks * 16, m0 = blockIdx.x / blocks * 16;
    const TW* w_row = W + (size_t)min(n0 + l16, N - 1) * K;         // rows beyond the last read it and are not stored
    const float* x_row = X + (size_t)min(m0 + l16, M - 1) * K;
    const int part = part_of(K);
    const int k_lo = wave * part, k_hi = min(K, k_lo + part);
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int AHEAD = 8;       // 16-number pieces asked for together
    int k = k_lo;
    for (; k + 16 * AHEAD <= k_hi; k += 16 * AHEAD) {
        f32x4 w[AHEAD], x[AHEAD];
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
            w[j] = four<VEC>(w_row, k + 16 * j + h4, K);
            x[j] = four<VEC>(x_row, k + 16 * j + h4, K);
        }
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) acc = mul16(w[j], x[j], acc);
    }
    for (; k < k_hi; k += 16) {
        const f32x4 w = four<VEC>(w_row, k + h4, K);
        acc = mul16(w, four<VEC>(x_row, k + h4, K), acc);
    }
    *reinterpret_cast<f32x4*>(part_s[wave][lane]) = acc;
    __syncthreads();
    // a thread an output: the runs' sums in order
    if (threadIdx.x < 256) {
        const int at = threadIdx.x;             // place in the fragment: column 16 numbers of n long
        const int n = n0 + (at & 15), m = m0 + (at >> 4);
        const int from = 16 * ((at & 15) >> 2) + (at >> 4);
        float total = 0.0f;
#pragma unroll
        for (int p = 0; p < KPARTS; ++p) total += part_s[p][from][at & 3];
        if (m < M && n < N) Y[(size_t)m * N + n] = total;
    }
}

// A wave stages its own steps of 32 numbers of k in its own part of LDS, so no wave waits for another before the sums.  A row's 128
// bytes lie at 128 times the row in it, 16 byte piece c at place c ^ (row / 2 mod 8): reads and writes then meet every bank once.  A lane
// reads what others of its wave wrote: LDS is in order within a wave, and the wave's barriers keep the compiler to that order.
template <typename TW, int NT, int MT, bool VEC>
__global__ void __launch_bounds__(ROWS_THREADS, 2)
gemm_f32_tiles_kernel(const float* __restrict__ X, const TW* __restrict__ W, float* __restrict__ Y, int M, int N, int K, int n_tiles, int m_tiles) {
    constexpr int ROWS = 16 * (NT + MT), LOADS = ROWS / 8, READS = NT + MT, STAGE = ROWS * STEP, PRODUCTS = 4 * NT * MT;
    __shared__ __attribute__((aligned(16))) float lds[KPARTS * (STAGE > NT * MT * 256 ? STAGE : NT * MT * 256)];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KIPP_WAVE), lane = threadIdx.x & (KIPP_WAVE - 1);
    const int l16 = lane & 15, h4 = 4 * (lane >> 4);
    // workgroups id, id + 8, .. share a die and its L2: a die takes a run of tiles, those of the same rows of W one after the other
    const int tiles = n_tiles * m_tiles, per_die = (tiles + XCDS - 1) / XCDS;
    const int turn = blockIdx.x / XCDS, tile = (blockIdx.x % XCDS) * per_die + turn;
    if (turn >= per_die || tile >= tiles) return;       // uniform over the workgroup
    // The last rows of W are a whole tile that ends with them (the launcher has checked that there are so many): outputs that two
    // tiles have are the same bits in both.
    const int n0 = min(tile / m_tiles * (16 * NT), N - 16 * NT), m0 = tile % m_tiles * (16 * MT);
    // From memory a lane takes four numbers, eight lanes a row's 32: load i brings rows 8 i + lane / 8, first W's, then X's.
    const TW* w_base = W + (size_t)n0 * K;
    const float* x_base = X + (size_t)m0 * K;
    const int ld_row = lane >> 3, ld_k = 4 * (lane & 7);
    const uint32_t w_src = (uint32_t)ld_row * (uint32_t)K + ld_k;
    uint32_t x_src[2 * MT];             // rows of X beyond the last read it and are not stored
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) x_src[i] = (uint32_t)min(8 * i + ld_row, M - 1 - m0) * (uint32_t)K + ld_k;
    float* stage = lds + wave * STAGE;
    float* put_at[2];                   // of even and odd i
    const float* take_at[2];            // of a step's two halves
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        put_at[j] = stage + ld_row * STEP + (ld_k ^ (4 * ((4 * j + (ld_row >> 1)) & 7)));
        take_at[j] = stage + l16 * STEP + ((16 * j + h4) ^ (4 * ((l16 >> 1) & 7)));
    }
    const int part = part_of(K);
    const int k_lo = wave * part, k_hi = min(K, k_lo + part);
    f32x4 acc[NT][MT];
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) acc[a][b] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 next[LOADS], op[2][READS];    // a step on its way; operands of the two halves of the one that is multiplied, W's and then X's
    auto fetch = [&](int i, int k0) {
        next[i] = i < 2 * NT ? four_inside<VEC>(w_base + ((size_t)(8 * i) * K + k0) + w_src)
                             : four_inside<VEC>(x_base + k0 + x_src[i < 2 * NT ? 0 : i - 2 * NT]);
    };
    auto put = [&](int i) { *reinterpret_cast<f32x4*>(put_at[i & 1] + 8 * i * STEP) = next[i]; };
    auto take = [&](int j, int r) { op[j][r] = *reinterpret_cast<const f32x4*>(take_at[j] + 16 * r * STEP); };
    // The sums side by side: an instruction does not wait for the one before.
    auto product = [&](int j, int p) {
        const int i = p / (NT * MT), a = p / MT % NT, b = p % MT;
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(op[j][a][i], op[j][NT + b][i], acc[a][b], 0, 0, 0);
    };
    // A step's first half is in registers when its products begin.  Behind them go, one at a time, the reads of its second half, then a
    // write of the next step into LDS with the request for the same piece of the one after it; behind the second half's products the
    // reads of the next step's first half.  (The two waves of a SIMD begin together, so neither fills the other's gaps, and sixteen
    // requests behind one another held every wave up for a quarter of its step.)  The order is pinned, or the compiler gathers them.
    const int steps = k_hi > k_lo ? (k_hi - k_lo) / STEP : 0, last = k_lo + (steps - 1) * STEP;
    if (steps > 0) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) fetch(i, k_lo);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            put(i);
            fetch(i, min(k_lo + STEP, last));
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < READS; ++r) take(0, r);
        for (int k0 = k_lo; k0 <= last; k0 += STEP) {       // behind the last step it is asked for again
            const int ahead = min(k0 + 2 * STEP, last);
            constexpr int ITEMS = READS + LOADS;
#pragma unroll
            for (int p = 0; p < PRODUCTS; ++p) {
                product(0, p);
#pragma unroll
                for (int q = p * ITEMS / PRODUCTS; q < (p + 1) * ITEMS / PRODUCTS; ++q) {
                    if (q < READS) {
                        take(1, q);
                    } else {
                        if (q == READS) __builtin_amdgcn_wave_barrier();
                        put(q - READS);
                        fetch(q - READS, ahead);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int p = 0; p < PRODUCTS; ++p) {
                product(1, p);
                if (p < READS) take(0, p);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    const int rest = k_lo + steps * STEP;
    if (rest < k_hi) {                              // what K leaves of a step
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            next[i] = i < 2 * NT ? four<VEC>(w_base + (size_t)(8 * i + ld_row) * K, rest + ld_k, K)
                                 : four<VEC>(x_base + x_src[i < 2 * NT ? 0 : i - 2 * NT] - ld_k, rest + ld_k, K);
            put(i);
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (rest + 16 * j >= k_hi) continue;
#pragma unroll
            for (int r = 0; r < READS; ++r) take(j, r);
#pragma unroll
            for (int p = 0; p < PRODUCTS; ++p) product(j, p);
        }
    }
    __syncthreads();                                // every wave is done with its part of LDS
    f32x4(*part_s)[NT * MT][KIPP_WAVE] = reinterpret_cast<f32x4(*)[NT * MT][KIPP_WAVE]>(lds);
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) part_s[wave][a * MT + b][lane] = acc[a][b];
    __syncthreads();
    const bool fours = (N & 3) == 0 && ((uintptr_t)Y & 15) == 0;
    for (int f = wave; f < NT * MT; f += KPARTS) {      // a wave a fragment: the runs' sums in order
        f32x4 total = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int p = 0; p < KPARTS; ++p) total += part_s[p][f][lane];
        const int m = m0 + 16 * (f % MT) + l16, n = n0 + 16 * (f / MT) + h4;
        if (m >= M) continue;
        float* y = Y + (size_t)m * N + n;
        if (fours) {
            *reinterpret_cast<f32x4*>(y) = total;
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v) y[v] = total[v];
        }
    }
}

template <typename TW, int NT, int MT, bool VEC>
static void launch_tiles(const float* X, const TW* W, float* Y, int M, int N, int K, hipStream_t stream) {
    const int n_tiles = (N + 16 * NT - 1) / (16 * NT), m_tiles = (M + 16 * MT - 1) / (16 * MT);
    const int grid = (n_tiles * m_tiles + XCDS - 1) / XCDS * XCDS;
    hipLaunchKernelGGL((gemm_f32_tiles_kernel<TW, NT, MT, VEC>), dim3(grid), dim3(ROWS_THREADS), 0, stream, X, W, Y, M, N, K, n_tiles, m_tiles);
}

// What the busiest compute unit takes for its tiles of nt x mt, one after the other, in products of one fragment: a tile's first requests
// and its sums cost two of them whatever it is (measured with K of 2,560, 4,096 and 9,728, us a round of tiles: 4 x 4 45, 64, 146;
// 4 x 3 35, 50, 114; 4 x 2 25, 36, 81; 2 x 3 20, 29, 65; 2 x 2 15, 21, 49).
static long long tile_price(int M, int N, int nt, int mt) {
    const long long tiles = (long long)((N + 16 * nt - 1) / (16 * nt)) * ((M + 16 * mt - 1) / (16 * mt));
    return (tiles + UNITS - 1) / UNITS * (nt * mt + 2);
}

template <typename TW, bool VEC>
static int launch(const float* X, const TW* W, float* Y, int M, int N, int K, hipStream_t stream) {
    if (M <= 16 || N < 32) {        // tiles hold 32 rows of W or more
        hipLaunchKernelGGL((gemm_f32_rows_kernel<TW, VEC>), dim3((N + 15) / 16 * ((M + 15) / 16)), dim3(ROWS_THREADS), 0, stream, X, W, Y, M, N, K);
        return KIPP_LAUNCH_CHECK();
    }
    static const int shapes[5][2] = {{4, 4}, {4, 3}, {4, 2}, {2, 3}, {2, 2}};
    int best = 4;
    for (int i = 3; i >= 0; --i)
        if (N >= 64 || shapes[i][0] == 2)
            if (tile_price(M, N, shapes[i][0], shapes[i][1]) <= tile_price(M, N, shapes[best][0], shapes[best][1])) best = i;
    switch (best) {
        case 0: launch_tiles<TW, 4, 4, VEC>(X, W, Y, M, N, K, stream); break;
        case 1: launch_tiles<TW, 4, 3, VEC>(X, W, Y, M, N, K, stream); break;
        case 2: launch_tiles<TW, 4, 2, VEC>(X, W, Y, M, N, K, stream); break;
        case 3: launch_tiles<TW, 2, 3, VEC>(X, W, Y, M, N, K, stream); break;
        default: launch_tiles<TW, 2, 2, VEC>(X, W, Y, M, N, K, stream); break;
    }
    return KIPP_LAUNCH_CHECK();
}

extern "C" int kipp_gemm_f32(const float* X, const void* W, int w_dtype, float* Y, int M, int N, int K,
                             hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0) return -1;
    const bool vec = K % 4 == 0 && ((uintptr_t)X & 15) == 0 && ((uintptr_t)W & (w_dtype == KIPP_BF16 ? 7 : 15)) == 0;
    if (w_dtype == KIPP_BF16)
        return vec ? launch<bf16_t, true>(X, (const bf16_t*)W, Y, M, N, K, stream) : launch<bf16_t, false>(X, (const bf16_t*)W, Y, M, N, K, stream);
    return vec ? launch<float, true>(X, (const float*)W, Y, M, N, K, stream) : launch<float, false>(X, (const float*)W, Y, M, N, K, stream);
}
