// True 32-bit matrix product for the float32 path: Y[M,N] = X[M,K] . W[N,K]^T
// with W stored [out][in] row-major like every projection of the model
// (/root/reference/src/kipp.c:2233-2244).  Products and sums are float32 throughout, on the
// matrix cores' float32 instruction (v_mfma_f32_16x16x4_f32: 155 TFLOP/s in a large product here, twice the plain FMA's rate).
//
// An output's bits depend on its two rows and K alone, not on M, on the tile it falls in or on what else is in the
// batch.  K is cut into KPARTS runs of `part_of(K)` numbers (the last ones shorter or empty); a run is one chain of
// instructions, four numbers of k each (16 j + i, + 4, + 8, + 12 for i = 0..3, j counting up from the run's start), and the runs' sums are added
// in order.  All kernels below do exactly that, W always the instruction's first operand and X its second.
//
//   rows   up to 16 rows of X a workgroup (32 or 64 for short K): 16 rows of W, a wave a run of K, straight from memory into the instruction's
//          operands (16 bytes a lane), the runs' sums added through LDS.  Bound by the read of W (5.9 TB/s for the head's matrix).  A 16-column fragment of
//          X is multiplied whether its rows are there or not: at one row the matrix cores could feed 19 TB/s.
//   tiles  more rows: 64 or 32 rows of W times 64, 48 or 32 of X a workgroup, a wave a run of K here too, so that every wave of a
//          workgroup multiplies all of its outputs and none waits for another in the walk.  Bound by the instruction's rate (80 %
//          of it at 1,024 rows) and, below a few rounds of tiles, by what the last round leaves idle: the shape goes by that.
//   shared 64 x 64 outputs a workgroup of four waves, which meet at a barrier every 32 numbers of k: short K in many tiles, where a run a wave
//          does not pay (`form_of`).
// Measured at the 4B shape, W in turn from several copies, us: one row against 19,456 x 2,560 37 (5.4 TB/s), 2,560 x 9,728 25, the head's
// 151,936 x 2,560 264 (5.9 TB/s).  The tiles, against 19,456 x 2,560 / 6,144 x 2,560 / 2,560 x 4,096 / 2,560 x 9,728, beside what these
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
#define SHARED_TILE 64
#define SHARED_THREADS 256
#define PITCH 36            // floats from a row to the next of a shared tile's operands in LDS: 16 bytes a lane spread over the banks

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
template <typename TW, int MT, bool VEC>
__global__ void __launch_bounds__(ROWS_THREADS, MT == 1 ? 6 : 2)
gemm_f32_rows_kernel(const float* __restrict__ X, const TW* __restrict__ W, float* __restrict__ Y, int M, int N, int K) {
    __shared__ __attribute__((aligned(16))) float part_s[KPARTS][MT][KIPP_WAVE][4];
    const int wave = threadIdx.x / KIPP_WAVE, lane = threadIdx.x & (KIPP_WAVE - 1);
    const int l16 = lane & 15, h4 = 4 * (lane >> 4);
    const int blocks = (N + 15) / 16, n0 = blockIdx.x % blocks * 16, m0 = blockIdx.x / blocks * (16 * MT);
    const TW* w_row = W + (size_t)min(n0 + l16, N - 1) * K;         // rows beyond the last read it and are not stored
    const float* x_row[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) x_row[i] = X + (size_t)min(m0 + 16 * i + l16, M - 1) * K;
    const int part = part_of(K);
    const int k_lo = wave * part, k_hi = min(K, k_lo + part);
    f32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    // Pieces of 16 numbers.  A long run has AHEAD of them on their way: a piece's place is asked for again as soon as it has been multiplied.  The
    // pieces of a short one are asked for one after the other, and so is what K ends with: asked for under conditions, or with 82 registers (two workgroups a
    // compute unit; now 80 and three), they cost more than they gain.  The line lies where all of the first AHEAD are there (numbers one at a
    // time: two pieces of more than a wave's first few, where each is four requests).  One row, us, eight asked for together and the rest one by one / six
    // ahead whatever the run / now: against 151,936 / 19,456 / 6,144 x 2,560 and 2,560 x 4,096 / 9,728 324 / 46.2 / 19.9 / 14.9 / 33.3, 266 / 38.8 / 17.3 / 12.7 / 26.0,
    // 264 / 37.5 / 16.2 / 12.2 / 25.3; 19,456 x 16 / 128 / 256 / 768 / 1,024 2.9 / 4.9 / 6.9 / 16.9 / 18.5, 4.9 / 6.5 / 7.8 / 14.4 / 21.3, 2.9 / 4.9 / 6.9 / 11.8 / 16.5; 64 x 16 / 512 1.9 / 2.8,
    // 2.3 / 3.3, 2.0 / 2.9; 19,456 x 37 / 501 4.8 / 21.3, 4.6 / 12.1, 4.0 / 11.1.  32 rows against 1,024 x 256 3.5, 3.7, 3.5.
    constexpr int AHEAD = MT > 1 ? 3 : (VEC ? 6 : 5);
    const int whole = max(k_hi - k_lo, 0) / 16;
    int k = k_lo;
    if (MT == 4 || (whole >= (VEC ? AHEAD : 2) && (VEC || MT == 2 || K > 128))) {
        constexpr bool full = VEC && MT < 4;        // AHEAD pieces are there
        f32x4 w[AHEAD], x[AHEAD][MT];
        auto ask = [&](int j, int piece) {
            const int at = k_lo + 16 * piece + h4;
            w[j] = four_inside<VEC>(w_row + at);
#pragma unroll
            for (int i = 0; i < MT; ++i) x[j][i] = four_inside<VEC>(x_row[i] + at);
        };
        auto take = [&](int j) {
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i] = mul16(w[j], x[j][i], acc[i]);
        };
#pragma unroll
        for (int j = 0; j < AHEAD; ++j)
            if (full || j < whole) ask(j, j);
        int piece = 0;
        for (; piece + 2 * AHEAD <= whole; piece += AHEAD) {
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) {
                take(j);
                ask(j, piece + AHEAD + j);
            }
        }
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
            if (full || piece + j < whole) take(j);
            if (piece + AHEAD + j < whole) ask(j, piece + AHEAD + j);
        }
#pragma unroll
        for (int j = 0; j < AHEAD; ++j)
            if (piece + AHEAD + j < whole) take(j);
        k = k_lo + 16 * whole;
    }
    for (; k < k_hi; k += 16) {
        const f32x4 last = four<VEC>(w_row, k + h4, K);
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i] = mul16(last, four<VEC>(x_row[i], k + h4, K), acc[i]);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) *reinterpret_cast<f32x4*>(part_s[wave][i][lane]) = acc[i];
    __syncthreads();
    // a thread an output: the runs' sums in order
    for (int e = threadIdx.x; e < MT * 256; e += ROWS_THREADS) {
        const int i = e >> 8, at = e & 255;             // fragment; place in it: column 16 numbers of n long
        const int n = n0 + (at & 15), m = m0 + 16 * i + (at >> 4);
        const int from = 16 * ((at & 15) >> 2) + (at >> 4);
        float total = 0.0f;
#pragma unroll
        for (int p = 0; p < KPARTS; ++p) total += part_s[p][i][from][at & 3];
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

// Four waves of 32 x 32 share a step of 64 rows of either operand, the next one's on its way in registers; a run's sums are added where it ends.
template <typename TW, bool VEC>
__global__ void __launch_bounds__(SHARED_THREADS)
gemm_f32_shared_kernel(const float* __restrict__ X, const TW* __restrict__ W, float* __restrict__ Y, int M, int N, int K) {
    __shared__ __attribute__((aligned(16))) float w_s[2][SHARED_TILE * PITCH];
    __shared__ __attribute__((aligned(16))) float x_s[2][SHARED_TILE * PITCH];
    const int tid = threadIdx.x;
    const int wave = tid / KIPP_WAVE, lane = tid & (KIPP_WAVE - 1);
    const int l16 = lane & 15, h4 = 4 * (lane >> 4);
    const int n0 = blockIdx.x * SHARED_TILE, m0 = blockIdx.y * SHARED_TILE;
    const int wn = (wave & 1) * 32, wm = (wave >> 1) * 32;
    // from memory a thread takes 16 bytes of rows tid / 8 and tid / 8 + 32: eight lanes a row's 128 bytes
    const int ld_row = tid >> 3, ld_k = (tid & 7) * 4;
    const TW* w_row[2];
    const float* x_row[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        w_row[i] = W + (size_t)min(n0 + ld_row + 32 * i, N - 1) * K;
        x_row[i] = X + (size_t)min(m0 + ld_row + 32 * i, M - 1) * K;
    }
    f32x4 w_r[2], x_r[2];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            w_r[i] = four<VEC>(w_row[i], k0 + ld_k, K);
            x_r[i] = four<VEC>(x_row[i], k0 + ld_k, K);
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            *reinterpret_cast<f32x4*>(&w_s[buf][(ld_row + 32 * i) * PITCH + ld_k]) = w_r[i];
            *reinterpret_cast<f32x4*>(&x_s[buf][(ld_row + 32 * i) * PITCH + ld_k]) = x_r[i];
        }
    };
    f32x4 acc[2][2], total[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = total[a][b] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    const int part = part_of(K);
    int until = part;           // where the run under way ends
    fetch(0);
    stage(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += STEP, buf ^= 1) {
        const bool more = k0 + STEP < K;
        if (more) fetch(k0 + STEP);
#pragma unroll
        for (int j = 0; j < STEP; j += 16) {
            if (k0 + j >= K) break;
            f32x4 w[2], x[2];
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                w[a] = *reinterpret_cast<const f32x4*>(&w_s[buf][(wn + 16 * a + l16) * PITCH + j + h4]);
                x[a] = *reinterpret_cast<const f32x4*>(&x_s[buf][(wm + 16 * a + l16) * PITCH + j + h4]);
            }
            // the four sums side by side: an instruction does not wait for the one before
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[a][i], x[b][i], acc[a][b], 0, 0, 0);
        }
        if (k0 + STEP == until || !more) {
            until += part;
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    total[a][b] += acc[a][b];
                    acc[a][b] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
                }
        }
        if (more) stage(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int m = m0 + wm + 16 * b + l16, n = n0 + wn + 16 * a + h4;
            if (m >= M) continue;
            float* y = Y + (size_t)m * N + n;
            if ((N & 3) == 0 && ((uintptr_t)Y & 15) == 0) {
                if (n < N) *reinterpret_cast<f32x4*>(y) = total[a][b];
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (n + v < N) y[v] = total[a][b][v];
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

// The kernel of a product: 1, 2 or 4 (rows, so many fragments of X), 0 (shared tiles) or 10 nt + mt (tiles).
// A short K is a few steps for every wave of a tile, or none for most: its eight sums through LDS, the requests ahead of what is there and the part of a
// step that K ends with then cost more than the products.  Up to 32 rows the kernel for rows is the faster one up to the K below (17 rows and K of 256 by
// 19 %, 500 by 30 %, 32 rows and 512 by 5 %).  With more rows the prices, in us, were fitted to 3,773 products (32 to 19,456 rows of W, 65 to 4,096 of
// X, K from 16 to 4,100; shared tiles 5 % off, tiles 8 %): a round of shared tiles by its steps, and of tiles by the steps of a run, fragments, runs and what
// the last run takes longer where K ends inside a step; numbers one at a time (`vec` false) cost both more.  By them 8,422 products take 0.2 % more than
// the faster way in the mean, 25 % at most; tiles alone take up to 4.2 times as long (2,048 rows against 9,728 x 16 / 64 / 256 / 768, us, shared and
// tiles: 23 / 95, 41 / 106, 114 / 158, 302 / 327; against 2,560 x 192 30 / 40, and 2,560 x 1,100 122 / 137).
static int form_of(int M, int N, int K, bool vec) {
    if (M <= 16 || N < 32) return 1;        // tiles hold 32 rows of W or more
    const long long shared = (long long)((M + SHARED_TILE - 1) / SHARED_TILE) * ((N + SHARED_TILE - 1) / SHARED_TILE);
    const bool few = M <= 64 || (M <= 256 && shared < 192), rest = K % STEP != 0;
    if (M <= 32) {
        const int most = vec ? (rest ? 1616 : 1040) - 16 * M : 224, most_wide = vec && rest ? 320 : 64;
        if (K <= (N <= 4096 ? most : min(most, most_wide))) return 2;
    }
    if (few && K < STEP) return M <= 32 ? 2 : 4;
    static const int shapes[5][2] = {{4, 4}, {4, 3}, {4, 2}, {2, 3}, {2, 2}};
    int best = 4;
    for (int i = 3; i >= 0; --i)
        if (N >= 64 || shapes[i][0] == 2)
            if (tile_price(M, N, shapes[i][0], shapes[i][1]) <= tile_price(M, N, shapes[best][0], shapes[best][1])) best = i;
    const int nt = shapes[best][0], mt = shapes[best][1];
    // a tile's offsets into X have 32 bits, and a launch less than 2^32 threads, 2^16 tiles down a grid's second side
    const long long tiles = tile_price(M, N, nt, mt) / (nt * mt + 2) * UNITS;
    if (K > 1 << 26 || tiles >= 1LL << 23) return 0;
    if (!few && (M + SHARED_TILE - 1) / SHARED_TILE < 1 << 16) {
        const int part = part_of(K), steps = part / STEP, runs = (K + part - 1) / part;
        const int longer = rest ? max(0, (K - (runs - 1) * part) / STEP + 2 - (runs > 1 ? steps : 0)) : 0;
        const long long rounds = tile_price(M, N, nt, mt) / (nt * mt + 2), shared_rounds = (shared + UNITS - 1) / UNITS;
        const double tile = 0.18 + 0.50 * steps + (0.217 * steps + 0.038 * runs) * nt * mt + 0.29 * longer + (vec ? 0.0 : (0.56 + 0.02 * nt * mt) * steps);
        const double shared_tile = 1.21 + (vec ? 0.876 : 1.42) * ((K + STEP - 1) / STEP);
        if (2.23 + shared_tile * (1.0 + 0.664 * (shared_rounds - 1)) < 2.15 + tile * (1.0 + 0.968 * (rounds - 1))) return 0;
    }
    return 10 * nt + mt;
}

template <typename TW, int MT, bool VEC>
static void launch_rows(const float* X, const TW* W, float* Y, int M, int N, int K, hipStream_t stream) {
    const dim3 grid((N + 15) / 16 * ((M + 16 * MT - 1) / (16 * MT)));
    hipLaunchKernelGGL((gemm_f32_rows_kernel<TW, MT, VEC>), grid, dim3(ROWS_THREADS), 0, stream, X, W, Y, M, N, K);
}

template <typename TW, bool VEC>
static int launch(const float* X, const TW* W, float* Y, int M, int N, int K, hipStream_t stream) {
    switch (form_of(M, N, K, VEC)) {
        case 1: launch_rows<TW, 1, VEC>(X, W, Y, M, N, K, stream); break;
        case 2: launch_rows<TW, 2, VEC>(X, W, Y, M, N, K, stream); break;
        case 4: launch_rows<TW, 4, VEC>(X, W, Y, M, N, K, stream); break;
        case 44: launch_tiles<TW, 4, 4, VEC>(X, W, Y, M, N, K, stream); break;
        case 43: launch_tiles<TW, 4, 3, VEC>(X, W, Y, M, N, K, stream); break;
        case 42: launch_tiles<TW, 4, 2, VEC>(X, W, Y, M, N, K, stream); break;
        case 23: launch_tiles<TW, 2, 3, VEC>(X, W, Y, M, N, K, stream); break;
        case 22: launch_tiles<TW, 2, 2, VEC>(X, W, Y, M, N, K, stream); break;
        default: {
            const dim3 grid((N + SHARED_TILE - 1) / SHARED_TILE, (M + SHARED_TILE - 1) / SHARED_TILE);
            hipLaunchKernelGGL((gemm_f32_shared_kernel<TW, VEC>), grid, dim3(SHARED_THREADS), 0, stream, X, W, Y, M, N, K);
        }
    }
    return KIPP_LAUNCH_CHECK();
}

extern "C" int kipp_gemm_f32_form(int M, int N, int K) { return form_of(M, N, K, K % 4 == 0); }

extern "C" int kipp_gemm_f32(const float* X, const void* W, int w_dtype, float* Y, int M, int N, int K,
                             hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0) return -1;
    const bool vec = K % 4 == 0 && ((uintptr_t)X & 15) == 0 && ((uintptr_t)W & (w_dtype == KIPP_BF16 ? 7 : 15)) == 0;
    if (w_dtype == KIPP_BF16)
        return vec ? launch<bf16_t, true>(X, (const bf16_t*)W, Y, M, N, K, stream) : launch<bf16_t, false>(X, (const bf16_t*)W, Y, M, N, K, stream);
    return vec ? launch<float, true>(X, (const float*)W, Y, M, N, K, stream) : launch<float, false>(X, (const float*)W, Y, M, N, K, stream);
}
