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
//   rows   up to 64 rows of X a workgroup: 16 rows of W, a wave a run of K, straight from memory into the instruction's
//          operands (16 bytes a lane), the runs' sums added through LDS.  Bound by the read of W.  A 16-column fragment of
//          X is multiplied whether its rows are there or not: at one row the matrix cores could feed 19 TB/s.
//   tiles  64 x 64 outputs a workgroup, a wave 32 x 32, X and W staged through LDS 32 numbers of k at a time, the next
//          step's on their way in registers.  Bound by the instruction's rate and, below a few hundred tiles, by idle
//          compute units.
// Measured at the 4B shape, before (one plain FMA chain an output, 64 x 64 tiles at every M) and now: one row against 19,456 x 2,560
// 402 and 46 us (4.3 TB/s), 2,560 x 9,728 1,160 and 34 us, the head's 151,936 x 2,560 913 and 325 us (4.8 TB/s);
// 333 rows against 19,456 x 2,560 614 and 422 us (79 TFLOP/s), 2,560 x 9,728 1,220 and 274 us (240 tiles for 256 compute units).
#include "common.h"

#define KPARTS 8
#define STEP 32             // numbers of k a tile step brings into LDS; a run is a multiple of it
#define TILE 64
#define PITCH 36            // floats from a row to the next in LDS: 16 bytes a lane spread over the banks
#define THREADS 256
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

// 16 numbers of k: lane l holds those at 4 (l / 16) .. + 3 of row l % 16 of either operand.
__device__ __forceinline__ f32x4 mul16(f32x4 w, f32x4 x, f32x4 acc) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[i], acc, 0, 0, 0);
    return acc;
}

// The sums of a fragment lie in lane l as rows 4 (l / 16) .. + 3 (of W) of column l % 16 (a row of X).
template <typename TW, int MT, bool VEC>
__global__ void __launch_bounds__(ROWS_THREADS)
gemm_f32_rows_kernel(const float* __restrict__ X, const TW* __restrict__ W, float* __restrict__ Y, int M, int N, int K) {
    __shared__ __attribute__((aligned(16))) float part_s[KPARTS][MT][KIPP_WAVE][4];
    const int wave = threadIdx.x / KIPP_WAVE, lane = threadIdx.x & (KIPP_WAVE - 1);
    const int l16 = lane & 15, h4 = 4 * (lane >> 4);
    const int n0 = blockIdx.x * 16, m0 = blockIdx.y * (16 * MT);
    const TW* w_row = W + (size_t)min(n0 + l16, N - 1) * K;         // rows beyond the last read it and are not stored
    const float* x_row[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) x_row[i] = X + (size_t)min(m0 + 16 * i + l16, M - 1) * K;
    const int part = part_of(K);
    const int k_lo = wave * part, k_hi = min(K, k_lo + part);
    f32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int AHEAD = MT == 1 ? 8 : (MT == 2 ? 6 : 4);       // 16-number pieces asked for together
    int k = k_lo;
    for (; k + 16 * AHEAD <= k_hi; k += 16 * AHEAD) {
        f32x4 w[AHEAD], x[AHEAD][MT];
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
            w[j] = four<VEC>(w_row, k + 16 * j + h4, K);
#pragma unroll
            for (int i = 0; i < MT; ++i) x[j][i] = four<VEC>(x_row[i], k + 16 * j + h4, K);
        }
#pragma unroll
        for (int j = 0; j < AHEAD; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i] = mul16(w[j], x[j][i], acc[i]);
    }
    for (; k < k_hi; k += 16) {
        const f32x4 w = four<VEC>(w_row, k + h4, K);
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i] = mul16(w, four<VEC>(x_row[i], k + h4, K), acc[i]);
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

template <typename TW, bool VEC>
__global__ void __launch_bounds__(THREADS)
gemm_f32_tiles_kernel(const float* __restrict__ X, const TW* __restrict__ W, float* __restrict__ Y, int M, int N, int K) {
    __shared__ __attribute__((aligned(16))) float w_s[2][TILE * PITCH];
    __shared__ __attribute__((aligned(16))) float x_s[2][TILE * PITCH];
    const int tid = threadIdx.x;
    const int wave = tid / KIPP_WAVE, lane = tid & (KIPP_WAVE - 1);
    const int l16 = lane & 15, h4 = 4 * (lane >> 4);
    const int n0 = blockIdx.x * TILE, m0 = blockIdx.y * TILE;
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

template <typename TW, bool VEC>
static int launch(const float* X, const TW* W, float* Y, int M, int N, int K, hipStream_t stream) {
    const int m_tiles = (M + TILE - 1) / TILE, n_tiles = (N + TILE - 1) / TILE;
    // Tiles need a workgroup for most of the 256 compute units; the other kernel has N / 16 workgroups for 64 rows, but
    // reads each of its operands from the caches for 16 rows of W only.
    if (M <= 64 || (M <= 256 && m_tiles * n_tiles < 192)) {
        const dim3 block(ROWS_THREADS);
        const int nb = (N + 15) / 16;
#define KIPP_ROWS(MT) hipLaunchKernelGGL((gemm_f32_rows_kernel<TW, MT, VEC>), dim3(nb, (M + 16 * MT - 1) / (16 * MT)), block, 0, stream, X, W, Y, M, N, K)
        if (M <= 16) KIPP_ROWS(1);
        else if (M <= 32) KIPP_ROWS(2);
        else KIPP_ROWS(4);
#undef KIPP_ROWS
    } else {
        hipLaunchKernelGGL((gemm_f32_tiles_kernel<TW, VEC>), dim3(n_tiles, m_tiles), dim3(THREADS), 0, stream, X, W, Y, M, N, K);
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
