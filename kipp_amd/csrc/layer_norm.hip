// Layer norm with weight and bias over rows of the float32 residual stream, and the step between two sublayers
// whose input and result are both normed:
//
//     LN(u)[c] = (u[c] - mean u) / sqrt(var u + eps) * w[c] + b[c],   var u = mean (u - mean u)^2
//
//     norm   out = scale * LN(sum of the slabs of u)                                  (any output type)
//     step   x <- x + mult * LN_post(sum of the slabs of delta) [+ extra];  out = LN_next(x)   (out optional)
//
// One workgroup a row; the row stays in registers, so it is read once, and what the step reads beside it is asked for before the
// first sum.  Bound by its reads: 2,048 rows of 2,560, 2 or 3 slabs (about 100 MB) 33 us; 39 with the
// residual stream asked for behind the sums and a slab behind the other.  A lane holds ten columns at most, wider rows have more
// lanes, and a workgroup of 1,024 keeps to 64 registers, so that two share a compute unit.  2,048 rows of 4,096, 5,120 and 8,192, one
// slab, us: norm 13.1, 15.9, 25.0, step 27.8, 36.3, 53; with 20 or 32 columns a lane of 256 (two or one waves a SIMD) 19, 22, 40 and
// 46, 54, 119; with columns read again instead of held 17, 20, 33 and 31, 36, 53.  The
// mean is taken first and the variance from the deviations, both summed over the workgroup in an order that the
// width alone fixes: a row's result does not depend on what else is in the launch.  All arithmetic is float32.
#include "common.h"
#include <math.h>

#define LN_MAX_WIDTH 8192

struct RowStats {
    float mean, inv;
};

template <int THREADS, int ITEMS>
__device__ __forceinline__ RowStats row_stats(const float (&v)[ITEMS], int width, float eps, float* scratch) {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
        if ((int)threadIdx.x + i * THREADS < width) s += v[i];
    const float mean = block_sum(s, scratch) / (float)width;
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
        if ((int)threadIdx.x + i * THREADS < width) {
            const float dlt = v[i] - mean;
            ss = fmaf(dlt, dlt, ss);
        }
    const float var = block_sum(ss, scratch) / (float)width;
    RowStats r;
    r.mean = mean;
    r.inv = 1.0f / sqrtf(var + eps);
    return r;
}

// v[i] = src at this lane's columns (columns beyond the row's read its last one and are not used)
template <int THREADS, int ITEMS>
__device__ __forceinline__ void load_row(float (&v)[ITEMS], const float* __restrict__ src, int width) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) v[i] = src[min((int)threadIdx.x + i * THREADS, width - 1)];
}

// The slabs added in order: the first 1 + AHEAD are asked for before any is used.
template <int THREADS, int AHEAD, int ITEMS>
__device__ __forceinline__ void load_slabs(float (&v)[ITEMS], const float* __restrict__ src, int parts, size_t part_stride, int width) {
    load_row<THREADS>(v, src, width);
    float more[AHEAD][ITEMS];
#pragma unroll
    for (int p = 1; p <= AHEAD; ++p)
        if (p < parts) load_row<THREADS>(more[p - 1], src + p * part_stride, width);
#pragma unroll
    for (int p = 1; p <= AHEAD; ++p)
        if (p < parts) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) v[i] += more[p - 1][i];
        }
    for (int p = 1 + AHEAD; p < parts; ++p) {
        load_row<THREADS>(more[0], src + p * part_stride, width);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) v[i] += more[0][i];
    }
}

template <typename TO, int THREADS, int ITEMS, int AHEAD>
__global__ void __launch_bounds__(THREADS, THREADS == 1024 ? 8 : 1)
layer_norm_kernel(const float* __restrict__ u, int parts, size_t part_stride, const float* __restrict__ w,
                  const float* __restrict__ b, float eps, float scale, TO* __restrict__ out, int width) {
    __shared__ float scratch[16];
    const size_t row = blockIdx.x;
    float v[ITEMS];
    load_slabs<THREADS, AHEAD>(v, u + row * width, parts, part_stride, width);
    const RowStats st = row_stats<THREADS>(v, width, eps, scratch);
    TO* dst = out + row * width;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int c = (int)threadIdx.x + i * THREADS;
        if (c < width) store_f(dst, c, ((v[i] - st.mean) * st.inv * w[c] + b[c]) * scale);
    }
}

template <typename TO, int THREADS, int ITEMS, int AHEAD>
__global__ void __launch_bounds__(THREADS, THREADS == 1024 ? 8 : 1)
sandwich_step_kernel(float* __restrict__ x, const float* __restrict__ delta, int parts, size_t part_stride,
                     const float* __restrict__ post_w, const float* __restrict__ post_b, float post_eps, float mult,
                     const float* __restrict__ extra, const float* __restrict__ next_w, const float* __restrict__ next_b,
                     float next_eps, TO* __restrict__ out, int width) {
    __shared__ float scratch[16];
    const size_t row = blockIdx.x;
    float* xr = x + row * width;
    float v[ITEMS], old[ITEMS];
    load_row<THREADS>(old, xr, width);
    load_slabs<THREADS, AHEAD>(v, delta + row * width, parts, part_stride, width);
    const RowStats st = row_stats<THREADS>(v, width, post_eps, scratch);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int c = (int)threadIdx.x + i * THREADS;
        if (c < width) {
            float nx = old[i] + mult * ((v[i] - st.mean) * st.inv * post_w[c] + post_b[c]);
            if (extra != nullptr) nx += extra[row * width + c];
            xr[c] = nx;
            v[i] = nx;
        }
    }
    if (out == nullptr) return;
    const RowStats nt = row_stats<THREADS>(v, width, next_eps, scratch);
    TO* dst = out + row * width;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int c = (int)threadIdx.x + i * THREADS;
        if (c < width) store_f(dst, c, (v[i] - nt.mean) * nt.inv * next_w[c] + next_b[c]);
    }
}

// LAUNCH(lanes, columns a lane, slabs asked for behind the first).  FIVE: which build rows of up to 5,120 take.
#define KIPP_LN_BUILDS(LAUNCH, FIVE)                       \
    do {                                                   \
        if (width <= 256 * 10) LAUNCH(256, 10, 3);         \
        else if (width <= 512 * 6) LAUNCH(512, 6, 2);      \
        else if (width <= 512 * 8) LAUNCH(512, 8, 2);      \
        else if (width <= 5120) FIVE;                      \
        else if (width <= 1024 * 6) LAUNCH(1024, 6, 2);    \
        else LAUNCH(1024, 8, 1);                           \
    } while (0)

extern "C" int kipp_layer_norm(const float* u, int parts, const float* w, const float* b, float eps, float scale, void* out,
                               int out_dtype, int rows, int width, hipStream_t stream) {
    if (rows <= 0) return 0;
    if (width <= 0 || width > LN_MAX_WIDTH || parts <= 0) return -1;
    const size_t part_stride = (size_t)rows * width;
#define KIPP_LN(THREADS, ITEMS, AHEAD)                                                                                                             \
    hipLaunchKernelGGL((layer_norm_kernel<KIPP_LN_TO, THREADS, ITEMS, AHEAD>), dim3(rows), dim3(THREADS), 0, stream, u, parts, part_stride, w, b, eps, \
                       scale, (KIPP_LN_TO*)out, width)
    if (out_dtype == KIPP_F32) {
#define KIPP_LN_TO float
        KIPP_LN_BUILDS(KIPP_LN, KIPP_LN(512, 10, 2));
#undef KIPP_LN_TO
    } else if (out_dtype == KIPP_BF16) {
#define KIPP_LN_TO bf16_t
        KIPP_LN_BUILDS(KIPP_LN, KIPP_LN(512, 10, 2));
#undef KIPP_LN_TO
    } else {
        return -2;
    }
#undef KIPP_LN
    return KIPP_LAUNCH_CHECK();
}

extern "C" int kipp_sandwich_step(float* x, const float* delta, int parts, const float* post_w, const float* post_b, float post_eps,
                                  float mult, const float* extra, const float* next_w, const float* next_b, float next_eps,
                                  void* out, int out_dtype, int rows, int width, hipStream_t stream) {
    if (rows <= 0) return 0;
    if (width <= 0 || width > LN_MAX_WIDTH || parts <= 0) return -1;
    if (out != nullptr && (next_w == nullptr || next_b == nullptr)) return -1;
    const size_t part_stride = (size_t)rows * width;
#define KIPP_SS(THREADS, ITEMS, AHEAD)                                                                                                             \
    hipLaunchKernelGGL((sandwich_step_kernel<KIPP_SS_TO, THREADS, ITEMS, AHEAD>), dim3(rows), dim3(THREADS), 0, stream, x, delta, parts, part_stride, \
                       post_w, post_b, post_eps, mult, extra, next_w, next_b, next_eps, (KIPP_SS_TO*)out, width)
    if (out == nullptr || out_dtype == KIPP_F32) {
#define KIPP_SS_TO float
        KIPP_LN_BUILDS(KIPP_SS, KIPP_SS(1024, 5, 2));
#undef KIPP_SS_TO
    } else if (out_dtype == KIPP_BF16) {
#define KIPP_SS_TO bf16_t
        KIPP_LN_BUILDS(KIPP_SS, KIPP_SS(1024, 5, 2));
#undef KIPP_SS_TO
    } else {
        return -2;
    }
#undef KIPP_SS
    return KIPP_LAUNCH_CHECK();
}
