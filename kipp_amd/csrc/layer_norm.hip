// Layer norm with weight and bias over rows of the float32 residual stream, and the step between two sublayers
// whose input and result are both normed:
//
//     LN(u)[c] = (u[c] - mean u) / sqrt(var u + eps) * w[c] + b[c],   var u = mean (u - mean u)^2
//
//     norm   out = scale * LN(sum of the slabs of u)                                  (any output type)
//     step   x <- x + mult * LN_post(sum of the slabs of delta) [+ extra];  out = LN_next(x)   (out optional)
//
// One workgroup a row; the row stays in registers, so it is read once, and what the step reads beside it (the weights too) is asked for before the
// first sum.  Bound by its reads and, at these sizes, by their number: a lane takes eight columns as two loads of 16 bytes.  2,048 rows of 2,560 / 4,096 / 5,120 /
// 8,192, three slabs, us, in turn from three copies: step 25, 36, 52, 74, norm 13, 23, 31, 45; one slab 21, 24, 35, 55 and 9, 11, 16.5, 24.  With a
// column a load, which is five times the requests: step 28, 43, 58, 84, norm 16, 26, 31.5, 49; 22, 28, 40, 59 and 11, 13, 15.5, 30.
// Rows whose width is no multiple of 4, or that begin at no multiple of 16 bytes, are taken a column a load: up to ten columns a lane, wider rows more lanes
// (2,048 rows of 2,561 / 4,097 / 5,118, one slab, us: step 20, 35, 42, norm 11.5, 15, 17; with 1,024 lanes for all of them 30, 35, 42 and 17, 19, 20).  The
// mean is taken first and the variance from the deviations, both summed over the workgroup in an order that the
// width and that alignment fix: a row's result does not depend on what else is in the launch.  All arithmetic is float32.
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

typedef __attribute__((ext_vector_type(4))) float f32x4;

// A lane's columns of a row: four at 4 t and four at 4 (t + lanes); behind the row's end its last four, which are not used.
struct Wide {
    int at[2];
    bool live[2];
    __device__ __forceinline__ explicit Wide(int width) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int c = 4 * ((int)threadIdx.x + i * (int)blockDim.x);
            live[i] = c < width;
            at[i] = live[i] ? c : width - 4;
        }
    }
    __device__ __forceinline__ void load(f32x4 (&v)[2], const float* __restrict__ src) const {
#pragma unroll
        for (int i = 0; i < 2; ++i) v[i] = *reinterpret_cast<const f32x4*>(src + at[i]);
    }
    __device__ __forceinline__ void store(float* dst, const f32x4 (&v)[2]) const {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (live[i]) *reinterpret_cast<f32x4*>(dst + at[i]) = v[i];
    }
    __device__ __forceinline__ void store(bf16_t* dst, const f32x4 (&v)[2]) const {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (live[i])
                *reinterpret_cast<uint2*>(dst + at[i]) = make_uint2((uint32_t)f32_to_bf16(v[i][0]) | ((uint32_t)f32_to_bf16(v[i][1]) << 16),
                                                                    (uint32_t)f32_to_bf16(v[i][2]) | ((uint32_t)f32_to_bf16(v[i][3]) << 16));
    }
    __device__ __forceinline__ RowStats stats(const f32x4 (&v)[2], int width, float eps, float* scratch) const {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (live[i]) s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
        RowStats r;
        r.mean = block_sum(s, scratch) / (float)width;
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (live[i])
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float dlt = v[i][j] - r.mean;
                    ss = fmaf(dlt, dlt, ss);
                }
        r.inv = 1.0f / sqrtf(block_sum(ss, scratch) / (float)width + eps);
        return r;
    }
};

// SLABS slabs are asked for together.
template <int SLABS>
__device__ __forceinline__ void load_wide_slabs(const Wide& lane, f32x4 (&v)[2], const float* __restrict__ src, int parts, size_t part_stride) {
    f32x4 more[SLABS - 1][2];
    lane.load(v, src);
#pragma unroll
    for (int p = 1; p < SLABS; ++p)
        if (p < parts) lane.load(more[p - 1], src + p * part_stride);
#pragma unroll
    for (int p = 1; p < SLABS; ++p)
        if (p < parts) {
#pragma unroll
            for (int i = 0; i < 2; ++i) v[i] += more[p - 1][i];
        }
    for (int p = SLABS; p < parts; ++p) {
        lane.load(more[0], src + p * part_stride);
#pragma unroll
        for (int i = 0; i < 2; ++i) v[i] += more[0][i];
    }
}

template <typename TO>
__global__ void __launch_bounds__(1024)
layer_norm_wide_kernel(const float* __restrict__ u, int parts, size_t part_stride, const float* __restrict__ w, const float* __restrict__ b,
                       float eps, float scale, TO* __restrict__ out, int width) {
    __shared__ float scratch[16];
    const size_t row = blockIdx.x;
    const Wide lane(width);
    f32x4 v[2], wv[2], bv[2];
    lane.load(wv, w);
    lane.load(bv, b);
    load_wide_slabs<4>(lane, v, u + row * width, parts, part_stride);
    const RowStats st = lane.stats(v, width, eps, scratch);
#pragma unroll
    for (int i = 0; i < 2; ++i) v[i] = ((v[i] - st.mean) * st.inv * wv[i] + bv[i]) * scale;
    lane.store(out + row * width, v);
}

// CROWDED: rows of more than 4,096 columns, 576 lanes and more, and of 2,564 to 3,584, six and seven waves, of which 94 registers leave room for two or
// three workgroups: 64 registers, so that two and three, and four and five, share a compute unit, for which the weights and the fourth slab are asked
// for when they are wanted (2,048 rows of 3,072, one and three slabs, us: 20.8, 28.5; with 94 registers 25.0, 32.0; a column a load 22.1, 30.5).
template <typename TO, bool CROWDED>
__global__ void __launch_bounds__(1024, CROWDED ? 8 : 4)
sandwich_step_wide_kernel(float* __restrict__ x, const float* __restrict__ delta, int parts, size_t part_stride,
                          const float* __restrict__ post_w, const float* __restrict__ post_b, float post_eps, float mult,
                          const float* __restrict__ extra, const float* __restrict__ next_w, const float* __restrict__ next_b,
                          float next_eps, TO* __restrict__ out, int width) {
    __shared__ float scratch[16];
    const size_t row = blockIdx.x;
    const Wide lane(width);
    f32x4 v[2], old[2], ev[2], pw[2], pb[2], nw[2], nb[2];
    lane.load(old, x + row * width);
    if (extra != nullptr) lane.load(ev, extra + row * width);
    auto post = [&]() {
        lane.load(pw, post_w);
        lane.load(pb, post_b);
    };
    auto next = [&]() {
        lane.load(nw, next_w);
        lane.load(nb, next_b);
    };
    if (!CROWDED) {
        post();
        if (out != nullptr) next();
    }
    load_wide_slabs<CROWDED ? 3 : 4>(lane, v, delta + row * width, parts, part_stride);
    const RowStats st = lane.stats(v, width, post_eps, scratch);
    if (CROWDED) post();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        v[i] = old[i] + mult * ((v[i] - st.mean) * st.inv * pw[i] + pb[i]);
        if (extra != nullptr) v[i] += ev[i];
    }
    lane.store(x + row * width, v);
    if (out == nullptr) return;
    const RowStats nt = lane.stats(v, width, next_eps, scratch);
    if (CROWDED) next();
#pragma unroll
    for (int i = 0; i < 2; ++i) v[i] = (v[i] - nt.mean) * nt.inv * nw[i] + nb[i];
    lane.store(out + row * width, v);
}

static bool wide_rows(int width, const void* a, const void* b, const void* c, const void* d, const void* e, const void* f, const void* g) {
    return width % 4 == 0 && (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c | (uintptr_t)d | (uintptr_t)e | (uintptr_t)f | (uintptr_t)g) & 15) == 0;
}

static dim3 wide_lanes(int width) { return dim3((width / 8 + KIPP_WAVE - 1 + (width % 8 != 0)) / KIPP_WAVE * KIPP_WAVE); }

// LAUNCH(lanes, columns a lane, slabs asked for behind the first): rows a column a load.  FIVE: which build rows of up to 5,120 take.
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
    if (wide_rows(width, u, w, b, out, nullptr, nullptr, nullptr)) {
        if (out_dtype == KIPP_F32)
            hipLaunchKernelGGL(layer_norm_wide_kernel<float>, dim3(rows), wide_lanes(width), 0, stream, u, parts, part_stride, w, b, eps, scale, (float*)out, width);
        else if (out_dtype == KIPP_BF16)
            hipLaunchKernelGGL(layer_norm_wide_kernel<bf16_t>, dim3(rows), wide_lanes(width), 0, stream, u, parts, part_stride, w, b, eps, scale, (bf16_t*)out, width);
        else
            return -2;
        return KIPP_LAUNCH_CHECK();
    }
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
    if (wide_rows(width, x, delta, post_w, post_b, extra, out, nullptr) && wide_rows(width, next_w, next_b, nullptr, nullptr, nullptr, nullptr, nullptr)) {
#define KIPP_SW(TO, CROWDED)                                                                                                                              \
    hipLaunchKernelGGL((sandwich_step_wide_kernel<TO, CROWDED>), dim3(rows), wide_lanes(width), 0, stream, x, delta, parts, part_stride, post_w, post_b, \
                       post_eps, mult, extra, next_w, next_b, next_eps, (TO*)out, width)
        if (out != nullptr && out_dtype != KIPP_F32 && out_dtype != KIPP_BF16) return -2;
        const bool crowded = width > 4096 || (width > 2560 && width <= 3584), narrow = out != nullptr && out_dtype == KIPP_BF16;
        if (crowded && narrow) KIPP_SW(bf16_t, true);
        else if (crowded) KIPP_SW(float, true);
        else if (narrow) KIPP_SW(bf16_t, false);
        else KIPP_SW(float, false);
#undef KIPP_SW
        return KIPP_LAUNCH_CHECK();
    }
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
