// Row-wise steps around the products over many rows: the embedding, the residual sum with the norm of a sublayer's output
// (for experts: with their weighted sum), the norm in front of the head.  The residual is fp32 throughout; one workgroup
// per row.
#include "dense.h"
#include "dense_kernels.h"
#include <type_traits>

namespace w4a16 {

namespace {

constexpr int kRowThreads = 256;

__device__ __forceinline__ float row_total(float v, float *red) {
    v = wave_reduce<false>(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}

template <class T>
__global__ void __launch_bounds__(kRowThreads) embed_rows_kernel(const int32_t *tokens, const T *embed, float scale, float *res, T *h, int width) {
    const size_t m = blockIdx.x;
    const T *row = embed + (size_t)tokens[m] * width;
    for (int i = 4 * threadIdx.x; i < width; i += 4 * kRowThreads) {
        float e[4];
        load4(row + i, e);
#pragma unroll
        for (int j = 0; j < 4; ++j) e[j] *= scale;
        store4(res + m * width + i, e[0], e[1], e[2], e[3]);
        store4(h + m * width + i, e[0], e[1], e[2], e[3]);
    }
}

// What bounds the two kernels below: round trips where there are few rows (every operand comes from the last-level cache, written by other XCDs), the copy rate where there are many.  So
// a thread asks for all that its elements are made of at once, up to AT parts or experts' outputs of them, and keeps in registers what a second pass reads (QUADS of four elements; 0: any
// width, by way of LDS).  In a graph, before / now, 64 rows of 2048: one part 2.6 / 2.35 us, eight 4.0 / 2.95, eight experts 4.2 / 3.1; 300 rows of 2880, eight parts 9.3 / 5.9;
// 1024 rows of 2048, eight experts 10.2 / 8.9; 2048 rows of 2048, eight experts 16.1 / 16.2.

// y[m] of a row's four elements: the sum of `parts` matrices [M][width] (a product's slices along K), in their order
// (in turn: a loop with no bounds to look at; 520 rows of 6144, two parts 11.3 -> 10.2 us)
template <int AT>
__device__ __forceinline__ void load_parts(const float *y, int parts, size_t size, float (&v)[4]) {
    if constexpr (AT == 1) {
        load4(y, v);
        for (int s = 1; s < parts; ++s) {
            float u[4];
            load4(y + s * size, u);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] += u[j];
        }
        return;
    }
    for (int s0 = 0; s0 < parts; s0 += AT) {
        float u[AT][4];
#pragma unroll
        for (int s = 0; s < AT; ++s) load4(y + (s0 + s < parts ? s0 + s : parts - 1) * size, u[s]);
#pragma unroll
        for (int s = 0; s < AT; ++s)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = s0 + s == 0 ? u[s][j] : s0 + s < parts ? v[j] + u[s][j] : v[j];
    }
}

// the weighted sum of a row's `top` outputs
template <int AT, class Y>
__device__ __forceinline__ void load_weighted(const Y *y, const float *weights, int top, int width, float (&v)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = 0.f;
    if constexpr (AT == 1) {
        for (int s = 0; s < top; ++s) {
            float u[4];
            load4(y + (size_t)s * width, u);
            const float wt = weights[s];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = fmaf(wt, u[j], v[j]);
        }
        return;
    }
    for (int s0 = 0; s0 < top; s0 += AT) {
        float u[AT][4], wt[AT];
#pragma unroll
        for (int s = 0; s < AT; ++s) {
            const int at = s0 + s < top ? s0 + s : top - 1;
            load4(y + (size_t)at * width, u[s]);
            wt[s] = weights[at];
        }
#pragma unroll
        for (int s = 0; s < AT; ++s)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = s0 + s < top ? fmaf(wt[s], u[s][j], v[j]) : v[j];
    }
}

__device__ __forceinline__ void squares(const float (&v)[4], float &ss) {
#pragma unroll
    for (int j = 0; j < 4; ++j) ss = fmaf(v[j], v[j], ss);
}

// Y: type of y; top > 0: y holds `top` rows per token, summed with the router's weights
template <class T, class Y, int QUADS, int AT>
__global__ void __launch_bounds__(kRowThreads) residual_norm_kernel(float *res, const Y *y, int parts, const float *weights, int top, const float *norm_w,
                                                                    float eps, int true_width, T *h, int width) {
    extern __shared__ float sum_lds[];
    __shared__ float red[4];
    const size_t m = blockIdx.x;
    float ss = 0.f;
    auto sum = [&](int i, float (&v)[4]) {
        if (top > 0) load_weighted<AT>(y + m * top * width + i, weights + m * top, top, width, v);
        else if constexpr (sizeof(Y) == 4) load_parts<AT>(y + m * width + i, parts, (size_t)gridDim.x * width, v);
    };
    auto finish = [&](int i, float rstd, const float (&v)[4], const float (&w)[4], float (&x)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = fmaf(v[j] * rstd, w[j], x[j]);
        store4(res + m * width + i, x[0], x[1], x[2], x[3]);
        if (h) store4(h + m * width + i, x[0], x[1], x[2], x[3]);
    };
    if constexpr (QUADS > 0) {
        float v[QUADS][4], w[QUADS][4], x[QUADS][4];
#pragma unroll
        for (int q = 0; q < QUADS; ++q) {
            const int i = 4 * (threadIdx.x + q * kRowThreads), at = i < width ? i : width - 4;   // (past the end the last ones, left out of the sum)
            sum(at, v[q]);
            load4(norm_w + at, w[q]);
            load4(res + m * width + at, x[q]);
        }
#pragma unroll
        for (int q = 0; q < QUADS; ++q)
            if (4 * (int)(threadIdx.x + q * kRowThreads) < width) squares(v[q], ss);
        const float rstd = 1.0f / sqrtf(row_total(ss, red) / (float)true_width + eps);
#pragma unroll
        for (int q = 0; q < QUADS; ++q)
            if (const int i = 4 * (threadIdx.x + q * kRowThreads); i < width) finish(i, rstd, v[q], w[q], x[q]);
        return;
    }
    for (int i = 4 * threadIdx.x; i < width; i += 4 * kRowThreads) {
        float v[4];
        sum(i, v);
        store4(sum_lds + i, v[0], v[1], v[2], v[3]);   // read back by the same thread
        squares(v, ss);
    }
    const float rstd = 1.0f / sqrtf(row_total(ss, red) / (float)true_width + eps);
    for (int i = 4 * threadIdx.x; i < width; i += 4 * kRowThreads) {
        float v[4], w[4], x[4];
        load4(sum_lds + i, v);
        load4(norm_w + i, w);
        load4(res + m * width + i, x);
        finish(i, rstd, v, w, x);
    }
}

template <class T>
__global__ void __launch_bounds__(kRowThreads) norm_rows_kernel(const float *res, const int32_t *rows, const float *norm_w, float eps, int true_width, T *out,
                                                                int width) {
    __shared__ float red[4];
    const float *x = res + (size_t)(rows ? rows[blockIdx.x] : (int)blockIdx.x) * width;
    float ss = 0.f;
    for (int i = 4 * threadIdx.x; i < width; i += 4 * kRowThreads) {
        float v[4];
        load4(x + i, v);
#pragma unroll
        for (int j = 0; j < 4; ++j) ss = fmaf(v[j], v[j], ss);
    }
    const float rstd = 1.0f / sqrtf(row_total(ss, red) / (float)true_width + eps);
    for (int i = 4 * threadIdx.x; i < width; i += 4 * kRowThreads) {
        float v[4], w[4];
        load4(x + i, v);
        load4(norm_w + i, w);
        store4(out + (size_t)blockIdx.x * width + i, v[0] * rstd * w[0], v[1] * rstd * w[1], v[2] * rstd * w[2], v[3] * rstd * w[3]);
    }
}

// the residual brought up to date and its norm: what the sublayers of a model with norms on their inputs read
template <class T, int QUADS, int AT>
__global__ void __launch_bounds__(kRowThreads) add_norm_rows_kernel(float *res, const float *y, int parts, const int32_t *tokens, const T *embed,
                                                                    float scale, const float *norm_w, float eps, int true_width, T *h, int width) {
    extern __shared__ float sum_lds[];
    __shared__ float red[4];
    const size_t m = blockIdx.x;
    const T *row = tokens ? embed + (size_t)tokens[m] * width : nullptr;
    float ss = 0.f;
    auto value = [&](int i, float (&v)[4]) {
        if (row) {
            load4(row + i, v);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] *= scale;
        } else {
            load4(res + m * width + i, v);
            if (y) {
                float u[4];
                load_parts<AT>(y + m * width + i, parts, (size_t)gridDim.x * width, u);
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] += u[j];
            }
        }
    };
    auto finish = [&](int i, float rstd, const float (&v)[4], const float (&w)[4]) {
        store4(h + m * width + i, v[0] * rstd * w[0], v[1] * rstd * w[1], v[2] * rstd * w[2], v[3] * rstd * w[3]);
    };
    if constexpr (QUADS > 0) {
        float v[QUADS][4], w[QUADS][4];
#pragma unroll
        for (int q = 0; q < QUADS; ++q) {
            const int i = 4 * (threadIdx.x + q * kRowThreads), at = i < width ? i : width - 4;
            value(at, v[q]);
            if (h) load4(norm_w + at, w[q]);
        }
        // (past the end the last elements again, which another thread writes: nothing of them is kept)
#pragma unroll
        for (int q = 0; q < QUADS; ++q)
            if (const int i = 4 * (threadIdx.x + q * kRowThreads); i < width) {
                if (row || y) store4(res + m * width + i, v[q][0], v[q][1], v[q][2], v[q][3]);
                squares(v[q], ss);
            }
        if (!h) return;
        const float rstd = 1.0f / sqrtf(row_total(ss, red) / (float)true_width + eps);
#pragma unroll
        for (int q = 0; q < QUADS; ++q)
            if (const int i = 4 * (threadIdx.x + q * kRowThreads); i < width) finish(i, rstd, v[q], w[q]);
        return;
    }
    for (int i = 4 * threadIdx.x; i < width; i += 4 * kRowThreads) {
        float v[4];
        value(i, v);
        if (row || y) store4(res + m * width + i, v[0], v[1], v[2], v[3]);
        store4(sum_lds + i, v[0], v[1], v[2], v[3]);   // read back by the same thread
        squares(v, ss);
    }
    if (!h) return;
    const float rstd = 1.0f / sqrtf(row_total(ss, red) / (float)true_width + eps);
    for (int i = 4 * threadIdx.x; i < width; i += 4 * kRowThreads) {
        float v[4], w[4];
        load4(sum_lds + i, v);
        load4(norm_w + i, w);
        finish(i, rstd, v, w);
    }
}

// f(quads a thread, parts at a time) with the kernel's constants for M rows of `parts`.  Over `few` rows the other workgroups of a CU cover the round trips, and fewer registers keep
// more of them there: loads in turn again, and by way of LDS where a row has more quads than `quads_few` of few rows, `quads_many` of many.  (2048 rows of 2048, eight parts at a time
// 27.2 us, in turn 25.9; 1024 rows, two parts 5.4 / 4.9; eight experts 8.9 / 10.2, at 2048 rows 16.6 / 16.2.)  By way of LDS also where half a workgroup or more has no quad and would
// ask for many operands of one all the same (registers / LDS, 2048 rows, eight experts of 512 5.6 / 4.7, of 256 5.1 / 4.2, four 4.1 / 3.7; but one or two of 512 3.0 / 3.2, eight of 768 4.0 / 4.3,
// 520 rows of eight of 512 3.3 / 3.5).
template <class F>
void row_form(int M, int few, int width, int quads_few, int quads_many, int parts, F f) {
    auto with_parts = [&](auto quads) {
        if (parts <= 1 || M > few) f(quads, std::integral_constant<int, 1>());
        else if (parts <= 2) f(quads, std::integral_constant<int, 2>());
        else if (parts <= 4) f(quads, std::integral_constant<int, 4>());
        else f(quads, std::integral_constant<int, 8>());
    };
    const int quads = (width + 4 * kRowThreads - 1) / (4 * kRowThreads), most = M > few ? quads_many : quads_few;
    const bool narrow = M > 1024 && width <= 512 && width <= 128 * parts;
    if (quads > most || narrow) with_parts(std::integral_constant<int, 0>());
    else if (quads == 1) with_parts(std::integral_constant<int, 1>());
    else if (quads == 2) with_parts(std::integral_constant<int, 2>());
    else with_parts(std::integral_constant<int, 4>());
}

}  // namespace

hipError_t launch_add_norm_rows(int dtype, float *res, const float *y, int parts, const int32_t *tokens, const void *embed, float scale, const float *norm_w,
                                float eps, int true_width, void *h, int M, int width, hipStream_t stream) {
    row_form(M, 512, width, 2, 0, y ? parts : 1, [&](auto quads, auto at) {
        constexpr int QUADS = decltype(quads)::value, AT = decltype(at)::value;
        const size_t lds = QUADS ? 0 : (size_t)width * sizeof(float);   // (the C ABI keeps width within 64 KiB)
        if (dtype == kF32)
            hipLaunchKernelGGL((add_norm_rows_kernel<float, QUADS, AT>), dim3(M), dim3(kRowThreads), lds, stream, res, y, parts, tokens, static_cast<const float *>(embed), scale,
                               norm_w, eps, true_width, static_cast<float *>(h), width);
        else
            hipLaunchKernelGGL((add_norm_rows_kernel<bf16, QUADS, AT>), dim3(M), dim3(kRowThreads), lds, stream, res, y, parts, tokens, static_cast<const bf16 *>(embed), scale,
                               norm_w, eps, true_width, static_cast<bf16 *>(h), width);
    });
    return hipGetLastError();
}

hipError_t launch_embed_rows(int dtype, const int32_t *tokens, const void *embed, float scale, float *res, void *h, int M, int width,
                             hipStream_t stream) {
    if (dtype == kF32)
        hipLaunchKernelGGL(embed_rows_kernel<float>, dim3(M), dim3(kRowThreads), 0, stream, tokens, static_cast<const float *>(embed), scale, res,
                           static_cast<float *>(h), width);
    else
        hipLaunchKernelGGL(embed_rows_kernel<bf16>, dim3(M), dim3(kRowThreads), 0, stream, tokens, static_cast<const bf16 *>(embed), scale, res,
                           static_cast<bf16 *>(h), width);
    return hipGetLastError();
}

hipError_t launch_residual_norm_rows(int dtype, float *res, const void *y, int parts, const float *weights, int top, const float *norm_w, float eps,
                                     int true_width, void *h, int M, int width, hipStream_t stream) {
    if (!weights) top = 0;
    row_form(M, top > 0 ? 1024 : 512, width, top > 0 ? 2 : 4, 2, top > 0 ? top : parts, [&](auto quads, auto at) {
        constexpr int QUADS = decltype(quads)::value, AT = decltype(at)::value;
        const size_t lds = QUADS ? 0 : (size_t)width * sizeof(float);   // (the C ABI keeps width within 64 KiB)
        if (dtype == kF32)
            hipLaunchKernelGGL((residual_norm_kernel<float, float, QUADS, AT>), dim3(M), dim3(kRowThreads), lds, stream, res, static_cast<const float *>(y), parts, weights, top,
                               norm_w, eps, true_width, static_cast<float *>(h), width);
        else if (top > 0)
            hipLaunchKernelGGL((residual_norm_kernel<bf16, bf16, QUADS, AT>), dim3(M), dim3(kRowThreads), lds, stream, res, static_cast<const bf16 *>(y), parts, weights, top,
                               norm_w, eps, true_width, static_cast<bf16 *>(h), width);
        else
            hipLaunchKernelGGL((residual_norm_kernel<bf16, float, QUADS, AT>), dim3(M), dim3(kRowThreads), lds, stream, res, static_cast<const float *>(y), parts, weights, top,
                               norm_w, eps, true_width, static_cast<bf16 *>(h), width);
    });
    return hipGetLastError();
}

hipError_t launch_norm_rows(int dtype, const float *res, const int32_t *rows, const float *norm_w, float eps, int true_width, void *out, int n,
                            int width, hipStream_t stream) {
    if (dtype == kF32)
        hipLaunchKernelGGL(norm_rows_kernel<float>, dim3(n), dim3(kRowThreads), 0, stream, res, rows, norm_w, eps, true_width, static_cast<float *>(out),
                           width);
    else
        hipLaunchKernelGGL(norm_rows_kernel<bf16>, dim3(n), dim3(kRowThreads), 0, stream, res, rows, norm_w, eps, true_width, static_cast<bf16 *>(out),
                           width);
    return hipGetLastError();
}

}  // namespace w4a16
