// One-token products with dense weights for gfx950: y[N] = W[N, K] x[K], W row-major in the element type.
//
// HBM-bound: every byte of W is read once.  A wavefront owns R consecutive rows at a time and reads each as coalesced
// 1 KiB pieces (8 consecutive k per lane), R x U of them in flight; x lies in LDS in the element type.  The row sums are
// fp32, added over the 64 lanes by a butterfly.  The workgroups walk the rows with a stride (at most kMaxBlocks of them),
// so that what a workgroup does to get x is done once per workgroup and not once per row group.
//
// The intake computes x where another kernel would otherwise be launched for it: the embedding row, or the residual
// stream with the normed output of the previous sublayer added (every workgroup redoes this small sum from L2; one of
// them stores it), or the final norm of that, or the norm of the stream with the previous sublayer's output added.  The first
// weights are requested before it is waited for.  The row sums can be combined in pairs: activation of a gate row times an up row.
#include "dense.h"
#include "dense_kernels.h"

namespace w4a16 {

namespace {

constexpr int kGemvWaves = 4, kGemvThreads = 64 * kGemvWaves;
constexpr int kMaxBlocks = 1024;
constexpr int kPiece = 512;   // elements of a row that a wave reads at once
constexpr int kIntakeNormedEmbed = 8;   // kIntakeNormed of an embedding row

template <class T>
struct GemvParams {
    const T *w;
    T *out;
    float *out_f32;
    unsigned long long *keys;
    int n_valid, K, N, groups;
    const T *x;
    const float *res, *y, *norm_w, *final_w;
    float eps;
    int width;
    float *res_out;
    T *h_out;
    const T *embed;
    const int32_t *token;
    float scale;
    RowOutput ro;
};

// sum over the workgroup, for every thread
__device__ __forceinline__ float block_sum(float v, float *red) {
    v = wave_reduce<false>(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = red[0];
#pragma unroll
    for (int i = 1; i < kGemvWaves; ++i) s += red[i];
    return s;
}

// x into LDS (K elements, zeros up to the next piece).  QUADS > 0: for up to 1024 QUADS elements.  What x is made of is asked for in front of the
// first weights (a wave's loads return in order) and all at once, and kept in registers from one pass over x to the next.  (Behind the weights, a
// round trip per 1024 elements and pass: gate and up of 2 x 8192 x 2048 behind a norm 14.1 -> 12.8 us = 5.3 TB/s, a router of 64 x 2048 behind a residual 4.5 -> 3.3 us.)
// QUADS 0, any length: every pass asks for what it uses, behind the weights.  (Registers in batches, every pass all operands of them anew,
// took 13.5 us instead of 10.5 for 2112 x 5120 behind a final norm.)  An x that is there already comes as it is, 8192 elements at a time.
template <class T, int MODE, int QUADS>
struct Intake {
    static constexpr int kKept = QUADS > 0 ? QUADS : 1, kStep = 4 * kGemvThreads;   // quads of a thread; elements between them
    static constexpr bool kRow = MODE == kIntakeEmbed || MODE == kIntakeNormedEmbed, kNormed = MODE == kIntakeNormed || MODE == kIntakeNormedEmbed;
    static constexpr bool kPlain = MODE == kIntakePlain, kAhead = kPlain || QUADS > 0;
    static constexpr int kY = 1, kRest = 2, kLast = 4, kAll = 7;   // operands: y; what else makes the value; final_w
    struct Operands {
        floatx4 res, y, norm, last;
    };
    const GemvParams<T> &p;
    T *xs;
    float *red;
    const T *row = nullptr;   // of the embedding
    Vec8<T> x[4];
    Operands kept[kKept];

    __device__ __forceinline__ static floatx4 quad_of(const float *v) { return *reinterpret_cast<const floatx4 *>(v); }
    template <int WHAT>
    __device__ __forceinline__ Operands load(int i) const {
        Operands o;
        if constexpr (kRow) {
            float e[4];
            load4(row + i, e);
            o.res = floatx4{e[0], e[1], e[2], e[3]} * p.scale;
        } else {
            // (without y: read all the same where operands are kept, and not used)
            if constexpr (WHAT & kRest) o.res = quad_of(p.res + i);
            if (WHAT & kY)
                if (kAhead || p.y) o.y = quad_of((kAhead && !p.y ? p.res : p.y) + i);
            if ((MODE == kIntakeResidual || MODE == kIntakeFinal) && (WHAT & kRest))
                if (kAhead || p.y) o.norm = quad_of((kAhead && !p.y ? p.res : p.norm_w) + i);
        }
        if constexpr ((MODE == kIntakeFinal || kNormed) && (WHAT & kLast)) o.last = quad_of(p.final_w + i);
        return o;
    }
    __device__ __forceinline__ void load_plain(int q) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int i = 8 * ((int)threadIdx.x + (4 * q + b) * kGemvThreads);
            x[b] = load8(p.x + (i < p.K ? i : p.K - 8));
        }
    }
    __device__ __forceinline__ void begin() {
        if constexpr (kRow) row = p.embed + (size_t)p.token[0] * p.K;
        if constexpr (kPlain) load_plain(0);
        else if constexpr (kAhead) {
#pragma unroll
            for (int b = 0; b < kKept; ++b) {
                const int i = 4 * (int)threadIdx.x + b * kStep;
                kept[b] = load<kAll>(i < p.K ? i : p.K - 4);   // (past the end the last ones)
            }
        }
    }
    __device__ __forceinline__ static float squares(floatx4 v, float ss) {
#pragma unroll
        for (int j = 0; j < 4; ++j) ss = fmaf(v[j], v[j], ss);
        return ss;
    }
    __device__ __forceinline__ float rstd_of(float ss) const { return 1.0f / sqrtf(block_sum(ss, red) / (float)p.width + p.eps); }
    // f(operands, first element) over all of x
    template <int WHAT, class F>
    __device__ __forceinline__ void pass(F f) const {
        if constexpr (kAhead) {
#pragma unroll
            for (int b = 0; b < kKept; ++b)
                if (const int i = 4 * (int)threadIdx.x + b * kStep; i < p.K) f(kept[b], i);
        } else {
            for (int i = 4 * (int)threadIdx.x; i < p.K; i += kStep) f(load<WHAT>(i), i);
        }
    }
    __device__ __forceinline__ void finish() {
        const int kl = (p.K + kPiece - 1) / kPiece * kPiece;
        for (int i = p.K + 8 * (int)threadIdx.x; i < kl; i += 8 * kGemvThreads) store8(xs + i, zero8<T>());
        if constexpr (kPlain) {
            for (int q = 0; q * 4 * 8 * kGemvThreads < p.K; ++q) {
                if (q > 0) load_plain(q);
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const int i = 8 * ((int)threadIdx.x + (4 * q + b) * kGemvThreads);
                    if (i < p.K) store8(xs + i, x[b]);
                }
            }
            return;
        }
        float rstd = 0.f;
        if constexpr (MODE == kIntakeResidual || MODE == kIntakeFinal) {
            if (p.y) {
                float ss = 0.f;
                pass<kY>([&](const Operands &o, int) { ss = squares(o.y, ss); });
                rstd = rstd_of(ss);
            }
        }
        auto value = [&](const Operands &o) {   // the new residual
            if constexpr (kRow) return o.res;
            if constexpr (MODE == kIntakeNormed) return p.y ? o.res + o.y : o.res;
            floatx4 v = o.res;
            if (p.y) {
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = fmaf(o.y[j] * rstd, o.norm[j], v[j]);
            }
            return v;
        };
        auto keep = [&](int i, floatx4 v) {
            if (blockIdx.x != 0) return;
            if (p.res_out) store4(p.res_out + i, v[0], v[1], v[2], v[3]);
            if constexpr (!kNormed)
                if (p.h_out) store4(p.h_out + i, v[0], v[1], v[2], v[3]);
        };
        if constexpr (MODE == kIntakeEmbed || MODE == kIntakeResidual) {
            pass<kY | kRest>([&](const Operands &o, int i) {
                const floatx4 v = value(o);
                store4(xs + i, v[0], v[1], v[2], v[3]);
                keep(i, v);
            });
        } else {
            float ss = 0.f;
            pass<kY | kRest>([&](const Operands &o, int i) {
                const floatx4 v = value(o);
                ss = squares(v, ss);
                if constexpr (kNormed) keep(i, v);
            });
            const float r2 = rstd_of(ss);
            pass<kAll>([&](const Operands &o, int i) {
                const floatx4 v = value(o);
                store4(xs + i, v[0] * r2 * o.last[0], v[1] * r2 * o.last[1], v[2] * r2 * o.last[2], v[3] * r2 * o.last[3]);
            });
        }
    }
};

// (PAIR: rows 2 o and 2 o + 1 of the walk are the gate and the up row of output o.)  Past the end: read in range, left out of the
// sum or never stored; no branch, behind which nobody could count the requests that are on their way.
template <class T, int R, int U, bool PAIR>
__device__ __forceinline__ void request(Vec8<T> (&w)[R][U], const T *base, int K, int N, int row0, int c0) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int row = row0 + r < N ? row0 + r : N - 1;
        if constexpr (PAIR) row = (row >> 5) * 32 + ((row & 31) >> 1) + 16 * (row & 1);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = (c0 + u) * kPiece + 8 * lane;
            w[r][u] = stream8(base + (size_t)row * K + (k < K ? k : K - 8));
        }
    }
}

template <class T, int R, int U, int MODE, bool PAIR, int QUADS>
__global__ void __launch_bounds__(kGemvThreads) dense_gemv_kernel(const GemvParams<T> p) {
    extern __shared__ __attribute__((aligned(16))) char gemv_lds[];
    __shared__ float red[kGemvWaves];
    T *xs = reinterpret_cast<T *>(gemv_lds);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int stride = gridDim.x * kGemvWaves;
    const int pieces = (p.K + kPiece - 1) / kPiece;
    int g = blockIdx.x * kGemvWaves + wave;
    Vec8<T> w[R][U];
    Intake<T, MODE, QUADS> in{p, xs, red};
    in.begin();
    __builtin_amdgcn_sched_barrier(0);
    request<T, R, U, PAIR>(w, p.w, p.K, p.N, g * R, 0);
    __builtin_amdgcn_sched_barrier(0);
    in.finish();
    __syncthreads();
    unsigned long long best = 0;
    for (; g < p.groups; g += stride) {
        float acc[R];
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = 0.f;
        for (int c0 = 0; c0 < pieces; c0 += U) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (c0 + u >= pieces) break;   // uniform
                const Vec8<T> xv = load8(xs + (c0 + u) * kPiece + 8 * lane);
                const bool in = (c0 + u) * kPiece + 8 * lane < p.K;
#pragma unroll
                for (int r = 0; r < R; ++r) acc[r] = dot8(in ? w[r][u] : zero8<T>(), xv, acc[r]);
            }
            if (c0 + U < pieces) request<T, R, U, PAIR>(w, p.w, p.K, p.N, g * R, c0 + U);
        }
        if (g + stride < p.groups) request<T, R, U, PAIR>(w, p.w, p.K, p.N, (g + stride) * R, 0);
        float mine = 0.f;
        if constexpr (PAIR) {
#pragma unroll
            for (int r = 0; r < R; r += 2) {
                const float a = wave_reduce<false>(acc[r]), b = wave_reduce<false>(acc[r + 1]);
                mine = lane == r / 2 ? (p.ro.gate == kGateGelu ? gelu_tanh_of<float>(a) : silu_f32(a)) * b : mine;
            }
            const int o = g * (R / 2) + lane;
            if (lane < R / 2 && 2 * o < p.N) p.out[o] = from_float<T>(mine);
            continue;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float s = wave_reduce<false>(acc[r]);
            mine = lane == r ? s : mine;
        }
        const int row = g * R + lane;
        if (lane < R && row < p.N) {
            if (row >= p.ro.silu_begin && row < p.ro.silu_end) mine = silu_f32(mine);
            if (p.out_f32) p.out_f32[row] = mine;
            else p.out[row] = from_float<T>(mine);
            if (p.keys && row < p.n_valid) {
                const unsigned long long key = ((unsigned long long)order_key(mine) << 32) | (0xFFFFFFFFu - (uint32_t)row);
                best = key > best ? key : best;
            }
        }
    }
    if (p.keys) {
        best = wave_max_u64(best);
        if (lane == 0) p.keys[blockIdx.x * kGemvWaves + wave] = best;
    }
}

// AT keys of a thread at a time: a round trip for up to 4096 of them with 4, where fewer ask for one each
template <int AT>
__global__ void __launch_bounds__(1024) argmax_keys_kernel(const unsigned long long *keys, int n, int32_t *token, int32_t *position,
                                                           int32_t *history) {
    __shared__ unsigned long long part[16];
    const int32_t here = position ? position[0] : 0;   // (every thread: asked for with the keys)
    unsigned long long best = 0;
    for (int i0 = threadIdx.x; i0 < n; i0 += AT * 1024) {
        unsigned long long k[AT];
#pragma unroll
        for (int j = 0; j < AT; ++j) k[j] = keys[i0 + 1024 * j < n ? i0 + 1024 * j : i0];
#pragma unroll
        for (int j = 0; j < AT; ++j) best = k[j] > best ? k[j] : best;
    }
    best = wave_max_u64(best);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 1; i < 16; ++i) best = part[i] > best ? part[i] : best;
        const int32_t id = (int32_t)(0xFFFFFFFFu - (uint32_t)(best & 0xFFFFFFFFull));
        if (token) token[0] = id;
        if (position) {
            const int32_t next = here + 1;   // the position of the chosen token
            position[0] = next;
            if (history) history[next] = id;
        }
    }
}

template <class T, int R, int U, int QUADS>
hipError_t launch_mode(const GemvParams<T> &p, int mode, int grid, size_t lds, hipStream_t stream) {
    auto run = [&](auto kernel) {
        if (lds > 48 * 1024) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(kGemvThreads), lds, stream, p);
        return hipGetLastError();
    };
    if (p.ro.gate) {
        if constexpr (R >= 2)
            return mode != kIntakeNormed ? run(&dense_gemv_kernel<T, R, U, kIntakePlain, true, 2>)
                   : p.embed             ? run(&dense_gemv_kernel<T, R, U, kIntakeNormedEmbed, true, QUADS>)
                                         : run(&dense_gemv_kernel<T, R, U, kIntakeNormed, true, QUADS>);
        return hipErrorInvalidValue;
    }
    if constexpr (R > 1 && QUADS != 2) return hipErrorInvalidValue;   // (without a gate rows past 2048 come one to a wave)
    else
        switch (mode == kIntakeNormed && p.embed ? (int)kIntakeNormedEmbed : mode) {
            case kIntakePlain: return run(&dense_gemv_kernel<T, R, U, kIntakePlain, false, 2>);
            case kIntakeResidual: return run(&dense_gemv_kernel<T, R, U, kIntakeResidual, false, QUADS>);
            case kIntakeEmbed: return run(&dense_gemv_kernel<T, R, U, kIntakeEmbed, false, QUADS>);
            case kIntakeNormed: return run(&dense_gemv_kernel<T, R, U, kIntakeNormed, false, QUADS>);
            case kIntakeNormedEmbed: return run(&dense_gemv_kernel<T, R, U, kIntakeNormedEmbed, false, QUADS>);
            default: return run(&dense_gemv_kernel<T, R, U, kIntakeFinal, false, QUADS>);
        }
}

// By the length of x: two or four quads of its operands in a thread's registers (four: up to 150, three waves to a SIMD in fp32), which is faster wherever they
// fit, or passes that ask for them.  4096 x 4096 behind a final norm, four quads / passes / passes with batches of two quads: 10.2 / 11.6 / 14.7 us,
// fp32 15.7 / 20.8 / 21.0; 64 x 4096 4.2 / 5.9 / 5.7; 2112 x 5120, passes / batches of four quads / of two: 10.5 / 15.3 / 13.5.
template <class T, int R, int U>
hipError_t launch_length(const GemvParams<T> &p, int mode, int grid, size_t lds, hipStream_t stream) {
    if (p.K <= 2048) return launch_mode<T, R, U, 2>(p, mode, grid, lds, stream);
    if (p.K <= 4096) return launch_mode<T, R, U, 4>(p, mode, grid, lds, stream);
    return launch_mode<T, R, U, 0>(p, mode, grid, lds, stream);
}

int rows_per_wave(int K, int N) { return K > 2048 || N < 512 ? 1 : K > 1024 ? 2 : 4; }

template <class T>
hipError_t launch_typed(const void *w, const RowIntake &in, void *out, float *out_f32, unsigned long long *keys, int n_valid, int K, int N,
                        const RowOutput &ro, hipStream_t stream) {
    GemvParams<T> p;
    p.ro = ro;
    p.w = static_cast<const T *>(w);
    p.out = static_cast<T *>(out);
    p.out_f32 = out_f32;
    p.keys = keys;
    p.n_valid = n_valid;
    p.K = K;
    p.N = N;
    p.x = static_cast<const T *>(in.x);
    p.res = in.res;
    p.y = in.y;
    p.norm_w = in.norm_w;
    p.final_w = in.final_w;
    p.eps = in.eps;
    p.width = in.width;
    p.res_out = in.res_out;
    p.h_out = static_cast<T *>(in.h_out);
    p.embed = static_cast<const T *>(in.embed);
    p.token = in.token;
    p.scale = in.scale;
    const int R = ro.gate && K > 1024 ? 2 : ro.gate ? 4 : rows_per_wave(K, N);
    p.groups = (N + R - 1) / R;
    const int need = (p.groups + kGemvWaves - 1) / kGemvWaves, grid = need < kMaxBlocks ? need : kMaxBlocks;
    const size_t lds = (size_t)((K + kPiece - 1) / kPiece) * kPiece * sizeof(T);
    switch (R) {
        case 1: return launch_length<T, 1, 8>(p, in.mode, grid, lds, stream);
        case 2: return launch_length<T, 2, 4>(p, in.mode, grid, lds, stream);
        default: return launch_mode<T, 4, 2, 2>(p, in.mode, grid, lds, stream);   // (K <= 1024)
    }
}

}  // namespace

int dense_gemv_blocks(int K, int N) {
    const int R = rows_per_wave(K, N), per = R * kGemvWaves;
    const int need = (N + per - 1) / per;
    return need < kMaxBlocks ? need : kMaxBlocks;
}

hipError_t launch_dense_gemv(int dtype, const void *w, const RowIntake &in, void *out, float *out_f32, unsigned long long *keys, int n_valid,
                             int K, int N, hipStream_t stream, const RowOutput &ro) {
    return dtype == kF32 ? launch_typed<float>(w, in, out, out_f32, keys, n_valid, K, N, ro, stream)
                         : launch_typed<bf16>(w, in, out, out_f32, keys, n_valid, K, N, ro, stream);
}

hipError_t launch_argmax_keys(const unsigned long long *keys, int n, int32_t *token, int32_t *position, int32_t *history, hipStream_t stream) {
    hipLaunchKernelGGL(n <= 1024 ? &argmax_keys_kernel<1> : &argmax_keys_kernel<4>, dim3(1), dim3(1024), 0, stream, keys, n, token, position, history);
    return hipGetLastError();
}

}  // namespace w4a16
