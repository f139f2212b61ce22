// Mixture of experts behind a grouped sigmoid router, for gfx950.
//
// Choice: score s = sigmoid(logit); choice score s + correction; the experts form `groups` equal groups of neighbours,
// a group counts as much as the sum of its two largest choice scores; the `top` experts with the largest choice scores
// among the `keep` best groups are taken, each with weight s.  Everything in fp32; ties go to the lower index.  One
// wavefront chooses for one token.
//
// One token: the gate / up product makes the choice itself (every workgroup, from the same logits: cheaper than a launch)
// and the first workgroup of a slot leaves it for the down product, which adds the experts' outputs with their weights.
// Many tokens: the choices become (token, slot) entries sorted by expert and cut into row tiles, on which dense_gemm.hip
// runs one grouped product each for gate / up and down.
#include "dense.h"
#include "dense_kernels.h"

namespace w4a16 {

namespace {

constexpr int kMoeWaves = 4, kMoeThreads = 64 * kMoeWaves;
constexpr int kMoePiece = 512;

// Called by one whole wavefront, which owns experts lane + 64 j, j < PL; choice: LDS scratch of r.experts floats, group: of
// r.groups floats (both of this wave).  ids / weights [top] may be LDS or global.
template <int PL>
__device__ __forceinline__ void choose_experts(const Router &r, const float *logits, float *choice, float *group, int32_t *ids,
                                               float *weights) {
    const int lane = threadIdx.x & 63;
    const int size = r.experts / r.groups;
    float score[PL], c[PL];
#pragma unroll
    for (int j = 0; j < PL; ++j) {
        const int e = lane + 64 * j;
        score[j] = 0.f;
        c[j] = -INFINITY;
        if (e < r.experts) {
            score[j] = sigmoid_f32(logits[e]);
            c[j] = score[j] + r.correction[e];
            choice[e] = c[j];
        }
    }
    if (r.groups > 1) {
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        for (int g = lane; g < r.groups; g += 64) {
            float a = -INFINITY, b = -INFINITY;   // the two largest
            for (int i = 0; i < size; ++i) {
                const float v = choice[g * size + i];
                b = fmaxf(b, fminf(a, v));
                a = fmaxf(a, v);
            }
            group[g] = size > 1 ? a + b : a;
        }
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        // experts outside the kept groups count as minus infinity
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            const int e = lane + 64 * j;
            if (e >= r.experts) continue;
            const int g = e / size;
            const float mine = group[g];
            int better = 0;
            for (int o = 0; o < r.groups; ++o) {
                const float v = group[o];
                better += v > mine || (v == mine && o < g);
            }
            if (better >= r.keep) c[j] = -INFINITY;
        }
    }
    for (int s = 0; s < r.top; ++s) {
        float best = c[0];
#pragma unroll
        for (int j = 1; j < PL; ++j) best = fmaxf(best, c[j]);
        best = wave_reduce<true>(best);
        bool found = false;   // wave-uniform; the lowest index among equals: the first j, its lowest lane
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            const unsigned long long hit = found ? 0ull : __ballot(c[j] == best);
            if (hit) {
                found = true;
                if (lane == __builtin_ctzll(hit)) {
                    ids[s] = lane + 64 * j;
                    weights[s] = score[j];
                    c[j] = -INFINITY;
                }
            }
        }
    }
}

template <class F>
auto with_lanes(int experts, F f) {
    if (experts <= 64) return f(std::integral_constant<int, 1>());
    if (experts <= 256) return f(std::integral_constant<int, 4>());
    return f(std::integral_constant<int, kMaxExperts / 64>());
}

template <int PL>
__global__ void __launch_bounds__(kMoeThreads) moe_select_kernel(const Router r, int parts, int tokens, int32_t *ids, float *weights) {
    extern __shared__ float select_lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, t = blockIdx.x * kMoeWaves + wave;
    if (t >= tokens) return;   // whole waves leave; no workgroup barrier below
    float *mine = select_lds + wave * (r.experts + r.groups);
    const float *logits = r.logits + (size_t)t * r.ld;
    if (parts > 1) {   // the router's product in slices along K, up to eight of them on their way; a lane reads back what it wrote
        float *sum = select_lds + kMoeWaves * (r.experts + r.groups) + wave * r.experts;
        const size_t size = (size_t)tokens * r.ld;
        for (int e = lane; e < r.experts; e += 64) {
            float z = 0.f;
            for (int s0 = 0; s0 < parts; s0 += 8) {
                float x[8];
#pragma unroll
                for (int s = 0; s < 8; ++s) x[s] = logits[(s0 + s < parts ? s0 + s : s0) * size + e];
#pragma unroll
                for (int s = 0; s < 8; ++s) z = s0 + s < parts ? z + x[s] : z;
            }
            sum[e] = z;
        }
        logits = sum;
    }
    choose_experts<PL>(r, logits, mine, mine + r.experts, ids + (size_t)t * r.top, weights + (size_t)t * r.top);
}

// One workgroup: sort the entries by expert (counting sort) and cut every expert's run into tiles of bm entries, or even ones where they
// are tall.  What bounds it: one CU's LDS additions, several lanes of a wave to a counter, and its stores.  An entry's place in its expert's run is what its
// addition returned, kept for the first kPlanKept entries of a thread; more entries are counted
// behind them and placed in a second pass.  Sums over the experts go by wave
// shuffles.  Lanes of a wave belong to runs all over the list, a cache line to a lane: thousands of entries are put in order in LDS and leave it side by side (up to kPlanDirect
// that costs 0.15 us more than it saves).  A wave whose entries are one expert's makes one addition.  16384 entries of 64 experts: 15.8 -> 12.4 us (before: two passes of
// additions, scans of ten barriers each), in a graph 10.1 -> 6.8 by way of LDS; of 256 11.8 -> 6.8, of one 19.3 -> 8.6; 4096 of 64 5.4 -> 4.8.
constexpr int kPlanDirect = 2048;
constexpr int kPlanKept = 16;
__global__ void __launch_bounds__(1024) moe_plan_kernel(const int32_t *ids, int entries, int experts, int bm, int max_tiles, int32_t *order,
                                                        int32_t *tiles) {
    __shared__ int count[kMaxExperts], first[kMaxExperts], sums[2][16];
    __shared__ uint16_t sorted[1024 * kPlanKept];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    int e[kPlanKept], place[kPlanKept];
#pragma unroll
    for (int j = 0; j < kPlanKept; ++j) e[j] = t + 1024 * j < entries ? ids[t + 1024 * j] : -1;
    count[t] = 0;   // kMaxExperts == number of threads
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPlanKept; ++j) {
        if (e[j] < 0) continue;
        const unsigned long long here = __ballot(1);
        if (__ballot(e[j] == __builtin_amdgcn_readfirstlane(e[j])) == here) {   // one expert: an addition for all of them
            const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(here >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)here, 0));
            int base = 0;
            if (rank == 0) base = atomicAdd(&count[e[j]], __popcll(here));
            place[j] = __builtin_amdgcn_readfirstlane(base) + rank;
        } else {
            place[j] = atomicAdd(&count[e[j]], 1);
        }
    }
    if (entries > 1024 * kPlanKept) {   // (behind the kept ones: those have the first places of each run)
        __syncthreads();
        for (int i = t + 1024 * kPlanKept; i < entries; i += 1024) atomicAdd(&count[ids[i]], 1);
    }
    __syncthreads();
    // exclusive prefix sums of the counts and of the tiles per expert
    const int n = count[t], parts = (n + bm - 1) / bm;
    int runs = n, cut = parts;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
        const int r = __shfl_up(runs, d), c = __shfl_up(cut, d);
        if (lane >= d) runs += r, cut += c;
    }
    if (lane == 63) sums[0][wave] = runs, sums[1][wave] = cut;
    __syncthreads();
    int total = 0;
    runs -= n;
    cut -= parts;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
        if (w < wave) runs += sums[0][w], cut += sums[1][w];
        total += sums[1][w];
    }
    first[t] = runs;
    const int each = bm > 256 && bm % 64 == 0 && n ? ((n + parts - 1) / parts + 31) / 32 * 32 : bm;
    if (t < experts)
        for (int i = 0; i < parts; ++i) {
            int32_t *row = tiles + 4 * (cut + i);
            const int left = n - i * each;
            row[0] = t;
            row[1] = runs + i * each;
            row[2] = left < each ? left : each;
            row[3] = 0;
        }
    if (t == 0) tiles[4 * max_tiles] = total;
    __syncthreads();
    if (entries > kPlanDirect && entries <= 1024 * kPlanKept) {
#pragma unroll
        for (int j = 0; j < kPlanKept; ++j)
            if (e[j] >= 0) sorted[first[e[j]] + place[j]] = (uint16_t)(t + 1024 * j);
        __syncthreads();
        for (int i = t; i < entries; i += 1024) order[i] = sorted[i];
        return;
    }
#pragma unroll
    for (int j = 0; j < kPlanKept; ++j)
        if (e[j] >= 0) order[first[e[j]] + place[j]] = t + 1024 * j;
    if (entries <= 1024 * kPlanKept) return;
    // the rest take the places from the end of their expert's run
    for (int i = t + 1024 * kPlanKept; i < entries; i += 1024) {
        const int x = ids[i];
        order[first[x] + atomicSub(&count[x], 1) - 1] = i;
    }
}

template <class T>
struct MoeGemv {
    Router r;
    const T *x, *w;
    T *h;
    float *y;
    int32_t *ids;
    float *weights;
    int K, ff, N, top;
};

// h[slot] = silu(gate x) * (up x); blockIdx.y = slot; a wave owns P neighbouring gate rows and the matching up rows
template <class T, int P, int U, int PL>
__global__ void __launch_bounds__(kMoeThreads) moe_gate_up_gemv_kernel(const MoeGemv<T> p) {
    extern __shared__ __attribute__((aligned(16))) char moe_lds[];
    __shared__ int32_t ids[kMaxTop];
    __shared__ float weights[kMaxTop];
    const int kl = (p.K + kMoePiece - 1) / kMoePiece * kMoePiece;
    T *xs = reinterpret_cast<T *>(moe_lds);
    float *scratch = reinterpret_cast<float *>(xs + kl);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, slot = blockIdx.y;
    if (wave == 0) choose_experts<PL>(p.r, p.r.logits, scratch, scratch + p.r.experts, ids, weights);
    else {
        for (int i = 8 * (tid - 64); i < p.K; i += 8 * (kMoeThreads - 64)) store8(xs + i, load8(p.x + i));
        for (int i = p.K + 8 * (tid - 64); i < kl; i += 8 * (kMoeThreads - 64)) store8(xs + i, zero8<T>());
    }
    __syncthreads();
    if (blockIdx.x == 0 && tid == 0) {
        p.ids[slot] = ids[slot];
        p.weights[slot] = weights[slot];
    }
    const T *w = p.w + (size_t)ids[slot] * 2 * p.ff * p.K;
    const int pieces = kl / kMoePiece;
    for (int f0 = (blockIdx.x * kMoeWaves + wave) * P; f0 < p.ff; f0 += gridDim.x * kMoeWaves * P) {
        float g[P], u[P];
#pragma unroll
        for (int j = 0; j < P; ++j) g[j] = u[j] = 0.f;
        // P divides 16, so the P rows lie in one block of 16 gate rows, the up rows 16 further on
        const T *gate = w + (size_t)(f0 / 16 * 32 + f0 % 16) * p.K + 8 * lane, *up = gate + (size_t)16 * p.K;
        for (int c0 = 0; c0 < pieces; c0 += U) {
            Vec8<T> wg[P][U], wu[P][U];
#pragma unroll
            for (int j = 0; j < P; ++j)
#pragma unroll
                for (int c = 0; c < U; ++c) {
                    const int k = (c0 + c) * kMoePiece;
                    const bool in = k + 8 * lane < p.K;
                    wg[j][c] = in ? stream8(gate + (size_t)j * p.K + k) : zero8<T>();
                    wu[j][c] = in ? stream8(up + (size_t)j * p.K + k) : zero8<T>();
                }
#pragma unroll
            for (int c = 0; c < U; ++c) {
                const int pc = c0 + c < pieces ? c0 + c : pieces - 1;
                const Vec8<T> xv = load8(xs + pc * kMoePiece + 8 * lane);
#pragma unroll
                for (int j = 0; j < P; ++j) {
                    g[j] = dot8(wg[j][c], xv, g[j]);
                    u[j] = dot8(wu[j][c], xv, u[j]);
                }
            }
        }
        float mine = 0.f;
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const float v = silu_f32(wave_reduce<false>(g[j])) * wave_reduce<false>(u[j]);
            mine = lane == j ? v : mine;
        }
        if (lane < P) p.h[(size_t)slot * p.ff + f0 + lane] = from_float<T>(mine);
    }
}

// y[n] = sum_s weight_s (down_s h_s)[n]; a wave owns a row, the pieces of all slots run through one loop, U of them in flight.  What bounds it:
// HBM, behind two round trips, the choice's and the weights'.  So h is asked for first, a wave's pieces at once, then
// the choice, a slot to a lane, and the weights before h is stored to LDS, all of a row where it is U pieces.  (No branch and no wait between
// the requests: addresses past the end are clamped.)  8 experts of 2048 x 1024 (33.5 MB), one product behind the other: 8.5 -> 8.0 us = 4.2 TB/s (a
// round trip per slot for h before).
template <class T, int U>
__global__ void __launch_bounds__(kMoeThreads, 2) moe_down_gemv_kernel(const MoeGemv<T> p) {
    extern __shared__ __attribute__((aligned(16))) char moe_lds[];
    T *hs = reinterpret_cast<T *>(moe_lds);
    constexpr int H = 4;   // pieces of h that a wave has in flight
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pieces = (p.ff + kMoePiece - 1) / kMoePiece, items = p.top * pieces, stride = gridDim.x * kMoeWaves;
    const int last = p.ff - 8;   // (ff is a multiple of 64)
    // element offset of this lane's chunk in piece i: slot i / pieces, and whether the piece has that much
    auto chunk = [&](int i, int &slot, bool &in) {
        slot = i / pieces;
        const int k = (i - slot * pieces) * kMoePiece + 8 * lane;
        in = k <= last;
        return in ? k : last;
    };
    Vec8<T> hv[H];
    auto request_h = [&](int i0) {
#pragma unroll
        for (int j = 0; j < H; ++j) {
            int slot;
            bool in;
            const int k = chunk(min(i0 + kMoeWaves * j, items - 1), slot, in);
            hv[j] = load8(p.h + (size_t)slot * p.ff + k);
            if (!in) hv[j] = zero8<T>();
        }
    };
    request_h(wave);
    const int id = p.ids[lane < p.top ? lane : 0];   // (top <= 32)
    const float weight = p.weights[lane < p.top ? lane : 0];
    int n = blockIdx.x * kMoeWaves + wave;
    Vec8<T> w[U];
    float wt[U];
    auto request = [&](int row, int i0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int slot;
            bool in;
            const int k = chunk(min(i0 + u, items - 1), slot, in);
            const int expert = __builtin_amdgcn_readlane(id, slot);
            const float x = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, weight), slot));
            wt[u] = x;
            w[u] = stream8(p.w + ((size_t)expert * p.N + row) * p.ff + k);
        }
    };
    request(min(n, p.N - 1), 0);
    for (int i0 = wave;;) {
#pragma unroll
        for (int j = 0; j < H; ++j)
            if (i0 + kMoeWaves * j < items) store8(hs + (i0 + kMoeWaves * j) * kMoePiece + 8 * lane, hv[j]);   // (slot s, piece c) lies at s * kl + c * 512
        i0 += kMoeWaves * H;
        if (i0 >= items) break;
        request_h(i0);
    }
    __syncthreads();
    float acc = 0.f;
    for (int i0 = 0; n < p.N;) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (i0 + u >= items) break;   // uniform; nothing is added for what is not there, not even 0 times an infinity
            int slot;
            bool in;
            const int i = i0 + u;
            chunk(i, slot, in);
            const Vec8<T> row = in ? w[u] : zero8<T>();
            acc = fmaf(wt[u], dot8(row, load8(hs + i * kMoePiece + 8 * lane), 0.f), acc);
        }
        __builtin_amdgcn_sched_barrier(0);   // (the next weights go into the same registers)
        i0 += U;
        if (i0 >= items) {
            const float sum = wave_reduce<false>(acc);
            if (lane == 0) p.y[n] = sum;
            acc = 0.f;
            i0 = 0;
            n += stride;
            if (n >= p.N) break;
        }
        request(n, i0);
    }
}

template <class F>
hipError_t with_lds(F kernel, size_t lds) {
    if (lds <= 48 * 1024) return hipSuccess;
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

template <class T>
hipError_t gate_up(const Router &r, const void *x, const void *w, void *h, int32_t *ids, float *weights, int K, int ff, hipStream_t stream) {
    MoeGemv<T> p{};
    p.r = r;
    p.x = static_cast<const T *>(x);
    p.w = static_cast<const T *>(w);
    p.h = static_cast<T *>(h);
    p.ids = ids;
    p.weights = weights;
    p.K = K;
    p.ff = ff;
    p.top = r.top;
    const size_t lds = (size_t)((K + kMoePiece - 1) / kMoePiece) * kMoePiece * sizeof(T) + (size_t)(r.experts + r.groups) * sizeof(float);
    const int P = K > 1024 ? 1 : 2;
    int gx = (ff + kMoeWaves * P - 1) / (kMoeWaves * P);
    const dim3 grid(gx, r.top), block(kMoeThreads);
    auto run = [&](auto kernel) {
        const hipError_t e = with_lds(kernel, lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kernel, grid, block, lds, stream, p);
        return hipGetLastError();
    };
    return with_lanes(r.experts, [&](auto pl) {
        constexpr int PL = decltype(pl)::value;
        return P == 1 ? run(&moe_gate_up_gemv_kernel<T, 1, 4, PL>) : run(&moe_gate_up_gemv_kernel<T, 2, 2, PL>);
    });
}

template <class T>
hipError_t down(const void *h, const void *w, const int32_t *ids, const float *weights, float *y, int top, int ff, int N, hipStream_t stream) {
    MoeGemv<T> p{};
    p.h = const_cast<T *>(static_cast<const T *>(h));
    p.w = static_cast<const T *>(w);
    p.ids = const_cast<int32_t *>(ids);
    p.weights = const_cast<float *>(weights);
    p.y = y;
    p.ff = ff;
    p.N = N;
    p.top = top;
    const size_t lds = (size_t)top * ((ff + kMoePiece - 1) / kMoePiece) * kMoePiece * sizeof(T);
    // Pieces in flight: 4 in fp32 (twice the registers) and where a row is no more, else 8.  (Requests past a row's end read its last piece again: with 16 for
    // every row, 2 experts of 2048 x 1024 took 6.2 us, 4.0 with 4; 8 of them 8.65, 8.0 with 8.)
    auto kernel = sizeof(T) == 4 || top * ((ff + kMoePiece - 1) / kMoePiece) <= 4 ? &moe_down_gemv_kernel<T, 4> : &moe_down_gemv_kernel<T, 8>;
    const hipError_t e = with_lds(kernel, lds);
    if (e != hipSuccess) return e;
    const int need = (N + kMoeWaves - 1) / kMoeWaves;
    hipLaunchKernelGGL(kernel, dim3(need < 1024 ? need : 1024), dim3(kMoeThreads), lds, stream, p);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_moe_gate_up_gemv(int dtype, const Router &r, const void *x, const void *w_gate_up, void *h, int32_t *ids, float *weights, int K,
                                   int ff, hipStream_t stream) {
    return dtype == kF32 ? gate_up<float>(r, x, w_gate_up, h, ids, weights, K, ff, stream)
                         : gate_up<bf16>(r, x, w_gate_up, h, ids, weights, K, ff, stream);
}

hipError_t launch_moe_down_gemv(int dtype, const void *h, const void *w_down, const int32_t *ids, const float *weights, float *y, int top, int ff,
                                int N, hipStream_t stream) {
    return dtype == kF32 ? down<float>(h, w_down, ids, weights, y, top, ff, N, stream) : down<bf16>(h, w_down, ids, weights, y, top, ff, N, stream);
}

hipError_t launch_moe_select(const Router &r, int parts, int tokens, int32_t *ids, float *weights, hipStream_t stream) {
    const size_t lds = (size_t)kMoeWaves * (r.experts * (parts > 1 ? 2 : 1) + r.groups) * sizeof(float);   // (48 KiB at most)
    return with_lanes(r.experts, [&](auto pl) {
        hipLaunchKernelGGL(moe_select_kernel<decltype(pl)::value>, dim3((tokens + kMoeWaves - 1) / kMoeWaves), dim3(kMoeThreads), lds, stream, r, parts,
                           tokens, ids, weights);
        return hipGetLastError();
    });
}

int moe_max_tiles(int entries, int experts, int bm) { return entries / bm + (entries < experts ? entries : experts); }

hipError_t launch_moe_plan(const int32_t *ids, int entries, int experts, int bm, int32_t *order, int32_t *tiles, hipStream_t stream) {
    hipLaunchKernelGGL(moe_plan_kernel, dim3(1), dim3(1024), 0, stream, ids, entries, experts, bm, moe_max_tiles(entries, experts, bm), order, tiles);
    return hipGetLastError();
}

}  // namespace w4a16
