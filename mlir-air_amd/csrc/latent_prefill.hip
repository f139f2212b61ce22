// Causal attention of a long portion on expanded keys and values, for gfx950: queries [dim | rot] per head (rotated by
// latent_prepare), keys = the head's dim columns of the expanded matrix followed by the rotated part of the cache row that
// all heads share, values = the head's vdim columns, a learned sink per head in the denominator, and the output gate
// applied before the only store.  WINDOW is the same kernel on grouped keys and values of their own projections
// (head_attention.hip): rows [key | value] of one matrix per key / value head, positions going round in a ring of rows, a limit to
// how far back a query sees, neither sink nor gate.
//
// Both products are computed transposed, so that a lane owns one query from the scores to the output:
//   S^T[key, q] = K . Q^T      A = K rows from LDS, B = Q^T held in registers
//   O^T[d, q]  += V^T . P^T    A = V^T (transposing LDS read), B = P^T built from the lane's own S^T registers
// The D layout gives a lane keys 4 g .. + 3 of each 16-key block; the k slots of the second product are defined as exactly
// those keys, so P never moves between lanes.  Four waves of QB blocks of 16 queries each share the K and V rows going through
// LDS; the next block of keys travels global -> registers while one is multiplied.  With SETS = 2 a second set of four waves
// takes the odd key blocks for the same queries, and the two partial results are merged through LDS at the end (with gates a block of queries by
// each set): the longest rows take half as long, and two waves share a SIMD.  (2048 tokens, 16 heads of 128 + 64 / 128: merge, gates and stores by one
// set 7.8 of 65 us, gates by an exponential and a division each and asked for one by one; now 3.7 of 62.)  The grid puts the longest rows first.  The running maximum may lag the true one by 2^8 (as in prefill_attention.hip), so
// rescaling is rare; the row sum is a product with a row of ones.
//
// Head sizes that are common have kernels of their own (EXACT: everything unrolled); any other size runs on the next
// larger register allotment with uniform bounds.
//
// What bounds it: the chain of a block of keys.  In the kernels of their own four operands are on their way from LDS while one is multiplied (five to six spill), and
// no load of the queries can be in flight when the loop begins.  (Before, every block waited for the next one to arrive from memory and for most of its LDS reads one
// by one.  us, 2048 tokens: 16 heads of 128 + 64 / 128 62.6 -> 56.1, 8 heads 53.0 -> 43.2; 16 windowed heads of 128 over 4, window 1024 32.9 -> 29.7, window 2048 50.2 -> 43.6; of 64,
// window 2048 32.9 -> 26.9.  Taken back on top: the keys stored beside the softmax and the values beside the scores, the two sets half a block apart: 2 to 40 % slower.)
#include <algorithm>

#include "dense.h"
#include "dense_kernels.h"

namespace w4a16 {

namespace {

constexpr int kSetThreads = 256;
constexpr float kMasked = -1.0e30f;
constexpr float kNoMax = -1.0e20f;   // "no score yet": far below any score, far above a masked one
constexpr float kLazy = 8.0f;

template <class T>
struct PrefillArgs {
    const T *q, *kv, *cache;
    T *out;
    long ldq, ldkv, ldo;
    int ldc, rot_off;        // cache row length, start of the rotated part in it
    int heads, dim, rot, vdim;
    int v_off, gate_off;     // columns of the values in kv, of the gate in q's matrix
    int M, total;            // queries, keys (the queries are the last M positions)
    float scale_log2;
    const float *sink;
    long head_q, group_q, head_k, head_v;   // elements between two heads' queries, key / value heads' queries, keys, values
    int group, window, ring;                // query heads per key / value head
    float out_scale;
};

// v sigmoid(z); a z that is not a number stays one (told by its bits: this file is compiled without NaNs)
__device__ __forceinline__ float gated(float v, float z) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, z);
    return __builtin_bit_cast(float, (bits & 0x7FFFFFFFu) > 0x7F800000u ? bits : __builtin_bit_cast(uint32_t, gated_f32(v, z)));
}

template <class T>
__device__ __forceinline__ Vec8<T> ones8();
template <>
__device__ __forceinline__ Vec8<bf16> ones8<bf16>() { return {u32x4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u}}; }
template <>
__device__ __forceinline__ Vec8<float> ones8<float>() { return {floatx4{1.f, 1.f, 1.f, 1.f}, floatx4{1.f, 1.f, 1.f, 1.f}}; }

// NQ: K-steps of 32 of a score; NV: 16-column tiles of the output; EXACT: the sizes are exactly these, otherwise at most
// these.  blockIdx.z picks a range of 16 NV value columns.
// (EXACT addresses K and V rows with 32-bit offsets: the expanded matrix is smaller than 4 GiB.)
template <class T, int NQ, int NV, int QB, int KB, int SETS, bool EXACT, bool WINDOW>
__global__ void __launch_bounds__(SETS * kSetThreads, SETS) latent_prefill_kernel(const PrefillArgs<T> p) {
    constexpr int NKK = KB / 16, NT = KB / 32, QW = 64 * QB;
    extern __shared__ __attribute__((aligned(16))) char pf_lds[];
    const int tid = threadIdx.x & (kSetThreads - 1), lane = tid & 63;   // thread within its set
    const int wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int set = SETS == 1 ? 0 : wave8 >> 2, wave = wave8 & 3;
    const int ql = lane & 15, g = lane >> 4;
    const int head = blockIdx.x, item = gridDim.y - 1 - blockIdx.y;
    const int qd = EXACT ? 32 * NQ : p.dim + p.rot;
    const int vcol0 = EXACT ? 0 : blockIdx.z * 16 * NV;
    const int vd = EXACT ? 16 * NV : (p.vdim - vcol0 < 16 * NV ? p.vdim - vcol0 : 16 * NV);
    const int nq = qd / 32, nv = vd / 16;
    const int kp = qd + 16 / (int)sizeof(T), vp = vd + 32 / (int)sizeof(T);
    T *kt = reinterpret_cast<T *>(pf_lds) + set * KB * (kp + vp);
    T *vt = kt + KB * kp;

    const int pos0 = p.total - p.M;
    const int q0 = item * QW + 16 * QB * wave;                    // first query row of this wave
    const int item_end = (item + 1) * QW < p.M ? (item + 1) * QW : p.M;
    const int blocks = (pos0 + item_end + KB - 1) / KB;
    const int wave_last = pos0 + q0 + 16 * QB - 1;                // last position of this wave's queries
    const int kvh = WINDOW ? head / p.group : head;
    // blocks that are wholly in front of the window of every query of the item are left out, and of those of a wave by the wave
    const int item_first = WINDOW ? pos0 + item * QW - p.window + 1 : 0, first = item_first > 0 ? item_first / KB : 0;
    const int wave_first = WINDOW ? pos0 + q0 - p.window + 1 : 0;

    Vec8<T> qf[QB][NQ];
    floatx4 o[QB][NV], l[QB];
    float m[QB];
    int qpos[QB];
#pragma unroll
    for (int b = 0; b < QB; ++b) {
        const int qi = q0 + 16 * b + ql;
        qpos[b] = pos0 + qi;
        const T *row = p.q + (size_t)(qi < p.M ? qi : p.M - 1) * p.ldq + (WINDOW ? kvh * p.group_q + (head - kvh * p.group) * p.head_q : (size_t)head * qd) + 8 * g;
#pragma unroll
        for (int ks = 0; ks < NQ; ++ks)
            if (EXACT || ks < nq) qf[b][ks] = load8(row + 32 * ks);
#pragma unroll
        for (int d = 0; d < NV; ++d) o[b][d] = floatx4{0.f, 0.f, 0.f, 0.f};
        l[b] = floatx4{0.f, 0.f, 0.f, 0.f};
        m[b] = kNoMax;
    }

    // the queries have arrived before the first block is asked for: with these loads possibly in flight the compiler waits for everything asked for since,
    // the next block included, in front of the first product of every block
    if constexpr (EXACT) __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)

    // a chunk is 8 elements of a row; the first dim of a K row come from the expanded matrix, the rest from the cache
    const T *k_base = p.kv + kvh * p.head_k, *v_base = p.kv + p.v_off + kvh * p.head_v + vcol0, *r_base = p.cache + p.rot_off;
    auto row_of = [&](int kb, int i) {   // row of key kb + i of a block (a ring holds whole blocks)
        if constexpr (WINDOW) return kb % p.ring + (kb + i < p.total ? i : p.total - 1 - kb);
        const int key = kb + i;
        return key < p.total ? key : p.total - 1;
    };
    auto at = [&](const T *base, int row, long ld, int e) -> Vec8<T> {
        if constexpr (EXACT) return load8(reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + (uint32_t)(row * (uint32_t)ld + e) * (uint32_t)sizeof(T)));
        return load8(base + (size_t)row * ld + e);
    };
    auto k_chunk = [&](int kb, int c, int cpr) -> Vec8<T> {
        const int row = row_of(kb, c / cpr), e = 8 * (c % cpr);
        return WINDOW || e < p.dim ? at(k_base, row, p.ldkv, e) : at(r_base, row, p.ldc, e - p.dim);
    };
    auto v_chunk = [&](int kb, int c, int cpr) -> Vec8<T> {
        return at(v_base, row_of(kb, c / cpr), p.ldkv, 8 * (c % cpr));
    };
    constexpr int CK = 4 * NQ, CV = 2 * NV;                       // chunks per row (EXACT)
    constexpr int NCK = EXACT ? KB * CK / kSetThreads : 1, NCV = EXACT ? KB * CV / kSetThreads : 1;
    static_assert(!EXACT || (KB * CK % kSetThreads == 0 && KB * CV % kSetThreads == 0), "whole chunks per thread");
    Vec8<T> kreg[NCK], vreg[NCV];
    auto fetch = [&](int it) {
        if constexpr (EXACT) {
#pragma unroll
            for (int i = 0; i < NCK; ++i) kreg[i] = k_chunk(it * KB, tid + kSetThreads * i, CK);
#pragma unroll
            for (int i = 0; i < NCV; ++i) vreg[i] = v_chunk(it * KB, tid + kSetThreads * i, CV);
        }
    };
    auto stage = [&](int it) {
        if constexpr (EXACT) {
#pragma unroll
            for (int i = 0; i < NCK; ++i) {
                const int c = tid + kSetThreads * i;
                store8(kt + (c / CK) * kp + 8 * (c % CK), kreg[i]);
            }
#pragma unroll
            for (int i = 0; i < NCV; ++i) {
                const int c = tid + kSetThreads * i;
                store8(vt + (c / CV) * vp + 8 * (c % CV), vreg[i]);
            }
        } else {
            const int ck = qd / 8, cv = vd / 8;
            for (int c = tid; c < KB * ck; c += kSetThreads) store8(kt + (c / ck) * kp + 8 * (c % ck), k_chunk(it * KB, c, ck));
            for (int c = tid; c < KB * cv; c += kSetThreads) store8(vt + (c / cv) * vp + 8 * (c % cv), v_chunk(it * KB, c, cv));
        }
    };

    if (first + set < blocks) fetch(first + set);
    for (int it0 = first; it0 < blocks; it0 += SETS) {
        const int it = it0 + set, kb = it * KB;
        if (it < blocks) stage(it);
        __syncthreads();
        if (it + SETS < blocks) fetch(it + SETS);
        if (it < blocks && kb <= wave_last && (!WINDOW || kb + KB > wave_first)) {
            floatx4 s[NKK][QB];
            if constexpr (EXACT) {   // kAhead operands are on their way from LDS (left to itself the compiler asks for one, waits, multiplies)
                constexpr int N = NKK * NQ, kAhead = 4;
                Vec8<T> a[kAhead];
#pragma unroll
                for (int kk = 0; kk < NKK; ++kk)
#pragma unroll
                    for (int b = 0; b < QB; ++b) s[kk][b] = floatx4{0.f, 0.f, 0.f, 0.f};
                auto ask = [&](int n) { a[n % kAhead] = load8(kt + (16 * (n / NQ) + ql) * kp + 32 * (n % NQ) + 8 * g); };
#pragma unroll
                for (int n = 0; n < kAhead; ++n) ask(n);
#pragma unroll
                for (int n = 0; n < N; ++n) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int b = 0; b < QB; ++b) s[n / NQ][b] = mma32(a[n % kAhead], qf[b][n % NQ], s[n / NQ][b]);
                    if (n + kAhead < N) ask(n + kAhead);
                }
                __builtin_amdgcn_sched_barrier(0);
            } else {
#pragma unroll
                for (int kk = 0; kk < NKK; ++kk) {
#pragma unroll
                    for (int b = 0; b < QB; ++b) s[kk][b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int ks = 0; ks < NQ; ++ks)
                        if (ks < nq) {
                            const Vec8<T> a = load8(kt + (16 * kk + ql) * kp + 32 * ks + 8 * g);
#pragma unroll
                            for (int b = 0; b < QB; ++b) s[kk][b] = mma32(a, qf[b][ks], s[kk][b]);
                        }
                }
            }
            // s[kk][b][r]: key kb + 16 kk + 4 g + r against query qpos[b]
            const bool masked = kb + KB - 1 > pos0 + q0;
            float bm[QB];
            bool lag = false;
#pragma unroll
            for (int b = 0; b < QB; ++b) {
                if (masked) {
                    int last = qpos[b] - kb - 4 * g;   // (in here: in front of the products it would take registers)
                    if constexpr (EXACT) asm volatile("" : "+v"(last));
#pragma unroll
                    for (int kk = 0; kk < NKK; ++kk)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (16 * kk + r > last) s[kk][b][r] = kMasked;
                }
                if (WINDOW && kb <= wave_last - p.window) {
                    int hidden = qpos[b] - p.window - kb - 4 * g;
                    if constexpr (EXACT) asm volatile("" : "+v"(hidden));
#pragma unroll
                    for (int kk = 0; kk < NKK; ++kk)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (16 * kk + r <= hidden) s[kk][b][r] = kMasked;
                }
                float v = kMasked;
#pragma unroll
                for (int kk = 0; kk < NKK; ++kk) {
                    v = fmaxf(fmaxf(v, s[kk][b][0]), s[kk][b][1]);
                    v = fmaxf(fmaxf(v, s[kk][b][2]), s[kk][b][3]);
                }
                bm[b] = max_over_lane_groups(v);
                lag = lag || (bm[b] - m[b]) * p.scale_log2 > kLazy;
            }
            if (__builtin_amdgcn_ballot_w64(lag) != 0) {   // (always at a query's first visible key)
#pragma unroll
                for (int b = 0; b < QB; ++b) {
                    const float mn = fmaxf(m[b], bm[b]);
                    const float alpha = __builtin_amdgcn_exp2f((m[b] - mn) * p.scale_log2);
                    m[b] = mn;
                    l[b] *= alpha;
#pragma unroll
                    for (int d = 0; d < NV; ++d) o[b][d] *= alpha;
                }
            }
            Vec8<T> pb[QB][NT];
#pragma unroll
            for (int b = 0; b < QB; ++b) {
                const float msc = m[b] * p.scale_log2;
#pragma unroll
                for (int kk = 0; kk < NKK; ++kk)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[kk][b][r] = __builtin_amdgcn_exp2f(fmaf(s[kk][b][r], p.scale_log2, -msc));
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    pb[b][t] = pair8<T>(s[2 * t][b], s[2 * t + 1][b]);
                    l[b] = mma32(ones8<T>(), pb[b][t], l[b]);
                }
            }
            if constexpr (EXACT) {
                constexpr int N = NT * NV, kAhead = 4;
                Vec8<T> a[kAhead];
                auto ask = [&](int n) { a[n % kAhead] = column8(vt + 32 * (n / NV) * vp, vp, 16 * (n % NV)); };
#pragma unroll
                for (int n = 0; n < kAhead; ++n) ask(n);
#pragma unroll
                for (int n = 0; n < N; ++n) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int b = 0; b < QB; ++b) o[b][n % NV] = mma32(a[n % kAhead], pb[b][n / NV], o[b][n % NV]);
                    if (n + kAhead < N) ask(n + kAhead);
                }
                __builtin_amdgcn_sched_barrier(0);
            } else
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int d = 0; d < NV; ++d)
                    if (d < nv) {
                        const Vec8<T> a = column8(vt + 32 * t * vp, vp, 16 * d);
#pragma unroll
                        for (int b = 0; b < QB; ++b) o[b][d] = mma32(a, pb[b][t], o[b][d]);
                    }
        }
        __syncthreads();
    }

    // The same wave and lane of the other set holds the same queries and output elements.  Where there are gates each set finishes one block
    // of queries, so that both work on them; without, the exchange both ways costs more than it shares (4 heads of 64 over 2, 2048 tokens 15.3 -> 15.6 us).
    constexpr bool kShare = SETS == 2 && QB == 2 && !WINDOW;
    if constexpr (SETS == 2) {
        constexpr int NREG = (kShare ? 1 : QB) * (4 * NV + 2);
        float *mine = reinterpret_cast<float *>(pf_lds) + (wave + (kShare ? 4 * set : 0)) * NREG * 64 + lane;   // what this wave takes
        float *other = reinterpret_cast<float *>(pf_lds) + (wave + (kShare ? 4 * (set ^ 1) : 0)) * NREG * 64 + lane;
        auto give = [&](int b, float *to) {
#pragma unroll
            for (int d = 0; d < NV; ++d)
#pragma unroll
                for (int r = 0; r < 4; ++r) to[(d * 4 + r) * 64] = o[b][d][r];
            to[4 * NV * 64] = m[b];
            to[(4 * NV + 1) * 64] = l[b][0];
        };
        // (own: this wave's part counts as set b's of block b.  Written out, so that a query's result does not depend on who adds the parts up.)
        auto take = [&](int b, const float *from, auto own) {
            const float m1 = from[4 * NV * 64], l1 = from[(4 * NV + 1) * 64];
            const float mm = fmaxf(m[b], m1);
            const float f0 = __builtin_amdgcn_exp2f((m[b] - mm) * p.scale_log2), f1 = __builtin_amdgcn_exp2f((m1 - mm) * p.scale_log2);
            auto sum = [&](float mine, float got, bool first) { return first ? fmaf(mine, f0, got * f1) : fmaf(got, f1, mine * f0); };
            m[b] = mm;
            l[b][0] = sum(l[b][0], l1, !own);
#pragma unroll
            for (int d = 0; d < NV; ++d)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[b][d][r] = sum(o[b][d][r], from[(d * 4 + r) * 64], own);
        };
        if constexpr (kShare) {
            if (set == 0) give(1, other);
            else give(0, other);
            __syncthreads();
            if (set == 0) take(0, mine, std::true_type());
            else take(1, mine, std::true_type());
        } else {
            if (set == 1) {
#pragma unroll
                for (int b = 0; b < QB; ++b) give(b, other + b * (4 * NV + 2) * 64);
            }
            __syncthreads();
            if (set == 1) return;
            take(0, mine, std::true_type());
            if constexpr (QB == 2) take(1, mine + (4 * NV + 2) * 64, std::false_type());
        }
    }

    const float snk = WINDOW ? 0.f : p.sink[head] * 1.4426950408889634f;
    auto finish = [&](int b) {
        const int qi = q0 + 16 * b + ql;
        if (qi >= p.M) return;
        const float inv = WINDOW ? p.out_scale / l[b][0] : 1.0f / (l[b][0] + exp2f(snk - m[b] * p.scale_log2));
        const int col = head * p.vdim + vcol0 + 4 * g;
        const T *gate = p.q + (size_t)qi * p.ldq + p.gate_off + col;
        T *dst = p.out + (size_t)qi * p.ldo + col;
        float z[WINDOW ? 1 : NV][4];
        if constexpr (!WINDOW) {   // all of them on their way before the first is used
#pragma unroll
            for (int d = 0; d < NV; ++d)
                if (EXACT || d < nv) load4(gate + 16 * d, z[d]);
        }
#pragma unroll
        for (int d = 0; d < NV; ++d)
            if (EXACT || d < nv) {
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    v[r] = o[b][d][r] * inv;
                    if constexpr (!WINDOW) v[r] = sizeof(T) == 2 ? gated(v[r], z[d][r]) : v[r] * sigmoid_f32(z[d][r]);
                }
                store4(dst + 16 * d, v[0], v[1], v[2], v[3]);
            }
    };
    if constexpr (kShare) {
        if (set == 0) finish(0);
        else finish(1);
    } else {
#pragma unroll
        for (int b = 0; b < QB; ++b) finish(b);
    }
}

constexpr size_t kLdsLimit = 160 * 1024;

template <class T, int NQ, int NV, int QB, int KB, int SETS, bool EXACT, bool WINDOW = false>
hipError_t launch(const PrefillArgs<T> &p, hipStream_t stream) {
    const int vd = p.vdim < 16 * NV ? p.vdim : 16 * NV;
    size_t lds = (size_t)SETS * KB * ((p.dim + p.rot + 16 / sizeof(T)) + (vd + 32 / sizeof(T))) * sizeof(T);
    const size_t exchange = SETS == 2 ? 4 * QB * (4 * NV + 2) * 64 * sizeof(float) : 0;
    if (lds < exchange) lds = exchange;
    if (lds > kLdsLimit) return hipErrorInvalidValue;
    auto kernel = &latent_prefill_kernel<T, NQ, NV, QB, KB, SETS, EXACT, WINDOW>;
    if (lds > 48 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const int items = (p.M + 64 * QB - 1) / (64 * QB);
    hipLaunchKernelGGL(kernel, dim3(p.heads, items, (p.vdim + 16 * NV - 1) / (16 * NV)), dim3(SETS * kSetThreads), lds, stream, p);
    return hipGetLastError();
}

template <class T>
PrefillArgs<T> args_of(const LatentShape &s, const LatentRows &r, const void *kv, long ldkv, const float *sink, void *out, long ldo) {
    PrefillArgs<T> p{};
    p.q = static_cast<const T *>(r.proj);
    p.kv = static_cast<const T *>(kv);
    p.cache = static_cast<const T *>(r.cache);
    p.out = static_cast<T *>(out);
    p.ldq = r.ld;
    p.ldkv = ldkv;
    p.ldo = ldo;
    p.ldc = s.rank + s.rot;
    p.rot_off = s.rank;
    p.heads = s.heads;
    p.dim = s.dim;
    p.rot = s.rot;
    p.vdim = s.vdim;
    p.v_off = s.heads * s.dim;
    p.gate_off = r.gate_off;
    p.M = r.M;
    p.total = r.pos + r.M;
    p.scale_log2 = s.scale * 1.4426950408889634f;
    p.sink = sink;
    p.head_k = s.dim;
    p.head_v = s.vdim;
    return p;
}

template <class T>
PrefillArgs<T> args_of(const HeadShape &s, const HeadRows &r, const void *q, void *out, long ldo) {
    PrefillArgs<T> p{};
    p.q = static_cast<const T *>(q);
    p.kv = p.cache = static_cast<const T *>(r.cache);
    p.out = static_cast<T *>(out);
    p.group = s.heads / s.kv_heads;
    p.ldq = (long)p.group * s.dim;
    p.head_q = s.dim;
    p.group_q = (long)r.M * p.ldq;
    p.ldkv = s.dim + s.vdim;
    p.ldo = ldo;
    p.heads = s.heads;
    p.dim = s.dim;
    p.vdim = s.vdim;
    p.v_off = s.dim;
    p.head_k = p.head_v = (long)s.ring * p.ldkv;
    p.window = s.window;
    p.ring = s.ring;
    p.M = r.M;
    p.total = r.pos + r.M;
    p.scale_log2 = s.scale * 1.4426950408889634f;
    p.out_scale = s.out_scale;
    return p;
}

// Whether a workgroup takes 64 queries, 16 to a wave, instead of 128, for heads of 128 + 64 / 128 and of 128 / 128 behind long windows.  A block of 64 keys takes a wave set 2.6 us
// with 16 queries to a wave and 2.8 with 32 (staging, scores, softmax and outputs are a chain between two barriers, a workgroup has its CU to itself), so of 64 queries the longest
// item is done sooner, and launches of several items to a CU take 1.35 times as long.  The line: 256 CUs get all items done in the time of the longest.  us, 128 / 64 queries, 16 heads of
// 128 + 64 / 128: 128 tokens 13.3 / 9.2, 1000 31.6 / 24.9, 1500 43.2 / 35.2, 1800 50.2 / 45.6, 3000 80.2 / 108.8; 8 heads 3000 73.6 / 62.6; 32 heads 700 25.1 / 20.7, 1000 33.8 / 32.6, 2048
// 74.0 / 99.4.  Just past it 64 would still be faster alone (16 heads and 2048 tokens, 3 % more blocks than that, 56.0 / 52.8): the line is not fitted there.
template <class T>
long item_blocks(const PrefillArgs<T> &p, long first, long queries = 64) {   // blocks of 64 keys of the item of so many queries from position `first` on
    const long end = std::min<long>(first + queries, p.total), unseen = p.window > 0 && first >= p.window ? (first - p.window + 1) / 64 : 0;
    return (end + 63) / 64 - unseen;
}
template <class T>
bool few_queries(const PrefillArgs<T> &p) {
    long longest = 0, all = 0;
    for (long first = p.total - p.M; first < p.total; first += 64) {
        const long blocks = item_blocks(p, first);
        longest = std::max(longest, blocks);
        all += blocks;
    }
    return all * p.heads <= 256 * longest;
}

// Whether windowed heads that otherwise take 64 queries to a workgroup take 128 after all: 512 items of 64 or fewer, two to a CU, of which more than 256 are nearly as long as the
// longest.  Two long ones on a CU take 1.02 us a block of keys together, one alone 0.76, an item of 128 queries 0.93 (heads of 64); where lengths differ a long one shares with short ones.
// us, 128 / 64 queries, heads of 64: 8, window 2048, 4096 tokens 32.0 / 35.0, window 1024 19.8 / 21.4; heads of 128 (windows up to 768): 16 of them, 2048 tokens, window 640 23.2 / 25.1,
// but 4096 tokens 46.8 / 45.6.  The two wave sets of 128 queries take blocks in turn, so an odd number costs them one more.
template <class T>
bool even_round(const PrefillArgs<T> &p, bool wide) {
    const long items = (p.M + 63) / 64 * (long)p.heads, start = p.total - p.M;
    if (items <= 256 || items > 512) return false;
    long longest = 0, tall = 0, longest128 = 0;
    for (long first = start; first < p.total; first += 64) longest = std::max(longest, item_blocks(p, first));
    for (long first = start; first < p.total; first += 64) tall += 10 * item_blocks(p, first) >= 9 * longest;
    for (long first = start; first < p.total; first += 128) longest128 = std::max(longest128, item_blocks(p, first, 128));
    return tall * p.heads > 256 && (wide ? longest >= 10 && longest128 % 2 == 0 : longest >= 17);
}

}  // namespace

bool latent_prefill_supported(int dtype, const LatentShape &s) {
    (void)dtype;
    return s.dim + s.rot <= 512;
}

hipError_t launch_latent_prefill(int dtype, const LatentShape &s, const LatentRows &r, const void *kv, long ldkv, const float *sink, void *out,
                                 long ldo, hipStream_t stream) {
    const int nq = (s.dim + s.rot) / 32, nv = s.vdim / 16;
    if (dtype == kF32) {
        const PrefillArgs<float> p = args_of<float>(s, r, kv, ldkv, sink, out, ldo);
        if (nq <= 4 && nv <= 4) return launch<float, 4, 4, 1, 32, 1, false>(p, stream);
        if (nq <= 8 && nv <= 8) return launch<float, 8, 8, 1, 32, 1, false>(p, stream);
        return launch<float, 16, 16, 1, 32, 1, false>(p, stream);
    }
    const PrefillArgs<bf16> p = args_of<bf16>(s, r, kv, ldkv, sink, out, ldo);
    if ((double)p.total * ldkv * sizeof(bf16) < 4e9) {
        if (nq == 6 && nv == 8) return few_queries(p) ? launch<bf16, 6, 8, 1, 32, 2, true>(p, stream) : launch<bf16, 6, 8, 2, 64, 2, true>(p, stream);
        // (two workgroups to a CU: 4 to 64 heads, 128 to 4096 tokens 1.0 to 1.4 times as fast as with 128 queries)
        if (nq == 4 && nv == 4) return launch<bf16, 4, 4, 1, 64, 2, true>(p, stream);
        if (nq == 3 && nv == 4) return launch<bf16, 3, 4, 1, 64, 2, true>(p, stream);
    }
    if (nq <= 4 && nv <= 4) return launch<bf16, 4, 4, 1, 64, 1, false>(p, stream);
    if (nq <= 8 && nv <= 8) return launch<bf16, 8, 8, 1, 64, 1, false>(p, stream);
    return launch<bf16, 16, 16, 1, 32, 1, false>(p, stream);
}

bool head_prefill_supported(int dtype, const HeadShape &s) {
    (void)dtype;
    return s.dim <= 512;
}

hipError_t launch_head_prefill(int dtype, const HeadShape &s, const HeadRows &r, const void *q, void *out, long ldo, hipStream_t stream) {
    const int nq = s.dim / 32, nv = s.vdim / 16;
    if (dtype == kF32) {
        const PrefillArgs<float> p = args_of<float>(s, r, q, out, ldo);
        if (nq <= 4 && nv <= 4) return launch<float, 4, 4, 1, 32, 1, false, true>(p, stream);
        if (nq <= 8 && nv <= 8) return launch<float, 8, 8, 1, 32, 1, false, true>(p, stream);
        return launch<float, 16, 16, 1, 32, 1, false, true>(p, stream);
    }
    const PrefillArgs<bf16> p = args_of<bf16>(s, r, q, out, ldo);
    if ((double)s.ring * (s.dim + s.vdim) * sizeof(bf16) < 4e9) {
        // (128 / 64, also behind 96 + 32 / 64 above: bounds were asked at every operand.  16 heads, 2048 tokens, window 1024 74 -> 25.5 us, 300 30 -> 13.8; 96 + 32 / 64, 16 heads, 2048
        // tokens 141 -> 34.2, 1000 71.5 -> 16.6.  By 128 queries 24.6, 14.6, 39.0, 22.0; blocks of 32 keys 0 to 4 % slower.)
        // (windows of few blocks are mostly start and end, which the smaller items share a CU for: 16 to 64 heads, 1024 to 4096 tokens, windows of 64 to 256 1.03 to 1.4 times
        // as fast, of 384 to 700 0.99 to 1.3)
        if (nq == 4 && nv == 8)
            return (p.window <= 768 && !even_round(p, true)) || few_queries(p) ? launch<bf16, 4, 8, 1, 32, 2, true, true>(p, stream) : launch<bf16, 4, 8, 2, 64, 2, true, true>(p, stream);
        if (nq == 4 && nv == 4) return launch<bf16, 4, 4, 1, 64, 2, true, true>(p, stream);
        if (nq == 2 && nv == 4) return even_round(p, false) ? launch<bf16, 2, 4, 2, 64, 2, true, true>(p, stream) : launch<bf16, 2, 4, 1, 32, 2, true, true>(p, stream);
    }
    if (nq <= 4 && nv <= 4) return launch<bf16, 4, 4, 1, 64, 1, false, true>(p, stream);
    if (nq <= 8 && nv <= 8) return launch<bf16, 8, 8, 1, 64, 1, false, true>(p, stream);
    return launch<bf16, 16, 16, 1, 32, 1, false, true>(p, stream);
}

}  // namespace w4a16
