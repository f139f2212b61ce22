// Single-query (decode) GQA attention over a bf16 KV cache, with the half-split RoPE of the new
// token's Q and K and the cache append fused in.
//
// Input is the fresh, un-rotated projection vector qkv = [Q (n_heads * HD) | K (n_kv * HD) |
// V (n_kv * HD)] of the current token.  HBM-bound on the cache: every cached K and V element is
// read by the workgroups of its (kv head, sequence chunk), as few or as many as there is room for
// (launch_decode_attention), and used for the G query heads that each has.
//
//   grid  = (nsplit sequence chunks, n_kv heads x groups of G of their query heads), 4 waves per workgroup
//   lanes = HD / 8 lanes share one cache position (16-byte loads), so a wave covers 64 / (HD / 8)
//           positions per load; each lane group keeps a private online-softmax state
//           (m, l, acc[8]) per query head and the states are merged at the end: across lane
//           groups with shuffles, across waves through LDS, across chunks by the combine kernel
//   the chunk that holds `pos` rotates K, takes the new token's K and V from registers and stores
//   them into the caches at its end, once per KV head
//
// Rounding points follow the reference's decode step: Q and K are rounded to bf16 after RoPE,
// scores, softmax and the weighted sum are fp32, the output is rounded to bf16 once.
#include "common.h"
#include "kernels.h"

namespace w4a16 {

namespace {

constexpr float kNegBig = kAttnNegBig;
constexpr float kLog2e = 1.4426950408889634f;

struct AttnParams {
    const uint16_t *qkv;
    const uint16_t *lut;      // [HD]: cos[0..HD/2), sin[0..HD/2) at position pos
    uint16_t *k_cache;        // [n_kv, max_seq, HD]
    uint16_t *v_cache;
    uint16_t *out;            // [n_heads * HD]
    float *part_ml;           // [n_heads, nsplit, 2]
    float *part_acc;          // [n_heads, nsplit, HD]
    int pos, max_seq, n_heads, n_kv, nsplit, chunk;
    int log2_sharers;         // of the workgroups that have query heads of one KV head
    float scale;
};

__device__ __forceinline__ void unpack8(const u32x4 v, float (&f)[8]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        f[2 * j] = __builtin_bit_cast(float, v[j] << 16);
        f[2 * j + 1] = __builtin_bit_cast(float, v[j] & 0xFFFF0000u);
    }
}

// 2^x for x <= 0 as the bare v_exp_f32: the library routine's rescaling of very negative arguments only
// changes results below 2^-126, which vanish against the running sums they are added to.
__device__ __forceinline__ float exp2_nonpos(float x) { return __builtin_amdgcn_exp2f(x); }

// Sum over a group of LPP = 8 or 16 neighbouring lanes (a group never crosses a row of 16 lanes), every lane
// of the group receiving the sum: an xor butterfly on data-parallel-primitive moves (quad permutes for
// distances 1 and 2, half-row and row mirrors for 4 and 8: once the quads agree, mirroring meets the
// partner quad), i.e. full-rate VALU adds instead of LDS-routed shuffles.  Bit-identical to the butterfly
// with shuffles: every step adds the same two partial sums.
template <int LPP>
__device__ __forceinline__ float group_sum(float s) {
    static_assert(LPP == 8 || LPP == 16, "lane groups of 8 or 16");
    s = dpp_add<0xB1>(s);    // quad_perm [1, 0, 3, 2]
    s = dpp_add<0x4E>(s);    // quad_perm [2, 3, 0, 1]
    s = dpp_add<0x141>(s);   // row_half_mirror
    if constexpr (LPP == 16) s = dpp_add<0x140>(s);   // row_mirror
    return s;
}

// Half-split RoPE of the eight elements x of one head's half, y the same places of the other half, rounded to bf16 (returned as floats).
__device__ __forceinline__ void rope8(const u32x4 xr, const u32x4 yr, const float (&c)[8], const float (&s)[8], bool low, float (&out)[8]) {
    float x[8], y[8];
    unpack8(xr, x);
    unpack8(yr, y);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        // low half: x1 cos - x2 sin; high half: x2 cos + x1 sin (x is the lane's own element)
        const float r = low ? x[j] * c[j] - y[j] * s[j] : x[j] * c[j] + y[j] * s[j];
        out[j] = bf16_bits_to_float(float_to_bf16_bits(r));
    }
}

// Over the lanes with equal `sub` (one per position), every one of them receiving the result.
template <int LPP, bool MAX>
__device__ __forceinline__ float slots_reduce(float v) {
    if constexpr (LPP == 8) {
        const float o = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xF, 0xF, true));   // row_ror:8
        v = MAX ? fmaxf(v, o) : v + o;
    }
    v = swap_reduce<16, MAX>(v, v);
    return swap_reduce<32, MAX>(v, v);
}

// What bounds it: latencies in a row, at 64 positions a workgroup: the fresh qkv and the cache (requested together, qkv first, so that it is rotated
// while the cache is on its way; the new token's K and V are taken from registers, not read back), the scores' sums, one maximum per wave and head,
// and the sums over positions.  Those halve
// what a lane holds with every exchange (v_permlane*_swap: half the values go each way), 28 exchanges for a head group of 4, where full
// butterflies of (m, l, acc) took 120 shuffles through LDS.   32 heads of 64 over 8, 1000 positions: 7.3 -> 4.9 us; -> 4.5 a layer of
// the model since the new token's row and the queries are no longer asked for one after the other behind the cache.  Only the chunk that appends
// the new K and V asks for them: with all chunks, merge included, 32 heads of 64 over 8 at 4000 positions 7.5 us, 32 heads of 128 at 2000 8.6; 7.2 and 7.8.
template <int HD, int G, int UN>
__global__ void __launch_bounds__(256) attn_partial_kernel(const AttnParams p) {
    constexpr int LPP = HD / 8;        // lanes per position
    constexpr int PPW = 64 / LPP;      // positions per wave and load
    constexpr int STATE = 4 + HD;      // m, l, -, -, acc[HD] per head
    constexpr int STEP = UN * 4 * PPW;   // positions per lane and trip, per workgroup and trip
    __shared__ __attribute__((aligned(16))) float sh[4 * G * STATE];

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int sub = lane % LPP, slot = lane / LPP;
    const int split = blockIdx.x, kvh = blockIdx.y >> p.log2_sharers, head0 = blockIdx.y * G;
    const int seq_len = p.pos + 1;
    const int t0 = split * p.chunk;
    const int t1 = min(seq_len, t0 + p.chunk);
    const int nq = p.n_heads * HD, nkv = p.n_kv * HD;

    uint16_t *kc = p.k_cache + (size_t)kvh * p.max_seq * HD + 8 * sub;
    uint16_t *vc = p.v_cache + (size_t)kvh * p.max_seq * HD + 8 * sub;

    // rotation and this lane's slices of qkv; of the new K and V where the chunk that holds `pos` appends them
    const bool low = 8 * sub < HD / 2;
    const int other = low ? 8 * sub + HD / 2 : 8 * sub - HD / 2, turn = low ? 8 * sub : other;
    auto raw = [](const uint16_t *at) { return *reinterpret_cast<const u32x4 *>(at); };
    const u32x4 cos_raw = raw(p.lut + turn), sin_raw = raw(p.lut + HD / 2 + turn);
    u32x4 qx[G], qy[G];
#pragma unroll
    for (int h = 0; h < G; ++h) {
        const uint16_t *src = p.qkv + (size_t)(head0 + h) * HD;
        qx[h] = raw(src + 8 * sub);
        qy[h] = raw(src + other);
    }
    const uint16_t *k_row = p.qkv + nq + kvh * HD;
    const bool owner = t0 <= p.pos && p.pos < t1;
    u32x4 kx, ky, knew, vnew;
    if (owner) kx = raw(k_row + 8 * sub), ky = raw(k_row + other), vnew = raw(k_row + nkv + 8 * sub);

    u32x4 kraw[UN], vraw[UN];
    auto request = [&](int tb) {
#pragma unroll
        for (int i = 0; i < UN; ++i) {
            const int t = tb + i * 4 * PPW;
            const size_t at = (size_t)min(t, t1 - 1) * HD;   // in range (t1 >= 1, also where the chunk is empty); a clamped slot's result is discarded
            kraw[i] = *reinterpret_cast<const u32x4 *>(kc + at);
            vraw[i] = *reinterpret_cast<const u32x4 *>(vc + at);
        }
    };
    int tb = t0 + wave * PPW + slot;
    request(tb);

    __builtin_amdgcn_sched_barrier(0);
    float cos[8], sin[8];
    unpack8(cos_raw, cos);
    unpack8(sin_raw, sin);
    if (owner) {
        float kr[8];
        rope8(kx, ky, cos, sin, low, kr);
#pragma unroll
        for (int j = 0; j < 4; ++j) knew[j] = pack_bf16x2(kr[2 * j], kr[2 * j + 1]);
    }
    // rotated, bf16-rounded query slices of the G heads, pre-scaled for exp2
    float q[G][8];
#pragma unroll
    for (int h = 0; h < G; ++h) {
        rope8(qx[h], qy[h], cos, sin, low, q[h]);
#pragma unroll
        for (int j = 0; j < 8; ++j) q[h][j] *= p.scale * kLog2e;
    }

    float m[G], l[G], acc[G * 8];   // m of the wave; l and acc of the lane's positions
#pragma unroll
    for (int h = 0; h < G; ++h) m[h] = kNegBig, l[h] = 0.f;
#pragma unroll
    for (int n = 0; n < G * 8; ++n) acc[n] = 0.f;

    for (int base = t0; base < t1; base += STEP, tb += STEP) {   // (the same number of trips for every lane)
        float s[UN][G], v[UN][8];
        bool live[UN];
#pragma unroll
        for (int i = 0; i < UN; ++i) {
            const int t = tb + i * 4 * PPW;
            live[i] = t < t1;
            float k[8];
            const bool fresh = owner && t == p.pos;
            unpack8(fresh ? knew : kraw[i], k);
            unpack8(fresh ? vnew : vraw[i], v[i]);
#pragma unroll
            for (int h = 0; h < G; ++h) {
                float d = 0.f;
#pragma unroll
                for (int j = 0; j < 8; ++j) d = fmaf(q[h][j], k[j], d);
                s[i][h] = group_sum<LPP>(d);
            }
        }
        if (base + STEP < t1) request(tb + STEP);
#pragma unroll
        for (int h = 0; h < G; ++h) {
            float mn = m[h];
#pragma unroll
            for (int i = 0; i < UN; ++i) mn = fmaxf(mn, live[i] ? s[i][h] : kNegBig);
            mn = slots_reduce<LPP, true>(mn);
            const float corr = exp2_nonpos(m[h] - mn);
            m[h] = mn;
            l[h] *= corr;
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[8 * h + j] *= corr;
#pragma unroll
            for (int i = 0; i < UN; ++i) {
                const float pr = live[i] ? exp2_nonpos(s[i][h] - mn) : 0.f;
                l[h] += pr;
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[8 * h + j] = fmaf(pr, live[i] ? v[i][j] : 0.f, acc[8 * h + j]);
            }
        }
    }

    if (owner && blockIdx.y == kvh << p.log2_sharers && threadIdx.x < LPP) {   // (behind the loop: no wait in it counts stores)
        *reinterpret_cast<u32x4 *>(kc + (size_t)p.pos * HD) = knew;
        *reinterpret_cast<u32x4 *>(vc + (size_t)p.pos * HD) = vnew;
    }

    // sums over the wave's positions: lanes 32 .. 63 go on with the upper half of the values, odd rows of lanes with the upper half of theirs
    constexpr int NV = G * 8, QV = NV / 4;
#pragma unroll
    for (int n = 0; n < NV / 2; ++n) acc[n] = swap_reduce<32, false>(acc[n], acc[n + NV / 2]);
#pragma unroll
    for (int n = 0; n < QV; ++n) acc[n] = swap_reduce<16, false>(acc[n], acc[n + QV]);
    if constexpr (LPP == 8) {
#pragma unroll
        for (int n = 0; n < QV; ++n) acc[n] = dpp_add<0x128>(acc[n]);
    }
#pragma unroll
    for (int h = 0; h < G; ++h) l[h] = slots_reduce<LPP, false>(l[h]);
    if (LPP == 16 || !(lane & 8)) {
        const int first = (lane & 32 ? NV / 2 : 0) + (lane & 16 ? QV : 0);
#pragma unroll
        for (int n = 0; n < QV; ++n) sh[(wave * G + (first + n) / 8) * STATE + 4 + 8 * sub + (first + n) % 8] = acc[n];
    }
    if (lane == 0) {
#pragma unroll
        for (int h = 0; h < G; ++h) {
            sh[(wave * G + h) * STATE] = m[h];
            sh[(wave * G + h) * STATE + 1] = l[h];
        }
    }
    __syncthreads();

    // merge the four waves; one thread per (head, element)
    for (int idx = threadIdx.x; idx < G * HD; idx += 256) {
        const int h = idx / HD, e = idx % HD;
        float mn = kNegBig;
#pragma unroll
        for (int w = 0; w < 4; ++w) mn = fmaxf(mn, sh[(w * G + h) * STATE]);
        float ls = 0.f, as = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float *src = sh + (w * G + h) * STATE;
            const float c = exp2f(src[0] - mn);
            ls += src[1] * c;
            as += src[4 + e] * c;
        }
        const int head = head0 + h;
        if (p.nsplit == 1) {
            p.out[(size_t)head * HD + e] = float_to_bf16_bits(as / ls);
        } else {
            const size_t slot_idx = (size_t)head * p.nsplit + split;
            if (e == 0) {
                p.part_ml[2 * slot_idx] = mn;
                p.part_ml[2 * slot_idx + 1] = ls;
            }
            p.part_acc[slot_idx * HD + e] = as;
        }
    }
}

// out[head] = sum_s acc_s 2^(m_s - M) / sum_s l_s 2^(m_s - M); grid = n_heads, block = HD threads.
// The chunk weights are computed once by the first wave (lane s owns chunk s, nsplit <= 32).
__global__ void attn_combine_kernel(const float *part_ml, const float *part_acc, uint16_t *out, int nsplit, int hd) {
    __shared__ float wgt[kMaxAttnSplit];
    __shared__ float inv_l;
    const int head = blockIdx.x, e = threadIdx.x;
    // every load of the kernel is requested up front: one memory round trip in total
    const float *src = part_acc + (size_t)head * nsplit * hd + e;
    float a[kMaxAttnSplit];
#pragma unroll
    for (int s = 0; s < kMaxAttnSplit; ++s) a[s] = s < nsplit ? src[(size_t)s * hd] : 0.f;
    if (e < 64) {
        const bool live = e < nsplit;
        const float m = live ? part_ml[2 * ((size_t)head * nsplit + e)] : kNegBig;
        const float l = live ? part_ml[2 * ((size_t)head * nsplit + e) + 1] : 0.f;
        const float mn = wave_reduce<true>(m);
        const float c = exp2f(m - mn);
        const float ls = wave_reduce<false>(l * c);
        if (e < kMaxAttnSplit) wgt[e] = live ? c : 0.f;
        if (e == 0) inv_l = 1.0f / ls;
    }
    __syncthreads();
    float as = 0.f;
#pragma unroll
    for (int s = 0; s < kMaxAttnSplit; ++s) as = fmaf(a[s], wgt[s], as);
    out[(size_t)head * hd + e] = float_to_bf16_bits(as * inv_l);
}

template <int HD>
hipError_t launch_g(int g, bool longer, const AttnParams &p, dim3 grid, hipStream_t stream) {
    switch (g) {
        case 1:
            if (longer) hipLaunchKernelGGL((attn_partial_kernel<HD, 1, 4>), grid, dim3(256), 0, stream, p);
            else hipLaunchKernelGGL((attn_partial_kernel<HD, 1, 2>), grid, dim3(256), 0, stream, p);
            break;
        case 2: hipLaunchKernelGGL((attn_partial_kernel<HD, 2, 2>), grid, dim3(256), 0, stream, p); break;
        case 4: hipLaunchKernelGGL((attn_partial_kernel<HD, 4, 2>), grid, dim3(256), 0, stream, p); break;
        case 8: hipLaunchKernelGGL((attn_partial_kernel<HD, 8, 2>), grid, dim3(256), 0, stream, p); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

// Whether one workgroup a query head takes all positions, two or four a lane and trip, and writes the result: every trip takes a chain of 0.6 us, chunks end in a
// launch that merges them.  us of the whole attention in a graph, 32 heads of 64 over 8, in chunks (four heads of a KV head to a workgroup, then the rule
// of launch_decode_attention) / whole: 64 positions 3.8 / 2.9 (one chunk), 128 5.9, 4.7 / 3.2, 256 5.9, 4.9 / 4.1, 384 6.0, 5.2 / 4.8,
// 512 5.9, 5.0 / 5.5.  Heads of 128: 64 4.8 / 3.2, 128 7.0, 5.6 / 4.1, 256 7.0, 5.8 / 5.5, 300 7.2, 6.1 / 6.2.  (16 waves instead of four 1.8 more, 8 waves
// 0.4 to 0.9.)
static bool attention_whole(int seq_len, int head_dim) { return seq_len <= (head_dim == 64 ? 384 : 256); }

int attention_nsplit(int seq_len, int head_dim) {
    if (attention_whole(seq_len, head_dim)) return 1;
    int n = (seq_len + 63) / 64;   // >= 64 positions per chunk
    if (n > kMaxAttnSplit) n = kMaxAttnSplit;
    return n;
}

size_t attention_workspace_bytes(int n_heads, int head_dim) {
    return (size_t)n_heads * kMaxAttnSplit * (2 + (size_t)head_dim) * sizeof(float);
}

hipError_t launch_decode_attention(const uint16_t *qkv, const uint16_t *lut_row, uint16_t *k_cache, uint16_t *v_cache,
                                   uint16_t *out, int pos, int max_seq, int n_heads, int n_kv, int head_dim,
                                   void *workspace, hipStream_t stream, bool combine) {
    AttnParams p;
    p.qkv = qkv;
    p.lut = lut_row;
    p.k_cache = k_cache;
    p.v_cache = v_cache;
    p.out = out;
    p.pos = pos;
    p.max_seq = max_seq;
    p.n_heads = n_heads;
    p.n_kv = n_kv;
    p.nsplit = attention_nsplit(pos + 1, head_dim);
    const int ppb = 4 * (64 / (head_dim / 8));   // positions per workgroup iteration
    p.chunk = (((pos + 1 + p.nsplit - 1) / p.nsplit + ppb - 1) / ppb) * ppb;
    p.scale = 1.0f / sqrtf((float)head_dim);
    p.part_ml = reinterpret_cast<float *>(workspace);
    p.part_acc = p.part_ml + (size_t)n_heads * kMaxAttnSplit * 2;
    // Query heads of a KV head to a workgroup: one if that makes a workgroup a CU at most, else two or four (a head costs a workgroup 0.3 to 0.9 us, but each that is not
    // there reads the cache again).  us with 4 / 2 / 1 heads, merge included: 32 heads of 64 over 8, 512 positions (64 / 128 / 256 workgroups) 6.0 / 5.2 / 5.0, 1000 (128 / 256 / 512)
    // 6.4 / 5.7 / 5.9, 1700 6.8 / 6.9 / 7.6; 32 of 128 over 4 at 1000 7.3 / 6.1 / 6.3, with all eight heads 9.7; 64 of 128 over 8 at 4000 12.8 / 13.1 / 14.4, with eight 13.3.
    // All eight heads of a KV head where that leaves two workgroups a CU and the cache is so long that reading it is what takes the time: with eight / four, 128 heads of
    // 128 over 16 at 3000 17.3 / 16.4, 6000 25.5 / 26.1, 12000 37.7 / 39.5, 32000 83.9 / 89.9, of 64 8000 18.6 / 18.1, 12200 23.4 / 24.1, 32000 47.0 / 49.0; 64 of 128 over 8 (one
    // workgroup a CU) at 32000 52.0 / 50.8.
    const int group = n_heads / n_kv;
    int g = 1;
    while (g < group && g < 4 && p.nsplit * n_heads / g > 256) g *= 2;
    if (g == 4 && group == 8 && p.nsplit * n_kv >= 512 && (long)pos * head_dim >= 5120 * 128) g = 8;
    if (p.nsplit == 1) {
        p.chunk = pos + 1;
        g = 1;
    }
    p.log2_sharers = __builtin_ctz(group / g);
    const dim3 grid(p.nsplit, n_heads / g);
    const bool longer = p.nsplit == 1 && pos >= ppb * 2;   // than two positions a lane
    hipError_t e = head_dim == 64 ? launch_g<64>(g, longer, p, grid, stream) : launch_g<128>(g, longer, p, grid, stream);
    if (e != hipSuccess || p.nsplit == 1 || !combine) return e;
    hipLaunchKernelGGL(attn_combine_kernel, dim3(n_heads), dim3(head_dim), 0, stream, p.part_ml, p.part_acc, out,
                       p.nsplit, head_dim);
    return hipGetLastError();
}

// Half-split RoPE of `rows` independent rows of `dim` elements, each with its own LUT row
// (cos then sin).  One thread rotates 8 consecutive elements of one row; dim % 16 == 0.
__global__ void __launch_bounds__(256) rope_rows_kernel(const uint16_t *x, const uint16_t *lut, uint16_t *out, int rows,
                                                        int dim) {
    const int per_row = dim >> 3;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= rows * per_row) return;
    const int row = t / per_row, e0 = 8 * (t % per_row);
    const int half = dim >> 1;
    const bool low = e0 < half;
    const int i0 = low ? e0 : e0 - half;
    const uint16_t *src = x + (size_t)row * dim;
    const uint16_t *l = lut + (size_t)row * dim;
    float a[8], b[8], c[8], s[8];
    unpack8(*reinterpret_cast<const u32x4 *>(src + e0), a);
    unpack8(*reinterpret_cast<const u32x4 *>(src + (low ? e0 + half : e0 - half)), b);
    unpack8(*reinterpret_cast<const u32x4 *>(l + i0), c);
    unpack8(*reinterpret_cast<const u32x4 *>(l + half + i0), s);
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        // products of two bf16 values are exact in fp32: one rounding to fp32, one to bf16, as in NumPy
        const float r0 = low ? a[2 * j] * c[2 * j] - b[2 * j] * s[2 * j] : a[2 * j] * c[2 * j] + b[2 * j] * s[2 * j];
        const float r1 = low ? a[2 * j + 1] * c[2 * j + 1] - b[2 * j + 1] * s[2 * j + 1]
                             : a[2 * j + 1] * c[2 * j + 1] + b[2 * j + 1] * s[2 * j + 1];
        o[j] = pack_bf16x2(r0, r1);
    }
    *reinterpret_cast<u32x4 *>(out + (size_t)row * dim + e0) = o;
}

hipError_t launch_rope_rows(const uint16_t *x, const uint16_t *lut, uint16_t *out, int rows, int dim, hipStream_t stream) {
    const int threads = rows * (dim >> 3);
    hipLaunchKernelGGL(rope_rows_kernel, dim3((threads + 255) / 256), dim3(256), 0, stream, x, lut, out, rows, dim);
    return hipGetLastError();
}

}  // namespace w4a16
