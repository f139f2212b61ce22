// Shared device helpers for the gfx950 W4A16 kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace w4a16 {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kGroup = 128;

// AWQ order: bit position 4*i of a word holds natural column kPackOrder[i] of its block.
__host__ __device__ constexpr int pack_order(int i) { return ((i & 3) << 1) | (i >> 2); }      // 0,2,4,6,1,3,5,7
// Bit-position index that holds natural column j.
__host__ __device__ constexpr int unpack_pos(int j) { return ((j & 1) << 2) | (j >> 1); }      // 0,4,1,5,2,6,3,7

__device__ __forceinline__ float bf16_bits_to_float(uint32_t bits16) {
    return __builtin_bit_cast(float, bits16 << 16);
}

// Two fp32 -> packed bf16 pair (round-to-nearest-even, v_cvt_pk_bf16_f32): low half = a.
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
    bf16x2 v;
    v.x = static_cast<__bf16>(a);
    v.y = static_cast<__bf16>(b);
    return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ uint16_t float_to_bf16_bits(float a) {
    __bf16 v = static_cast<__bf16>(a);
    return __builtin_bit_cast(uint16_t, v);
}

// Nibble at bit-position index `pos` of `w` as float (exact).
__device__ __forceinline__ float nibble_f32(uint32_t w, int pos) {
    return static_cast<float>((w >> (4 * pos)) & 0xFu);
}

// The 8 nibbles of one AWQ word as floats in NATURAL column order.  The even/odd
// nibble split lets every conversion be a byte-select convert (v_cvt_f32_ubyteN).
__device__ __forceinline__ void unpack8_f32(uint32_t w, float (&q)[8]) {
    const uint32_t e = w & 0x0F0F0F0Fu;          // positions 0,2,4,6 -> columns 0,4,1,5
    const uint32_t o = (w >> 4) & 0x0F0F0F0Fu;   // positions 1,3,5,7 -> columns 2,6,3,7
    q[0] = static_cast<float>(e & 0xFFu);
    q[4] = static_cast<float>((e >> 8) & 0xFFu);
    q[1] = static_cast<float>((e >> 16) & 0xFFu);
    q[5] = static_cast<float>(e >> 24);
    q[2] = static_cast<float>(o & 0xFFu);
    q[6] = static_cast<float>((o >> 8) & 0xFFu);
    q[3] = static_cast<float>((o >> 16) & 0xFFu);
    q[7] = static_cast<float>(o >> 24);
}

// v + the value that the DPP control CTRL moves to this lane
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// Two lane halves (SWAP 32) or neighbouring rows of 16 lanes (SWAP 16): first + second of the values that each pair of lanes holds of `a`
// in the one lane, of `b` in the other.
template <int SWAP, bool MAX>
__device__ __forceinline__ float swap_reduce(float a, float b) {
    const auto r = SWAP == 32 ? __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false)
                              : __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    const unsigned first = r[0], second = r[1];   // (a bit cast of an element itself reads the vector's first one)
    const float x = __builtin_bit_cast(float, first), y = __builtin_bit_cast(float, second);
    return MAX ? fmaxf(x, y) : x + y;
}
// Maximum / sum over the 64 lanes of a wavefront, every lane receiving the result: the four steps inside a row of
// 16 lanes on DPP moves (quad permutes for distances 1 and 2, half-row and row mirrors for 4 and 8: once the
// quads agree, mirroring meets the partner quad), the two steps across rows by exchanging rows and halves of two copies, which then hold a
// lane's own value and its partner's (a shuffle goes through LDS; the same sums,
// bit for bit.  The choice of 8 experts by one wave, eight maxima one after the other: 14.5 -> 14.0 us for the launch that makes it).
template <bool MAX>
__device__ __forceinline__ float wave_reduce(float v) {
    auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
    auto dpp = [&](auto ctrl) {
        constexpr int CTRL = decltype(ctrl)::value;
        const int moved = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true);
        v = op(v, __builtin_bit_cast(float, moved));
    };
    dpp(std::integral_constant<int, 0xB1>());    // quad_perm [1, 0, 3, 2]
    dpp(std::integral_constant<int, 0x4E>());    // quad_perm [2, 3, 0, 1]
    dpp(std::integral_constant<int, 0x141>());   // row_half_mirror
    dpp(std::integral_constant<int, 0x140>());   // row_mirror
    v = swap_reduce<16, MAX>(v, v);   // rows (0, 1) and (2, 3) exchanged
    return swap_reduce<32, MAX>(v, v);   // halves exchanged
}

// Maximum / sum over the 16 lanes of a DPP row, every lane of the row receiving it (the four in-row steps of wave_reduce).
template <bool MAX>
__device__ __forceinline__ float row_reduce16(float v) {
    auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
    auto dpp = [&](auto ctrl) {
        constexpr int CTRL = decltype(ctrl)::value;
        v = op(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true)));
    };
    dpp(std::integral_constant<int, 0xB1>());    // quad_perm [1, 0, 3, 2]
    dpp(std::integral_constant<int, 0x4E>());    // quad_perm [2, 3, 0, 1]
    dpp(std::integral_constant<int, 0x141>());   // row_half_mirror
    dpp(std::integral_constant<int, 0x140>());   // row_mirror
    return v;
}
__device__ __forceinline__ float row_sum16(float v) { return row_reduce16<false>(v); }

// max over the four lanes ql, ql + 16, ql + 32, ql + 48
__device__ __forceinline__ float max_over_lane_groups(float v) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);   // rows (0, 1) and (2, 3) exchanged
    v = fmaxf(__builtin_bit_cast(float, (uint32_t)a[0]), __builtin_bit_cast(float, (uint32_t)a[1]));
    const uint32_t w = __builtin_bit_cast(uint32_t, v);
    const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);   // halves exchanged
    return fmaxf(__builtin_bit_cast(float, (uint32_t)b[0]), __builtin_bit_cast(float, (uint32_t)b[1]));
}

// Sum of n matrices `stride` floats apart at one place, in their order, AT of them asked for together (one after the other each costs a round trip to the last-level cache)
template <int AT>
__device__ __forceinline__ floatx4 sum_parts(const float *p, size_t stride, int n) {
    floatx4 sum;
    for (int k0 = 0; k0 < n; k0 += AT) {
        floatx4 v[AT];
#pragma unroll
        for (int k = 0; k < AT; ++k) v[k] = *reinterpret_cast<const floatx4 *>(p + (size_t)(k0 + k < n ? k0 + k : n - 1) * stride);
#pragma unroll
        for (int k = 0; k < AT; ++k) sum = k0 + k == 0 ? v[k] : k0 + k < n ? sum + v[k] : sum;
    }
    return sum;
}

// silu(g) in the reference's tanh form (matvec_int4_swiglu_rms.py:512-514), fp32
__device__ __forceinline__ float silu_tanh(float g) { return g * 0.5f * (tanhf(g * 0.5f) + 1.0f); }

// z sigmoid(v) with the error of z / (1 + expf(-v)) in fp32 (half a unit of 2^-24 on average, two and a half at most) over its whole range,
// in 19 instructions instead of 27, none of them a division's.  A wide tile's store has up to 256 of them to a lane, alone on its SIMD:
// 2048 x 11264 x 2048 with silu on 4096 columns 96 us with the division, 91 with this, 83 with the bare hardware exponential and
// reciprocal, whose argument is rounded behind log2 e (30 units at v = -60).
// Over all bf16 gates rms 0.30 and at most 2.1 units of 2^-24 (0.33 and 2.2 with the division and expf); int4 gate and up of 4096 x 14336 for 2048 tokens
// 387 -> 384 us with it.
// e = e^-|v|: the product with log2 e is cut at a whole number n before it is rounded; s / (1 + e), s = 1 or for v < 0 e, by the hardware's
// reciprocal and one step that takes back its error and that of 1 + e.  (Past 150 e is 0.)
__device__ __forceinline__ float gated_f32(float z, float v) {
    const float a = __builtin_amdgcn_fmed3f(fabsf(v), 0.0f, 150.0f);
    const float n = rintf(-1.44269502f * a), x = fmaf(-1.92596303e-8f, a, fmaf(-1.44269502f, a, -n));   // log2 e in two parts
    const float e = ldexpf(__builtin_amdgcn_exp2f(x), (int)n), s = v < 0.0f ? e : 1.0f;
    const float d = 1.0f + e, r = __builtin_amdgcn_rcpf(d), q = s * r;
    return z * fmaf(fmaf(-q, e - (d - 1.0f), fmaf(-d, q, s)), r, q);
}

// "No score yet" of the attention partials: finite, so differences of two of them are 0, not NaN.
constexpr float kAttnNegBig = -1e30f;

// Agent-scope (all XCDs) relaxed accesses for data exchanged between workgroups.
__device__ __forceinline__ void store_agent(float *p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_agent(const float *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A wave-uniform pointer pinned to scalar registers: loads and copies through it take the form "scalar base + 32-bit lane offset", and
// the per-lane part stays one VGPR (left alone the compiler folds the lane offset into a 64-bit VGPR base per stream and spends two
// VGPRs and a 64-bit add on every request).  The offset's zero extension has to be in the same basic block as its request to fold
// into the instruction: a loop makes its offsets opaque once per turn.
typedef const __attribute__((address_space(1))) char *gptr;
__device__ __forceinline__ gptr scalar_ptr(const void *p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    asm volatile("" : "+s"(lo), "+s"(hi));
    return reinterpret_cast<gptr>(((uint64_t)hi << 32) | lo);
}

}  // namespace w4a16
