// Stream-order cells (wstream.h) -> the bf16 weights of the dense dequant, in registers.
#pragma once

#include "common.h"

namespace w4a16 {

// Eight weights of one dword (rows 8 lg .. 8 lg + 7 of the lane's column) as the four registers of a B operand, bf16(sf q + c0): any scale of either order
__device__ __forceinline__ bf16x8 dequant_operand(uint32_t w, float sf, float c0) {
    uint32_t e = w & 0x0F0F0F0Fu;          // nibbles 0, 2, 4, 6 -> rows 0, 4, 1, 5
    uint32_t o = (w >> 4) & 0x0F0F0F0Fu;   // nibbles 1, 3, 5, 7 -> rows 2, 6, 3, 7
    // kept opaque: the compiler would otherwise fold the masks into one v_bfe_u32 per nibble in front of every
    // convert (two instructions per weight) instead of the byte-select converts v_cvt_f32_ubyte0..3 (one)
    asm volatile("" : "+v"(e), "+v"(o));
    const float k0 = fmaf(static_cast<float>(e & 0xFFu), sf, c0), k4 = fmaf(static_cast<float>((e >> 8) & 0xFFu), sf, c0);
    const float k1 = fmaf(static_cast<float>((e >> 16) & 0xFFu), sf, c0), k5 = fmaf(static_cast<float>(e >> 24), sf, c0);
    const float k2 = fmaf(static_cast<float>(o & 0xFFu), sf, c0), k6 = fmaf(static_cast<float>((o >> 8) & 0xFFu), sf, c0);
    const float k3 = fmaf(static_cast<float>((o >> 16) & 0xFFu), sf, c0), k7 = fmaf(static_cast<float>(o >> 24), sf, c0);
    const u32x4 b = {pack_bf16x2(k0, k1), pack_bf16x2(k2, k3), pack_bf16x2(k4, k5), pack_bf16x2(k6, k7)};
    return __builtin_bit_cast(bf16x8, b);
}

// The same eight weights of the AWQ order in 17 vector instructions instead of 23.  A nibble behind the exponent of the half-precision 1024 is 1024 + q
// (bits 0 .. 3 of a half) or 1024 + 16 q (bits 4 .. 7), two weights a mask, and a multiply-add that takes a half as it is does conversion and scale in
// one: (1024 + q) s - (1024 + z) s = (q - z) s and (1024 + 16 q) s / 16 - (64 + z) s, exact in fp32 (11 x 8 bits), so
// the rounded weights are the same bits.  From scales of 2^117 on the offsets may be infinite, and then so is, or no number at all, every weight of the group and
// every result of its column: the kernels look for that behind their loop (awq_overflowed) and take such columns again with the form above
// (without such scales 300 rows of 4096 x 11008 and 2048 of 4096 x 14336 take as long as without the look).  300 rows of 4096 x 11008 48.2 -> 44.5 us, 512 of 4096 x 4096 30.4 -> 29.1, tiled 2048 of 4096 x 14336
// 178.5 -> 176.6.  (Q4NX keeps the 23: min' - 1024 s is not exact for a minimum that is small against the scale.)
struct AwqScale {
    float s, c, s16, c16;   // s, -(1024 + z) s, s / 16, -(64 + z) s
};
__device__ __forceinline__ AwqScale awq_scale(uint32_t md) {
    const float s = __builtin_bit_cast(float, md << 16), nz = __builtin_bit_cast(float, md & 0xFFFF0000u);   // nz = -(128 + z)
    return {s, (nz - 896.0f) * s, s * 0.0625f, (nz + 64.0f) * s};
}
constexpr uint32_t kLowNibbles = 0x000F000Fu, kHighNibbles = 0x00F000F0u, kHalf1024 = 0x64006400u;
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
// `low`, `high`, `magic`: the three constants in registers
__device__ __forceinline__ bf16x8 dequant_operand_awq(uint32_t w, const AwqScale &d, uint32_t low, uint32_t high, uint32_t magic) {
    const uint32_t w8 = w >> 8;
    auto pair = [](uint32_t n, float s, float c) __attribute__((always_inline)) {
        const f16x2 h = __builtin_bit_cast(f16x2, n);
        return pack_bf16x2(fmaf(static_cast<float>(h.x), s, c), fmaf(static_cast<float>(h.y), s, c));
    };
    const u32x4 b = {pair((w & low) | magic, d.s, d.c), pair((w & high) | magic, d.s16, d.c16), pair((w8 & low) | magic, d.s, d.c),
                     pair((w8 & high) | magic, d.s16, d.c16)};
    return __builtin_bit_cast(bf16x8, b);
}

// AWQ order: scale word -> scale s and -z s (exact: (128 + z) - 128 and an 8 x 8 bit product), for dequant_operand
__device__ __forceinline__ void decode_md(uint32_t md, float &sf, float &c0) {
    sf = __builtin_bit_cast(float, md << 16);
    const float nz = __builtin_bit_cast(float, md & 0xFFFF0000u);   // -(128 + z)
    c0 = (nz + 128.0f) * sf;
}
// Whether a column of the wave may have had a weight of AwqScale that is not finite, by two results of it, of different rows of x (one row may itself hold
// an infinity).
__device__ __forceinline__ bool awq_overflowed(float a, float b) { return !__builtin_isfinite(a) && !__builtin_isfinite(b); }

// Q4NX order: scale word -> scale s and min' (two bf16 halves)
__device__ __forceinline__ void decode_md_q4(uint32_t md, float &sf, float &c0) {
    sf = __builtin_bit_cast(float, md << 16);
    c0 = __builtin_bit_cast(float, md & 0xFFFF0000u);
}

}  // namespace w4a16
