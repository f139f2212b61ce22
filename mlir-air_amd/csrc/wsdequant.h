// Stream-order cells (wstream.h) -> the bf16 weights of the dense dequant, in registers.
#pragma once

#include "common.h"

namespace w4a16 {

// eight weights of one dword (rows 8 lg .. 8 lg + 7 of the lane's column) as the four registers of a B operand
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

// Q4NX order: scale word -> scale s and min' (two bf16 halves)
__device__ __forceinline__ void decode_md_q4(uint32_t md, float &sf, float &c0) {
    sf = __builtin_bit_cast(float, md << 16);
    c0 = __builtin_bit_cast(float, md & 0xFFFF0000u);
}

// scale word -> scale s and -z * s (exact: (128 + z) - 128 and an 8 x 8 bit product)
__device__ __forceinline__ void decode_md(uint32_t md, float &sf, float &c0) {
    sf = __builtin_bit_cast(float, md << 16);
    const float nz = __builtin_bit_cast(float, md & 0xFFFF0000u);   // -(128 + z)
    c0 = (nz + 128.0f) * sf;
}

}  // namespace w4a16
