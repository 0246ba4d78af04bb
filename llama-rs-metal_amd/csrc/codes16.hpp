// Affine codes as f16 pairs: code - 2^(BITS-1), exact for 2, 4 and 8 bits.
//
// A masked code OR'ed into the mantissa of a power of two is that power plus
// the code; one packed f16 addition takes the power and the code's centre
// away.  1.1 instructions a code at 4 bits against 1.4 for byte conversions to
// F32, and the centred values make sums of code * x smaller than unsigned ones
// (and their rounding with them).
#pragma once
#include "device_common.hpp"

namespace moehip {

namespace codes16 {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t cu32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t as_u32(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ f16x2 as_h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
// Exponents that place code bits at a value's units: two f16 of 2^10 (units at
// bit 0), 2^8 (bit 2), 2^6 (bit 4) and 2^4 (bit 6), in vector registers, so
// that v_and_or_b32 takes mask and magic as they are.
struct Magic {
    uint32_t u0 = 0x64006400u, u2 = 0x5c005c00u, u4 = 0x54005400u, u6 = 0x4c004c00u;
    __device__ __forceinline__ void pin() {
        asm("" : "+v"(u0));
        asm("" : "+v"(u2));
        asm("" : "+v"(u4));
        asm("" : "+v"(u6));
    }
};
// (w & mask | magic) + off as two f16: off takes the magic and the code's
// centre away
__device__ __forceinline__ uint32_t code_pair(uint32_t w, uint32_t mask, uint32_t magic, float off) {
    const f16x2 o = {(_Float16)off, (_Float16)off};
    return as_u32(as_h2((w & mask) | magic) + o);
}

// The 8 codes of one fragment as f16 code - 2^(BITS-1), in the order (0, 4),
// (1, 5), (2, 6), (3, 7) -- the order the input rows are stored in.
//   8-bit: w0 codes 0-3, w1 codes 4-7; 4-bit: w0; 2-bit: half `sel` of w0
template <int BITS>
__device__ __forceinline__ f16x8 code_frag(uint32_t w0, uint32_t w1, int sel, const Magic &mg) {
    cu32x4 o;
    if constexpr (BITS == 4) {
        const uint32_t w8 = w0 >> 8;
        o[0] = code_pair(w0, 0x000f000fu, mg.u0, -1032.f);  // 1024 + c
        o[1] = code_pair(w0, 0x00f000f0u, mg.u4, -72.f);    // 64 + c
        o[2] = code_pair(w8, 0x000f000fu, mg.u0, -1032.f);
        o[3] = code_pair(w8, 0x00f000f0u, mg.u4, -72.f);
    } else if constexpr (BITS == 8) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            o[i] = code_pair(__builtin_amdgcn_perm(w1, w0, 0x0c040c00u + i * 0x00010001u), 0xffffffffu, mg.u0,
                             -1152.f);
    } else {
        const uint32_t t = __builtin_amdgcn_perm(w0, w0, sel ? 0x0c030c02u : 0x0c010c00u);
        o[0] = code_pair(t, 0x00030003u, mg.u0, -1026.f);  // 1024 + c
        o[1] = code_pair(t, 0x000c000cu, mg.u2, -258.f);   // 256 + c
        o[2] = code_pair(t, 0x00300030u, mg.u4, -66.f);    // 64 + c
        o[3] = code_pair(t, 0x00c000c0u, mg.u6, -18.f);    // 16 + c
    }
    return __builtin_bit_cast(f16x8, o);
}

}  // namespace codes16

}  // namespace moehip
