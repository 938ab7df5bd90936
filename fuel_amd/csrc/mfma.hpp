// Int8 MFMA building blocks shared by the batched QMatMul kernels
// (mmq.hip, mmq_skinny.hip): operand vector types and the byte-plane
// arithmetic that turns k-quant codes and sub-block scales into exact int8
// MFMA operands.
#pragma once

#include "common.hpp"

namespace frq {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// Four nibble bytes (<= 15) times a small factor (<= 7), byte by byte: each
// product is <= 105, so two 16-bit lane multiplies (one full-rate packed
// instruction) produce them without carries between bytes.
__device__ __forceinline__ int bytes_times(uint32_t q, uint32_t f) {
    const u16x2 p = __builtin_bit_cast(u16x2, q) * u16x2{(unsigned short)f, (unsigned short)f};
    return __builtin_bit_cast(int, p);
}

// Factor and offset of q6_planes for the 16-element scale sc, one copy per
// 16-bit lane.
__device__ __forceinline__ void q6_factors(int sc, uint32_t& sc16, uint32_t& c16) {
    const uint32_t f = (uint32_t)sc & 0xffffu, c = (uint32_t)(128 - 32 * sc) & 0xffffu;
    sc16 = f | (f << 16);
    c16 = c | (c << 16);
}

// Four 6-bit codes u (bytes of q, <= 63) -> w = (u - 32) * sc split into signed
// byte planes, w = 256 wh + wl.  Each 16-bit lane holds w + 128 exactly (|w| <=
// 4096), so the arithmetic runs two codes per packed instruction: even bytes,
// then odd bytes.  The high byte of w + 128 is wh and its low byte, less 128,
// is wl: two byte permutes and one exclusive or (a 128 wh + wl split took two
// shifts more per four codes).
__device__ __forceinline__ void q6_planes(uint32_t q, uint32_t sc16, uint32_t c16, int& wl, int& wh) {
    const u16x2 ev = __builtin_bit_cast(u16x2, q & 0x00ff00ffu);
    const u16x2 od = __builtin_bit_cast(u16x2, __builtin_amdgcn_perm(0u, q, 0x0c030c01u));  // bytes 1, 3
    const u16x2 f = __builtin_bit_cast(u16x2, sc16), c = __builtin_bit_cast(u16x2, c16);
    const uint32_t pe = __builtin_bit_cast(uint32_t, ev * f + c), po = __builtin_bit_cast(uint32_t, od * f + c);
    // interleave the four lanes' low and high bytes back into code order
    wl = (int)(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
    wh = (int)__builtin_amdgcn_perm(po, pe, 0x07030501u);
}

}  // namespace frq
