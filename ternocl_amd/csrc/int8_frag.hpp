// int8_frag.hpp -- operand order of the s8 x s2 GEMMs: the packed word's int8
// fragment, the matching byte transpose of the activations, and the in-GEMM
// quantization.
#pragma once

#include "common.hpp"

namespace tcl {
namespace {

typedef int i32x4_t __attribute__((ext_vector_type(4)));

__host__ __device__ constexpr int ldsa_of(int M) { return (M + 31) & ~31; }

constexpr uint32_t kCodeLut = 0xFFFE0100u;  // int8 of code 0, 1, 2, 3

// out[i] byte b = byte i of d[b] (4 x 4 byte transpose)
__device__ __forceinline__ void transpose4x4(const uint32_t d[4], uint32_t o[4]) {
    const uint32_t p0 = __builtin_amdgcn_perm(d[1], d[0], 0x06020400u);  // d0.b0 d1.b0 d0.b2 d1.b2
    const uint32_t p1 = __builtin_amdgcn_perm(d[1], d[0], 0x07030501u);  // d0.b1 d1.b1 d0.b3 d1.b3
    const uint32_t p2 = __builtin_amdgcn_perm(d[3], d[2], 0x06020400u);
    const uint32_t p3 = __builtin_amdgcn_perm(d[3], d[2], 0x07030501u);
    o[0] = __builtin_amdgcn_perm(p2, p0, 0x05040100u);
    o[1] = __builtin_amdgcn_perm(p3, p1, 0x05040100u);
    o[2] = __builtin_amdgcn_perm(p2, p0, 0x07060302u);
    o[3] = __builtin_amdgcn_perm(p3, p1, 0x07060302u);
}

// B fragment of one word: dword i byte b = int8 value of row 4b + i.
__device__ __forceinline__ i32x4_t decode_s2(uint32_t w) {
    i32x4_t r;
    r[0] = (int)__builtin_amdgcn_perm(kCodeLut, kCodeLut, w & 0x03030303u);
    r[1] = (int)__builtin_amdgcn_perm(kCodeLut, kCodeLut, (w >> 2) & 0x03030303u);
    r[2] = (int)__builtin_amdgcn_perm(kCodeLut, kCodeLut, (w >> 4) & 0x03030303u);
    r[3] = (int)__builtin_amdgcn_perm(kCodeLut, kCodeLut, (w >> 6) & 0x03030303u);
    return r;
}

// In-GEMM quantization (the reference's QMODE 1, int2_int8_dpas.cl:61-68 and
// quant8x32 :70-99): the int8 of a DT activation is the low byte of
// fma(a, sa, 1.5 * 2^23), which rounds a * sa (exact in fp32) to the nearest
// even integer; |a * sa| <= 127.06 by the construction of sa, so it equals
// quant_a's saturating conversion for every finite input.
template <bool BF16>
__device__ __forceinline__ uint32_t q8_bits(uint32_t h, float sa) {
    return __float_as_uint(__builtin_fmaf(dt2f<BF16>(h), sa, 12582912.0f));
}

}  // namespace
}  // namespace tcl
