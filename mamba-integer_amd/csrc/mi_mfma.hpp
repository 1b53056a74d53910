// Ternary unpack, the int8 MFMA and the int8 epilogue pieces of the BitLinear kernels.
#pragma once

#include "mi_common.hpp"

namespace mi {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef long long v2l __attribute__((ext_vector_type(2)));  // (sum r, sum r^2) pairs

// 16 ternary weights of one packed word -> 16 int8 in k order (4 dwords).
// (word >> 2j) & 0x03030303 holds the 2-bit codes of weights 4j..4j+3 in byte
// order; v_perm_b32 against the byte table {0x00, 0x01, 0xFE, 0xFF} (byte c =
// value of code c, both permute sources equal) sign-extends all four at once.
__device__ __forceinline__ v4i unpack16(uint32_t w) {
    const uint32_t lut = 0xFFFE0100u;
    v4i r;
    r[0] = (int)__builtin_amdgcn_perm(lut, lut, w & 0x03030303u);
    r[1] = (int)__builtin_amdgcn_perm(lut, lut, (w >> 2) & 0x03030303u);
    r[2] = (int)__builtin_amdgcn_perm(lut, lut, (w >> 4) & 0x03030303u);
    r[3] = (int)__builtin_amdgcn_perm(lut, lut, (w >> 6) & 0x03030303u);
    return r;
}

// D(16x16) += A(16x64) * B(64x16), int8 in, int32 accumulate (gfx950).
__device__ __forceinline__ v4i mfma_i8(v4i a, v4i b, v4i c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

// The low bytes of four values as one dword (three v_perm_b32).
__device__ __forceinline__ uint32_t pack4(int v0, int v1, int v2, int v3) {
    return __builtin_amdgcn_perm(__builtin_amdgcn_perm((uint32_t)v3, (uint32_t)v2, 0x0c0c0400u),
                                 __builtin_amdgcn_perm((uint32_t)v1, (uint32_t)v0, 0x0c0c0400u), 0x05040100u);
}

// Exact squareplus of spec rule 4.4 on four conv outputs c (Q10) -> int8 (Q4):
// q = min((v + isqrt(v^2 + 2^22) + 64) >> 7, 127), v = c within +-51200, which
// is floor((v + s + 64) / 128) of the real s = sqrt(v^2 + 2^22).  q >= k where
// v >= T/2 - 2^21/T, T = 128 k - 64; for k >= 2 an integer v stays 1/(2k - 1)
// or more away from that, so (v + s) stays 64/s > 0.0057 away from T, while
// the rounding of v^2 + 2^22 and v_sqrt_f32 (1 ulp) move it by 0.0013 at most
// (s < 11100 there): nearest-rounding (v + s) / 128 gives q.  k = 1 holds from
// v = -32736 up, which is tested on the integers: q of a smaller v is 0, and
// the float form sees v from -20000 (q = 1) to 8000 (q = 127, where every
// larger v stays).  v_cvt_pk_u8_f32 rounds and packs.  ~8 instructions a value
// against ~24 of the integer root (float estimate corrected by two squares and
// compares); the in_proj GEMM with conv of 16384 x 768 -> 3072 72 -> 60 us,
// of 2000 rows 14.5 -> 13.6.
constexpr int32_t kSqpZero = -32736;   // q = 0 below it

__device__ __forceinline__ uint32_t sqp_byte(int32_t c, int r, uint32_t o) {
    const float v = (float)clamp32(c, -20000, 8000);
    const float f = __builtin_amdgcn_sqrtf(__builtin_fmaf(v, v, 4194304.0f)) + v;
    return __builtin_amdgcn_cvt_pk_u8_f32(f * 0.0078125f, r, o);
}
__device__ __forceinline__ int sqp1(int32_t c) { return c < kSqpZero ? 0 : (int)sqp_byte(c, 0, 0); }
__device__ __forceinline__ uint32_t sqp4(int32_t c0, int32_t c1, int32_t c2, int32_t c3) {
    const int32_t c[4] = {c0, c1, c2, c3};
    uint32_t o = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) o = sqp_byte(c[r], r, o);
    if (min(min(c0, c1), min(c2, c3)) < kSqpZero) {
#pragma unroll
        for (int r = 0; r < 4; ++r) o &= c[r] < kSqpZero ? ~(255u << (8 * r)) : ~0u;
    }
    return o;
}

}  // namespace mi
