// What the f32 products on the bf16 instructions (gemm_f32_split.hip, gemm_f32_ks_split.hip) ask of the values they split.
#pragma once
#include "common.h"

namespace mg {

// Three bf16 parts hold x exactly, with no infinity on the way, for zero and for 2^-102 <= |x| < 2^60. A thread's values so far:
// most: the largest magnitude (a NaN is none: it stays one in the parts); least: the smallest magnitude's bits, times two and less
// one, so that a zero is the largest there. Of the f32 bits, not of the first part's: up to 2^-134 that one is a zero (and the parts lose x).
struct PartsRange {
    float most;
    unsigned least;
    __device__ __forceinline__ void begin() {
        most = 0.f;
        least = ~0u;
    }
    __device__ __forceinline__ void look(float x, float y) {
        const unsigned a = 2u * __float_as_uint(x) - 1u, b = 2u * __float_as_uint(y) - 1u;
#ifdef MG_HOST_AUDIT
        most = max(most, max(fabsf(x), fabsf(y)));
        least = min(least, min(a, b));
#else
        asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(most) : "v"(x), "v"(y));
        asm("v_min3_u32 %0, %1, %2, %0" : "+v"(least) : "v"(a), "v"(b));
#endif
    }
    __device__ __forceinline__ bool beyond() const { return most >= 0x1p60f || least < 2u * (25u << 23) - 1u; }
};

}  // namespace mg
