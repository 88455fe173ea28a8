// Device-side arithmetic shared by every kernel that produces qsi8: the exact float sequence of
// the reference's generated C, so that outputs are bit-identical.
//
//   conv / FullyConnected : fp32_to_int8(act((float)acc * src_scale * flt_scale / dst_scale))
//                           (BareMetal/Activation.cpp:47-56,105-114; ConvKernel.cpp:374-380)
//   fp32_to_int8          : int r = roundf(x); clamp to [-128,127]   (half away from zero)
//
// Built with -ffp-contract=off: no multiply may fuse with a following add, and the division is the
// correctly rounded IEEE one (hipcc's default for fp32 `/`); int->float conversion rounds to
// nearest even exactly like the host's cvtsi2ss.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <memory>

#include "megcc_gfx950.h"

namespace mg {

template <int ACT>
__host__ __device__ __forceinline__ float act_apply(float x) {
    if (ACT == MEGCC_NONLINE_RELU) {
        return x > 0 ? x : 0;
    } else if (ACT == MEGCC_NONLINE_H_SWISH) {
        // res * min(max(res + 3, 0.f), 6.f) * (1.f / 6.f) with the generated min/max helpers
        float t = x + 3;
        float mx = t > 0.f ? t : 0.f;
        float mn = mx > 6.f ? 6.f : mx;
        return x * mn * (1.f / 6.f);
    } else if (ACT == MEGCC_NONLINE_SIGMOID) {
        return 1.f / (expf(-x) + 1.f);
    }
    return x;
}

// (int)x by the instruction's name: it saturates and turns NaN into 0, where the conversion in the language is undefined
// for what an int cannot hold
__device__ __forceinline__ int cvt_i32(float x) {
    int r = 0;
#ifndef MG_HOST_AUDIT  // (a host build that looks at addresses only)
    asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(x));
#endif
    return r;
}

__host__ __device__ __forceinline__ int fp32_to_int8(float v) {
    // (on the host, where nothing saturates, clamped as a float)
#if defined(__HIP_DEVICE_COMPILE__)
    // Half away from zero is truncation of the value plus the largest float below a half (the same for every
    // float, checked one by one; a half itself would carry 0.49999997 up): four instructions for nine.
    const int i = cvt_i32(v + __builtin_copysignf(0x1.fffffep-2f, v));
    return i > 127 ? 127 : (i < -128 ? -128 : i);
#else
    float r = roundf(v);
    r = r > 127.f ? 127.f : r;
    r = r < -128.f ? -128.f : r;
    return (int)r;
#endif
}

// acc already includes the int32 bias. (Rounded like fp32_to_int8, but clamped while it is a float, which the compiler can
// see through: FullyConnected tiles lost 2 % to the instruction by name.)
template <int ACT>
__host__ __device__ __forceinline__ int requant_conv(int acc, float s_src, float s_flt, float s_dst) {
    const float v = act_apply<ACT>((float)acc * s_src * s_flt / s_dst);
#if defined(__HIP_DEVICE_COMPILE__)
    return (int)__builtin_amdgcn_fmed3f(v + __builtin_copysignf(0x1.fffffep-2f, v), -128.f, 127.f);
#else
    return fp32_to_int8(v);
#endif
}

// ---- exact requantisation at a third of the instructions ---------------------------------------
// For IDENTITY and RELU the int8 result only depends on which integer the scaled value rounds to,
// so it can be taken from ONE multiply by c = fl(fl(s_src*s_flt)/s_dst) whenever that product is
// safely away from a rounding boundary:
//     v = fl(fl(fl(a*s_src)*s_flt)/s_dst)  (the reference, three roundings)
//     g = fl(a*c)                          (three roundings too, c is computed on the host)
// both are within 3*2^-24 relative of the real quotient, so |v - g| <= 6*2^-24*|v| < 2^-14 for
// |v| < 129. If the distance of g to the nearest integer r is below 0.5 - 2^-13, v rounds (half
// away from zero, like roundf) to the same r; beyond +-129 both clamp. Only lanes closer than
// 2^-13 to a tie (about one in 4000; exact ties included) take the reference's own sequence.
// RELU commutes with the rounding: roundf(max(v,0)) == max(roundf(v),0).
struct RequantFast {
    float c;       // fl(fl(s_src*s_flt)/s_dst); 0 disables the fast path (extreme scales)
    float s_src, s_flt, s_dst;
};

// host side: c, or 0 when a scale is so extreme that the error bound above does not hold
static inline RequantFast make_requant_fast(float s_src, float s_flt, float s_dst) {
    RequantFast q;
    q.s_src = s_src;
    q.s_flt = s_flt;
    q.s_dst = s_dst;
    const float p = s_src * s_flt;
    const float c = p / s_dst;
    auto mid = [](float x) { return x > 1e-30f && x < 1e30f; };
    const bool sane = mid(s_src) && mid(s_flt) && mid(p) && mid(s_dst) && mid(c);
    q.c = sane ? c : 0.f;
    return q;
}

template <int ACT>
__device__ __forceinline__ int requant_conv_fast(int acc, const RequantFast& q) {
    static_assert(ACT == MEGCC_NONLINE_IDENTITY || ACT == MEGCC_NONLINE_RELU, "monotone only");
    const float a = (float)acc;
    const float g = a * q.c;
    const float r = __builtin_rintf(g);  // nearest, ties to even: ties never use this result
    const float d = __builtin_fabsf(g - r);
    int out;
    if (__builtin_expect((!(d <= 0.5f - 0x1p-13f) && __builtin_fabsf(g) < 129.f) || q.c == 0.f, 0)) {
        out = requant_conv<ACT>(acc, q.s_src, q.s_flt, q.s_dst);
    } else {
        const float lo = ACT == MEGCC_NONLINE_RELU ? 0.f : -128.f;
        out = (int)__builtin_amdgcn_fmed3f(r, lo, 127.f);  // (clamped as a float: an int holds it)
    }
    return out;
}

// run-time activation selector (a uniform branch) for kernels that are not templated on it
__device__ __forceinline__ int requant_conv_rt(int act, int acc, float s0, float s1, float s2) {
    switch (act) {
        case MEGCC_NONLINE_RELU:
            return requant_conv<MEGCC_NONLINE_RELU>(acc, s0, s1, s2);
        case MEGCC_NONLINE_H_SWISH:
            return requant_conv<MEGCC_NONLINE_H_SWISH>(acc, s0, s1, s2);
        case MEGCC_NONLINE_SIGMOID:
            return requant_conv<MEGCC_NONLINE_SIGMOID>(acc, s0, s1, s2);
        default:
            return requant_conv<MEGCC_NONLINE_IDENTITY>(acc, s0, s1, s2);
    }
}

// ---- exact requantisation by threshold table ---------------------------------------------------
// For a monotone activation (IDENTITY, RELU) the reference's F(acc) = fp32_to_int8(act(acc * s_src
// * s_flt / s_dst)) is a non-decreasing step function of the integer accumulator, so it is fully
// described by 255 thresholds T[j] = max{a : F(a) < j}, j = -127..127:  F(a) = lo + #{j : a > T[j]}.
// The table is built with the reference's literal float sequence (a search over int32 per level) - on
// the host, once per (activation, scales) and cached, since x86-64 SSE arithmetic and the device's
// are the same IEEE operations; it travels to the kernel as an argument and each workgroup copies
// it to LDS. A kernel then needs only ONE estimate per output:
// with g = fl((float)a * c), c = fl(fl(s_src*s_flt)/s_dst), the true value is within 2^-14 of g
// while |g| < 129, so F(a) is floor(g) or floor(g)+1 (clamped), and the table decides which:
//     m = clamp(floor(g), lo, 126);   F(a) = m + (a > T[m + 1])
// No rounding-mode reasoning, no near-tie special case, bit-exact by construction.
static constexpr int REQUANT_TABLE_ENTRIES = 256;  // entry j + 127, last one unused

// (int)floorf(x) in one instruction (saturating like the plain conversion)
__device__ __forceinline__ int cvt_floor_i32(float x) {
    int r = 0;
#ifndef MG_HOST_AUDIT
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
#endif
    return r;
}

struct RequantTable {
    int t[REQUANT_TABLE_ENTRIES];
};

// H_SWISH joins the monotone activations: the reference applies it to the value already divided by
// the output scale, h(v) = v * min(max(v + 3, 0), 6) * (1/6), so its dip (-0.375 at v = -1.5) never
// reaches -0.5 and F is 0 for every v < 0; for v >= 0 both factors grow with v and every float
// rounding keeps the order, so F is a non-decreasing step function from 0 to 127 and the same table
// describes it exactly. The estimate is h(g) itself: |h(g) - h(v)| <= 1.5 * 2^-14, far inside the
// quarter that the look-up tolerates (m = floor(h(g) + 0.25), F = m or m + 1).
static inline bool requant_table_act(int act) {
    return act == MEGCC_NONLINE_IDENTITY || act == MEGCC_NONLINE_RELU || act == MEGCC_NONLINE_H_SWISH;
}

// host: the table for (act in {IDENTITY, RELU, H_SWISH}, scales); requant_table.hip
std::shared_ptr<const RequantTable> requant_table_for(int act, float s_src, float s_flt, float s_dst);

// the lower candidate m (clamped to [lowest output, 126]) of the output for accumulator acc
template <int ACT>
__device__ __forceinline__ int requant_table_candidate(int acc, float c) {
    static_assert(ACT == MEGCC_NONLINE_IDENTITY || ACT == MEGCC_NONLINE_RELU || ACT == MEGCC_NONLINE_H_SWISH,
                  "monotone only");
    constexpr int LO = ACT == MEGCC_NONLINE_IDENTITY ? -128 : 0;
    float g = (float)acc * c;
    if (ACT == MEGCC_NONLINE_H_SWISH) {
        const float t = __builtin_fminf(__builtin_fmaxf(g + 3.f, 0.f), 6.f);
        g = __builtin_fmaf(g * t, 1.f / 6.f, 0.25f);
    }
    const int m = cvt_floor_i32(g);  // saturating conversion
    return m < LO ? LO : (m > 126 ? 126 : m);
}

// table: pointer to entry 0 (LDS)
template <int ACT>
__device__ __forceinline__ int requant_conv_table(int acc, float c, const int* table) {
    const int m = requant_table_candidate<ACT>(acc, c);
    return m + (acc > table[m + 128] ? 1 : 0);
}

// ---- exact requantisation by ONE fused multiply-add, where the host can prove it ----------------
// The table look-up costs 7-8 vector instructions and an LDS read per output, and layers with few
// multiply-adds per output (pointwise with 32..128 input channels, depthwise) are bound by exactly
// that. For IDENTITY and RELU the candidate
//     F'(a) = clamp(floor(fma((float)a, c', d)), lo, 127)
// is a non-decreasing step function of a like F itself, so F' == F on all of int32 iff the two
// agree on both sides of every step of F - 2 x 255 evaluations. The host looks for a pair (c', d)
// near (c, 0.5) that passes that check against the reference's literal float sequence (for each
// c' within a few ulps of c the feasible d form an interval; its middle is then verified with the
// exact fmaf) and caches the answer per (activation, scales). Scales with exact ties whose
// roundings land on either side (0.02 * 0.01 / 0.05 ...) have no such pair and keep the table;
// calibrated scales of real networks almost always have one. 4 instructions per output, no LDS.
struct RequantAffine {
    float c, d;  // d == 0: no exact pair exists (or the activation is not IDENTITY / RELU)
};
RequantAffine requant_affine_for(int act, float s_src, float s_flt, float s_dst);
// what a launch uses: the pair (and the launch is noted as "+affine") when `table` - the kernel is the
// table instantiation for IDENTITY / RELU - and the switch "noaffine" is off; else d == 0. Call it
// after note_kernel().
RequantAffine requant_affine_pick(bool table, int act, float s_src, float s_flt, float s_dst);

template <int ACT>
__device__ __forceinline__ int requant_conv_affine(int acc, float c, float d) {
    constexpr int LO = ACT == MEGCC_NONLINE_RELU ? 0 : -128;
    const int m = cvt_floor_i32(__builtin_fmaf((float)acc, c, d));  // saturating conversion
    return m < LO ? LO : (m > 127 ? 127 : m);
}

// bytes 0 of a, b, c, d -> one dword
__device__ __forceinline__ uint32_t pack4_perm(int a, int b, int c, int d) {
    const uint32_t lo = __builtin_amdgcn_perm((uint32_t)b, (uint32_t)a, 0x0c0c0400u);
    const uint32_t hi = __builtin_amdgcn_perm((uint32_t)d, (uint32_t)c, 0x0c0c0400u);
    return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

// bytes 1 and 3 of two pairs of 16-bit values -> one dword: their floor by 256
__device__ __forceinline__ uint32_t pack4_high(uint32_t ab, uint32_t cd) {
    return __builtin_amdgcn_perm(cd, ab, 0x07050301u);
}
// two ints saturated to 16 bits
__device__ __forceinline__ uint32_t pack2_sat(int a, int b) {
#ifndef MG_HOST_AUDIT
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pk_i16(a, b));
#else
    return (uint32_t)(a ^ b);
#endif
}
// IDENTITY's clamp and the packing of whole outputs: times 256 with saturation two by two, of which the upper bytes are the outputs. 5
// instructions for four of them; the clamp of every one by itself and pack4_perm took 7 (us, 16 x 128 -> 256 28 x 28 3x3 10.22 / 10.13, 34 x 44 ->
// 60 67 x 67 16.17 / 16.07; with mode 4 15 for 19, 32 x 64 -> 64 56 x 56 pointwise 5.71 / 5.35).
__device__ __forceinline__ uint32_t pack4_clamp(int a, int b, int c, int d) {
    uint32_t ab = pack2_sat(a, b), cd = pack2_sat(c, d);
#ifndef MG_HOST_AUDIT
    asm("v_pk_mad_i16 %0, %0, %1, 0 clamp" : "+v"(ab) : "s"(0x01000100));
    asm("v_pk_mad_i16 %0, %0, %1, 0 clamp" : "+v"(cd) : "s"(0x01000100));
#endif
    return pack4_high(ab, cd);
}

// ---- four outputs at a time, without a table ------------------------------------------------------
// v_cvt_pk_u8_f32 rounds to nearest (ties to even), saturates to 0..255 and puts the byte where it
// belongs, which makes the floor, the clamp and the byte shuffling of the forms above unnecessary. In RELU's
// (and H_SWISH's) case the byte is 2 out (+ 1): 0..255 covers 0..127.5, and the one bit that is dropped
// afterwards turns the rounding into a floor; in IDENTITY's it is out + 128. The value converted is
//     mode 1: fma((float)a, c, d)              mode 2: fma(((float)a * s1) * s2, c, d)
// - mode 2 repeats the reference's own first two roundings (or one of them: s2 = 1) and finds constants
// where mode 1 has none (many input channels: c is small, and so is the room between the steps). All of
// it is non-decreasing in a, so it equals the reference on all of int32 iff it does on both sides of each
// of its steps: the host search (requant_table.hip) checks exactly that. (IDENTITY has no mode 2.)
//     mode 4 (IDENTITY): requant_conv_affine's pair, which more scales have - the 128 cost the sum one bit.
//     mode 6 (IDENTITY): trunc(fma(x, c, copysign(d, x))) with mode 2's x: half away from zero is one function of the magnitude, so an
// exact tie is a step like any other, and only the steps of one sign bound c and d. Most of IDENTITY's scales that have neither of
// the above up to a K of a thousand (300 input channels, calibrated scales: 116 of 157).
//     mode 3: the reference's own sequence, for scales with exact ties whose roundings land on either side and for
// H_SWISH. Its division costs two instructions: with c + d the 48-bit reciprocal of s_dst, v = fma(x, c, x d) is
// the quotient to 2^-47 before its one rounding, so it is the correctly rounded one but for quotients that close
// to halfway between two floats, where it is the float on the other side; the host checks every accumulator
// whose output that could change. Half away from zero is then exact for every float: truncation of v plus the
// largest float below a half, and for outputs that are never negative the conversion of 2 v plus that float
// (ties to even: 2 v + 0.5 of v = k + 0.5 is 2 k + 1.5, which goes to the even 2 k + 2).
//     mode 5: mode 1 without its conversion, for kernels whose sums start from requant_bias(): the bits of the sum are then
// those of the float 1.5 * 2^23 + a + m as long as |a + m| < 2^22, where all steps lie (it is asked for), and beyond
// that floats that still grow with a. d is about 10^4 / c of its last bit there, too coarse to put it between the
// steps; the whole number m, a few hundred at most, shifts them until a float falls there.
// Vector instructions for four outputs: 10 (mode 5), 14, 18 - 22, 15 (mode 4), 29 (mode 6), and mode 3 30 (RELU), 37 (IDENTITY), 46 (H_SWISH); the
// threshold table's look-ups took 35 (H_SWISH 51) and four gathers from LDS, and its 1 KB among a launch's
// arguments 0.7 us of the host's time.
// (mode 0: none of these was proven; s1, s2, c are then the reference's three scales, for requant_conv)
struct RequantPack {
    float s1, s2, c, d;
    int mode;
    bool affine() const { return mode != 0 && mode != 3; }
};
// `affine`: any mode, else 3 or 0
RequantPack requant_pack_for(int act, float s_src, float s_flt, float s_dst, bool affine);
// mode 5, or mode 0 where it has no constants
RequantPack requant_shifted_for(int act, float s_src, float s_flt, float s_dst);
// for kernels whose sums start from requant_start(): mode 5 where there is one, else 2, 4, 6, 3 or 0 (mode 1 as mode 2 with products by
// one); `affine` as above
RequantPack requant_started_for(int act, float s_src, float s_flt, float s_dst, bool affine);
// A bias for mode 5. Clamped: sums of a few thousand products on top of +-2^29 have the outputs of the largest and the smallest sums.
__device__ __forceinline__ int requant_bias(int bias, const RequantPack& q) {
    return (bias > (1 << 29) ? 1 << 29 : bias < -(1 << 29) ? -(1 << 29) : bias) + __builtin_bit_cast(int, q.s1);
}
__device__ __forceinline__ int requant_start(int bias, const RequantPack& q) {
    return q.mode == 5 ? requant_bias(bias, q) : bias;  // (uniform)
}
// what a launch uses: modes 1, 2, 4 and 6 unless the switch "noaffine" is on (a launch with them is noted as "+affine")
RequantPack requant_pack_pick(int act, float s_src, float s_flt, float s_dst);

// MODE, ACT compile-time; channels (or pixels) 0..3 of one dword
template <int MODE, int ACT>
__device__ __forceinline__ uint32_t requant_pack4(int a0, int a1, int a2, int a3, const RequantPack& q) {
    const int a[4] = {a0, a1, a2, a3};
    uint32_t r = 0;
    if constexpr (MODE == 3) {
        constexpr float HALF = 0x1.fffffep-2f;
        int o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float x = (float)a[i] * q.s1 * q.s2;
            float v = __builtin_fmaf(x, q.c, x * q.d);  // (RELU: twice the quotient)
            if (ACT == MEGCC_NONLINE_IDENTITY) {
                o[i] = cvt_i32(v + __builtin_copysignf(HALF, v));
                continue;
            }
            if (ACT == MEGCC_NONLINE_H_SWISH)
                v = v * __builtin_amdgcn_fmed3f(v + 3, 0.f, 6.f) * (2.f * (1.f / 6.f));
            r = __builtin_amdgcn_cvt_pk_u8_f32(v + HALF, i, r);
        }
        if (ACT == MEGCC_NONLINE_IDENTITY)
            return pack4_clamp(o[0], o[1], o[2], o[3]);
        return (r >> 1) & 0x7f7f7f7fu;
    } else if constexpr (MODE == 6) {
        int o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float x = (float)a[i] * q.s1 * q.s2;
            o[i] = cvt_i32(__builtin_fmaf(x, q.c, __builtin_copysignf(q.d, x)));
        }
        return pack4_clamp(o[0], o[1], o[2], o[3]);
    } else if constexpr (MODE == 4) {
        // (256 times the value, which changes no rounding: the floor of its floor by 256, and saturation at 16 bits is the clamp)
        const float c = q.c * 256.f, d = q.d * 256.f;
        int o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            o[i] = cvt_floor_i32(__builtin_fmaf((float)a[i], c, d));
        return pack4_high(pack2_sat(o[0], o[1]), pack2_sat(o[2], o[3]));
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float x = MODE == 5 ? __builtin_bit_cast(float, a[i]) : (float)a[i];
            if (MODE == 2)
                x = x * q.s1 * q.s2;
            r = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(x, q.c, q.d), i, r);
        }
        return ACT == MEGCC_NONLINE_RELU ? (r >> 1) & 0x7f7f7f7fu : r ^ 0x80808080u;
    }
}

// N accumulators -> N / 4 dwords (each 4 consecutive ones), the form by a uniform branch. ACT < 0: the literal sequence of
// `act` (mode 0, SIGMOID), whose scales stand where mode 0 has them. STARTED: the sums started from requant_start().
// The empty volatile statement keeps each form inside its branch: the compiler otherwise computes one of them ahead of the
// branch and throws it away, 80 instructions of 120. (On the four constants: on the sums themselves it copied every
// one of them: 16 x 300 -> 300 56 x 56 pointwise 21.6 / 19.9 us, of IDENTITY 23.9 / 22.2, 11 x 296 -> 208 86 x 101 31.6 / 29.7.)
template <int ACT, bool STARTED = false, int N>
__device__ __forceinline__ void requant_dwords(int (&a)[N], uint32_t (&out)[N / 4], const RequantPack& q, int act = ACT) {
    RequantPack p = q;
    auto here = [&]() __attribute__((always_inline)) {
#ifndef MG_HOST_AUDIT
        asm volatile("" : "+s"(p.s1), "+s"(p.s2), "+s"(p.c), "+s"(p.d));
#endif
    };
    if constexpr (ACT < 0) {
#pragma unroll
        for (int i = 0; i < N / 4; ++i) {
            int r[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                r[e] = requant_conv_rt(act, a[4 * i + e], q.s1, q.s2, q.c);
            out[i] = pack4_perm(r[0], r[1], r[2], r[3]);
        }
    } else if constexpr (ACT == MEGCC_NONLINE_H_SWISH) {
#pragma unroll
        for (int i = 0; i < N / 4; ++i)
            out[i] = requant_pack4<3, ACT>(a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3], q);
    } else if (q.mode == (STARTED ? 5 : 1)) {  // (uniform)
        here();
#pragma unroll
        for (int i = 0; i < N / 4; ++i)
            out[i] = requant_pack4<STARTED ? 5 : 1, ACT>(a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3], p);
    } else if (ACT == MEGCC_NONLINE_RELU ? q.mode == 2 : q.mode == 4) {
        here();
#pragma unroll
        for (int i = 0; i < N / 4; ++i)
            out[i] = requant_pack4<ACT == MEGCC_NONLINE_RELU ? 2 : 4, ACT>(a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3], p);
    } else if (ACT == MEGCC_NONLINE_IDENTITY && q.mode == 6) {
        here();
#pragma unroll
        for (int i = 0; i < N / 4; ++i)
            out[i] = requant_pack4<6, ACT>(a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3], p);
    } else {
        here();
#pragma unroll
        for (int i = 0; i < N / 4; ++i)
            out[i] = requant_pack4<3, ACT>(a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3], p);
    }
}

// One form for a whole epilogue: f(form) in the branch of q's mode, form(a0, a1, a2, a3) -> dword. For epilogues of many separate
// dwords, whose every one had the branches in front of it (64 x 64 outputs a wave: sixteen times; 34 x 44 -> 60 67 x 67 3x3 17.4 / 16.1 us).
template <int MODE, int ACT>
struct RequantForm {
    RequantPack q;
    int act;
    __device__ __forceinline__ uint32_t operator()(int a0, int a1, int a2, int a3) const {
        if constexpr (MODE < 0)
            return pack4_perm(requant_conv_rt(act, a0, q.s1, q.s2, q.c), requant_conv_rt(act, a1, q.s1, q.s2, q.c),
                              requant_conv_rt(act, a2, q.s1, q.s2, q.c), requant_conv_rt(act, a3, q.s1, q.s2, q.c));
        else
            return requant_pack4<MODE, ACT>(a0, a1, a2, a3, q);
    }
};
template <int ACT, typename F>
__device__ __forceinline__ void requant_by_form(const RequantPack& q, int act, F f) {
    RequantPack p = q;
    auto here = [&]() __attribute__((always_inline)) {
#ifndef MG_HOST_AUDIT
        asm volatile("" : "+s"(p.s1), "+s"(p.s2), "+s"(p.c), "+s"(p.d));  // (as in requant_dwords)
#endif
    };
    if constexpr (ACT < 0) {
        f(RequantForm<-1, ACT>{p, act});
    } else if constexpr (ACT == MEGCC_NONLINE_H_SWISH) {
        f(RequantForm<3, ACT>{p, act});
    } else if (q.mode == 1) {  // (uniform)
        here();
        f(RequantForm<1, ACT>{p, act});
    } else if (ACT == MEGCC_NONLINE_RELU ? q.mode == 2 : q.mode == 4) {
        here();
        f(RequantForm<ACT == MEGCC_NONLINE_RELU ? 2 : 4, ACT>{p, act});
    } else if (ACT == MEGCC_NONLINE_IDENTITY && q.mode == 6) {
        here();
        f(RequantForm<6, ACT>{p, act});
    } else {
        here();
        f(RequantForm<3, ACT>{p, act});
    }
}

// The same for kernels whose sums started from requant_start(), RELU.
template <typename F>
__device__ __forceinline__ void requant_by_started_form(const RequantPack& q, F f) {
    constexpr int RELU = MEGCC_NONLINE_RELU;
    RequantPack p = q;
    auto here = [&]() __attribute__((always_inline)) {
#ifndef MG_HOST_AUDIT
        asm volatile("" : "+s"(p.s1), "+s"(p.s2), "+s"(p.c), "+s"(p.d));  // (as in requant_dwords)
#endif
    };
    if (q.mode == 5) {  // (uniform)
        here();
        f(RequantForm<5, RELU>{p, RELU});
    } else if (q.mode == 2) {
        here();
        f(RequantForm<2, RELU>{p, RELU});
    } else {
        here();
        f(RequantForm<3, RELU>{p, RELU});
    }
}

// fp32_to_int8(sum * sdiv) (RELU: of max(sum, 0) * sdiv) of 4 N sums, QADD's and QFUSE_ADD_RELU's last step (elemwise.hip). RELU's
// is never negative where sdiv is not, and the conversion above serves: 3 vector instructions a value for 6.
template <bool RELU, int N>
__device__ __forceinline__ void requant_sums(float (&sum)[4 * N], uint32_t (&out)[N], float sdiv) {
    if (RELU && (int)__builtin_bit_cast(unsigned, sdiv) > 0) {  // (uniform; the sign and what is no number, without a vector compare)
#pragma unroll
        for (int i = 0; i < N; ++i) {
            uint32_t r = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#ifndef MG_HOST_AUDIT
                asm volatile("" : "+v"(sum[4 * i + e]));  // (as in requant_dwords)
#endif
                r = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(sum[4 * i + e] * sdiv, 2.f, 0x1.fffffep-2f), e, r);
            }
            out[i] = (r >> 1) & 0x7f7f7f7fu;
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            int r[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float s = sum[4 * i + e];
                r[e] = fp32_to_int8((RELU ? (s > 0 ? s : 0) : s) * sdiv);
            }
            out[i] = pack4_perm(r[0], r[1], r[2], r[3]);
        }
    }
}

// host side: the estimate above is valid (else kernels use the literal sequence per element)
static inline bool requant_table_ok(float s_src, float s_flt, float s_dst) {
    const RequantFast q = make_requant_fast(s_src, s_flt, s_dst);
    return q.c != 0.f && q.c * 2147483648.f > 1000.f;
}

__device__ __forceinline__ uint32_t pack4(int a, int b, int c, int d) {
    return (uint32_t)(a & 0xff) | ((uint32_t)(b & 0xff) << 8) | ((uint32_t)(c & 0xff) << 16) |
           ((uint32_t)(d & 0xff) << 24);
}

__device__ __forceinline__ int sbyte(uint32_t w, int i) {
    return (int)(int8_t)(w >> (8 * i));
}

// an f32 layer's activation
__device__ __forceinline__ float f32_act(int act, float x) {
    switch (act) {
        case MEGCC_NONLINE_RELU: return act_apply<MEGCC_NONLINE_RELU>(x);
        case MEGCC_NONLINE_H_SWISH: return act_apply<MEGCC_NONLINE_H_SWISH>(x);
        case MEGCC_NONLINE_SIGMOID: return act_apply<MEGCC_NONLINE_SIGMOID>(x);
        default: return x;
    }
}

}  // namespace mg
