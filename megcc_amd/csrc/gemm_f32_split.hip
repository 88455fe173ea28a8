// f32 MatMul of any transposition by v_mfma_f32_32x32x16_bf16 at f32 accuracy.
//
// What bounds the f32 kernel (gemm_f32.hip) on a large product is the rate of the f32 matrix instructions, a
// sixteenth of the bf16 ones'. An f32 value has 24 significant bits and is exactly the sum of three bf16 values,
// x = x1 + x2 + x3 (x1 = x rounded to bf16, x2 = the rest rounded, x3 = what is left: 7 bits or fewer). Of the
// nine products of two such sums six are multiplied - all but a2 b3, a3 b2, a3 b3, which are below 2^-26 of a b,
// a quarter of what rounding one f32 product costs - each of them exact in f32.
//   * Error of the sums. An instruction rounds the running sum once per 16 steps of K where the f32 instruction
//     does so 8 times, but there are six of them. So K up to 512 keeps the five small products in a sum of their own
//     (a rounding of it costs 2^-8), and beyond that one running sum is closed every 128 steps into a second set of
//     registers. Against 64 bits, relative error here / by the f32 instructions (gemm_f32.hip, the same operands):
//     4096^3 2.0e-7 / 4.1e-7, 2048^3 1.8e-7 / 4.1e-7, K = 768 1.7e-7 / 5.0e-7, 333 0.9e-7 / 3.3e-7, 64 0.5e-7 / 1.4e-7.
//   * The decomposition is exact, and no infinity appears on the way, for zero and for 2^-102 <= |x| < 2^60. A
//     workgroup looks at every value it splits, asks after the first stage and every chain of 8 (K up to 512, whose sum of
//     small products runs through, is one chain) whether one lay outside, and then multiplies the rest from that chain
//     on with v_mfma_f32_32x32x2_f32, running sums closed every 512 steps of K: Inf, NaN and extreme values come
//     out as of an f32 product. With such values all over (a soft-max of wide logits; us, here / the f32 kernel):
//     4096^3 1040 / 1080, 2048^3 160 / 155 (gemm_f32_ks), 1999 x 333 x 2500 52 / 54. One, late in every tile: 740 / 1080,
//     121 / 155, and for K up to 512, where it costs both passes, 81 / 54.
//   * Workgroup: 128 x 128 outputs, 4 waves of 64 x 64, 16 steps of K a stage, two stages in LDS (50 KB),
//     the next one's values in registers. Two workgroups share a CU, so that one splits while the other multiplies.
//     A thread fetches 8 steps of K of one row - two 16-byte loads, or 8 dword loads of 256 contiguous bytes a wave
//     where the rows are the contiguous axis - splits them and writes one 16-byte piece per part, just what
//     a lane of the instruction reads: no bank conflicts either way.
//   * Loads are unconditional from clamped rows (their results are not stored); the last K % 16 steps are fetched
//     element by element and masked.
// Measured (us, before: the f32 kernels): 4096^3 1087 -> 709 (194 TFLOP/s of the product, 1.16 PFLOP/s of bf16), 2048^3 139 ->
// 107, 1536^3 100 -> 69, 1999 x 333 x 2500 58 -> 33, 4096 x 77 x 4096 40 -> 28.
// The matrix units are busy 60 % of 4096^3, at the 1.85 GHz the card holds under this load (2.4 without); the
// rest is the split's vector instructions, which both cost issue slots and power.
// Fp32MatMulM4N12.cpp:9-158 is the loop replaced.
#include "common.h"
#include "conv_mfma_i8.h"
#include "f32_parts.h"
#include "gemm_f32_ks.h"
#include "gemm_f32_split.h"

namespace mg {

typedef float sp_v16f __attribute__((ext_vector_type(16)));
typedef float sp_v4f __attribute__((ext_vector_type(4)));
typedef float sp_v2f __attribute__((ext_vector_type(2)));
typedef unsigned sp_v4u __attribute__((ext_vector_type(4)));
typedef __bf16 sp_v2b __attribute__((ext_vector_type(2)));
typedef __bf16 sp_v8b __attribute__((ext_vector_type(8)));

struct SplitParams {
    const float* A;
    const float* B;
    float* C;
    unsigned a_bytes, b_bytes;
    unsigned a_row, a_k, b_row, b_k;  // byte strides: of A's rows / B's columns, and along K
    int M, N, K;
    long ldc;
    XcdOrder xo;
};

static constexpr int SP_T = 128, SP_K = 16;
static constexpr int SP_CHAIN = 8;      // stages per running sum
static constexpr int SP_SHORT_K = 512;  // up to here the five small products have a sum of their own
// an LDS piece: 16 bytes of each of the 128 rows; 64 bytes behind each keep the two halves of a stage, which
// neighbouring threads write, on different banks
static constexpr int SP_PIECE = SP_T * 16 + 64;
static constexpr int SP_OPERAND = 6 * SP_PIECE;  // [part][half of the 16 steps][row]

// one operand's part of a thread: 8 steps of K of one row
template <bool KFAST>
struct SplitSide {
    __amdgpu_buffer_rsrc_t rsrc;
    unsigned off, k_bytes;
    int row, half;

    __device__ __forceinline__ SplitSide(const float* p, unsigned bytes, unsigned row_bytes, unsigned k_stride, int first, int rows) {
        rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00020000);
        row = KFAST ? threadIdx.x >> 1 : threadIdx.x & 127;
        half = KFAST ? threadIdx.x & 1 : threadIdx.x >> 7;
        k_bytes = k_stride;
        off = (unsigned)min(first + row, rows - 1) * row_bytes + (unsigned)(8 * half) * k_stride;
    }
    __device__ __forceinline__ void load(int k0, float (&v)[8]) const {
        if (KFAST) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const sp_v4u t = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off + 16 * i, k0 * 4, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[4 * i + e] = __uint_as_float(t[e]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                v[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)off, (int)((unsigned)(k0 + i) * k_bytes), 0));
        }
    }
    // (steps from K on: the last one's value is fetched instead and dropped)
    __device__ __forceinline__ void load_tail(int k0, int K, float (&v)[8]) const {
        const unsigned base = off - (unsigned)(8 * half) * k_bytes;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = k0 + 8 * half + i;
            const float t = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(base + (unsigned)min(k, K - 1) * k_bytes), 0, 0));
            v[i] = k < K ? t : 0.f;
        }
    }
    // splits the 8 values into LDS
    __device__ __forceinline__ void store(char* lds, const float (&v)[8], PartsRange& range) const {
        sp_v4u part[3];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            sp_v2f x = {v[2 * i], v[2 * i + 1]};
            range.look(x[0], x[1]);
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                const unsigned b = __builtin_bit_cast(unsigned, __builtin_convertvector(x, sp_v2b));
                part[p][i] = b;
                x[0] -= __uint_as_float(b << 16);
                x[1] -= __uint_as_float(b & 0xffff0000u);
            }
        }
#pragma unroll
        for (int p = 0; p < 3; ++p)
            *(sp_v4u*)(lds + (2 * p + half) * SP_PIECE + row * 16) = part[p];
    }
    // the same 8 values as they are: [half][first or second 4 steps][row]
    __device__ __forceinline__ void store_f32(char* lds, const float (&v)[8]) const {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            *(sp_v4f*)(lds + (2 * half + i) * SP_PIECE + row * 16) = sp_v4f{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
    }
};

template <bool AK, bool BK, bool SHORT>
__global__ void __launch_bounds__(256, 2) gemm_f32_split_kernel(SplitParams q) {
    __shared__ __attribute__((aligned(16))) char lds[2][2 * SP_OPERAND];
    __shared__ int beyond;  // some thread has split a value that the parts cannot hold
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    int tx, ty;
    xcd_tile(q.xo, blockIdx.x, blockIdx.y, gridDim.x, gridDim.y, tx, ty);
    const int m0 = ty * SP_T, n0 = tx * SP_T;
    const SplitSide<AK> sa(q.A, q.a_bytes, q.a_row, q.a_k, m0, q.M);
    const SplitSide<BK> sb(q.B, q.b_bytes, q.b_row, q.b_k, n0, q.N);
    const int full = q.K / SP_K;
    const char* const at = &lds[0][0] + (lane >> 5) * SP_PIECE + (wm + (lane & 31)) * 16;
    const char* const bt = &lds[0][0] + SP_OPERAND + (lane >> 5) * SP_PIECE + (wn + (lane & 31)) * 16;

    sp_v16f acc[2][2], sum[2][2];
    auto clear = [&](sp_v16f (&t)[2][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    t[i][j][e] = 0.f;
    };
    clear(acc);
    clear(sum);
    auto close = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    sum[i][j][e] += acc[i][j][e];
                    acc[i][j][e] = 0.f;
                }
    };
    auto multiply = [&](int buf) __attribute__((always_inline)) {
        sp_v8b a[3][2], b[3][2];
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[p][i] = *(const sp_v8b*)(at + buf * (2 * SP_OPERAND) + 2 * p * SP_PIECE + i * 512);
                b[p][i] = *(const sp_v8b*)(bt + buf * (2 * SP_OPERAND) + 2 * p * SP_PIECE + i * 512);
            }
        // (neighbouring instructions add to different sums)
#define MG_SP_MUL(SUM, PA, PB)                                                                              \
    _Pragma("unroll") for (int i = 0; i < 2; ++i) _Pragma("unroll") for (int j = 0; j < 2; ++j) SUM[i][j] = \
            __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[PA][i], b[PB][j], SUM[i][j], 0, 0, 0)
        // Smallest products first: each running sum of what x = x1 + x2 + x3 times a power of two leaves behind is
        // then a float (x3, x2 + x3, x), so selecting values (a one-hot column, a permutation) and products of whole
        // numbers that fit 24 bits are exact, as in f32. x1 + x3 in that order need not be a float.
        sp_v16f(&small)[2][2] = SHORT ? sum : acc;
        MG_SP_MUL(small, 0, 2);
        MG_SP_MUL(small, 2, 0);
        MG_SP_MUL(small, 1, 1);
        MG_SP_MUL(small, 0, 1);
        MG_SP_MUL(small, 1, 0);
        MG_SP_MUL(acc, 0, 0);
#undef MG_SP_MUL
    };
    float va[8], vb[8];
    PartsRange range;
    range.begin();
    auto split = [&](int buf) __attribute__((always_inline)) {
        sa.store(&lds[buf][0], va, range);
        sb.store(&lds[buf][SP_OPERAND], vb, range);
    };
    // Whether a thread has met such a value: report(), a barrier, reported(). Every thread then reads the same, since
    // at least one more barrier (a stage's) lies in front of the next report().
    auto report = [&]() __attribute__((always_inline)) {
        if (range.beyond())
            beyond = 1;
    };
    auto reported = [&]() __attribute__((always_inline)) {
        return __builtin_amdgcn_readfirstlane(*(volatile int*)&beyond) != 0;
    };
    // Steps of K whose products are in the sums for good: all of a chain, once no value of it has been reported.
    // (SHORT's sum of small products runs through: one chain, nothing is for good before its end.)
    int kept = 0;
    bool f32 = false;
    sa.load(0, va);
    sb.load(0, vb);
    if (threadIdx.x == 0)
        beyond = 0;
    __syncthreads();
    split(0);  // (K is at least two stages)
    sa.load(SP_K, va);
    sb.load(SP_K, vb);
    report();
    __syncthreads();
    f32 = reported();
    for (int s0 = 0; s0 < full && !f32; s0 += SHORT ? full : SP_CHAIN) {
        if (!SHORT && s0) {
            close();
            kept = s0 * SP_K;
        }
        const int s1 = SHORT ? full : min(s0 + SP_CHAIN, full);
        // (the last two rounds fetch and split the last stage again, for no reader, rather than branch)
        for (int s = s0; s < s1; ++s) {
            multiply(s & 1);
            split((s + 1) & 1);
            const int k0 = min(s + 2, full - 1) * SP_K;
            sa.load(k0, va);
            sb.load(k0, vb);
            __syncthreads();
        }
        report();  // (of the stage behind the chain as well)
        __syncthreads();
        f32 = reported();
    }
    if (!f32 && full * SP_K < q.K) {
        sa.load_tail(full * SP_K, q.K, va);
        sb.load_tail(full * SP_K, q.K, vb);
        split(0);  // (every reader of either buffer is behind the loop's last barrier)
        __syncthreads();
        report();
        __syncthreads();
        f32 = reported();
        multiply(0);
    }
    if (f32) {
        // the rest in f32, from the chain on that met the value
        clear(acc);
        if (SHORT)
            clear(sum);
        __syncthreads();  // (a wave may still be in the multiply just above, reading what is written next)
        if (!SHORT) {
            sa.load(kept, va);  // (a chain begins with a whole stage)
            sb.load(kept, vb);
        }
        for (int k0 = kept; k0 < q.K; k0 += SP_K) {
            // (the next stage in flight while this one is multiplied, but for SHORT, whose bf16 loop would spill registers)
            const int buf = (k0 / SP_K) & 1, kf = SHORT ? k0 : k0 + SP_K;
            if (!SHORT) {
                sa.store_f32(&lds[buf][0], va);
                sb.store_f32(&lds[buf][SP_OPERAND], vb);
            }
            if (kf + SP_K <= q.K) {
                sa.load(kf, va);
                sb.load(kf, vb);
            } else if (SHORT || kf < q.K) {
                sa.load_tail(kf, q.K, va);
                sb.load_tail(kf, q.K, vb);
            }
            if (SHORT) {
                sa.store_f32(&lds[buf][0], va);
                sb.store_f32(&lds[buf][SP_OPERAND], vb);
            }
            __syncthreads();
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                // half h of the wave multiplies steps 8 h + 4 c ... + 3 (piece 2 h + c)
                sp_v4f a[2], b[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    a[i] = *(const sp_v4f*)(at + buf * (2 * SP_OPERAND) + ((lane >> 5) + c) * SP_PIECE + i * 512);
                    b[i] = *(const sp_v4f*)(bt + buf * (2 * SP_OPERAND) + ((lane >> 5) + c) * SP_PIECE + i * 512);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
            }
            if ((k0 & 511) == 512 - SP_K)
                close();
        }
    }
    // register e of a tile: row 8 (e / 4) + 4 (lane / 32) + e % 4, column lane % 32
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int n = n0 + wn + j * 32 + (lane & 31);
        if (n >= q.N)
            continue;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + wm + i * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                if (m < q.M)
                    q.C[(size_t)m * q.ldc + n] = acc[i][j][e] + sum[i][j][e];
            }
    }
}

// Against the kernel for few tiles (gemm_f32_ks.hip) on its scale of cycles of the busiest CU: a tile that has a
// CU to itself counts 118 a step of K, two that share one 205, and 12000 to start and store. Both sides
// measured (us): 2048^3 110 here / 139 there, 1536^3 69 / 100, 1824 x 2002 x 2524 152 / 166; 735 x 3147 x 3000 152 /
// 144, 512 x 4096 x 4096 (128 tiles: half the CUs) 183 / 136, 1024 x 1000 x 2048 49 / 46, 640 x 2000 x 1900 92 / 51
// stay there.
static bool split_wins(const GevmArgs& v) {
    const long tiles = ((long)(v.M + SP_T - 1) / SP_T) * ((v.N + SP_T - 1) / SP_T);
    const long per_cu = (tiles + num_cus() - 1) / num_cus();
    return 12000.0 + (double)v.K * (205.0 * (double)(per_cu / 2) + 118.0 * (double)(per_cu & 1)) < gemm_f32_ks_cycles(v);
}

static unsigned side_bytes(long rows, long row, long k, long K) {
    return (unsigned)(4 * ((rows - 1) * row + (K - 1) * k + 1));
}

bool gemm_f32_split_supported(const GevmArgs& v) {
    const long limit = (1L << 31) - 65536;
    return v.K >= 2 * SP_K && 4 * ((long)(v.M - 1) * v.a_rs + (long)(v.K - 1) * v.a_cs + 1) < limit &&
           4 * ((long)(v.K - 1) * v.b_rs + (long)(v.N - 1) * v.b_cs + 1) < limit && (v.a_cs == 1 || v.a_rs == 1) &&
           (v.b_cs == 1 || v.b_rs == 1) && (v.M + SP_T - 1) / SP_T < 65536 && split_wins(v);
}

TinyNNStatus gemm_f32_split_launch(const GevmArgs& v, int ta, int tb) {
    SplitParams q = {};
    q.A = v.A;
    q.B = v.B;
    q.C = v.C;
    q.M = v.M;
    q.N = v.N;
    q.K = v.K;
    q.ldc = v.ldc;
    q.a_row = (unsigned)v.a_rs * 4u;
    q.a_k = (unsigned)v.a_cs * 4u;
    q.b_row = (unsigned)v.b_cs * 4u;
    q.b_k = (unsigned)v.b_rs * 4u;
    q.a_bytes = side_bytes(v.M, v.a_rs, v.a_cs, v.K);
    q.b_bytes = side_bytes(v.N, v.b_cs, v.b_rs, v.K);
    const dim3 grid((unsigned)((q.N + SP_T - 1) / SP_T), (unsigned)((q.M + SP_T - 1) / SP_T));
    q.xo = options().no_xcdorder ? XcdOrder{0} : make_xcd_order((int)grid.x, (int)grid.y, 4L * (q.M + q.N) * q.K);
    note_kernel("gemm_f32_split", SP_T, SP_T, q.xo.w);
#define MG_SP_K(AK_, BK_) (v.K <= SP_SHORT_K ? gemm_f32_split_kernel<AK_, BK_, true> : gemm_f32_split_kernel<AK_, BK_, false>)
    void (*kern)(SplitParams) = !ta ? (tb ? MG_SP_K(true, true) : MG_SP_K(true, false))
                                    : (tb ? MG_SP_K(false, true) : MG_SP_K(false, false));
#undef MG_SP_K
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, stream(), q);
    return check_launch("gemm_f32_split");
}

}  // namespace mg
