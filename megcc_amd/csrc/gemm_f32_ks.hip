// f32 products with too few output tiles for the tiled kernel of gemm_f32.hip, on the matrix cores
// (v_mfma_f32_32x32x2_f32): MatMul of any transposition and NCHW dense convolution (rows = output
// channels, columns = output pixels, K = (ic, fh, fw)).
//
// What bounds such a product is how few workgroups its 128 x 128 tiles are and, behind a split of K over
// workgroups, a second kernel that adds the slices. Here a workgroup owns ONE tile of 32 MT x 32 NT outputs
// and its waves share K: the tile is small, so there are enough of them for every CU, and the partial sums
// meet in LDS at the end of the same launch.
//   * No wave multiplies what another one does, so nothing is staged: operands go from memory to the
//     registers the MFMA reads. A step is 8 values of K: lane half h holds k = 8 s + 4 h + i for the MFMA i
//     of the step (any assignment of K to the two halves gives the same products as long as both operands
//     use it), so an operand that is contiguous along K is one 16-byte load per lane and step, one that is
//     contiguous along its rows is four dword loads of 128 contiguous bytes per half wave.
//   * RING steps are in flight per wave; all loads are unconditional buffer loads (offsets beyond the
//     operand's bytes read zero and touch nothing).
//   * Convolution: the column of a lane is a pixel; the offset of k = (ic, fh, fw) in the image and the tap
//     it belongs to come from a table in LDS the workgroup makes once; a tap outside the image turns the
//     offset into an out-of-range one with one shift and one and-or.
//   * The last K % 8 values are one more step of one wave, fetched element by element at the start and
//     masked on both sides (a row's neighbour may hold anything, Inf included).
// Sums: a wave closes its running sums every 64 values of K into a second set of registers; the waves' sums are
// added in wave order. (Without that, relative error against 64 bits of 64 x 4096 x 4096 4.1e-7, of 197 x 771 x 1003
// 2.5e-7, where the tiled kernel's slices of K had 3.0e-7 and 1.7e-7.) Fp32MatMulM4N12.cpp:9-158, Fp32Im2col.cpp:88-218 are the loops replaced.
// Measured (us, before: the tiled kernel with its slice sums in a second launch, or conv_f32_small.hip):
// 64 x 4096 x 4096 35.4 -> 24.0 (2.9 TB/s and 90 TFLOP/s), 197 x 771 x 1003 nt 19.9 -> 7.5,
// 8 x 284 x 736 16.5 -> 4.0, 1623 x 3660 x 316 73 -> 41; convolution 32 -> 32 on 56 x 56 6.9 -> 5.1, N=8
// 64 -> 64 on 56 x 56 55 -> 29, N=8 128 -> 128 165 -> 82.
#include "common.h"
#include "conv_geom.h"
#include "conv_mfma_i8.h"
#include "epilogue.h"
#include "gemm_f32_ks.h"

namespace mg {

typedef float ks_v16f __attribute__((ext_vector_type(16)));
typedef float ks_v4f __attribute__((ext_vector_type(4)));

enum { KS_CONTIG = 0, KS_STRIDED = 1, KS_CONV = 2, KS_CONV1 = 3 };  // along K: contiguous, strided, gathered, 1x1 filter

struct KsParams {
    const float* A;
    const float* B;
    float* C;
    const float* bias;
    unsigned a_bytes, b_bytes;
    unsigned a_row, a_k, b_row, b_k;  // byte strides: of A's rows / B's columns, and along K
    int M, N, K, ldc;
    int act;
    // convolution
    int ic, ih, iw, ow, ohw, fh, fw, sh, sw, ph, pw, dh, dw;
    FastDiv d_ohw, d_ow, d_taps, d_fw;
    XcdOrder xo;
};

__device__ __forceinline__ float ks_act(int act, float x) {
    switch (act) {
        case MEGCC_NONLINE_RELU: return act_apply<MEGCC_NONLINE_RELU>(x);
        case MEGCC_NONLINE_H_SWISH: return act_apply<MEGCC_NONLINE_H_SWISH>(x);
        case MEGCC_NONLINE_SIGMOID: return act_apply<MEGCC_NONLINE_SIGMOID>(x);
        default: return x;
    }
}

static constexpr int KS_MAX_WAVES = 8;
static constexpr int KS_MAX_CONV_K = 4096;  // table entries (8 bytes each)

template <int AM, int BMODE, int MT, int NT, bool TAIL>
__global__ void __launch_bounds__(64 * KS_MAX_WAVES) gemm_f32_ks_kernel(KsParams q) {
    constexpr int RING = 4;
    constexpr bool GATHER = BMODE == KS_CONV, CONV = GATHER || BMODE == KS_CONV1;
    static_assert(!CONV || NT == 1, "one pixel per lane");
    extern __shared__ __attribute__((aligned(16))) float ks_lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), W = blockDim.x >> 6;
    const int h = lane >> 5, c = lane & 31;
    int tx, ty;
    xcd_tile(q.xo, blockIdx.x, blockIdx.y, gridDim.x, gridDim.y, tx, ty);
    const int m0 = ty * (32 * MT), n0 = tx * (32 * NT);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)q.A, 0, (int)q.a_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)q.B, 0, (int)q.b_bytes, 0x00020000);

    // Whole steps, dealt to the waves RING at a time where K is long - 4 steps are one 128-byte line of an
    // operand that is contiguous along K, fetched by one wave back to back instead of by four waves that
    // drift apart - and one at a time where that would leave waves without work.
    const int full = q.K >> 3;
    const bool lines = full >= 4 * RING * W;
    const int s_wave = lines ? RING : 1, s_ring = lines ? 1 : W;  // step = j0 * W + wave * s_wave + r * s_ring
    const int rounds = full / (RING * W), over = full - rounds * (RING * W);
    const int nj = lines ? rounds * RING + min(max(over - RING * wave, 0), RING)
                         : full > wave ? (full - wave + W - 1) / W : 0;

    // byte offset of (row, k = 4 h) of each operand tile
    unsigned aoff[MT], boff[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
        aoff[i] = (unsigned)min(m0 + i * 32 + c, q.M - 1) * q.a_row + (unsigned)(4 * h) * q.a_k;
    int* const tab = (int*)ks_lds;
    int* const pix = tab + (GATHER ? (q.K + 7) / 8 * 16 : 0);  // [offset, outside, image, place in it][32]
    if (CONV) {
        // The lane's pixel and, for a gather, the table: per k the byte offset and 31 - tap (0 - the bit
        // that is always set - beyond K), in groups of four: 4 offsets, 4 shifts. One wave works out the 32
        // pixels and the others the table: done by every wave, the index arithmetic was half of a small
        // layer's time.
        if (wave == 0 && lane < 32) {
            const int p = min(n0 + lane, q.N - 1);
            const int img = (int)fdiv(p, q.d_ohw), rem = p - img * q.ohw;
            const int oh = (int)fdiv(rem, q.d_ow), ow = rem - oh * q.ow;
            const int ih0 = oh * q.sh - q.ph, iw0 = ow * q.sw - q.pw;
            pix[lane] = (((img * q.ic) * q.ih + ih0) * q.iw + iw0) * 4;
            if (GATHER) {  // a bit per tap that lies outside the image (bit 31 always set)
                unsigned cols = 0, out = 0x80000000u;
                for (int x = 0; x < q.fw; ++x)
                    cols |= (unsigned)((unsigned)(iw0 + x * q.dw) >= (unsigned)q.iw) << x;
                const unsigned all = (1u << q.fw) - 1;
                for (int y = 0; y < q.fh; ++y)
                    out |= ((unsigned)(ih0 + y * q.dh) < (unsigned)q.ih ? cols : all) << (y * q.fw);
                pix[32 + lane] = (int)out;
            }
            pix[64 + lane] = img;
            pix[96 + lane] = rem;
        } else if (GATHER && wave > 0) {
            const int taps = q.fh * q.fw;
            for (int k = tid - 64; k < (q.K + 7) / 8 * 8; k += blockDim.x - 64) {
                const int ic = (int)fdiv(k, q.d_taps), t = k - ic * taps;
                const int y = (int)fdiv(t, q.d_fw), x = t - y * q.fw;
                const int e = (k >> 2) * 8 + (k & 3);
                tab[e] = ((ic * q.ih + y * q.dh) * q.iw + x * q.dw) * 4;
                tab[e + 4] = k < q.K ? 31 - t : 0;
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < NT; ++j)
            boff[j] = (unsigned)min(n0 + j * 32 + c, q.N - 1) * q.b_row + (unsigned)(4 * h) * q.b_k;
    }
    unsigned outside = 0;
    int img = 0, rem = 0;

    auto load_a = [&](int s, ks_v4f (&v)[MT]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            if (AM == KS_CONTIG) {
                v[i] = __builtin_bit_cast(ks_v4f, __builtin_amdgcn_raw_buffer_load_b128(ra, (int)(aoff[i] + (unsigned)s * 32u), 0, 0));
            } else {
                const unsigned o = aoff[i] + (unsigned)s * (8u * q.a_k);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra, (int)(o + (unsigned)e * q.a_k), 0, 0));
            }
        }
    };
    auto load_b = [&](int s, ks_v4f (&v)[NT]) __attribute__((always_inline)) {
        if (GATHER) {
            const v4i o = *(const v4i*)(tab + (2 * s + h) * 8), sh = *(const v4i*)(tab + (2 * s + h) * 8 + 4);
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const unsigned off = (boff[j] + (unsigned)o[e]) | ((outside << sh[e]) & 0x80000000u);
                    v[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, (int)off, 0, 0));
                }
            return;
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            if (BMODE == KS_CONTIG) {
                v[j] = __builtin_bit_cast(ks_v4f, __builtin_amdgcn_raw_buffer_load_b128(rb, (int)(boff[j] + (unsigned)s * 32u), 0, 0));
            } else {
                const unsigned o = boff[j] + (unsigned)s * (8u * q.b_k);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, (int)(o + (unsigned)e * q.b_k), 0, 0));
            }
        }
    };
    ks_v16f acc[MT][NT], sum[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                acc[i][j][e] = sum[i][j][e] = 0.f;
    auto close = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    sum[i][j][e] += acc[i][j][e];
                    acc[i][j][e] = 0.f;
                }
    };
    auto multiply = [&](const ks_v4f (&a)[MT], const ks_v4f (&b)[NT]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
    };

    // the step behind the last whole one, element by element
    ks_v4f at[MT], bt[NT];
    auto tail_k = [&](int e) { return min(full * 8 + 4 * h + e, q.K - 1) - 4 * h; };
    if (TAIL)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                at[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra, (int)(aoff[i] + (unsigned)tail_k(e) * q.a_k), 0, 0));
    ks_v4f av[RING][MT], bv[RING][NT];
    const int s0 = wave * s_wave;
    auto step = [&](int j0, int r) { return min(j0 * W + s0 + r * s_ring, full - 1); };
    if (nj > 0)
        static_for<RING>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            load_a(step(0, r), av[r]);
        });
    if (CONV) {
        __syncthreads();
        boff[0] = (unsigned)pix[c] + (BMODE == KS_CONV1 ? (unsigned)(4 * h) * q.b_k : 0u);
        outside = GATHER ? (unsigned)pix[32 + c] : 0u;
        img = pix[64 + c];
        rem = pix[96 + c];
    }
    if (TAIL && GATHER)
        load_b(full, bt);
    if (TAIL && !GATHER)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                bt[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, (int)(boff[j] + (unsigned)tail_k(e) * q.b_k), 0, 0));
    if (nj > 0) {
        static_for<RING>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            load_b(step(0, r), bv[r]);
        });
        // (whole groups with nothing under a condition: behind a conditional load the compiler has to assume
        //  fewer loads in flight than there are, and waits for more of them)
        int j0 = 0;
        for (; j0 + 2 * RING <= nj; j0 += RING) {
            static_for<RING>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                multiply(av[r], bv[r]);
                load_a((j0 + RING) * W + s0 + r * s_ring, av[r]);
                load_b((j0 + RING) * W + s0 + r * s_ring, bv[r]);
            });
            if (j0 & RING)
                close();
        }
        for (; j0 < nj; j0 += RING)
            static_for<RING>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                if (j0 + r < nj) {
                    multiply(av[r], bv[r]);
                    if (j0 + r + RING < nj) {
                        load_a(step(j0 + RING, r), av[r]);
                        load_b(step(j0 + RING, r), bv[r]);
                    }
                }
            });
    }
    if (TAIL && wave == (lines ? W - 1 : full % W)) {  // (the wave whose turn it is)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const bool in = full * 8 + 4 * h + e < q.K;
#pragma unroll
            for (int i = 0; i < MT; ++i)
                at[i][e] = in ? at[i][e] : 0.f;
#pragma unroll
            for (int j = 0; j < NT; ++j)
                bt[j][e] = in ? bt[j][e] : 0.f;
        }
        multiply(at, bt);
    }

    // the waves' sums meet in LDS: [wave][tile][register][lane]
    if (CONV)
        __syncthreads();  // (the table's room is used again)
    constexpr int TILE = MT * NT * 1024;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                ks_lds[wave * TILE + ((i * NT + j) * 16 + e) * 64 + lane] = acc[i][j][e] + sum[i][j][e];
    __syncthreads();
    // register e of a tile: row 8 * (e / 4) + 4 * h + e % 4, column c. Wave w finishes registers w, w + W, ...
    for (int r = wave; r < MT * NT * 16; r += W) {
        const int t = r >> 4, e = r & 15, i = t / NT, j = t - i * NT;
        float v = 0.f;
#pragma unroll 4
        for (int w = 0; w < W; ++w)
            v += ks_lds[w * TILE + r * 64 + lane];
        const int m = m0 + i * 32 + 8 * (e >> 2) + 4 * h + (e & 3), n = n0 + j * 32 + c;
        if (m >= q.M || n >= q.N)
            continue;
        if (CONV) {
            q.C[((size_t)img * q.M + m) * q.ohw + rem] = ks_act(q.act, v + (q.bias ? q.bias[m] : 0.f));
        } else {
            q.C[(size_t)m * q.ldc + n] = v;
        }
    }
}

// ---- choice of tile and waves -------------------------------------------------------------------------
struct KsPlan {
    int mt, nt, waves;
    double cost;  // estimated cycles of the busiest CU
};

// Cycles of the busiest CU: its tiles' MFMAs (K / 2 of 64 cycles per 32 x 32 outputs, over four SIMDs) plus
// what its operands cost on their way through the CU's 64-byte-a-cycle port - half of that where a lane's 16
// bytes lie a row apart from its neighbours' - plus a round of latency for every set of workgroups that fits
// it at once. (Fitted: 2048^3 nt measured 248 / 203 / 159 us with tiles of 32x32 / 32x64 / 64x64, this says 238 /
// 208 / 178.)
static KsPlan ks_plan(long M, long N, long K, bool a_contig, bool b_contig, bool conv) {
    KsPlan best = {0, 0, 0, 1e30};
    static const int kResident[] = {0, 5, 3, 0, 2};
    for (int mt = 1; mt <= (conv ? 1 : 2); ++mt)
        for (int nt = 1; nt <= (conv ? 1 : 2); ++nt) {
            const long tiles = ((M + 32 * mt - 1) / (32 * mt)) * ((N + 32 * nt - 1) / (32 * nt));
            const long per_cu = (tiles + num_cus() - 1) / num_cus();
            const double mfma = 8.0 * mt * nt, load = mt * (a_contig ? 3.5 : 2.0) + nt * (b_contig ? 3.5 : 2.0);
            const double cost = (double)per_cu * K * (mfma + load) +
                                (mt * nt == 4 ? 5000.0 : 3000.0) * (double)((per_cu + kResident[mt * nt] - 1) / kResident[mt * nt]);
            if (cost < best.cost * 0.98) {
                // eight waves where a CU has one tile of a long K, or where there are few tiles (64 x 4096 x 4096:
                // 29.5 us with 4, 23.5 with 8, 25.2 with 16; 197 x 771 x 1003: 8.2, 9.8, 9.7)
                const int w = per_cu <= 1 && (K >= 1024 || tiles <= num_cus() / 2) ? 8 : 4;
                best = {mt, nt, w, cost};
            }
        }
    return best;
}

// What the tiled kernel of gemm_f32.hip would take on the same scale: 128 x 128 tiles (4096^3: 1.14 times the
// MFMA cycles, 2048^3, one tile a CU and nothing to overlap with: 1.5 times, 175 us where 64 x 64 tiles take 151; a
// convolution's gather makes it 1.7 times that); it splits K and adds the slices in a second kernel below 192 tiles, where it never won.
static bool ks_wins(long M, long N, long K, bool conv, const KsPlan& p) {
    if (p.mt == 0)
        return false;
    const long tiles = ((M + 127) / 128) * ((N + 127) / 128), per_cu = (tiles + num_cus() - 1) / num_cus();
    if (tiles < 192)
        return true;
    return p.cost < (double)K * 128.0 * (per_cu == 1 ? 1.55 : 1.14 * (double)per_cu) * (conv ? 1.7 : 1.0);
}

template <int AM, int BMODE>
static TinyNNStatus ks_launch(KsParams& q, const KsPlan& p, const char* what) {
    const bool tail = (q.K & 7) != 0;
    constexpr bool CONV = BMODE == KS_CONV || BMODE == KS_CONV1;
#define MG_KS_T(MT_, NT_) (tail ? gemm_f32_ks_kernel<AM, BMODE, MT_, NT_, true> : gemm_f32_ks_kernel<AM, BMODE, MT_, NT_, false>)
    void (*kern)(KsParams);
    if constexpr (CONV)  // (wider tiles never measured better for a convolution)
        kern = MG_KS_T(1, 1);
    else
        kern = p.mt == 1 ? (p.nt == 1 ? MG_KS_T(1, 1) : MG_KS_T(1, 2)) : (p.nt == 1 ? MG_KS_T(2, 1) : MG_KS_T(2, 2));
#undef MG_KS_T
    const dim3 grid((unsigned)((q.N + 32 * p.nt - 1) / (32 * p.nt)), (unsigned)((q.M + 32 * p.mt - 1) / (32 * p.mt)));
    q.xo = options().no_xcdorder ? XcdOrder{0} : make_xcd_order((int)grid.x, (int)grid.y);
    note_kernel(what, p.mt * 32, p.nt * 32, p.waves, q.xo.w);
    size_t lds = (size_t)p.waves * p.mt * p.nt * 4096;
    const size_t table = (BMODE == KS_CONV ? (size_t)(q.K + 7) / 8 * 64 : 0) + (CONV ? 512 : 0);
    if (lds < table)
        lds = table;
    if (lds > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        MG_REQUIRE(e == hipSuccess, TinyNN_ERROR_RUNTIME, "%s: LDS attribute: %s", what, hipGetErrorString(e));
    }
    hipLaunchKernelGGL(kern, grid, dim3(64 * p.waves), lds, stream(), q);
    return check_launch(what);
}

static KsPlan matmul_plan(const GevmArgs& v) {
    return ks_plan(v.M, v.N, v.K, v.a_cs == 1, v.b_cs != 1, false);
}
static KsPlan conv_plan(const ConvGeom& g) {
    return ks_plan(g.oc, (long)g.n * g.oh * g.ow, (long)g.ic * g.fh * g.fw, true, false, true);
}

double gemm_f32_ks_cycles(const GevmArgs& v) {
    return matmul_plan(v).cost;
}

// Rows of B that are contiguous along a long K, few of them: a wave's 32 lanes read 32 lines of one channel's stride,
// and too few CUs share the chain. The tiled kernel's slices of K over the whole chip are faster there (16 x 4096 x
// 1024 nt 25.2 us here, 20.1 there; 64 x 4096 x 2048 31.1 / 25.7; at K = 2500, 16 x 512, 14.1 / 18.9).
static bool long_rows_of_few(const GevmArgs& v) {
    return v.b_cs != 1 && v.K > 3400 && (long)((v.M + 31) / 32) * ((v.N + 31) / 32) <= num_cus() / 2;
}

bool gemm_f32_ks_supported(const GevmArgs& v) {
    if (long_rows_of_few(v))
        return false;
    const long as = 4 * ((long)(v.M - 1) * v.a_rs + (long)(v.K - 1) * v.a_cs + 1);
    const long bs = 4 * ((long)(v.K - 1) * v.b_rs + (long)(v.N - 1) * v.b_cs + 1);
    return v.K >= 1 && as < (1L << 31) - 65536 && bs < (1L << 31) - 65536 && (v.a_cs == 1 || v.a_rs == 1) &&
           (v.b_cs == 1 || v.b_rs == 1) && ks_wins(v.M, v.N, v.K, false, matmul_plan(v));
}

TinyNNStatus gemm_f32_ks_launch(const GevmArgs& v, int ta, int tb) {
    KsParams q = {};
    q.A = v.A;
    q.B = v.B;
    q.C = v.C;
    q.M = v.M;
    q.N = v.N;
    q.K = v.K;
    q.ldc = (int)v.ldc;
    q.a_row = (unsigned)v.a_rs * 4u;
    q.a_k = (unsigned)v.a_cs * 4u;
    q.b_row = (unsigned)v.b_cs * 4u;
    q.b_k = (unsigned)v.b_rs * 4u;
    q.a_bytes = (unsigned)(4 * ((long)(v.M - 1) * v.a_rs + (long)(v.K - 1) * v.a_cs + 1));
    q.b_bytes = (unsigned)(4 * ((long)(v.K - 1) * v.b_rs + (long)(v.N - 1) * v.b_cs + 1));
    const KsPlan p = matmul_plan(v);
    return !ta ? (tb ? ks_launch<KS_CONTIG, KS_CONTIG>(q, p, "gemm_f32_ks") : ks_launch<KS_CONTIG, KS_STRIDED>(q, p, "gemm_f32_ks"))
               : (tb ? ks_launch<KS_STRIDED, KS_CONTIG>(q, p, "gemm_f32_ks") : ks_launch<KS_STRIDED, KS_STRIDED>(q, p, "gemm_f32_ks"));
}

bool conv_f32_ks_supported(const ConvGeom& g) {
    const long P = (long)g.n * g.oh * g.ow, K = (long)g.ic * g.fh * g.fw;
    return g.fmt == MEGCC_FMT_NCHW && g.groups == 1 && g.fh * g.fw <= 31 && K >= 1 && K <= KS_MAX_CONV_K && P >= 1 &&
           P < (1L << 30) && (long)g.n * g.ic * g.ih * g.iw < (1L << 29) - 65536 && (long)g.oc * K < (1L << 29) - 65536 &&
           P * g.oc < (1L << 31) && g.fh * g.fw >= 1 && ks_wins(g.oc, P, K, true, conv_plan(g));
}

TinyNNStatus conv_f32_ks_launch(const ConvGeom& g, const void* src, const void* flt, const void* bias, void* dst) {
    KsParams q = {};
    q.A = (const float*)flt;
    q.B = (const float*)src;
    q.C = (float*)dst;
    q.bias = (const float*)bias;
    q.M = g.oc;
    q.ohw = g.oh * g.ow;
    q.N = g.n * q.ohw;
    q.K = g.ic * g.fh * g.fw;
    q.a_row = (unsigned)q.K * 4u;
    q.a_k = 4u;
    q.a_bytes = (unsigned)((long)g.oc * q.K * 4);
    q.b_bytes = (unsigned)((long)g.n * g.ic * g.ih * g.iw * 4);
    q.act = g.act;
    q.ic = g.ic, q.ih = g.ih, q.iw = g.iw, q.ow = g.ow;
    q.fh = g.fh, q.fw = g.fw, q.sh = g.sh, q.sw = g.sw, q.ph = g.ph, q.pw = g.pw, q.dh = g.dh, q.dw = g.dw;
    q.d_ohw = make_fastdiv(q.ohw);
    q.d_ow = make_fastdiv(g.ow);
    q.d_taps = make_fastdiv(g.fh * g.fw);
    q.d_fw = make_fastdiv(g.fw);
    q.b_k = (unsigned)(g.ih * g.iw) * 4u;
    const KsPlan p = conv_plan(g);
    if (g.fh == 1 && g.fw == 1 && g.ph == 0 && g.pw == 0)
        return ks_launch<KS_CONTIG, KS_CONV1>(q, p, "conv_f32_gemm_ks");
    return ks_launch<KS_CONTIG, KS_CONV>(q, p, "conv_f32_gemm_ks");
}

}  // namespace mg
