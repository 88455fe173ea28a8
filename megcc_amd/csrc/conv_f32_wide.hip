// f32 NCHW dense convolution of many pixels on the matrix cores (v_mfma_f32_32x32x2_f32, v_mfma_f32_16x16x4_f32): rows = output
// channels, columns = output pixels, K = (ic, fh, fw).
//
// gemm_f32_ks.hip gives every 32 x 32 tile a workgroup of its own, whose waves share K: with thousands of tiles each pays for its
// table, its pixels' places, four sets of sums through LDS and two barriers, for 17 steps of K at 15 channels 3x3, and an output of
// 11 channels is multiplied as 32. Here a wave owns 32 pixels and 16, 32 or 64 channels for the whole of K:
//   * one table and one barrier for four waves, sums from the registers to memory;
//   * 16 rows (v_mfma_f32_16x16x4_f32, two tiles along the pixels) where 32 would be work on rows that are not there;
//   * a step is 4 values of K for every group of lanes (8 or 16 in all): one 16-byte load of the filter a lane and row, four
//     dwords of 32 or 16 neighbouring pixels; four steps in flight, a step's offsets from the table in LDS (written once: byte
//     offset and tap of every k) a step earlier still. A tap outside the image or a k beyond K turns the offset into one
//     beyond the operand, which reads zero and touches nothing. Left to itself the compiler puts the four steps' loads
//     behind their products (64 -> 64 112 x 112 N=16 160 us for 151 with 64 channels).
//   * The last K % 8 (16) values are one more step, masked on both sides (a row's neighbour may hold anything, Inf included).
//   * Running sums are closed every 8 (K up to 63), 16 or 32 values of K. Relative error against 64 bits, gemm_f32_ks.hip / here: 8 -> 9 3x3 0.93e-7 / 0.89e-7,
//     126 -> 74 1x1 1.13e-7 / 0.99e-7, 32 -> 32 3x3 1.59e-7 / 1.12e-7, 96 -> 11 3x3 1.53e-7 / 1.28e-7, 100 -> 128 3x3 1.52e-7 / 1.47e-7; it grows with
//     the number of closings, up to CwPlan's longest K (128 -> 96 3x3 1.55e-7 / 1.74e-7, which is why it stays there).
// Bound: f32 MFMA (by counter 0.43 - 0.67 of the cycles a CU is busy: 96 -> 11 and 64 -> 64 below; profiles/conv_f32_wide__drawn_layers.txt), launch and a wave's prologue for
// short K. Eight steps in flight: no
// faster (96 -> 11 39.7 for 40.0). Fp32Im2col.cpp:88-218 is the loop replaced.
// Measured (us, gemm_f32_ks.hip / here): 3x3 96 -> 11 77 x 77 N=9 39.0 / 29.2, 15 -> 81 83 x 83 N=13 44 / 35, 3 -> 8 112 x 112 N=16 15.4 / 11.4, 7 -> 118
// 83 x 24 N=8 13.0 / 8.6, 64 -> 64 112 x 112 N=16 164 / 154, 52 -> 121 42 x 42 N=7 26 / 23.6; 1x1 126 -> 74 97 x 87 N=5 25.8 / 15.9,
// 86 -> 19 63 x 86 N=10 11.5 / 7.5, 12 -> 107 25 x 88 N=14 12.4 / 8.0, 128 -> 128 112 x 112 N=8 51.6 / 43.6. Of 47 drawn layers the three slowest
// beside it take 2 % longer.
#include "common.h"
#include "conv_geom.h"
#include "conv_mfma_i8.h"
#include "epilogue.h"
#include "gemm_f32_ks.h"

namespace mg {

typedef float cw_v16f __attribute__((ext_vector_type(16)));
typedef float cw_v4f __attribute__((ext_vector_type(4)));
template <int R>
struct CwTile {
    typedef cw_v16f Sums;
    static __device__ __forceinline__ Sums multiply(float a, float b, Sums c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
};
template <>
struct CwTile<16> {
    typedef cw_v4f Sums;
    static __device__ __forceinline__ Sums multiply(float a, float b, Sums c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
};

static constexpr int CW_WAVES = 4, CW_THREADS = 64 * CW_WAVES;

struct CwParams {
    const float* src;
    const float* flt;
    const float* bias;
    float* dst;
    unsigned src_bytes, flt_bytes, plane;  // of an input channel: bytes
    int total, per_xcd;                    // workgroups: in all, of an XCD
    int M, N, K, act;
    int ic, ih, iw, ohw, fh, fw, sh, sw, ph, pw, dh, dw;
    FastDiv d_tiles, d_ohw, d_ow, d_taps, d_fw;  // d_tiles: tiles of output channels
};

// R: side of an output tile; MT, NT: tiles of a wave along the channels, along the pixels; GATHER: a filter of more than 1 x 1 or
// padding; TAIL: K is no whole number of steps; SHORT: sums are closed after every step (MT = 1)
template <int R, int MT, int NT, bool GATHER, bool TAIL, bool SHORT>
__global__ void __launch_bounds__(CW_THREADS, 3) conv_f32_wide_kernel(CwParams q) {
    constexpr int RING = 4;  // steps in flight
    constexpr int H = 64 / R, KS = 4 * H, SUMS = R * R / 64;  // groups of lanes along K, values of K a step, sums of a tile per lane
    typedef typename CwTile<R>::Sums Sums;
    extern __shared__ __attribute__((aligned(16))) float cw_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane / R, c = lane & (R - 1);
    const int place = (int)(blockIdx.x & 7) * q.per_xcd + (int)(blockIdx.x >> 3);
    if (place >= q.total)  // (the whole workgroup)
        return;
    const int block = (int)fdiv(place, q.d_tiles), m0 = (place - block * (int)q.d_tiles.d) * (R * MT);
    const int n0 = (block * CW_WAVES + wave) * (R * NT);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)q.flt, 0, (int)q.flt_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)q.src, 0, (int)q.src_bytes, 0x00020000);
    const unsigned OOB = 0x80000000u;
    const int full = q.K / KS;

    unsigned aoff[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
        aoff[i] = (unsigned)(min(m0 + i * R + c, q.M - 1) * q.K + 4 * h) * 4u;
    // (no bias: some other value, not used)
    const float mine = (q.bias ? q.bias : q.flt)[min(m0 + min(tid, R * MT - 1), q.M - 1)];
    cw_v4f av[RING][MT], bv[RING][NT];
    auto load_a = [&](int s, cw_v4f (&v)[MT]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
            v[i] = __builtin_bit_cast(cw_v4f, __builtin_amdgcn_raw_buffer_load_b128(ra, (int)aoff[i], s * (4 * KS), 0));
    };
    if (full > 0)
#pragma unroll
        for (int r = 0; r < RING; ++r)
            load_a(min(r, full - 1), av[r]);

    // The table, for the workgroup: per k the byte offset and 31 - tap (0 - the bit that is always set - beyond K), in groups of
    // four: 4 offsets, 4 shifts. Behind it the tile's biases.
    int* const tab = (int*)cw_lds;
    float* const bias = cw_lds + (GATHER ? (q.K + KS - 1) / KS * (2 * KS) : 0);
    if (GATHER) {
        const int taps = q.fh * q.fw;
        for (int k = tid; k < (q.K + KS - 1) / KS * KS; k += CW_THREADS) {
            const int ic = (int)fdiv(k, q.d_taps), t = k - ic * taps;
            const int y = (int)fdiv(t, q.d_fw), x = t - y * q.fw;
            const int e = (k >> 2) * 8 + (k & 3);
            tab[e] = ((ic * q.ih + y * q.dh) * q.iw + x * q.dw) * 4;
            tab[e + 4] = k < q.K ? 31 - t : 0;
        }
    }
    // the lane's pixels: byte offset of the first value, a bit per tap outside the image (bit 31 always set), place in the result
    unsigned boff[NT], outside[NT];
    int to[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int p = min(n0 + j * R + c, q.N - 1);
        const int img = (int)fdiv(p, q.d_ohw), rem = p - img * q.ohw;
        const int oh = (int)fdiv(rem, q.d_ow), ow = rem - oh * (int)q.d_ow.d;
        const int ih0 = oh * q.sh - q.ph, iw0 = ow * q.sw - q.pw;
        boff[j] = (unsigned)((((img * q.ic) * q.ih + ih0) * q.iw + iw0) * 4) + (GATHER ? 0u : (unsigned)(4 * h) * q.plane);
        to[j] = img * q.M * q.ohw + rem;
        outside[j] = OOB;
        if (GATHER) {
            unsigned cols = 0;
            for (int x = 0; x < q.fw; ++x)
                cols |= (unsigned)((unsigned)(iw0 + x * q.dw) >= (unsigned)q.iw) << x;
            const unsigned all = (1u << q.fw) - 1;
            for (int y = 0; y < q.fh; ++y)
                outside[j] |= ((unsigned)(ih0 + y * q.dh) < (unsigned)q.ih ? cols : all) << (y * q.fw);
        }
    }
    if (tid < R * MT)
        bias[tid] = q.bias ? mine : 0.f;
    lds_barrier();
    if (n0 >= q.N)
        return;

    // a step's offsets and taps (GATHER), and its loads
    struct Step {
        v4i o, sh;
    };
    auto look = [&](int s) __attribute__((always_inline)) -> Step {
        const int* const at = tab + (H * s + h) * 8;
        return GATHER ? Step{*(const v4i*)at, *(const v4i*)(at + 4)} : Step{};
    };
    auto load_b = [&](int s, const Step& t, cw_v4f (&v)[NT]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const unsigned off = GATHER ? (boff[j] + (unsigned)t.o[e]) | ((outside[j] << t.sh[e]) & OOB) : boff[j];
                v[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, (int)off, GATHER ? 0 : (int)((unsigned)(s * KS + e) * q.plane), 0));
            }
    };
    // Running sums, closed into `sum`: with 16 and 32 channels every two steps (SHORT: every step), while the products go to the other set of registers, so that
    // the additions stand between them; with 64 every four (a second set would leave two waves a SIMD for three). 16 channels have
    // two chains a tile, so no chain is longer than 16 (8) or 32 values.
    constexpr int SETS = MT == 1 ? 2 : 1, GROUP = MT == 1 ? (SHORT ? 1 : 2) : RING, CHAINS = R == 16 ? 2 : 1;
    Sums acc[SETS][CHAINS][MT][NT], sum[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < SUMS; ++e)
                sum[i][j][e] = acc[SETS - 1][0][i][j][e] = acc[SETS - 1][CHAINS - 1][i][j][e] = 0.f;
    auto multiply = [&](const cw_v4f (&a)[MT], const cw_v4f (&b)[NT], int set, bool first) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[set][e % CHAINS][i][j] = CwTile<R>::multiply(a[i][e], b[j][e], first && e < CHAINS ? Sums{} : acc[set][e % CHAINS][i][j]);
    };
    auto close = [&](int set) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < SUMS; ++e)
                    sum[i][j][e] += CHAINS == 2 ? acc[set][0][i][j][e] + acc[set][CHAINS - 1][i][j][e] : acc[set][0][i][j][e];
    };
    // what lies behind the last whole step, element by element: beyond K zeros on both sides
    cw_v4f at[MT], bt[NT];
    if (TAIL) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int k = full * KS + 4 * h + e;
                at[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra, (int)(k < q.K ? aoff[i] + (unsigned)(full * KS + e) * 4u : OOB), 0, 0));
            }
        if (GATHER) {
            load_b(full, look(full), bt);
        } else {
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int k = full * KS + 4 * h + e;
                    bt[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, (int)(k < q.K ? boff[j] + (unsigned)(full * KS + e) * q.plane : OOB), 0, 0));
                }
        }
    }
    Step t = {};  // of the step to load next
    if (full > 0) {
#pragma unroll
        for (int r = 0; r < RING; ++r)
            load_b(min(r, full - 1), look(min(r, full - 1)), bv[r]);
        t = look(min(RING, full - 1));
    }
    __builtin_amdgcn_sched_barrier(0);
    if (SHORT && TAIL)  // (in front of the steps: behind them a rest costs one more rounding of the whole sum, K = 33 0.76e-7 for 0.73e-7)
        multiply(at, bt, SETS - 1, true);
    int s = 0;
    for (; s + RING <= full; s += RING) {
        static_for<RING>([&](auto rc) __attribute__((always_inline)) {
            constexpr int r = decltype(rc)::value, set = r / GROUP % SETS;
            constexpr bool begins = r % GROUP == 0;
            const Step now = t;
            t = look(min(s + RING + r + 1, full - 1));
            multiply(av[r], bv[r], set, begins);
            if (SETS == 2 && begins)
                close(1 - set);
            const int next = min(s + RING + r, full - 1);
            load_a(next, av[r]);
            load_b(next, now, bv[r]);
#ifndef MG_HOST_AUDIT
            // one step stays one step, its address arithmetic (and the sums before) between the products
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // LDS reads
#pragma unroll
            for (int i = 0; i < 4 * MT * NT; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // a product
                __builtin_amdgcn_sched_group_barrier(0x2, (GATHER ? 12 / (4 * MT) + 1 : 1) + (SETS == 2 && begins ? CHAINS * SUMS / 4 : 0), 0);  // vector instructions
            }
            __builtin_amdgcn_sched_group_barrier(0x20, MT + 4 * NT, 0);  // loads
            __builtin_amdgcn_sched_barrier(0);
#endif
        });
        if (SETS == 1)
            close(0);
    }
    if (SETS == 2)
        close(1);
    const bool rest = s < full;
    static_for<RING - 1>([&](auto rc) __attribute__((always_inline)) {
        constexpr int r = decltype(rc)::value;
        if (s + r < full) {
            multiply(av[r], bv[r], 0, SHORT || r == 0);
            if (SHORT)  // (not from the other set's registers: with those in use to the end four waves a SIMD are left for five)
                close(0);
        }
    });
    if (!SHORT && rest)
        close(0);
    if (TAIL && !SHORT) {
        multiply(at, bt, 0, true);
        close(0);
    }
    // register e of a tile: row 8 * (e / 4) + 4 * h + e % 4 (16 x 16: 4 * h + e), column c
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int e4 = 0; e4 < SUMS / 4; ++e4) {
            const int row = i * R + 8 * e4 + 4 * h;
            const cw_v4f b = *(const cw_v4f*)(bias + row);
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const bool there = n0 + j * R + c < q.N;
                float* const out = q.dst + to[j] + (size_t)(m0 + row) * q.ohw;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (there && m0 + row + e < q.M)
                        out[(size_t)e * q.ohw] = f32_act(q.act, sum[i][j][e4 * 4 + e] + b[e]);
            }
        }
}

struct CwPlan {
    int r, mt, nt;
    long shortest, longest;  // K
    double us;               // estimated
};

// Up to this K sums are closed after every step, and rows of 64 begin behind the other: longer chains' error would be larger than that of the four
// waves' shorter ones in gemm_f32_ks.hip, which had these layers before (relative error there / with chains of 16 / here: 32 channels K = 24 0.69e-7 / 0.94e-7 /
// 0.69e-7, 48 0.84 / 0.86 / 0.77, 63 0.88 / 0.92 / 0.82, 12 channels K = 48 0.84 / 0.96 / 0.75, 100 channels K = 72 in rows of 64 0.93 / 1.08, of 32 / 0.90). Such layers
// take up to 4 % longer for it, 40 channels of K = 63, for two tiles of 32 in place of one of 64, 9 (15 x 7 -> 40 62 x 62 11.1 / 12.2 us; 15.6 there).
// (K = 9 of a 1x1 filter alone is left with more than in conv_f32_small.hip, whose waves add two or three values each: 0.63e-7 for 0.61e-7.)
static constexpr long CW_SHORT_K = 63, CW_LONG_CHAINS = 129;

// A workgroup puts one wave on each SIMD of a CU: its MFMAs, 0.45 - 1 us for the
// prologue and end of every set of 256 workgroups, 4 for launch and first operands; pixels that do not
// follow one another cost the loads' way 1.8 times (108 -> 9 87 x 69 stride 2 N=11 23.3 / 23.7, 27 -> 38 86 x 86 stride 2 N=9 14.4 / 14.7). Rows of 16 cost a third more than rows of
// 32, 64 a twentieth less. Estimated / measured us: 96 -> 11 77 x 77 N=9 in rows of 16, 32, 64 26 / 28, 36 / 40, 65 / 63; 15 -> 81 83 x 83 N=13 41 / 43, 30 / 35, 37 / 43;
// 64 -> 64 112 x 112 N=16 188 / 188, 144 / 154, 149 / 151; 6 -> 104 76 x 79 1x1 N=6 7.5 / 7.8, 6.8 / 6.8, 7.4 / 7.5. (64 pixels a wave for 32: 64 ->
// 64 162, 96 -> 11 49; 64 x 64 outputs 174, 74.)
static CwPlan cw_plan(const ConvGeom& g) {
    static const CwPlan kPlans[] = {{32, 1, 1, 1, 640, 0}, {32, 2, 1, CW_LONG_CHAINS, 960, 0}, {16, 1, 2, 1, 1152, 0}};
    const long N = (long)g.n * g.oh * g.ow, K = (long)g.ic * g.fh * g.fw;
    CwPlan best = {0, 0, 0, 0, 0, 1e30};
    const double each = g.sw > 1 && g.fw > 1 ? 1e-3 : 0.56e-3;
    for (CwPlan p : kPlans) {
        const long wgs = ((g.oc + p.r * p.mt - 1) / (p.r * p.mt)) * ((N + CW_WAVES * 32 - 1) / (CW_WAVES * 32));
        const double sets = (double)((wgs + num_cus() - 1) / num_cus());
        p.us = 4.0 + sets * ((p.r == 16 ? 0.5 : p.mt == 1 ? 0.45 : 1.0) + each * (double)K * (p.r == 16 ? 22.0 : p.mt == 1 ? 32.0 : 61.0));
        if (K >= p.shortest && K <= p.longest && p.us < best.us)
            best = p;
    }
    return best;
}

// Fewer pixels than this leave SIMDs without a wave, unless the waves of a workgroup share K (gemm_f32_ks.hip).
static constexpr long CW_MIN_PIXELS = 12288;

// What gemm_f32_ks.hip takes, or the tiled kernel of gemm_f32.hip where that is the quicker one, in us. Here, there;
// estimated / measured: 128 -> 128 56 x 56 N=16 165 / 165, 162 / 153 (stays there), 64 -> 64 112 x 112 N=16 144 / 154, 169 / 165; 24 -> 18 68 x 68
// N=3 6.7 / 7.8, 6.4 / 5.6 (stays); 64 -> 64 56 x 56 N=8 24.6 / 26.5, 29 / 28; 7 -> 118 83 x 24 N=8 6.5 / 8.6, 10 / 13.0; 13 -> 11 82 x 82
// stride 2 N=9 7 / 6.4, 5.4 / 5.4 (stays). The 0.93 where it is used: what both estimates are off by.
static double cw_others(const ConvGeom& g) {
    const long N = (long)g.n * g.oh * g.ow, K = (long)g.ic * g.fh * g.fw;
    const double tiles = (double)((((long)g.oc + 31) / 32 * ((N + 31) / 32) + num_cus() - 1) / num_cus());
    const long big = ((long)g.oc + 127) / 128 * ((N + 127) / 128), per_cu = (big + num_cus() - 1) / num_cus();
    // (up to 16 channels and a long K: its 16 x 16 tiles)
    const double ks = g.oc <= 16 && K >= 250 ? (double)(((N + 15) / 16 + num_cus() - 1) / num_cus()) * ((double)K * 6.2 + 1000.0)
                                             : tiles * (double)K * 11.8 + 1000.0 * (tiles + (tiles < 7.0 ? tiles : 7.0) - 2.0);
    const double tiled = big < 192 ? 1e30 : (double)K * 128.0 * (per_cu == 1 ? 1.55 : 1.14 * (double)per_cu) * 1.7 + 16000.0 * (double)per_cu;
    return 2.5 + (ks < tiled ? ks : tiled) / 2330.0;
}

bool conv_f32_wide_supported(const ConvGeom& g) {
    const long P = (long)g.n * g.oh * g.ow, K = (long)g.ic * g.fh * g.fw;
    return g.fmt == MEGCC_FMT_NCHW && g.groups == 1 && g.fh >= 1 && g.fw >= 1 && g.fh * g.fw <= 31 && K >= 1 && P >= CW_MIN_PIXELS &&
           P < (1L << 30) && (long)g.n * g.ic * g.ih * g.iw < (1L << 29) - 65536 && (long)g.oc * K < (1L << 29) - 65536 && P * g.oc < (1L << 31) &&
           cw_plan(g).us < 0.93 * cw_others(g);
}

template <int R, int MT, int NT, bool SHORT>
static void (*cw_kernel(bool gather, bool tail))(CwParams) {
    return gather ? (tail ? conv_f32_wide_kernel<R, MT, NT, true, true, SHORT> : conv_f32_wide_kernel<R, MT, NT, true, false, SHORT>)
                  : (tail ? conv_f32_wide_kernel<R, MT, NT, false, true, SHORT> : conv_f32_wide_kernel<R, MT, NT, false, false, SHORT>);
}

TinyNNStatus conv_f32_wide_launch(const ConvGeom& g, const void* src, const void* flt, const void* bias, void* dst) {
    CwParams q = {};
    q.src = (const float*)src;
    q.flt = (const float*)flt;
    q.bias = (const float*)bias;
    q.dst = (float*)dst;
    q.M = g.oc;
    q.ohw = g.oh * g.ow;
    q.N = g.n * q.ohw;
    q.K = g.ic * g.fh * g.fw;
    q.act = g.act;
    q.flt_bytes = (unsigned)((long)g.oc * q.K * 4);
    q.src_bytes = (unsigned)((long)g.n * g.ic * g.ih * g.iw * 4);
    q.plane = (unsigned)(g.ih * g.iw) * 4u;
    q.ic = g.ic, q.ih = g.ih, q.iw = g.iw;
    q.fh = g.fh, q.fw = g.fw, q.sh = g.sh, q.sw = g.sw, q.ph = g.ph, q.pw = g.pw, q.dh = g.dh, q.dw = g.dw;
    const CwPlan p = cw_plan(g);
    const int tiles = (q.M + p.r * p.mt - 1) / (p.r * p.mt), wide = CW_WAVES * p.r * p.nt;
    q.total = tiles * ((q.N + wide - 1) / wide);
    q.per_xcd = (q.total + 7) / 8;
    q.d_tiles = make_fastdiv((uint32_t)tiles);
    q.d_ohw = make_fastdiv((uint32_t)q.ohw);
    q.d_ow = make_fastdiv((uint32_t)g.ow);
    q.d_taps = make_fastdiv((uint32_t)(g.fh * g.fw));
    q.d_fw = make_fastdiv((uint32_t)g.fw);
    const bool gather = !(g.fh == 1 && g.fw == 1 && g.ph == 0 && g.pw == 0);
    const int ks = p.r == 32 ? 8 : 16;
    const bool tail = q.K % ks != 0;
    const bool brief = q.K <= CW_SHORT_K && q.K >= 2 * ks;  // (below two steps there is one chain and the rest)
    void (*const kern)(CwParams) = p.r == 16   ? (brief ? cw_kernel<16, 1, 2, true>(gather, tail) : cw_kernel<16, 1, 2, false>(gather, tail))
                                   : p.mt == 1 ? (brief ? cw_kernel<32, 1, 1, true>(gather, tail) : cw_kernel<32, 1, 1, false>(gather, tail))
                                               : cw_kernel<32, 2, 1, false>(gather, tail);
    const size_t lds = (gather ? (size_t)(q.K + ks - 1) / ks * ks * 8 : 0) + (size_t)p.r * p.mt * 4;
    note_kernel("conv_f32_wide", p.r * p.mt, p.r * p.nt);
    hipLaunchKernelGGL(kern, dim3((unsigned)(8 * q.per_xcd)), dim3(CW_THREADS), lds, stream(), q);
    return check_launch("conv_f32_wide");
}

}  // namespace mg
