// qsi8 dense NCHW44 convolution of any filter size, stride and dilation on the matrix cores
// (v_mfma_i32_32x32x32_i8) without staging: for the layers the LDS-direct kernel (conv_mfma_i8_dma.hip) has no
// variant for or leaves part of the chip idle on.
//
// What bounded those layers was the one-stage kernel's chain - gather a stage, barrier, multiply it with nothing in
// flight - on a handful of 128-pixel tiles, and for more than 9 taps the dot-product kernel's 12 vector instructions
// per 16 multiply-adds. Here nothing goes through LDS on the way in:
//   * a step is one tap of 32 input channels = one MFMA per 32 x 32 outputs. The filter operand of 32 channels is one
//     contiguous KB of the packed filter; the activation operand of 32 pixels is four dwords per lane, pixel = lane,
//     32 lanes on consecutive pixels of one channel group's plane;
//   * a tap outside the image turns the lane's offset into one beyond the tensor, which a buffer load answers with
//     zero; channel groups beyond the last meet zero filter rows, and offsets beyond the tensor read zero too. The
//     whole offset is in the lane's register: the range check sees all of it;
//   * RING steps are in flight per wave;
//   * the waves of a workgroup share K (KW groups) and the pixels (the rest): small layers split K so that every CU
//     has work; the groups' int32 sums meet in LDS, each group finishing its share of the tile.
// Bound by the loads' way through the CU's address and data path (64 x 64 outputs a wave: 64 cycles of it a step for
// 32 of its matrix units; on small layers too, 4 waves' steps of 5 loads each). Measured (us, before: the one-stage
// kernel of conv_mfma_i8.hip, beyond 9 taps conv_dot4.hip; then with steps beyond a wave's share fetched as zeros, the
// table read before the first operand and the arguments where they are used; now): 6 x 88 -> 148 57 x 43 stride 2
// 14.6, 7.1, 5.9 (5.3 with tiles by the rule at conv_gather_i8_launch); 4 x 24 -> 68 98 x 98 stride 2 14.8, 5.7, 4.15; 1 x 356 -> 52 68 x 81
// 21.2, 8.4, 7.5; 1 x 256 -> 256 28 x 28 8.0, 5.6, 4.8; 47 x 104 -> 48 89 x 89 95.8, 50.5, 40.3; 58 x 264 -> 320 70 x 70 stride 2 216, 176,
// 155; 5x5: 1 x 120 -> 280 19 x 19 134, 6.6, 5.6; 60 x 28 -> 20 63 x 63 137, 21.4, 17.0.
// Reference loop: BareMetal/ConvKernel.cpp:305-344.
#include "conv_mfma_i8.h"

namespace mg {

struct GatherParams {
    // (what is read together at the start of the kernel: gather_begin)
    const int8_t* src;
    const int8_t* wp;     // packed filter [chunk][tap][OCP][32], 16-byte halves swapped when (oc >> 3) & 1
    const int32_t* bias;  // [OC] or NULL
    int8_t* dst;
    unsigned src_bytes, wp_bytes;
    int P, OC, steps, taps, lkw;  // steps = chunks * taps; log2 of the groups that share K
    unsigned step_bytes;         // of the packed filter
    unsigned plane, image, row;  // bytes of the source
    int IH, IW, OHW, OW, FW, SH, SW, PH, PW, DH, DW;
    FastDiv dOHW, dOW, dTaps, dFW;
    int act;
    RequantPack rq;
    // (tiles in runs on the XCDs) pixel tiles; whether a channel tile hangs over, which is then behind all the others of
    // its XCD; the number of the others
    int ptiles, ragged;
    FastDiv dOct;
};

// The arguments as the first thing, in one round trip: asked for where they are used, up to four round trips one
// after the other stood in front of the first load.
__device__ __forceinline__ void gather_begin(const GatherParams& q) {
#ifndef MG_HOST_AUDIT
    asm volatile("" ::"s"(q.src), "s"(q.wp), "s"(q.bias), "s"(q.dst), "s"(q.src_bytes), "s"(q.wp_bytes), "s"(q.P), "s"(q.OC), "s"(q.steps), "s"(q.taps),
                 "s"(q.lkw), "s"(q.step_bytes), "s"(q.plane), "s"(q.image), "s"(q.row), "s"(q.IH), "s"(q.IW), "s"(q.OHW), "s"(q.OW), "s"(q.SH), "s"(q.SW),
                 "s"(q.PH), "s"(q.PW), "s"(q.DH), "s"(q.DW), "s"(q.dOHW.mul), "s"(q.dOW.mul), "s"(q.dTaps.mul), "s"(q.dFW.mul), "s"(q.rq.mode));
#endif
}

// ACT: an activation with a requantisation of its own (q.rq), or -1 (the literal sequence of q.act)
static constexpr int GATHER_LOG2_WAVES = 2, GATHER_WAVES = 1 << GATHER_LOG2_WAVES;  // of a workgroup

// RUNS: every XCD has an eighth of the pixel tiles, each with all its channel tiles, in a row (conv_gather_i8_launch); else a
// grid of pixel x channel tiles
template <int MT, int NT, int ACT, bool RUNS>
__global__ void __launch_bounds__(64 * GATHER_WAVES) conv_gather_i8_kernel(GatherParams q) {
    constexpr int RING = 4;  // steps in flight (8: no step faster, 256 -> 256 28 x 28 5.1 us for 5.0, 4 x 24 -> 68 4.9 for 4.2)
    extern __shared__ __attribute__((aligned(16))) int gather_lds[];
    gather_begin(q);
    int* const bias = gather_lds;  // [32 MT]
    int* const parts = bias + 32 * MT;
    const int lane = threadIdx.x & 63, col = lane & 31, kg = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // groups that share K, waves side by side in pixels
    const int kw = 1 << q.lkw, lpw = GATHER_LOG2_WAVES - q.lkw, pw = 1 << lpw;
    const int grp = wave >> lpw, sub = wave & (pw - 1);
    int tx = blockIdx.x, ty = blockIdx.y;
    if constexpr (RUNS) {
        const int xcd = tx & 7, i = tx >> 3, extra = q.ptiles & 7, mine = (q.ptiles >> 3) + (xcd < extra);
        const int first = xcd * (q.ptiles >> 3) + min(xcd, extra), whole = mine * (int)q.dOct.d;
        tx = (int)fdiv(i, q.dOct);
        ty = i - tx * (int)q.dOct.d;
        if (i >= whole) {
            tx = i - whole;
            ty = (int)q.dOct.d;
            if (!q.ragged || tx >= mine)  // (the whole workgroup: an XCD with a pixel tile less)
                return;
        }
        tx += first;
    }
    const int oc0 = ty * (32 * MT), p0 = (tx * pw + sub) * (32 * NT);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)q.src, 0, (int)q.src_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)q.wp, 0, (int)q.wp_bytes, 0x00020000);

    unsigned pix[NT];
    int ih0[NT], iw0[NT], img[NT], rem[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int p = min(p0 + 32 * j + col, q.P - 1);
        img[j] = (int)fdiv(p, q.dOHW);
        rem[j] = p - img[j] * q.OHW;
        const int oh = (int)fdiv(rem[j], q.dOW), ow = rem[j] - oh * q.OW;
        ih0[j] = oh * q.SH - q.PH;
        iw0[j] = ow * q.SW - q.PW;
        pix[j] = (unsigned)img[j] * q.image + (unsigned)kg * 4u * q.plane + (unsigned)ih0[j] * q.row + (unsigned)iw0[j] * 4u;
    }
    unsigned aoff[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int oc = oc0 + 32 * i + col;  // (below OCP, a multiple of every tile height)
        aoff[i] = (unsigned)oc * KROW + (((kg ^ (oc >> 3)) & 1) << 4);
    }
    v4i A[RING][MT], B[RING][NT];
    auto load = [&](int s, v4i (&a)[MT], v4i (&b)[NT]) __attribute__((always_inline)) {
        const bool over = s >= q.steps;
        const int sc = over ? q.steps - 1 : s;
        const int chunk = (int)fdiv(sc, q.dTaps), tap = sc - chunk * q.taps;
        const int fh = (int)fdiv(tap, q.dFW), fw = tap - fh * q.FW;
        const int dy = fh * q.DH, dx = fw * q.DW;
        const unsigned off = (unsigned)chunk * 8u * q.plane + (unsigned)dy * q.row + (unsigned)dx * 4u;
        const int bottom = over ? 0 : q.IH;
#pragma unroll
        for (int i = 0; i < MT; ++i)
            a[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, (int)(aoff[i] + (unsigned)sc * q.step_bytes), 0, 0));
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const bool in = (unsigned)(ih0[j] + dy) < (unsigned)bottom && (unsigned)(iw0[j] + dx) < (unsigned)q.IW;
            const unsigned o = in ? pix[j] + off : 0x80000000u;
#pragma unroll
            for (int c = 0; c < 4; ++c)
                b[j][c] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs, (int)(o + (unsigned)c * q.plane), 0, 0);
        }
    };
    v16i acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                acc[i][j][e] = 0;
    // group g takes steps g, g + kw, ...
    const int mine = (q.steps - grp + kw - 1) / kw;
#pragma unroll
    for (int r = 0; r < RING; ++r)
        load(grp + r * kw, A[r], B[r]);
    // What the outputs need is asked for behind the operands and waits in registers till the products are done.
    int bv = 0;
    if (q.bias && threadIdx.x < 32 * MT)
        bv = q.bias[min(oc0 + (int)threadIdx.x, q.OC - 1)];
    auto multiply = [&](const v4i (&a)[MT], const v4i (&b)[NT]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[i], b[j], acc[i][j], 0, 0, 0);
    };
    int t = 0;
    for (; t + 2 * RING <= mine; t += RING) {
#pragma unroll
        for (int r = 0; r < RING; ++r) {
            multiply(A[r], B[r]);
            load(grp + (t + r + RING) * kw, A[r], B[r]);
        }
    }
    // The last steps one by one: steps beyond the wave's share are neither asked for nor multiplied. (They read nothing,
    // but 18 steps of the 28 x 28 layer of 256 channels went through the CU's address path as 24.)
    for (; t < mine; t += RING) {
#pragma unroll
        for (int r = 0; r < RING; ++r)
            if (t + r < mine) {
                multiply(A[r], B[r]);
                if (t + r + RING < mine)
                    load(grp + (t + r + RING) * kw, A[r], B[r]);
            }
    }
    // [group][wave of it][quad][lane]: a quad is 4 neighbouring channels of the lane's pixel
    constexpr int QUADS = MT * NT * 4;
    if (threadIdx.x < 32 * MT)
        bias[threadIdx.x] = bv;
    if (kw > 1) {
#pragma unroll
        for (int x = 0; x < QUADS; ++x)
            if ((x & (kw - 1)) != grp) {
                const v16i& t = acc[x / (NT * 4)][x / 4 % NT];
                *(v4i*)(parts + ((wave * QUADS + x) * 64 + lane) * 4) =
                        v4i{t[x % 4 * 4], t[x % 4 * 4 + 1], t[x % 4 * 4 + 2], t[x % 4 * 4 + 3]};
            }
    }
    __syncthreads();
    requant_by_form<ACT>(q.rq, q.act, [&](const auto& form) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < QUADS; ++x) {
            if ((x & (kw - 1)) != grp)
                continue;
            const int i = x / (NT * 4), j = x / 4 % NT, e4 = x % 4;
            int s[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                s[e] = acc[i][j][e4 * 4 + e];
            // (the other groups from the one behind this wave's, no question which of them is its own: 256 -> 256 28 x 28 5.05 -> 4.75 us,
            // 512 -> 512 7 x 7 7.0 -> 6.65)
#pragma unroll
            for (int g = 1; g < GATHER_WAVES; ++g) {
                if (g >= kw)
                    break;
                const v4i o = *(const v4i*)(parts + (((((grp + g) & (kw - 1)) * pw + sub) * QUADS + x) * 64 + lane) * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    s[e] += o[e];
            }
            const int oc = oc0 + 32 * i + 8 * e4 + 4 * kg;
            const v4i bq = *(const v4i*)(bias + 32 * i + 8 * e4 + 4 * kg);
            if (oc >= q.OC || p0 + 32 * j + col >= q.P)
                continue;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                s[e] += bq[e];
            ((uint32_t*)q.dst)[((size_t)img[j] * (q.OC >> 2) + (oc >> 2)) * q.OHW + rem[j]] = form(s[0], s[1], s[2], s[3]);
        }
    });
}

size_t conv_mfma_packed_bytes(const ConvGeom& g);

bool conv_gather_i8_supported(const ConvGeom& g) {
    const long P = (long)g.n * g.oh * g.ow, src = (long)g.n * g.ic * g.ih * g.iw;
    return g.fmt == MEGCC_FMT_NCHW44 && g.groups == 1 && (g.ic & 3) == 0 && (g.oc & 3) == 0 && g.ic >= 4 && g.oc >= 4 &&
           g.fh >= 1 && g.fw >= 1 && P >= 1 && P < (1L << 31) - 512 && src < (1L << 31) &&
           // offsets before the first pixel and behind the last stay clear of the tensor's when they wrap
           (long)g.ih * g.iw * 4 * 12 < (1L << 31) && (long)g.fh * g.dh < (1L << 20) && (long)g.fw * g.dw < (1L << 20) &&
           (long)conv_mfma_packed_bytes(g) < (1L << 31) - 65536 && (long)((g.ic + 31) / 32) * g.fh * g.fw < (1L << 22) &&
           (g.oc + 31) / 32 < 65536;
}

// The layers this kernel takes from the LDS-direct one (its variant `picked`), by how many 32 x 32 tiles there are for a CU.
// Measured over 640 3x3 and 5x5 layers of 16 .. 512 channels, 7 x 7 .. 112 x 112, batch 1 .. 64 (us there / here):
//   * the small-layer variants 6 and 7, one 32-channel tile a workgroup: under two tiles a CU (256 -> 256 28 x 28 7.9 / 4.8,
//     128 -> 128 28 x 28 N=4 5.25 / 4.6, 512 -> 512 28 x 28 10.4 / 9.7, 64 -> 64 14 x 14 N=16 5.2 / 3.9; beyond, 256 -> 256 28 x 28 N=3
//     7.7 / 7.9, 512 -> 128 14 x 14 N=24 12.9 / 14.9); with 32 channels both are at a launch's time, 6 slightly below (4.3 / 4.45);
//   * 1 and 4, 128 (or 64) channels by 256 pixels on part of the CUs: under three (140 -> 96 24 x 22 N=8 7.6 / 5.2, 388 -> 80 39 x 39 N=4
//     13.8 / 10.4, 176 -> 96 57 x 68 N=2 8.2 / 6.55, 32 -> 64 56 x 56 N=3 4.8 / 4.6; beyond, 380 -> 112 17 x 16 N=24 13.7 / 14.6, 228 -> 68 37 x
//     43 N=12 11.8 / 13.4, 256 -> 64 28 x 28 N=22 10.4 / 10.9). From 128 channels on, where it is the taller tile that leaves CUs idle, under
//     seven, for up to 36 steps eight (424 -> 344 31 x 31 N=5 19.6 / 16.5, 248 -> 316 50 x 50 N=2 13.7 / 11.4, 64 -> 164 56 x 56 N=3 7.4 / 5.6; 232 -> 204 23 x 23 N=16
//     13.6 / 14.6), with a stride for up to 36 steps only (20 -> 316 28 x 19 N=35 6.4 / 5.4, 124 -> 340 54 x 66 N=6 10.2 / 10.0; 356 -> 184 25 x 25
//     N=53 19.2 / 27.6), and, of 1, under sixteen with 32 input channels (20 -> 208 21 x 21 N=23 6.3 / 5.2, 32 -> 276 23 x 23 N=21 7.5 / 6.2; 20 -> 464
//     19 x 19 N=25 7.7 / 8.1);
//   * 0, 128 by 512, with 32 input channels: under 32 (20 -> 268 31 x 31 N=24 10.4 / 9.0, 28 -> 188 47 x 47 N=19 12.2 / 9.6, 20 -> 76 27 x 35
//     N=55 8.7 / 7.6; beyond, 24 -> 240 55 x 55 N=17 13.2 / 14.4);
//   * 8 and 9, a filter row a stage: under six (128 -> 64 56 x 56 N=5 16.7 / 10.9, 64 -> 60 54 x 48 N=8 10.7 / 9.0, 72 -> 140 23 x 26
//     N=13 16.9 / 14.2; beyond, 172 -> 372 13 x 12 N=27 30.1 / 33.8) and under four (128 -> 32 56 x 56 stride 2 N=23 22.7 / 16.4), with
//     a stride under eight (80 -> 36 65 x 65 stride 2 N=30 20.1 / 17.2, 44 -> 224 42 x 42 15.1 / 12.0; beyond, 156 -> 496 64 x 72 N=4 30.5 /
//     36.3). Rows of 40 pixels and more without a stride, whose patches leave 9 a 128-pixel tile, however many there are (84 -> 116
//     102 x 112 N=9 95.7 / 50.1, 184 -> 192 60 x 60 N=10 92.4 / 54.1, 144 -> 512 97 x 97 N=3 107 / 79, 20 -> 152 110 x 110 N=35 177 / 88).
//     Layers of 48 channels and fewer with fewer tiles than that would gain too (32 -> 32 28 x 28 N=16 7.2 / 4.1) but are what the
//     row-split kernel is tested with.
bool conv_gather_i8_wins(const ConvGeom& g, int picked) {
    const long tiles = (((long)g.n * g.oh * g.ow + 31) / 32) * ((g.oc + 31) / 32), cus = num_cus();
    const int taps = g.fh * g.fw;
    const long steps = (long)((g.ic + 31) / 32) * taps;
    const bool stride = g.sh > 1 || g.sw > 1, wide = !stride && g.iw >= 40;
    switch (picked) {
        case 0: return taps > 1 && steps <= 9 && tiles < 32 * cus;
        case 6: return tiles < 2 * cus && steps > 9;
        case 7: return tiles < 2 * cus;
        case 1:
        case 4:
            return taps > 1 && (tiles < 3 * cus || (g.oc >= 128 && ((steps <= 36 ? tiles < 8 * cus : !stride && tiles < 7 * cus) ||
                                                                   (picked == 1 && tiles < 16 * cus && steps <= 9))));
        case 8: return tiles < 6 * cus && g.ic > 48;
        case 9: return g.ic > 48 ? tiles < (stride ? 8 : 4) * cus || wide : tiles >= 24 * cus && wide;
        default: return false;
    }
}

TinyNNStatus conv_gather_i8_launch(const ConvGeom& g, const void* src, const void* packed, const void* bias, void* dst) {
    GatherParams q = {};
    q.src = (const int8_t*)src;
    q.wp = (const int8_t*)packed;
    q.bias = (const int32_t*)bias;
    q.dst = (int8_t*)dst;
    q.src_bytes = (unsigned)((long)g.n * g.ic * g.ih * g.iw);
    q.wp_bytes = (unsigned)conv_mfma_packed_bytes(g);
    q.OHW = g.oh * g.ow;
    q.OW = g.ow;
    q.P = g.n * q.OHW;
    q.OC = g.oc;
    q.taps = g.fh * g.fw;
    q.steps = (g.ic + 31) / 32 * q.taps;
    q.step_bytes = (unsigned)((g.oc + OC_PAD - 1) / OC_PAD * OC_PAD * KROW);
    q.plane = (unsigned)(g.ih * g.iw) * 4u;
    q.image = (unsigned)(g.ic / 4) * q.plane;
    q.row = (unsigned)g.iw * 4u;
    q.IH = g.ih, q.IW = g.iw, q.FW = g.fw;
    q.SH = g.sh, q.SW = g.sw, q.PH = g.ph, q.PW = g.pw, q.DH = g.dh, q.DW = g.dw;
    q.dOHW = make_fastdiv(q.OHW);
    q.dOW = make_fastdiv(g.ow);
    q.dTaps = make_fastdiv(q.taps);
    q.dFW = make_fastdiv(g.fw);
    q.act = g.act;
    // 64 x 64 outputs a wave where that gives every SIMD one, else less. Groups share K (1300 layers, kw 1, 2 and 4):
    //   * 32 x 32: a long K however many tiles there are (7 x 124 -> 240 29 x 23 11.4 us with one group, 10.4 with four; 256 -> 256
    //     28 x 28 5.6 with four, 6.0 with eight); a shorter one until there are 1.6 waves a SIMD - the second round is then as short
    //     as the first (64 -> 64 28 x 28 N=24 6.5 with one, 5.5 with two, 32 -> 128 14 x 14 5x5 N=24 6.0 with two, 5.3 with four, 3 x 64 ->
    //     64 90 x 90 6.2 with one, 5.3 with two; beyond, 32 -> 128 90 x 90 stride 2 N=8 6.3, 6.1 and, with four, 6.95);
    //   * 64 x 32: the tiles are between one and two for a SIMD, two groups even out the last round (256 -> 256 56 x 56 N=3 19.7 with
    //     one, 15.2 with two, 13.4 with four; 20 -> 404 28 x 28 N=8 6.05, 5.4, 6.7), four where it is nearly empty (96 -> 32 56 x 56 5x5
    //     N=24 24.1, 18.6, 15.7; 1778 tiles, 20 -> 404 90 x 90 5x5 9.6, 8.7, 9.45);
    //   * 64 x 64: two where a SIMD has under four waves (10 x 452 -> 108 75 x 91 77.5 with one, 68.1 with two; 124 -> 240 28 x 28
    //     N=24 18.9, 17.7; 25 steps, 20 -> 404 56 x 56 N=3 11.8, 12.8).
    int mt = g.oc > 32 ? 2 : 1, nt = 2, kw = 1;
    const long full = 4L * num_cus();
    auto tiles = [&] { return (long)((q.P + 32 * nt - 1) / (32 * nt)) * ((g.oc + 32 * mt - 1) / (32 * mt)); };
    if (tiles() < full)
        nt = 1;
    if (tiles() < full)
        mt = 1;
    if (mt * nt == 1) {
        // With four groups a workgroup is one tile, and what bounds it is its CU's data path: 16 accesses of the L1 a step for 32 channels'
        // filter, some 68 for 32 pixels (a dword a lane) - a larger tile is fewer accesses an output, unless its rounds over the
        // CUs cost more. From 80 steps on with pixels too; a shorter K does not hide what the larger tile's sums cost (us 32 x 32 / 64
        // channels x 32 pixels / 64 x 64: 56 x 164 -> 60 18 x 17 5x5 stride 2 20.7 / 13.1 / 22.2, 10 x 428 -> 476 17 x 16 stride 2 17.6 / 11.4 /
        // 18.6, 13 x 196 -> 380 27 x 25 stride 2 16.6 / 10.9 / 10.9, 31 x 484 -> 172 30 x 22 5x5 stride 2 61.0 / 37.9 / 33.6, 9 x 176 -> 460
        // 13 x 13 5x5 16.3 / 14.4 / 13.5, 1 x 176 -> 364 95 x 101 stride 2 10.8 / 8.2 / 8.6; one round either way: 1 x 256 -> 256 28 x 28 4.8 /
        // 5.4 / 7.6; 420 layers of 5 us and more: 6 % in the mean, nothing by more than two runs differ).
        auto port = [&](int m, int n) {
            const long t = (long)((q.P + 32 * n - 1) / (32 * n)) * ((g.oc + 32 * m - 1) / (32 * m));
            return (t + num_cus() - 1) / num_cus() * (16 * m + 68 * n);
        };
        long least = port(1, 1);
        auto consider = [&](int m, int n, int steps) {
            if (q.steps >= steps && (m == 1 || g.oc > 32) && port(m, n) < least)
                least = port(m, n), mt = m, nt = n, kw = 4;
        };
        consider(2, 1, 25);
        consider(2, 2, 80);
        consider(1, 2, 80);
    }
    if (kw > 1) {
        // (as just chosen)
    } else if (mt * nt == 1) {
        while (kw < 4 && q.steps >= 8 * kw && (5 * tiles() * kw < 8 * full || q.steps >= 27))
            kw *= 2;
    } else if (mt * nt == 2) {
        kw = q.steps >= 25 && 4 * tiles() < 5 * full ? 4 : q.steps >= 8 ? 2 : 1;
    } else if (q.steps >= 36 && tiles() < 4 * full) {
        kw = 2;
    }
    // Where the image is more than an XCD's L2 holds, neighbouring pixels - rows of the image that both read - and a pixel
    // tile's channel tiles on one XCD (us without / with: 58 x 264 -> 320 70 x 70 stride 2 171 / 156, 21 x 116 -> 20 47 x 59
    // 10.4 / 8.9, 50 x 192 -> 20 58 x 42 stride 2 12.3 / 10.9, 47 x 104 -> 48 89 x 89 41.9 / 40.8, 10 x 136 -> 20 84 x 84 14.8 /
    // 14.9; in one kernel with the grid's order the arithmetic cost smaller layers 0.1 - 0.2 us). A channel tile that hangs over is the
    // quicker one and fills the last round best, behind the others: 23 x 36 -> 144 87 x 74 31.9 us without, 34.6 with the three side
    // by side, 31.7; 23 x 100 -> 144 48.6, 48.7, 46.0.
    const bool runs = q.src_bytes > (1u << 22) && !options().no_xcdorder;
    const int pw = GATHER_WAVES / kw;
    const int gx = (q.P + 32 * nt * pw - 1) / (32 * nt * pw), gy = (g.oc + 32 * mt - 1) / (32 * mt);
    q.ptiles = gx;
    q.ragged = g.oc % (32 * mt) != 0 && gy > 1;
    q.dOct = make_fastdiv(gy - q.ragged);
    const dim3 grid((unsigned)(runs ? (gx + 7) / 8 * 8 * gy : gx), (unsigned)(runs ? 1 : gy));
#define MG_GATHER_R(MT_, NT_, ACT_) (runs ? conv_gather_i8_kernel<MT_, NT_, ACT_, true> : conv_gather_i8_kernel<MT_, NT_, ACT_, false>)
#define MG_GATHER_A(MT_, NT_)                                                                \
    (q.rq.mode == 0                      ? MG_GATHER_R(MT_, NT_, -1)                         \
     : g.act == MEGCC_NONLINE_IDENTITY   ? MG_GATHER_R(MT_, NT_, MEGCC_NONLINE_IDENTITY)     \
     : g.act == MEGCC_NONLINE_RELU       ? MG_GATHER_R(MT_, NT_, MEGCC_NONLINE_RELU)         \
                                         : MG_GATHER_R(MT_, NT_, MEGCC_NONLINE_H_SWISH))
    q.lkw = kw == 4 ? 2 : kw == 2 ? 1 : 0;
    note_kernel("conv_mfma_i8_gather", 32 * mt, 32 * nt, kw);
    q.rq = requant_pack_pick(g.act, g.s_src, g.s_flt, g.s_dst);
    note_requant_affine(q.rq.affine());
    void (*kern)(GatherParams) = mt == 2 ? (nt == 2 ? MG_GATHER_A(2, 2) : MG_GATHER_A(2, 1))
                                         : (nt == 2 ? MG_GATHER_A(1, 2) : MG_GATHER_A(1, 1));
#undef MG_GATHER_A
#undef MG_GATHER_R
    const size_t lds = 32 * mt * 4 + (kw > 1 ? (size_t)GATHER_WAVES * mt * nt * 4096 : 0);
    if (lds > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        MG_REQUIRE(e == hipSuccess, TinyNN_ERROR_RUNTIME, "conv_gather_i8: LDS attribute: %s", hipGetErrorString(e));
    }
    hipLaunchKernelGGL(kern, grid, dim3(64 * GATHER_WAVES), lds, stream(), q);
    return check_launch("conv_gather_i8");
}

}  // namespace mg
