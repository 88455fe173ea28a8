// qsi8 FullyConnected ([M,K,1,1] x [N,K,1,1]) with any number of rows and any K: a tiled product on
// the matrix cores whose activation rows may start at any byte.
//
// The LDS-direct kernel wants rows that are whole 128-byte blocks and the one-stage kernel wants K to
// be a multiple of 4 (a channel group of NCHW44); a classifier over 491 or 2958 features has neither and
// ran on the one-output-per-thread kernel. Here
//   * the filter comes from the packed copy (K padded with zeros to whole 128-byte blocks, so what the
//     activations hold beyond K does not matter) straight into registers: one contiguous KB per 32
//     channels and 32 bytes of K;
//   * the activations of a block of K (tile rows x 128 bytes) go through LDS, fetched 16 bytes per
//     lane at whatever address the row has (8 lanes read one row's 128 bytes), rows of 128 bytes with
//     their 16-byte pieces at piece ^ (row & 7) so that operand reads of 8 neighbouring rows hit
//     different banks. Two LDS buffers; a block's loads, filter included, are issued before the block
//     ahead of it is multiplied;
//   * a load that would run past the end of the tensor is moved back to its last 16 bytes and the bytes
//     are shifted into place on their way into LDS: every access stays inside the operands;
//   * KW groups of four waves share K between them where the tiles alone would leave the chip idle; their
//     int32 sums meet in LDS (integer: the order does not matter);
//   * the output tile is put together in LDS and leaves as 16-byte row pieces: with an odd N no row
//     starts on a word, and byte stores from the accumulator layout would be 16 times the instructions.
// Bound by latency at the sizes of classifiers (a few blocks of K per workgroup: 225 x 117 x 3611 335 -> 4.8
// us, 2378 x 2958 x 70 799 -> 14.2 us, both from the one-output-per-thread kernel), by operand delivery at
// large ones (4000 x 4001 x 4001: 110 us = 1.16 POP/s).
// Reference loop: BareMetal/ConvKernel.cpp:305-344 on the [M,K,1,1] x [N,K,1,1] layer.
#include "conv_mfma_i8.h"

namespace mg {

struct FcTileParams {
    const int8_t* src;   // [M][K]
    const int8_t* wp;    // packed filter [K/32][OCP][32], 16-byte halves swapped when (oc >> 3) & 1
    const int32_t* bias; // [OC] or NULL
    int8_t* dst;         // [M][OC]
    unsigned last16;     // offset of the last 16 bytes of src
    int M, K, OC, OCP, nblk;  // nblk: blocks of 128 bytes of K
    int act;
    RequantPack rq;
    XcdOrder xo;  // tile order (set at launch from the grid)
};

// MT, NT: 32-channel and 32-row MFMA tiles per wave; a group of four waves makes 64 MT channels x 64 NT rows
template <int MT, int NT, int KW, int ACT>
__global__ void __launch_bounds__(256 * KW) fc_tile_kernel(FcTileParams q) {
    constexpr int BOC = 64 * MT, BR = 64 * NT;
    constexpr int STAGE = BR * 128;                      // bytes of one stage buffer
    constexpr int AL = 2 * NT;                           // 16-byte loads per thread and block
    constexpr int ACC = MT * NT * 16 * 256 * 4;          // bytes of a group's accumulators
    constexpr int OPITCH = BOC + 16;                     // row of the output tile in LDS
    constexpr int NEED0 = KW * 2 * STAGE, NEED1 = (KW - 1) * ACC, NEED2 = BR * OPITCH;
    constexpr int LDS = NEED0 > NEED1 ? (NEED0 > NEED2 ? NEED0 : NEED2) : (NEED1 > NEED2 ? NEED1 : NEED2);
    __shared__ __attribute__((aligned(16))) int8_t lds[LDS];
    const int tid = threadIdx.x & 255, lane = tid & 63;
    const int grp = KW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wn = wave & 1;
    const int col = lane & 31, kg = lane >> 5;
    int tx, ty;
    xcd_tile(q.xo, blockIdx.x, blockIdx.y, gridDim.x, gridDim.y, tx, ty);
    const int oc0 = tx * BOC, row0 = ty * BR;
    int8_t* const stage = lds + grp * (2 * STAGE);

    // activations: thread -> row (tid >> 3) + 32 i, piece tid & 7 of the block
    const int srow = tid >> 3, pc = tid & 7;
    unsigned roff[AL];
#pragma unroll
    for (int i = 0; i < AL; ++i)
        roff[i] = (unsigned)min(row0 + srow + 32 * i, q.M - 1) * (unsigned)q.K + (unsigned)pc * 16u;
    v4i ra[AL];
    auto act_load = [&](int blk) __attribute__((always_inline)) {
        const unsigned b = (unsigned)min(blk, q.nblk - 1) * 128u;
#pragma unroll
        for (int i = 0; i < AL; ++i)
            ra[i] = *(const v4i_any*)(q.src + min(roff[i] + b, q.last16));
    };
    auto act_store = [&](int blk, int buf) __attribute__((always_inline)) {
        const unsigned b = (unsigned)blk * 128u;
#pragma unroll
        for (int i = 0; i < AL; ++i) {
            v4i v = ra[i];
            const unsigned off = roff[i] + b;
            if (off > q.last16)  // (the end of the tensor, or a block beyond K)
                v = fc_tail_piece(v, off - q.last16);
            if (KW > 1 && blk >= q.nblk)
                v = v4i{0, 0, 0, 0};
            *(v4i*)(stage + buf * STAGE + (srow + 32 * i) * 128 + ((pc ^ (srow & 7)) << 4)) = v;
        }
    };
    const int8_t* arow[MT];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
        const int oc = oc0 + wm * (32 * MT) + mi * 32 + col;  // (< OCP: a multiple of every tile width)
        arow[mi] = q.wp + (size_t)oc * KROW + (((kg ^ (oc >> 3)) & 1) << 4);
    }
    const size_t cstep = (size_t)q.OCP * KROW;
    v4i A[2][MT][4];
    auto flt_load = [&](int blk, v4i (&a)[MT][4]) __attribute__((always_inline)) {
        const size_t o = (size_t)(min(blk, q.nblk - 1) * 4) * cstep;
#pragma unroll
        for (int mi = 0; mi < MT; ++mi)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                a[mi][c] = *(const v4i*)(arow[mi] + o + c * cstep);
    };
    v16i acc[MT][NT];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi)
#pragma unroll
        for (int ni = 0; ni < NT; ++ni)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                acc[mi][ni][e] = 0;
    auto multiply = [&](int buf, const v4i (&a)[MT][4]) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            v4i b[NT];
#pragma unroll
            for (int ni = 0; ni < NT; ++ni)
                b[ni] = *(const v4i*)(stage + buf * STAGE + (wn * (32 * NT) + ni * 32 + col) * 128 +
                                      (((c * 2 + kg) ^ (col & 7)) << 4));
#pragma unroll
            for (int mi = 0; mi < MT; ++mi)
#pragma unroll
                for (int ni = 0; ni < NT; ++ni)
                    acc[mi][ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[mi][c], b[ni], acc[mi][ni], 0, 0, 0);
        }
    };

    // group g multiplies blocks g, g + KW, ...; all groups take the same number of steps
    const int steps = (q.nblk + KW - 1) / KW;
    act_load(grp);
    flt_load(grp, A[0]);
    act_store(grp, 0);
    __syncthreads();
    for (int s = 0; s < steps; s += 2) {
        // (two steps per turn: the filter's register set is a compile-time choice)
        const int n1 = grp + (s + 1) * KW, n2 = grp + (s + 2) * KW;
        act_load(n1);
        flt_load(n1, A[1]);
        multiply(0, A[0]);
        act_store(n1, 1);
        __syncthreads();
        if (s + 1 >= steps)
            break;
        act_load(n2);
        flt_load(n2, A[0]);
        multiply(1, A[1]);
        act_store(n2, 0);
        __syncthreads();
    }

    if (KW > 1) {
        int* red = (int*)lds;
        if (grp > 0) {
#pragma unroll
            for (int mi = 0; mi < MT; ++mi)
#pragma unroll
                for (int ni = 0; ni < NT; ++ni)
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        red[(grp - 1) * (ACC / 4) + ((mi * NT + ni) * 16 + e) * 256 + tid] = acc[mi][ni][e];
        }
        __syncthreads();
        if (grp == 0) {
#pragma unroll
            for (int g = 0; g < KW - 1; ++g)
#pragma unroll
                for (int mi = 0; mi < MT; ++mi)
#pragma unroll
                    for (int ni = 0; ni < NT; ++ni)
#pragma unroll
                        for (int e = 0; e < 16; ++e)
                            acc[mi][ni][e] += red[g * (ACC / 4) + ((mi * NT + ni) * 16 + e) * 256 + tid];
        }
        __syncthreads();
    }
    // register e of a tile: channel 8 * (e / 4) + 4 * kg + e % 4, row = the lane's column
    if (grp == 0) {
#pragma unroll
        for (int mi = 0; mi < MT; ++mi)
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                const int ocl = wm * (32 * MT) + mi * 32 + e4 * 8 + kg * 4, oc = oc0 + ocl;
                int bv[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    bv[e] = q.bias ? q.bias[min(oc + e, q.OC - 1)] : 0;
#pragma unroll
                for (int ni = 0; ni < NT; ++ni) {
                    int a[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        a[e] = acc[mi][ni][e4 * 4 + e] + bv[e];
                    uint32_t d[1];
                    requant_dwords<ACT>(a, d, q.rq, q.act);
                    *(uint32_t*)(lds + (wn * (32 * NT) + ni * 32 + col) * OPITCH + ocl) = d[0];
                }
            }
    }
    __syncthreads();
    constexpr int PIECES = BOC / 16;
    for (int i = threadIdx.x; i < BR * PIECES; i += 256 * KW) {
        const int r = i / PIECES, p = i - r * PIECES;
        const int row = row0 + r, oc = oc0 + p * 16;
        if (row >= q.M || oc >= q.OC)
            continue;
        const v4i v = *(const v4i*)(lds + r * OPITCH + p * 16);
        int8_t* o = q.dst + (size_t)row * q.OC + oc;
        if (oc + 16 <= q.OC) {
            *(v4i_any*)o = v;
        } else {
#pragma unroll
            for (int b = 0; b < 15; ++b)
                if (oc + b < q.OC)
                    o[b] = (int8_t)((unsigned)v[b >> 2] >> (8 * (b & 3)));
        }
    }
}

bool fc_tile_supported(const ConvGeom& g) {
    return (long)g.n * g.ic >= 16 && (long)g.n * g.ic < (1L << 31) - 65536 && (long)g.n * g.oc < (1L << 31) && g.oc >= 1;
}

TinyNNStatus fc_tile_launch(const ConvGeom& g, const void* src, const void* packed, const void* bias, void* dst) {
    FcTileParams q = {};
    q.src = (const int8_t*)src;
    q.wp = (const int8_t*)packed;
    q.bias = (const int32_t*)bias;
    q.dst = (int8_t*)dst;
    q.last16 = (unsigned)((long)g.n * g.ic - 16);
    q.M = g.n;
    q.K = g.ic;
    q.OC = g.oc;
    q.OCP = (g.oc + OC_PAD - 1) / OC_PAD * OC_PAD;
    q.nblk = (g.ic + 127) / 128;
    q.act = g.act;
    q.rq = requant_pack_pick(g.act, g.s_src, g.s_flt, g.s_dst);
    // 128 x 128 tiles where they give every CU one; else 64 x 64, with up to four groups of waves sharing
    // K while the groups still have a block each and the chip is not full
    const long big = (long)((g.n + 127) / 128) * ((g.oc + 127) / 128);
    const long small = (long)((g.n + 63) / 64) * ((g.oc + 63) / 64);
    const bool wide = big >= num_cus();
    const int kw = wide || small >= 2L * num_cus() || q.nblk < 2 ? 1 : small >= num_cus() || q.nblk < 4 ? 2 : 4;
    const int act = q.rq.mode ? g.act : -1;
#define MG_FCT(MT_, NT_, KW_)                                                                        \
    (act == MEGCC_NONLINE_IDENTITY ? fc_tile_kernel<MT_, NT_, KW_, MEGCC_NONLINE_IDENTITY>           \
     : act == MEGCC_NONLINE_RELU   ? fc_tile_kernel<MT_, NT_, KW_, MEGCC_NONLINE_RELU>               \
     : act == MEGCC_NONLINE_H_SWISH ? fc_tile_kernel<MT_, NT_, KW_, MEGCC_NONLINE_H_SWISH>           \
                                   : fc_tile_kernel<MT_, NT_, KW_, -1>)
    void (*kern)(FcTileParams) = wide ? MG_FCT(2, 2, 1) : kw == 1 ? MG_FCT(1, 1, 1) : kw == 2 ? MG_FCT(1, 1, 2) : MG_FCT(1, 1, 4);
#undef MG_FCT
    const int b = wide ? 128 : 64;
    const dim3 grid((g.oc + b - 1) / b, (g.n + b - 1) / b);
    q.xo = options().no_xcdorder ? XcdOrder{0} : make_xcd_order((int)grid.x, (int)grid.y, (long)(q.M + q.OC) * q.K);
    note_kernel(q.xo.w ? "fc_tile_xo" : "fc_tile", b, kw);
    note_requant_affine(q.rq.affine());
    hipLaunchKernelGGL(kern, grid, dim3(256 * kw), 0, stream(), q);
    return check_launch("fc_tile");
}

}  // namespace mg
