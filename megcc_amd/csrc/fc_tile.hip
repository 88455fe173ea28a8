// qsi8 FullyConnected ([M,K,1,1] x [N,K,1,1]) with any number of rows and any K: a tiled product on
// the matrix cores whose activation rows may start at any byte.
//
// The LDS-direct kernel wants rows that are whole 128-byte blocks and the one-stage kernel wants K to
// be a multiple of 4 (a channel group of NCHW44); a classifier over 491 or 2958 features has neither. Here
//   * the filter comes from the packed copy (K padded with zeros to whole 128-byte blocks, so what the
//     activations hold beyond K does not matter) straight into registers: one contiguous KB per 32
//     channels and 32 bytes of K;
//   * rows that start at any byte are read as aligned words and the word behind them, and moved into
//     place by the address's last two bits (16-byte loads at odd bytes took half as long again: 1491 x 1457 x 666
//     12.9 us where 1491 x 1460 x 666 took 9.5); of the last row only, a piece that would run past the end of
//     the tensor is moved back to its last 16 bytes and shifted: every access stays in words of the operands;
//   * 128 x 128 and 64 x 64 parts: the activations of a block of K (part rows x 128 bytes) go through LDS, rows of
//     128 bytes with their 16-byte pieces at piece ^ (row & 7) so that operand reads of 8 neighbouring rows
//     hit different banks; two LDS buffers, the next block's loads are out while one is multiplied;
//   * few 64 x 64 parts over a long K: four groups of four waves share K, each with buffers of its own;
//   * 32 x 32 parts: four waves share K, each with a block's activations in 4 KB of LDS of its own; their int32 sums meet in
//     LDS, as those of the groups do (integer: the order does not matter);
//   * a part is put together in LDS and leaves as 16-byte row pieces: with an odd N no row
//     starts on a word, and byte stores from the accumulator layout would be 16 times the instructions.
// What bounds it: at the sizes of classifiers what ONE CU can fetch from beyond its L2 (about 20 bytes a clock: 0.36 us for the 16 KB of
// a block of a 64 x 64 part, however many of them are requested ahead and by however many groups of waves), so parts are as
// small as still gives every CU one, nothing is requested that is not used (a next block that is not there used to be
// requested again, and the bias was read where it is added: a round trip to memory before each part's end), and a
// second block in flight only costs registers (1500 x 260 x 1540 5.4 / 5.5 us with one / two, 2048 x 259 x 2052 8.0 / 8.3). us before / now: 3156 x 64 x 3456 15.5 / 7.8, 2048 x 259 x 2052 13.6 / 7.8,
// 1376 x 1598 x 17 9.8 / 4.6, 2378 x 2958 x 70 13.1 / 6.1, 225 x 515 x 361 7.8 / 3.9, 1491 x 1457 x 666 12.9 / 8.2, 1400 x 1601 x
// 1400 14.5 / 10.6. Large ones are bound by operand delivery (4000 x 4001 x 4001: 108 / 95 us = 1.35 POP/s).
// Reference loop: BareMetal/ConvKernel.cpp:305-344 on the [M,K,1,1] x [N,K,1,1] layer.
#include <type_traits>

#include "conv_mfma_i8.h"

namespace mg {

typedef int v4i_w __attribute__((ext_vector_type(4), aligned(4)));

struct FcTileParams {
    const int8_t* src;   // [M][K]
    const int8_t* wp;    // packed filter [K/32][OCP][32], 16-byte halves swapped when (oc >> 3) & 1
    const int32_t* bias; // [OC] or NULL
    int8_t* dst;         // [M][OC]
    unsigned last16;     // offset of the last 16 bytes of src
    unsigned src_off, last_word;  // ODD: src points to the word that holds the first byte, src_off its place in it
    int M, K, OC, OCP, nblk;  // nblk: blocks of 128 bytes of K
    int act;
    RequantPack rq;
    XcdOrder xo;  // tile order (set at launch from the grid)
};

// 16 bytes of the activations from any offset, in two halves so that the bytes are moved into place only where they are used. ODD: at any
// byte - aligned words and the one behind them, moved by the offset's last two bits
template <bool ODD>
struct FcPiece {
    v4i v;
    uint32_t next;
    __device__ __forceinline__ void load(const FcTileParams& q, unsigned off) {  // off <= last16
        if constexpr (ODD) {
            const unsigned a = (off + q.src_off) & ~3u;
            v = *(const v4i_w*)(q.src + a);
            next = *(const uint32_t*)(q.src + min(a + 16u, q.last_word));
        } else {
            v = *(const v4i_w*)(q.src + off);
        }
    }
    // LAST: of a row's last block, the only one that may reach past the end of the tensor
    template <bool LAST>
    __device__ __forceinline__ v4i bytes(const FcTileParams& q, unsigned off) const {
        v4i r = v;
        if constexpr (ODD) {
            const unsigned s = (((LAST && off > q.last16 ? q.last16 : off) + q.src_off) & 3u) * 8u;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                r[j] = (int)(uint32_t)((((uint64_t)(j < 3 ? (uint32_t)v[j < 3 ? j + 1 : 0] : next) << 32) | (uint32_t)v[j]) >> s);
        }
        if (LAST && off > q.last16)  // (a piece wholly beyond meets the packed filter's zeros, whatever it holds)
            r = fc_tail_piece(r, min(off - q.last16, 15u));
        return r;
    }
};

// pieces of one block of K from the places roff + b
template <bool ODD, int N>
__device__ __forceinline__ void fc_fetch(const FcTileParams& q, const unsigned (&roff)[N], unsigned b, FcPiece<ODD> (&piece)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i)
        piece[i].load(q, min(roff[i] + b, q.last16));
}

// 16 results of a row
__device__ __forceinline__ void fc_store_piece(const FcTileParams& q, int row, int oc, v4i v) {
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

// MT, NT: 32-channel and 32-row MFMA tiles per wave; a group of four waves makes 64 MT channels x 64 NT rows
// KW: groups of four waves that share K
template <int MT, int NT, int KW, bool ODD, int ACT>
__global__ void __launch_bounds__(256 * KW) fc_tile_kernel(FcTileParams q) {
    constexpr int BOC = 64 * MT, BR = 64 * NT;
    constexpr int STAGE = BR * 128;                      // bytes of one stage buffer
    constexpr int AL = 2 * NT;                           // 16-byte loads per thread and block
    constexpr int OPITCH = BOC + 16;                     // row of the output tile in LDS
    constexpr int ACC = MT * NT * 16 * 256 * 4;          // bytes of a group's accumulators
    constexpr int NEED0 = KW * 2 * STAGE, NEED1 = (KW - 1) * ACC, NEED2 = BR * OPITCH;
    constexpr int LDS = NEED0 > NEED1 ? (NEED0 > NEED2 ? NEED0 : NEED2) : (NEED1 > NEED2 ? NEED1 : NEED2);
    __shared__ __attribute__((aligned(16))) int8_t lds[LDS];
    __shared__ __attribute__((aligned(16))) int bias_lds[BOC];
    const int tid = threadIdx.x & 255, lane = tid & 63;
    const int grp = KW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wn = wave & 1;
    const int col = lane & 31, kg = lane >> 5;
    int tx, ty;
    xcd_tile(q.xo, blockIdx.x, blockIdx.y, gridDim.x, gridDim.y, tx, ty);
    const int oc0 = tx * BOC, row0 = ty * BR;
    int8_t* const stage = lds + grp * (2 * STAGE);
    // (the bias is asked for first and waits in LDS: read where it is added, a round trip to memory stood before every tile's end)
    const int boc = tid & (BOC - 1);
    const int bias_v = q.bias ? q.bias[min(oc0 + boc, q.OC - 1)] : 0;

    // activations: thread -> row (tid >> 3) + 32 i, piece tid & 7 of the block
    const int srow = tid >> 3, pc = tid & 7;
    unsigned roff[AL];
#pragma unroll
    for (int i = 0; i < AL; ++i)
        roff[i] = (unsigned)min(row0 + srow + 32 * i, q.M - 1) * (unsigned)q.K + (unsigned)pc * 16u;
    FcPiece<ODD> ra[AL];
    auto act_store = [&](int s, int blk, auto last) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < AL; ++i)
            *(v4i*)(stage + (s & 1) * STAGE + (srow + 32 * i) * 128 + ((pc ^ (srow & 7)) << 4)) =
                    ra[i].template bytes<decltype(last)::value>(q, roff[i] + (unsigned)blk * 128u);
    };
    const int8_t* arow[MT];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
        const int oc = oc0 + wm * (32 * MT) + mi * 32 + col;  // (< OCP: a multiple of every tile width)
        arow[mi] = q.wp + (size_t)oc * KROW + (((kg ^ (oc >> 3)) & 1) << 4);
    }
    const size_t cstep = (size_t)q.OCP * KROW;
    v4i A[MT][4];
    auto flt_load = [&](int blk) __attribute__((always_inline)) {
        const size_t o = (size_t)(blk * 4) * cstep;
#pragma unroll
        for (int mi = 0; mi < MT; ++mi)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                A[mi][c] = *(const v4i*)(arow[mi] + o + c * cstep);
    };
    v16i acc[MT][NT];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi)
#pragma unroll
        for (int ni = 0; ni < NT; ++ni)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                acc[mi][ni][e] = 0;
    auto multiply = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            v4i b[NT];
#pragma unroll
            for (int ni = 0; ni < NT; ++ni)
                b[ni] = *(const v4i*)(stage + (s & 1) * STAGE + (wn * (32 * NT) + ni * 32 + col) * 128 +
                                      (((c * 2 + kg) ^ (col & 7)) << 4));
#pragma unroll
            for (int mi = 0; mi < MT; ++mi)
#pragma unroll
                for (int ni = 0; ni < NT; ++ni)
                    acc[mi][ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[mi][c], b[ni], acc[mi][ni], 0, 0, 0);
        }
    };

    // Group g multiplies blocks g, g + KW, ...; all groups take the same number of steps, the last of which some may sit out. (One barrier
    // a step: a wave that has passed the one of the step between has left the buffer it stores to. The last step stands by
    // itself: nothing is asked for beyond it - a clamped request costs what a real one does.)
    const int steps = (q.nblk + KW - 1) / KW;
    int blk = KW == 1 ? 0 : min(grp, q.nblk - 1);
    fc_fetch(q, roff, (unsigned)blk * 128u, ra);
    flt_load(blk);
    bias_lds[boc] = bias_v;
    blk = grp;
    for (int s = 0; s + 1 < steps; ++s) {
        act_store(s, blk, std::false_type());
        __syncthreads();
        blk += KW;
        const int next = KW == 1 ? blk : min(blk, q.nblk - 1);
        fc_fetch(q, roff, (unsigned)next * 128u, ra);
        multiply(s);
        flt_load(next);
    }
    const bool mine = KW == 1 || blk < q.nblk;
    if (mine)
        act_store(steps - 1, blk, std::true_type());
    __syncthreads();
    if (mine)
        multiply(steps - 1);
    __syncthreads();
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
            for (int ni = 0; ni < NT; ++ni) {
                int a[16];
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4) {
                    const v4i bv = *(const v4i*)(bias_lds + wm * (32 * MT) + mi * 32 + e4 * 8 + kg * 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        a[e4 * 4 + e] = acc[mi][ni][e4 * 4 + e] + bv[e];
                }
                uint32_t d[4];
                requant_dwords<ACT>(a, d, q.rq, q.act);
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4)
                    *(uint32_t*)(lds + (wn * (32 * NT) + ni * 32 + col) * OPITCH + wm * (32 * MT) + mi * 32 + e4 * 8 + kg * 4) = d[e4];
            }
    }
    __syncthreads();
    constexpr int PIECES = BOC / 16;
    for (int i = threadIdx.x; i < BR * PIECES; i += 256 * KW) {
        const int r = i / PIECES, p = i - r * PIECES;
        const int row = row0 + r, oc = oc0 + p * 16;
        if (row >= q.M || oc >= q.OC)
            continue;
        fc_store_piece(q, row, oc, *(const v4i*)(lds + r * OPITCH + p * 16));
    }
}

// Parts of 32 channels x 32 rows: a workgroup of W waves that share K between them, each with 4 KB of LDS of its own for its block's
// activations (operands fetched a row a lane took a third longer where rows start at odd bytes: 512 x 4001 x 1024 14.3 / 9.4 us).
template <bool ODD, int ACT>
__global__ void __launch_bounds__(256) fc_quarter_kernel(FcTileParams q) {
    constexpr int W = 4;
    constexpr int OPITCH = 48;
    __shared__ __attribute__((aligned(16))) int8_t lds[W * 4096 + 32 * OPITCH];  // a block or the sums of each wave; the part
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, kg = lane >> 5;
    int tx, ty;
    xcd_tile(q.xo, blockIdx.x, blockIdx.y, gridDim.x, gridDim.y, tx, ty);
    const int oc0 = tx * 32, row0 = ty * 32;
    // (the bias of the four channels that this lane will finish)
    v4i bv = {0, 0, 0, 0};
    if (q.bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            bv[e] = q.bias[min(oc0 + wave * 8 + kg * 4 + e, q.OC - 1)];
    }
    // activations: lane -> row (lane >> 3) + 8 i, piece lane & 7 of the wave's block, through 4 KB of LDS of the wave's own
    int8_t* const stage = lds + wave * 4096;
    const int srow = lane >> 3, pc = lane & 7;
    unsigned roff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        roff[i] = (unsigned)min(row0 + srow + 8 * i, q.M - 1) * (unsigned)q.K + (unsigned)pc * 16u;
    const int oc = oc0 + col;
    const size_t cstep = (size_t)q.OCP * KROW;
    const int8_t* const arow = q.wp + (size_t)oc * KROW + (((kg ^ (oc >> 3)) & 1) << 4);
    FcPiece<ODD> ra[4];
    v4i A[4];
    auto flt_load = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            A[c] = *(const v4i*)(arow + (size_t)(blk * 4 + c) * cstep);
    };
    v16i acc;
#pragma unroll
    for (int e = 0; e < 16; ++e)
        acc[e] = 0;
    auto act_store = [&](int blk, auto last) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *(v4i*)(stage + (srow + 8 * i) * 128 + ((pc ^ srow) << 4)) =
                    ra[i].template bytes<decltype(last)::value>(q, roff[i] + (unsigned)blk * 128u);
    };
    // (a wave's LDS operations execute in order: no barrier)
    auto multiply = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const v4i b = *(const v4i*)(stage + col * 128 + (((c * 2 + kg) ^ (col & 7)) << 4));
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[c], b, acc, 0, 0, 0);
        }
    };
    // blocks wave, wave + W, ...
    if (wave < q.nblk) {
        int blk = wave;
        fc_fetch(q, roff, (unsigned)blk * 128u, ra);
        flt_load(blk);
        for (; blk + W < q.nblk; blk += W) {
            act_store(blk, std::false_type());
            fc_fetch(q, roff, (unsigned)(blk + W) * 128u, ra);
            multiply();
            flt_load(blk + W);
        }
        act_store(blk, std::true_type());
        multiply();
    }
    // register e: channel 8 * (e / 4) + 4 * kg + e % 4, row = the lane's column
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4)
        *(v4i*)(stage + e4 * 1024 + lane * 16) = v4i{acc[4 * e4], acc[4 * e4 + 1], acc[4 * e4 + 2], acc[4 * e4 + 3]};
    __syncthreads();
    int a[4] = {bv[0], bv[1], bv[2], bv[3]};
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const v4i v = *(const v4i*)(lds + w * 4096 + wave * 1024 + lane * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            a[e] += v[e];
    }
    uint32_t d[1];
    requant_dwords<ACT>(a, d, q.rq, q.act);
    int8_t* const out = lds + W * 4096;
    *(uint32_t*)(out + col * OPITCH + wave * 8 + kg * 4) = d[0];
    __syncthreads();
    if (tid < 64) {
        const int r = tid >> 1, p = tid & 1, row = row0 + r, o0 = oc0 + p * 16;
        if (row < q.M && o0 < q.OC)
            fc_store_piece(q, row, o0, *(const v4i*)(out + r * OPITCH + p * 16));
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
    const bool odd = (g.ic & 3) || ((uintptr_t)src & 3);
    q.src_off = odd ? (unsigned)((uintptr_t)src & 3) : 0;
    q.src -= q.src_off;
    q.last_word = (q.src_off + q.last16 + 15) & ~3u;
    // Parts of 128 x 128 (us for 128 / 64) from 16 blocks of K for each CU in the 128 x 128 squares of a chip full of them: 4000 x 600 x 4000
    // 21 / 25, 4000 x 1001 x 4000 30 / 43, 2500 x 1601 x 2500 24 / 31; below, 4000 x 300 x 4000 17 / 17, 2048 x 1001 x 2052 17 / 14,
    // 2049 x 67 x 2050 8.6 / 6.0. Parts of 32 x 32 (us for 32 / 64) while there are three to a CU: 300 x 2000 x 300 4.3 / 7.8, 512 x 4001 x
    // 1024 9.4 / 14.9, 898 x 1104 x 690 5.4 / 5.8, or four where a second round of squares would be nearly empty (1491 x 1457 x 666 8.2 / 9.6);
    // beyond, 832 x 515 x 960 5.1 / 4.7, 1400 x 515 x 1400 8.6 / 6.3. Squares in one round share a long K between four groups
    // (us for one / four groups: 832 x 4001 x 960 18.3 / 15.6, 1024 x 4096 x 1000 11.2 / 10.4, 832 x 2000 x 960 7.0 / 6.9, 960 x 1001 x 960 5.9 / 5.9)
    const long big = (long)((g.n + 127) / 128) * ((g.oc + 127) / 128);
    const long squares = (long)((g.n + 63) / 64) * ((g.oc + 63) / 64);
    const long quarters = (long)((g.n + 31) / 32) * ((g.oc + 31) / 32);
    const int part = big >= num_cus() && big * q.nblk >= 16L * num_cus() ? 128
                     : quarters > (squares > num_cus() ? 4L : 3L) * num_cus() ? 64 : 32;
    const int groups = part == 32 || (part == 64 && squares <= num_cus() && q.nblk >= 16) ? 4 : 1;
    const int act = q.rq.mode ? g.act : -1;
#define MG_FCA(KERN, ...)                                                       \
    (act == MEGCC_NONLINE_IDENTITY  ? KERN<__VA_ARGS__, MEGCC_NONLINE_IDENTITY> \
     : act == MEGCC_NONLINE_RELU    ? KERN<__VA_ARGS__, MEGCC_NONLINE_RELU>     \
     : act == MEGCC_NONLINE_H_SWISH ? KERN<__VA_ARGS__, MEGCC_NONLINE_H_SWISH>  \
                                    : KERN<__VA_ARGS__, -1>)
    void (*kern)(FcTileParams) = part == 32   ? odd ? MG_FCA(fc_quarter_kernel, true) : MG_FCA(fc_quarter_kernel, false)
                                 : part == 128 ? odd ? MG_FCA(fc_tile_kernel, 2, 2, 1, true) : MG_FCA(fc_tile_kernel, 2, 2, 1, false)
                                 : groups == 4  ? odd ? MG_FCA(fc_tile_kernel, 1, 1, 4, true) : MG_FCA(fc_tile_kernel, 1, 1, 4, false)
                                 : odd         ? MG_FCA(fc_tile_kernel, 1, 1, 1, true)
                                               : MG_FCA(fc_tile_kernel, 1, 1, 1, false);
#undef MG_FCA
    const dim3 grid((g.oc + part - 1) / part, (g.n + part - 1) / part);
    q.xo = options().no_xcdorder ? XcdOrder{0} : make_xcd_order((int)grid.x, (int)grid.y, (long)(q.M + q.OC) * q.K);
    note_kernel(q.xo.w ? "fc_tile_xo" : "fc_tile", part, groups);  // (the part's side, the groups of waves that share K in it)
    note_requant_affine(q.rq.affine());
    hipLaunchKernelGGL(kern, grid, dim3(part == 32 ? 256 : 256 * groups), 0, stream(), q);
    return check_launch("fc_tile");
}

}  // namespace mg
