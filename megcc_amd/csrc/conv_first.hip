// qsi8 first-layer convolution: NCHW input with 3 channels -> NCHW44 output, 3x3, stride 2, pad 1
// (the "hybrid" format NCHW_NCHW44 of MegCC's nchw44 layout pass; filter [OC/4, FH, FW, IC, 4oc],
// same loop nest and epilogue as BareMetal/ConvKernel.cpp:305-344,374-380).
//
// K = 27 is far too short for the matrix cores and the layer moves 3.7 bytes per MAC-quad, so
// this is a VALU kernel built around v_dot4_i32_i8:
//   * one thread = two horizontally adjacent output pixels (ow even) x all output channels. With
//     stride 2 and pad 1 the two pixels need input columns 4k-1 .. 4k+3 of three rows per channel:
//     the last byte of one aligned dword and the whole next one, so every load is an aligned dword
//     and consecutive lanes read consecutive dwords;
//   * per (channel, filter row) the 3 taps of a pixel are one dword (v_alignbyte / shift), the
//     matching weights one dword (w0, w1, w2, 0): 9 dot4 per pixel and output channel;
//   * weights are re-packed once per workgroup into LDS as [oc/4][ic*3+fh][4 oc] dwords and read
//     back as wave-wide broadcasts; bias and the 8 results of an oc group stay in registers and
//     leave as one 8-byte store (pixels ow, ow+1 of one NCHW44 plane).
// Only the top row and the left column can be padding for even IH, IW.
#include "common.h"
#include "conv_geom.h"
#include "epilogue.h"
#include "fastdiv.h"

namespace mg {

static constexpr int CF_THREADS = 256;
static constexpr int CF_MAX_OC = 128;
typedef int cf_v4i __attribute__((ext_vector_type(4)));

template <int ACT>
__global__ void __launch_bounds__(CF_THREADS) conv_first_q8_kernel(
        ConvGeom g, RequantFast rq, const int8_t* __restrict__ src, const int8_t* __restrict__ flt,
        const int32_t* __restrict__ bias, uint32_t* __restrict__ dst, int total_pairs,
        RequantTable table) {
    __shared__ __attribute__((aligned(16))) int wlds[CF_MAX_OC * 9];
    __shared__ __attribute__((aligned(16))) int blds[CF_MAX_OC];
    __shared__ int tbl[REQUANT_TABLE_ENTRIES];
    if (ACT >= 0)
        tbl[threadIdx.x] = table.t[threadIdx.x];
    const int oc4n = g.oc >> 2;
    // packed weight dword (g4, row = ic*3 + fh, o): bytes fw = 0, 1, 2 and a zero
    for (int i = threadIdx.x; i < g.oc * 9; i += CF_THREADS) {
        const int o = i & 3, row = (i >> 2) % 9, g4 = (i >> 2) / 9;
        const int ic = row / 3, fh = row - ic * 3;
        uint32_t w = 0;
#pragma unroll
        for (int fw = 0; fw < 3; ++fw) {
            const int8_t v = flt[((((size_t)g4 * 3 + fh) * 3 + fw) * 3 + ic) * 4 + o];
            w |= (uint32_t)(uint8_t)v << (8 * fw);
        }
        wlds[i] = (int)w;
    }
    for (int i = threadIdx.x; i < g.oc; i += CF_THREADS)
        blds[i] = bias ? bias[i] : 0;
    __syncthreads();

    const int ow2n = g.ow >> 1;
    const int iw4 = g.iw >> 2;  // dwords per input row
    for (int p = blockIdx.x * CF_THREADS + threadIdx.x; p < total_pairs; p += gridDim.x * CF_THREADS) {
        int r = p;
        const int ow2 = r % ow2n; r /= ow2n;
        const int oh = r % g.oh;
        const int n = r / g.oh;
        // x[row][0 / 1]: the 3 taps of pixel ow = 2*ow2 / 2*ow2 + 1 in (channel, filter row) `row`
        int xa[9], xb[9];
        const uint32_t* img = (const uint32_t*)(src + (size_t)n * 3 * g.ih * g.iw);
#pragma unroll
        for (int ic = 0; ic < 3; ++ic) {
#pragma unroll
            for (int fh = 0; fh < 3; ++fh) {
                const int ih = 2 * oh - 1 + fh;
                uint32_t cur = 0, prev = 0;
                if ((unsigned)ih < (unsigned)g.ih) {
                    const uint32_t* rowp = img + ((size_t)ic * g.ih + ih) * iw4;
                    cur = rowp[ow2];
                    if (ow2 > 0)
                        prev = rowp[ow2 - 1];
                }
                xa[ic * 3 + fh] = (int)__builtin_amdgcn_alignbyte(cur, prev, 3);  // prev.b3 cur.b0 cur.b1 (cur.b2)
                xb[ic * 3 + fh] = (int)(cur >> 8);                                // cur.b1 cur.b2 cur.b3 0
            }
        }
        uint32_t* out = dst + ((size_t)n * oc4n * g.oh + oh) * g.ow + 2 * ow2;
        for (int g4 = 0; g4 < oc4n; ++g4) {
            const cf_v4i bv = *(const cf_v4i*)(blds + g4 * 4);
            int a[4] = {bv[0], bv[1], bv[2], bv[3]}, b[4] = {bv[0], bv[1], bv[2], bv[3]};
#pragma unroll
            for (int row = 0; row < 9; ++row) {
                const cf_v4i w = *(const cf_v4i*)(wlds + (g4 * 9 + row) * 4);
#pragma unroll
                for (int o = 0; o < 4; ++o) {
                    a[o] = __builtin_amdgcn_sdot4(xa[row], w[o], a[o], false);
                    b[o] = __builtin_amdgcn_sdot4(xb[row], w[o], b[o], false);
                }
            }
            int ra[4], rb[4];
#pragma unroll
            for (int o = 0; o < 4; ++o) {
                if (ACT < 0) {
                    ra[o] = requant_conv_rt(g.act, a[o], g.s_src, g.s_flt, g.s_dst);
                    rb[o] = requant_conv_rt(g.act, b[o], g.s_src, g.s_flt, g.s_dst);
                } else {
                    ra[o] = requant_conv_table<(ACT < 0 ? 0 : ACT)>(a[o], rq.c, tbl);
                    rb[o] = requant_conv_table<(ACT < 0 ? 0 : ACT)>(b[o], rq.c, tbl);
                }
            }
            uint2 v;
            v.x = pack4_perm(ra[0], ra[1], ra[2], ra[3]);
            v.y = pack4_perm(rb[0], rb[1], rb[2], rb[3]);
            *(uint2*)(out + (size_t)g4 * g.oh * g.ow) = v;
        }
    }
}

// The same layer with 32 or 64 output channels on the matrix cores. K = 27 is short, but what the
// v_dot4 kernel above spends per output - 9 dot products next to the 10 instructions of the exact
// requantisation - is what an MFMA saves: here the reduction index is k = 4 * (ic * 3 + fh) + fw with a
// zero weight at fw = 3, so a lane's 16 K-bytes of the B operand are the 4 bytes at input columns
// 2 * ox - 1 .. 2 * ox + 2 of four (channel, filter row) pairs; 9 pairs x 4 bytes = 36 > 32, so a second
// MFMA takes the ninth pair.
// A wave takes 64 pixels a step, a lane the horizontally adjacent ones 2m and 2m + 1 - columns of two
// products with the same weights. Both are cut out of the same two aligned dwords (input columns
// 4m - 4 .. 4m + 3), so a pair of filter rows costs one 8-byte load for two pixels, the results leave as
// one 8-byte store a plane, and nothing but the very first pixel's dword is special. A wave's steps
// are consecutive (input rows that two output rows read are in its CU's L1), their number the same for
// every wave but the last ones. The requantisation needs no table: without
// one the arguments are an eighth.
// What bounds it: memory (N = 256: 141 MB in 27.5 us is what a large copy reaches), below 64 images the set-up and
// the first round trip. 3 x 224 x 224 -> 32 in us, with one pixel a lane, its filter bytes and biases loaded
// one by one and steps 8192 waves apart (the last round of four nearly empty at N = 64) / as it is:
// N = 1 3.5 / 3.3, 8 5.2 / 4.5, 32 9.0 / 7.7, 64 13.1 / 11.5, 128 20.0 / 15.8, 256 33.9 / 27.5.
typedef int cfm_v4i __attribute__((ext_vector_type(4)));
typedef int cfm_v2i __attribute__((ext_vector_type(2)));
typedef int cfm_v16i __attribute__((ext_vector_type(16)));
typedef uint32_t cfm_word __attribute__((aligned(1)));  // of a filter, which may begin at any byte

struct ConvFirstMfmaParams {
    const int8_t* src;
    const int8_t* flt;
    const int32_t* bias;
    uint32_t* dst;
    int src_bytes, dst_bytes;
    int IH, IW, OW2, OHW, pairs, steps, run, oc4n;
    int act;
    RequantPack rq;
    FastDiv dOW2, dOHW2;
};
static constexpr int CFM_WAVES = 5;  // waves a SIMD holds (N = 256 in us: 2 29.2, 3 28.5, 4 28.3, 5 27.5)

template <int MT, int ACT>
__global__ void __launch_bounds__(256) conv_first_mfma_kernel(ConvFirstMfmaParams q) {
    constexpr int OC = MT * 32;
    __shared__ __attribute__((aligned(16))) int wlds[9 * OC], blds[OC];
    const int tid = threadIdx.x, lane = tid & 63;
    const int col = lane & 31, kg = lane >> 5;
    // byte offset of this lane's (channel, filter row) pairs inside an image, relative to row 2 * oy - 1
    int pair_off[4];
    bool pair_top[4];  // the pair's filter row is 0: above the image when oy == 0
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int pair = 4 * kg + j, ic = pair / 3, fh = pair - ic * 3;
        pair_off[j] = (ic * q.IH + fh) * q.IW;
        pair_top[j] = fh == 0;
    }
    const int pair8_off = (2 * q.IH + 2) * q.IW;  // channel 2, filter row 2
    const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc((void*)q.src, 0, q.src_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rd =
            __builtin_amdgcn_make_buffer_rsrc((void*)q.dst, 0, q.dst_bytes, 0x00020000);
    const int OOB = (int)0x80000000u;
    // operands of a step (requested one step ahead: the loads fly during the epilogue before them)
    struct Step {
        cfm_v2i d[5];
        int out;  // byte offset of the two pixels in plane kg
        bool first;
    };
    auto request = [&](int t, int end) __attribute__((always_inline)) {
        Step r;
        const int p = t * 32 + col;
        const bool ok = t < end && p < q.pairs;
        const int n = fdiv(p, q.dOHW2), rem = p - n * (q.OHW >> 1);
        const int oy = fdiv(rem, q.dOW2), m = rem - oy * q.OW2;
        // the first pixels' left dword is padding: they load one dword further right and use the first one (the other may be
        // another row's, or beyond the images, where a buffer load reads nothing)
        r.first = m == 0;
        const int base = n * 3 * q.IH * q.IW + (2 * oy - 1) * q.IW + 4 * m - (r.first ? 0 : 4);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            r.d[j] = __builtin_amdgcn_raw_buffer_load_b64(rs, ok && !(pair_top[j] && oy == 0) ? base + pair_off[j] : OOB, 0, 0);
        r.d[4] = __builtin_amdgcn_raw_buffer_load_b64(rs, ok && kg == 0 ? base + pair8_off : OOB, 0, 0);
        r.out = ok ? 4 * ((n * q.oc4n + kg) * q.OHW + 2 * rem) : OOB;
        return r;
    };
    const int t0 = (blockIdx.x * 4 + (tid >> 6)) * q.run, t1 = min(t0 + q.run, q.steps);
    Step next = request(t0, t1);
    // ---- filter and bias once per workgroup: 15 single bytes and 16 biases a lane kept the address path busy for 3 us
    if (tid < OC / 4 * 9) {  // (channel group, pair): four channels' dwords (w0, w1, w2, 0)
        const int g4 = tid / 9, pair = tid - g4 * 9, ic = pair / 3, fh = pair - ic * 3;
        const cfm_word* f = (const cfm_word*)q.flt + (g4 * 3 + fh) * 9 + ic;
        const uint32_t f0 = f[0], f1 = f[3], f2 = f[6];
        const uint32_t lo = __builtin_amdgcn_perm(f1, f0, 0x05010400u), hi = __builtin_amdgcn_perm(f1, f0, 0x07030602u);
        *(cfm_v4i*)(wlds + pair * OC + g4 * 4) = cfm_v4i{
                (int)__builtin_amdgcn_perm(f2, lo, 0x0c040100u), (int)__builtin_amdgcn_perm(f2, lo, 0x0c050302u),
                (int)__builtin_amdgcn_perm(f2, hi, 0x0c060100u), (int)__builtin_amdgcn_perm(f2, hi, 0x0c070302u)};
    }
    if (tid >= 256 - OC)
        blds[tid - (256 - OC)] = q.bias ? q.bias[tid - (256 - OC)] : 0;
    __syncthreads();
    // filter rows of this lane's output channels: A1 = pairs 4 * kg .. 4 * kg + 3, A2 = pair 8
    cfm_v4i A1[MT], A2[MT], biasv[MT][4];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            A1[mi][j] = wlds[(4 * kg + j) * OC + mi * 32 + col];
        A2[mi] = cfm_v4i{kg == 0 ? wlds[8 * OC + mi * 32 + col] : 0, 0, 0, 0};
        // accumulator register e is channel 8 * (e / 4) + 4 * kg + e % 4 of the row tile
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4)
            biasv[mi][e4] = *(const cfm_v4i*)(blds + mi * 32 + e4 * 8 + kg * 4);
    }
    for (int t = t0; t < t1; ++t) {
        cfm_v4i be, bo;  // B operands of the even and the odd pixels
        int be8, bo8;
#pragma unroll
        for (int j = 0; j < 5; ++j) {
            const uint32_t lo = next.first ? 0u : (uint32_t)next.d[j][0], hi = (uint32_t)(next.first ? next.d[j][0] : next.d[j][1]);
            const int e = (int)__builtin_amdgcn_alignbyte(hi, lo, 3), o = (int)(hi >> 8);
            if (j < 4) {
                be[j] = e;
                bo[j] = o;
            } else {
                be8 = e;
                bo8 = o;
            }
        }
        const int out = next.out;
        next = request(t + 1, t1);
#pragma unroll
        for (int mi = 0; mi < MT; ++mi) {
            cfm_v16i ae, ao;
#pragma unroll
            for (int e = 0; e < 16; ++e)
                ae[e] = ao[e] = biasv[mi][e >> 2][e & 3];
            ae = __builtin_amdgcn_mfma_i32_32x32x32_i8(A1[mi], be, ae, 0, 0, 0);
            ao = __builtin_amdgcn_mfma_i32_32x32x32_i8(A1[mi], bo, ao, 0, 0, 0);
            ae = __builtin_amdgcn_mfma_i32_32x32x32_i8(A2[mi], cfm_v4i{be8, 0, 0, 0}, ae, 0, 0, 0);
            ao = __builtin_amdgcn_mfma_i32_32x32x32_i8(A2[mi], cfm_v4i{bo8, 0, 0, 0}, ao, 0, 0, 0);
            int a[32];  // by plane: four channels of the even pixel, of the odd one
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                a[e / 4 * 8 + e % 4] = ae[e];
                a[e / 4 * 8 + 4 + e % 4] = ao[e];
            }
            uint32_t d[8];
            requant_dwords<ACT>(a, d, q.rq, q.act);
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4)
                __builtin_amdgcn_raw_buffer_store_b64(cfm_v2i{(int)d[e4 * 2], (int)d[e4 * 2 + 1]}, rd, out, (mi * 8 + e4 * 2) * q.OHW * 4, 0);
        }
    }
}

static bool conv_first_mfma_ok(const ConvGeom& g) {
    return (g.oc == 32 || g.oc == 64) && (long)g.n * 3 * g.ih * g.iw < (1L << 31) &&
           (long)g.n * g.oc * g.oh * g.ow < (1L << 31) && !options().no_firstmfma;
}

static TinyNNStatus conv_first_mfma_launch(
        const ConvGeom& g, const void* src, const void* flt, const void* bias, void* dst) {
    ConvFirstMfmaParams q = {};
    q.src = (const int8_t*)src;
    q.flt = (const int8_t*)flt;
    q.bias = (const int32_t*)bias;
    q.dst = (uint32_t*)dst;
    q.src_bytes = (int)((long)g.n * 3 * g.ih * g.iw);
    q.dst_bytes = (int)((long)g.n * g.oc * g.oh * g.ow);
    q.IH = g.ih; q.IW = g.iw; q.OW2 = g.ow / 2;
    q.OHW = g.oh * g.ow;
    q.pairs = g.n * (q.OHW / 2);
    q.steps = (q.pairs + 31) / 32;
    q.oc4n = g.oc / 4;
    q.act = g.act;
    q.rq = requant_pack_pick(g.act, g.s_src, g.s_flt, g.s_dst);
    note_requant_affine(q.rq.affine());
    q.dOW2 = make_fastdiv(q.OW2);
    q.dOHW2 = make_fastdiv(q.OHW / 2);
    // as many waves as are resident at once, and of those only as many as the longest run of steps needs
    const int most = num_cus() * 4 * CFM_WAVES;
    q.run = (q.steps + most - 1) / most;
    const unsigned blocks = (unsigned)(((q.steps + q.run - 1) / q.run + 3) / 4);
    const int act = q.rq.mode ? g.act : -1;
#define MG_CFM(ACT_) (g.oc == 32 ? (const void*)conv_first_mfma_kernel<1, ACT_> : (const void*)conv_first_mfma_kernel<2, ACT_>)
    const void* kern = act == MEGCC_NONLINE_IDENTITY  ? MG_CFM(MEGCC_NONLINE_IDENTITY)
                       : act == MEGCC_NONLINE_RELU    ? MG_CFM(MEGCC_NONLINE_RELU)
                       : act == MEGCC_NONLINE_H_SWISH ? MG_CFM(MEGCC_NONLINE_H_SWISH)
                                                      : MG_CFM(-1);
#undef MG_CFM
    void* args[] = {&q};
    const hipError_t e = hipLaunchKernel(kern, dim3(blocks), dim3(256), args, 0, stream());
    MG_REQUIRE(e == hipSuccess, TinyNN_ERROR_RUNTIME, "conv_first_mfma: %s", hipGetErrorString(e));
    return check_launch("conv_first_mfma");
}

bool conv_first_supported(const ConvGeom& g) {
    return g.fmt == MEGCC_FMT_NCHW_NCHW44 && g.groups == 1 && g.ic == 3 && g.fh == 3 && g.fw == 3 &&
           g.sh == 2 && g.sw == 2 && g.ph == 1 && g.pw == 1 && g.dh == 1 && g.dw == 1 &&
           (g.iw & 3) == 0 && (g.ih & 1) == 0 && (g.oc & 3) == 0 && g.oc <= CF_MAX_OC &&
           g.ow * 2 == g.iw && g.oh * 2 == g.ih &&
           (long)g.n * g.oh * g.ow < (1L << 31);
}

TinyNNStatus conv_first_launch(
        const ConvGeom& g, const void* src, const void* flt, const void* bias, void* dst) {
    const long pairs = (long)g.n * g.oh * (g.ow / 2);
    if (pairs == 0)
        return TinyNN_SUCCESS;
    if (conv_first_mfma_ok(g)) {
        note_kernel("conv_first_mfma", g.oc / 32);
        return conv_first_mfma_launch(g, src, flt, bias, dst);
    }
    long blocks = (pairs + CF_THREADS - 1) / CF_THREADS;
    if (blocks > 256 * 16)
        blocks = 256 * 16;
    const RequantFast rq = make_requant_fast(g.s_src, g.s_flt, g.s_dst);
    // exact thresholds for the monotone activations; anything else (and extreme scales)
    // evaluates the literal sequence per output
    const bool tab = requant_table_act(g.act) && requant_table_ok(g.s_src, g.s_flt, g.s_dst);
    static const RequantTable no_table = {};
    std::shared_ptr<const RequantTable> kept;
    const RequantTable& table = tab ? *(kept = requant_table_for(g.act, g.s_src, g.s_flt, g.s_dst)) : no_table;
    auto kern = tab && g.act == MEGCC_NONLINE_IDENTITY ? conv_first_q8_kernel<MEGCC_NONLINE_IDENTITY>
              : tab && g.act == MEGCC_NONLINE_RELU     ? conv_first_q8_kernel<MEGCC_NONLINE_RELU>
              : tab && g.act == MEGCC_NONLINE_H_SWISH  ? conv_first_q8_kernel<MEGCC_NONLINE_H_SWISH>
                                                       : conv_first_q8_kernel<-1>;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(CF_THREADS), 0, stream(), g, rq,
                       (const int8_t*)src, (const int8_t*)flt, (const int32_t*)bias, (uint32_t*)dst,
                       (int)pairs, table);
    return check_launch("conv_first_q8");
}

}  // namespace mg
