// The head of a quantised MobileNet as ONE kernel: the f32 image to qsi8, the first convolution (3 channels, 3x3 stride 2,
// NCHW -> NCHW44, 32 channels), the channel-wise 3x3 and the pointwise 1x1 convolution behind it. As three kernels (the last two
// are conv_dw_pw's pair) the quantised image and the first convolution's result, the largest tensors of the network but one, go
// out and come back: 283 of the 642 MB of batch 256, and two launches of a network that is 18 of them.
//
// A workgroup of 8 waves owns a strip of rows of one image and walks down it two output rows a step. Four stages work at the
// same time, each a step behind the one that feeds it, one barrier a step:
//   A  four rows of the image, asked for a step earlier, are quantised into a ring of rows in LDS (every pixel once);
//   B  the first convolution, as in conv_first.hip (k = 4 (ic 3 + fh) + fw; the fourth bytes, where a filter row has no weight, take the
//      ninth pair (ic, fh), so that one product does): 32 pixels a wave, whose four bytes of a row are cut out of two dwords of the
//      ring. Its result goes to a second ring, channel group by channel group as NCHW44 has it; rows outside of the image
//      are written as the zeros the next layer pads with;
//   C  the channel-wise layer as in conv_dw_pw.hip: a product with a banded matrix, 16 channels x 64 pixels a wave, whose operands
//      are 16-byte pieces of the second ring and the pixels left and right of them;
//   D  the pointwise layer: 32 pixels a wave, the filter in registers, four channels of a pixel a store.
// So a strip pays three steps before its first result (and computes three rows that its neighbours compute too); how many
// strips an image has follows from how many images there are for a CU (stem_strips).
// The requantisations are those of epilogue.h, so the result is bit for bit the four operators'.
// What bounds it: a step's 1.4 us are the waves' operands out of LDS, products and conversions one after the other, about 0.65 us of
// them the vector ALU's; from 256 images on memory (359 MB). Measured (us, 3 x 224 x 224 -> 64, as three kernels / this one):
// N=1 9.5 / 5.7, 8 13.0 / 7.9, 32 26.6 / 16.7, 64 36.6 / 26.8, 128 59 / 47, 256 141 / 90. 112 registers are two waves a SIMD beside two of the
// 144 that conv_dw_pw has at 512 channels: in a network the tail of the forward before runs on the same CUs. (216 registers, all
// biases in them and the stages' operands asked for together took 1.29 us a step and made no network faster; with the conversion of
// every sum to a float, mode 1 for 5, 1.50.)
#include "common.h"
#include "conv_geom.h"
#include "conv_mfma_i8.h"
#include "epilogue.h"

namespace mg {

static constexpr int ST_THREADS = 512;
static constexpr int ST_C = 32;               // channels of the first and the channel-wise layer
static constexpr int ST_MAXW = 128;           // output pixels of a row
static constexpr int ST_T = 2 * ST_MAXW;      // places for a step's pixels
static constexpr int ST_IRING = 16, ST_IROW = 68;   // rows of the image ring; dwords of a row of one channel: 3 unused, one of padding, 64; behind the pixels another of padding
static constexpr int ST_CRING = 8, ST_CROW = 136;   // rows of the second ring; dwords of a channel group's row: 4 + 128 + 4, padding next to the pixels
static constexpr int ST_ALL_BUT_MFMA = 0x7f6;
typedef unsigned st_v2u __attribute__((ext_vector_type(2)));

struct StemParams {
    const float* image;
    const int8_t* flt0;    // [8][3][3][3][4]
    const int32_t* bias0;  // biases: or NULL
    const uint32_t* dflt;  // [8][3][3] dwords of 4 channel bytes
    const int32_t* dbias;
    const int8_t* wp;      // packed pointwise filter [OCP][32], halves swapped when (oc >> 3) & 1
    const int32_t* pbias;
    uint32_t* dst;
    int image_bytes, dst_bytes;
    int ih, iw, oh, ow, OC;
    int steps, strips;     // steps of two output rows of an image, workgroups of an image
    float scale;           // 1 / the quantised image's
    FastDiv d_strips, d_quads;  // d_quads: 16-byte pieces of an image row
    RequantPack r0, dq, pq;
};

// MT: 32-channel tiles of the pointwise layer; PACT: its activation (the other two have RELU). FMA: all three requantise by
// mode 5, else by whichever form.
template <int MT, int PACT, bool FMA>
__global__ void __launch_bounds__(ST_THREADS, 4) conv_stem_kernel(StemParams q) {
    __shared__ __attribute__((aligned(16))) uint32_t img[ST_IRING * 3 * ST_IROW + 1];  // (the widest rows' last padding is the next row's first dword)
    __shared__ __attribute__((aligned(16))) uint32_t first[ST_CRING * (ST_C / 4) * ST_CROW];
    __shared__ __attribute__((aligned(16))) v4i mid[2][2 * ST_T];  // [16 channels][pixel] pieces
    __shared__ __attribute__((aligned(16))) int b0[ST_C], db[ST_C], pb[32 * MT];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, kg = lane >> 5;     // 32-pixel products: pixel, half of K
    const int colq = lane & 15, kg4 = lane >> 4;   // banded product: group of 4 pixels, input row / pixel of the group
    const unsigned OOB = 0x80000000u;
    const int n = (int)fdiv(blockIdx.x, q.d_strips), strip = blockIdx.x - n * q.strips;
    const int s0 = strip * q.steps / q.strips, s1 = (strip + 1) * q.steps / q.strips;
    const __amdgpu_buffer_rsrc_t ri = __builtin_amdgcn_make_buffer_rsrc((void*)q.image, 0, q.image_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc((void*)q.dst, 0, q.dst_bytes, 0x00020000);

    // ---- A: a thread's pieces of 4 pixels (piece i of channel c, row k of the rows that come together)
    const int quads = q.iw >> 2;
    int k[2], place[2];  // row (far beyond any: no piece); dword of a ring row's channel
    unsigned goff[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int idx = tid + h * ST_THREADS;
        const int rc = (int)fdiv(idx, q.d_quads), i = idx - rc * quads;
        k[h] = rc * 11 >> 5;  // rc / 3 (rc < 15)
        const int c = rc - 3 * k[h];
        k[h] = rc < 15 ? k[h] : 1 << 20;
        goff[h] = (unsigned)((((n * 3 + c) * q.ih + k[h]) * q.iw + 4 * i) * 4);
        place[h] = c * ST_IROW + 4 + i;
    }
    float4 px[2];
    auto ask = [&](int row0, int rows) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool in = k[h] < rows && (unsigned)(row0 + k[h]) < (unsigned)q.ih;
            const v4i v = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                    ri, (int)(in ? goff[h] + (unsigned)(row0 * q.iw * 4) : OOB), 0, 0));
            px[h] = __builtin_bit_cast(float4, v);
        }
    };
    auto quantise = [&](int row0, int rows) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (k[h] < rows)
                img[((row0 + k[h]) & (ST_IRING - 1)) * (3 * ST_IROW) + place[h]] =
                        pack4_perm(fp32_to_int8(px[h].x * q.scale), fp32_to_int8(px[h].y * q.scale), fp32_to_int8(px[h].z * q.scale),
                                   fp32_to_int8(px[h].w * q.scale));
    };
    ask(4 * s0 - 3, 5);

    // ---- set-up: filters by way of `mid`, which stage C writes two barriers from here at the earliest
    auto start = [](int bias, const RequantPack& r) { return FMA ? requant_bias(bias, r) : bias; };
    int* const w0 = (int*)mid;              // [9 pairs][32]
    int* const wl = w0 + 9 * ST_C;          // [32][4]: per channel the channel-wise filter's 3 rows, one of zeros
    if (tid < ST_C / 4 * 9) {  // (channel group, pair (ic, fh)): four channels' dwords (w0, w1, w2, 0)
        typedef uint32_t word __attribute__((aligned(1)));
        const int g4 = tid / 9, pair = tid - g4 * 9, ic = pair / 3, fh = pair - ic * 3;
        const word* f = (const word*)q.flt0 + (g4 * 3 + fh) * 9 + ic;
        const uint32_t f0 = f[0], f1 = f[3], f2 = f[6];
        const uint32_t lo = __builtin_amdgcn_perm(f1, f0, 0x05010400u), hi = __builtin_amdgcn_perm(f1, f0, 0x07030602u);
        *(v4i*)(w0 + pair * ST_C + g4 * 4) =
                v4i{(int)__builtin_amdgcn_perm(f2, lo, 0x0c040100u), (int)__builtin_amdgcn_perm(f2, lo, 0x0c050302u),
                    (int)__builtin_amdgcn_perm(f2, hi, 0x0c060100u), (int)__builtin_amdgcn_perm(f2, hi, 0x0c070302u)};
    } else if (tid >= 128 && tid < 256) {
        const int i = tid - 128, dy = i & 3, sh = 8 * ((i >> 2) & 3);
        const uint32_t* w = q.dflt + ((i >> 4) * 3 + min(dy, 2)) * 3;
        const uint32_t v = ((w[0] >> sh) & 0xff) | (((w[1] >> sh) & 0xff) << 8) | (((w[2] >> sh) & 0xff) << 16);
        wl[i] = dy < 3 ? (int)v : 0;
    } else if (tid >= 256 && tid < 256 + ST_C) {
        b0[tid - 256] = start(q.bias0 ? q.bias0[tid - 256] : 0, q.r0);
    } else if (tid >= 320 && tid < 320 + ST_C) {
        db[tid - 320] = start(q.dbias ? q.dbias[tid - 320] : 0, q.dq);
    } else if (tid >= 384 && tid < 384 + 32 * MT) {
        pb[tid - 384] = start(q.pbias ? q.pbias[tid - 384] : 0, q.pq);
    } else if (tid >= 448 && tid < 448 + ST_IRING * 3) {
        img[(tid - 448) * ST_IROW + 3] = 0;
        img[(tid - 448) * ST_IROW + 4 + quads] = 0;
    }
    if (tid < ST_CRING * (ST_C / 4)) {
        first[tid * ST_CROW + 3] = 0;
        first[tid * ST_CROW + 4 + q.ow] = 0;
    }
    v4i P[MT];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
        const int oc = mi * 32 + col;
        P[mi] = *(const v4i*)(q.wp + oc * KROW + (((kg ^ (oc >> 3)) & 1) << 4));
    }
    quantise(4 * s0 - 3, 5);
    wait_vmcnt<0>();  // (the filters are there: no wait for them is left in the loop)
    ask(4 * s0 + 2, 4);
    __syncthreads();
    // rows of the first filter: pairs 4 kg .. + 3 of this half of K; the three weights of pair 8 where pairs 0 to 2 have their zeros
    v4i A1;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        A1[j] = w0[(4 * kg + j) * ST_C + col] | (kg == 0 && j < 3 ? w0[8 * ST_C + col] >> (8 * j) << 24 : 0);
    // ---- B: this lane's pixel of a step's two rows and where its bytes begin in a ring row
    const int slot = wave * 32 + col;
    const bool there = slot < 2 * q.ow;
    const int row = there && slot >= q.ow ? 1 : 0, x = there ? slot - row * q.ow : 0;
    const unsigned cut = (x & 1) ? 1 : 3;
    const int at = 3 + ((x + 1) >> 1);  // its first dword's place
    // ---- C: banded matrices and this lane's pieces
    const int quad = wave & 1, sub = wave >> 1;
    const int xg = q.ow >> 2;
    const int g = min(sub * 16 + colq, 2 * xg - 1), grow = g >= xg ? 1 : 0, gx = (g - grow * xg) * 4;
    const int grow_in = grow - 1 + min(kg4, 2);  // (the fourth quarter of K meets zero weights)
    v4i M[4];
    st_v2u Me[4];
    {
        const int bx = colq >> 2, sh = 8 * (colq & 3);
        auto selector = [&](int fw) { return (unsigned)fw < 3u ? (0x0c0c0c0cu & ~(0xffu << sh)) | ((unsigned)fw << sh) : 0x0c0c0c0cu; };
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const unsigned w = (unsigned)wl[((quad * 4 + p) * 4 + (colq & 3)) * 4 + kg4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                M[p][e] = (int)__builtin_amdgcn_perm(0u, w, selector(e + 1 - bx));
            Me[p] = st_v2u{__builtin_amdgcn_perm(0u, w, selector(-bx)), __builtin_amdgcn_perm(0u, w, selector(5 - bx))};
        }
    }
    const int ostep = q.oh * q.ow * 4;  // bytes of a channel group of the result
    const int obase = n * (q.OC >> 2) * ostep + (row * q.ow + x) * 4 + kg * ostep;

    auto bias_of = [&](const int* from, v16i& acc) __attribute__((always_inline)) {
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
            const v4i bv = *(const v4i*)(from + e4 * 8 + kg * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                acc[e4 * 4 + e] = bv[e];
        }
    };
    auto requant = [&](auto act, int (&a)[16], uint32_t (&d)[4], const RequantPack& r) __attribute__((always_inline)) {
        constexpr int ACT = decltype(act)::value;
        if constexpr (FMA) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                d[k] = requant_pack4<5, ACT>(a[4 * k], a[4 * k + 1], a[4 * k + 2], a[4 * k + 3], r);
        } else {
            requant_dwords<ACT>(a, d, r);
        }
    };
    auto sums = [&](const v16i& acc, int (&a)[16]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
            a[e] = acc[e];
    };
    // B, rows 2 i - 1 and 2 i of the first convolution
    auto first_words = [&](int i, uint32_t (&w)[5][2]) __attribute__((always_inline)) {
        const int y = 2 * i - 1 + row;
        int r[3];  // by filter row
#pragma unroll
        for (int f = 0; f < 3; ++f)
            r[f] = ((2 * y - 1 + f) & (ST_IRING - 1)) * (3 * ST_IROW) + at;
#pragma unroll
        for (int j = 0; j < 5; ++j) {  // pairs (channel, filter row) 4 kg + j, and 8
            const int lo = j < 4 ? r[j % 3] + j / 3 * ST_IROW : r[2] + 2 * ST_IROW;
            const int hi = j < 4 ? r[(j + 1) % 3] + (4 + j) / 3 * ST_IROW : lo;
            const uint32_t* const d = img + (kg ? hi : lo);
            w[j][0] = d[0];
            w[j][1] = d[1];
        }
    };
    auto first_products = [&](const uint32_t (&w)[5][2]) __attribute__((always_inline)) -> v16i {
        int b[5];
#pragma unroll
        for (int j = 0; j < 5; ++j)
            b[j] = (int)__builtin_amdgcn_alignbyte(w[j][1], w[j][0], cut);
        v16i acc;
        bias_of(b0, acc);
#pragma unroll
        for (int j = 0; j < 3; ++j)  // byte j of pair 8 in the place of pair j's fourth (the other half of K has no weight there)
            b[j] = (int)__builtin_amdgcn_perm((unsigned)b[4], (unsigned)b[j], 0x00020100u + ((4u + j) << 24));
        return __builtin_amdgcn_mfma_i32_32x32x32_i8(A1, v4i{b[0], b[1], b[2], b[3]}, acc, 0, 0, 0);
    };
    auto first_results = [&](int i, const v16i& acc) __attribute__((always_inline)) {
        const int y = 2 * i - 1 + row;
        int a[16];
        uint32_t d[4];
        sums(acc, a);
        requant(std::integral_constant<int, MEGCC_NONLINE_RELU>{}, a, d, q.r0);
        const bool in = (unsigned)y < (unsigned)q.oh;
        if (there) {
            uint32_t* const o = first + ((y & (ST_CRING - 1)) * (ST_C / 4) + kg) * ST_CROW + 4 + x;
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4)
                o[e4 * 2 * ST_CROW] = in ? d[e4] : 0u;
        }
    };
    // C, rows 2 t and 2 t + 1 of the channel-wise layer
    struct Pieces {
        v4i b[4], acc[4];
        st_v2u e[4];
    };
    auto dw_operands = [&](int t, Pieces& o) __attribute__((always_inline)) {
        const uint32_t* const src = first + (((2 * t + grow_in) & (ST_CRING - 1)) * (ST_C / 4) + quad * 4) * ST_CROW + 4 + gx;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            o.b[p] = *(const v4i*)(src + p * ST_CROW);
            o.e[p] = st_v2u{src[p * ST_CROW - 1], src[p * ST_CROW + 4]};
            o.acc[p] = *(const v4i*)(db + quad * 16 + p * 4);
        }
    };
    // (the short products first and every product where it stands, as conv_dw_pw.hip has it: a long product must not
    // read sums that the short one has not written yet)
    auto dw_products = [&](Pieces& o) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            o.acc[p] = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                    __builtin_bit_cast(long, Me[p]), __builtin_bit_cast(long, o.e[p]), o.acc[p], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(ST_ALL_BUT_MFMA);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            o.acc[p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(M[p], o.b[p], o.acc[p], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(ST_ALL_BUT_MFMA);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto dw_results = [&](int t, const Pieces& o) __attribute__((always_inline)) {
        int a[16];
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                a[p * 4 + e] = o.acc[p][e];
        uint32_t d[4];
        requant(std::integral_constant<int, MEGCC_NONLINE_RELU>{}, a, d, q.dq);
        mid[t & 1][quad * ST_T + (sub * 16 + colq) * 4 + kg4] = v4i{(int)d[0], (int)d[1], (int)d[2], (int)d[3]};
    };
    // D, rows 2 t and 2 t + 1 of the pointwise layer
    auto pointwise = [&](int t, const v4i& b) __attribute__((always_inline)) {
        const unsigned o = there && 2 * t + row < q.oh ? (unsigned)(obase + 2 * t * q.ow * 4) : OOB;
#pragma unroll
        for (int mi = 0; mi < MT; ++mi) {
            v16i acc;
            bias_of(pb + mi * 32, acc);
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(P[mi], b, acc, 0, 0, 0);
            int a[16];
            uint32_t d[4];
            sums(acc, a);
            requant(std::integral_constant<int, PACT>{}, a, d, q.pq);
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4)
                __builtin_amdgcn_raw_buffer_store_b32(d[e4], rd, (int)o, (mi * 8 + e4 * 2) * ostep, 0);
        }
    };
    const bool mine = wave * 32 < 2 * q.ow;       // pixels for this wave (B, D)
    const bool pieces = sub * 16 < 2 * xg;        // ... groups (C)
    for (int i = s0; i < s1 + 3; ++i) {
        if (i < s1) {
            quantise(4 * i + 2, 4);
            ask(i + 1 < s1 ? 4 * i + 6 : q.ih, 4);
        }
        if (i <= s1 && mine) {
            uint32_t w[5][2];
            first_words(i, w);
            first_results(i, first_products(w));
        }
        if (i - 2 >= s0 && i - 2 < s1 && pieces) {
            Pieces o;
            dw_operands(i - 2, o);
            dw_products(o);
            dw_results(i - 2, o);
        }
        if (i - 3 >= s0 && mine)
            pointwise(i - 3, mid[(i - 3) & 1][kg * ST_T + slot]);
        lds_barrier();
    }
}

// c0: the first convolution (its s_src the quantised image's scale), dw, pw. (The scales are conv_stem_launch's question.)
bool conv_stem_supported(const ConvGeom& c0, const ConvGeom& dw, const ConvGeom& pw, const void* image, const void* dst) {
    return c0.fmt == MEGCC_FMT_NCHW_NCHW44 && c0.groups == 1 && c0.ic == 3 && c0.oc == ST_C && c0.fh == 3 && c0.fw == 3 && c0.sh == 2 &&
           c0.sw == 2 && c0.ph == 1 && c0.pw == 1 && c0.dh == 1 && c0.dw == 1 && c0.act == MEGCC_NONLINE_RELU && c0.ih == 2 * c0.oh &&
           c0.iw == 2 * c0.ow && (c0.ow & 3) == 0 && c0.ow >= 4 && c0.ow <= ST_MAXW && c0.oh >= 1 &&
           dw.fmt == MEGCC_FMT_NCHW44 && dw.groups == ST_C && dw.ic == ST_C && dw.oc == ST_C && dw.fh == 3 && dw.fw == 3 && dw.sh == 1 &&
           dw.sw == 1 && dw.ph == 1 && dw.pw == 1 && dw.dh == 1 && dw.dw == 1 && dw.act == MEGCC_NONLINE_RELU && dw.n == c0.n &&
           dw.ih == c0.oh && dw.iw == c0.ow &&
           pw.fmt == MEGCC_FMT_NCHW44 && pw.groups == 1 && pw.ic == ST_C && (pw.oc == 32 || pw.oc == 64) && pw.fh == 1 && pw.fw == 1 &&
           pw.sh == 1 && pw.sw == 1 && pw.ph == 0 && pw.pw == 0 && (pw.act == MEGCC_NONLINE_IDENTITY || pw.act == MEGCC_NONLINE_RELU) &&
           pw.n == c0.n && pw.ih == c0.oh && pw.iw == c0.ow &&
           ((uintptr_t)image & 3) == 0 && ((uintptr_t)dst & 3) == 0 && (long)c0.n * 3 * c0.ih * c0.iw * 4 < (1L << 31) - (1 << 20) &&
           (long)pw.n * pw.oc * pw.oh * pw.ow < (1L << 31);
}

// Workgroups of an image: one for a CU, and a strip has three steps on top of its own. (A CU holds two, and on its own the kernel is
// the quicker for it: N=64 4 strips 26.8 us, 8 23.7; 256 1 90, 2 79. In a network their room is the other stream's: MobileNetV1
// batch 64 147 and 155, 256 488 and 487, 16 14 strips 94.3, 28 94.7.)
static int stem_strips(long n, int steps) {
    int best = 1;
    long least = 1L << 60;
    for (int k = 1; k <= steps; ++k) {
        const long time = ((steps + k - 1) / k + 3) * ((n * k + num_cus() - 1) / num_cus());
        if (time < least) {
            least = time;
            best = k;
        }
    }
    return best;
}

// `launch` false: only whether the scales have constants
TinyNNStatus conv_stem_launch(
        const ConvGeom& c0, const ConvGeom& dw, const ConvGeom& pw, const void* image, const void* flt0, const void* bias0, const void* dflt,
        const void* dbias, const void* packed, const void* pbias, void* dst, bool launch) {
    const ConvGeom* const layers[] = {&c0, &dw, &pw};
    if (!launch) {  // (there are constants whatever the switch says)
        for (const ConvGeom* g : layers)
            MG_REQUIRE(requant_pack_for(g->act, g->s_src, g->s_flt, g->s_dst, false).mode, TinyNN_ERROR_NO_IMPLEMENT,
                       "conv_stem: scales without proven constants");
        return TinyNN_SUCCESS;
    }
    if (c0.n == 0)
        return TinyNN_SUCCESS;
    StemParams q = {};
    q.image = (const float*)image;
    q.flt0 = (const int8_t*)flt0;
    q.bias0 = (const int32_t*)bias0;
    q.dflt = (const uint32_t*)dflt;
    q.dbias = (const int32_t*)dbias;
    q.wp = (const int8_t*)packed;
    q.pbias = (const int32_t*)pbias;
    q.dst = (uint32_t*)dst;
    q.image_bytes = (int)((long)c0.n * 3 * c0.ih * c0.iw * 4);
    q.dst_bytes = (int)((long)pw.n * pw.oc * pw.oh * pw.ow);
    q.ih = c0.ih, q.iw = c0.iw, q.oh = c0.oh, q.ow = c0.ow;
    q.OC = pw.oc;
    q.steps = (c0.oh + 1) / 2;
    q.strips = stem_strips(c0.n, q.steps);
    q.scale = 1.f / c0.s_src;  // (as the conversion on its own has it)
    q.d_strips = make_fastdiv(q.strips);
    q.d_quads = make_fastdiv(c0.iw / 4);
    RequantPack* const packs[] = {&q.r0, &q.dq, &q.pq};
    bool fma = !options().no_affine, affine = true;
    for (int l = 0; l < 3; ++l) {
        const ConvGeom& g = *layers[l];
        if (fma)
            *packs[l] = requant_shifted_for(g.act, g.s_src, g.s_flt, g.s_dst);
        fma = fma && packs[l]->mode == 5;
    }
    for (int l = 0; l < 3; ++l) {
        const ConvGeom& g = *layers[l];
        if (!fma)
            *packs[l] = requant_pack_pick(g.act, g.s_src, g.s_flt, g.s_dst);
        affine = affine && packs[l]->affine();
    }
    MG_REQUIRE(q.r0.mode && q.dq.mode && q.pq.mode, TinyNN_ERROR_NO_IMPLEMENT, "conv_stem: scales without proven constants");
#define MG_STEM(MT_, ACT_) (fma ? conv_stem_kernel<MT_, ACT_, true> : conv_stem_kernel<MT_, ACT_, false>)
    void (*const kern)(StemParams) = pw.oc == 64 ? (pw.act == MEGCC_NONLINE_RELU ? MG_STEM(2, MEGCC_NONLINE_RELU) : MG_STEM(2, MEGCC_NONLINE_IDENTITY))
                                                 : (pw.act == MEGCC_NONLINE_RELU ? MG_STEM(1, MEGCC_NONLINE_RELU) : MG_STEM(1, MEGCC_NONLINE_IDENTITY));
#undef MG_STEM
    note_kernel("conv_stem", pw.oc, q.strips);
    note_requant_affine(affine);
    hipLaunchKernelGGL(kern, dim3((unsigned)(c0.n * q.strips)), dim3(ST_THREADS), 0, stream(), q);
    return check_launch("conv_stem");
}

}  // namespace mg
