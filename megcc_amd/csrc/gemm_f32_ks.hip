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
// Where there are too few 32 x 32 tiles for every CU, 16 x 16 ones (v_mfma_f32_16x16x4_f32, steps of 16, one tile a workgroup).
// Measured (us, before: the tiled kernel with its slice sums in a second launch, or conv_f32_small.hip; with 32 x 32 tiles; now):
// 64 x 4096 x 4096 35.4, 24.0, 23.6 (2.9 TB/s and 90 TFLOP/s), 197 x 771 x 1003 nt 19.9, 7.5, 7.5, 8 x 284 x 736 16.5, 4.0, 3.7,
// 1623 x 3660 x 316 73, 38, 35, 64 x 1024 x 1000 7.5, 4.8 with 16 x 16, 50 x 4000 x 500 21.1, 10.9, 128 x 2048 x 512 nt 17.0, 9.1;
// convolution 32 -> 32 on 56 x 56 6.9, 5.0, 4.2, 64 -> 64 28 x 28 6.7, 4.4, N=8 64 -> 64 on 56 x 56 55, 28, 27.6.
#include "common.h"
#include "conv_geom.h"
#include "conv_mfma_i8.h"
#include "epilogue.h"
#include "gemm_f32_ks.h"

namespace mg {

bool conv_f32_small_supported(const ConvGeom& g);

typedef float ks_v16f __attribute__((ext_vector_type(16)));
typedef float ks_v4f __attribute__((ext_vector_type(4)));
// the sums of an R x R tile and its product with K = 64 / R
template <int R>
struct KsTile {
    typedef ks_v16f Sums;
    static __device__ __forceinline__ Sums multiply(float a, float b, Sums c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
};
template <>
struct KsTile<16> {
    typedef ks_v4f Sums;
    static __device__ __forceinline__ Sums multiply(float a, float b, Sums c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
};

enum { KS_CONTIG = 0, KS_STRIDED = 1, KS_CONV = 2, KS_CONV1 = 3 };  // along K: contiguous, strided, gathered, 1x1 filter

struct KsParams {
    const float* A;
    const float* B;
    float* C;
    const float* bias;
    unsigned a_bytes, b_bytes;
    unsigned a_row, a_k, b_row, b_k;  // byte strides: of A's rows / B's columns, and along K
    // tiles in strips of strip_w columns, row by row inside a strip; per_xcd: of them on each XCD (0: a grid of tiles)
    int tiles, per_xcd, strip_w, strips;
    FastDiv d_strip, d_w, d_last;
    int M, N, K, ldc;
    int lw;  // log2 of the waves
    int act;
    // convolution
    int ic, ih, iw, ow, ohw, fh, fw, sh, sw, ph, pw, dh, dw;
    FastDiv d_ohw, d_ow, d_taps, d_fw;
};

// The arguments as the first thing, in one round trip: asked for where they are used, two to five round trips one after
// the other stood in front of the first load.
template <bool CONV, bool STRIPS>
__device__ __forceinline__ void ks_begin(const KsParams& q) {
#ifndef MG_HOST_AUDIT
    asm volatile("" ::"s"(q.A), "s"(q.B), "s"(q.C), "s"(q.a_bytes), "s"(q.b_bytes), "s"(q.a_row), "s"(q.a_k), "s"(q.b_row), "s"(q.b_k), "s"(q.M),
                 "s"(q.N), "s"(q.K), "s"(q.ldc), "s"(q.lw));
    if (STRIPS)
        asm volatile("" ::"s"(q.tiles), "s"(q.per_xcd), "s"(q.strip_w), "s"(q.strips), "s"(q.d_strip.mul), "s"(q.d_w.mul), "s"(q.d_last.mul));
    if (CONV)
        asm volatile("" ::"s"(q.bias), "s"(q.act), "s"(q.ic), "s"(q.ih), "s"(q.iw), "s"(q.ow), "s"(q.ohw), "s"(q.fh), "s"(q.fw), "s"(q.sh), "s"(q.sw),
                     "s"(q.ph), "s"(q.pw), "s"(q.dh), "s"(q.dw), "s"(q.d_ohw.mul), "s"(q.d_ow.mul), "s"(q.d_taps.mul), "s"(q.d_fw.mul));
#endif
}

static constexpr int KS_MAX_WAVES = 8;
static constexpr int KS_MAX_CONV_K = 4096;  // table entries (8 bytes each)
static constexpr int KS_SHORT = 28;         // steps of a short K: up to seven for each of four waves

// STRIPS: tiles in strips on the XCDs (ks_launch); else a grid of tiles.
// SHORT: four waves of up to seven steps each, which never come to the loop that keeps the ring full and have no sums to close
// (32 x 32: 155 registers for 236 with 64 x 64 outputs). In one instantiation with a number of waves from the arguments and the
// strips' arithmetic, products of K under 230 had lost 2 - 6 % to the kernel before there were strips. us, that kernel, all in one, apart:
// 2882 x 226 x 641 nt 17.3, 18.3, 17.1, 2000 x 200 x 900 tn 13.0, 13.4, 11.7, 637 x 117 x 1589 tn 6.9, 7.0, 6.0, 3118 x 140 x 293
// 7.7, 7.8, 6.95, 2500 x 200 x 700 13.2, 13.4, 11.8; convolution 9 -> 101 77 x 77 N=2 10.8, 11.0, 9.8, 21 -> 69 26 x 30 N=13 9.5,
// 9.6, 9.2. (The number of waves fixed for a long K too: the addresses of all its steps spilled, 1024^3 tn 56.4 us for 21.6.)
template <int AM, int BMODE, int R, int MT, int NT, bool TAIL, bool STRIPS, bool SHORT>
__global__ void __launch_bounds__(64 * KS_MAX_WAVES) gemm_f32_ks_kernel(KsParams q) {
    constexpr int RING = 4;  // (full >> (2 + lw) below)
    constexpr bool GATHER = BMODE == KS_CONV, CONV = GATHER || BMODE == KS_CONV1;
    // lanes along an operand's rows, groups of lanes along K, values of K a step, sums of a tile per lane
    constexpr int H = 64 / R, KS = 4 * H, LKS = R == 32 ? 3 : 4, SUMS = R * R / 64;
    typedef typename KsTile<R>::Sums Sums;
    static_assert(!CONV || NT == 1, "one pixel per lane");
    extern __shared__ __attribute__((aligned(16))) float ks_lds[];
    ks_begin<CONV, STRIPS>(q);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lw = SHORT ? 2 : q.lw, W = 1 << lw;
    const int h = lane / R, c = lane & (R - 1);
    int tx = blockIdx.x, ty = blockIdx.y;
    if constexpr (STRIPS) {
        const int place = (tx & 7) * q.per_xcd + (tx >> 3);
        if (place >= q.tiles)  // (the whole workgroup)
            return;
        const int strip = (int)fdiv(place, q.d_strip), in = place - strip * (int)q.d_strip.d;
        const bool last = strip == q.strips - 1;
        ty = last ? (int)fdiv(in, q.d_last) : (int)fdiv(in, q.d_w);
        tx = strip * q.strip_w + in - ty * (int)(last ? q.d_last.d : q.d_w.d);
    }
    const int m0 = ty * (R * MT), n0 = tx * (R * NT);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)q.A, 0, (int)q.a_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)q.B, 0, (int)q.b_bytes, 0x00020000);

    // Whole steps, dealt to the waves RING at a time where K is long - 4 steps are one 128-byte line of an
    // operand that is contiguous along K, fetched by one wave back to back instead of by four waves that
    // drift apart - and one at a time where that would leave waves without work.
    // SHORT: a wave's steps follow one another too, as many for each wave; where both operands are contiguous along K that is
    // twice the lines a wave comes back to, more than the L1 holds, and the waves take the steps of a line in turn (us in
    // turn / one run: 2500 x 180 x 700 15.2 / 13.3, 1500 x 170 x 1500 16.3 / 15.1; nt 2882 x 226 x 641 17.1 / 18.9, 2500 x 224 x 700
    // 14.7 / 14.3, 274 x 186 x 2814 8.9 / 9.1).
    const int full = q.K >> LKS;
    const bool lines = !SHORT && full >= 4 * RING * W;
    const int s_wave = lines ? RING : 1, s_ring = lines ? 1 : W;  // step = j0 * W + wave * s_wave + r * s_ring
    const int rounds = full >> (2 + lw), over = full - (rounds << (2 + lw));
    const int nj = lines ? rounds * RING + min(max(over - RING * wave, 0), RING)
                         : full > wave ? (full - wave + W - 1) >> lw : 0;

    // byte offset of (row, k = 4 h) of each operand tile
    unsigned aoff[MT], boff[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
        aoff[i] = (unsigned)min(m0 + i * R + c, q.M - 1) * q.a_row + (unsigned)(4 * h) * q.a_k;
    int* const tab = (int*)ks_lds;
    int* const pix = tab + (GATHER ? (q.K + KS - 1) / KS * (2 * KS) : 0);  // [offset, outside, image, place in it][32]
    if (CONV) {
        // The lane's pixel and, for a gather, the table: per k the byte offset and 31 - tap (0 - the bit
        // that is always set - beyond K), in groups of four: 4 offsets, 4 shifts. One wave works out the 32
        // pixels and the others the table: done by every wave, the index arithmetic was half of a small
        // layer's time.
        if (wave == 0 && lane < R) {
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
            for (int k = tid - 64; k < (q.K + KS - 1) / KS * KS; k += 64 * W - 64) {
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
            boff[j] = (unsigned)min(n0 + j * R + c, q.N - 1) * q.b_row + (unsigned)(4 * h) * q.b_k;
    }
    unsigned outside = 0;
    int img = 0, rem = 0;

    auto load_a = [&](int s, ks_v4f (&v)[MT]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            if (AM == KS_CONTIG) {
                v[i] = __builtin_bit_cast(ks_v4f, __builtin_amdgcn_raw_buffer_load_b128(ra, (int)(aoff[i] + (unsigned)s * (4u * KS)), 0, 0));
            } else {
                const unsigned o = aoff[i] + (unsigned)s * ((unsigned)KS * q.a_k);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra, (int)(o + (unsigned)e * q.a_k), 0, 0));
            }
        }
    };
    auto load_b = [&](int s, ks_v4f (&v)[NT]) __attribute__((always_inline)) {
        if (GATHER) {
            const v4i o = *(const v4i*)(tab + (H * s + h) * 8), sh = *(const v4i*)(tab + (H * s + h) * 8 + 4);
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
                v[j] = __builtin_bit_cast(ks_v4f, __builtin_amdgcn_raw_buffer_load_b128(rb, (int)(boff[j] + (unsigned)s * (4u * KS)), 0, 0));
            } else {
                const unsigned o = boff[j] + (unsigned)s * ((unsigned)KS * q.b_k);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, (int)(o + (unsigned)e * q.b_k), 0, 0));
            }
        }
    };
    // (the one tile of 16 x 16 has a chain for each product of a step: four in flight, and shorter sums - relative error of
    // 100 x 500 x 600 1.65e-7 with one, 0.97e-7 with four, 1.54e-7 with 32 x 32 tiles)
    constexpr int CHAINS = R == 16 ? 4 : 1;
    Sums acc[CHAINS][MT][NT], sum[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < SUMS; ++e) {
                sum[i][j][e] = 0.f;
#pragma unroll
                for (int x = 0; x < CHAINS; ++x)
                    acc[x][i][j][e] = 0.f;
            }
    auto close = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < SUMS; ++e) {
                    sum[i][j][e] += CHAINS == 4 ? (acc[0][i][j][e] + acc[1 % CHAINS][i][j][e]) + (acc[2 % CHAINS][i][j][e] + acc[3 % CHAINS][i][j][e])
                                                : acc[0][i][j][e];
#pragma unroll
                    for (int x = 0; x < CHAINS; ++x)
                        acc[x][i][j][e] = 0.f;
                }
    };
    auto multiply = [&](const ks_v4f (&a)[MT], const ks_v4f (&b)[NT]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[e % CHAINS][i][j] = KsTile<R>::multiply(a[i][e], b[j][e], acc[e % CHAINS][i][j]);
    };

    // the step behind the last whole one, element by element
    ks_v4f at[MT], bt[NT];
    auto tail_k = [&](int e) { return min(full * KS + 4 * h + e, q.K - 1) - 4 * h; };
    if (TAIL)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                at[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra, (int)(aoff[i] + (unsigned)tail_k(e) * q.a_k), 0, 0));
    ks_v4f av[RING][MT], bv[RING][NT];
    constexpr bool RUN = SHORT && !(AM == KS_CONTIG && BMODE == KS_CONTIG);
    const int s0 = RUN ? wave * (full >> 2) + min(wave, full & 3) : wave * s_wave;
    auto step = [&](int j0, int r) { return min(RUN ? s0 + j0 + r : j0 * W + s0 + r * s_ring, full - 1); };
    if (nj > 0)
        static_for<RING>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            load_a(step(0, r), av[r]);
        });
    // (16 x 16: the bias of the row this lane finishes, asked for here, not behind the sums. 32 x 32 tiles, several a CU, fetch
    // theirs where they are used: with four prefetched and an epilogue unrolled for them, 21 -> 69 26 x 30 N=13 10.1 us for 9.6.)
    float bias = 0.f;
    if (CONV && R == 16 && q.bias)
        bias = q.bias[min(m0 + 4 * h + (wave & 3), q.M - 1)];
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
    // Few rows of a transposed B, which gevm_f32.hip had before: the last runs of a wave are closed after two steps, not four, else the error is up to
    // 1.13 times as large as there (relative error there / after four / two: K = 256 0.82e-7 / 0.93e-7 / 0.82e-7, 500 0.91 / 1.01 / 0.91, 1000 1.04 /
    // 1.04 / 1.00; after one, more roundings of the whole sum: K = 544 0.92 / 1.02 / 0.93 / 0.96). 0 - 4 % longer (2 x 300 x 1000 tt 3.63 / 3.66 us, 2 x 700 x 1000 4.36 / 4.54).
    const bool few = R == 16 && BMODE == KS_CONTIG && q.M <= 4;
    if (nj > 0) {
        static_for<RING>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            load_b(step(0, r), bv[r]);
        });
        // (whole groups with nothing under a condition: behind a conditional load the compiler has to assume
        //  fewer loads in flight than there are, and waits for more of them)
        int j0 = 0;
        for (; !SHORT && j0 + 2 * RING <= nj; j0 += RING) {
            static_for<RING>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                multiply(av[r], bv[r]);
                load_a((j0 + RING) * W + s0 + r * s_ring, av[r]);
                load_b((j0 + RING) * W + s0 + r * s_ring, bv[r]);
            });
            if (KS == 16 || (j0 & RING))  // (every 64 values of K)
                close();
        }
        for (; j0 < nj; j0 += RING) {
            static_for<RING>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                if (j0 + r < nj) {
                    multiply(av[r], bv[r]);
                    if (j0 + r + RING < nj) {
                        load_a(step(j0 + RING, r), av[r]);
                        load_b(step(j0 + RING, r), bv[r]);
                    }
                    if (few && r == 1)
                        close();
                }
            });
            if (KS == 16)
                close();
        }
    }
    if (TAIL && wave == (lines ? W - 1 : full & (W - 1))) {  // (the wave whose turn it is)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const bool in = full * KS + 4 * h + e < q.K;
#pragma unroll
            for (int i = 0; i < MT; ++i)
                at[i][e] = in ? at[i][e] : 0.f;
#pragma unroll
            for (int j = 0; j < NT; ++j)
                bt[j][e] = in ? bt[j][e] : 0.f;
        }
        multiply(at, bt);
    }

    if (R == 16)
        close();

    // the waves' sums meet in LDS: [wave][tile][register][lane]
    if (CONV)
        __syncthreads();  // (the table's room is used again)
    constexpr int TILE = MT * NT * R * R;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < SUMS; ++e)
                ks_lds[wave * TILE + ((i * NT + j) * SUMS + e) * 64 + lane] = R == 16 ? sum[i][j][e] : SHORT ? acc[0][i][j][e] : acc[0][i][j][e] + sum[i][j][e];
    __syncthreads();
    // register e of a tile: row 8 * (e / 4) + 4 * h + e % 4 (16 x 16: 4 * h + e), column c. Wave w finishes registers w, w + W, ...
    for (int r = wave; r < MT * NT * SUMS; r += W) {
        const int t = r / SUMS, e = r & (SUMS - 1), i = t / NT, j = t - i * NT;
        float v = 0.f;
#pragma unroll 4
        for (int w = 0; w < W; ++w)
            v += ks_lds[w * TILE + r * 64 + lane];
        const int m = m0 + i * R + (R == 32 ? 8 * (e >> 2) : 0) + 4 * h + (e & 3), n = n0 + j * R + c;
        if (m >= q.M || n >= q.N)
            continue;
        if (CONV) {
            q.C[((size_t)img * q.M + m) * q.ohw + rem] = f32_act(q.act, v + (R == 16 ? bias : q.bias ? q.bias[m] : 0.f));
        } else {
            q.C[(size_t)m * q.ldc + n] = v;
        }
    }
}

// ---- choice of tile and waves -------------------------------------------------------------------------
struct KsPlan {
    int r, mt, nt, waves;  // tiles of r mt x r nt
    double cost;           // estimated cycles of the busiest CU
};

// Cycles of the busiest CU: its tiles' MFMAs (K / 2 of 64 cycles per 32 x 32 outputs, over four SIMDs) plus
// what its operands cost on their way through the CU's 64-byte-a-cycle port - half of that where a lane's 16
// bytes lie a row apart from its neighbours' - plus a round of latency for every set of workgroups that fits
// it at once. (Fitted: 2048^3 nt measured 248 / 203 / 159 us with tiles of 32x32 / 32x64 / 64x64, this says 238 /
// 208 / 178.)
static KsPlan ks_plan(long M, long N, long K, bool a_contig, bool b_contig, bool conv) {
    KsPlan best = {0, 0, 0, 0, 1e30};
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
                // 29.5 us with 4, 23.5 with 8, 25.2 with 16; 197 x 771 x 1003: 7.5, 8.6, 9.7; 64 -> 64 28 x 28 N=4 8.0, 7.0;
                // 400 x 640 x 333 6.0, 6.2)
                const int w = per_cu <= 1 && (K >= 1024 || tiles <= num_cus() / 2 || (conv ? K >= 512 : K >= 700 && tiles <= num_cus() * 5L / 8)) ? 8 : 4;
                best = {32, mt, nt, w, cost};
            }
        }
    // 16 x 16 tiles (the same rate on the matrix cores, four times the workgroups) where 32 x 32 ones leave CUs without any: a
    // tile's own chain is a quarter (64 x 1024 x 1000 7.5 us with 32 x 32, 4.8 with 16 x 16; 128 x 2048 x 512 nt 17.0 / 9.1; 33 x 500 x
    // 200 5.6 / 3.6; convolution 64 -> 64 28 x 28 6.7 / 4.3). Two a CU are still one round (32 -> 32 56 x 56 4.9 / 4.2, 300 x 2000 x
    // 400 13.4 / 9.6), unless one row of 32 x 32 tiles is all there is and the other operand, beyond the L2s, would be read
    // twice (20 x 3000 x 4000 16.0 / 17.0); with more, the operands' way in costs more than the idle CUs (500^3 6.0 / 8.1, 8 -> 16 112 x 112 4.7 / 5.4).
    // Eight waves where four would have more than seven steps each (16 x 312 x 1000 nt 3.7 us with four, 4.4 with eight, 4.0 with
    // 32 x 32 tiles; 16 x 512 x 1000 nt 4.0, 4.0; convolution 64 -> 64 28 x 28 4.6, 4.4).
    const long small = ((M + 15) / 16) * ((N + 15) / 16);
    const bool one_row = ((M > 16 && M <= 32) || (N > 16 && N <= 32)) && K * (M > N ? M : N) > (1L << 22);
    if (small <= num_cus() || (small <= 2L * num_cus() && !one_row))
        best = {16, 1, 1, small <= num_cus() && K >= 16 * (KS_SHORT + 1) ? 8 : 4, (double)K * 4.75 * (small <= num_cus() ? 1.0 : 2.0) + 3000.0};
    // Few rows of a transposed B in 16 x 16 tiles however many there are: 32 x 64 ones, whose waves add up to 64 values in a row, had up to 1.96 times
    // the error of gevm_f32.hip, which took them before (2 x 330 x 9000 1.69e-7 for 0.86e-7, now 0.85e-7). Us: 2 x 330 x 9000 7.2 / 4.9, 2 x 1000 x 9000 13.4 / 9.3, 2 x
    // 128 x 30000 5.7 / 6.5 (gevm_f32.hip 13.1); A not transposed 4 x 300 x 12000 6.8 / 5.2, 4 x 64 x 20000 4.1 / 5.4 (gevm_f32.hip 9.9).
    else if (!conv && M <= 4 && b_contig)
        best = {16, 1, 1, 4, (double)((small + num_cus() - 1) / num_cus()) * ((double)K * 4.75 + 1000.0) + 2000.0};
    // A convolution of up to 16 channels and a long K in rows of 16 however many there are: half of a 32 x 32 tile's products are for
    // channels that are not there (us, 32 x 32 / 16 x 16: 114 -> 11 46 x 57 stride 2 N=13 18.1 / 15.4, 95 -> 12 58 x 58 N=3 13.8 / 9.7, 33 -> 12
    // 83 x 17 N=6 7.7 / 6.0, 32 -> 8 69 x 18 N=13 6.9 / 5.7, 30 -> 9 33 x 33 N=8 7.0 / 5.2; with eight waves 15.6, 11.4, 8.5, -, 7.6). Below, a tile's
    // set-up is what counts (12 -> 11 57 x 108 N=2 4.6 / 5.2, 8 -> 14 41 x 84 N=5 4.6 / 6.5); from 17 channels on 32 x 32 is mostly the
    // quicker one (19 -> 17 65 x 65 stride 2 N=6 4.9 / 6.9, 100 -> 37 34 x 34 N=7 14.5 / 16.0).
    else if (conv && M <= 16 && K >= 250)
        best = {16, 1, 1, 4, (double)((small + num_cus() - 1) / num_cus()) * ((double)K * 6.2 + 1000.0)};
    return best;
}

// What the tiled kernel of gemm_f32.hip would take on the same scale: 128 x 128 tiles (4096^3: 1.14 times the
// MFMA cycles, 2048^3, one tile a CU and nothing to overlap with: 1.5 times, 175 us where 64 x 64 tiles take 151; a
// convolution's gather makes it 1.7 times that); it splits K and adds the slices in a second kernel below 192 tiles, where it never won.
static bool ks_wins(long M, long N, long K, bool conv, const KsPlan& p) {
    if (p.mt == 0)
        return false;
    const long tiles = ((M + 127) / 128) * ((N + 127) / 128), per_cu = (tiles + num_cus() - 1) / num_cus();
    if (tiles < 192 || (!conv && p.r == 16))
        return true;
    return p.cost < (double)K * 128.0 * (per_cu == 1 ? 1.55 : 1.14 * (double)per_cu) * (conv ? 1.7 : 1.0);
}

template <int AM, int BMODE>
static TinyNNStatus ks_launch(KsParams& q, const KsPlan& p, const char* what) {
    const bool tail = (q.K & (p.r == 32 ? 7 : 15)) != 0;
    constexpr bool CONV = BMODE == KS_CONV || BMODE == KS_CONV1;
    const int tm = p.r * p.mt, tn = p.r * p.nt;
    const int gx = (q.N + tn - 1) / tn, gy = (q.M + tm - 1) / tm;
    q.tiles = gx * gy;
    // The order of common.h's XcdOrder, but where the number of tiles is no multiple of eight with the same number for every
    // XCD and up to seven workgroups without one: strips begin with an XCD more often (64 x 4096 x 1000 12.5 / 12.0 us). Then for
    // 16 x 16 tiles - a row of theirs is half a line, and two XCDs would fetch each (64 x 4096 x 1000 17.2 without, 12.0 with) -
    // and for operands beyond an L2 (64 x 3000 x 3900 28.3 / 20.0, 200 x 2000 x 1100 16.3 / 12.6, 64 x 250 x 3900 4.65 / 4.64; below,
    // 1109 x 309 x 402 nt 7.6 / 7.9), not for convolutions (18 -> 48 27 x 46 N=13 9.0 / 9.9, 11 -> 98 29 x 29 N=8 7.9 / 8.3).
    const bool odd = (q.tiles & 7) != 0, order = !odd || (!CONV && (p.r == 16 || 4L * (q.M + q.N) * q.K > (4L << 20)));
    const int w = options().no_xcdorder || !order ? 0 : xcd_strip(gx, q.tiles);
    q.per_xcd = w ? (q.tiles + 7) / 8 : 0;
    q.strip_w = w ? w : gx, q.strips = (gx + q.strip_w - 1) / q.strip_w;
    q.d_strip = make_fastdiv((uint32_t)(q.strip_w * gy));
    q.d_w = make_fastdiv((uint32_t)q.strip_w);
    q.d_last = make_fastdiv((uint32_t)(gx - (q.strips - 1) * q.strip_w));
    const dim3 grid((unsigned)(w ? 8 * q.per_xcd : gx), (unsigned)(w ? 1 : gy));
    const bool brief = p.waves == 4 && (q.K >> (p.r == 32 ? 3 : 4)) <= KS_SHORT;
#define MG_KS_B(R_, MT_, NT_, T_, S_) (brief ? gemm_f32_ks_kernel<AM, BMODE, R_, MT_, NT_, T_, S_, true> : gemm_f32_ks_kernel<AM, BMODE, R_, MT_, NT_, T_, S_, false>)
#define MG_KS_S(R_, MT_, NT_, T_) (w ? MG_KS_B(R_, MT_, NT_, T_, true) : MG_KS_B(R_, MT_, NT_, T_, false))
#define MG_KS_T(R_, MT_, NT_) (tail ? MG_KS_S(R_, MT_, NT_, true) : MG_KS_S(R_, MT_, NT_, false))
    void (*kern)(KsParams);
    if (p.r == 16)
        kern = MG_KS_T(16, 1, 1);
    else if constexpr (CONV)  // (wider tiles never measured better for a convolution)
        kern = MG_KS_T(32, 1, 1);
    else
        kern = p.mt == 1 ? (p.nt == 1 ? MG_KS_T(32, 1, 1) : MG_KS_T(32, 1, 2)) : (p.nt == 1 ? MG_KS_T(32, 2, 1) : MG_KS_T(32, 2, 2));
#undef MG_KS_T
#undef MG_KS_S
#undef MG_KS_B
    q.lw = p.waves == 8 ? 3 : 2;
    note_kernel(what, tm, tn, p.waves, w);
    size_t lds = (size_t)p.waves * tm * tn * 4;
    const size_t table = (BMODE == KS_CONV ? (size_t)(q.K + 15) / 16 * 128 : 0) + (CONV ? 512 : 0);
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
    return v.b_cs != 1 && v.K > 3400 && (long)((v.M + 31) / 32) * ((v.N + 31) / 32) <= num_cus() / 2 &&
           (long)((v.M + 15) / 16) * ((v.N + 15) / 16) > num_cus();
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

// Where the tiled kernel would be faster by ks_wins, conv_f32_small.hip stands in front of it for layers under 2^27 multiply-adds:
// those run here. Few are left of them behind conv_f32_wide.hip, 50 of 200000 drawn layers under 2^27 (us, there / here: 9 x 1->23 62 x 44 3x3 9.4 /
// 4.5, 8 x 10->183 9 x 169 1x1 20.9 / 9.3, 3 x 2->188 240 x 17 3x3 37.3 / 10.7, 5 x 7->9 63 x 78 1x1 4.2 / 3.7, 2 x 7->2 240 x 204 1x1 stride 2 3.4 / 3.5).
bool conv_f32_ks_supported(const ConvGeom& g) {
    const long P = (long)g.n * g.oh * g.ow, K = (long)g.ic * g.fh * g.fw;
    return g.fmt == MEGCC_FMT_NCHW && g.groups == 1 && g.fh * g.fw <= 31 && K >= 1 && K <= KS_MAX_CONV_K && P >= 1 &&
           P < (1L << 30) && (long)g.n * g.ic * g.ih * g.iw < (1L << 29) - 65536 && (long)g.oc * K < (1L << 29) - 65536 &&
           P * g.oc < (1L << 31) && g.fh * g.fw >= 1 && (conv_f32_small_supported(g) || ks_wins(g.oc, P, K, true, conv_plan(g)));
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
