// Channel-wise 3x3 (pad 1, stride 1 or 2) and the pointwise 1x1 convolution of its result as ONE kernel,
// qsi8 NCHW44: the block a MobileNet is made of. Run as two kernels the tensor between them goes out and
// comes back - a third of the bytes of the whole network - and every block pays a second launch. Here
// it stays in LDS:
//   A workgroup of 8 waves walks over tiles of T = 64 SUB output pixels (slots: groups of 4 pixels of a
//   row; a row's last group may hang over). Per tile
//   1. channel-wise: a job is 16 channels (4 plane sets) x 64 pixels. The multiply-adds are products with
//      banded matrices on the matrix cores, as in dwconv_mfma.hip but on v_mfma_i32_16x16x64_i8: a column
//      is a group of 4 output pixels, the rows are 4 pixels x 4 channels, and K is 3 input rows (one quarter
//      of the lanes each) x the group's own 4 pixels as they lie in memory - one aligned 16-byte load per
//      lane, no byte loaded twice. (K = 16 pixels of ONE row, three products, loaded each piece four times:
//      the L1's data path was busy 67 % of the kernel.) The pixels left and right of the group come from the
//      neighbouring columns, two row shifts (DPP) and a v_mfma_i32_16x16x32_i8; those of the first and last
//      column by one dword load. With stride 2 the group has 8 pixels, two products and the one on its left.
//      A lane ends up with the 4 channels of one pixel: one dword, no shuffles. Four plane sets make the 16
//      consecutive channels of a pixel the next product wants: one ds_write_b128. With up to 128 channels a
//      wave has one job per tile and keeps its banded matrices in registers, else they are rebuilt per job
//      from the filter in LDS by v_perm.
//   2. pointwise: rows = output channels (the packed filter, in registers for the workgroup's life where it
//      fits 8 chunks per wave, else streamed from L2 a few chunks ahead), columns = 32 pixels, the operand
//      one conflict-free ds_read_b128 per 32 channels; 4 consecutive accumulators are a dword of the result.
//   The next job's 12 loads fly while a job is requantised, the next tile's first ones while the pointwise
//   product runs; two tile buffers, one barrier per tile.
// Both requantisations are the exact ones of epilogue.h, so the result is bit for bit the two kernels'.
// Bound: HBM on the large maps, the vector ALU's requantisation and the filter's way from L2 on the small
// ones; with one tile a workgroup the way from the launch to the first load (dp_begin).
// Measured (N=64, us, one kernel / two): 32x112x112->64 19.8 / 32.0, 64 s2 -> 128 17.0 / 25.5, 128x56x56->128 17.4 / 27.9,
// 256x28x28->256 12.8 / 22.1, 512x14x14->512 9.5 / 21.5, 1024x7x7->1024 11.0 / 20.2; N=1: 4.0 / 7.0, 4.4 / 6.5, 3.9 / 7.1,
// 4.6 / 7.2, 6.2 / 7.9, 9.5 / 9.9; N=256: 86 / 117 and, 512 channels, 31.0 / 49.2. Before the arguments came in one round trip,
// slices followed the number of tiles and addresses were constants from one place, N=1: 5.1, 5.6, 5.2, 6.4, 9.7, 17.0; N=64, 512 and
// 1024 channels: 10.9, 18.3. (Two jobs' operands in flight, 16 waves of 128 registers, the whole filter in registers, jobs
// and products of two wave halves in opposite order: each slower, 512 channels N=1 by 0.4 - 1.6 us.)
#include <cstring>
#include <map>
#include <mutex>

#include "common.h"
#include "conv_dw_pw.h"
#include "conv_geom.h"
#include "conv_mfma_i8.h"
#include "epilogue.h"

namespace mg {

static constexpr int DP_THREADS = 512;
static constexpr int DP_ALL_BUT_MFMA = 0x7f6;  // what may cross a scheduling barrier: vector, scalar and memory instructions
typedef unsigned dp_v2u __attribute__((ext_vector_type(2)));

// All of the arguments in one round trip: the compiler otherwise asks for each where it is used, and nine round trips one
// after the other stood in front of the first load (3300 of a workgroup's 22000 cycles at 512 channels; 0.9 us of a launch).
__device__ __forceinline__ DwPwArgs dp_args(const DwPwParams* p) {
#ifdef MG_HOST_AUDIT
    return p->a;
#else
    typedef unsigned v16u __attribute__((ext_vector_type(16)));
    typedef const __attribute__((address_space(4))) v16u* lines;
    union {
        v16u v[4];
        DwPwArgs a;
    } u;
    const lines w = (lines)(uintptr_t)p;
    u.v[0] = w[0], u.v[1] = w[1], u.v[2] = w[2], u.v[3] = w[3];
    return u.a;
#endif
}

#ifndef MG_HOST_AUDIT
DwPwBlock* dw_pw_block_create() {
    return new DwPwBlock();
}
void dw_pw_block_destroy(DwPwBlock* b) {
    if (b && b->dev)
        megcc_gfx950_free(b->dev);
    delete b;
}
static TinyNNStatus dp_upload(DwPwBlock* b) {
    DwPwParams* const dev = (DwPwParams*)megcc_gfx950_malloc(sizeof(b->host));
    MG_REQUIRE(dev, TinyNN_ERROR_MEMORY_MALLOC, "conv_dw_pw: arguments");
    // (the copy is over before anything reads it, on whichever stream)
    TinyNNStatus st = megcc_gfx950_memcpy_h2d(dev, b->host, sizeof(b->host));
    if (st == TinyNN_SUCCESS && hipStreamSynchronize(stream()) != hipSuccess)
        st = fail(TinyNN_ERROR_RUNTIME, "conv_dw_pw: arguments");
    if (st != TinyNN_SUCCESS)
        megcc_gfx950_free(dev);
    else
        b->dev = dev;
    return st;
}
#endif

// a scalar whose origin the compiler does not know: sums made from it stay where they are written, instead of one register (and,
// beyond what there are, one spill) for every chunk and plane ahead of the loop
__device__ __forceinline__ int dp_opaque(int v) {
#ifndef MG_HOST_AUDIT
    asm volatile("" : "+s"(v));
#endif
    return v;
}

// LDS bytes of an instantiation
template <int KC, int SUB>
constexpr int dp_lds(int oc) {
    const int C = 32 * KC;
    return 2 * (64 * SUB) * C + C * 16 + C * 4 + oc * 4;
}

// S: stride; KC: 32-channel chunks; SUB: 64-pixel parts of a tile; MT, NT: 32-channel and 32-pixel tiles per
// wave of the pointwise product; RAG: IW % 4 (the input pixel right of a row's end is in its last piece)
// DACT, PACT: activations of the two layers (IDENTITY / RELU)
template <int S, int KC, int SUB, int MT, int NT, int RAG, int DACT, int PACT>
__global__ void __launch_bounds__(DP_THREADS, 2) conv_dw_pw_kernel(const DwPwParams* __restrict__ params) {
    constexpr int C = 32 * KC, NQ = 2 * KC, T = 64 * SUB;
    constexpr int JW = NQ * SUB / 8;                 // channel-wise jobs per wave and tile
    constexpr int WP = T / (32 * NT), WO = 8 / WP;   // waves along the pixels, along the channels
    constexpr bool KEEP_D = JW == 1 && S == 1, KEEP_P = KC * MT <= 8;
    // chunks of the pointwise filter in flight (not KEEP_P). More of them only stand in front of the channel-wise
    // operands: 8 for 4 chunks, 512 channels at N=256 33.1 for 32.2 us, stride 2 21.2 for 20.4
    constexpr int RING = MT == 1 || KC < 16 ? 8 : 4;
    static_assert(JW >= 1 && WP >= 1 && WO >= 1 && WP * WO == 8, "8 waves");
    const DwPwArgs q = dp_args(params);
    extern __shared__ __attribute__((aligned(16))) int8_t dp_lds_mem[];
    int8_t* const mid = dp_lds_mem;                             // [2][NQ][T] 16-byte pieces
    int* const wl = (int*)(mid + 2 * T * C);                    // [C][4]: per channel the filter's 3 rows
    int* const db = wl + C * 4;                                 // [C] bias
    int* const pb = db + C;                                     // [OC slice] bias
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ocs = WO * 32 * MT;                               // channels of a slice

    // Workgroup -> (slice, run of tiles). Each XCD gets a contiguous eighth of the tiles, and the runs with a tile more are the
    // first ones of every XCD: one to a CU, not two (the first runs of all were, and sat on the same XCDs: 784 tiles for two
    // workgroups a CU were four tiles for the CUs of three XCDs and two for the others).
    const int bx = blockIdx.x & 7, bi = blockIdx.x >> 3;
    const int xcd = q.xcds == 8 ? bx : 0, xi = q.xcds == 8 ? bi : q.per_xcd ? bx * q.per_xcd + bi : blockIdx.x;
    const int wi = (int)fdiv(xi, q.d_slices), slice = xi - wi * q.slices;
    const bool more = xcd < q.xcd_r, full = more && q.run_r + 1 == q.xcd_runs;  // (a tile more makes every run longer)
    const int run_q = q.run_q + (full ? 1 : 0), run_r = full ? 0 : q.run_r + (more ? 1 : 0);
    const int t_begin = xcd * q.xcd_q + min(xcd, q.xcd_r) + wi * run_q + min(wi, run_r), t_end = t_begin + run_q + (wi < run_r ? 1 : 0);

    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)q.src, 0, q.src_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc((void*)q.dst, 0, q.dst_bytes, 0x00020000);
    const unsigned OOB = 0x80000000u;
    const int colq = lane & 15, kg4 = lane >> 4;   // channel-wise: column, quarter of K / pixel of the group
    const int col = lane & 31, kg = lane >> 5;     // pointwise: column, half of K

    // what a lane (column colq, input row kg4) reads of a job: byte offsets in plane set 0
    struct Rows {
        unsigned off, offb;   // the group's pixels (S = 2: offb the second four)
        unsigned eoff;        // first / last column: the pixel left / right of the columns
        unsigned lmask, rmask;
        bool edge, edgeb;     // RAG: the piece (second piece) holds the pixel right of the row's end
    };
    auto rows_of = [&](int tile, int u) __attribute__((always_inline)) -> Rows {
        const int g = tile * (16 * SUB) + u * 16 + colq;
        const int rg = (int)fdiv(g, q.d_xg), x0 = (g - rg * q.xg) * 4;
        const int n = (int)fdiv(rg, q.d_oh), y = rg - n * q.oh;
        const int ix = S * x0, iy = S * y - 1 + kg4;
        const bool ok = g < q.groups && tile < t_end && kg4 < 3 && (unsigned)iy < (unsigned)q.ih;
        const unsigned o = (unsigned)(n * (C / 4) * q.plane + (iy * q.iw + ix) * 4);
        Rows r;
        r.off = ok ? o : OOB;
        r.offb = ok && ix + 4 < q.iw ? o + 16 : OOB;
        const bool l = x0 > 0, rt = ix + 4 < q.iw;
        r.lmask = l ? ~0u : 0u;
        r.rmask = rt ? ~0u : 0u;
        r.eoff = ok && colq == 0 && l ? o - 4 : S == 1 && ok && colq == 15 && rt ? o + 16 : OOB;
        r.edge = RAG != 0 && ix + 4 > q.iw;
        r.edgeb = RAG != 0 && ix + 4 <= q.iw && ix + 8 > q.iw;
        return r;
    };
    v4i B[4][S];
    unsigned E[4];
    // job i of this wave: channels 16 quad .. + 15, pixels 64 u .. + 63 of the tile
    // (several jobs a tile: tiles of 64 pixels)
    static_assert(JW == 1 || SUB == 1, "");
    const int quad0 = SUB == 1 ? wave : wave % NQ, sub0 = SUB == 1 ? 0 : wave / NQ;
    const int plane0 = quad0 * 4 * q.plane;
    auto request = [&](const Rows& r, int i) __attribute__((always_inline)) {
        int pl = dp_opaque(plane0 + i * (32 * q.plane));
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            B[p][0] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)r.off, pl, 0));
            if (S == 2)
                B[p][S - 1] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)r.offb, pl, 0));
            E[p] = __builtin_amdgcn_raw_buffer_load_b32(rs, (int)r.eoff, pl, 0);
            pl += q.plane;
        }
    };
    Rows rows = rows_of(t_begin, sub0), cur;
    request(rows, 0);

    // ---- set-up: filters, biases -----------------------------------------------------------
    // (all loads of a thread before its first store: a round trip for the whole set-up, not one per turn)
    constexpr int WI = (C * 4 + DP_THREADS - 1) / DP_THREADS, BI = (C + DP_THREADS - 1) / DP_THREADS;
    constexpr int PI = (WO * 32 * MT + DP_THREADS - 1) / DP_THREADS;
    uint32_t wv[WI][3];
    int dbv[BI], pbv[PI];
#pragma unroll
    for (int k = 0; k < WI; ++k) {
        const int i = min(tid + k * DP_THREADS, C * 4 - 1);
        const uint32_t* w = q.dflt + ((i >> 4) * 3 + min(i & 3, 2)) * 3;
#pragma unroll
        for (int j = 0; j < 3; ++j)
            wv[k][j] = w[j];
    }
    // (no bias: some other bytes, not used)
    const int32_t *dbp = q.dbias ? q.dbias : (const int32_t*)q.dflt, *pbp = q.pbias ? q.pbias : (const int32_t*)q.wp;
#pragma unroll
    for (int k = 0; k < BI; ++k)
        dbv[k] = dbp[min(tid + k * DP_THREADS, C - 1)];
#pragma unroll
    for (int k = 0; k < PI; ++k)
        pbv[k] = pbp[min(slice * ocs + tid + k * DP_THREADS, q.OC - 1)];
    // byte selectors of the banded matrices: row = (pixel colq >> 2, channel colq & 3) of the group, input row kg4;
    // the group's input pixel k meets it through filter column k + 1 - S px
    const int px = colq >> 2, sh = 8 * (colq & 3);
    auto selector = [&](int fw) { return (unsigned)fw < 3u ? (0x0c0c0c0cu & ~(0xffu << sh)) | ((unsigned)fw << sh) : 0x0c0c0c0cu; };
    unsigned sel[4 * S], sell = selector(-S * px), selr = selector(5 - px);  // (left: k = -1, right: k = 4)
#pragma unroll
    for (int k = 0; k < 4 * S; ++k)
        sel[k] = selector(k + 1 - S * px);
    // pointwise filter rows of this wave
    const int wo = wave % WO, wpx = wave / WO;
    const int oc_wave = slice * ocs + wo * (32 * MT);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)q.wp, 0, KC * KROW * q.OCP, 0x00020000);
    const int cstep = q.OCP * KROW;
    int prow[MT];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
        const int oc = min(oc_wave + mi * 32, q.OCP - 32) + col;
        prow[mi] = oc * KROW + (((kg ^ (oc >> 3)) & 1) << 4);
    }
    v4i P[KEEP_P ? KC : RING][MT];
    int next_chunk = 0;  // byte offset of the chunk to ask for next
    auto filter = [&](v4i (&P)[MT]) __attribute__((always_inline)) {
#pragma unroll
        for (int mi = 0; mi < MT; ++mi)
            P[mi] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, prow[mi], next_chunk, 0));
        next_chunk = dp_opaque(next_chunk + cstep);
    };
    // (what follows waits for the loads; nothing of the above may move behind it)
#ifndef MG_HOST_AUDIT
#pragma unroll
    for (int k = 0; k < 4 * S; ++k)
        asm volatile("" : "+v"(sel[k]));
    asm volatile("" : "+v"(sell), "+v"(selr), "+v"(prow[0]));
#endif
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < WI; ++k) {
        const int i = tid + k * DP_THREADS, dy = i & 3, sh = 8 * ((i >> 2) & 3);
        const uint32_t v = ((wv[k][0] >> sh) & 0xff) | (((wv[k][1] >> sh) & 0xff) << 8) | (((wv[k][2] >> sh) & 0xff) << 16);
        if (i < C * 4)
            wl[i] = dy < 3 ? (int)v : 0;  // (a fourth row of zeros)
    }
#pragma unroll
    for (int k = 0; k < BI; ++k)
        if (tid + k * DP_THREADS < C)
            db[tid + k * DP_THREADS] = requant_start(q.dbias ? dbv[k] : 0, q.dq);
#pragma unroll
    for (int k = 0; k < PI; ++k)
        if (tid + k * DP_THREADS < ocs)
            pb[tid + k * DP_THREADS] = requant_start(q.pbias ? pbv[k] : 0, q.pq);
    if (KEEP_P) {
#pragma unroll
        for (int c = 0; c < KC; ++c)
            filter(P[KEEP_P ? c : 0]);
    }
    lds_barrier();
    struct Band {
        v4i m[S];
        dp_v2u e;  // left, right
    };
    auto band_half = [&](unsigned w, int h) __attribute__((always_inline)) {
        v4i m;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            m[k] = (int)__builtin_amdgcn_perm(0u, w, sel[4 * h + k]);
        return m;
    };
    auto band_edges = [&](unsigned w) __attribute__((always_inline)) {
        return dp_v2u{__builtin_amdgcn_perm(0u, w, sell), S == 1 ? __builtin_amdgcn_perm(0u, w, selr) : 0u};
    };
    Band A[KEEP_D ? 4 : 1];
    if (KEEP_D) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const unsigned w = (unsigned)wl[((quad0 * 4 + p) * 4 + (colq & 3)) * 4 + kg4];
#pragma unroll
            for (int h = 0; h < S; ++h)
                A[KEEP_D ? p : 0].m[h] = band_half(w, h);
            A[KEEP_D ? p : 0].e = band_edges(w);
        }
    }

    // LDS places of a lane in job 0 and in the first pixel part of a product; everything else is a constant away
    const int* const wl0 = wl + ((quad0 * 4) * 4 + (colq & 3)) * 4 + kg4;
    const int* const db0 = db + quad0 * 16;
    const int mid0 = (quad0 * T + sub0 * 64 + colq * 4 + kg4) * 16;
    const int op0 = (kg * T + wpx * NT * 32 + col) * 16;
    // one channel-wise job: 16 channels (plane sets 4 quad ..), 64 pixels; `next` asks for what comes after it as soon as
    // its operands are consumed, so that those loads fly while this one is requantised
    auto channelwise = [&](int i, int8_t* m, auto next) __attribute__((always_inline)) {
        v4i acc[4];
        // the pixels left and right of each column's group
        unsigned L[4], R[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            L[p] = E[p];
            R[p] = E[p];
        }
#ifndef MG_HOST_AUDIT
        // (one block: a DPP read needs two cycles behind a vector write of its source)
        asm volatile(
                "s_nop 1\n\t"
                "v_and_b32_dpp %0, %4, %8 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
                "v_and_b32_dpp %1, %5, %8 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
                "v_and_b32_dpp %2, %6, %8 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
                "v_and_b32_dpp %3, %7, %8 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
                "s_nop 1"
                : "+v"(L[0]), "+v"(L[1]), "+v"(L[2]), "+v"(L[3])
                : "v"(B[0][S - 1][3]), "v"(B[1][S - 1][3]), "v"(B[2][S - 1][3]), "v"(B[3][S - 1][3]), "v"(cur.lmask));
        if (S == 1)
            asm volatile(
                    "s_nop 1\n\t"
                    "v_and_b32_dpp %0, %4, %8 row_shl:1 row_mask:0xf bank_mask:0xf\n\t"
                    "v_and_b32_dpp %1, %5, %8 row_shl:1 row_mask:0xf bank_mask:0xf\n\t"
                    "v_and_b32_dpp %2, %6, %8 row_shl:1 row_mask:0xf bank_mask:0xf\n\t"
                    "v_and_b32_dpp %3, %7, %8 row_shl:1 row_mask:0xf bank_mask:0xf\n\t"
                    "s_nop 1"
                    : "+v"(R[0]), "+v"(R[1]), "+v"(R[2]), "+v"(R[3])
                    : "v"(B[0][0][0]), "v"(B[1][0][0]), "v"(B[2][0][0]), "v"(B[3][0][0]), "v"(cur.rmask));
#endif
        // The short products of all four plane sets first, and every product where it stands (a scheduling
        // barrier behind each that only products may not cross). Products of ONE shape take their sums from the one
        // before at any distance; between the two shapes the sum must have been written: a 16x16x64 product
        // directly behind its 16x16x32 one has read channels 0 and 1 of the last pixels before that. A short
        // product takes 4 passes of 4 cycles and a few cycles to write; the three products in between alone
        // take 12 passes. (The build's code is checked for the three: test_mfma_order.py.)
        unsigned w[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            acc[p] = *(const v4i*)(db0 + i * 128 + p * 4);
            if (!KEEP_D)
                w[p] = (unsigned)wl0[(i * 32 + p) * 16];
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const dp_v2u al = KEEP_D ? A[KEEP_D ? p : 0].e : band_edges(w[p]), bl = {L[p], S == 1 ? R[p] : L[p]};
            acc[p] = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                    __builtin_bit_cast(long, al), __builtin_bit_cast(long, bl), acc[p], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(DP_ALL_BUT_MFMA);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < S; ++h)
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                v4i b = B[p][h];
                if (RAG)
                    b[RAG] = (h == 0 ? cur.edge : cur.edgeb) ? 0 : b[RAG];
                acc[p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                        KEEP_D ? A[KEEP_D ? p : 0].m[h] : band_half(w[p], h), b, acc[p], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(DP_ALL_BUT_MFMA);
            }
        __builtin_amdgcn_sched_barrier(0);
        next();
        int a[16];
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                a[p * 4 + e] = acc[p][e];
        uint32_t d[4];
        requant_dwords<DACT, true>(a, d, q.dq);
        *(v4i*)(m + mid0 + i * (8 * T * 16)) = v4i{(int)d[0], (int)d[1], (int)d[2], (int)d[3]};
    };
    // ---- pointwise: where a column's results go. (Stores are issued whether or not the place exists: what is under no
    // condition the compiler can count, and the next tile then waits for its loads, not for these stores.)
    const int ostep = q.oh * q.ow * 4;  // bytes of a plane set of the result
    auto where = [&](int t, int ni) __attribute__((always_inline)) {
        const int s = (wpx * NT + ni) * 32 + col;
        const int g = t * (16 * SUB) + (s >> 2);
        const int rg = (int)fdiv(g, q.d_xg), x = (g - rg * q.xg) * 4 + (s & 3);
        const int n = (int)fdiv(rg, q.d_oh), y = rg - n * q.oh;
        const unsigned o = (unsigned)((n * (q.OC >> 2) * q.oh + y) * q.ow + x) * 4u + (unsigned)(kg * ostep);
        return g < q.groups && x < q.ow ? o : OOB;
    };
    auto bias_of = [&](int mi, v16i& acc) __attribute__((always_inline)) {
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
            const v4i bv = *(const v4i*)(pb + wo * (32 * MT) + mi * 32 + e4 * 8 + kg * 4);
#pragma unroll
            for (int k = 0; k < 4; ++k)
                acc[e4 * 4 + k] = bv[k];
        }
    };
    auto finish = [&](int mi, unsigned w, const v16i& acc) __attribute__((always_inline)) {
        int a[16];
#pragma unroll
        for (int e = 0; e < 16; ++e)
            a[e] = acc[e];
        uint32_t d[4];
        requant_dwords<PACT, true>(a, d, q.pq);
        // (OC is a multiple of 32: all of the tile's channels exist or none)
        const bool there = oc_wave + mi * 32 < q.OC;
        const unsigned o = there ? w : OOB;
        const int plane = there ? (oc_wave + mi * 32) >> 2 : 0;
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4)
            __builtin_amdgcn_raw_buffer_store_b32(d[e4], rd, (int)o, (plane + e4 * 2) * ostep, 0);
    };
    auto operand = [&](const int8_t* m, int c, int ni) __attribute__((always_inline)) {
        return *(const v4i*)(m + op0 + c * (2 * T * 16) + ni * 512);
    };
    // (KEEP_P: nothing in flight from here, the loop's own waits are then exact)
    if (KEEP_P)
        wait_vmcnt<0>();
    for (int t = t_begin, buf = 0; t < t_end; ++t, buf ^= 1) {
        int8_t* const m = mid + buf * (T * C);
        cur = rows;
        static_for<JW>([&](auto ii) {
            constexpr int i = decltype(ii)::value;
            channelwise(i, m, [&]() __attribute__((always_inline)) {
                if (i + 1 < JW) {
                    request(rows, i + 1);
                } else if (KEEP_P) {
                    rows = rows_of(t + 1, sub0);
                    request(rows, 0);
                } else {
                    // the pointwise filter's first chunks
                    next_chunk = 0;
#pragma unroll
                    for (int c = 0; c < RING; ++c)
                        filter(P[c]);
                }
            });
        });
        lds_barrier();
        if constexpr (KEEP_P) {
            // one 32 x 32 tile after the other: 16 accumulators live, four waves to a SIMD
#pragma unroll
            for (int ni = 0; ni < NT; ++ni) {
                const unsigned w = where(t, ni);
#pragma unroll
                for (int mi = 0; mi < MT; ++mi) {
                    v16i acc;
                    bias_of(mi, acc);
#pragma unroll
                    for (int c = 0; c < KC; ++c)
                        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(P[c][mi], operand(m, c, ni), acc, 0, 0, 0);
                    finish(mi, w, acc);
                }
            }
        } else {
            v16i acc[MT][NT];
#pragma unroll
            for (int mi = 0; mi < MT; ++mi) {
                bias_of(mi, acc[mi][0]);
#pragma unroll
                for (int ni = 1; ni < NT; ++ni)
                    acc[mi][ni] = acc[mi][0];
            }
            static_for<KC>([&](auto cc) {
                constexpr int c = decltype(cc)::value, slot = c % RING;
#pragma unroll
                for (int ni = 0; ni < NT; ++ni) {
                    const v4i b = operand(m, c, ni);
#pragma unroll
                    for (int mi = 0; mi < MT; ++mi)
                        acc[mi][ni] = __builtin_amdgcn_mfma_i32_32x32x32_i8(P[slot][mi], b, acc[mi][ni], 0, 0, 0);
                }
                if (c + RING < KC)
                    filter(P[slot]);
                // the next tile's first job, behind the last chunk of the filter: loads come back in the order they
                // were issued, and one asked for after these would wait for them
                if (c + (RING < KC ? RING : KC) == KC) {
                    rows = rows_of(t + 1, sub0);
                    request(rows, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
#pragma unroll
            for (int ni = 0; ni < NT; ++ni) {
                const unsigned w = where(t, ni);
#pragma unroll
                for (int mi = 0; mi < MT; ++mi)
                    finish(mi, w, acc[mi][ni]);
            }
        }
    }
}

// the instantiation for C channels and OC: SUB, MT, NT
struct DpShape {
    int kc, sub, mt, nt;
};
static bool dp_shape(int c, int oc, long groups, DpShape* s) {
    // Slices of 128 or 256 channels while every slice of a tile has a CU to itself: the channel-wise layer is worked out
    // once a slice, but a workgroup's filter, products and requantisation are a quarter or half of 512 channels'. With two
    // slices to a CU that is no gain (us, with slices of 512 / 256 / 128 channels: 512 14 x 14 N=1 9.1 / - / 7.0, N=32
    // 9.6 / 8.3 / 11.7, N=64 10.5 / - / 19.9; 1024 7 x 7 N=1 13.3 / - / 10.5, N=64 14.3 / 12.4 / 18.5; 256 -> 512 stride 2 N=1
    // 7.1 / - / 5.4, N=64 8.4 / - / 12.5).
    const long tiles = (groups + 15) / 16;
    if (c == 256 || c == 512 || c == 1024)
        for (int nt = 1; nt <= 2; ++nt)
            if (tiles * ((oc + 128 * nt - 1) / (128 * nt)) <= num_cus()) {
                *s = {c / 32, 1, 1, nt};
                return true;
            }
    switch (c) {
        case 32: *s = {1, 4, 2, 1}; break;                        // 64 channels a slice
        case 64: *s = {2, 2, 2, 1}; break;                        // 128
        case 128: *s = oc <= 128 ? DpShape{4, 1, 1, 1} : DpShape{4, 1, 1, 2}; break;  // 128 / 256
        case 256: *s = oc <= 256 ? DpShape{8, 1, 1, 2} : DpShape{8, 1, 2, 2}; break;  // 256 / 512
        case 512: *s = {16, 1, 2, 2}; break;                      // 512
        case 1024: *s = {32, 1, 2, 2}; break;
        default: return false;
    }
    return true;
}

// (but for the scales: whether there are constants for them is asked when the arguments are written, not on every forward)
bool conv_dw_pw_supported(const ConvGeom& dw, const ConvGeom& pw, const void* src, const void* dst) {
    DpShape s;
    return dw.fmt == MEGCC_FMT_NCHW44 && dw.groups == dw.ic && dw.ic == dw.oc && dw.fh == 3 && dw.fw == 3 && dw.ph == 1 &&
           dw.pw == 1 && dw.dh == 1 && dw.dw == 1 && dw.sh == dw.sw && (dw.sh == 1 || dw.sh == 2) &&
           pw.fmt == MEGCC_FMT_NCHW44 && pw.groups == 1 && pw.fh == 1 && pw.fw == 1 && pw.sh == 1 && pw.sw == 1 && pw.ph == 0 &&
           pw.pw == 0 && pw.ic == dw.oc && (pw.oc & 31) == 0 && dp_shape(dw.ic, pw.oc, 0, &s) &&
           dw.act == MEGCC_NONLINE_RELU &&
           (pw.act == MEGCC_NONLINE_IDENTITY || pw.act == MEGCC_NONLINE_RELU) &&
           ((uintptr_t)src & 15) == 0 && ((uintptr_t)dst & 3) == 0 && (long)dw.n * dw.ic * dw.ih * dw.iw < (1L << 31) &&
           (long)pw.n * pw.oc * pw.oh * pw.ow < (1L << 31) && (long)dw.ih * dw.iw < (1L << 24) && dw.oh > 0 && dw.ow > 0;
}

template <int S, int KC, int SUB, int MT, int NT>
static void (*dp_kernel(int rag, int dact, int pact))(const DwPwParams*) {
    // (MobileNets use RELU behind both layers; a RELU-less pointwise layer is the linear bottleneck)
#define MG_DP_ACT(R_)                                                                                                   \
    (dact == MEGCC_NONLINE_RELU                                                                                          \
             ? (pact == MEGCC_NONLINE_RELU ? conv_dw_pw_kernel<S, KC, SUB, MT, NT, R_, MEGCC_NONLINE_RELU, MEGCC_NONLINE_RELU>        \
                                           : conv_dw_pw_kernel<S, KC, SUB, MT, NT, R_, MEGCC_NONLINE_RELU, MEGCC_NONLINE_IDENTITY>)   \
             : nullptr)
    return rag == 0 ? MG_DP_ACT(0) : rag == 1 ? MG_DP_ACT(1) : rag == 2 ? MG_DP_ACT(2) : MG_DP_ACT(3);
#undef MG_DP_ACT
}

// workgroups of `kern` one CU holds at a time; 0 where it cannot have its LDS. Asked for once per kernel (its LDS
// size goes with it).
static int dp_resident(const void* kern, size_t lds) {
    static std::map<const void*, int> cache;
    static std::mutex lock;
    std::lock_guard<std::mutex> guard(lock);
    auto it = cache.find(kern);
    if (it != cache.end())
        return it->second;
    int n = 0;
    if (lds > 48 * 1024 && hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, DP_THREADS, lds) != hipSuccess || n < 1)
        n = 1;
    return cache[kern] = n;
}

// `affine`: with the proven multiply-adds, where there are any
static TinyNNStatus dp_plan(
        const ConvGeom& dw, const ConvGeom& pw, const void* src, const void* dflt, const void* dbias, const void* packed,
        const void* pbias, void* dst, bool affine, DwPwParams& all, DpLaunch& l) {
    memset(all.words, 0, sizeof(all.words));
    DwPwArgs& q = all.a;
    DpShape s;
    q.xg = (dw.ow + 3) / 4;
    q.groups = dw.n * dw.oh * q.xg;
    MG_REQUIRE(dp_shape(dw.ic, pw.oc, q.groups, &s), TinyNN_ERROR_NO_IMPLEMENT, "conv_dw_pw: %d channels", dw.ic);
    q.src = (const uint32_t*)src;
    q.dflt = (const uint32_t*)dflt;
    q.dbias = (const int32_t*)dbias;
    q.wp = (const int8_t*)packed;
    q.pbias = (const int32_t*)pbias;
    q.dst = (uint32_t*)dst;
    q.src_bytes = (int)((long)dw.n * dw.ic * dw.ih * dw.iw);
    q.dst_bytes = (int)((long)pw.n * pw.oc * pw.oh * pw.ow);
    q.ih = dw.ih, q.iw = dw.iw, q.oh = dw.oh, q.ow = dw.ow;
    q.OC = pw.oc;
    q.OCP = (pw.oc + OC_PAD - 1) / OC_PAD * OC_PAD;
    q.plane = dw.ih * dw.iw * 4;
    const int tiles = (q.groups + 16 * s.sub - 1) / (16 * s.sub);
    const int wo = 8 / (64 * s.sub / (32 * s.nt)), ocs = wo * 32 * s.mt;
    q.slices = (pw.oc + ocs - 1) / ocs;
    q.d_xg = make_fastdiv(q.xg);
    q.d_oh = make_fastdiv(q.oh);
    q.d_slices = make_fastdiv(q.slices);
    q.dq = requant_started_for(dw.act, dw.s_src, dw.s_flt, dw.s_dst, affine);
    q.pq = requant_started_for(pw.act, pw.s_src, pw.s_flt, pw.s_dst, affine);
    MG_REQUIRE(q.dq.mode && q.pq.mode, TinyNN_ERROR_NO_IMPLEMENT, "conv_dw_pw: scales without proven constants");
    const int rag = dw.iw & 3;
    DwPwKernel kern = nullptr;
    size_t lds = 0;
#define MG_DP(KC_, SUB_, MT_, NT_)                                                                               \
    if (s.kc == KC_ && s.mt == MT_ && s.nt == NT_) {                                                                   \
        kern = dw.sh == 1 ? dp_kernel<1, KC_, SUB_, MT_, NT_>(rag, dw.act, pw.act) : dp_kernel<2, KC_, SUB_, MT_, NT_>(rag, dw.act, pw.act); \
        lds = (size_t)dp_lds<KC_, SUB_>(ocs);                                                                          \
    }
    MG_DP(1, 4, 2, 1)
    MG_DP(2, 2, 2, 1)
    MG_DP(4, 1, 1, 1)
    MG_DP(4, 1, 1, 2)
    MG_DP(8, 1, 1, 1)
    MG_DP(8, 1, 1, 2)
    MG_DP(8, 1, 2, 2)
    MG_DP(16, 1, 1, 1)
    MG_DP(16, 1, 1, 2)
    MG_DP(16, 1, 2, 2)
    MG_DP(32, 1, 1, 1)
    MG_DP(32, 1, 1, 2)
    MG_DP(32, 1, 2, 2)
#undef MG_DP
    MG_REQUIRE(kern, TinyNN_ERROR_NO_IMPLEMENT, "conv_dw_pw: no instance");
    const int resident = dp_resident((const void*)kern, lds);
    MG_REQUIRE(resident > 0, TinyNN_ERROR_RUNTIME, "conv_dw_pw: %d bytes of LDS", (int)lds);
    // as many workgroups as are resident, each with a run of tiles
    long runs = (long)num_cus() * resident / q.slices;
    if (runs < 1)
        runs = 1;
    if (runs > tiles)
        runs = tiles;
    q.xcds = runs % 8 == 0 ? 8 : 1;
    q.xcd_q = tiles / q.xcds, q.xcd_r = tiles - q.xcd_q * q.xcds;
    q.xcd_runs = (int)runs / q.xcds;
    q.per_xcd = runs * q.slices % 8 == 0 ? (int)runs * q.slices / 8 : 0;
    q.run_q = q.xcd_q / q.xcd_runs, q.run_r = q.xcd_q - q.run_q * q.xcd_runs;
    l = {kern, lds, (unsigned)(runs * q.slices)};
    return TinyNN_SUCCESS;
}

TinyNNStatus conv_dw_pw_launch(
        const ConvGeom& dw, const ConvGeom& pw, const void* src, const void* dflt, const void* dbias, const void* packed,
        const void* pbias, void* dst, DwPwBlock* block, bool prepare) {
    const bool affine = !options().no_affine;
#ifdef MG_HOST_AUDIT
    DwPwBlock here;
    block = &here;
    TinyNNStatus st = dp_plan(dw, pw, src, dflt, dbias, packed, pbias, dst, affine, here.host[!affine], here.launch);
    if (st != TinyNN_SUCCESS)
        return st;
    const DwPwParams* const args = &here.host[!affine];
#else
    if (prepare) {
        MG_REQUIRE(!block->dev, TinyNN_ERROR_RUNTIME, "conv_dw_pw: prepared before");
        for (int i = 0; i < 2; ++i) {
            TinyNNStatus st = dp_plan(dw, pw, src, dflt, dbias, packed, pbias, dst, i == 0, block->host[i], block->launch);
            if (st != TinyNN_SUCCESS)
                return st;
        }
        block->act = pw.act;
        return dp_upload(block);
    }
    MG_REQUIRE(block->dev, TinyNN_ERROR_RUNTIME, "conv_dw_pw: not prepared");
    const DwPwParams* const args = block->dev + !affine;
#endif
    const DwPwArgs& q = block->host[!affine].a;
    MG_REQUIRE(q.src == src && q.dflt == dflt && q.dbias == dbias && q.wp == packed && q.pbias == pbias && q.dst == dst,
               TinyNN_ERROR_RUNTIME, "conv_dw_pw: not the operands it was prepared for");
    note_kernel("conv_dw_pw", dw.ic / 32, dw.sh, q.slices);
    note_requant_affine(q.dq.affine() && q.pq.affine());
    hipLaunchKernelGGL(block->launch.kern, dim3(block->launch.workgroups), dim3(DP_THREADS), block->launch.lds, stream(), args);
    return check_launch("conv_dw_pw");
}

}  // namespace mg
