// A run of blocks - channel-wise 3x3 (pad 1, stride 1, RELU), then the pointwise 1x1 convolution of its result back to the same
// number of channels (RELU) - as ONE kernel, qsi8 NCHW44, 256 or 512 channels on maps of up to 14 x 15 pixels: the middle of a
// MobileNet (five blocks of 512 channels at 14 x 14). One workgroup holds one image for the whole run in LDS (146 KB with 512 channels, 74 with 256), which
// every layer overwrites in place. As one kernel a block (conv_dw_pw.hip) a workgroup's tile of 64 pixels waits for its pixels
// from HBM in every one of its four channel-wise jobs, takes the whole filter (256 KB) for every tile, and each block
// begins when the last tile of the one before is done.
//
// In LDS: [channels / 16][16 rows][16 slots] pieces of 16 channels; map row y is row y + 1, the rows around it and the slots
// past its width hold zeros (the padding), which nothing overwrites.
//   Channel-wise: a wave has the 2 or 4 plane groups of 16 channels whose pointwise results it will also write, so no other wave
//   is waited for. A product v_mfma_i32_16x16x64_i8 has 16 channels x 16 pixels of a row, K = 16 channels x 4 of the 9 filter taps,
//   the filter's bytes on a diagonal; two rows of outputs share three operands, each one ds_read_b128 a lane, of which one serves the next two as well. A lane ends up
//   with 4 channels of a pixel: a dword, written where the row was read once the rows below have been read.
//   Pointwise: a wave has 32 or 64 output channels; four, then three parts of 32 pixels (two map rows), requantised to registers, so that one
//   wave of a SIMD multiplies while the other requantises. When all waves are through, the results take the pixels' place. The
//   filter is streamed, four chunks of 32 channels ahead, across the parts and the layers: 512 KB a layer and image.
// Two barriers a layer. Both requantisations are the exact ones of epilogue.h: bit for bit the layers one by one.
// Bound: the matrix cores (19700 of a layer's 35400 cycles) and the vector ALU's issue (4000 instructions a SIMD with the products, 3.3 to 5 cycles each
// with two waves), which overlap in the pointwise half only. Counters: profiles/conv_blocks__5_blocks_14x14.txt.
// Measured (five blocks of 512 channels 14 x 14, us, pair by pair / as one kernel): N=64 60 / 76, 128 88 / 78, 256 146 / 94, 512 264 / 170; 256
// channels N=128 55 / 38, 256 76 / 43; MobileNetV1 batch 256 495 / 444. With the requantisation behind the barrier, where no wave
// multiplies, 96.8 for 91.5; operands moved by a lane (DPP) instead of three taps of a product 106; one channel group at a time 96.8 for 94.5.
#include <cstring>
#include <vector>

#include "common.h"
#include "conv_dw_pw.h"
#include "conv_mfma_i8.h"
#include "epilogue.h"

namespace mg {

static constexpr int CB_THREADS = 512, CB_ROWS = 16, CB_QUAD = CB_ROWS * 256;  // bytes of 16 channels' map
static constexpr int CB_PARTS = 7, CB_COLS = 15;  // parts of 32 pixels: 14 map rows; a row's last slot stays zero
// behind the maps: what the channel-wise operands of the last rows may reach into (read, met by zeros)
static constexpr int CB_PAD = 1024, CB_FRONT = 256;  // (in front of them zeros: the pixel left of the first map's first row)
struct BlockLayer {
    const uint32_t* dflt;  // [C/4][3][3] dwords of 4 channel bytes
    const int32_t* dbias;  // or NULL
    const int8_t* wp;      // packed pointwise filter [C/32][C][32], halves swapped when (oc >> 3) & 1
    const int32_t* pbias;  // or NULL
    RequantPack dq, pq;
};
template <int MT>
struct CbLds {
    static constexpr int C = 256 * MT, MAP = CB_FRONT + C / 16 * CB_QUAD + CB_PAD;
    static constexpr int FLT = C / 4 * 9, LAYER = FLT + 2 * C + 4;  // dwords of a layer: filter, biases, a zero
    static constexpr int BYTES = MAP + 2 * LAYER * 4;
};

// MT: 32-channel tiles of a wave; C = 256 MT
template <int MT>
__global__ void __launch_bounds__(CB_THREADS, 2) conv_blocks_kernel(
        const uint32_t* __restrict__ src, uint32_t* __restrict__ dst, const BlockLayer* __restrict__ layers, int count, int h, int w) {
    typedef CbLds<MT> L;
    constexpr int C = L::C, KC = C / 32, PQ = 2 * MT, RING = 4;
    extern __shared__ __attribute__((aligned(16))) int8_t cb_lds[];
    int8_t* const map = cb_lds + CB_FRONT;
    int* const par = (int*)(cb_lds + L::MAP);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hw4 = h * w * 4, image = C * h * w;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)src + (size_t)blockIdx.x * image), 0, image, 0x00020000);
    const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc((void*)((char*)dst + (size_t)blockIdx.x * image), 0, image, 0x00020000);
    const unsigned OOB = 0x80000000u;

    // ---- a layer's filter and biases, from memory to registers and to LDS
    constexpr int WI = (L::FLT + CB_THREADS - 1) / CB_THREADS;
    unsigned wv[WI];
    int dbv, pbv;
    auto ask = [&](const BlockLayer& q) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < WI; ++k)
            wv[k] = q.dflt[min(tid + k * CB_THREADS, L::FLT - 1)];
        // (no bias: some other bytes, not used)
        dbv = (q.dbias ? q.dbias : (const int32_t*)q.dflt)[min(tid, C - 1)];
        pbv = (q.pbias ? q.pbias : (const int32_t*)q.wp)[min(tid, C - 1)];
    };
    auto keep = [&](const BlockLayer& q, int* to) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < WI; ++k)
            if (tid + k * CB_THREADS < L::FLT)
                to[tid + k * CB_THREADS] = (int)wv[k];
        if (tid < C) {
            to[L::FLT + tid] = requant_start(q.dbias ? dbv : 0, q.dq);
            to[L::FLT + C + tid] = requant_start(q.pbias ? pbv : 0, q.pq);
        }
        if (tid == 0)
            to[L::FLT + 2 * C] = 0;
    };
    ask(layers[0]);

    // ---- pointwise filter: rows of this wave, RING chunks ahead
    const int col = lane & 31, kg = lane >> 5;
    int prow[MT];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
        const int oc = wave * (32 * MT) + mi * 32 + col;
        prow[mi] = oc * KROW + (((kg ^ (oc >> 3)) & 1) << 4);
    }
    __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)layers[0].wp, 0, KC * KROW * C, 0x00020000);
    v4i P[RING][MT];
    auto filter = [&](int c, v4i (&P)[MT]) __attribute__((always_inline)) {
#pragma unroll
        for (int mi = 0; mi < MT; ++mi)
            P[mi] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, prow[mi], c * (C * KROW), 0));
    };

    // ---- the image
    if (tid < CB_FRONT / 4)
        ((int*)cb_lds)[tid] = 0;
    {
        const int slot = tid & 255, y = (slot >> 4) - 1, x = slot & 15;
        const unsigned o = (unsigned)y < (unsigned)h && x < w ? (unsigned)((y * w + x) * 4) : OOB;
        const int half = __builtin_amdgcn_readfirstlane(tid >> 8);
#pragma unroll 4
        for (int k = 0; k < C / 32; ++k) {
            const int quad = 2 * k + half;
            v4i v;
#pragma unroll
            for (int p = 0; p < 4; ++p)
                v[p] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs, (int)o, (quad * 4 + p) * hw4, 0);
            *(v4i*)(map + quad * CB_QUAD + slot * 16) = v;
        }
    }
    keep(layers[0], par);
#pragma unroll
    for (int c = 0; c < RING; ++c)
        filter(c, P[c]);
    lds_barrier();

    // Channel-wise: pixel of the row, quarter of K / of the channels. Two rows of outputs take four rows of three pixels, twelve
    // operands of 16 channels, four to a product: the first row's three and the second's first, the second's and the fourth's
    // others, the third row's three and the fourth's first - what the next two rows begin with, already read. from[] is where a
    // lane's quarter of the first two lies, tap[] the filter's place that it meets (-1: none).
    const int colq = lane & 15, kg4 = lane >> 4;
    int from[2], tap[3][2];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int row = k == 1 ? (kg4 & 2) + 1 : kg4 / 3 + k, f = k == 1 ? 1 + (kg4 & 1) : kg4 % 3;
        if (k < 2)
            from[k] = row * 256 + (colq + f - 1) * 16;
#pragma unroll
        for (int r = 0; r < 2; ++r)
            tap[k][r] = (unsigned)(row - r) < 3u ? (row - r) * 3 + f : -1;
    }
    int diagonal[4];  // the byte of a quarter's 16 that is the lane's own channel
#pragma unroll
    for (int j = 0; j < 4; ++j)
        diagonal[j] = (colq >> 2) == j ? 0xff << 8 * (colq & 3) : 0;
    const unsigned inside = colq < w ? ~0u : 0u;  // (slots past the map's width stay zero)
    for (int l = 0; l < count; ++l) {
        const BlockLayer& q = layers[l];
        const int* const now = par + (l & 1) * L::LAYER;
        const bool last = l + 1 == count;
        if (!last)
            ask(layers[l + 1]);
        // ---- channel-wise
        requant_by_started_form(q.dq, [&](auto form) __attribute__((always_inline)) {
#pragma unroll 1
            for (int i = 0; i < PQ; i += 2) {
                // two maps of 16 channels at a time: one's products and reads stand between the other's
                v4i A[2][3][2], bias[2], U[2][2], M[2];
                const int8_t* in = map + (wave * PQ + i) * CB_QUAD;
                int8_t* out = map + (wave * PQ + i) * CB_QUAD + 256 + colq * 16 + kg4 * 4;
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const int quad = wave * PQ + i + m;
                    const int* const wl = now + (quad * 4 + (colq >> 2)) * 9;
#pragma unroll
                    for (int k = 0; k < 3; ++k)
#pragma unroll
                        for (int r = 0; r < 2; ++r) {
                            // (a select by lane costs as much as five of these: 17 cycles an instruction for 3.3)
                            const int v = *(tap[k][r] >= 0 ? wl + tap[k][r] : now + L::FLT + 2 * C);
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                A[m][k][r][j] = v & diagonal[j];
                        }
                    bias[m] = *(const v4i*)(now + L::FLT + quad * 16 + kg4 * 4);
#pragma unroll
                    for (int r = 0; r < 2; ++r)
                        U[r][m] = *(const v4i*)(in + from[0] + r * 512 + m * CB_QUAD);
                    M[m] = *(const v4i*)(in + from[1] + m * CB_QUAD);
                }
                // the sums of the next two rows, of which u has the filter's first rows and v the last ones; then u has what the two after
                // those end with
                auto product = [&](v4i (&acc)[2][2], v4i (&u)[2], const v4i (&v)[2]) __attribute__((always_inline)) {
                    in += 512;
#pragma unroll
                    for (int k = 0; k < 3; ++k)
#pragma unroll
                        for (int m = 0; m < 2; ++m) {
#pragma unroll
                            for (int r = 0; r < 2; ++r)
                                acc[m][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                                        A[m][k][r], k == 0 ? u[m] : k == 1 ? M[m] : v[m], k ? acc[m][r] : bias[m], 0, 0, 0);
                            if (k == 0)
                                u[m] = *(const v4i*)(in + from[0] + 512 + m * CB_QUAD);
                            else if (k == 1)
                                M[m] = *(const v4i*)(in + from[1] + m * CB_QUAD);
                        }
                };
                auto finish = [&](int y, const v4i (&acc)[2][2]) __attribute__((always_inline)) {
                    const unsigned mask[2] = {inside, inside & (unsigned)((y + 1 - h) >> 31)};  // (a row past the map's height stays zero)
#pragma unroll
                    for (int m = 0; m < 2; ++m)
#pragma unroll
                        for (int r = 0; r < 2; ++r)
                            *(unsigned*)(out + m * CB_QUAD + r * 256) =
                                    form(acc[m][r][0], acc[m][r][1], acc[m][r][2], acc[m][r][3]) & mask[r];
                    out += 512;
                };
                // (two rows' products stand in front of the two before's requantisation; what they read in front of what that writes)
                v4i acc[2][2][2];
                product(acc[0], U[0], U[1]);
                int y = 0;
#pragma unroll 1
                for (; y + 4 < h; y += 4) {
                    product(acc[1], U[1], U[0]);
                    finish(y, acc[0]);
                    product(acc[0], U[0], U[1]);
                    finish(y + 2, acc[1]);
                }
                if (y + 2 < h) {
                    product(acc[1], U[1], U[0]);
                    finish(y, acc[0]);
                    finish(y + 2, acc[1]);
                } else {
                    finish(y, acc[0]);
                }
            }
        });
        // (the other layer's place: the barriers of the layer before are behind its last readers)
        if (!last)
            keep(layers[l + 1], par + ((l + 1) & 1) * L::LAYER);
        lds_barrier();
        // ---- pointwise: parts T0 .. T0 + NT - 1, requantised
        const int* const pb = now + L::FLT + C + wave * (32 * MT) + kg * 4;
        const int8_t* const op = map + kg * CB_QUAD + 256 + col * 16;
        uint32_t result[CB_PARTS][MT][4];
        auto parts = [&](auto t0, auto nt) __attribute__((always_inline)) {
            constexpr int T0 = decltype(t0)::value, NT = decltype(nt)::value;
            v16i acc[MT][NT], bias[MT];
#pragma unroll
            for (int mi = 0; mi < MT; ++mi)
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4) {
                    const v4i bv = *(const v4i*)(pb + mi * 32 + e4 * 8);
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        bias[mi][e4 * 4 + k] = bv[k];
                }
            v4i b[2][NT];
#pragma unroll
            for (int t = 0; t < NT; ++t)
                b[0][t] = *(const v4i*)(op + (T0 + t) * 512);
            static_for<KC>([&](auto cc) __attribute__((always_inline)) {
                constexpr int c = decltype(cc)::value, slot = c % RING;
                if (c + 1 < KC)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        b[(c + 1) & 1][t] = *(const v4i*)(op + (c + 1) * (2 * CB_QUAD) + (T0 + t) * 512);
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int mi = 0; mi < MT; ++mi)
                        acc[mi][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(P[slot][mi], b[c & 1][t], c ? acc[mi][t] : bias[mi], 0, 0, 0);
                // behind the last parts' last chunk comes the next layer's first (behind the last layer nothing: a buffer of no bytes)
                if (T0 > 0 && c + RING == KC)
                    rw = __builtin_amdgcn_make_buffer_rsrc((void*)layers[last ? l : l + 1].wp, 0, last ? 0 : KC * KROW * C, 0x00020000);
                filter((c + RING) % KC, P[slot]);
                __builtin_amdgcn_sched_barrier(0);
            });
            requant_by_started_form(q.pq, [&](auto form) __attribute__((always_inline)) {
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int mi = 0; mi < MT; ++mi)
#pragma unroll
                        for (int e4 = 0; e4 < 4; ++e4)
                            result[T0 + t][mi][e4] =
                                    form(acc[mi][t][e4 * 4], acc[mi][t][e4 * 4 + 1], acc[mi][t][e4 * 4 + 2], acc[mi][t][e4 * 4 + 3]);
            });
            __builtin_amdgcn_sched_barrier(0);
        };
        parts(std::integral_constant<int, 0>{}, std::integral_constant<int, 4>{});
        parts(std::integral_constant<int, 4>{}, std::integral_constant<int, 3>{});
        if (!last)
            lds_barrier();
#pragma unroll
        for (int t = 0; t < CB_PARTS; ++t) {
            const int y = 2 * t + (col >> 4), x = col & 15;
            const bool there = y < h && x < w;
#pragma unroll
            for (int mi = 0; mi < MT; ++mi) {
                uint32_t(&d)[4] = result[t][mi];
                if (last) {
                    const unsigned o = there ? (unsigned)((y * w + x) * 4 + kg * hw4) : OOB;
#pragma unroll
                    for (int e4 = 0; e4 < 4; ++e4)
                        __builtin_amdgcn_raw_buffer_store_b32(d[e4], rd, (int)o, (wave * (8 * MT) + mi * 8 + e4 * 2) * hw4, 0);
                } else {
                    // lanes 0 - 31 take the tile's first 16 channels of their pixel, lanes 32 - 63 the others
                    const auto p = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
                    const auto r = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
                    int8_t* const out = map + (wave * PQ + kg) * CB_QUAD + 256 + t * 512 + col * 16;
                    if (there)
                        *(v4i*)(out + mi * (2 * CB_QUAD)) = v4i{(int)p[0], (int)p[1], (int)r[0], (int)r[1]};
                }
            }
        }
    }
}

struct BlocksRun {
    BlockLayer* dev = nullptr;  // [2][count]: as DwPwBlock's two forms
    int count = 0, n = 0, h = 0, w = 0, mt = 0;
    bool affine = false;  // every layer of the first form by proven multiply-adds
    const uint32_t* src = nullptr;
    uint32_t* dst = nullptr;
};

static const void* cb_kernel(int mt) {
    return mt == 2 ? (const void*)conv_blocks_kernel<2> : (const void*)conv_blocks_kernel<1>;
}
static int cb_lds_bytes(int mt) {
    return mt == 2 ? CbLds<2>::BYTES : CbLds<1>::BYTES;
}

// A workgroup an image, two a CU with 256 channels: where fewer images leave CUs without one, runs are not even timed (us, pair by pair / as one
// kernel: five blocks of 512 channels N=64 60 / 76, 96 78 / 77, 104 81 / 77, 128 88 / 78; of 256 N=32 26 / 36, 52 45 / 36, 80 48 / 37). A tie
// alone loses beside the other stream: MobileNetV1 batch 88 191 / 198, 96 199 / 206, but 104 229 / 224, 112 243 / 222.
bool conv_blocks_takes(const Tensor& x) {
    const uint32_t* d = x.layout.dims;
    return x.layout.nr_dim == 5 && (d[1] == 64 || d[1] == 128) && (options().fuse_blocks || 5L * d[0] >= (d[1] == 128 ? 2L : 1L) * num_cus()) &&
           d[2] <= 2 * CB_PARTS && d[3] <= CB_COLS;
}

void conv_blocks_destroy(BlocksRun* run) {
    if (run && run->dev)
        megcc_gfx950_free(run->dev);
    delete run;
}

BlocksRun* conv_blocks_create(const DwPwBlock* const* blocks, int count) {
    if (count < 2)
        return nullptr;
    const DwPwArgs& first = blocks[0]->host[0].a;
    const int c = first.OC, h = first.oh, w = first.ow;
    if ((c != 256 && c != 512) || h > 2 * CB_PARTS || w > CB_COLS)
        return nullptr;
    std::vector<BlockLayer> layers(2 * (size_t)count);
    bool affine = true;
    for (int i = 0; i < count; ++i) {
        const DwPwArgs& a = blocks[i]->host[0].a;
        // (as many channels, rows and columns in as out: stride 1)
        if (blocks[i]->act != MEGCC_NONLINE_RELU || a.OC != c || a.OCP != c || a.src_bytes != a.dst_bytes || a.ih != h || a.iw != w || a.oh != h ||
            a.ow != w || a.src_bytes != first.src_bytes || (i && a.src != blocks[i - 1]->host[0].a.dst))
            return nullptr;
        for (int form = 0; form < 2; ++form) {
            const DwPwArgs& f = blocks[i]->host[form].a;
            layers[(size_t)(form * count + i)] = {f.dflt, f.dbias, f.wp, f.pbias, f.dq, f.pq};
        }
        affine = affine && a.dq.affine() && a.pq.affine();
    }
    BlocksRun* r = new BlocksRun();
    r->count = count, r->h = h, r->w = w, r->mt = c / 256, r->affine = affine;
    r->n = (int)(first.src_bytes / ((long)c * h * w));
    r->src = first.src;
    r->dst = blocks[count - 1]->host[0].a.dst;
    const size_t bytes = layers.size() * sizeof(BlockLayer);
    r->dev = (BlockLayer*)megcc_gfx950_malloc(bytes);
    // (the copy is over before anything reads it, on whichever stream)
    if (!r->dev || hipFuncSetAttribute(cb_kernel(r->mt), hipFuncAttributeMaxDynamicSharedMemorySize, cb_lds_bytes(r->mt)) != hipSuccess ||
        megcc_gfx950_memcpy_h2d(r->dev, layers.data(), bytes) != TinyNN_SUCCESS || hipStreamSynchronize(stream()) != hipSuccess) {
        conv_blocks_destroy(r);
        return nullptr;
    }
    return r;
}

TinyNNStatus conv_blocks_launch(const BlocksRun* r) {
    const bool affine = !options().no_affine;
    note_kernel("conv_blocks", r->mt * 256, r->count);
    note_requant_affine(affine && r->affine);
    const BlockLayer* const layers = r->dev + (affine ? 0 : r->count);
    if (r->mt == 2)
        hipLaunchKernelGGL(conv_blocks_kernel<2>, dim3(r->n), dim3(CB_THREADS), CbLds<2>::BYTES, stream(), r->src, r->dst, layers, r->count, r->h, r->w);
    else
        hipLaunchKernelGGL(conv_blocks_kernel<1>, dim3(r->n), dim3(CB_THREADS), CbLds<1>::BYTES, stream(), r->src, r->dst, layers, r->count, r->h, r->w);
    return check_launch("conv_blocks");
}

}  // namespace mg
