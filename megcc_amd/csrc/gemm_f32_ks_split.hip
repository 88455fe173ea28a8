// f32 MatMul of middle size, any transposition, by v_mfma_f32_32x32x16_bf16 at f32 accuracy.
//
// Between the products of many 128 x 128 tiles (gemm_f32_split.hip) and those of one round of small ones (gemm_f32_ks.hip) lie
// the ones whose tiles of 32 x 32 or 64 x 64 outputs are bound by the f32 instructions, by what a CU fetches - each multiplies 32
// or 64 values of one operand with every value of the other - and by a last round that leaves CUs idle. The parts are those of
// gemm_f32_split.hip (x = x1 + x2 + x3 in bf16, six of the nine products, each exact in f32):
//   * A workgroup of 8 waves owns 64 rows of one operand, L, and 64, 128 or 256 of the other, R. L's values are split once
//     for the workgroup, into LDS, 64 steps of K a stage, two stages ahead. A wave has 32 rows of R to itself: its values go from
//     memory to the registers the instruction reads and are split there, so 16 steps of K cost a wave 12 products
//     (384 cycles of the matrix unit), 4 pairs a lane to split and six 16-byte reads of LDS. (Both operands through LDS, 64 x 64
//     outputs, a wave 64 x 32: 8 pairs, nine reads and six writes; 512 x 4096 x 4096 140 us for 111, 1912 x 1206 x 1078 51 for 41.)
//   * With 64 (128) rows of R four (two) groups of waves share a stage's K; their sums meet in LDS. A workgroup may take a slice
//     of K; a second kernel then adds the slices in order.
//   * The five small products have sums of their own, of which a rounding costs 2^-8 of one of the large product's; both
//     are closed every 8 or 16 steps of a wave into a third set. Relative error against 64 bits 0.7 - 1.0e-7 (K = 360 ... 4096),
//     where gemm_f32_ks.hip has 1.0 - 1.7e-7.
//   * Which operand is L is the launch's choice (SWAP: L's rows are the result's columns).
//   * A wave splits step j + 1 while it multiplies step j; R's next four steps and L's next two stages are in flight.
//   * Values outside 2^-102 <= |x| < 2^60 (zero is fine) are met as in gemm_f32_split.hip: a workgroup that finds one in a
//     chain of stages multiplies its slice from that chain on by v_mfma_f32_32x32x2_f32.
//   * Stages behind the last come from a buffer of no bytes (zeros), the last K % 64 steps element by element, masked.
// Measured (us, gemm_f32_ks.hip / here): 512 x 4096 x 4096 154 / 109 (158 TFLOP/s of the product), 1912 x 1206 x 1078 58 / 41, 83 x 2794 x 3689
// nt 41 / 28.5, 1381 x 2795 x 925 nt 92 / 71, 3713 x 2717 x 528 138 / 110, 947 x 2247 x 657 nt 47 / 38. A wave's 16 steps take 0.74 - 0.9 us
// beside a second wave's, the products alone 0.4 (at 1.85 GHz): with half of the products left out 0.75 of the time, without R's
// split 0.83, every stage read from one place the same, so no one of them bounds it: by counter the matrix units are busy 0.47 of
// a CU's cycles at 512 x 4096 x 4096, 0.42 - 0.26 for the others (profiles/f32_products__few_rows_and_middle_size.txt).
// Fp32MatMulM4N12.cpp:9-158 is the loop replaced.
#include "common.h"
#include "conv_mfma_i8.h"
#include "f32_parts.h"
#include "gemm_f32_ks.h"
#include "gemm_f32_split.h"

namespace mg {

typedef float kp_v16f __attribute__((ext_vector_type(16)));
typedef float kp_v4f __attribute__((ext_vector_type(4)));
typedef float kp_v2f __attribute__((ext_vector_type(2)));
typedef unsigned kp_v4u __attribute__((ext_vector_type(4)));
typedef __bf16 kp_v2b __attribute__((ext_vector_type(2)));
typedef __bf16 kp_v8b __attribute__((ext_vector_type(8)));

enum { KP_CONTIG = 0, KP_STRIDED = 1 };  // along K

struct KpSide {
    const float* p;
    unsigned bytes, row, k;  // byte strides: of rows, along K
    int rows;
};
struct KpParams {
    KpSide l, r;
    float* C;
    int K, ldc, M, N;
    // workgroups on an XCD, in all; tiles of a slice of K; a slice's steps (a multiple of 64); tiles run along L's first or R's
    int per_xcd, total, tiles, chunk, l_first;
    int sliced;
    FastDiv d_tiles, d_run;
};

static constexpr int KP_L = 64, KP_K = 64, KP_STEP = 16;
// an LDS piece: 16 bytes of each of the 64 rows; the 16 bytes behind each keep the eight octets of a stage, which
// neighbouring threads write, on different banks
static constexpr int KP_PIECE = KP_L * 16 + 16;
static constexpr int KP_STAGE = 24 * KP_PIECE;  // [part][octet of the 64 steps][row]
static constexpr int KP_RING = 4;               // steps of R in flight

// Splits 8 values into three parts each, and looks at them.
// `ones`: -1 in the lower half, in the upper half of a register: the rest behind a part is one v_dot2 (exact) instead of a
// shift or a mask and a subtraction. (As constants the compiler gives the instruction its inline -1.0, whose lower half is 0.)
struct KpSplit {
    unsigned ones[2];
    PartsRange range;
    __device__ __forceinline__ void begin() {
        ones[0] = 0x0000bf80u, ones[1] = 0xbf800000u;
#ifndef MG_HOST_AUDIT
        asm volatile("" : "+v"(ones[0]), "+v"(ones[1]));
#endif
        range.begin();
    }
    __device__ __forceinline__ void split(const float (&v)[8], kp_v4u (&part)[3]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            kp_v2f x = {v[2 * i], v[2 * i + 1]};
            range.look(x[0], x[1]);
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                const kp_v2b b = __builtin_convertvector(x, kp_v2b);
                part[p][i] = __builtin_bit_cast(unsigned, b);
                if (p < 2) {
                    x[0] = __builtin_amdgcn_fdot2_f32_bf16(b, __builtin_bit_cast(kp_v2b, ones[0]), x[0], false);
                    x[1] = __builtin_amdgcn_fdot2_f32_bf16(b, __builtin_bit_cast(kp_v2b, ones[1]), x[1], false);
                }
            }
        }
    }
};

// what a lane reads of an operand: 8 steps of K, an octet, of one row
template <int MODE>
struct KpLane {
    const float* base;
    unsigned bytes, off, k_bytes;

    // `octet`: of what is loaded at a time
    __device__ __forceinline__ KpLane(const KpSide& s, int r, int octet) {
        base = s.p;
        bytes = s.bytes;
        k_bytes = s.k;
        off = (unsigned)min(r, s.rows - 1) * s.row + (unsigned)(8 * octet) * s.k;
    }
    // from step k0 on; `there`: there is such a stage (else zeros)
    __device__ __forceinline__ void load(int k0, bool there, float (&v)[8]) const {
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, there ? (int)bytes : 0, 0x00020000);
        if (MODE == KP_CONTIG) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const kp_v4u t = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off + 16 * i, k0 * 4, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[4 * i + e] = __uint_as_float(t[e]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                v[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)off, (int)((unsigned)(k0 + i) * k_bytes), 0));
        }
    }
    // (steps from `end` on: the last one's value is fetched instead and dropped)
    __device__ __forceinline__ void load_tail(int k0, int octet, int end, float (&v)[8]) const {
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00020000);
        const unsigned start = off - (unsigned)(8 * octet) * k_bytes;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = k0 + 8 * octet + i;
            const float t = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(start + (unsigned)min(k, end - 1) * k_bytes), 0, 0));
            v[i] = k < end ? t : 0.f;
        }
    }
};

// LM, RM: how the operands lie along K; KG: groups of waves that share a stage's K; SWAP: L's rows are the result's columns
template <int LM, int RM, int KG, bool SWAP>
__global__ void __launch_bounds__(512, 2) gemm_f32_ks_split_kernel(KpParams q) {
    constexpr int WN = 8 / KG, OWN = 4 / KG;    // waves along R; steps of a stage that are a wave's own
    constexpr int BODY = KG == 4 ? 4 : 2;       // stages of the loop's body: whole turns of R's ring and of L's two buffers
    constexpr int CHAIN = KG == 4 ? 8 : 4;      // stages per running sum
    constexpr bool AHEAD = KG == 2;             // L's operands are read a step ahead (the others would spill)
    constexpr int MEET = KG == 1 ? 16 : 8 * 32 * 64 * 4;
    __shared__ __attribute__((aligned(16))) char lds[4 * KP_STAGE > MEET ? 4 * KP_STAGE : MEET];
    __shared__ int beyond;  // some thread has split a value that the parts cannot hold
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5;
    const int wn = wave % WN, kg = wave / WN;
    // an XCD has a run of (slice, tile): slices one after the other, so that what the tiles of a slice share is in its L2
    const int place = (int)(blockIdx.x & 7) * q.per_xcd + (int)(blockIdx.x >> 3);
    if (place >= q.total)  // (the whole workgroup)
        return;
    const int z = (int)fdiv(place, q.d_tiles), in = place - z * q.tiles;
    const int major = (int)fdiv(in, q.d_run), minor = in - major * (int)q.d_run.d;
    const int l0 = (q.l_first ? minor : major) * KP_L, r0 = (q.l_first ? major : minor) * (32 * WN) + wn * 32;
    const int k_begin = z * q.chunk, k_end = min(k_begin + q.chunk, q.K);
    const int full = (k_end - k_begin) / KP_K, rest = k_begin + full * KP_K;
    // L: a thread splits one octet of one row a stage
    const int lrow = LM == KP_CONTIG ? tid >> 3 : lane, loct = LM == KP_CONTIG ? tid & 7 : wave;
    const KpLane<LM> sl(q.l, l0 + lrow, loct);
    const KpLane<RM> sr(q.r, r0 + (lane & 31), half);
    char* const lput = lds + loct * KP_PIECE + lrow * 16;
    const char* const lget = lds + half * KP_PIECE + (lane & 31) * 16;

    kp_v16f acc[2], small[2], sum[2];
    auto clear = [&](kp_v16f (&t)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                t[i][e] = 0.f;
    };
    clear(acc);
    clear(small);
    clear(sum);
    // (the small products first: what they add up to is then rounded as one of the large products' sums is)
    auto close = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                sum[i][e] += acc[i][e] + small[i][e];
        clear(acc);
        clear(small);
    };
    KpSplit sp;
    sp.begin();
    float vl[2][8], vr[KP_RING][8];
    kp_v4u pr[2][3];
    kp_v8b fl[AHEAD ? 2 : 1][3][2];
    auto load_l = [&](int s, float (&v)[8]) __attribute__((always_inline)) {
        const bool there = s < full;
        sl.load(k_begin + (there ? s : 0) * KP_K, there, v);
    };
    // step j of this wave: stage j / OWN, its steps OWN kg ... there
    auto load_r = [&](int j, float (&v)[8]) __attribute__((always_inline)) {
        const int s = j / OWN;
        const bool there = s < full;
        sr.load(k_begin + (there ? s * KP_K + (OWN * kg + j % OWN) * KP_STEP : 0), there, v);
    };
    auto put_l = [&](int buf, const float (&v)[8]) __attribute__((always_inline)) {
        kp_v4u part[3];
        sp.split(v, part);
#pragma unroll
        for (int p = 0; p < 3; ++p)
            *(kp_v4u*)(lput + buf * KP_STAGE + 8 * p * KP_PIECE) = part[p];
    };
    auto get_l = [&](int buf, int i16, kp_v8b (&fl)[3][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                fl[p][i] = *(const kp_v8b*)(lget + buf * KP_STAGE + (8 * p + 2 * i16) * KP_PIECE + i * 512);
    };
    auto multiply = [&](const kp_v8b (&fl)[3][2], const kp_v4u (&b)[3]) __attribute__((always_inline)) {
#define MG_KP_MUL(SUM, PL, PR)                                                                                                     \
    _Pragma("unroll") for (int i = 0; i < 2; ++i) SUM[i] =                                                                         \
            SWAP ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(kp_v8b, b[PR]), fl[PL][i], SUM[i], 0, 0, 0)          \
                 : __builtin_amdgcn_mfma_f32_32x32x16_bf16(fl[PL][i], __builtin_bit_cast(kp_v8b, b[PR]), SUM[i], 0, 0, 0)
        // smallest products first (gemm_f32_split.hip says why)
        MG_KP_MUL(small, 0, 2);
        MG_KP_MUL(acc, 0, 0);
        MG_KP_MUL(small, 2, 0);
        MG_KP_MUL(small, 1, 1);
        MG_KP_MUL(small, 0, 1);
        MG_KP_MUL(small, 1, 0);
#undef MG_KP_MUL
    };
    // Whether a thread has met such a value: report(), a barrier, reported(). Every thread then reads the same, since
    // at least one more barrier (a stage's) lies in front of the next report().
    auto report = [&]() __attribute__((always_inline)) {
        if (sp.range.beyond())
            beyond = 1;
    };
    auto reported = [&]() __attribute__((always_inline)) {
        return __builtin_amdgcn_readfirstlane(*(volatile int*)&beyond) != 0;
    };
    // the vector instructions of the next step's split go between the products of this one
    auto order = [&](auto vector) __attribute__((always_inline)) {
#ifndef MG_HOST_AUDIT
        __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);  // LDS reads
#pragma unroll
        for (int i = 0; i < 12; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                  // a product
            __builtin_amdgcn_sched_group_barrier(0x2, decltype(vector)::value, 0);  // vector instructions
        }
        __builtin_amdgcn_sched_barrier(0);
#endif
    };
    int kept = k_begin;  // steps of K whose products are in the sums for good
    bool f32 = false;
    load_l(0, vl[0]);
    load_l(1, vl[1]);
#pragma unroll
    for (int j = 0; j < KP_RING; ++j)
        load_r(j, vr[j]);
    if (tid == 0)
        beyond = 0;
    __builtin_amdgcn_sched_barrier(0);
    put_l(0, vl[0]);
    load_l(2, vl[0]);
    put_l(1, vl[1]);
    load_l(3, vl[1]);
    sp.split(vr[0], pr[0]);
    load_r(KP_RING, vr[0]);
    lds_barrier();
    if (AHEAD)
        get_l(0, OWN * kg, fl[0]);
    report();
    lds_barrier();
    f32 = reported();
    for (int s0 = 0; s0 < full && !f32; s0 += CHAIN) {
        if (s0) {
            close();
            kept = k_begin + s0 * KP_K;
        }
        const int s1 = min(s0 + CHAIN, full);
        for (int s = s0; s < s1; s += BODY) {
            static_for<BODY * OWN>([&](auto jc) {
                constexpr int j = decltype(jc)::value, st = j / OWN, t = j % OWN, next = (j + 1) % KP_RING;
                // (a stage lies in LDS two stages ahead: one barrier a stage orders its writes, in front of it, and the reads of
                // what was in its place)
                if (t == OWN - 1) {
                    lds_barrier();
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (AHEAD)
                    get_l((s + (j + 1) / OWN) & 3, OWN * kg + (j + 1) % OWN, fl[(j + 1) & 1 & AHEAD]);
                else
                    get_l((s + st) & 3, OWN * kg + t, fl[0]);
                if (t == 0) {
                    put_l((s + st + 2) & 3, vl[st & 1]);
                    load_l(s + st + 4, vl[st & 1]);
                }
                sp.split(vr[next], pr[(j + 1) & 1]);
                load_r(s * OWN + j + 1 + KP_RING, vr[next]);
                multiply(fl[j & 1 & AHEAD], pr[j & 1]);
                order(std::integral_constant<int, t == 0 ? 8 : 4>{});
            });
        }
        report();  // (of what lies behind the chain as well)
        lds_barrier();
        f32 = reported();
    }
    if (!f32 && rest < k_end) {
        sl.load_tail(rest, loct, k_end, vl[0]);
        __syncthreads();
        put_l(0, vl[0]);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < OWN; ++t) {
            sr.load_tail(rest + (OWN * kg + t) * KP_STEP, half, k_end, vr[0]);
            sp.split(vr[0], pr[0]);
            get_l(0, OWN * kg + t, fl[0]);
            multiply(fl[0], pr[0]);
        }
        report();
        __syncthreads();
        f32 = reported();
    }
    if (f32) {
        // the rest in f32, from the chain on that met the value
        clear(acc);
        clear(small);
        for (int k0 = kept; k0 < k_end; k0 += KP_K) {
            __syncthreads();  // (the stage before, or a wave still in the loop above, is read to its end)
            sl.load_tail(k0, loct, k_end, vl[0]);
            // [octet][first or second 4 steps][row]
#pragma unroll
            for (int i = 0; i < 2; ++i)
                *(kp_v4f*)(lds + (2 * loct + i) * KP_PIECE + lrow * 16) = kp_v4f{vl[0][4 * i], vl[0][4 * i + 1], vl[0][4 * i + 2], vl[0][4 * i + 3]};
            __syncthreads();
#pragma unroll 1
            for (int t = 0; t < OWN; ++t) {
                sr.load_tail(k0 + (OWN * kg + t) * KP_STEP, half, k_end, vr[0]);
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const char* const at = lds + (2 * (2 * (OWN * kg + t) + half) + c) * KP_PIECE + (lane & 31) * 16;
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const kp_v4f l = *(const kp_v4f*)(at + i * 512);
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            acc[i] = SWAP ? __builtin_amdgcn_mfma_f32_32x32x2f32(vr[0][4 * c + e], l[e], acc[i], 0, 0, 0)
                                          : __builtin_amdgcn_mfma_f32_32x32x2f32(l[e], vr[0][4 * c + e], acc[i], 0, 0, 0);
                    }
                }
            }
            if ((((k0 - k_begin) / KP_K) & 7) == 7)
                close();
        }
    }
    close();
    // the waves that share rows of R meet in LDS: wave kg finishes registers kg 32 / KG ... of the 32
    constexpr int MINE = 32 / KG;
    float* const meet = (float*)lds;
    if (KG > 1) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                meet[(wave * 32 + i * 16 + e) * 64 + lane] = sum[i][e];
        __syncthreads();
    }
    float* const out = q.sliced ? q.C + (size_t)z * q.M * q.N : q.C;
    // register e of a 32 x 32 tile: row 8 (e / 4) + 4 half + e % 4, column lane % 32
#pragma unroll
    for (int x = 0; x < MINE; ++x) {
        const int reg = KG > 1 ? kg * MINE + x : x, i = reg >> 4, e = reg & 15;
        float v = 0.f;
        if (KG == 1) {
            v = sum[x >> 4][x & 15];
        } else {
#pragma unroll
            for (int g = 0; g < KG; ++g)
                v += meet[((g * WN + wn) * 32 + reg) * 64 + lane];
        }
        const int row = 8 * (e >> 2) + 4 * half + (e & 3);
        const int m = SWAP ? r0 + row : l0 + i * 32 + row, n = SWAP ? l0 + i * 32 + (lane & 31) : r0 + (lane & 31);
        if (m < q.M && n < q.N) {
            if (q.sliced) {
                out[(size_t)m * q.N + n] = v;
            } else {
                out[(size_t)m * q.ldc + n] = v;
            }
        }
    }
}

// ---- choice ---------------------------------------------------------------------------------------------
// Estimated cycles of the busiest CU, on the scale of gemm_f32_ks.hip (2.33 GHz): 16 steps of K of the 8 waves of a workgroup, one a
// CU, 2250 (2100 with two groups of waves, 1720 where every wave has its own rows of R: L is split less often), 4500 for the
// first operands and the end of each and 4000 for a rest of K; for slices of K a second launch and their way out and back in at 5
// TB/s. Estimated / measured us: 512 x 4096 x 4096 111 / 109, 1912 x 1206 x 1078 43 / 41, 1381 x 2795 x 925 nt 69 / 71, 947 x 2247 x 657 nt 37 /
// 38, 83 x 2794 x 3689 nt 30 / 28.5, 3713 x 2717 x 528 114 / 110, 2240 x 474 x 1804 tt 60 / 56 (there 46); 64 x 4096 x 4096, which stays with
// gemm_f32_ks.hip, 24.5 / 24.5 for 24 - 25.6.
static double kp_cost(long M, long N, long K, int kg, int slices, bool swap) {
    const long wide = 256 / kg, l = swap ? N : M, r = swap ? M : N;
    const long chunk = ((K + slices - 1) / slices + KP_K - 1) / KP_K, body = kg == 4 ? 4 : 2;
    const long turns = (chunk + body - 1) / body * body * (4 / kg);
    const long wgs = ((l + KP_L - 1) / KP_L) * ((r + wide - 1) / wide) * slices;
    const double each = (double)turns * (kg == 1 ? 1720.0 : kg == 2 ? 2100.0 : 2250.0) + 4500.0 + (slices == 1 && K % KP_K ? 4000.0 : 0.0);
    const double add = slices == 1 ? 0.0 : 4000.0 + 4.0 * (double)(2 * slices + 1) * (double)M * (double)N / 2146.0;
    return (double)((wgs + num_cus() - 1) / num_cus()) * each + 8000.0 + add;
}

// Below some 20 us nothing is won (197 x 771 x 1003 nt 7.9 us there, 12.7 here), and working the plan out costs the host 1 us.
static bool kp_plan(const GevmArgs& v, size_t room, KpPlan* plan) {
    const long M = v.M, N = v.N, K = v.K;
    double best = 0.97 * gemm_f32_ks_cycles(v);
    if (best < 45000.0)
        return false;
    plan->kg = 0;
    const long most = (long)(room / ((size_t)M * N * 4));
    for (int kg = 1; kg <= 4; kg *= 2)
        for (int swap = 0; swap < (kg == 4 ? 1 : 2); ++swap)
            for (int s = 1; s == 1 || (s <= 16 && s <= most && s * 128L <= K); ++s) {
                const double cost = kp_cost(M, N, K, kg, s, swap != 0);
                if (cost < best) {
                    best = cost;
                    *plan = {kg, s, swap != 0};
                }
            }
    return plan->kg != 0;
}

static long side_bytes(long rows, long row, long steps, long k) {
    return 4 * ((rows - 1) * row + (steps - 1) * k + 1);
}

template <int LM, int RM, bool SWAP>
static TinyNNStatus kp_launch(KpParams& q, const KpPlan& p, const Workspace* ws) {
    const int wide = 256 / p.kg;
    const int gl = (q.l.rows + KP_L - 1) / KP_L, gr = (q.r.rows + wide - 1) / wide;
    q.tiles = gl * gr;
    q.chunk = ((q.K + p.slices - 1) / p.slices + KP_K - 1) / KP_K * KP_K;
    const int slices = (q.K + q.chunk - 1) / q.chunk;
    q.total = q.tiles * slices;
    q.per_xcd = (q.total + 7) / 8;
    // (tiles along the shorter side first: a run of an XCD is then about square)
    q.l_first = (long)gl * KP_L <= (long)gr * wide;
    q.d_tiles = make_fastdiv((uint32_t)q.tiles);
    q.d_run = make_fastdiv((uint32_t)(q.l_first ? gl : gr));
    q.sliced = slices > 1;
    float* const C = q.C;
    if (q.sliced)
        q.C = (float*)ws->ptr;
    note_kernel("gemm_f32_ks_split", KP_L, wide, slices, SWAP);
    void (*kern)(KpParams) = p.kg == 1 ? gemm_f32_ks_split_kernel<LM, RM, 1, SWAP> : p.kg == 2 ? gemm_f32_ks_split_kernel<LM, RM, 2, SWAP> : gemm_f32_ks_split_kernel<LM, RM, 4, false>;
    hipLaunchKernelGGL(kern, dim3(8 * q.per_xcd), dim3(512), 0, stream(), q);
    if (q.sliced)
        gemm_f32_add_slices(q.C, slices, q.M, q.N, C, q.ldc);
    return check_launch("gemm_f32_ks_split");
}

TinyNNStatus gemm_f32_ks_split_launch(const GevmArgs& v, int ta, int tb, const KpPlan& p, const Workspace* ws) {
    KpParams q = {};
    const KpSide a = {v.A, (unsigned)side_bytes(v.M, v.a_rs, v.K, v.a_cs), (unsigned)v.a_rs * 4u, (unsigned)v.a_cs * 4u, v.M};
    const KpSide b = {v.B, (unsigned)side_bytes(v.N, v.b_cs, v.K, v.b_rs), (unsigned)v.b_cs * 4u, (unsigned)v.b_rs * 4u, v.N};
    q.C = v.C;
    q.M = v.M;
    q.N = v.N;
    q.K = v.K;
    q.ldc = (int)v.ldc;
    q.l = p.swap ? b : a;
    q.r = p.swap ? a : b;
    const bool lk = p.swap ? tb : !ta, rk = p.swap ? !ta : tb;  // contiguous along K
#define MG_KP(L_, R_) (p.swap ? kp_launch<L_, R_, true>(q, p, ws) : kp_launch<L_, R_, false>(q, p, ws))
    return lk ? (rk ? MG_KP(KP_CONTIG, KP_CONTIG) : MG_KP(KP_CONTIG, KP_STRIDED)) : (rk ? MG_KP(KP_STRIDED, KP_CONTIG) : MG_KP(KP_STRIDED, KP_STRIDED));
#undef MG_KP
}

bool gemm_f32_ks_split(const GevmArgs& v, int ta, int tb, const Workspace* ws, TinyNNStatus* status) {
    const long limit = (1L << 31) - 65536;
    KpPlan p;
    if ((double)v.M * v.N * v.K < 4e8 || v.K < KP_K || side_bytes(v.M, v.a_rs, v.K, v.a_cs) >= limit || side_bytes(v.N, v.b_cs, v.K, v.b_rs) >= limit ||
        !(v.a_cs == 1 || v.a_rs == 1) || !(v.b_cs == 1 || v.b_rs == 1) || (long)v.M * v.N >= (1L << 31) ||
        !kp_plan(v, ws && ws->ptr && ((uintptr_t)ws->ptr & 3) == 0 ? ws->size : 0, &p))
        return false;
    *status = gemm_f32_ks_split_launch(v, ta, tb, p, ws);
    return true;
}

}  // namespace mg
