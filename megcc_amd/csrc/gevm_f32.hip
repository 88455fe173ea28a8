// f32 MatMul with at most 4 rows (C[M,N] = A[M,K] * B, M <= 4): the reference's gevm / gemv case
// (GeneralIntrinsic/MatMulKernel/Fp32Gevm.cpp:50-119 for M <= 4, BareMetal/MatrixMul.cpp:43-120).
// The layer is ONE pass over B, a few MB: what counts is that every byte of B is requested at
// once - the whole matrix is smaller than the bandwidth-latency product of the chip - and that it
// is one launch. No matrix cores (2 flops per 4 bytes of B).
//   * B row-major [K,N] (not transposed): a workgroup owns 16 columns, a lane 4 of them (one
//     16-byte load per row) and every (16 W)-th row, W the waves of the workgroup: 4 to 16, so that all of a
//     K up to 2048 is asked for at once. The partial sums of a column meet by shifts within 16 lanes and then in
//     LDS, in a fixed order. Neighbouring workgroups, which share lines of 128 bytes, run on one XCD.
//   * B transposed [N,K]: a wave owns 1 or 2 rows of B (= outputs), a lane 16-byte pieces of them
//     along K, 8 in flight; the lanes' partial sums meet by swaps of half waves and rows and by shifts, in a fixed order.
// A 16-byte load needs 4-byte alignment only. The last columns (the end of K) come from a load that begins up to three
// places earlier; what another lane counts as well is dropped.
// Measured (us, before - four waves a workgroup, 16-byte loads only where every row was aligned, a wave four rows - / now):
// 1 x 1024 x 1000 3.75 / 3.6, 1 x 2346 x 311 12.6 / 4.2, 1 x 4000 x 1000 10.7 / 5.9, 1 x 4000 x 3530 27 / 11.5 (4.9 TB/s),
// 4 x 544 x 311 6.2 / 4.0; B transposed 1 x 1024 x 1000 4.3 / 3.2, 1 x 2346 x 311 12.9 / 3.5, 1 x 4000 x 1000 8.6 / 3.8,
// 3 x 544 x 1000 8.3 / 3.2, 4 x 4000 x 311 21.4 / 7.4.
// The order of the additions differs from the reference's ascending k; f32 results are held to the
// 1e-4 tolerance like the tiled GEMM, not to bit equality.
#include "common.h"
#include "gevm_f32.h"

namespace mg {
namespace {

constexpr int GV_UNROLL = 8;  // 16-byte loads requested before the first one is used

typedef float gv_v4f __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ void gv_load(const float* p, float (&v)[4]) {
    const gv_v4f t = *(const gv_v4f*)p;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        v[j] = t[j];
}

// lane i of every 16 gets what lane i + BY of them holds (0 beyond them)
template <int BY>
__device__ __forceinline__ float gv_shift(float v) {
#ifdef MG_HOST_AUDIT
    return v;
#else
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x100 | BY, 0xf, 0xf, true));
#endif
}

// lanes 0 - 31 (of 32: 0 - 15) get their own and what the other 32 (16) hold
template <int BY>
__device__ __forceinline__ float gv_fold(float v) {
#ifdef MG_HOST_AUDIT
    return v;
#else
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const auto p = BY == 32 ? __builtin_amdgcn_permlane32_swap(u, u, false, false) : __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
#endif
}

// B[k, n] at B + k * b_rs + n (rows contiguous), N >= 4; waves: up to 16
template <int M>
__global__ void __launch_bounds__(1024) gevm_f32_cols_kernel(GevmArgs q, int waves, int per_xcd) {
    __shared__ float red[64][M][16];
    const int tid = threadIdx.x, cg = tid & 3, kg = tid >> 2, rows = 16 * waves;
    const int block = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    const int n0 = block * 16 + cg * 4;
    if (block * 16 >= q.N)  // (the whole workgroup)
        return;
    const int first = min(n0, q.N - 4);
    float acc[M][4];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            acc[m][j] = 0.f;
    for (int k0 = kg; k0 < q.K; k0 += rows * GV_UNROLL) {
        // No load stands under a condition (the compiler would wait for every outstanding
        // load at each join, one round trip per row): rows beyond K read row K - 1, and their products are replaced by 0.
        float b[GV_UNROLL][4], a[GV_UNROLL][M];
#pragma unroll
        for (int u = 0; u < GV_UNROLL; ++u) {
            const int k = min(k0 + u * rows, q.K - 1);
            gv_load(q.B + (size_t)k * q.b_rs + first, b[u]);
#pragma unroll
            for (int m = 0; m < M; ++m)
                a[u][m] = q.A[(size_t)m * q.a_rs + (size_t)k * q.a_cs];
        }
#pragma unroll
        for (int u = 0; u < GV_UNROLL; ++u) {
            const bool ok = k0 + u * rows < q.K;
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[m][j] += ok ? a[u][m] * b[u][j] : 0.f;
        }
    }
    // the four of 16 lanes that hold a column, then (m, column) adds those of the workgroup in ascending order
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float s = acc[m][j];
            s += gv_shift<8>(s);
            s += gv_shift<4>(s);
            if ((tid & 15) < 4 && first + j >= n0)  // (the columns in front of n0 are another lane's, or another workgroup's)
                red[tid >> 4][m][first + j - block * 16] = s;
        }
    __syncthreads();
    if (tid < M * 16) {
        const int m = tid >> 4, c = tid & 15, n = block * 16 + c;
        if (n < q.N) {
            float s = 0.f;
            for (int w = 0; w < 4 * waves; w += 4) {  // (four in flight)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    s += red[w + i][m][c];
            }
            q.C[(size_t)m * q.ldc + n] = s;
        }
    }
}

// B[k, n] at B + n * b_cs + k (B stored transposed, rows of K contiguous), A's rows contiguous too, K >= 4
template <int M, int R>
__global__ void __launch_bounds__(256) gevm_f32_rows_kernel(GevmArgs q) {
    constexpr int U = GV_UNROLL / R;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = (blockIdx.x * 4 + wave) * R;  // this wave's outputs
    if (n0 >= q.N)
        return;
    float acc[M][R];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int r = 0; r < R; ++r)
            acc[m][r] = 0.f;
    for (int k0 = lane * 4; k0 < q.K; k0 += 256 * U) {
        // (no load under a condition, as above: rows beyond N read row N - 1, pieces beyond K the last one)
        float b[U][R][4], a[U][M][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(k0 + u * 256, q.K - 4);
#pragma unroll
            for (int r = 0; r < R; ++r)
                gv_load(q.B + (size_t)min(n0 + r, q.N - 1) * q.b_cs + k, b[u][r]);
#pragma unroll
            for (int m = 0; m < M; ++m)
                gv_load(q.A + (size_t)m * q.a_rs + k, a[u][m]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int own = k0 + u * 256 - min(k0 + u * 256, q.K - 4);  // (elements in front of it are another lane's)
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[m][r] += j >= own ? a[u][m][j] * b[u][r][j] : 0.f;
        }
    }
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float s = acc[m][r];
            // (halves first: behind the shifts the few values of a K just over 64 are one more rounding of the whole sum, K = 66 0.76e-7 for 0.73e-7)
            s = gv_fold<32>(s);
            s = gv_fold<16>(s);
            s += gv_shift<8>(s);
            s += gv_shift<4>(s);
            s += gv_shift<2>(s);
            s += gv_shift<1>(s);
            if (lane == 0 && n0 + r < q.N)
                q.C[(size_t)m * q.ldc + n0 + r] = s;
        }
}

template <int M>
void launch_cols(const GevmArgs& q) {
    const int blocks = (q.N + 15) / 16, per_xcd = (blocks + 7) / 8;
    // waves: K dealt evenly to the fewest rounds of 16 of them
    const int per_wave = 16 * GV_UNROLL, rounds = (int)((q.K + 16L * per_wave - 1) / (16 * per_wave));
    int waves = (int)((q.K + (long)rounds * per_wave - 1) / ((long)rounds * per_wave));
    waves = waves < 4 ? 4 : waves;
    hipLaunchKernelGGL((gevm_f32_cols_kernel<M>), dim3(8 * per_xcd), dim3(64 * waves), 0, stream(), q, waves, per_xcd);
}

template <int M>
void launch_rows(const GevmArgs& q) {
    if (M == 1 && q.N <= 2048)
        hipLaunchKernelGGL((gevm_f32_rows_kernel<M, 1>), dim3((q.N + 3) / 4), dim3(256), 0, stream(), q);
    else
        hipLaunchKernelGGL((gevm_f32_rows_kernel<M, 2>), dim3((q.N + 7) / 8), dim3(256), 0, stream(), q);
}

}  // namespace

static bool by_columns(const GevmArgs& q) {
    return q.b_cs == 1 && q.N >= 4;
}

bool gevm_f32_supported(const GevmArgs& q) {
    return q.M >= 1 && q.M <= 4 && q.N >= 1 && q.K >= 1 && (by_columns(q) || (q.b_rs == 1 && q.K >= 4 && q.a_cs == 1));
}

// Against the matrix cores (gemm_f32_ks.hip), whose tiles have 16 rows whatever M is. They win where this kernel's loads of A,
// M to one of B, are what a CU is busy with: four rows of a long K (us, here / there: 4 x 1000 x 1000 4.6 / 4.7, 4 x
// 1300 x 1000 5.4 / 5.0, which stays, 4 x 1537 x 1000 6.0 / 5.5, 4 x 2346 x 311 7.2 / 6.5, 4 x 4096 x 1300 11.2 / 10.3), three of many columns
// as well (3 x 4096 x 1300 11.3 / 10.0; 3 x 2048 x 1300 5.6 / 5.5, 3 x 4096 x 1024 7.7 / 8.2), and both above 2048 columns from K = 513 on (4 x 513 x 3530 4.3 / 3.8,
// 4 x 800 x 2049 4.3 / 3.9, 4 x 1000 x 3530 5.0 / 5.2, 4 x 1500 x 3000 5.5 / 5.2; 3 x 513 x 3530 3.9 / 3.8, 3 x 800 x 3530 4.6 / 4.2, 3 x 1000 x 3530 4.9 / 5.0, 3 x 1024 x 4096 4.3 / 4.0). Below 64 of their tiles two XCDs fetch each line of B (xcd_strip): a long K of four rows and 37 tiles
// or more stays here (4 x 3000 x 650 7.5 / 9.3, 4 x 4000 x 1000 9.3 / 10.7; 4 x 4000 x 400 8.7 / 8.1, 4 x 4000 x 1010 9.3 / 8.5, 4 x 2600 x 580
// 7.3 / 6.5). Two rows stay: mostly faster, 7 % slower at worst but for 4096 x 4096 (2 x 4000 x 1400 9.6 / 9.0, 2 x 4096 x 4096 16.0 / 13.9). B transposed
// stays but for four rows of many columns and a short K (4 x 300 x 3000 4.3 / 3.4, 4 x 544 x 3530 4.3 / 3.9, 4 x 560 x 8192 5.7 / 4.4; 4 x 600 x 3530 4.3 / 4.4,
// 4 x 1000 x 3530 4.3 / 5.3, 4 x 4000 x 311 7.4 / 11.9, 4 x 4096 x 4096 13.9 / 13.4), though a K just beyond the first round of
// four rows' loads would be better off there (4 x 1200 x 1000 4.9 / 4.7).
bool gevm_f32_wins(const GevmArgs& q) {
    if (!by_columns(q))
        return !(q.M == 4 && q.N > 2048 && q.K <= 560);
    if (q.M <= 2 || q.K <= 512)
        return true;
    if (q.N > 2048)
        return false;
    if (q.M == 4)
        return q.K <= 1536 || (q.K >= 2800 && q.N > 36 * 16 && q.N <= 63 * 16);
    return q.N <= 1280 || q.K <= 2560;
}

TinyNNStatus gevm_f32_launch(const GevmArgs& q) {
    const bool cols = by_columns(q);
#define MG_GEVM(M_) (cols ? launch_cols<M_>(q) : launch_rows<M_>(q))
    switch (q.M) {
        case 1: MG_GEVM(1); break;
        case 2: MG_GEVM(2); break;
        case 3: MG_GEVM(3); break;
        default: MG_GEVM(4); break;
    }
#undef MG_GEVM
    return check_launch("gevm_f32");
}

}  // namespace mg
