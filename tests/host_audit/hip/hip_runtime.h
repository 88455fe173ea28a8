// Stand-in for <hip/hip_runtime.h> used by tests/host_audit/audit.cpp ONLY: it lets the library's
// own kernel sources (megcc_amd/csrc/*.hip, included as they are) be compiled as plain host C++
// and run one GPU thread after the other, so that every address a kernel computes is dereferenced
// on the host, on buffers fenced by inaccessible pages. Values do not matter here - threads do not
// see each other's LDS writes, matrix-core and cross-lane builtins return an operand - only the
// index arithmetic is exercised, and that arithmetic never depends on loaded values in the
// audited kernels.
#pragma once
#include <math.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>

#define MG_HOST_AUDIT 1
#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __shared__
#define __launch_bounds__(...)

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
struct uint3_ {
    unsigned x, y, z;
};
inline thread_local uint3_ threadIdx, blockIdx;
inline thread_local dim3 blockDim, gridDim;

struct float4 {
    float x, y, z, w;
} __attribute__((aligned(16)));
inline float4 make_float4(float x, float y, float z, float w) { return float4{x, y, z, w}; }
struct float2 {
    float x, y;
} __attribute__((aligned(8)));
inline float2 make_float2(float x, float y) { return float2{x, y}; }
struct int4 {
    int x, y, z, w;
} __attribute__((aligned(16)));
struct int2 {
    int x, y;
} __attribute__((aligned(8)));
struct uint4 {
    unsigned x, y, z, w;
} __attribute__((aligned(16)));
struct uint2 {
    unsigned x, y;
} __attribute__((aligned(8)));

using std::max;
using std::min;
inline int min(int a, unsigned b) { return a < (int)b ? a : (int)b; }
inline long min(long a, int b) { return a < b ? a : (long)b; }
inline long max(long a, int b) { return a > b ? a : (long)b; }

typedef int hipError_t;
typedef void* hipStream_t;
enum { hipSuccess = 0, hipFuncAttributeMaxDynamicSharedMemorySize = 8 };
inline const char* hipGetErrorString(hipError_t) { return "host audit"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipFuncSetAttribute(const void*, int, int) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }

inline hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { return *n = 1, hipSuccess; }

// Buffer loads and stores: dwords whose whole offset, the lane's and the scalar one, lies beyond the buffer read zero
// or are dropped (each dword for itself, as the hardware does it), everything else is dereferenced.
struct audit_rsrc {
    char* p;
    unsigned bytes;
};
typedef unsigned audit_v4u __attribute__((ext_vector_type(4)));
// Most kernels lean on that here and there. Where `audit_strict` is set only offsets with the top bit, which is how a kernel says
// that it means none, and buffers of no bytes may lie beyond: anything else ends the run as an access out of bounds.
extern bool audit_strict;
void audit_beyond(const char* what, unsigned off, unsigned soff, unsigned bytes);
inline bool audit_inside(audit_rsrc r, unsigned off, unsigned soff, const char* what) {
    if ((unsigned long long)off + soff < r.bytes)
        return true;
    if (audit_strict && r.bytes && !(off >> 31))
        audit_beyond(what, off, soff, r.bytes);
    return false;
}
inline unsigned audit_load(audit_rsrc r, unsigned off, unsigned soff) {
    return audit_inside(r, off, soff, "load") ? *(volatile unsigned*)(r.p + off + soff) : 0;
}
inline audit_v4u audit_load4(audit_rsrc r, unsigned off, unsigned soff) {
    return audit_v4u{audit_load(r, off, soff), audit_load(r, off + 4, soff), audit_load(r, off + 8, soff), audit_load(r, off + 12, soff)};
}
inline void audit_store(unsigned v, audit_rsrc r, unsigned off, unsigned soff) {
    if (audit_inside(r, off, soff, "store"))
        *(volatile unsigned*)(r.p + off + soff) = v;
}
#define __amdgpu_buffer_rsrc_t audit_rsrc
#define __builtin_amdgcn_make_buffer_rsrc(ptr, stride, bytes, flags) (audit_rsrc{(char*)(ptr), (unsigned)(bytes)})
#define __builtin_amdgcn_raw_buffer_load_b32(r, off, soff, aux) audit_load(r, (unsigned)(off), (unsigned)(soff))
#define __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, aux) audit_load4(r, (unsigned)(off), (unsigned)(soff))
#define __builtin_amdgcn_raw_buffer_store_b32(v, r, off, soff, aux) audit_store(v, r, (unsigned)(off), (unsigned)(soff))

inline float __uint_as_float(unsigned u) {
    float f;
    memcpy(&f, &u, 4);
    return f;
}

inline unsigned __float_as_uint(float f) {
    unsigned u;
    memcpy(&u, &f, 4);
    return u;
}

inline void __syncthreads() {}
template <typename T>
inline T __shfl_down(T v, int, int = 64) { return v; }
template <typename T>
inline T __shfl_xor(T v, int, int = 64) { return v; }
template <typename T>
inline T __shfl(T v, int, int = 64) { return v; }
inline unsigned __umulhi(unsigned a, unsigned b) { return (unsigned)(((unsigned long long)a * b) >> 32); }

#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_sched_barrier(x) ((void)0)
template <typename A, typename B, typename C>
inline C audit_sums(const A&, const B&, const C& c, int, int, int) { return c; }
#define __builtin_amdgcn_mfma_f32_32x32x2f32(...) audit_sums(__VA_ARGS__)
#define __builtin_amdgcn_mfma_f32_16x16x4f32(...) audit_sums(__VA_ARGS__)
#define __builtin_amdgcn_mfma_f32_32x32x16_bf16(...) audit_sums(__VA_ARGS__)
#define __builtin_amdgcn_mfma_i32_32x32x32_i8(...) audit_sums(__VA_ARGS__)
#define __builtin_amdgcn_mfma_i32_16x16x64_i8(...) audit_sums(__VA_ARGS__)
#define __builtin_amdgcn_mfma_i32_16x16x32_i8(...) audit_sums(__VA_ARGS__)
#define __builtin_amdgcn_fdot2_f32_bf16(a, b, c, clamp) (c)
struct audit_pair {
    unsigned v[2];
    unsigned operator[](int i) const { return v[i]; }
};
#define __builtin_amdgcn_permlane32_swap(a, b, x, y) (audit_pair{{(unsigned)(a), (unsigned)(b)}})
#define __builtin_amdgcn_sdot4(a, b, c, clamp) (c)
#define __builtin_amdgcn_fmed3f(x, lo, hi) (lo)
#define __builtin_amdgcn_cvt_pk_u8_f32(x, i, r) (r)
#define __builtin_amdgcn_perm(a, b, sel) ((a) ^ (b) ^ (sel))
#define __builtin_amdgcn_alignbyte(hi, lo, n) ((hi) ^ (lo) ^ (n))
#define __builtin_amdgcn_s_barrier() ((void)0)
#define __builtin_amdgcn_s_waitcnt(x) ((void)0)
#define __builtin_amdgcn_fence(...) ((void)0)
#define __builtin_amdgcn_kernarg_segment_ptr() ((const char*)0)

// every block, every thread, one after the other
void audit_dynamic_lds(size_t bytes);
template <typename K, typename... Args>
inline void host_audit_launch(K kernel, dim3 grid, dim3 block, size_t lds_bytes, Args... args) {
    audit_dynamic_lds(lds_bytes);
    gridDim = grid;
    blockDim = block;
    for (unsigned bz = 0; bz < grid.z; ++bz)
        for (unsigned by = 0; by < grid.y; ++by)
            for (unsigned bx = 0; bx < grid.x; ++bx) {
                blockIdx = uint3_{bx, by, bz};
                for (unsigned tz = 0; tz < block.z; ++tz)
                    for (unsigned ty = 0; ty < block.y; ++ty)
                        for (unsigned tx = 0; tx < block.x; ++tx) {
                            threadIdx = uint3_{tx, ty, tz};
                            kernel(args...);
                        }
            }
}
#define hipLaunchKernelGGL(kernel, grid, block, lds_bytes, strm, ...) \
    host_audit_launch(kernel, dim3(grid), dim3(block), (size_t)(lds_bytes), __VA_ARGS__)
