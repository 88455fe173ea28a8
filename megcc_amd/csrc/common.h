// Shared host-side helpers of libmegcc_gfx950.so: error reporting, the library stream, Tensor
// inspection. Host code, plus the tile-order helper the tiled kernels share; the other device helpers live in epilogue.h.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "megcc_gfx950.h"

namespace mg {

// One stream for every launch and copy, default priority, created on first use.
hipStream_t stream();
// The library stream itself, whatever stream() currently answers.
hipStream_t main_stream();
// While `on`, stream() answers `s` on this thread: the model runtime launches the last operators of a
// forward on a second stream this way (model.cpp). The kernels' launch code is unchanged.
void set_stream_override(hipStream_t s, bool on);
// Streams megcc_gfx950_wait() synchronises besides the library stream.
void register_aux_stream(hipStream_t s);
void unregister_aux_stream(hipStream_t s);

// How often the host has waited for the library stream, and for that and all of the streams above.
struct HostWaits {
    unsigned long library, all;
};
HostWaits host_waits();

// Compute units of the current device (256 when the query fails).
int num_cus();

// Records a message for megcc_gfx950_last_error() and returns `st`.
TinyNNStatus fail(TinyNNStatus st, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

#define MG_REQUIRE(cond, st, ...)          \
    do {                                   \
        if (!(cond))                       \
            return ::mg::fail(st, __VA_ARGS__); \
    } while (0)

// Tile order of a 2-D grid of gx x gy workgroups for the chip's eight XCDs. Workgroups are handed to
// the XCDs in turn (workgroup i runs on XCD i % 8) and every XCD has an L2 of its own, so with the
// plain order each XCD touches every row panel of one operand. Here XCD x takes the x-th eighth (the first
// ones of a tile more where the number is no multiple of 8) of an order that walks the grid in strips of `w`
// columns, row by row inside a strip: the tiles one XCD owns are then a compact rectangle and each
// operand panel is fetched by the one or two XCDs that need it. w = 0 keeps the plain order. Any w >= 1
// gives a bijection. Where the number is no multiple of 8, only for operands (`bytes`) of more than half an L2
// (without / with, us: FullyConnected 246 x 3742 x 2207 16.2 / 14.8, 591 x 1822 x 2221 15.3 / 13.9, 873 x 4053 x 3853
// 48.0 / 44.4, 2355 x 717 x 2650 18.9 / 18.3; below, 898 x 1104 x 690 7.5 / 7.7, 3844 x 171 x 2463 19.3 / 20.4).
struct XcdOrder {
    int w;
};
// the strip for `tiles` tiles in rows of gx; 0: too few
inline int xcd_strip(int gx, long tiles) {
    if (tiles < 64)
        return 0;
    // w ~ sqrt(tiles per XCD / 2): the half of its share an XCD has resident at a time is about square
    // (a round of workgroups streams its panels through the 4 MB L2 once; the next round starts over)
    int w = 1;
    while ((long)w * w * 8 <= tiles / 8)
        w *= 2;
    return w < gx ? w : gx;
}
inline XcdOrder make_xcd_order(int gx, int gy, long bytes) {
    return {((long)gx * gy & 7) != 0 && bytes <= (2L << 20) ? 0 : xcd_strip(gx, (long)gx * gy)};
}
__device__ __forceinline__ void xcd_tile(XcdOrder o, int bx, int by, int gx, int gy, int& tx, int& ty) {
    tx = bx;
    ty = by;
    if (o.w == 0)
        return;
    const int nb = gx * gy, lb = by * gx + bx;
    const int place = (lb & 7) * (nb >> 3) + min(lb & 7, nb & 7) + (lb >> 3);
    const int strip = place / (o.w * gy), rem = place - strip * (o.w * gy);
    const int w = min(o.w, gx - strip * o.w);
    ty = rem / w;
    tx = strip * o.w + rem - ty * w;
}

// Kernel-selection overrides: each one takes a kernel (or a variant of one) out of the dispatch so
// that the regression tests can reach the kernels that serve the shapes behind it. Read from the
// environment (MEGCC_NOPWS=1, ...) ONCE, when the library first consults them; later changes go
// through megcc_gfx950_set_option(). Nothing on a launch path scans the environment.
struct Options {
    bool no_pws, no_gevm, no_fcb, no_small, no_pm768, no_pm, no_dma512, no_pm256, no_dma, no_fcs, no_pwshare, no_hybrid, no_dot4, no_f32small, dw_generic, no_dwmfma, no_dwnchw, no_fuse_softmax, no_graph, no_poolrows, no_firstmfma, no_rowsplit, no_fuse_chain, no_fuse_pwdw, fuse_pwdw, no_fcone, no_xcdorder, no_affine, no_pipeline, no_fuse_dwpw, fuse_dwpw, no_fuse_stem, fuse_stem, no_f32split, no_f32ks, no_fuse_blocks, fuse_blocks;
};
Options& options();

// Which kernel variant the most recent dispatch on this thread selected: `name` (a string literal)
// and up to five numbers that identify the instantiation; megcc_gfx950_last_kernel() formats them.
void note_kernel(const char* name, int a = -1, int b = -1, int c = -1, int d = -1, int e = -1);

// A kernel that requantises by the proven fused multiply-add (epilogue.h) says so after its
// note_kernel(): megcc_gfx950_last_kernel() then ends in "+affine".
void note_requant_affine(bool on);

// conv_api.hip: looks up the address of the static scratch array of
// megcc_gfx950_conv2d_noalloc on the current device (once per device; later calls return at once).
TinyNNStatus noalloc_scratch_setup();

// conv_api.hip: a channel-wise 3x3 convolution and the pointwise convolution of its result as one kernel
// (model runtime only). CHECK: whether the kernel takes the pair; PREPARE, once: everything a launch on these operands needs is
// in the pair's block, which belongs to the caller and keeps the kernel's arguments on the device; RUN: the launch, nothing else.
struct DwPwBlock;
DwPwBlock* dw_pw_block_create();
void dw_pw_block_destroy(DwPwBlock* block);
enum class DwPw { CHECK, PREPARE, RUN };
TinyNNStatus dw_pw_run(
        const MegccPwDwAttr* attr, Tensor** inputs, int nr_input, Tensor** outputs, int nr_output, DwPwBlock* block, DwPw what);
// conv_blocks.hip: consecutive prepared pairs as one kernel, where it takes them (else NULL). What a launch needs is kept with it.
struct BlocksRun;
bool conv_blocks_takes(const Tensor& x);  // of these channels, rows and columns
BlocksRun* conv_blocks_create(const DwPwBlock* const* blocks, int count);
void conv_blocks_destroy(BlocksRun* run);
TinyNNStatus conv_blocks_launch(const BlocksRun* run);
// whether it could take the pair, before memory is planned and the pointwise filter packed
bool dw_pw_takes(
        const MegccConvAttr* dw_attr, const MegccConvAttr* pw_attr, const Tensor* src, const Tensor* dw_flt, const Tensor* mid,
        const Tensor* pw_flt, const Tensor* dst);

// conv_api.hip: the image's conversion to qsi8, the first convolution of the quantised image, the channel-wise 3x3 and the pointwise
// convolution behind it as one kernel (model runtime only). inputs: f32 image, then each layer's filter [, bias], the
// pointwise one packed; the scales of the three tensors in between. `launch` false: only whether the kernel takes them.
struct StemAttr {
    MegccConvAttr first, dw, pw;
    float s_image, s_first, s_mid;
};
TinyNNStatus stem_run(const StemAttr& attr, Tensor** inputs, int nr_input, Tensor** outputs, int nr_output, bool launch);

// After a kernel launch: surfaces launch-configuration errors as TinyNN_ERROR_RUNTIME.
TinyNNStatus check_launch(const char* what);

// device.cpp: small reads of device memory by a blocking caller, through pinned memory of their own. A copy to pageable memory and the
// wait for it took 28 us behind a forward of 100; here a kernel writes the bytes and then a number to pinned memory, and the host
// looks for the number: less than the wait for the stream alone (us behind 280 of work: 4 KB 316 / 285, 64 KB 348 / 290,
// the wait with no copy 288). Reads of more than HOST_STAGE_BYTES, and one while another thread's is under way, go by the copy.
static constexpr size_t HOST_STAGE_BYTES = 64 << 10;
struct HostStage;
HostStage* host_stage_create();  // NULL: no pinned memory
void host_stage_destroy(HostStage* stage);
TinyNNStatus host_stage_read(HostStage* stage, void* host, const void* src, size_t bytes);
// relayout.hip: `bytes` bytes to pinned memory, then `number` behind them all
TinyNNStatus copy_to_host_launch(const void* src, void* pinned, size_t bytes, unsigned* where, unsigned number);

// relayout.hip: copies `src` (layout sl) to `dst` (layout dl), elements of `es` bytes; one launch.
TinyNNStatus strided_copy(
        const void* src, const Layout& sl, void* dst, const Layout& dl, size_t es, const char* who);

inline size_t nr_elem(const Layout& l) {
    size_t n = 1;
    for (int i = 0; i < l.nr_dim; ++i)
        n *= l.dims[i];
    return n;
}

// Dense row-major strides (dims of extent 1 may carry any stride).
inline bool is_contiguous(const Layout& l) {
    long expect = 1;
    for (int i = l.nr_dim - 1; i >= 0; --i) {
        if (l.dims[i] != 1 && l.stride[i] != expect)
            return false;
        expect *= l.dims[i];
    }
    return true;
}

// Lowest and highest element offset a layout touches, relative to its first element; false when
// it has no elements.
inline bool view_span(const Layout& l, long long* lo, long long* hi) {
    *lo = *hi = 0;
    for (int i = 0; i < l.nr_dim; ++i) {
        if (l.dims[i] == 0)
            return false;
        const long long reach = (long long)(l.dims[i] - 1) * l.stride[i];
        (reach < 0 ? *lo : *hi) += reach;
    }
    return true;
}

inline bool is_q8(const Tensor* t) {
    return t->dtype.type_enum == TinyNN_QINT8 || t->dtype.type_enum == TinyNN_INT8;
}
inline bool is_q32(const Tensor* t) {
    return t->dtype.type_enum == TinyNN_QINT32 || t->dtype.type_enum == TinyNN_INT;
}
inline bool is_f32(const Tensor* t) {
    return t->dtype.type_enum == TinyNN_FLOAT;
}
inline size_t dtype_size(const Tensor* t) {
    switch (t->dtype.type_enum) {
        case TinyNN_FLOAT:
        case TinyNN_INT:
        case TinyNN_QINT32:
            return 4;
        case TinyNN_FLOAT16:
        case TinyNN_INT16:
            return 2;
        default:
            return 1;
    }
}

inline unsigned ceil_div(size_t a, size_t b) {
    return (unsigned)((a + b - 1) / b);
}

// NULL / pointer checks shared by every entry point (the reference kernels TINYNN_ASSERT these).
TinyNNStatus check_io(
        Tensor** inputs, int nr_input, int want_in_min, int want_in_max, Tensor** outputs,
        int nr_output, const char* who);

}  // namespace mg
