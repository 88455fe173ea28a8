// Host-side bounds audit of kernels that load unconditionally from clamped indices.
//
// Linked with the library's OWN kernel sources (test_bounds_audit.py lists them) compiled as host C++ against tests/host_audit/hip/hip_runtime.h,
// where a launch runs every thread of every workgroup one after the other on the CPU. The operand
// buffers are fenced: each sits at the very end (then, in a second pass, at the very start) of a
// mapping whose neighbouring page is inaccessible, so a load or store one element outside a tensor
// ends the process with SIGSEGV instead of reading a stray value. Nothing here restates an index
// formula: the addresses dereferenced are the ones the kernels compute.
//
// stdin: one case per line, stdout: "ok <line> -> <kernel noted>" per case; exit status 0 when all of them ran.
//   mm     M K N ta tb lda_pad ldb_pad ws     f32 MatMul through megcc_gfx950_matmul (gemm / gevm); ws = 1: with split-K room
//   conv   n ic ih iw oc k s p d bias ws      f32 NCHW convolution through the implicit GEMM
//   small  n ic ih iw oc k s p d bias         f32 NCHW convolution through conv_f32_small (k = 1 or 3)
//   dwf32  n c ih iw k s p bias               f32 channel-wise layer in NCHW44
//   first  n ic ih iw oc k s p bias           f32 first layer, NCHW source -> NCHW44 result
//   fcone  M K OC packed_bytes bias           qsi8 FullyConnected, M <= 64, one launch
//   fcgevm M K OC packed_bytes bias           qsi8 FullyConnected, M <= 4
//   fctile M K OC packed_bytes bias cus       qsi8 FullyConnected, any M and K, on a chip of that many CUs
//   ks     M K N ta tb lda_pad ldb_pad        f32 MatMul whose waves share K (whatever the dispatch would choose)
//   split  M K N ta tb lda_pad ldb_pad        f32 MatMul on the bf16 instructions, K >= 32 (likewise)
//   gather n ic ih iw oc k s p d bias packed_bytes       qsi8 dense NCHW44 convolution without staging
//   dwpw   n c oc h w stride bias packed_bytes           qsi8 channel-wise 3x3 + pointwise 1x1 in one kernel
//   pw     n ic ih iw oc stride bias packed_bytes cus    qsi8 pointwise NCHW44 layer, streaming, on a chip of that many CUs
//   ksplit M K N ta tb lda_pad ldb_pad ldc_pad kg slices swap   f32 MatMul of middle size on the bf16 instructions, by that plan
//   wide   n ic ih iw oc k s p d bias cus                f32 NCHW convolution of many pixels, on a chip of that many CUs
//   blocks n c h w count bias                            qsi8 run of channel-wise 3x3 + pointwise 1x1 blocks in one kernel
//   asked  n c h w cus                                   whether that one would be timed, noted as "conv_blocks_takes:1,0" or 0
//   stem   n oh ow oc act bias packed_bytes cus          f32 image -> qsi8 -> first convolution -> channel-wise -> pointwise in one kernel
#include <hip/hip_runtime.h>
#include <sanitizer/asan_interface.h>
#include <signal.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <sys/mman.h>
#include <unistd.h>

#include <sstream>
#include <string>
#include <vector>

#include "common.h"
#include "conv_dw_pw.h"
#include "conv_geom.h"
#include "epilogue.h"
#include "gemm_f32_ks.h"
#include "gemm_f32_split.h"
#include "gevm_f32.h"

namespace mg {
// what the kernel sources expect from the rest of the library
hipStream_t stream() { return nullptr; }
static int g_cus = 256;
int num_cus() { return g_cus; }
TinyNNStatus fail(TinyNNStatus st, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vfprintf(stderr, fmt, ap);
    va_end(ap);
    fputc('\n', stderr);
    return st;
}
Options& options() {
    static Options o = {};
    return o;
}
static std::string g_noted;
void note_kernel(const char* name, int a, int b, int, int, int) { g_noted = std::string(name) + ":" + std::to_string(a) + "," + std::to_string(b); }
void note_requant_affine(bool) {}
// (of the case at hand: the library's own figure, which the test passes in)
static size_t g_packed_bytes = 0;
size_t conv_mfma_packed_bytes(const ConvGeom&) { return g_packed_bytes; }
TinyNNStatus check_launch(const char*) { return TinyNN_SUCCESS; }
TinyNNStatus check_io(Tensor** in, int nin, int lo, int hi, Tensor** out, int nout, const char* who) {
    if (!in || !out || nin < lo || nin > hi || nout != 1)
        return fail(TinyNN_ERROR_OUT_OF_RANGE, "%s: operand count", who);
    return TinyNN_SUCCESS;
}
// dynamic LDS of fc_stream.hip / fc_gevm_q8.hip (`extern __shared__ ... name[]`)
__attribute__((aligned(16))) int8_t lds[160 * 1024];
__attribute__((aligned(16))) int fg_lds[40 * 1024];
// ... of gemm_f32_ks.hip, conv_gather_i8.hip and conv_dw_pw.hip
__attribute__((aligned(16))) float ks_lds[40 * 1024];
__attribute__((aligned(16))) int gather_lds[40 * 1024];
__attribute__((aligned(16))) int8_t dp_lds_mem[160 * 1024];

// ... of conv_f32_wide.hip and conv_blocks.hip, where what lies behind a launch's size is out of bounds too
__attribute__((aligned(16))) float cw_lds[40 * 1024];
__attribute__((aligned(16))) int8_t cb_lds[160 * 1024];

size_t gemm_f32_workspace_bytes(long M, long N, long K, bool conv);
size_t conv_f32_gemm_workspace_bytes(const ConvGeom& g);
TinyNNStatus conv_f32_gemm_launch(const ConvGeom&, const void*, const void*, const void*, void*, const Workspace*);
bool conv_f32_small_supported(const ConvGeom& g);
TinyNNStatus conv_f32_small_launch(const ConvGeom&, const void*, const void*, const void*, void*);
bool dwconv44_f32_supported(const ConvGeom&);
TinyNNStatus dwconv44_f32_launch(const ConvGeom&, const void*, const void*, const void*, void*);
bool conv_first_f32_supported(const ConvGeom&);
TinyNNStatus conv_first_f32_launch(const ConvGeom&, const void*, const void*, const void*, void*);
bool fc_one_supported(const ConvGeom& g, const void* src);
TinyNNStatus fc_one_launch(const ConvGeom&, const void*, const void*, const void*, void*);
bool fc_gevm_q8_supported(const ConvGeom& g);
TinyNNStatus fc_gevm_q8_launch(const ConvGeom&, const void*, const void*, const void*, void*);
bool fc_tile_supported(const ConvGeom& g);
TinyNNStatus fc_tile_launch(const ConvGeom&, const void*, const void*, const void*, void*);
bool conv_gather_i8_supported(const ConvGeom& g);
TinyNNStatus conv_gather_i8_launch(const ConvGeom&, const void*, const void*, const void*, void*);
bool conv_pw_stream_supported(const ConvGeom& g);
bool conv_pw_stream_takes_stride(const ConvGeom& g);
TinyNNStatus conv_pw_stream_launch(const ConvGeom&, const void*, const void*, const void*, void*);
bool conv_stem_supported(const ConvGeom&, const ConvGeom&, const ConvGeom&, const void*, const void*);
TinyNNStatus conv_stem_launch(
        const ConvGeom&, const ConvGeom&, const ConvGeom&, const void*, const void*, const void*, const void*, const void*, const void*,
        const void*, void*, bool);
bool conv_dw_pw_supported(const ConvGeom& dw, const ConvGeom& pw, const void* src, const void* dst);
TinyNNStatus conv_dw_pw_launch(
        const ConvGeom&, const ConvGeom&, const void*, const void*, const void*, const void*, const void*, void*, DwPwBlock*, bool);
}  // namespace mg

void* megcc_gfx950_malloc(size_t n) { return malloc(n); }
void megcc_gfx950_free(void* p) { free(p); }
TinyNNStatus megcc_gfx950_memcpy_h2d(void* dst, const void* src, size_t n) { return memcpy(dst, src, n), TinyNN_SUCCESS; }

bool audit_strict = false;
void audit_dynamic_lds(size_t bytes) {
    using namespace mg;
    for (auto lds : {std::make_pair((char*)cw_lds, sizeof(cw_lds)), std::make_pair((char*)cb_lds, sizeof(cb_lds))}) {
        __asan_unpoison_memory_region(lds.first, lds.second);
        if (bytes < lds.second)
            __asan_poison_memory_region(lds.first + bytes, lds.second - bytes);
    }
}

// the bf16 conversion of the compiler's vector types (its value does not matter here)
extern "C" __bf16 __truncsfbf2(float) { return __builtin_bit_cast(__bf16, (unsigned short)0); }

extern "C" TinyNNStatus megcc_gfx950_matmul(
        const MegccMatMulAttr*, Tensor**, int, Tensor**, int, const Workspace*, const RuntimeOpt*);

static std::string g_case;
void audit_beyond(const char* what, unsigned off, unsigned soff, unsigned bytes) {
    fprintf(stderr, "OUT OF BOUNDS: %s at %u + %u of %u bytes while running: %s\n", what, off, soff, bytes, g_case.c_str());
    _exit(3);
}
static void on_fault(int, siginfo_t* info, void*) {
    char buf[512];
    int n = snprintf(buf, sizeof(buf), "OUT OF BOUNDS: access at %p while running: %s\n", info->si_addr,
                     g_case.c_str());
    (void)!write(2, buf, n);
    _exit(3);
}

// what operands hold. As floats: 2.4e-38, which the bf16 parts of f32 products cannot hold, and 0.75
static const int kFills[] = {0x01, 0x3f};
static int g_fill = kFills[0];

// `bytes` usable bytes whose end (at_end) or start touches an inaccessible page
struct Fenced {
    void* map = nullptr;
    size_t map_bytes = 0;
    char* ptr = nullptr;
    Fenced(size_t bytes, bool at_end, size_t align) {
        const size_t page = 4096, body = (bytes + page - 1) / page * page + page;
        map_bytes = body + 2 * page;
        map = mmap(nullptr, map_bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
        if (map == MAP_FAILED) {
            perror("mmap");
            exit(2);
        }
        char* base = (char*)map;
        mprotect(base, page, PROT_NONE);
        mprotect(base + page + body, page, PROT_NONE);
        if (at_end) {
            // the last byte right below the fence, moved down only as far as `align` demands
            size_t start = page + body - bytes;
            start -= start % align;
            ptr = base + start;
        } else {
            ptr = base + page;
        }
        memset(ptr, g_fill, bytes);
    }
    ~Fenced() { munmap(map, map_bytes); }
};

static Tensor tensor2d(void* p, int rows, int cols, long ld) {
    Tensor t;
    memset(&t, 0, sizeof(t));
    t.ptr = p;
    t.dtype.type_enum = TinyNN_FLOAT;
    t.layout.nr_dim = 2;
    t.layout.dims[0] = rows;
    t.layout.dims[1] = cols;
    t.layout.stride[0] = (int)ld;
    t.layout.stride[1] = 1;
    return t;
}

static bool run_case(const std::string& line, bool at_end) {
    using namespace mg;
    std::stringstream ss(line);
    std::string kind;
    ss >> kind;
    g_cus = 256;
    audit_dynamic_lds(sizeof(cb_lds));  // (all of either)
    memset(cw_lds, 0, sizeof(cw_lds));
    memset(cb_lds, 0, sizeof(cb_lds));
    audit_strict = kind == "ksplit" || kind == "wide" || kind == "blocks";
    if (kind == "mm") {
        int M, K, N, ta, tb, pa, pb, ws;
        ss >> M >> K >> N >> ta >> tb >> pa >> pb >> ws;
        const int ar = ta ? K : M, ac = ta ? M : K, br = tb ? N : K, bc = tb ? K : N;
        const long lda = ac + pa, ldb = bc + pb;
        // a padded last row ends with its last element, not with its padding
        Fenced A(((size_t)(ar - 1) * lda + ac) * 4, at_end, 16), B(((size_t)(br - 1) * ldb + bc) * 4, at_end, 16),
                Cm((size_t)M * N * 4, at_end, 16);
        const size_t wsb = ws ? gemm_f32_workspace_bytes(M, N, K, false) : 0;
        Fenced W(wsb ? wsb : 16, at_end, 16);
        Tensor a = tensor2d(A.ptr, ar, ac, lda), b = tensor2d(B.ptr, br, bc, ldb), c = tensor2d(Cm.ptr, M, N, N);
        Tensor *in[2] = {&a, &b}, *out[1] = {&c};
        MegccMatMulAttr attr;
        memset(&attr, 0, sizeof(attr));
        attr.transpose_a = ta;
        attr.transpose_b = tb;
        Workspace w = {wsb ? W.ptr : nullptr, wsb, 0};
        return megcc_gfx950_matmul(&attr, in, 2, out, 1, &w, nullptr) == TinyNN_SUCCESS;
    }
    if (kind == "ks" || kind == "split") {
        int M, K, N, ta, tb, pa, pb;
        ss >> M >> K >> N >> ta >> tb >> pa >> pb;
        const int ar = ta ? K : M, ac = ta ? M : K, br = tb ? N : K, bc = tb ? K : N;
        const long lda = ac + pa, ldb = bc + pb;
        Fenced A(((size_t)(ar - 1) * lda + ac) * 4, at_end, 16), B(((size_t)(br - 1) * ldb + bc) * 4, at_end, 16),
                Cm((size_t)M * N * 4, at_end, 16);
        const GevmArgs v = {(const float*)A.ptr, (const float*)B.ptr, (float*)Cm.ptr, M, N, K, ta ? 1 : lda, ta ? lda : 1,
                            tb ? 1 : ldb, tb ? ldb : 1, N};
        return (kind == "ks" ? gemm_f32_ks_launch(v, ta, tb) : gemm_f32_split_launch(v, ta, tb)) == TinyNN_SUCCESS;
    }
    if (kind == "ksplit") {
        int M, K, N, ta, tb, pa, pb, pc;
        KpPlan plan;
        ss >> M >> K >> N >> ta >> tb >> pa >> pb >> pc >> plan.kg >> plan.slices >> plan.swap;
        const int ar = ta ? K : M, ac = ta ? M : K, br = tb ? N : K, bc = tb ? K : N;
        const long lda = ac + pa, ldb = bc + pb, ldc = N + pc;
        Fenced A(((size_t)(ar - 1) * lda + ac) * 4, at_end, 4), B(((size_t)(br - 1) * ldb + bc) * 4, at_end, 4),
                Cm(((size_t)(M - 1) * ldc + N) * 4, at_end, 4), W((size_t)plan.slices * M * N * 4, at_end, 4);
        const GevmArgs v = {(const float*)A.ptr, (const float*)B.ptr, (float*)Cm.ptr, M, N, K, ta ? 1 : lda, ta ? lda : 1,
                            tb ? 1 : ldb, tb ? ldb : 1, ldc};
        const Workspace w = {plan.slices > 1 ? W.ptr : nullptr, plan.slices > 1 ? (size_t)plan.slices * M * N * 4 : 0, 0};
        return gemm_f32_ks_split_launch(v, ta, tb, plan, &w) == TinyNN_SUCCESS;
    }
    if (kind == "wide") {
        ConvGeom g;
        memset(&g, 0, sizeof(g));
        int k, s, p, d, bias;
        ss >> g.n >> g.ic >> g.ih >> g.iw >> g.oc >> k >> s >> p >> d >> bias >> g_cus;
        g.fh = g.fw = k, g.sh = g.sw = s, g.ph = g.pw = p, g.dh = g.dw = d;
        g.oh = (g.ih + 2 * p - (d * (k - 1) + 1)) / s + 1;
        g.ow = (g.iw + 2 * p - (d * (k - 1) + 1)) / s + 1;
        g.groups = 1, g.fmt = MEGCC_FMT_NCHW, g.act = MEGCC_NONLINE_RELU, g.has_bias = bias;
        Fenced src((size_t)g.n * g.ic * g.ih * g.iw * 4, at_end, 4), flt((size_t)g.oc * g.ic * k * k * 4, at_end, 4), b((size_t)g.oc * 4, at_end, 4),
                dst((size_t)g.n * g.oc * g.oh * g.ow * 4, at_end, 4);
        // (the second time every thread finds the whole table, which the threads of a workgroup write one after the other here)
        return conv_f32_wide_launch(g, src.ptr, flt.ptr, bias ? b.ptr : nullptr, dst.ptr) == TinyNN_SUCCESS &&
               conv_f32_wide_launch(g, src.ptr, flt.ptr, bias ? b.ptr : nullptr, dst.ptr) == TinyNN_SUCCESS;
    }
    if (kind == "blocks") {
        int n, c, h, w, count, bias;
        ss >> n >> c >> h >> w >> count >> bias;
        const size_t image = (size_t)n * c * h * w;
        Fenced src(image, at_end, 4), dst(image, at_end, 4), df((size_t)c * 9, at_end, 4), db((size_t)c * 4, at_end, 4), wp((size_t)c * c, at_end, 16),
                pb((size_t)c * 4, at_end, 4);
        std::vector<DwPwBlock> blocks((size_t)count);
        std::vector<const DwPwBlock*> run;
        for (int i = 0; i < count; ++i) {
            DwPwArgs a;
            memset(&a, 0, sizeof(a));
            // (what lies between two blocks is neither read nor written)
            a.src = i ? blocks[(size_t)i - 1].host[0].a.dst : (const uint32_t*)src.ptr;
            a.dst = i + 1 < count ? (uint32_t*)(uintptr_t)(64 * (i + 1)) : (uint32_t*)dst.ptr;
            a.dflt = (const uint32_t*)df.ptr, a.wp = (const int8_t*)wp.ptr;
            a.dbias = bias ? (const int32_t*)db.ptr : nullptr, a.pbias = bias ? (const int32_t*)pb.ptr : nullptr;
            a.src_bytes = a.dst_bytes = (int)image;
            a.ih = a.oh = h, a.iw = a.ow = w, a.OC = a.OCP = c;
            a.dq.mode = a.pq.mode = 2;
            blocks[(size_t)i].host[0].a = blocks[(size_t)i].host[1].a = a;
            blocks[(size_t)i].act = MEGCC_NONLINE_RELU;
            run.push_back(&blocks[(size_t)i]);
        }
        BlocksRun* r = conv_blocks_create(run.data(), count);
        if (!r) {
            fprintf(stderr, "not a conv_blocks run: %s\n", line.c_str());
            return false;
        }
        const TinyNNStatus st = conv_blocks_launch(r);
        conv_blocks_destroy(r);
        return st == TinyNN_SUCCESS;
    }
    if (kind == "asked") {
        int n, c, h, w;
        ss >> n >> c >> h >> w >> g_cus;
        Tensor x = tensor2d(nullptr, 1, 1, 1);
        const uint32_t dims[5] = {(uint32_t)n, (uint32_t)c / 4, (uint32_t)h, (uint32_t)w, 4};
        x.layout.nr_dim = 5;
        std::copy(dims, dims + 5, x.layout.dims);
        note_kernel("conv_blocks_takes", conv_blocks_takes(x), 0, 0, 0, 0);
        return true;
    }
    if (kind == "gather") {
        ConvGeom g;
        memset(&g, 0, sizeof(g));
        int k, s, p, d, bias;
        ss >> g.n >> g.ic >> g.ih >> g.iw >> g.oc >> k >> s >> p >> d >> bias >> g_packed_bytes;
        g.fh = g.fw = k, g.sh = g.sw = s, g.ph = g.pw = p, g.dh = g.dw = d;
        g.oh = (g.ih + 2 * p - (d * (k - 1) + 1)) / s + 1;
        g.ow = (g.iw + 2 * p - (d * (k - 1) + 1)) / s + 1;
        // (an activation without a threshold table: there is no kernel-argument segment to read one from)
        g.groups = 1, g.fmt = MEGCC_FMT_NCHW44, g.act = MEGCC_NONLINE_SIGMOID, g.has_bias = bias;
        g.s_src = g.s_flt = 0.01f, g.s_dst = 0.1f;
        Fenced src((size_t)g.n * g.ic * g.ih * g.iw, at_end, 4), wp(g_packed_bytes, at_end, 16), b((size_t)g.oc * 4, at_end, 4),
                dst((size_t)g.n * g.oc * g.oh * g.ow, at_end, 4);
        if (!conv_gather_i8_supported(g)) {
            fprintf(stderr, "not a conv_gather_i8 layer: %s\n", line.c_str());
            return false;
        }
        return conv_gather_i8_launch(g, src.ptr, wp.ptr, bias ? b.ptr : nullptr, dst.ptr) == TinyNN_SUCCESS;
    }
    if (kind == "dwpw") {
        ConvGeom dw, pw;
        memset(&dw, 0, sizeof(dw));
        int oc, stride, bias;
        ss >> dw.n >> dw.ic >> oc >> dw.ih >> dw.iw >> stride >> bias >> g_packed_bytes;
        dw.oc = dw.groups = dw.ic, dw.fh = dw.fw = 3, dw.sh = dw.sw = stride, dw.ph = dw.pw = dw.dh = dw.dw = 1;
        dw.oh = (dw.ih - 1) / stride + 1, dw.ow = (dw.iw - 1) / stride + 1;
        dw.fmt = MEGCC_FMT_NCHW44, dw.act = MEGCC_NONLINE_RELU, dw.has_bias = bias;
        dw.s_src = dw.s_flt = 0.01f, dw.s_dst = 0.1f;
        pw = dw;
        pw.oc = oc, pw.groups = 1, pw.ih = dw.oh, pw.iw = dw.ow, pw.fh = pw.fw = pw.sh = pw.sw = 1, pw.ph = pw.pw = 0;
        Fenced src((size_t)dw.n * dw.ic * dw.ih * dw.iw, at_end, 16), df((size_t)dw.ic * 9, at_end, 4), db((size_t)dw.ic * 4, at_end, 4),
                wp(g_packed_bytes, at_end, 16), pb((size_t)oc * 4, at_end, 4), dst((size_t)dw.n * oc * dw.oh * dw.ow, at_end, 4);
        if (!conv_dw_pw_supported(dw, pw, src.ptr, dst.ptr)) {
            fprintf(stderr, "not a conv_dw_pw pair: %s\n", line.c_str());
            return false;
        }
        return conv_dw_pw_launch(dw, pw, src.ptr, df.ptr, bias ? db.ptr : nullptr, wp.ptr, bias ? pb.ptr : nullptr, dst.ptr, nullptr,
                                 false) == TinyNN_SUCCESS;
    }
    if (kind == "pw") {
        ConvGeom g;
        memset(&g, 0, sizeof(g));
        int s, bias;
        ss >> g.n >> g.ic >> g.ih >> g.iw >> g.oc >> s >> bias >> g_packed_bytes >> g_cus;
        g.fh = g.fw = g.dh = g.dw = 1, g.sh = g.sw = s;
        g.oh = (g.ih - 1) / s + 1, g.ow = (g.iw - 1) / s + 1;
        g.groups = 1, g.fmt = MEGCC_FMT_NCHW44, g.act = MEGCC_NONLINE_RELU, g.has_bias = bias;
        g.s_src = g.s_flt = 0.01f, g.s_dst = 0.1f;
        Fenced src((size_t)g.n * g.ic * g.ih * g.iw, at_end, 4), wp(g_packed_bytes, at_end, 16), b((size_t)g.oc * 4, at_end, 4),
                dst((size_t)g.n * g.oc * g.oh * g.ow, at_end, 4);
        if (!(s == 1 ? conv_pw_stream_supported(g) : conv_pw_stream_takes_stride(g))) {
            fprintf(stderr, "not a conv_pw_stream layer: %s\n", line.c_str());
            return false;
        }
        return conv_pw_stream_launch(g, src.ptr, wp.ptr, bias ? b.ptr : nullptr, dst.ptr) == TinyNN_SUCCESS;
    }
    if (kind == "stem") {
        ConvGeom c0, dw, pw;
        memset(&c0, 0, sizeof(c0));
        int oc, act, bias;
        ss >> c0.n >> c0.oh >> c0.ow >> oc >> act >> bias >> g_packed_bytes >> g_cus;
        c0.ic = 3, c0.oc = 32, c0.ih = 2 * c0.oh, c0.iw = 2 * c0.ow, c0.fh = c0.fw = 3, c0.sh = c0.sw = 2;
        c0.ph = c0.pw = c0.dh = c0.dw = c0.groups = 1, c0.fmt = MEGCC_FMT_NCHW_NCHW44, c0.act = MEGCC_NONLINE_RELU, c0.has_bias = bias;
        c0.s_src = 1.f / 127, c0.s_flt = 0.0051f, c0.s_dst = 0.037f;
        dw = c0;
        dw.ic = dw.oc = dw.groups = 32, dw.ih = c0.oh, dw.iw = c0.ow, dw.sh = dw.sw = 1, dw.fmt = MEGCC_FMT_NCHW44;
        pw = dw;
        pw.oc = oc, pw.groups = pw.fh = pw.fw = 1, pw.ph = pw.pw = 0, pw.act = act ? MEGCC_NONLINE_RELU : MEGCC_NONLINE_IDENTITY;
        Fenced image((size_t)c0.n * 3 * c0.ih * c0.iw * 4, at_end, 4), f0(8 * 27 * 4, at_end, 1), b0(32 * 4, at_end, 4), df(32 * 9, at_end, 4),
                db(32 * 4, at_end, 4), wp(g_packed_bytes, at_end, 16), pb((size_t)oc * 4, at_end, 4),
                dst((size_t)c0.n * oc * c0.oh * c0.ow, at_end, 4);
        if (!conv_stem_supported(c0, dw, pw, image.ptr, dst.ptr)) {
            fprintf(stderr, "not a conv_stem chain: %s\n", line.c_str());
            return false;
        }
        return conv_stem_launch(c0, dw, pw, image.ptr, f0.ptr, bias ? b0.ptr : nullptr, df.ptr, bias ? db.ptr : nullptr, wp.ptr,
                                bias ? pb.ptr : nullptr, dst.ptr, true) == TinyNN_SUCCESS;
    }
    if (kind == "conv" || kind == "small") {
        ConvGeom g;
        memset(&g, 0, sizeof(g));
        int k, s, p, d, bias, ws = 0;
        ss >> g.n >> g.ic >> g.ih >> g.iw >> g.oc >> k >> s >> p >> d >> bias;
        if (kind == "conv")
            ss >> ws;
        g.fh = g.fw = k, g.sh = g.sw = s, g.ph = g.pw = p, g.dh = g.dw = d;
        g.oh = (g.ih + 2 * p - (d * (k - 1) + 1)) / s + 1;
        g.ow = (g.iw + 2 * p - (d * (k - 1) + 1)) / s + 1;
        g.groups = 1, g.fmt = MEGCC_FMT_NCHW, g.act = MEGCC_NONLINE_RELU, g.has_bias = bias;
        Fenced src((size_t)g.n * g.ic * g.ih * g.iw * 4, at_end, 16), flt((size_t)g.oc * g.ic * k * k * 4, at_end, 16),
                b((size_t)g.oc * 4, at_end, 4), dst((size_t)g.n * g.oc * g.oh * g.ow * 4, at_end, 16);
        if (kind == "small") {
            if (!conv_f32_small_supported(g)) {
                fprintf(stderr, "not a conv_f32_small layer: %s\n", line.c_str());
                return false;
            }
            return conv_f32_small_launch(g, src.ptr, flt.ptr, bias ? b.ptr : nullptr, dst.ptr) == TinyNN_SUCCESS;
        }
        const size_t wsb = ws ? conv_f32_gemm_workspace_bytes(g) : 0;
        Fenced W(wsb ? wsb : 16, at_end, 16);
        Workspace w = {wsb ? W.ptr : nullptr, wsb, 0};
        return conv_f32_gemm_launch(g, src.ptr, flt.ptr, bias ? b.ptr : nullptr, dst.ptr, &w) == TinyNN_SUCCESS;
    }
    if (kind == "dwf32" || kind == "first") {
        ConvGeom g;
        memset(&g, 0, sizeof(g));
        int k, s, p, bias;
        ss >> g.n >> g.ic >> g.ih >> g.iw;
        if (kind == "first")
            ss >> g.oc;
        else
            g.oc = g.ic;
        ss >> k >> s >> p >> bias;
        g.fh = g.fw = k, g.sh = g.sw = s, g.ph = g.pw = p, g.dh = g.dw = 1;
        g.oh = (g.ih + 2 * p - k) / s + 1;
        g.ow = (g.iw + 2 * p - k) / s + 1;
        g.groups = kind == "first" ? 1 : g.ic;
        g.fmt = kind == "first" ? MEGCC_FMT_NCHW_NCHW44 : MEGCC_FMT_NCHW44;
        g.act = MEGCC_NONLINE_H_SWISH, g.has_bias = bias;
        const size_t taps = (size_t)k * k * (kind == "first" ? (size_t)g.ic * g.oc : (size_t)g.ic);
        Fenced src((size_t)g.n * g.ic * g.ih * g.iw * 4, at_end, 16), flt(taps * 4, at_end, 16),
                b((size_t)g.oc * 4, at_end, 16), dst((size_t)g.n * g.oc * g.oh * g.ow * 4, at_end, 16);
        if (kind == "first") {
            if (!conv_first_f32_supported(g)) {
                fprintf(stderr, "not a conv_first_f32 layer: %s\n", line.c_str());
                return false;
            }
            return conv_first_f32_launch(g, src.ptr, flt.ptr, bias ? b.ptr : nullptr, dst.ptr) == TinyNN_SUCCESS;
        }
        if (!dwconv44_f32_supported(g)) {
            fprintf(stderr, "not a dwconv44_f32 layer: %s\n", line.c_str());
            return false;
        }
        return dwconv44_f32_launch(g, src.ptr, flt.ptr, bias ? b.ptr : nullptr, dst.ptr) == TinyNN_SUCCESS;
    }
    if (kind == "fcone" || kind == "fcgevm" || kind == "fctile") {
        ConvGeom g;
        memset(&g, 0, sizeof(g));
        long packed;
        int bias;
        ss >> g.n >> g.ic >> g.oc >> packed >> bias;
        if (kind == "fctile")
            ss >> g_cus;
        g.ih = g.iw = g.oh = g.ow = g.fh = g.fw = g.sh = g.sw = g.dh = g.dw = 1;
        g.groups = 1, g.fmt = MEGCC_FMT_NCHW, g.act = MEGCC_NONLINE_RELU, g.has_bias = bias;
        g.s_src = g.s_flt = 0.01f, g.s_dst = 0.1f;
        Fenced src((size_t)g.n * g.ic, at_end, 16), wp((size_t)packed, at_end, 16), b((size_t)g.oc * 4, at_end, 4),
                dst((size_t)g.n * g.oc, at_end, g.oc % 4 ? 1 : 4);
        if (kind == "fctile") {
            if (!fc_tile_supported(g)) {
                fprintf(stderr, "not an fc_tile layer: %s\n", line.c_str());
                return false;
            }
            return fc_tile_launch(g, src.ptr, wp.ptr, bias ? b.ptr : nullptr, dst.ptr) == TinyNN_SUCCESS;
        }
        if (kind == "fcone") {
            if (!fc_one_supported(g, src.ptr)) {
                fprintf(stderr, "not an fc_one layer: %s\n", line.c_str());
                return false;
            }
            return fc_one_launch(g, src.ptr, wp.ptr, bias ? b.ptr : nullptr, dst.ptr) == TinyNN_SUCCESS;
        }
        if (!fc_gevm_q8_supported(g)) {
            fprintf(stderr, "not an fc_gevm_q8 layer: %s\n", line.c_str());
            return false;
        }
        return fc_gevm_q8_launch(g, src.ptr, wp.ptr, bias ? b.ptr : nullptr, dst.ptr) == TinyNN_SUCCESS;
    }
    fprintf(stderr, "unknown case kind: %s\n", line.c_str());
    return false;
}

int main() {
    struct sigaction sa;
    memset(&sa, 0, sizeof(sa));
    sa.sa_sigaction = on_fault;
    sa.sa_flags = SA_SIGINFO;
    sigaction(SIGSEGV, &sa, nullptr);
    sigaction(SIGBUS, &sa, nullptr);
    char buf[512];
    int n = 0;
    while (fgets(buf, sizeof(buf), stdin)) {
        std::string line(buf);
        while (!line.empty() && (line.back() == '\n' || line.back() == ' '))
            line.pop_back();
        if (line.empty() || line[0] == '#')
            continue;
        const bool parts = line.rfind("split ", 0) == 0 || line.rfind("ksplit ", 0) == 0;
        for (int fill : kFills) {
            if (fill != kFills[0] && !parts)
                continue;
            g_fill = fill;
            for (int at_end = 1; at_end >= 0; --at_end) {
                g_case = line + (at_end ? "  [buffers end at a fence]" : "  [buffers start at a fence]");
                if (!run_case(line, at_end != 0)) {
                    fprintf(stderr, "FAILED: %s\n", g_case.c_str());
                    return 1;
                }
            }
        }
        g_fill = kFills[0];
        printf("ok %s -> %s\n", line.c_str(), mg::g_noted.c_str());
        fflush(stdout);
        ++n;
    }
    printf("audited %d cases\n", n);
    return 0;
}
