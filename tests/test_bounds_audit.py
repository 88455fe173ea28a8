"""Host-side bounds audit of the kernels that issue their loads unconditionally from clamped
indices or through range-checked buffers (gemm_f32: all four transpositions and the implicit-GEMM gather; gemm_f32_ks,
gemm_f32_split and gemm_f32_ks_split: all four transpositions; conv_f32_wide; conv_blocks; gevm_f32; conv_f32_small; the f32 NCHW44 channel-wise and first-layer kernels;
fc_one32 / fc_one; every part of fc_tile; fc_gevm_q8; conv_gather_i8; conv_pw_stream / conv_pw_share with and without a stride; conv_dw_pw;
conv_stem). Not gemm_f32_ks's convolution, whose addresses come through LDS from other threads. tests/host_audit/audit.cpp links the library's own kernel sources,
compiled as host C++ against a stand-in HIP header that runs every thread of every workgroup on
the CPU, and fences each operand buffer with inaccessible pages: one element outside a tensor ends
the run. No GPU involved; the shapes are every case of the GPU sweeps plus a seeded sweep of ragged
shapes aimed at the tile edges."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

from cases import ConvCase, MatMulCase
from megcc_amd import abi, runtime

HERE = os.path.dirname(os.path.abspath(__file__))
AUDIT_DIR = os.path.join(HERE, "host_audit")
CSRC = os.path.join(os.path.dirname(HERE), "megcc_amd", "csrc")
CLANG = "/opt/rocm/llvm/bin/clang++"
SOURCES = ["gemm_f32", "gevm_f32", "conv_f32_small", "conv_f32_nchw44", "fc_stream", "fc_gevm_q8", "fc_tile", "gemm_f32_ks",
           "gemm_f32_split", "conv_gather_i8", "conv_pw_stream", "conv_dw_pw", "conv_stem", "requant_table"]
# compiled with the address sanitizer (host code, like all of it), so that an access beyond a workgroup's LDS ends the run as well
CHECKED = ["gemm_f32_ks_split", "conv_f32_wide", "conv_blocks"]

pytestmark = pytest.mark.skipif(not os.path.exists(CLANG), reason="needs ROCm's clang++ for the kernels' vector types")


def compile_audit(out_dir, replace=None, have=None):
    """replace: {source name: path of another file to compile in its place}; have: folder with the objects of the others"""
    os.makedirs(out_dir, exist_ok=True)
    flags = ["-x", "c++", "-std=c++17", "-O1", "-g", "-I" + AUDIT_DIR, "-I" + CSRC,
             "-I" + os.path.join(os.path.dirname(HERE), "include"), "-ffp-contract=off", "-Wno-unknown-attributes"]
    objs = []
    jobs = []
    for name in SOURCES + CHECKED + ["audit"]:
        src = os.path.join(AUDIT_DIR, "audit.cpp") if name == "audit" else os.path.join(CSRC, name + ".hip")
        if replace and name in replace:
            src = replace[name]
        obj = os.path.join(out_dir, name + ".o")
        if have and not (replace and name in replace):
            objs.append(os.path.join(have, name + ".o"))
            continue
        objs.append(obj)
        last = ["-O0", "-g0"] if name in ("conv_dw_pw", "conv_pw_stream") else []  # (some 100 instances: half a minute with the optimiser)
        # (without the optimiser, which leaves out loads that only the stood-in instructions use)
        last += ["-O0", "-g0", "-fsanitize=address"] if name in CHECKED else []
        jobs.append(subprocess.Popen([CLANG] + flags + last + ["-c", src, "-o", obj], stderr=subprocess.PIPE, text=True))
    for j in jobs:
        err = j.communicate()[1]
        assert j.returncode == 0, err[-4000:]
    exe = os.path.join(out_dir, "audit")
    subprocess.check_call([CLANG, "-fsanitize=address", "-o", exe] + objs)
    return exe


@pytest.fixture(scope="module")
def audit_exe(tmp_path_factory):
    return compile_audit(str(tmp_path_factory.mktemp("host_audit")))


def packed_bytes(case):
    """size of the packed filter the layer's init step produces (host code of the library)"""
    arrays = {"src": None}
    desc = runtime.parse_symbol(case.symbol())
    tin = [abi.make_tensor(None, case.src_shape(), abi.QINT8, case.scales[0], b"src"),
           abi.make_tensor(None, case.flt_shape(), abi.QINT8, case.scales[1], b"flt")]
    if case.bias:
        tin.append(abi.make_tensor(None, case.bias_shape(), abi.QINT32, case.scales[0] * case.scales[1], b"bias"))
    w = abi.Tensor()
    runtime.check(runtime.lib().megcc_gfx950_call_init(C.byref(desc), abi.tensor_array(tin), len(tin), C.byref(w),
                                                       None, None), "init(describe)")
    n = 1
    for i in range(w.layout.nr_dim):
        n *= w.layout.dims[i]
    return n


def line_of(case, with_ws=1):
    if isinstance(case, MatMulCase):
        return "mm %d %d %d %d %d 0 0 %d" % (case.m, case.k, case.n, case.trans_a, case.trans_b, with_ws)
    assert isinstance(case, ConvCase)
    if case.dtype == "f32":
        macs = case.n * case.oh * case.ow * case.oc * case.ic * case.fh * case.fw
        small = case.fh in (1, 3) and case.fh == case.fw and macs <= 2 ** 27
        kind = "small" if small else "conv"
        tail = "" if small else " %d" % with_ws
        return "%s %d %d %d %d %d %d %d %d %d %d%s" % (kind, case.n, case.ic, case.ih, case.iw, case.oc, case.fh,
                                                       case.sh, case.ph, case.dh, int(case.bias), tail)
    kind = "fcgevm" if case.n <= 4 else "fcone"
    return "%s %d %d %d %d %d" % (kind, case.n, case.ic, case.oc, packed_bytes(case), int(case.bias))


FC_TILE_PARTS = [(130, 65, 150), (131, 260, 149), (129, 127, 193), (100, 2049, 101), (128, 2052, 98), (130, 2049, 129), (200, 1924, 130)]


def audit_lines():
    import test_gpu_parity as gp
    lines = []
    for _, case in gp.F32_SWEEP:
        if isinstance(case, ConvCase) and case.fmt != abi.FMT_NCHW:
            continue  # (NCHW44 layers reach the same kernel through relayouts of dense copies)
        lines.append(line_of(case))
    for case in gp.FC_SWEEP:
        if isinstance(case, ConvCase) and case.ic > 8192:
            continue  # (fc_stream: loads under range tests, not audited here)
        lines.append(line_of(case))
    r = np.random.Generator(np.random.PCG64(2024))
    # MatMul: every transposition x {inside, ragged} x {with, without split-K room}, padded rows, skinny tiles
    for i in range(40):
        m = int(r.choice([1, 2, 3, 4, 5, 31, 64, 65, 127, 128, 129, 200]))
        k = int(r.choice([1, 2, 15, 16, 17, 64, 100, 128, 513, 1040, 2049]))
        n = int(r.choice([1, 3, 4, 5, 63, 127, 128, 129, 255, 256, 257, 1000, 1024]))
        lines.append("mm %d %d %d %d %d %d %d %d" % (m, k, n, r.integers(0, 2), r.integers(0, 2),
                                                       r.choice([0, 1, 4, 7]), r.choice([0, 1, 4, 7]), r.integers(0, 2)))
    # implicit GEMM: pixel counts around multiples of the 128 / 256 pixel tiles, ragged K, few channels
    for i in range(24):
        k = int(r.choice([1, 3, 5]))
        s, d = int(r.integers(1, 3)), int(r.integers(1, 3)) if k == 3 else 1
        p = int(r.integers(0, k // 2 + 2))
        ic, oc = int(r.choice([1, 3, 16, 33, 64, 100])), int(r.choice([1, 5, 63, 64, 65, 128, 130]))
        ih, iw, n = int(r.integers(6, 40)), int(r.integers(6, 40)), int(r.integers(1, 6))
        if ih + 2 * p < d * (k - 1) + 1 or iw + 2 * p < d * (k - 1) + 1:
            continue
        lines.append("conv %d %d %d %d %d %d %d %d %d %d %d" % (n, ic, ih, iw, oc, k, s, p, d, r.integers(0, 2),
                                                               r.integers(0, 2)))
    lines.append("conv 3 86 45 42 117 5 2 3 1 1 1")  # 1584 = 12 x 128 + 48 pixels: the ragged last tile once read past the tensor
    # small layers: one pixel, one channel, rows shorter than the window, strides, dilation
    for (n, ic, ih, iw, oc, k, s, p, d) in [(1, 1, 1, 1, 1, 1, 1, 0, 1), (1, 1, 3, 3, 1, 3, 1, 1, 1), (2, 3, 5, 7, 5, 3, 2, 1, 1),
                                            (1, 32, 56, 56, 32, 3, 1, 1, 1), (3, 7, 9, 11, 13, 3, 1, 2, 2), (1, 5, 2, 2, 3, 3, 1, 1, 1),
                                            (4, 9, 17, 3, 6, 1, 2, 0, 1), (1, 64, 13, 13, 66, 3, 1, 0, 1), (5, 2, 8, 64, 3, 3, 2, 1, 2)]:
        lines.append("small %d %d %d %d %d %d %d %d %d 1" % (n, ic, ih, iw, oc, k, s, p, d))
    # f32 NCHW44: channel-wise tiles of 4 x 64 pixels with halos, first layers of 256-pixel blocks
    for _, case in gp.F32_NCHW44:
        if case.sparse == abi.GROUP and case.fh in (3, 5):
            lines.append("dwf32 %d %d %d %d %d %d %d %d" % (case.n, case.ic, case.ih, case.iw, case.fh, case.sh,
                                                          case.ph, int(case.bias)))
        elif case.fmt == abi.FMT_NCHW_NCHW44:
            lines.append("first %d %d %d %d %d %d %d %d %d" % (case.n, case.ic, case.ih, case.iw, case.oc, case.fh,
                                                             case.sh, case.ph, int(case.bias)))
    for i in range(16):
        k, s = int(r.choice([3, 5])), int(r.integers(1, 3))
        ih, iw = int(r.integers(1, 20)), int(r.choice([1, 2, 63, 64, 65, 127, 129, 200]))
        p = int(r.integers(0, k // 2 + 2))
        if ih + 2 * p < k or iw + 2 * p < k:
            continue
        lines.append("dwf32 %d %d %d %d %d %d %d %d" % (r.integers(1, 4), 4 * r.integers(1, 5), ih, iw, k, s, p,
                                                      r.integers(0, 2)))
    for i in range(12):
        k, s = int(r.choice([3, 5, 7])), int(r.integers(1, 3))
        ih, iw = int(r.integers(3, 40)), int(r.integers(3, 70))
        p = int(r.integers(0, k // 2 + 2))
        if ih + 2 * p < k or iw + 2 * p < k:
            continue
        lines.append("first %d %d %d %d %d %d %d %d %d" % (r.integers(1, 4), r.integers(1, 5), ih, iw,
                                                         4 * r.choice([1, 2, 8, 9, 16]), k, s, p, r.integers(0, 2)))
    # f32 products whose waves share K and those on the bf16 instructions: edges of the 32 / 64 / 128 tiles, K with and
    # without a rest, every transposition, padded rows
    for i in range(32):
        m, n = (int(r.choice([1, 5, 31, 32, 33, 64, 65, 127, 128, 129, 200])) for _ in range(2))
        k = int(r.choice([1, 3, 7, 8, 9, 31, 64, 100, 300]))
        tail = "%d %d %d %d" % (r.integers(0, 2), r.integers(0, 2), r.choice([0, 1, 4, 7]), r.choice([0, 1, 4, 7]))
        lines.append("ks %d %d %d %s" % (m, k, n, tail))
        lines.append("split %d %d %d %s" % (m, 32 + int(r.choice([0, 1, 15, 16, 17, 100, 143, 500])), n, tail))
    # ... 16 x 16 tiles up to two a CU, in strips with workgroups left over; then 32 x 32
    for m, k, n in ((15, 17, 16), (17, 15, 33), (100, 33, 300), (357, 16, 301), (40, 300, 1700), (513, 9, 530), (600, 31, 700)):
        for t in range(4):
            lines.append("ks %d %d %d %d %d 0 0" % (m, k, n, t & 1, t >> 1))
    # ... those of middle size, by every plan: rows and columns beyond tiles of 64, 128 and 256; K of less than a stage of 64, of stages and chains with
    # and without a rest; slices, the last one of less than a stage; padded rows of all three
    plans = [(kg, slices, swap) for kg in (1, 2, 4) for slices in (1, 2, 3) for swap in (0, 1) if not (kg == 4 and swap)]
    for t in range(4):
        for i, plan in enumerate(plans):
            for k in ((64, 65, 191), (128, 577, 63), (66, 260, 1))[i % 3]:
                m, n = (int(r.choice([1, 31, 64, 65, 100, 129])) for _ in range(2))
                lines.append("ksplit %d %d %d %d %d %d %d %d %d %d %d" % ((m, k, n, t & 1, t >> 1) + tuple(int(r.choice([0, 1, 4, 7])) for _ in range(3)) + plan))
    for plan in plans:
        lines.append("ksplit 70 1100 270 %d %d 0 3 5 %d %d %d" % ((plan[0] & 1, plan[2]) + plan))
    # convolutions of many pixels, tiles of 16, 32 and 64 channels: K below a step, of steps, of turns of four and with a rest, taps outside,
    # a stride, a dilation, pixels beyond the last wave
    for n, ic, ih, iw, oc, k, st, p, d in (
            (1, 1, 1, 1, 1, 1, 1, 0, 1), (3, 1, 5, 9, 7, 1, 1, 0, 1), (1, 7, 11, 12, 16, 1, 1, 0, 1), (2, 8, 8, 8, 17, 1, 1, 0, 1), (2, 9, 9, 15, 31, 1, 2, 0, 1), (1, 33, 12, 11, 33, 1, 1, 0, 1),
            (1, 64, 16, 16, 64, 1, 1, 0, 1), (1, 65, 13, 10, 65, 1, 1, 0, 1), (2, 130, 9, 9, 130, 1, 1, 0, 1), (1, 1, 9, 17, 12, 3, 1, 1, 1), (3, 2, 7, 7, 9, 3, 2, 1, 1), (2, 5, 10, 14, 40, 5, 1, 2, 1),
            (1, 9, 16, 15, 15, 3, 1, 2, 2), (1, 16, 13, 11, 70, 3, 1, 1, 1), (2, 3, 21, 23, 24, 5, 2, 2, 1), (1, 40, 12, 13, 64, 3, 1, 0, 1), (2, 128, 8, 9, 11, 3, 1, 1, 1), (1, 100, 9, 9, 128, 3, 1, 1, 1),
            (1, 17, 3, 90, 18, 1, 1, 1, 1), (1, 70, 12, 12, 8, 3, 1, 1, 1), (1, 96, 10, 13, 80, 3, 2, 1, 1),
            (1, 5, 12, 13, 11, 3, 1, 1, 1), (1, 48, 9, 10, 10, 1, 1, 0, 1), (1, 63, 9, 9, 14, 1, 2, 0, 1), (2, 6, 11, 9, 40, 3, 1, 1, 1), (1, 16, 9, 9, 20, 1, 1, 0, 1)):  # (short K)
        lines.append("wide %d %d %d %d %d %d %d %d %d %d %d" % (n, ic, ih, iw, oc, k, st, p, d, oc & 1, 1 + 7 * (ic & 1)))
    # runs of blocks: every kind of map, both numbers of channels
    for n, h, w, count in ((1, 1, 1, 3), (2, 1, 15, 2), (1, 2, 3, 2), (1, 14, 1, 2), (2, 3, 5, 2), (1, 7, 7, 3), (1, 9, 11, 2), (1, 13, 15, 2), (2, 14, 14, 5), (2, 14, 15, 2)):
        for c in (256, 512):
            lines.append("blocks %d %d %d %d %d %d" % (n, c, h, w, count, (h + w + c // 256) & 1))
    # FullyConnected of any K on tiles: rows at any byte, the tensor's last 16 bytes anywhere in a piece
    for m, k, oc in ((65, 5, 9), (64, 1, 3), (16, 1, 1), (65, 129, 67), (70, 295, 70), (225, 515, 361), (66, 128, 64), (130, 260, 257),
                     (100, 1123, 65), (65, 127, 129), (300, 33, 31)):
        case = ConvCase(abi.FMT_NCHW, abi.DENSE, m, k, 1, 1, oc, 1, 1, 0, abi.RELU, scales=(0.01, 0.01, 0.1))
        lines.append("fctile %d %d %d %d %d 256" % (m, k, oc, packed_bytes(case), i & 1))
    # ... and each part at its smallest, on a chip of four CUs: 64 x 64 alone, with four groups, 128 x 128; rows at odd bytes and on words
    for m, k, oc in FC_TILE_PARTS:
        case = ConvCase(abi.FMT_NCHW, abi.DENSE, m, k, 1, 1, oc, 1, 1, 0, abi.RELU, scales=(0.01, 0.01, 0.1))
        lines.append("fctile %d %d %d %d %d 4" % (m, k, oc, packed_bytes(case), k & 1))
    # qsi8 layers without staging, and channel-wise + pointwise pairs: the shapes of their GPU tests
    for case in gp.GATHER:
        if case.n * case.oh * case.ow <= 6000:
            lines.append("gather %d %d %d %d %d %d %d %d %d %d %d" % (case.n, case.ic, case.ih, case.iw, case.oc, case.fh, case.sh,
                                                                     case.ph, case.dh, int(case.bias), packed_bytes(case)))
    import test_dw_pw
    for n, c, oc, h, w, s, act, _ in test_dw_pw.PAIRS:
        n = min(n, 3)
        if n * c * h * w <= 1 << 19:
            pw = ConvCase(abi.FMT_NCHW44, abi.DENSE, n, c, (h - 1) // s + 1, (w - 1) // s + 1, oc, 1, 1, 0, act, scales=(0.01, 0.01, 0.1))
            lines.append("dwpw %d %d %d %d %d %d %d %d" % (n, c, oc, h, w, s, (h + w) & 1, packed_bytes(pw)))
    # pointwise layers, on a chip small enough that the shared form and several tiles a wave are among them; with a stride the shapes
    # of their GPU test with fewer images, without one channels and pixels off every tile
    for case in gp.STRIDED_1X1_IN_PLACE:
        n = min(case.n, 8)
        if n * case.oh * case.ow >= 32 and case.ic * case.ih * case.iw <= 1 << 18:
            lines.append("pw %d %d %d %d %d %d %d %d 8" % (n, case.ic, case.ih, case.iw, case.oc, case.sh, int(case.bias), packed_bytes(case)))
    for n, ic, h, w, oc in ((1, 32, 6, 7, 64), (2, 20, 13, 5, 36), (1, 68, 8, 4, 100), (3, 256, 7, 7, 64), (1, 512, 9, 9, 32), (2, 1024, 5, 4, 64), (1, 136, 9, 7, 44),
                            (4, 512, 11, 7, 128), (1, 384, 9, 7, 64), (3, 260, 8, 5, 36)):
        case = ConvCase(abi.FMT_NCHW44, abi.DENSE, n, ic, h, w, oc, 1, 1, 0, abi.RELU, scales=(0.01, 0.01, 0.1))
        lines.append("pw %d %d %d %d %d 1 %d %d 4" % (n, ic, h, w, oc, h & 1, packed_bytes(case)))
    # the head of a network in one kernel: the shapes of its GPU test, as one strip an image and as several
    import test_stem
    for n, oh, ow, oc, act, bias, _ in test_stem.CASES:
        pw = ConvCase(abi.FMT_NCHW44, abi.DENSE, min(n, 3), 32, oh, ow, oc, 1, 1, 0, act, scales=(0.01, 0.01, 0.1))
        for cus in (1, 16):
            lines.append("stem %d %d %d %d %d %d %d %d" % (min(n, 3), oh, ow, oc, int(act == abi.RELU), int(bias), packed_bytes(pw), cus))
    # qsi8 FullyConnected: 1..64 rows, K = 1..32 blocks of 128 (and beyond 4096), channel counts off every tile size
    for i in range(24):
        m = int(r.choice([1, 2, 3, 4, 5, 31, 32, 33, 63, 64]))
        k = int(r.choice([128, 256, 384, 512, 1024, 2048, 4096, 4224, 8192])) if m > 4 else int(r.choice([1, 31, 32, 33, 100, 1024, 4095]))
        oc = int(r.choice([1, 3, 31, 32, 33, 63, 64, 65, 255, 256, 257, 1000]))
        case = ConvCase(abi.FMT_NCHW, abi.DENSE, m, k, 1, 1, oc, 1, 1, 0, abi.RELU, scales=(0.01, 0.01, 0.1),
                        bias=bool(r.integers(0, 2)))
        lines.append(line_of(case))
    return lines


def test_every_load_and_store_of_the_clamped_kernels_stays_inside_its_tensor(audit_exe):
    lines = audit_lines()
    assert len(lines) > 150
    r = subprocess.run([audit_exe], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=1500)
    assert r.returncode == 0, "bounds audit failed:\n%s\n%s" % (r.stdout[-1500:], r.stderr[-3000:])
    assert "audited %d cases" % len(lines) in r.stdout
    ran = {line.split(" -> ")[1] for line in r.stdout.splitlines() if " -> " in line}
    for kernel in ("fc_tile:32,4", "fc_tile:64,1", "fc_tile:64,4", "fc_tile:128,1", "conv_pw_share:16,-1", "conv_pw_stream:1,0",
                   "gemm_f32_ks_split:64,256", "gemm_f32_ks_split:64,128", "gemm_f32_ks_split:64,64", "conv_f32_wide:16,32", "conv_f32_wide:32,32",
                   "conv_f32_wide:64,32", "conv_blocks:256,3", "conv_blocks:512,5", "conv_pw_stream:8,1", "conv_pw_stream:12,0", "conv_pw_stream:12,1", "conv_pw_stream:32,0", "conv_stem:64,1", "conv_stem:32,1", "conv_stem:64,14"):
        assert kernel in ran, (kernel, sorted(ran))


def test_which_runs_of_blocks_are_asked_for(audit_exe):
    """images for two fifths of the CUs with 512 channels, a fifth with 256 (host code of the library)"""
    ask = {"102 512 14 14 256": 0, "103 512 14 14 256": 1, "103 512 14 15 256": 1, "103 512 15 14 256": 0, "103 512 14 16 256": 0, "51 256 14 14 256": 0,
           "52 256 14 14 256": 1, "52 512 14 14 256": 0, "200 384 14 14 256": 0, "200 128 14 14 256": 0, "52 512 7 7 128": 1, "1 256 1 1 5": 1, "1 512 1 1 5": 0}
    r = subprocess.run([audit_exe], input="".join("asked %s\n" % a for a in ask), capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr[-500:]
    assert r.stdout.splitlines()[:-1] == ["ok asked %s -> conv_blocks_takes:%d,0" % a for a in ask.items()]


def test_the_audit_sees_the_out_of_bounds_read_a_missing_clamp_causes(audit_exe, tmp_path):
    """the audit itself, pinned by a mutation: without the clamp of the gather's column the surplus
    columns of a ragged last pixel tile read up to one image past the tensor; the audit must die on it"""
    src = open(os.path.join(CSRC, "gemm_f32.hip")).read()
    clamp = "const int cn = min(n0 + tid % BN, q.N - 1);"
    assert src.count(clamp) == 1
    mutated = tmp_path / "gemm_f32.hip"
    mutated.write_text(src.replace(clamp, "const int cn = n0 + tid % BN;"))
    exe = compile_audit(str(tmp_path / "build"), replace={"gemm_f32": str(mutated)}, have=os.path.dirname(audit_exe))
    r = subprocess.run([exe], input="conv 3 86 45 42 117 5 2 3 1 1 1\n", capture_output=True, text=True, timeout=300)
    assert r.returncode == 3 and "OUT OF BOUNDS" in r.stderr, (r.returncode, r.stderr[-500:])


@pytest.mark.parametrize("line", ["fctile 65 129 67 65536 0 256", "fctile 130 65 150 65536 0 4", "fctile 100 2049 101 1048576 1 4",
                                  "fctile 130 2049 129 1048576 1 4"])
def test_the_audit_sees_a_row_read_past_the_end_of_its_tensor(audit_exe, tmp_path_factory, line):
    """likewise for loads at any byte, in every part: without the step back to the tensor's last 16 bytes"""
    if not _no_clamp:
        src = open(os.path.join(CSRC, "fc_tile.hip")).read()
        clamp = "min(roff[i] + b, q.last16)"
        assert src.count(clamp) == 1
        folder = tmp_path_factory.mktemp("no_clamp")
        mutated = folder / "fc_tile.hip"
        mutated.write_text(src.replace(clamp, "(roff[i] + b)"))
        _no_clamp.append(compile_audit(str(folder / "build"), replace={"fc_tile": str(mutated)}, have=os.path.dirname(audit_exe)))
    r = subprocess.run([_no_clamp[0]], input=line + "\n", capture_output=True, text=True, timeout=300)
    assert r.returncode == 3 and "OUT OF BOUNDS" in r.stderr, (r.returncode, r.stderr[-500:])


@pytest.mark.parametrize("source,was,by,line", [
    # pixels beyond the last one; the result's rows below an odd last one (both also without the buffer's own range check)
    ("conv_pw_stream", "return tile < tend && p < q.P", "return true || (tile < tend && p < q.P)", "pw 3 20 13 11 36 2 0 65536 8"),
    ("conv_stem", "there && 2 * t + row < q.oh ?", "there ?", "stem 1 7 12 32 0 0 32768 1"),
])
def test_the_audit_sees_a_missing_range_test(audit_exe, tmp_path, source, was, by, line):
    src = open(os.path.join(CSRC, source + ".hip")).read()
    assert was in src
    mutated = tmp_path / (source + ".hip")
    mutated.write_text(src.replace(was, by).replace("make_buffer_rsrc((void*)q.src, 0, q.src_bytes", "make_buffer_rsrc((void*)q.src, 0, 0x7fffffff")
                       .replace("make_buffer_rsrc((void*)q.dst, 0, q.dst_bytes", "make_buffer_rsrc((void*)q.dst, 0, 0x7fffffff"))
    exe = compile_audit(str(tmp_path / "build"), replace={source: str(mutated)}, have=os.path.dirname(audit_exe))
    r = subprocess.run([exe], input=line + "\n", capture_output=True, text=True, timeout=300)
    assert r.returncode == 3 and "OUT OF BOUNDS" in r.stderr, (r.returncode, r.stderr[-500:])


@pytest.mark.parametrize("source,was,by,line,what", [
    # a row behind the operand's last; a channel behind the last, stored and of the filter; one value more of a stage in LDS than there is room for; a
    # layer's last parameter behind the LDS that was asked for
    ("gemm_f32_ks_split", "min(r, s.rows - 1)", "r", "ksplit 70 128 130 0 0 0 0 0 1 1 0", "OUT OF BOUNDS: load"),
    ("conv_f32_wide", "if (there && m0 + row + e < q.M)", "if (there)", "wide 1 4 5 7 3 1 1 0 1 1 1", "OUT OF BOUNDS: access"),
    ("conv_f32_wide", "min(m0 + i * R + c, q.M - 1)", "(m0 + i * R + c)", "wide 1 16 5 7 3 1 1 0 1 1 1", "OUT OF BOUNDS: load"),
    ("gemm_f32_ks_split", "lds[4 * KP_STAGE > MEET ? 4 * KP_STAGE : MEET]", "lds[4 * KP_STAGE - 32]", "ksplit 64 256 64 0 1 0 0 0 1 1 0", "AddressSanitizer"),
    ("conv_blocks", "BYTES = MAP + 2 * LAYER * 4;", "BYTES = MAP + 2 * LAYER * 4 - 16;", "blocks 1 256 3 5 2 1", "AddressSanitizer"),
])
def test_the_audit_sees_an_access_beyond_a_buffer_or_the_lds(audit_exe, tmp_path, source, was, by, line, what):
    src = open(os.path.join(CSRC, source + ".hip")).read()
    assert src.count(was) == 1
    mutated = tmp_path / (source + ".hip")
    mutated.write_text(src.replace(was, by))
    exe = compile_audit(str(tmp_path / "build"), replace={source: str(mutated)}, have=os.path.dirname(audit_exe))
    r = subprocess.run([exe], input=line + "\n", capture_output=True, text=True, timeout=300)
    assert r.returncode != 0 and what in r.stderr, (r.returncode, r.stderr[-500:])


_no_clamp = []
