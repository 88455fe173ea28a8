"""Which kernel takes a layer does not depend on the requantisation's constants, and asking for them costs a lock and, for new scales, a
search: what decides on kernels does not ask. The library's own functions, with its num_cus() and requant_pack_for() replaced
by ones that need no device and count."""
import os
import subprocess

import pytest

import megcc_amd

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CLANG = "/opt/rocm/llvm/bin/clang++"
LIB = os.path.join(os.path.dirname(megcc_amd.__file__), "libmegcc_gfx950.so")

PROGRAM = r"""
#include <stdio.h>
#include "conv_mfma_i8.h"
namespace mg {
static int asked = 0;
int num_cus() { return 256; }
RequantPack requant_pack_for(int, float, float, float, bool) {
    ++asked;
    return {1.f, 1.f, 1.f, 0.f, 3};
}
bool conv_mfma_dma_config(const ConvGeom&, bool fc, int variant, bool b128_ok, PipeConfig*);
bool conv_dw_pw_supported(const ConvGeom& dw, const ConvGeom& pw, const void* src, const void* dst);
bool conv_stem_supported(const ConvGeom& c0, const ConvGeom& dw, const ConvGeom& pw, const void* image, const void* dst);
}
using namespace mg;
static ConvGeom layer(int n, int ic, int oc, int h, int w, int k, int s, int groups) {
    ConvGeom g = {};
    g.n = n, g.ic = ic, g.oc = oc, g.ih = h, g.iw = w, g.fh = g.fw = k, g.sh = g.sw = s, g.ph = g.pw = k / 2, g.dh = g.dw = 1;
    g.oh = (h - 1) / s + 1, g.ow = (w - 1) / s + 1, g.groups = groups, g.fmt = MEGCC_FMT_NCHW44, g.act = MEGCC_NONLINE_RELU;
    g.s_src = 0.02f, g.s_flt = 0.01f, g.s_dst = 0.05f;
    return g;
}
int main() {
    int taken = 0;
    for (int k : {1, 3, 5})
        for (int s : {1, 2})
            for (int c : {32, 128, 256})
                for (int variant = 0; variant < 10; ++variant)
                    for (int act : {MEGCC_NONLINE_IDENTITY, MEGCC_NONLINE_RELU, MEGCC_NONLINE_H_SWISH}) {
                        ConvGeom g = layer(4, c, c, 56, 56, k, s, 1);
                        g.act = (MegccNonline)act;
                        PipeConfig pc;
                        if (conv_mfma_dma_config(g, false, variant, true, &pc)) {
                            ++taken;
                            if (!pc.kernel || !pc.literal || pc.kernel == pc.literal)
                                return printf("variant %d: no two forms\n", variant), 1;
                        }
                    }
    const ConvGeom dw = layer(2, 32, 32, 112, 112, 3, 1, 32), pw = layer(2, 32, 64, 112, 112, 1, 1, 1);
    ConvGeom c0 = layer(2, 3, 32, 224, 224, 3, 2, 1);
    c0.fmt = MEGCC_FMT_NCHW_NCHW44;
    const bool pair = conv_dw_pw_supported(dw, pw, nullptr, nullptr), head = conv_stem_supported(c0, dw, pw, nullptr, nullptr);
    printf("variants %d pair %d head %d asked %d\n", taken, pair, head, asked);
    return 0;
}
"""


@pytest.mark.skipif(not os.path.exists(CLANG) or not os.path.exists(LIB), reason="needs ROCm's clang++ and the built library")
def test_the_choice_of_a_kernel_does_not_ask_for_constants(tmp_path):
    src, exe = tmp_path / "question.cpp", str(tmp_path / "question")
    src.write_text(PROGRAM)
    subprocess.check_call([CLANG, "-std=c++17", "-O1", "-Wno-unknown-attributes", "-ffp-contract=off", "-I" + os.path.join(HERE, "host_audit"),
                           "-I" + os.path.join(ROOT, "megcc_amd", "csrc"), "-I" + os.path.join(ROOT, "include"), str(src), "-o", exe, "-rdynamic",
                           LIB, "-Wl,-rpath," + os.path.dirname(LIB)])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    words = r.stdout.split()
    assert int(words[1]) > 50 and words[3] == "1" and words[5] == "1" and words[7] == "0", r.stdout
