"""The order of the matrix instructions in the build's own code of conv_dw_pw.hip (CPU: disassembles the object the
Makefile leaves behind). A 16x16x64 product that adds to the sums of a 16x16x32 one must have three other products
between the two; the compiler is free to move them unless it is told not to."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
OBJECT = os.path.join(os.path.dirname(HERE), "megcc_amd", "csrc", "build", "conv_dw_pw.o")
LLVM = "/opt/rocm/llvm/bin"

pytestmark = pytest.mark.skipif(not os.path.exists(OBJECT), reason="needs the object file of the build")


def test_three_products_between_a_short_product_and_the_long_one_behind_it(tmp_path):
    fat, code = str(tmp_path / "fat"), str(tmp_path / "code")
    subprocess.check_call([LLVM + "/llvm-objcopy", "--dump-section=.hip_fatbin=" + fat, OBJECT, str(tmp_path / "copy.o")])
    subprocess.check_call([LLVM + "/clang-offload-bundler", "--type=o", "--unbundle", "--input=" + fat, "--output=" + code,
                           "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"])
    text = subprocess.run([LLVM + "/llvm-objdump", "-d", code], capture_output=True, text=True, check=True).stdout
    pairs = 0
    near = []
    for kernel in re.split(r"(?m)^[0-9a-f]+ <", text)[1:]:
        products = re.findall(r"(v_mfma_i32_\w+) (v\[\d+:\d+\]), [^,]+, [^,]+, (v\[\d+:\d+\]|-?\w+)", kernel)
        writer = {}
        for k, (name, out, add) in enumerate(products):
            if "16x16x64" in name and add in writer and "16x16x32" in products[writer[add]][0]:
                pairs += 1
                if k - writer[add] - 1 < 3:
                    near.append((kernel.split(">")[0], k, k - writer[add] - 1))
            writer[out] = k
    assert pairs > 500, pairs
    assert not near, "%d of %d pairs: %s" % (len(near), pairs, near[:3])
