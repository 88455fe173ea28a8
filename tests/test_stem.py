"""The head of a quantised network - the f32 image's conversion to qsi8, the first 3x3 stride-2 convolution, the channel-wise 3x3
and the pointwise convolution behind it - as one kernel (model runtime), against the oracle operator by operator: bit for bit."""
import os
import re
import subprocess

import numpy as np
import pytest

from cases import ConvCase
from megcc_amd import abi, runtime
from test_dw_pw import starts_as_floats, swept_biases

CALIBRATED, TIES = (1.0 / 127, 0.0051, 0.037, 0.0047, 0.021, 0.0049, 0.043), (1.0 / 127, 0.01, 0.02, 0.01, 0.02, 0.01, 0.05)


def _layers(n, oh, ow, oc, act, bias, s):
    a = abi
    c0 = ConvCase(a.FMT_NCHW_NCHW44, a.DENSE, n, 3, 2 * oh, 2 * ow, 32, 3, 2, 1, a.RELU, scales=(s[0], s[1], s[2]), bias=bias)
    dw = ConvCase(a.FMT_NCHW44, a.GROUP, n, 32, oh, ow, 32, 3, 1, 1, a.RELU, scales=(s[2], s[3], s[4]), bias=bias)
    pw = ConvCase(a.FMT_NCHW44, a.DENSE, n, 32, oh, ow, oc, 1, 1, 0, act, scales=(s[4], s[5], s[6]), bias=bias)
    return c0, dw, pw


# one row and the narrowest rows, an odd number of rows, rows at and around 32-pixel places, the widest; more strips than
# one per image, several images a strip row apart; both numbers of output channels, both activations, no biases
CASES = [(1, 1, 4, 64, abi.RELU, True, CALIBRATED), (3, 7, 12, 32, abi.IDENTITY, False, CALIBRATED), (2, 2, 16, 64, abi.RELU, True, TIES),
         (5, 15, 36, 32, abi.RELU, True, CALIBRATED), (2, 33, 64, 64, abi.IDENTITY, True, TIES), (1, 112, 112, 64, abi.RELU, True, CALIBRATED),
         (70, 9, 60, 64, abi.RELU, False, CALIBRATED), (2, 40, 128, 64, abi.RELU, True, CALIBRATED), (300, 6, 20, 32, abi.RELU, True, TIES)]


@pytest.mark.gpu
@pytest.mark.parametrize("n,oh,ow,oc,act,bias,s", CASES)
def test_head_of_a_network_as_one_kernel(n, oh, ow, oc, act, bias, s):
    print("GPU case:", n, oh, ow, oc, act, bias, flush=True)
    layers = _layers(n, oh, ow, oc, act, bias, s)
    rng = np.random.default_rng(n * 1000 + oh)
    image = rng.uniform(-1.3, 1.3, (n, 3, 2 * oh, 2 * ow)).astype(np.float32)
    image.reshape(-1)[:4] = [np.float32(0.5 / 127), np.float32(-0.5 / 127), 1e9, -1e9]  # halves; beyond the range
    scaled = image * (np.float32(1) / np.float32(s[0]))
    x = np.clip(np.copysign(np.floor(np.abs(scaled.astype(np.float64)) + 0.5), scaled), -128, 127).astype(np.int8)
    m = runtime.Model()
    ids = [m.tensor("image", image.shape, abi.FLOAT), m.tensor("q", image.shape, abi.QINT8, s[0])]
    m.mark_input(ids[0])
    m.opr("GI_kernel_typecvt_f32qsi8", [ids[0]], [ids[1]])
    for k, case in enumerate(layers):
        arrays = case.gen(seed=31 + k)
        arrays["src"] = x
        if bias:
            arrays["bias"].reshape(-1)[:2] = [2 * 10**9, -2 * 10**9]
        x = case.run_port(arrays)
        weights = [m.weight("w%d" % k, arrays["flt"], abi.QINT8, case.scales[1])]
        if bias:
            weights.append(m.weight("b%d" % k, arrays["bias"], abi.QINT32, float(np.float32(case.scales[0]) * np.float32(case.scales[1]))))
        ids.append(m.tensor("y%d" % k, case.dst_shape(), abi.QINT8, case.scales[2]))
        m.opr(case.symbol(), [ids[-2]] + weights, [ids[-1]])
    m.mark_output(ids[-1])
    runtime.set_option("fusestem", 1)
    try:
        m.finalize()
    finally:
        runtime.set_option("fusestem", 0)
    assert m.nr_kernel == 1
    for noaffine in (0, 1):
        runtime.set_option("noaffine", noaffine)
        try:
            m.set_input(ids[0], image)
            m.forward()
            assert runtime.last_kernel().startswith("conv_stem"), runtime.last_kernel()
            got = m.get(ids[-1])
        finally:
            runtime.set_option("noaffine", 0)
        bad = np.argwhere(got != x)
        assert bad.size == 0, "%d differ, first at %s: %d, expected %d" % (len(bad), bad[0], got[tuple(bad[0])], x[tuple(bad[0])])
    for k in range(m.nr_opr):  # operators one by one find their tensors
        m.run_opr(k)
    assert np.array_equal(m.get(ids[-1]), x)
    m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("noaffine", [0, 1])
@pytest.mark.parametrize("swept,act", [("first", abi.RELU), ("dw", abi.RELU), ("pw", abi.RELU), ("pw", abi.IDENTITY)])
def test_every_sum_between_the_lowest_and_the_highest_output(swept, act, noaffine):
    """two of the three layers pass their source on, the third one's sums are all whole numbers over the whole range of its outputs, for
    sums that start as floats (epilogue.h, mode 5) and, noaffine, for those that do not"""
    oc = 64
    channels, values = (oc, 128) if swept == "pw" else (32, 256 if swept == "first" else 128)
    lowest = -128 if act == abi.IDENTITY else 0
    ratio = (127 - lowest + 48) / (channels * values)
    unit = 0.5
    s = [unit, 1.0, unit, 1.0, unit, 1.0, unit]  # (source, filter, result = next source, ...) of layers whose outputs are their sums
    layer = ["first", "dw", "pw"].index(swept)
    s[2 * layer + 1] = 0.0097
    out = float(np.float32(unit) * np.float32(0.0097)) / ratio
    s[2 * layer + 2:] = [out if k % 2 == 0 else 1.0 for k in range(2 * layer + 2, 7)]
    layers = _layers(1, 16, 16, oc, act, True, s)
    assert starts_as_floats(layers[layer].act, layers[layer].scales)
    q = np.zeros((1, 3, 32, 32), np.int8)
    x = np.arange(256) - 128 if swept == "first" else np.arange(256) % 128
    q[:, :, ::2, ::2] = x.reshape(16, 16).astype(np.int8)  # (the pixels under the filters' centres)
    image = q.astype(np.float32) * np.float32(unit)
    m = runtime.Model()
    ids = [m.tensor("image", image.shape, abi.FLOAT), m.tensor("q", image.shape, abi.QINT8, unit)]
    m.mark_input(ids[0])
    m.opr("GI_kernel_typecvt_f32qsi8", [ids[0]], [ids[1]])
    want = q
    for k, case in enumerate(layers):
        arrays = case.gen(seed=k)
        arrays["src"] = want
        f = arrays["flt"]
        f[...] = 0
        if k == 0:
            f[:, 1, 1, 0, :] = 1
        elif k == 1:
            f.reshape(8, 9, 4)[:, 4] = 1
        else:
            for o in range(oc // 4):
                for i in range(4):
                    f[o, o % 8, 0, 0, i, i] = 1
        arrays["bias"].reshape(-1)[...] = swept_biases(channels, values, ratio, lowest) if k == layer else 0
        want = case.run_port(arrays)
        weights = [m.weight("w%d" % k, f, abi.QINT8, case.scales[1]),
                   m.weight("b%d" % k, arrays["bias"], abi.QINT32, float(np.float32(case.scales[0]) * np.float32(case.scales[1])))]
        ids.append(m.tensor("y%d" % k, case.dst_shape(), abi.QINT8, case.scales[2]))
        m.opr(case.symbol(), [ids[-2]] + weights, [ids[-1]])
    assert set(np.unique(want)) == set(range(lowest, 128))
    m.mark_output(ids[-1])
    runtime.set_option("fusestem", 1)
    try:
        m.finalize()
    finally:
        runtime.set_option("fusestem", 0)
    assert m.nr_kernel == 1
    m.set_input(ids[0], image)
    runtime.set_option("noaffine", noaffine)
    try:
        m.forward()
    finally:
        runtime.set_option("noaffine", 0)
    got = m.get(ids[-1])
    assert runtime.last_kernel().startswith("conv_stem"), runtime.last_kernel()
    bad = np.argwhere(got != want)
    assert bad.size == 0, "%d differ, first at %s: %d, expected %d" % (len(bad), bad[0], got[tuple(bad[0])], want[tuple(bad[0])])
    m.close()


OBJECT = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "megcc_amd", "csrc", "build", "conv_stem.o")
LLVM = "/opt/rocm/llvm/bin"


@pytest.mark.skipif(not os.path.exists(OBJECT), reason="needs the object file of the build")
def test_three_products_between_a_short_product_and_the_long_one_behind_it(tmp_path):
    """the build's own code: a 16x16x64 product that adds to the sums of a 16x16x32 one has three others in between"""
    fat, code = str(tmp_path / "fat"), str(tmp_path / "code")
    subprocess.check_call([LLVM + "/llvm-objcopy", "--dump-section=.hip_fatbin=" + fat, OBJECT, str(tmp_path / "copy.o")])
    subprocess.check_call([LLVM + "/clang-offload-bundler", "--type=o", "--unbundle", "--input=" + fat, "--output=" + code,
                           "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"])
    text = subprocess.run([LLVM + "/llvm-objdump", "-d", code], capture_output=True, text=True, check=True).stdout
    pairs, near = 0, []
    for kernel in re.split(r"(?m)^[0-9a-f]+ <", text)[1:]:
        products = re.findall(r"(v_mfma_i32_\w+) (v\[\d+:\d+\]), [^,]+, [^,]+, (v\[\d+:\d+\]|-?\w+)", kernel)
        writer = {}
        for k, (name, out, add) in enumerate(products):
            if "16x16x64" in name and add in writer and "16x16x32" in products[writer[add]][0]:
                pairs += 1
                if k - writer[add] - 1 < 3:
                    near.append((kernel.split(">")[0], k))
            writer[out] = k
    assert pairs >= 8 * 4, pairs
    assert not near, near
