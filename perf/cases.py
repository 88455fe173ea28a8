"""The work this library is used for, as cases that can be timed and compared.

A case is one of six kinds of call through the public entry points:

  net       a MobileNetV1-int8 forward through the model runtime (runtime.Model): the deployed network.
            "host": the image comes from and the probabilities go back to host memory, as in an
            application that classifies what it receives; otherwise both stay in HBM.
  conv      one qsi8 NCHW44 convolution with bias, activation and requantisation (megcc_gfx950_call), the
            operator nearly all arithmetic of a quantised network is in
  fc        one qsi8 FullyConnected: a 1x1 NCHW convolution on [M,K,1,1], as MegCC lowers it
  matmul    one f32 MatMul in any of its four transposes
  conv_f32  one f32 NCHW convolution with bias and ReLU
  chain     channel-wise 3x3 -> max-pool 2x2 -> add + ReLU through the model runtime, the memory-bound
            end of a quantised network

"calibrated": scales under which the activations use the int8 range, as a calibrated network's do; the
other scales are those of the benchmark's configurations, whose outputs mostly saturate.
"""
import ctypes as C
import math

import numpy as np
import torch

from megcc_amd import abi, runtime

_TORCH = {abi.FLOAT: torch.float32, abi.QINT8: torch.int8, abi.QINT32: torch.int32}
_NUMPY = {torch.float32: "<f4", torch.int8: "|i1", torch.int32: "<i4"}

# (stride of the channel-wise layer, output channels of the pointwise layer) of each block
_BLOCKS = [(1, 64), (2, 128), (1, 128), (2, 256), (1, 256), (2, 512), (1, 512), (1, 512), (1, 512), (1, 512),
           (1, 512), (2, 1024), (1, 1024)]
_IMAGE, _CLASSES = 224, 1000


def listed():
    return [
        # one image in, one set of probabilities out: the latency an application sees
        {"name": "net_b1_host", "kind": "net", "batch": 1, "host": True},
        # batched serving, and the largest batch of the configurations
        {"name": "net_b64", "kind": "net", "batch": 64, "host": False},
        {"name": "net_b256", "kind": "net", "batch": 256, "host": False},
        # 3x3 layers: one of a single image (latency), the largest of the configurations (arithmetic)
        {"name": "conv_n1_c256_28", "kind": "conv", "n": 1, "ic": 256, "oc": 256, "h": 28, "w": 28, "k": 3,
         "stride": 1, "act": "RELU", "calibrated": False},
        {"name": "conv_n32_c256_56", "kind": "conv", "n": 32, "ic": 256, "oc": 256, "h": 56, "w": 56, "k": 3,
         "stride": 1, "act": "RELU", "calibrated": False},
        # a down-sampling layer of a network whose images are not square and whose channels are no power of two
        {"name": "conv_n6_s2_ragged", "kind": "conv", "n": 6, "ic": 88, "oc": 148, "h": 57, "w": 43, "k": 3,
         "stride": 2, "act": "RELU", "calibrated": True},
        # the classifier of a batch of 64
        {"name": "fc_64x4096x4096", "kind": "fc", "m": 64, "k": 4096, "n": 4096, "calibrated": False},
        # f32 products: the same classifier, odd sizes with transposed operands, a square one bound by arithmetic
        {"name": "matmul_64x4096x4096", "kind": "matmul", "m": 64, "k": 4096, "n": 4096, "ta": False, "tb": False},
        {"name": "matmul_odd_nt", "kind": "matmul", "m": 197, "k": 771, "n": 1003, "ta": False, "tb": True},
        {"name": "matmul_4096", "kind": "matmul", "m": 4096, "k": 4096, "n": 4096, "ta": False, "tb": False},
        # one f32 layer of a single image
        {"name": "conv_f32_n1_c32_56", "kind": "conv_f32", "n": 1, "ic": 32, "oc": 32, "h": 56, "w": 56, "k": 3,
         "stride": 1},
        # the memory-bound chain at its largest
        {"name": "chain_n64_c512_112", "kind": "chain", "n": 64, "c": 512, "h": 112, "w": 112, "stride": 1,
         "calibrated": False},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["net", "conv", "conv", "fc", "matmul", "conv_f32", "chain"])
    while True:
        if kind == "net":
            batch = _log_int(rng, 1, 256)
            case = {"kind": kind, "batch": batch, "host": batch <= 8 and rng.random() < 0.5}
        elif kind == "conv":
            h = _log_int(rng, 7, 112)
            w = h if rng.random() < 0.5 else max(7, min(112, int(h * rng.uniform(0.6, 1.5))))
            case = {"kind": kind, "n": _log_int(rng, 1, 64), "ic": 4 * _log_int(rng, 4, 128),
                    "oc": 4 * _log_int(rng, 4, 128), "h": h, "w": w, "k": rng.choice([1, 1, 3, 3, 3, 5]),
                    "stride": rng.choice([1, 1, 2]), "act": rng.choice(["IDENTITY", "RELU", "RELU", "H_SWISH"]),
                    "calibrated": rng.random() < 0.75}
        elif kind == "fc":
            case = {"kind": kind, "m": _log_int(rng, 1, 4096), "k": _log_int(rng, 64, 4096),
                    "n": _log_int(rng, 10, 4096), "calibrated": rng.random() < 0.75}
        elif kind == "matmul":
            case = {"kind": kind, "m": _log_int(rng, 1, 4096), "k": _log_int(rng, 64, 4096),
                    "n": _log_int(rng, 16, 4096), "ta": rng.random() < 0.25, "tb": rng.random() < 0.5}
        elif kind == "conv_f32":
            h = _log_int(rng, 7, 112)
            case = {"kind": kind, "n": _log_int(rng, 1, 16), "ic": _log_int(rng, 3, 128),
                    "oc": _log_int(rng, 8, 128), "h": h, "w": h if rng.random() < 0.5 else _log_int(rng, 7, 112),
                    "k": rng.choice([1, 3, 3]), "stride": rng.choice([1, 1, 2])}
        else:
            h = _log_int(rng, 14, 112)
            case = {"kind": kind, "n": _log_int(rng, 1, 64), "c": 4 * _log_int(rng, 4, 128), "h": h, "w": h,
                    "stride": rng.choice([1, 2]), "calibrated": rng.random() < 0.75}
        # no more work than the largest listed case of the kind, and more than a launch
        w = work(case)
        most = {"conv": 1.2e11, "conv_f32": 2e10}.get(kind, math.inf)
        if w["flops"] <= most and w["bytes"] / 1e11 + w["flops"] / 3e13 >= 5e-6:
            return case


# ---- one operator through the kernel ABI ---------------------------------------------------------------

class _Operator:
    """An operator as the TinyNN VM holds it: device tensors, workspace, the weight the init protocol
    returned. `tensors`: (torch tensor, scale, name), inputs then the one output."""

    def __init__(self, symbol, tensors):
        lib = runtime.lib()
        self.desc = runtime.parse_symbol(symbol)
        self.keep = [t for t, _, _ in tensors]
        kinds = {v: k for k, v in _TORCH.items()}
        make = [abi.make_tensor(t.data_ptr(), t.shape, abi.QINT32 if t.dtype == torch.int32 else kinds[t.dtype],
                                scale, name) for t, scale, name in tensors]
        self.tensors, self.output, self.nr_input = make, tensors[-1][0], len(make) - 1
        ins = abi.tensor_array(make[:-1])
        size = C.c_size_t(0)
        runtime.check(lib.megcc_gfx950_call_workspace(self.desc, ins, self.nr_input, 1, size), "workspace")
        self.workspace = abi.Workspace()
        if size.value:
            scratch = torch.empty(size.value, dtype=torch.uint8, device="cuda")
            self.keep.append(scratch)
            self.workspace.ptr, self.workspace.size = scratch.data_ptr(), size.value
        count = C.c_int(0)
        runtime.check(lib.megcc_gfx950_call_init(self.desc, ins, self.nr_input, None, count, None), "init")
        if count.value:
            weight = abi.Tensor()
            runtime.check(lib.megcc_gfx950_call_init(self.desc, ins, self.nr_input, weight, None, None), "init")
            packed = torch.empty(weight.layout.dims[0], dtype=torch.int8, device="cuda")
            self.keep.append(packed)
            weight.ptr = packed.data_ptr()
            torch.cuda.synchronize()  # the library has a stream of its own
            runtime.check(lib.megcc_gfx950_call_init(self.desc, ins, self.nr_input, weight, count, None), "init")
            for i, t in enumerate(make[:-1]):
                if t.name == weight.name:
                    make[i] = weight
        self.ins, self.outs = abi.tensor_array(make[:-1]), abi.tensor_array(make[-1:])
        self.call = lib.megcc_gfx950_call
        torch.cuda.synchronize()

    def run(self):
        runtime.check(self.call(self.desc, self.ins, self.nr_input, self.outs, 1, self.workspace, None), "call")
        return self.output


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _int8(gen, *shape, low=-128):
    return torch.randint(low, 128, shape, dtype=torch.int8, device="cuda", generator=gen)


def _bias(gen, *shape):
    return torch.randint(-1000, 1001, shape, dtype=torch.int32, device="cuda", generator=gen)


def _uniform(gen, *shape, span=1.0):
    return torch.rand(shape, device="cuda", generator=gen).mul_(2 * span).sub_(span)


def _empty(dtype, *shape):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _out(h, k, stride):
    return (h + 2 * (k // 2) - k) // stride + 1


def _scales(case, seed, taps, config):
    """(source, filter, destination) scales: the configuration's, or calibrated ones - about 36 destination
    steps to a standard deviation of the sums, and no round numbers"""
    if not case["calibrated"]:
        return config
    r = np.random.default_rng([seed, 77])
    s, f = config[0] * r.uniform(0.8, 1.2), config[1] * r.uniform(0.8, 1.2)
    return s, f, s * f * 74.0 * 73.0 * math.sqrt(taps) / 36.0 * r.uniform(0.9, 1.1)


def _bias_scale(s, f):
    return float(np.float32(s) * np.float32(f))


def _conv(case, seed):
    g, n, ic, oc, k = _generator(seed), case["n"], case["ic"], case["oc"], case["k"]
    oh, ow = _out(case["h"], k, case["stride"]), _out(case["w"], k, case["stride"])
    s, f, d = _scales(case, seed, ic * k * k, (0.02, 0.01, 0.05))
    act = "" if case["act"] == "IDENTITY" else "_" + case["act"]
    symbol = "kernel_conv2d_%dx%d_NCHW44_DENSE_p%dx%d_s%dx%d_d1x1_qsi8qsi8qsi32qsi8_bias%s" % (
        k, k, k // 2, k // 2, case["stride"], case["stride"], act)
    return _Operator(symbol, [
        (_int8(g, n, ic // 4, case["h"], case["w"], 4), s, b"src"),
        (_int8(g, oc // 4, ic // 4, k, k, 4, 4, low=-127), f, b"flt"),
        (_bias(g, 1, oc // 4, 1, 1, 4), _bias_scale(s, f), b"bias"),
        (_empty(torch.int8, n, oc // 4, oh, ow, 4), d, b"dst")])


def _fc(case, seed):
    g, m, k, n = _generator(seed), case["m"], case["k"], case["n"]
    s, f, d = _scales(case, seed, k, (0.01, 0.01, 0.1))
    return _Operator("kernel_conv2d_1x1_NCHW_DENSE_p0x0_s1x1_d1x1_qsi8qsi8qsi32qsi8_bias", [
        (_int8(g, m, k, 1, 1), s, b"src"), (_int8(g, n, k, 1, 1, low=-127), f, b"flt"),
        (_bias(g, 1, n, 1, 1), _bias_scale(s, f), b"bias"), (_empty(torch.int8, m, n, 1, 1), d, b"dst")])


def _matmul(case, seed):
    g, m, k, n, ta, tb = _generator(seed), case["m"], case["k"], case["n"], case["ta"], case["tb"]
    name = "gevm" if m <= 4 and not ta else "fp32_matmul_4x12"
    return _Operator("GI_kernel_%s_%s%s" % (name, "t" if ta else "n", "t" if tb else "n"), [
        (_uniform(g, *((k, m) if ta else (m, k))), 1.0, b"a"), (_uniform(g, *((n, k) if tb else (k, n))), 1.0, b"b"),
        (_empty(torch.float32, m, n), 1.0, b"c")])


def _conv_f32(case, seed):
    g, n, ic, oc, k, s = _generator(seed), case["n"], case["ic"], case["oc"], case["k"], case["stride"]
    symbol = "GI_kernel_conv2d_im2col_%dx%d_NCHW_DENSE_p%dx%d_s%dx%d_d1x1_bias_RELUf32" % (k, k, k // 2, k // 2, s, s)
    return _Operator(symbol, [
        (_uniform(g, n, ic, case["h"], case["w"]), 1.0, b"src"), (_uniform(g, oc, ic, k, k), 1.0, b"flt"),
        (_uniform(g, 1, oc, 1, 1, span=0.1), 1.0, b"bias"),
        (_empty(torch.float32, n, oc, _out(case["h"], k, s), _out(case["w"], k, s)), 1.0, b"dst")])


# ---- models --------------------------------------------------------------------------------------------

class _Device:
    """a model's tensor as an array torch can look at; keeps the model, whose arena it is part of"""

    def __init__(self, model, tid):
        self.model = model
        shape, kind = model.shapes[tid]
        self.__cuda_array_interface__ = {
            "shape": shape, "typestr": _NUMPY[_TORCH[kind]], "version": 2,
            "data": (runtime.lib().megcc_gfx950_model_tensor_ptr(model.h, tid), False)}


def _view(model, tid):
    view = torch.as_tensor(_Device(model, tid), device="cuda")
    view.owner = model  # a caller may keep an output longer than the program's state
    return view


class _Forward:
    """forward passes with inputs and outputs resident in HBM"""

    def __init__(self, model, inputs, output):
        self.model = model
        for tid, value in inputs:
            _view(model, tid).copy_(value)
        self.output = _view(model, output)
        torch.cuda.synchronize()

    def run(self):
        self.model.forward()
        return self.output


class _HostForward:
    """one image batch in host memory to probabilities in host memory"""

    def __init__(self, model, image_id, image, output):
        self.model, self.image_id, self.image, self.out_id = model, image_id, image, output

    def run(self):
        self.model.set_input(self.image_id, self.image)
        self.model.forward()
        return self.model.get(self.out_id)


class _Quantised:
    """qsi8 layers of a model under construction; `rms`: of the current tensor's values, which the calibrated
    scales follow from"""

    def __init__(self, model, rng):
        self.model, self.rng, self.nr = model, rng, 0

    def conv(self, x, src_scale, rms, symbol, src_taps, flt_shape, bias_shape, dst_shape, dst_scale=None):
        sigma = math.sqrt(src_taps) * 73.0 * rms  # of the int32 sums
        flt_scale = self.rng.uniform(0.004, 0.006) if dst_scale is None else dst_scale * 36.0 / (sigma * src_scale)
        if dst_scale is None:
            dst_scale = src_scale * flt_scale * sigma / 40.0
        self.nr += 1
        m, r, name = self.model, self.rng, "l%d" % self.nr
        w = m.weight(name + ".w", r.integers(-127, 128, flt_shape, dtype=np.int8), abi.QINT8, flt_scale)
        b = m.weight(name + ".b", r.integers(-1000, 1001, bias_shape, dtype=np.int32), abi.QINT32,
                     _bias_scale(src_scale, flt_scale))
        y = m.tensor(name, dst_shape, abi.QINT8, dst_scale)
        m.opr(symbol, [x, w, b], [y])
        return y, dst_scale


def _net(case, seed):
    b, r = case["batch"], np.random.default_rng(seed)
    m = runtime.Model()
    image = m.tensor("image", (b, 3, _IMAGE, _IMAGE), abi.FLOAT)
    m.mark_input(image)
    scale = 1.0 / 127.0
    x = m.tensor("quantised", (b, 3, _IMAGE, _IMAGE), abi.QINT8, scale)
    m.opr("GI_kernel_typecvt_f32qsi8", [image], [x])
    q = _Quantised(m, r)
    name = "kernel_conv2d_%s_d1x1_qsi8qsi8qsi32qsi8_bias"
    hw, c, rms = _IMAGE // 2, 32, 28.0  # (of a ReLU's outputs with 40 steps to a standard deviation)
    x, scale = q.conv(x, scale, 73.0, name % "3x3_NCHW_NCHW44_DENSE_p1x1_s2x2" + "_RELU", 27, (c // 4, 3, 3, 3, 4),
                      (1, c // 4, 1, 1, 4), (b, c // 4, hw, hw, 4))
    for stride, oc in _BLOCKS:
        hw //= stride
        x, scale = q.conv(x, scale, rms, name % ("3x3_NCHW44_GROUP_p1x1_s%dx%d" % (stride, stride)) + "_RELU", 9,
                          (c // 4, 1, 1, 3, 3, 4), (1, c // 4, 1, 1, 4), (b, c // 4, hw, hw, 4))
        x, scale = q.conv(x, scale, rms, name % "1x1_NCHW44_DENSE_p0x0_s1x1" + "_RELU", c,
                          (oc // 4, c // 4, 1, 1, 4, 4), (1, oc // 4, 1, 1, 4), (b, oc // 4, hw, hw, 4))
        c = oc
    pooled = m.tensor("pooled", (b, c // 4, 1, 1, 4), abi.QINT8, scale)
    m.opr("GI_kernel_pooling_AVERAGE_NCHW44_p0x0_s%dx%d_w%dx%d_qsi8qsi8_qsi8qsi8_fallback" % (hw, hw, hw, hw), [x], [pooled])
    x = m.alias("flat", pooled, (b, c, 1, 1))
    x, scale = q.conv(x, scale, 17.0, name % "1x1_NCHW_DENSE_p0x0_s1x1", c, (_CLASSES, c, 1, 1), (1, _CLASSES, 1, 1),
                      (b, _CLASSES, 1, 1), dst_scale=0.05)
    f32 = {n: m.tensor(n, (b, w), abi.FLOAT) for n, w in (
        ("logits", _CLASSES), ("max", 1), ("sub", _CLASSES), ("exp", _CLASSES), ("sum", 1), ("softmax", _CLASSES))}
    for symbol, ins, out in (
            ("GI_kernel_typecvt_qsi8f32", [x], "logits"),
            ("kernel_reduce_MAX_DEFAULT_a1_f32f32", ["logits"], "max"),
            ("kernel_elementwise_SUB_f32f32f32", ["logits", "max"], "sub"),
            ("kernel_elementwise_EXP_f32f32", ["sub"], "exp"),
            ("kernel_reduce_SUM_DEFAULT_a1_f32f32", ["exp"], "sum"),
            ("kernel_elementwise_TRUE_DIV_f32f32f32", ["exp", "sum"], "softmax")):
        m.opr(symbol, [f32.get(i, i) for i in ins], [f32[out]])
    m.mark_output(f32["softmax"])
    m.finalize()
    if case["host"]:
        pixels = r.uniform(-1, 1, (b, 3, _IMAGE, _IMAGE)).astype(np.float32)
        return _HostForward(m, image, pixels, f32["softmax"])
    return _Forward(m, [(image, _uniform(_generator(seed), b, 3, _IMAGE, _IMAGE))], f32["softmax"])


def _chain(case, seed):
    n, c, h, w = case["n"], case["c"], case["h"], case["w"]
    oh, ow = _out(h, 3, case["stride"]), _out(w, 3, case["stride"])
    half = (n, c // 4, oh // 2, ow // 2, 4)
    s, f, d = _scales(case, seed, 9, (0.02, 0.01, 0.05))
    r, g = np.random.default_rng(seed), _generator(seed)
    m = runtime.Model()
    x = m.tensor("x", (n, c // 4, h, w, 4), abi.QINT8, s)
    other = m.tensor("other", half, abi.QINT8, 0.01)
    m.mark_input(x)
    m.mark_input(other)
    flt = m.weight("w", r.integers(-127, 128, (c // 4, 1, 1, 3, 3, 4), dtype=np.int8), abi.QINT8, f)
    bias = m.weight("b", r.integers(-1000, 1001, (1, c // 4, 1, 1, 4), dtype=np.int32), abi.QINT32, _bias_scale(s, f))
    conv = m.tensor("conv", (n, c // 4, oh, ow, 4), abi.QINT8, d)
    m.opr("kernel_conv2d_3x3_NCHW44_GROUP_p1x1_s%dx%d_d1x1_qsi8qsi8qsi32qsi8_bias_RELU" % (
        case["stride"], case["stride"]), [x, flt, bias], [conv])
    pool = m.tensor("pool", half, abi.QINT8, d)
    m.opr("GI_kernel_pooling_MAX_NCHW44_p0x0_s2x2_w2x2_qsi8qsi8_qsi8qsi8_fallback", [conv], [pool])
    out = m.tensor("out", half, abi.QINT8, d)
    m.opr("kernel_elementwise_multitype_QFUSE_ADD_RELU_qsi8qsi8qsi8", [pool, other], [out])
    m.mark_output(out)
    m.finalize()
    return _Forward(m, [(x, _int8(g, n, c // 4, h, w, 4)), (other, _int8(g, *half))], out)


_PREPARE = {"net": _net, "conv": _conv, "fc": _fc, "matmul": _matmul, "conv_f32": _conv_f32, "chain": _chain}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return state.run()


def work(case):
    kind = case["kind"]
    if kind == "net":
        weights, macs, c, hw = 0, 0, 3, _IMAGE // 2
        layers = [(27, 32, hw)]
        c = 32
        for stride, oc in _BLOCKS:
            hw //= stride
            layers += [(9, c, hw), (c, oc, hw)]
            c = oc
        for taps, oc, size in layers + [(c, _CLASSES, 1)]:
            weights += oc * (taps + 4)
            macs += oc * taps * size * size
        return {"bytes": weights + case["batch"] * 4 * (3 * _IMAGE * _IMAGE + _CLASSES),
                "flops": 2 * macs * case["batch"]}
    if kind in ("conv", "conv_f32"):
        size = 1 if kind == "conv" else 4
        pixels = case["n"] * _out(case["h"], case["k"], case["stride"]) * _out(case["w"], case["k"], case["stride"])
        taps = case["ic"] * case["k"] * case["k"]
        return {"bytes": size * (case["n"] * case["ic"] * case["h"] * case["w"] + case["oc"] * taps + case["oc"] * pixels) +
                4 * case["oc"], "flops": 2 * case["oc"] * taps * pixels}
    if kind == "chain":
        oh, ow = _out(case["h"], 3, case["stride"]), _out(case["w"], 3, case["stride"])
        planes, half = case["n"] * case["c"], (oh // 2) * (ow // 2)
        return {"bytes": planes * (case["h"] * case["w"] + 2 * half) + 13 * case["c"], "flops": planes * (18 * oh * ow + 6 * half)}
    m, k, n = case["m"], case["k"], case["n"]
    size = 1 if kind == "fc" else 4
    return {"bytes": size * (m * k + k * n + m * n) + (4 * n if kind == "fc" else 0), "flops": 2 * m * k * n}


def tolerance(case):
    # quantised results are whole numbers, the same for every implementation; f32 sums differ by their order
    if case["kind"] == "net":
        return {"rel": 1e-5}  # (soft-max of whole logits)
    return {"rel": 1e-5} if case["kind"] in ("matmul", "conv_f32") else "exact"
