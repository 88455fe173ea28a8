"""A channel-wise 3x3 convolution and the pointwise 1x1 convolution of its result as one kernel (the model
runtime's conv_dw_pw), against the oracle's two convolutions run one after the other, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from cases import ConvCase
from megcc_amd import abi, runtime
from megcc_amd import abi as A
from oracle import port

pytestmark = pytest.mark.gpu

TIES = (0.02, 0.01, 0.05)            # exact ties: both layers requantise by the reference's own sequence
GENERIC = (0.0213, 0.0097, 0.0371)

PAIRS = [
    # (n, c, oc, h, w, stride, pointwise act, scales): every channel count with a kernel of its own at the extents of
    # MobileNets, then rows whose last group of 4 pixels hangs over by 1, 2, 3, tiles that cross images, fewer
    # pixels than a tile, one row, output channels that leave part of the last slice empty
    (1, 32, 64, 112, 112, 1, A.RELU, GENERIC), (1, 64, 128, 112, 112, 2, A.RELU, TIES),
    (2, 128, 128, 56, 56, 1, A.RELU, GENERIC), (2, 128, 256, 56, 56, 2, A.RELU, GENERIC),
    (3, 256, 256, 28, 28, 1, A.RELU, TIES), (3, 256, 512, 28, 28, 2, A.RELU, GENERIC),
    (5, 512, 512, 14, 14, 1, A.RELU, GENERIC), (5, 512, 1024, 14, 14, 2, A.RELU, TIES),
    (7, 1024, 1024, 7, 7, 1, A.RELU, GENERIC), (64, 512, 512, 14, 14, 1, A.RELU, GENERIC),
    (2, 32, 64, 9, 5, 1, A.IDENTITY, TIES), (2, 32, 96, 6, 13, 2, A.RELU, GENERIC), (3, 64, 160, 5, 7, 1, A.RELU, GENERIC),
    (3, 64, 32, 7, 6, 2, A.IDENTITY, GENERIC), (1, 128, 64, 1, 3, 1, A.RELU, TIES), (2, 128, 160, 11, 9, 2, A.RELU, GENERIC),
    (1, 256, 96, 2, 2, 1, A.IDENTITY, GENERIC), (2, 256, 320, 10, 15, 2, A.RELU, TIES), (1, 512, 544, 3, 31, 1, A.RELU, GENERIC),
    (1, 1024, 64, 4, 5, 2, A.RELU, TIES), (1, 1024, 1056, 5, 6, 1, A.IDENTITY, GENERIC), (40, 32, 64, 33, 17, 1, A.RELU, TIES),
]


@pytest.mark.parametrize("cfg", PAIRS, ids=lambda c: "n%d_c%d_oc%d_%dx%d_s%d_a%d_%s" % (c[:7] + ("ties" if c[7] is TIES else "gen",)))
def test_pair_in_one_kernel(cfg):
    n, c, oc, h, w, stride, act, scales = cfg
    port.set_threads(8)
    dw = ConvCase(A.FMT_NCHW44, A.GROUP, n, c, h, w, c, 3, stride, 1, A.RELU, scales=scales, flt_range=(-30, 30))
    s2 = (scales[2], scales[1], scales[2] if scales is TIES else scales[2] * scales[1] * 4.0e3 * c ** 0.5 / 36.0)
    pw = ConvCase(A.FMT_NCHW44, A.DENSE, n, c, dw.oh, dw.ow, oc, 1, 1, 0, act, scales=s2)
    a0, a1 = dw.gen(51), pw.gen(52)
    a1["src"] = dw.run_port(a0)
    want = pw.run_port(a1)
    assert len(np.unique(want)) > 20
    bias_scale = lambda k: float(np.float32(k.scales[0]) * np.float32(k.scales[1]))
    for fused in (True, False):
        runtime.set_option("fusedwpw", int(fused))
        runtime.set_option("nofusedwpw", int(not fused))
        try:
            m = runtime.Model()
            x = m.tensor("x", dw.src_shape(), abi.QINT8, dw.scales[0])
            m.mark_input(x)
            t = x
            for k, case, arrays in (("dw", dw, a0), ("pw", pw, a1)):
                y = m.tensor(k, case.dst_shape(), abi.QINT8, case.scales[2])
                m.opr(case.symbol(), [t, m.weight(k + ".w", arrays["flt"], abi.QINT8, case.scales[1]),
                                      m.weight(k + ".b", arrays["bias"], abi.QINT32, bias_scale(case))], [y])
                t = y
            m.mark_output(t)
            m.finalize()
        finally:
            runtime.set_option("fusedwpw", 0)
            runtime.set_option("nofusedwpw", 0)
        assert m.nr_kernel == (1 if fused else 2)
        m.set_input(x, a0["src"])
        for _ in range(2):
            m.forward()
        got = m.get(t)
        print(runtime.last_kernel())
        assert runtime.last_kernel().startswith("conv_dw_pw") == fused, runtime.last_kernel()
        bad = int((got != want).sum())
        assert bad == 0, "%s: %d of %d differ" % ("one kernel" if fused else "two kernels", bad, got.size)
        m.close()


def _block(c, oc, n=3, h=20, w=18, pairs=2):
    """`pairs` channel-wise + pointwise pairs behind an operator, all tensors in the arena but the first and the last:
    (model, ids of its tensors in order, the oracle's results in order, lifetimes (begin, end, bytes) of the arena's)"""
    from cases import MultiTypeCase
    bias_scale = lambda k: float(np.float32(k.scales[0]) * np.float32(k.scales[1]))
    pre = MultiTypeCase(A.Q_RELU, (n, c // 4, h, w, 4), (0.03, 0.01, GENERIC[0]))
    x0 = np.random.default_rng(61).integers(-128, 128, pre.shape).astype(np.int8)
    m = runtime.Model()
    ids, want = [m.tensor("x0", pre.shape, abi.QINT8, 0.03)], [x0]
    m.mark_input(ids[0])
    ids.append(m.tensor("x", pre.shape, abi.QINT8, GENERIC[0]))
    want.append(pre.run_port({"a": x0, "b": None}))
    m.opr(pre.symbol(), [ids[0]], [ids[1]])
    scale = GENERIC[0]
    for p in range(pairs):
        dw = ConvCase(A.FMT_NCHW44, A.GROUP, n, c, h, w, c, 3, 1, 1, A.RELU, scales=(scale,) + GENERIC[1:], flt_range=(-30, 30))
        pw = ConvCase(A.FMT_NCHW44, A.DENSE, n, c, h, w, oc, 1, 1, 0, A.RELU, scales=(GENERIC[2], GENERIC[1], GENERIC[2] * 5))
        for case in (dw, pw):
            arrays = case.gen(70 + len(ids))
            arrays["src"] = want[-1]
            want.append(case.run_port(arrays))
            name = "t%d" % len(ids)
            ids.append(m.tensor(name, case.dst_shape(), abi.QINT8, case.scales[2]))
            m.opr(case.symbol(), [ids[-2], m.weight(name + ".w", arrays["flt"], abi.QINT8, case.scales[1]),
                                  m.weight(name + ".b", arrays["bias"], abi.QINT32, bias_scale(case))], [ids[-1]])
        scale, c = pw.scales[2], oc
    m.mark_output(ids[-1])
    bytes_of = [int(np.prod(t.shape)) for t in want]
    last = len(ids) - 2
    life = [(k - 1, k + 1, bytes_of[k]) for k in range(1, len(ids) - 1)] + [(last, last + 2, bytes_of[-1])]
    return m, ids, want, life


def _planned(life):
    _, arena, _ = runtime.plan_memory(*[[r[k] for r in life] for k in (0, 1, 2)], 256)
    return int(arena)


def test_a_pair_the_kernel_does_not_take_costs_no_memory():
    """24 channels: no kernel of its own. The arena is that of the operators as they are"""
    m, ids, want, life = _block(24, 24)
    m.finalize()
    assert m.nr_kernel == 5
    assert m.arena_bytes == _planned(life)
    m.set_input(ids[0], want[0])
    m.forward()
    assert np.array_equal(m.get(ids[-1]), want[-1])
    m.close()


@pytest.mark.parametrize("switch", ["fusedwpw", "nofusedwpw", None])
def test_the_tensor_inside_a_pair_is_planned_for_operators_run_one_by_one(switch):
    """as one kernel the pair needs no memory for the tensor in between; operators run one by one get one place for all
    of them, and forwards before and behind are as they were"""
    m, ids, want, life = _block(64, 64)
    if switch:
        runtime.set_option(switch, 1)
    try:
        m.finalize()
    finally:
        if switch:
            runtime.set_option(switch, 0)
    kernels = m.nr_kernel
    if switch:
        assert kernels == (3 if switch == "fusedwpw" else 5)
    up = lambda v: (v + 255) // 256 * 256
    if kernels == 3:  # sources and results of the pairs (one operator longer), one tensor in between
        ends = [(b, e + 1, s) for b, e, s in life[0:-1:2]] + [life[-1]]
        assert m.arena_bytes == up(_planned(ends)) + up(max(s for _, _, s in life[1:-1:2]))
    elif kernels == 5:
        assert m.arena_bytes == _planned(life)
    for _ in range(2):
        m.set_input(ids[0], want[0])
        m.forward()
        assert np.array_equal(m.get(ids[-1]), want[-1])
        for k in range(len(ids) - 1):
            m.run_opr(k)
            assert np.array_equal(m.get(ids[k + 1]), want[k + 1]), k
    m.close()


@pytest.mark.parametrize("graph", [True, False])
def test_the_requantisation_is_switched_between_forwards(graph):
    """the switch "noaffine" changes what a pair is launched with: at the forward that is captured, between replays and
    between plain launches, every forward runs and gives the oracle's result"""
    m, ids, want, _ = _block(64, 64, pairs=4)
    runtime.set_option("fusedwpw", 1)
    try:
        m.finalize()
    finally:
        runtime.set_option("fusedwpw", 0)
    assert m.nr_kernel == 5  # (the fewest a forward is captured with)
    m.set_input(ids[0], want[0])
    runtime.set_option("no_graph", int(not graph))
    try:
        for k in range(1, 15):
            runtime.set_option("noaffine", int(k in (1, 4, 6, 7, 11, 13)))
            m.forward()
            # (a replayed graph launches nothing of its own; the pair's layers have multiply-adds for these scales)
            if not graph:
                assert runtime.last_kernel().endswith("+affine") == (k not in (1, 4, 6, 7, 11, 13)), k
            if k != 2:  # (forwards 2 and 3 are timed as a pair, one behind the other)
                assert np.array_equal(m.get(ids[-1]), want[-1]), k
        assert m.launch_mode()[0] == -1 or (graph and m.launch_mode()[0] == 1)
    finally:
        runtime.set_option("noaffine", 0)
        runtime.set_option("no_graph", 0)
    m.close()


class _Pack(C.Structure):
    _fields_ = [("s1", C.c_float), ("s2", C.c_float), ("c", C.c_float), ("d", C.c_float), ("mode", C.c_int)]


def starts_as_floats(act, scales):
    """whether sums of that layer start as floats (epilogue.h, mode 5): the library's own answer"""
    f = runtime.lib()._ZN2mg19requant_shifted_forEifff
    f.argtypes, f.restype = [C.c_int] + [C.c_float] * 3, _Pack
    return f(act, *scales).mode == 5


def swept_biases(channels, values, ratio, lowest):
    """`values` consecutive sums a channel, from 24 outputs below `lowest` to 24 above 127; the channels at the ends, which
    saturate, far beyond 2^22 and 2^29"""
    bias = int(np.floor((lowest - 24) / ratio)) + values * np.arange(channels, dtype=np.int64)
    bias[[0, -1, -2]] = [-(2 ** 30), 2 ** 30, 2 ** 22 + 3]
    return bias.astype(np.int32)


PASS = (0.5, 1.0, 0.5)  # scales of a layer whose outputs are its sums


@pytest.mark.parametrize("noaffine", [0, 1])
@pytest.mark.parametrize("swept,act", [("dw", A.RELU), ("pw", A.RELU), ("pw", A.IDENTITY)])
@pytest.mark.parametrize("c", [32, 64, 128, 512])
def test_every_sum_between_the_lowest_and_the_highest_output(c, swept, act, noaffine):
    """one layer passes its source on, the other's sums are all whole numbers over the whole range of its outputs: both sides of every
    step, for sums that start as floats and (noaffine) for those that do not"""
    values = 256 if swept == "dw" else 128
    lowest = -128 if act == A.IDENTITY and swept == "pw" else 0
    ratio = (127 - lowest + 48) / (c * values)
    scales = (0.0131, 0.0097, 0.0131 * 0.0097 / ratio)
    if swept == "pw":
        scales = (PASS[2], 0.0097, PASS[2] * 0.0097 / ratio)
    dw = ConvCase(A.FMT_NCHW44, A.GROUP, 1, c, 16, values // 16, c, 3, 1, 1, A.RELU, scales=scales if swept == "dw" else PASS)
    s2 = scales if swept == "pw" else (scales[2], 1.0, scales[2])
    pw = ConvCase(A.FMT_NCHW44, A.DENSE, 1, c, 16, values // 16, c, 1, 1, 0, act, scales=s2)
    assert starts_as_floats(act if swept == "pw" else A.RELU, scales)
    a0, a1 = dw.gen(1), pw.gen(2)
    x = np.arange(values) - (128 if swept == "dw" else 0)
    a0["src"] = np.broadcast_to(x.astype(np.int8).reshape(1, 1, 16, values // 16, 1), a0["src"].shape).copy()
    a0["flt"][...] = 0
    a0["flt"].reshape(c // 4, 9, 4)[:, 4] = 1
    a1["flt"][...] = 0
    w = a1["flt"].reshape(c // 4, c // 4, 4, 4)  # [output group][input group][input][output]
    for k in range(4):
        w[np.arange(c // 4), np.arange(c // 4), k, k] = 1
    for arrays, mine in ((a0, swept == "dw"), (a1, swept == "pw")):
        arrays["bias"].reshape(-1)[...] = swept_biases(c, values, ratio, lowest) if mine else 0
    a1["src"] = dw.run_port(a0)
    want = pw.run_port(a1)
    assert set(np.unique(want)) == set(range(lowest, 128))
    bias_scale = lambda k: float(np.float32(k.scales[0]) * np.float32(k.scales[1]))
    m = runtime.Model()
    t = x = m.tensor("x", dw.src_shape(), abi.QINT8, dw.scales[0])
    m.mark_input(x)
    for k, case, arrays in (("dw", dw, a0), ("pw", pw, a1)):
        y = m.tensor(k, case.dst_shape(), abi.QINT8, case.scales[2])
        m.opr(case.symbol(), [t, m.weight(k + ".w", arrays["flt"], abi.QINT8, case.scales[1]),
                              m.weight(k + ".b", arrays["bias"], abi.QINT32, bias_scale(case))], [y])
        t = y
    m.mark_output(t)
    runtime.set_option("fusedwpw", 1)
    try:
        m.finalize()
    finally:
        runtime.set_option("fusedwpw", 0)
    assert m.nr_kernel == 1
    m.set_input(x, a0["src"])
    runtime.set_option("noaffine", noaffine)
    try:
        m.forward()
    finally:
        runtime.set_option("noaffine", 0)
    got = m.get(t)
    assert runtime.last_kernel().startswith("conv_dw_pw")
    bad = np.argwhere(got != want)
    assert bad.size == 0, "%d differ, first at %s: %d, expected %d" % (len(bad), bad[0], got[tuple(bad[0])], want[tuple(bad[0])])
    m.close()


def test_a_pair_with_ratios_near_a_millionth():
    """scales for which there are no multiply-adds but the reference's sequence is proven: the pair is one kernel like any other"""
    n, c, scales = 2, 64, (0.001, 0.001, 0.9)
    dw = ConvCase(A.FMT_NCHW44, A.GROUP, n, c, 9, 12, c, 3, 1, 1, A.RELU, scales=scales)
    pw = ConvCase(A.FMT_NCHW44, A.DENSE, n, c, 9, 12, c, 1, 1, 0, A.IDENTITY, scales=(0.9, 0.001, 0.9 * 0.001 / 9.0e-7))
    a0, a1 = dw.gen(5), pw.gen(6)
    for case, arrays, lowest in ((dw, a0, 0), (pw, a1, -128)):
        ratio = case.scales[0] * case.scales[1] / case.scales[2]
        arrays["bias"].reshape(-1)[...] = np.linspace((lowest - 2) / ratio, 129 / ratio, c).astype(np.int32)
    a1["src"] = dw.run_port(a0)
    want = pw.run_port(a1)
    bias_scale = lambda k: float(np.float32(k.scales[0]) * np.float32(k.scales[1]))
    m = runtime.Model()
    t = x = m.tensor("x", dw.src_shape(), abi.QINT8, dw.scales[0])
    m.mark_input(x)
    for k, case, arrays in (("dw", dw, a0), ("pw", pw, a1)):
        y = m.tensor(k, case.dst_shape(), abi.QINT8, case.scales[2])
        m.opr(case.symbol(), [t, m.weight(k + ".w", arrays["flt"], abi.QINT8, case.scales[1]),
                              m.weight(k + ".b", arrays["bias"], abi.QINT32, bias_scale(case))], [y])
        t = y
    m.mark_output(t)
    runtime.set_option("fusedwpw", 1)
    try:
        m.finalize()
    finally:
        runtime.set_option("fusedwpw", 0)
    assert m.nr_kernel == 1
    m.set_input(x, a0["src"])
    m.forward()
    assert np.array_equal(m.get(t), want)
    m.close()
