"""Runs of channel-wise 3x3 + pointwise 1x1 blocks that one workgroup an image keeps in LDS (the model runtime's conv_blocks),
against the oracle's convolutions run one after the other, bit for bit."""
import numpy as np
import pytest

from cases import ConvCase
from megcc_amd import abi, runtime
from megcc_amd import abi as A
from oracle import port

pytestmark = pytest.mark.gpu

TIES = (0.02, 0.01, 0.05)  # exact ties: both layers requantise by the reference's own sequence
GENERIC = (0.0213, 0.0097, 0.0371)

RUNS = [
    # (n, c, h, w, blocks, scales): a MobileNet's; the largest map; odd numbers of rows and slots; fewer rows than a part; one row,
    # one column, one pixel; more images than there are CUs; parts that have no rows at all
    (3, 512, 14, 14, 5, GENERIC), (2, 512, 14, 14, 2, TIES), (2, 512, 14, 15, 3, GENERIC), (3, 256, 13, 15, 3, GENERIC),
    (2, 256, 14, 15, 2, TIES), (2, 512, 7, 7, 2, GENERIC), (2, 256, 1, 15, 2, GENERIC), (2, 512, 14, 1, 2, GENERIC),
    (5, 256, 1, 1, 4, GENERIC), (300, 256, 3, 5, 2, GENERIC), (2, 512, 9, 11, 2, GENERIC),
]


def _run(cfg, seed=0):
    """(model under construction, its source, the oracle's result, the last tensor)"""
    n, c, h, w, blocks, scales = cfg
    m = runtime.Model()
    x = t = m.tensor("x", (n, c // 4, h, w, 4), abi.QINT8, scales[0])
    m.mark_input(x)
    src = want = np.random.default_rng(seed + 1).integers(-128, 128, (n, c // 4, h, w, 4)).astype(np.int8)
    s = scales[0]
    for b in range(blocks):
        # (sums of 9 and of c products that use the int8 range)
        mid = scales[2] if scales is TIES else s * scales[1] * 1.1e3 / 36.0
        out = scales[2] if scales is TIES else mid * scales[1] * 2.0e3 * c ** 0.5 / 36.0
        dw = ConvCase(A.FMT_NCHW44, A.GROUP, n, c, h, w, c, 3, 1, 1, A.RELU, scales=(s, scales[1], mid), flt_range=(-30, 30))
        pw = ConvCase(A.FMT_NCHW44, A.DENSE, n, c, h, w, c, 1, 1, 0, A.RELU, scales=(mid, scales[1], out))
        for k, case in (("dw", dw), ("pw", pw)):
            arrays = case.gen(seed + 10 * b + (k == "pw"))
            arrays["src"] = want
            want = case.run_port(arrays)
            name = "%s%d" % (k, b)
            y = m.tensor(name, case.dst_shape(), abi.QINT8, case.scales[2])
            m.opr(case.symbol(), [t, m.weight(name + ".w", arrays["flt"], abi.QINT8, case.scales[1]),
                                  m.weight(name + ".b", arrays["bias"], abi.QINT32,
                                           float(np.float32(case.scales[0]) * np.float32(case.scales[1])))], [y])
            t = y
        s = out
    m.mark_output(t)
    return m, x, src, want, t


@pytest.mark.parametrize("cfg", RUNS, ids=lambda c: "n%d_c%d_%dx%d_b%d_%s" % (c[:5] + ("ties" if c[5] is TIES else "gen",)))
def test_run_of_blocks_in_one_kernel(cfg):
    port.set_threads(8)
    m, x, src, want, t = _run(cfg)
    assert cfg[2] * cfg[3] < 4 or len(np.unique(want)) > 20
    for switch in ("fusedwpw", "fuseblocks"):
        runtime.set_option(switch, 1)
    try:
        m.finalize()
    finally:
        for switch in ("fusedwpw", "fuseblocks"):
            runtime.set_option(switch, 0)
    assert m.nr_kernel == 1
    m.set_input(x, src)
    for affine in (True, False):
        runtime.set_option("noaffine", int(not affine))
        try:
            for _ in range(2):
                m.forward()
            got = m.get(t)
        finally:
            runtime.set_option("noaffine", 0)
        print(runtime.last_kernel(), flush=True)
        assert runtime.last_kernel().startswith("conv_blocks:%d,%d" % (cfg[1], cfg[4])), runtime.last_kernel()
        bad = int((got != want).sum())
        assert bad == 0, "%d of %d differ" % (bad, got.size)
    m.close()


def test_operators_of_a_run_one_by_one():
    """run_opr and the tensors between the blocks have their places in the plan, and a forward behind them is as it was"""
    m, x, src, want, t = _run((2, 512, 14, 14, 3, GENERIC), 5)
    for switch in ("fusedwpw", "fuseblocks"):
        runtime.set_option(switch, 1)
    try:
        m.finalize()
    finally:
        for switch in ("fusedwpw", "fuseblocks"):
            runtime.set_option(switch, 0)
    m.set_input(x, src)
    for i in range(m.nr_opr):
        m.run_opr(i)
    assert np.array_equal(m.get(t), want)
    m.forward()
    assert np.array_equal(m.get(t), want)
    m.close()
