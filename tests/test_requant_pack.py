"""The qsi8 kernels' requantisation on the accumulators where it can go wrong: both sides of every step of the output, two
apart, as the biases of a pointwise layer whose source is zero. Expected: the oracle's literal float sequence, bit for bit.
The scales reach each form (a multiply-add, the reference's first two roundings in front of one, the literal sequence with
its division as two multiply-adds, the literal sequence itself for ratios under 5e-7) for each activation."""
import math

import numpy as np
import pytest

from cases import ConvCase
from megcc_amd import abi, runtime


def _calibrated(taps, seed):
    r = np.random.default_rng(seed)
    s, f = 0.02 * r.uniform(0.8, 1.2), 0.01 * r.uniform(0.8, 1.2)
    return s, f, s * f * 74.0 * 73.0 * math.sqrt(taps) / 36.0 * r.uniform(0.9, 1.1)


SCALES = [(0.02, 0.01, 0.05), (0.01, 0.01, 0.1), (0.25, 0.5, 0.125), (0.5, 0.5, 0.1), (0.0013, 0.00127, 0.9), (0.001, 0.001, 0.9), (0.0008, 0.0008, 1.3), (0.0005, 0.0005, 0.9),
          *[_calibrated(t, 7 * t + k) for t in (9, 64, 256, 300, 800, 4096) for k in range(3)]]


@pytest.mark.gpu
@pytest.mark.parametrize("noaffine", [0, 1])
@pytest.mark.parametrize("act", [abi.IDENTITY, abi.RELU, abi.H_SWISH, abi.SIGMOID])
@pytest.mark.parametrize("scales", SCALES, ids=["%.4g,%.4g,%.4g" % s for s in SCALES])
def test_both_sides_of_every_step(scales, act, noaffine):
    case = ConvCase(abi.FMT_NCHW44, abi.DENSE, 1, 32, 8, 8, 1024, 1, 1, 0, act, scales=scales)
    arrays = case.gen(3)
    arrays["src"][...] = 0
    c = float(np.float32(scales[0])) * float(np.float32(scales[1])) / float(np.float32(scales[2]))
    v = np.arange(-127, 128) - 0.5
    if act == abi.H_SWISH:
        v = np.where((v > 0) & (v < 3), 0.5 * (np.sqrt(9 + 24 * np.abs(v)) - 3), v)
    elif act == abi.SIGMOID:
        v = v / 20
    acc = np.clip(np.floor(v / c)[:, None] + np.arange(-1, 3), -2.0e9, 2.0e9).astype(np.int64).reshape(-1)
    # (the reference's conversion of a scaled value of 2^31 and more is undefined: the largest accumulator stays below)
    acc = np.concatenate([acc, [0, 1, -1, int(min(2.0e9, 2.0e9 / c))]])
    arrays["bias"][...] = acc.astype(np.int32).reshape(arrays["bias"].shape)
    runtime.set_option("noaffine", noaffine)
    try:
        ins, outs = case.specs(arrays)
        got = runtime.run_symbol(case.symbol(), ins, outs)
    finally:
        runtime.set_option("noaffine", 0)
    want = case.run_port(arrays)
    bad = np.argwhere(got != want)
    assert bad.size == 0, "accumulator %d: %d, expected %d" % (
        acc[bad[0][1] * 4 + bad[0][4]], got[tuple(bad[0])], want[tuple(bad[0])])
