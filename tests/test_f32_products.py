"""f32 products and convolutions at the sizes where a kernel or the choice between kernels can go wrong, against 64 bits."""
import numpy as np
import pytest

from cases import ConvCase, MatMulCase
from megcc_amd import abi as A
from megcc_amd import runtime

pytestmark = pytest.mark.gpu


def run(case, arrays):
    print("GPU case:", repr(case), flush=True)
    ins, outs = case.specs(arrays)
    return runtime.run_symbol(case.symbol(), ins, outs)


def check_product(case, seed, own=None):
    arrays = case.gen(seed=seed)
    got = run(case, arrays)
    if own:
        assert runtime.last_kernel().startswith(own), runtime.last_kernel()
    a, b = arrays["a"].astype(np.float64), arrays["b"].astype(np.float64)
    a, b = a.T if case.trans_a else a, b.T if case.trans_b else b
    # f32 sums of K products in any order: each of the K - 1 additions (and the product) rounds by 2^-24 of a partial
    # sum of magnitudes
    bound = (case.k + 1) * 2.0 ** -24 * (np.abs(a) @ np.abs(b))
    bad = np.abs(got - a @ b) > bound
    assert not bad.any(), "%r: %d of %d" % (case, bad.sum(), bad.size)


# fewer columns (steps of K) than a 16-byte load, one more than a multiple; one round of four waves, one more row, one
# round of 16, one more; columns of two workgroups and of every XCD
FEW = [(m, k, n, ta, tb) for m in (1, 2, 3, 4) for k, n in ((1, 1), (3, 5), (4, 4), (5, 3), (511, 17), (513, 19), (2048, 16), (2049, 133), (4100, 33))
       for ta, tb in ((False, False), (False, True), (True, False), (True, True)) if not (ta and m % 2)]


@pytest.mark.parametrize("m,k,n,ta,tb", FEW)
def test_few_rows(m, k, n, ta, tb):
    check_product(MatMulCase(m, k, n, ta, tb), 61)


def test_few_rows_of_values_that_are_not_finite():
    """a row or column beyond the operands (the clamped loads repeat the last one) leaves no trace, an Inf inside does"""
    case = MatMulCase(2, 515, 18)
    arrays = case.gen(seed=62)
    arrays["b"][514, 17] = np.inf
    got = run(case, arrays)
    assert np.isfinite(got[:, :17]).all() and not np.isfinite(got[:, 17]).any()
    case = MatMulCase(2, 515, 18, trans_b=True)
    arrays = case.gen(seed=62)
    arrays["b"][17, 514] = np.inf
    got = run(case, arrays)
    assert np.isfinite(got[:, :17]).all() and not np.isfinite(got[:, 17]).any()


@pytest.mark.parametrize("n,ic,h,w,oc,k", [(13, 12, 50, 100, 34, 1), (5, 3, 90, 91, 9, 3), (4, 5, 98, 98, 64, 1)])
def test_layers_of_many_pixels_and_few_channels(n, ic, h, w, oc, k):
    case = ConvCase(A.FMT_NCHW, A.DENSE, n, ic, h, w, oc, k, 1, k // 2, A.RELU, dtype="f32")
    arrays = case.gen(seed=63)
    got, want = run(case, arrays), case.run_port(arrays)
    assert runtime.last_kernel().startswith("conv_f32_gemm_ks"), runtime.last_kernel()
    assert np.abs(got - want).max() <= 1e-4 * max(1.0, np.abs(want).max())
