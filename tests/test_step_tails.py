"""Kernels whose waves walk K in steps with a ring of operands in flight: shares below, at and beyond the ring and its
multiples, where the last steps are taken one by one."""
import numpy as np
import pytest

from cases import ConvCase, MatMulCase
from golden_cases import unsat
from megcc_amd import abi as A
from megcc_amd import runtime
from oracle import port

import test_dw_pw
from test_gpu_parity import _product, compare, run_gpu

pytestmark = pytest.mark.gpu


# (input channels, filter, stride): 9, 18, 25, 27, 36, 45, 49, 63 steps, shared by one, two or four waves
@pytest.mark.parametrize("ic,k,stride", [(4, 3, 2), (36, 3, 2), (32, 5, 2), (68, 3, 2), (100, 3, 2),
                                         (132, 3, 2), (20, 7, 2), (200, 3, 2)])
@pytest.mark.parametrize("ties", [True, False])
@pytest.mark.parametrize("bias", [True, False])
def test_shares_of_k_in_dense_layers_without_staging(ic, k, stride, ties, bias):
    d = unsat(ic * k * k) if ties else unsat(ic * k * k) * 1.0371
    case = ConvCase(A.FMT_NCHW44, A.DENSE, 2, ic, 17, 14, 36, k, stride, k // 2, A.RELU, bias=bias, scales=(0.02, 0.01, d))
    arrays = case.gen(seed=41)
    got = run_gpu(case, arrays)
    assert runtime.last_kernel().startswith("conv_mfma_i8_gather"), runtime.last_kernel()
    compare(got, case.run_port(arrays), repr(case))


# both sides of the border between the LDS-direct kernel (by its variants) and the one without staging, channels and pixels that
# fill no whole tile among them
@pytest.mark.parametrize("n,ic,ih,iw,oc,k,stride,kernel", [
    (5, 128, 28, 28, 100, 3, 1, "gather"), (6, 128, 28, 28, 100, 3, 1, "dma:6"), (2, 32, 28, 28, 64, 3, 1, "dma:6"), (2, 64, 28, 28, 64, 3, 1, "gather"),
    (10, 96, 14, 14, 232, 3, 1, "gather"), (11, 96, 14, 14, 232, 3, 1, "dma:7"), (7, 32, 14, 14, 64, 3, 1, "gather"),
    (8, 76, 24, 22, 96, 3, 1, "gather"), (5, 88, 48, 38, 80, 3, 1, "dma:1"), (6, 40, 56, 55, 100, 3, 2, "gather"),
    (2, 76, 57, 68, 96, 3, 1, "gather"), (24, 44, 17, 16, 112, 3, 1, "dma:4"),
    (8, 56, 30, 29, 84, 5, 1, "gather"), (14, 52, 24, 24, 196, 5, 1, "dma:8"),
    (5, 52, 46, 44, 100, 5, 2, "gather"), (7, 64, 26, 21, 268, 5, 1, "dma:9")])
def test_layers_on_both_sides_of_the_staging_border(n, ic, ih, iw, oc, k, stride, kernel):
    port.set_threads(8)
    case = ConvCase(A.FMT_NCHW44, A.DENSE, n, ic, ih, iw, oc, k, stride, k // 2, A.RELU, scales=(0.02, 0.01, unsat(ic * k * k)))
    arrays = case.gen(seed=48)
    got = run_gpu(case, arrays)
    assert runtime.last_kernel().startswith("conv_mfma_i8_" + kernel), runtime.last_kernel()
    compare(got, case.run_port(arrays), repr(case))


# the groups that share K: one, two and four with 32 x 32, 64 x 32, 32 x 64 and 64 x 64 outputs a wave, on both sides of each line
@pytest.mark.parametrize("n,ic,ih,iw,oc,k,stride,kernel", [
    (36, 60, 28, 30, 36, 3, 2, "32,32,4"), (70, 60, 29, 30, 64, 3, 2, "32,32,2"), (130, 60, 29, 30, 64, 3, 2, "32,32,1"),
    (80, 20, 29, 30, 100, 3, 2, "64,32,2"), (80, 80, 29, 30, 100, 3, 2, "64,32,4"), (100, 68, 29, 30, 100, 3, 2, "64,32,2"),
    (28, 56, 41, 59, 16, 3, 1, "32,64,2"), (24, 40, 56, 55, 16, 5, 1, "32,64,4"),
    (150, 20, 29, 30, 100, 3, 2, "64,64,1"), (150, 100, 29, 30, 100, 3, 2, "64,64,2"),
    # one tile a workgroup, its size by what its operands cost: from 25 steps on two channel tiles, from 80 on pixels too
    (16, 60, 29, 30, 100, 3, 2, "32,32,4"), (16, 20, 29, 30, 100, 5, 2, "64,32,4"), (20, 256, 29, 30, 100, 3, 2, "64,32,4"),
    (20, 260, 29, 30, 100, 3, 2, "64,64,4"), (40, 256, 29, 30, 28, 3, 2, "32,32,4"), (40, 260, 29, 30, 28, 3, 2, "32,64,4")])
def test_groups_that_share_k(n, ic, ih, iw, oc, k, stride, kernel):
    port.set_threads(8)
    case = ConvCase(A.FMT_NCHW44, A.DENSE, n, ic, ih, iw, oc, k, stride, k // 2, A.RELU, scales=(0.02, 0.01, unsat(ic * k * k)))
    arrays = case.gen(seed=49)
    got = run_gpu(case, arrays)
    assert runtime.last_kernel().split("+")[0] == "conv_mfma_i8_gather:" + kernel, runtime.last_kernel()
    compare(got, case.run_port(arrays), repr(case))


# images beyond an XCD's L2, whose tiles are dealt to the XCDs in runs: one, two and several channel tiles, the last one whole or hanging over,
# a number of pixel tiles that is and is not a multiple of eight
@pytest.mark.parametrize("n,ic,ih,iw,oc,k,stride", [(21, 116, 47, 59, 20, 3, 1), (17, 64, 66, 66, 72, 3, 2), (67, 132, 23, 21, 36, 3, 2), (35, 52, 58, 58, 352, 3, 2), (23, 36, 87, 74, 144, 3, 1),
                                                    (23, 36, 87, 74, 64, 3, 1)])
@pytest.mark.parametrize("plain", [0, 1])
def test_tiles_in_runs_on_the_xcds(n, ic, ih, iw, oc, k, stride, plain):
    port.set_threads(8)
    assert n * ic * ih * iw > 1 << 22
    case = ConvCase(A.FMT_NCHW44, A.DENSE, n, ic, ih, iw, oc, k, stride, k // 2, A.RELU, scales=(0.02, 0.01, unsat(ic * k * k)))
    arrays = case.gen(seed=42)
    runtime.set_option("noxcdorder", plain)
    try:
        got = run_gpu(case, arrays)
        assert runtime.last_kernel().startswith("conv_mfma_i8_gather"), runtime.last_kernel()
    finally:
        runtime.set_option("noxcdorder", 0)
    compare(got, case.run_port(arrays), repr(case))


# rows, columns and K at the edges of the 16 x 16 tiles and their steps of 16, four and eight waves; tiles that are no multiple
# of eight, in strips; one and two tiles a CU, and the first size beyond
@pytest.mark.parametrize("m,k,n", [(5, 1, 5), (16, 15, 16), (17, 16, 15), (15, 17, 33), (33, 63, 31), (31, 64, 49), (16, 65, 32), (48, 255, 16),
                                   (33, 256, 17), (64, 257, 100), (100, 1031, 130), (357, 40, 301), (200, 300, 700), (40, 1300, 1700),
                                   (512, 70, 256), (512, 270, 257), (23, 2000, 3100), (64, 300, 3900), (200, 90, 1111)])
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
def test_f32_products_of_few_tiles(m, k, n, ta, tb):
    case = MatMulCase(m, k, n, trans_a=ta, trans_b=tb)
    arrays = case.gen(seed=43)
    got = run_gpu(case, arrays)
    assert runtime.last_kernel().startswith("gemm_f32_ks:"), runtime.last_kernel()
    # each of the k products and sums is rounded once, in whatever order
    bound = _product(case, {x: np.abs(v) for x, v in arrays.items()}) * (k * 2.0 ** -24)
    assert np.all(np.abs(got - _product(case, arrays)) <= bound)
    assert np.array_equal(run_gpu(case, {x: np.round(8 * v) for x, v in arrays.items()}), _product(case, {x: np.round(8 * v) for x, v in arrays.items()}))


# 32 x 32, 32 x 64 and 64 x 64 tiles, with and without strips, at the edges of the steps, of the four waves' shares and of the
# short loop (28 steps of 8); 16 x 16 ones at theirs (28 of 16)
@pytest.mark.parametrize("m,n,ks", [(700, 800, (1, 7, 8, 9, 33, 224, 231, 232)), (637, 1589, (17, 32, 224, 232)), (2500, 700, (1, 31, 72, 226, 231, 233)),
                                    (2562, 675, (8, 100, 224)), (60, 500, (447, 448, 463, 464))])
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
def test_f32_products_of_short_k(m, n, ks, ta, tb):
    for k in ks:
        test_f32_products_of_few_tiles(m, k, n, ta, tb)


# the same edges in K = (channel, row, column) and pixels
@pytest.mark.parametrize("n,ic,ih,iw,oc,k", [(2, 1, 77, 77, 101, 3), (2, 9, 77, 77, 101, 3), (13, 21, 26, 30, 69, 3), (9, 24, 28, 30, 69, 3), (9, 25, 28, 29, 69, 3),
                                             (9, 26, 29, 29, 69, 3), (5, 224, 33, 31, 70, 1), (5, 232, 33, 31, 70, 1), (5, 3, 35, 51, 70, 1)])
def test_f32_convolutions_of_short_k(n, ic, ih, iw, oc, k):
    port.set_threads(8)
    case = ConvCase(A.FMT_NCHW, A.DENSE, n, ic, ih, iw, oc, k, 1, k // 2, A.RELU, dtype="f32")
    arrays = case.gen(seed=47)
    got = run_gpu(case, arrays)
    assert runtime.last_kernel().startswith("conv_f32_gemm_ks:32,32"), runtime.last_kernel()
    compare(got, case.run_port(arrays), repr(case))


@pytest.mark.parametrize("n,ic,ih,iw,oc,k,stride", [(1, 1, 4, 4, 16, 3, 1), (1, 5, 9, 9, 17, 3, 1), (2, 28, 13, 11, 33, 3, 2), (1, 29, 14, 15, 15, 3, 1),
                                                    (1, 64, 28, 28, 64, 3, 1), (1, 32, 56, 56, 32, 3, 1), (3, 100, 14, 13, 30, 1, 1), (1, 21, 17, 16, 40, 5, 2)])
@pytest.mark.parametrize("bias", [True, False])
def test_f32_convolutions_of_few_tiles(n, ic, ih, iw, oc, k, stride, bias):
    port.set_threads(8)
    case = ConvCase(A.FMT_NCHW, A.DENSE, n, ic, ih, iw, oc, k, stride, k // 2, A.RELU, dtype="f32", bias=bias)
    arrays = case.gen(seed=44)
    got = run_gpu(case, arrays)
    assert runtime.last_kernel().startswith("conv_f32_gemm_ks:16,16"), runtime.last_kernel()
    compare(got, case.run_port(arrays), repr(case))


GENERIC, TIES = test_dw_pw.GENERIC, test_dw_pw.TIES


# (n, c, oc, h, w, stride, activation, scales) with slices of 128, 256 and 512 channels of the result, the last one in part
@pytest.mark.parametrize("cfg", [
    (1, 256, 160, 9, 10, 1, A.RELU, TIES), (2, 512, 288, 5, 6, 2, A.RELU, GENERIC), (1, 1024, 96, 6, 7, 1, A.IDENTITY, GENERIC), (1, 1024, 416, 7, 8, 2, A.RELU, TIES),
    (20, 512, 512, 14, 13, 1, A.RELU, GENERIC), (66, 512, 544, 14, 15, 2, A.RELU, TIES), (40, 1024, 1056, 7, 7, 1, A.RELU, GENERIC), (17, 256, 288, 28, 27, 1, A.RELU, GENERIC),
    (70, 1024, 32, 20, 12, 1, A.RELU, TIES), (280, 1024, 32, 19, 13, 2, A.RELU, GENERIC), (70, 512, 32, 20, 10, 1, A.RELU, GENERIC), (280, 512, 64, 20, 11, 2, A.IDENTITY, TIES),
    (280, 256, 288, 20, 11, 2, A.RELU, GENERIC), (40, 256, 288, 28, 28, 1, A.RELU, TIES)], ids=lambda c: "n%d_c%d_oc%d_%dx%d_s%d_a%d" % c[:7])
def test_slices_of_channel_wise_pointwise_pairs(cfg):
    test_dw_pw.test_pair_in_one_kernel(cfg)


# image widths from the smallest the kernel takes, one output row, steps of 64 pixels that end inside a row, inside an image and
# behind the last one, one and two steps a wave; every form of the requantisation
@pytest.mark.parametrize("n,ih,iw", [(1, 2, 4), (3, 2, 4), (50, 6, 4), (1, 2, 8), (3, 2, 8), (1, 6, 12), (5, 10, 36), (2, 4, 132), (1, 34, 260), (30, 224, 224)])
@pytest.mark.parametrize("oc", [32, 64])
@pytest.mark.parametrize("act,noaffine", [(A.RELU, 0), (A.IDENTITY, 0), (A.RELU, 1), (A.IDENTITY, 1), (A.H_SWISH, 0), (A.SIGMOID, 0)])
def test_first_layer_steps(n, ih, iw, oc, act, noaffine):
    port.set_threads(8)
    if n == 30 and (noaffine or act in (A.H_SWISH, A.SIGMOID)):
        pytest.skip("the same steps as with the other activations")
    case = ConvCase(A.FMT_NCHW_NCHW44, A.DENSE, n, 3, ih, iw, oc, 3, 2, 1, act, bias=n != 3, scales=(0.02, 0.01, unsat(27)))
    arrays = case.gen(seed=45)
    runtime.set_option("noaffine", noaffine)
    try:
        got = run_gpu(case, arrays)
        assert runtime.last_kernel().startswith("conv_first_mfma"), runtime.last_kernel()
    finally:
        runtime.set_option("noaffine", 0)
    compare(got, case.run_port(arrays), repr(case))


# a filter that begins at any byte, and the narrowest images with it
@pytest.mark.parametrize("n,ih,iw", [(1, 2, 4), (5, 10, 36)])
@pytest.mark.parametrize("oc", [32, 64])
@pytest.mark.parametrize("at", [1, 2, 3])
def test_first_layer_filters_off_a_dword(n, ih, iw, oc, at):
    case = ConvCase(A.FMT_NCHW_NCHW44, A.DENSE, n, 3, ih, iw, oc, 3, 2, 1, A.RELU, scales=(0.02, 0.01, unsat(27)))
    arrays = case.gen(seed=46)
    ins, outs = case.specs(arrays)
    ins[1].array = np.concatenate([np.full(at, 77, np.int8), arrays["flt"].ravel()])
    ins[1].offset = at
    got = runtime.run_symbol(case.symbol(), ins, outs)
    assert runtime.last_kernel().startswith("conv_first_mfma"), runtime.last_kernel()
    compare(got, case.run_port(arrays), repr(case))
