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


# either side of every line between the kernel for few rows and the matrix cores, and the shapes whose times the lines follow from
GEVM, KS = "gevm_f32", "gemm_f32_ks:"


@pytest.mark.parametrize("m,k,n,tb,own", [
    (4, 1024, 1000, False, GEVM), (4, 1536, 1000, False, GEVM), (4, 1536, 2048, False, GEVM), (4, 512, 4096, False, GEVM), (4, 513, 2049, False, KS), (3, 512, 2049, False, GEVM), (3, 513, 2049, False, KS), (4, 1537, 1000, False, KS), (4, 2346, 311, False, KS), (4, 4096, 1300, False, KS),
    (4, 2799, 650, False, KS), (4, 2800, 650, False, GEVM), (4, 4000, 576, False, KS), (4, 4000, 577, False, GEVM), (4, 4000, 1000, False, GEVM),
    (4, 4000, 1008, False, GEVM), (4, 4000, 1009, False, KS), (3, 1024, 3530, False, KS), (3, 1025, 2048, False, GEVM), (3, 1025, 2049, False, KS), (2, 1024, 3530, False, GEVM),
    (3, 2560, 1281, False, GEVM), (3, 2561, 1281, False, KS), (3, 4096, 1280, False, GEVM), (3, 4096, 1300, False, KS), (2, 4000, 1400, False, GEVM),
    (4, 560, 2048, True, GEVM), (4, 560, 2049, True, KS), (4, 561, 3530, True, GEVM), (4, 1024, 3530, True, GEVM), (4, 4000, 311, True, GEVM), (3, 4096, 4096, True, GEVM)])
def test_which_kernel_few_rows_run_on(m, k, n, tb, own):
    case = MatMulCase(m, k, n, False, tb)
    check_product(case, 67, own)
    if own == GEVM:
        assert runtime.last_kernel() == GEVM


def tree_of_sums(a, b):
    """one pass over B: four rounded products a lane, and another four every 256, then a tree over 64 lanes"""
    lanes = np.zeros((64, a.shape[1], b.shape[1]), np.float32)
    for at in range(len(a)):
        lanes[at // 4 % 64] += a[at][:, None] * b[at]
    while len(lanes) > 1:
        lanes = lanes[:len(lanes) // 2] + lanes[len(lanes) // 2:]
    return lanes[0]


def check_against_tree(case, seed, kernel, most):
    arrays = case.gen(seed=seed)
    got, exact = run(case, arrays), product64(case, arrays)
    assert runtime.last_kernel().startswith(kernel), runtime.last_kernel()
    sums = tree_of_sums(arrays["a"] if case.trans_a else np.ascontiguousarray(arrays["a"].T), np.ascontiguousarray(arrays["b"].T))
    error, tree = np.linalg.norm(got - exact), np.linalg.norm(sums - exact)
    print("relative error", error / np.linalg.norm(exact), "of the tree", tree / np.linalg.norm(exact))
    assert error <= most * tree


@pytest.mark.parametrize("m,k,n", [(1, 66, 20000), (2, 66, 8000), (3, 68, 6000), (4, 70, 2048), (1, 200, 9000), (4, 260, 2000), (2, 1030, 3000)])
def test_few_rows_of_a_transposed_b_are_as_precise_as_a_tree_of_sums(m, k, n):
    check_against_tree(MatMulCase(m, k, n, False, True), 79, GEVM, 1.005)


# (6000 outputs and more: the ratio of the norms of two such sets of errors spreads by some 1.3 %)
@pytest.mark.parametrize("m,k,n,ta", [
    (4, 64, 1500, True), (4, 256, 1500, True), (3, 300, 2000, True), (2, 500, 3000, True), (4, 600, 1500, True), (2, 200, 9000, True), (4, 330, 9000, True),
    (4, 1000, 9000, True), (4, 16, 30000, True), (4, 64, 2049, False), (4, 256, 3000, False), (4, 464, 3000, False), (4, 560, 9000, False)])
def test_few_rows_of_a_transposed_b_on_the_matrix_cores_are_as_precise_as_a_tree_of_sums(m, k, n, ta):
    check_against_tree(MatMulCase(m, k, n, ta, True), 78, KS + "16,16", 1.05)


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


# (layers that the tiled kernel is estimated faster for, with the kernel for small layers in front of it, and not the one of whole K a wave)
@pytest.mark.parametrize("n,ic,h,w,oc,k", [(5, 7, 63, 78, 9, 1), (9, 1, 62, 44, 23, 3), (8, 10, 9, 169, 183, 1)])
def test_layers_of_many_pixels_and_few_channels(n, ic, h, w, oc, k):
    case = ConvCase(A.FMT_NCHW, A.DENSE, n, ic, h, w, oc, k, 1, k // 2, A.RELU, dtype="f32")
    arrays = case.gen(seed=63)
    got, want = run(case, arrays), case.run_port(arrays)
    assert runtime.last_kernel().startswith("conv_f32_gemm_ks:32,32"), runtime.last_kernel()
    assert np.abs(got - want).max() <= 1e-4 * max(1.0, np.abs(want).max())


def convolution64(case, arrays, mag=False):
    import torch
    f = np.abs if mag else np.array
    flt, src = (torch.from_numpy(f(arrays[x]).astype(np.float64)) for x in ("flt", "src"))
    bias = torch.from_numpy(f(arrays["bias"]).astype(np.float64).reshape(-1)) if case.bias else None
    return torch.nn.functional.conv2d(src, flt, bias, stride=(case.sh, case.sw), padding=(case.ph, case.pw)).numpy()


# a wave has its pixels for the whole of K: tiles of 16, 32 and 64 channels, full and with one channel more or less; K of less
# than a step, of whole steps and turns of four and with a rest; as few pixels as it takes, and waves without any; taps outside
WIDE = [("32,32", 1, 17, 96, 96, 128, 1, 1), ("32,32", 11, 18, 97, 68, 68, 1, 2), ("32,32", 11, 5, 22, 63, 63, 3, 1), ("32,32", 13, 15, 81, 83, 83, 3, 1),
        ("32,32", 4, 31, 64, 67, 67, 1, 1), ("32,32", 8, 12, 33, 41, 41, 3, 1), ("32,32", 4, 32, 32, 112, 112, 3, 1), ("32,32", 10, 86, 19, 63, 86, 1, 1), ("16,32", 7, 6, 12, 77, 77, 3, 1), ("16,32", 16, 89, 15, 101, 16, 3, 1),
        ("16,32", 16, 3, 8, 112, 112, 3, 1), ("16,32", 16, 3, 16, 112, 112, 3, 2), ("16,32", 14, 51, 35, 95, 49, 1, 2), ("64,32", 8, 64, 64, 56, 56, 3, 1),
        ("64,32", 7, 52, 121, 42, 42, 3, 1), ("64,32", 4, 25, 60, 79, 79, 5, 1)]


@pytest.mark.parametrize("tile,n,ic,oc,h,w,k,stride", WIDE)
@pytest.mark.parametrize("act,bias", [(A.RELU, True), (A.IDENTITY, False)])
def test_layers_of_many_pixels(tile, n, ic, oc, h, w, k, stride, act, bias):
    case = ConvCase(A.FMT_NCHW, A.DENSE, n, ic, h, w, oc, k, stride, k // 2, act, dtype="f32", bias=bias)
    arrays = case.gen(seed=64)
    got = run(case, arrays)
    assert runtime.last_kernel().startswith("conv_f32_wide"), runtime.last_kernel()
    want = convolution64(case, arrays)
    # each of the products and sums (and the bias's) is rounded once, in whatever order
    bound = (ic * k * k + 2) * 2.0 ** -24 * convolution64(case, arrays, mag=True)
    assert np.all(np.abs(got - (np.maximum(want, 0) if act == A.RELU else want)) <= bound)
    # an Inf stays where it belongs: in a channel's filter (the last value, beside the next channel's), in a pixel
    arrays["flt"][oc // 2, -1, -1, -1] = np.inf
    assert np.isfinite(np.delete(run(case, arrays), oc // 2, axis=1)).all()
    arrays = case.gen(seed=64)
    arrays["src"][n - 1, ic - 1, h - 1, w - 1] = np.inf
    got = run(case, arrays)
    assert np.isfinite(got[:n - 1]).all() and np.isfinite(got[n - 1, :, :(h - k) // stride - 1]).all()


# other windows' places: a dilation, no padding and more than half a window, strides of two and three
@pytest.mark.parametrize("n,ic,oc,h,w,k,stride,pad,dilate", [(12, 8, 30, 71, 83, 3, 1, 2, 2), (10, 12, 20, 60, 75, 3, 1, 0, 1), (18, 3, 16, 98, 90, 5, 2, 4, 1), (6, 10, 40, 60, 70, 1, 1, 1, 1),
                                                             (42, 6, 62, 103, 101, 3, 3, 1, 1), (4, 5, 70, 66, 61, 5, 1, 4, 2)])
def test_layers_of_many_pixels_of_other_windows(n, ic, oc, h, w, k, stride, pad, dilate):
    import torch
    case = ConvCase(A.FMT_NCHW, A.DENSE, n, ic, h, w, oc, k, stride, pad, A.IDENTITY, dtype="f32", dilate=dilate)
    arrays = case.gen(seed=68)
    got = run(case, arrays)
    assert runtime.last_kernel().startswith("conv_f32_wide:"), runtime.last_kernel()
    want, mag = (torch.nn.functional.conv2d(*(torch.from_numpy(f(arrays[x]).astype(np.float64)) for x in ("src", "flt")),
                                            torch.from_numpy(f(arrays["bias"]).astype(np.float64).reshape(-1)), stride=stride, padding=pad,
                                            dilation=dilate).numpy() for f in (np.array, np.abs))
    assert np.all(np.abs(got - want) <= (ic * k * k + 2) * 2.0 ** -24 * mag)


# up to 16 channels and a long K on fewer pixels, or more than it takes: 16 x 16 tiles with four waves sharing K
@pytest.mark.parametrize("n,ic,oc,h,w,k,stride", [(8, 28, 16, 33, 33, 3, 1), (3, 250, 16, 53, 52, 1, 1), (13, 114, 11, 46, 57, 3, 2), (3, 95, 1, 65, 65, 3, 1)])
def test_layers_of_few_channels_and_a_long_k(n, ic, oc, h, w, k, stride):
    case = ConvCase(A.FMT_NCHW, A.DENSE, n, ic, h, w, oc, k, stride, k // 2, A.IDENTITY, dtype="f32")
    arrays = case.gen(seed=66)
    got = run(case, arrays)
    assert runtime.last_kernel().startswith("conv_f32_gemm_ks:16,16,4"), runtime.last_kernel()
    bound = (ic * k * k + 2) * 2.0 ** -24 * convolution64(case, arrays, mag=True)
    assert np.all(np.abs(got - convolution64(case, arrays)) <= bound)


@pytest.mark.parametrize("oc", [12, 32, 40])
@pytest.mark.parametrize("ic,k", [(16, 1), (24, 1), (3, 3), (32, 1), (39, 1), (48, 1), (7, 3), (63, 1)])
def test_layers_of_many_pixels_and_short_k_are_as_precise_as_sums_of_eight(oc, ic, k):
    """as the kernel that shares K among waves had them: no chain of a short K is longer than the eight values of a step"""
    case = ConvCase(A.FMT_NCHW, A.DENSE, 7, ic, 96, 96, oc, k, 1, k // 2, A.IDENTITY, dtype="f32", bias=False)
    arrays = case.gen(seed=69)
    got = run(case, arrays)[:2]
    assert runtime.last_kernel().startswith("conv_f32_wide:"), runtime.last_kernel()
    flt = arrays["flt"].reshape(oc, -1)
    src = np.pad(arrays["src"][:2], ((0, 0), (0, 0), (k // 2, k // 2), (k // 2, k // 2)))
    cols = np.stack([src[:, c, y:y + 96, x:x + 96] for c in range(ic) for y in range(k) for x in range(k)])  # [K][image][row][column]
    exact = np.tensordot(flt.astype(np.float64), cols.astype(np.float64), 1)
    total = np.float32(0)
    for k0 in range(0, len(cols), 8):
        chain = np.zeros(exact.shape, np.float32)
        for j in range(k0, min(k0 + 8, len(cols))):  # (a product is exact in 64 bits, and one rounding to 32 follows the addition)
            chain = (chain + flt[:, j, None, None, None].astype(np.float64) * cols[j].astype(np.float64)).astype(np.float32)
        total = total + chain
    exact, total = exact.swapaxes(0, 1), total.swapaxes(0, 1)
    error, of_eight = np.linalg.norm(got - exact), np.linalg.norm(total - exact)
    print("relative error", error / np.linalg.norm(exact), "of sums of eight", of_eight / np.linalg.norm(exact))
    # (the same sums in another order: some 200000 roundings of each kind, whose norms differ by less than 1 %, and instructions of two products)
    assert error <= 1.03 * of_eight


@pytest.mark.parametrize("ic", [33, 34, 41])
def test_layers_of_many_pixels_and_a_short_k_with_a_rest(ic):
    """a rest behind the steps of eight is no further rounding of the whole sum: as precise as where a chain of eight goes on with it"""
    case = ConvCase(A.FMT_NCHW, A.DENSE, 7, ic, 50, 50, 85, 1, 1, 0, A.IDENTITY, dtype="f32", bias=False)
    arrays = case.gen(seed=70)
    got = run(case, arrays)
    assert runtime.last_kernel().startswith("conv_f32_wide:"), runtime.last_kernel()
    flt, cols = arrays["flt"].reshape(85, ic).astype(np.float64), arrays["src"].swapaxes(0, 1).astype(np.float64)
    exact = np.tensordot(flt, cols, 1)
    total, chain = np.zeros(exact.shape, np.float32), np.zeros(exact.shape, np.float32)
    for j in range(ic):
        chain = (chain + flt[:, j, None, None, None] * cols[j]).astype(np.float32)
        if (j % 8 == 7 and j < ic // 8 * 8 - 1) or j == ic - 1:
            total, chain = total + chain, np.zeros(exact.shape, np.float32)
    exact, total = exact.swapaxes(0, 1), total.swapaxes(0, 1)
    error, of_chains = np.linalg.norm(got - exact), np.linalg.norm(total - exact)
    print("relative error", error / np.linalg.norm(exact), "of the chains", of_chains / np.linalg.norm(exact))
    assert error <= 1.02 * of_chains


def test_layers_of_many_pixels_reach_every_tile():
    for tile, n, ic, oc, h, w, k, stride in WIDE:
        case = ConvCase(A.FMT_NCHW, A.DENSE, n, ic, h, w, oc, k, stride, k // 2, A.SIGMOID, dtype="f32")
        arrays = case.gen(seed=65)
        got = run(case, arrays)
        assert runtime.last_kernel() == "conv_f32_wide:" + tile, runtime.last_kernel()
        want = convolution64(case, arrays)
        assert np.abs(got - 1 / (1 + np.exp(-want))).max() <= 1e-5


def product64(case, arrays):
    a, b = arrays["a"].astype(np.float64), arrays["b"].astype(np.float64)
    return (a.T if case.trans_a else a) @ (b.T if case.trans_b else b)


# products of middle size on the bf16 parts, a workgroup's waves sharing K, and the plan each is to have (rows of either operand, slices of K, which
# one is staged; None: not there): every transposition with either operand staged, one wave, two and four to a stage's K, whole and in slices; K with and
# without a rest of a stage, rows and columns beyond whole tiles
MIDDLE = [(512, 4096, 4096, "nn", "64,256,2,0"), (512, 4096, 4096, "nt", "64,256,2,0"), (512, 4096, 4096, "tn", "64,256,2,0"),
          (512, 4096, 4096, "tt", "64,256,2,0"), (1912, 1206, 1078, "nn", "64,128,1,1"), (1912, 1206, 1078, "nt", "64,128,1,1"),
          (1912, 1206, 1078, "tn", None), (1912, 1206, 1078, "tt", "64,128,1,1"), (83, 2794, 3689, "nn", None), (83, 2794, 3689, "nt", "64,256,8,0"),
          (83, 2794, 3689, "tn", None), (83, 2794, 3689, "tt", None), (947, 2247, 657, "nn", "64,64,3,0"), (947, 2247, 657, "nt", "64,64,3,0"),
          (947, 2247, 657, "tn", None), (947, 2247, 657, "tt", "64,64,3,0"), (1381, 2795, 925, "nn", "64,128,3,1"),
          (1381, 2795, 925, "nt", "64,128,3,1"), (1381, 2795, 925, "tn", None), (1381, 2795, 925, "tt", "64,128,3,1"),
          (3713, 2717, 528, "nn", "64,256,3,1"), (3713, 2717, 528, "nt", "64,256,3,1"), (3713, 2717, 528, "tn", None), (3713, 2717, 528, "tt", None),
          (320, 4095, 1100, "nn", "64,128,5,0"), (320, 4095, 1100, "nt", "64,128,5,0"), (320, 4095, 1100, "tn", "64,128,5,0"),
          (320, 4095, 1100, "tt", "64,128,5,0"), (2500, 1216, 400, "nn", None), (2500, 1216, 400, "nt", "64,256,3,0"), (2500, 1216, 400, "tn", None),
          (2500, 1216, 400, "tt", None), (1290, 1088, 1290, "nn", "64,128,1,0"), (1290, 1088, 1290, "nt", "64,128,1,0"),
          (1290, 1088, 1290, "tn", "64,128,1,0"), (1290, 1088, 1290, "tt", "64,128,1,0"), (1741, 1791, 471, "nn", "64,64,1,0"),
          (1026, 226, 3702, "nn", "64,256,1,0"), (2464, 223, 1597, "nn", "64,256,1,1"), (2942, 1274, 259, "nt", "64,64,1,0"),
          (1044, 211, 3628, "nt", "64,256,1,0"), (3660, 204, 1047, "nt", "64,256,1,1"), (1545, 3559, 605, "tn", "64,64,1,0"),
          (40, 3715, 2862, "tn", "64,64,5,0"), (3366, 1021, 563, "tn", "64,128,1,1"), (2927, 4073, 34, "tn", "64,128,11,1"),
          (3249, 237, 1222, "tn", "64,256,1,0"), (3620, 331, 1047, "tn", "64,256,1,1"), (2831, 2293, 70, "tn", "64,256,9,1"),
          (1152, 1791, 679, "tt", "64,64,1,0"), (1551, 246, 2436, "tt", "64,256,1,0"), (2466, 218, 1537, "tt", "64,256,1,1"),
          (1641, 3724, 66, "tt", "64,256,15,1")]


@pytest.mark.parametrize("m,k,n,t,plan", MIDDLE)
def test_products_of_middle_size(m, k, n, t, plan):
    case = MatMulCase(m, k, n, t[0] == "t", t[1] == "t")
    arrays = case.gen(seed=71)
    got, want = run(case, arrays), product64(case, arrays)
    assert runtime.last_kernel().startswith("gemm_f32_ks_split:" + plan if plan else KS), runtime.last_kernel()
    # each of the k products and sums is rounded once, in whatever order
    bound = product64(case, {x: np.abs(v) for x, v in arrays.items()}) * (k * 2.0 ** -24)
    assert np.all(np.abs(got - want) <= bound)
    if plan:
        runtime.set_option("nof32split", 1)
        try:
            in_f32 = run(case, arrays)
            assert runtime.last_kernel().startswith(("gemm_f32_ks:", "gemm_f32:")), runtime.last_kernel()
        finally:
            runtime.set_option("nof32split", 0)
        assert np.linalg.norm(got - want) <= np.linalg.norm(in_f32 - want)
        # whole numbers whose sums fit 24 bits: no rounding is due
        whole = {x: np.round(8 * v) for x, v in arrays.items()}
        assert np.array_equal(run(case, whole), product64(case, whole))


def test_products_of_middle_size_are_of_every_form():
    seen = {(t,) + tuple(plan.split(",")[1:2]) + (plan.split(",")[3], plan.split(",")[2] != "1") for _, _, _, t, plan in MIDDLE if plan}
    every = {(t, tile, swap, sliced) for t in ("nn", "nt", "tn", "tt") for tile in ("64", "128", "256") for swap in ("0", "1") for sliced in (False, True)
             if not (tile == "64" and swap == "1")}  # (64 rows of either: never swapped)
    assert seen == every, every - seen


@pytest.mark.parametrize("m,k,n,tb", [(1912, 1206, 1078, False), (947, 2247, 657, True), (83, 2794, 3689, True), (512, 4096, 4096, False)])
@pytest.mark.parametrize("value", [2.0 ** -120, 2.0 ** 70, np.inf, np.nan])
def test_products_of_middle_size_that_meet_a_value_the_parts_cannot_hold(m, k, n, tb, value):
    """one value at step `at` of K, of either operand: what its tile had summed before must neither be lost nor counted
    twice, and an infinity must not have been in the bf16 product"""
    case = MatMulCase(m, k, n, False, tb)
    arrays = case.gen(seed=73)
    for name in "ab":
        arrays[name] = np.where(arrays[name] == 0, np.float32(1), arrays[name])
    want0, mag0 = product64(case, arrays), product64(case, {x: np.abs(v) for x, v in arrays.items()})
    a, b = arrays["a"], arrays["b"].T if tb else arrays["b"]
    for at in (0, 63, 64, 255, 256, 511, 704, k // 2, k - 65, k - 1):
        for side in "ab":
            changed = dict(arrays)
            changed[side] = arrays[side].copy()
            row = 70
            (changed["a"] if side == "a" else (changed["b"].T if tb else changed["b"]).T)[row, at] = value
            got = run(case, changed)
            assert runtime.last_kernel().startswith("gemm_f32_ks_split"), runtime.last_kernel()
            want, mag = want0.copy(), mag0.copy()
            with np.errstate(invalid="ignore"):
                if side == "a":
                    want[row] += (value - np.float64(a[row, at])) * b[at].astype(np.float64)
                    mag[row] += abs(value) * np.abs(b[at])
                    line = (row, slice(None))
                else:
                    want[:, row] += (value - np.float64(b[at, row])) * a[:, at].astype(np.float64)
                    mag[:, row] += abs(value) * np.abs(a[:, at])
                    line = (slice(None), row)
                if not np.isfinite(value):
                    assert np.array_equal(np.isnan(got[line]), np.isnan(want[line]))
                    assert np.array_equal(got[line][np.isinf(want[line])], want[line][np.isinf(want[line])])
                    got[line] = want[line] = mag[line] = 0
            assert np.all(np.abs(got - want) <= mag * ((k + 2) * 2.0 ** -24)), (side, at)


@pytest.mark.parametrize("m,k,n,tb", [(1912, 1206, 1078, False), (947, 2247, 657, True), (83, 2794, 3689, True), (512, 4096, 4096, False)])
@pytest.mark.parametrize("value", [2.0 ** -133, 2.0 ** -134, 2.0 ** -140, 2.0 ** -149])
@pytest.mark.parametrize("side", ["a", "b"])
def test_products_of_middle_size_of_values_below_every_bf16(m, k, n, tb, value, side):
    """a row of them times values near 2^58 is made of ordinary numbers: none of them may go for a zero, and a zero is none of them"""
    case = MatMulCase(m, k, n, False, tb)
    check_tiny_values(case, "gemm_f32_ks_split", value, side)


def check_tiny_values(case, kernel, value, side):
    arrays = case.gen(seed=74)
    rng = np.random.default_rng(75)
    a, b = arrays["a"].T if case.trans_a else arrays["a"], arrays["b"].T if case.trans_b else arrays["b"]
    tiny, other = (a, b) if side == "a" else (b.T, a.T)  # (views)
    row, at = 70, rng.choice(case.k, 9, replace=False)
    other[:] = (other * 2.0 ** 57).astype(np.float32)
    tiny[row] = 0
    tiny[row, at] = (value * rng.choice([-1, 1], 9)).astype(np.float32)
    got, want = run(case, arrays), product64(case, arrays)
    assert runtime.last_kernel().startswith(kernel), runtime.last_kernel()
    mag = product64(case, {x: np.abs(v) for x, v in arrays.items()})
    line = (row, slice(None)) if side == "a" else (slice(None), row)
    assert mag[line].min() > 2.0 ** -100
    assert np.all(np.abs(got - want) <= mag * ((case.k + 1) * 2.0 ** -24))


@pytest.mark.parametrize("m,k,n,ta,tb", [(2040, 512, 1999, False, False), (1930, 531, 1925, True, True), (2900, 145, 3001, False, True)])
@pytest.mark.parametrize("value", [2.0 ** -133, 2.0 ** -134, 2.0 ** -149])
@pytest.mark.parametrize("side", ["a", "b"])
def test_products_of_many_tiles_of_values_below_every_bf16(m, k, n, ta, tb, value, side):
    check_tiny_values(MatMulCase(m, k, n, ta, tb), "gemm_f32_split", value, side)


def padded(arrays, case, pads):
    """the operands and the result with rows longer than they are wide, what lies between filled with NaN"""
    ins, outs = case.specs(arrays)
    for s, pad in zip(ins + outs, pads):
        rows, cols = s.shape
        s.strides = (cols + pad, 1)
        if s in ins:
            wide = np.full((rows, cols + pad), np.nan, np.float32)
            wide[:, :cols] = s.array
            s.array = wide
    outs[0].storage = (case.m, case.n + pads[2])
    return ins, outs


# ... with room for all of the slices, for two of them, for less, none, and a workspace that floats cannot be stored to
@pytest.mark.parametrize("m,k,n,t,plan", [p for p in MIDDLE if p[4] and p[4].split(",")[2] != "1"][::4])
def test_products_of_middle_size_with_less_workspace(m, k, n, t, plan):
    case = MatMulCase(m, k, n, t[0] == "t", t[1] == "t")
    arrays = case.gen(seed=76)
    want = product64(case, arrays)
    bound = product64(case, {x: np.abs(v) for x, v in arrays.items()}) * (k * 2.0 ** -24)
    op = runtime.PreparedOp(runtime.parse_symbol(case.symbol()), *case.specs(arrays))
    size, ptr = op.ws.size, op.ws.ptr
    slices = int(plan.split(",")[2])
    assert size >= slices * m * n * 4
    for room, at, most in ((slices * m * n * 4, ptr, slices), (2 * m * n * 4, ptr, 2), (2 * m * n * 4 - 1, ptr, 1), (0, None, 1), (size - 1, ptr + 1, 1)):
        op.ws.size, op.ws.ptr = room, at
        op.poison_outputs()
        op.launch()
        kernel = runtime.last_kernel()
        if kernel.startswith("gemm_f32_ks_split"):
            assert int(kernel.split(",")[2]) <= most, (kernel, room)
        else:
            assert kernel.startswith(("gemm_f32_ks:", "gemm_f32:")) and most < slices, (kernel, room)
        assert np.all(np.abs(op.result() - want) <= bound), (kernel, room)


PADDED = [(512, 1219, 640, "nn"), (83, 2794, 3689, "nt"), (1290, 1088, 1290, "tt"), (2927, 4073, 34, "tn"), (1, 700, 333, "nn"), (3, 513, 130, "nt"), (4, 2900, 700, "nn"),
          (2, 260, 75, "tn"), (70, 90, 66, "nn"), (2040, 145, 1999, "tn")]


@pytest.mark.parametrize("m,k,n,t", PADDED)
@pytest.mark.parametrize("pads", [(3, 0, 0), (0, 1, 0), (0, 0, 5), (4, 8, 12), (1, 3, 7)])
def test_products_of_padded_rows(m, k, n, t, pads):
    """whichever kernel takes them, nothing between the rows is read into a sum or written"""
    case = MatMulCase(m, k, n, t[0] == "t", t[1] == "t")
    arrays = case.gen(seed=77)
    op = runtime.PreparedOp(runtime.parse_symbol(case.symbol()), *padded(arrays, case, pads))
    before = op.result()
    op.launch()
    print("GPU case:", repr(case), pads, runtime.last_kernel(), flush=True)
    got = op.result()
    bound = product64(case, {x: np.abs(v) for x, v in arrays.items()}) * ((k + 1) * 2.0 ** -24)
    assert np.all(np.abs(got[:, :n] - product64(case, arrays)) <= bound)
    assert got[:, n:].tobytes() == before[:, n:].tobytes()
