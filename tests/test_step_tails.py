"""Kernels whose waves walk K in steps with a ring of operands in flight: shares below, at and beyond the ring and its
multiples, where the last steps are taken one by one."""
import pytest

from cases import ConvCase
from golden_cases import unsat
from megcc_amd import abi as A
from megcc_amd import runtime
from oracle import port
from test_gpu_parity import compare, run_gpu

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
