"""The small GEMMs and convolutions without tiles in LDS: ragged ends, every result type and requant tail, the residual add; against
the oracle, and against the records' own kernels."""
import numpy as np
import pytest

from helpers import assert_bit_exact, check_own_kernels, families, oracle_eval, run_on_gpu
from torq_compiler_amd import workloads as w

pytestmark = pytest.mark.gpu

CASES = [
    lambda: w.fully_connected_workload(17, 16, 1, realistic=True), lambda: w.fully_connected_workload(33, 48, 33, realistic=True),
    lambda: w.fully_connected_workload(49, 960, 160), lambda: w.fully_connected_workload(64, 1040, 36, shift=7), lambda: w.fully_connected_workload(31, 2064, 70, shift=0),
    lambda: w.fully_connected_workload(40, 1024, 31, shift=62), lambda: w.matmul_workload(1, 20, 80, 45, constant_rhs=True, out_dtype=np.int32),
    lambda: w.matmul_workload(2, 33, 96, 40, constant_rhs=True),
    lambda: w.conv2d_workload(N=2, H=7, W=9, C=16, O=33, realistic=True), lambda: w.conv2d_workload(N=1, H=8, W=8, C=304, O=64, input_zp=-90),
    lambda: w.conv2d_workload(N=3, H=13, W=11, C=48, O=24, KH=5, KW=3, stride=(2, 1), pad=(1, 1, 2, 2), output_min=-128, realistic=True),
    lambda: w.conv2d_workload(N=1, H=33, W=35, C=80, O=8, KH=2, KW=2, stride=(2, 2), pad=(0, 1, 1, 0), realistic=True, nhwc=False),
    lambda: w.conv2d_workload(N=1, H=160, W=160, C=16, O=16, realistic=True),  # four waves per workgroup
    lambda: w.pointwise_add_workload(N=1, H=7, W=7, C=96, O=32), lambda: w.pointwise_add_workload(N=2, H=9, W=5, C=64, O=48, other_first=True),
]


@pytest.mark.parametrize("make", CASES, ids=range(len(CASES)))
def test_direct(device, make):
    wl = make()
    print("[gpu-case]", wl.name, flush=True)
    want = oracle_eval(wl)[0]
    launched = []
    got, _ = run_on_gpu(device, wl, via="device", launched=launched)
    assert "igemm_direct_i8" in families(launched), launched
    assert_bit_exact(got[0], want, wl.name)
    check_own_kernels(device, wl, [want], "device")
