"""int8 results whose rows are no whole 16 columns, requantised in registers by the ring kernels and conv_patch_i8: every length behind the last whole
16, rows that begin at any alignment; against the oracle and against the op's own kernel."""
import pytest

from helpers import assert_bit_exact, check_own_kernels, families, oracle_eval, run_on_gpu
from torq_compiler_amd import workloads as w

pytestmark = pytest.mark.gpu


def check(device, wl, family, epilogue=None):
    print("[gpu-case]", wl.name, flush=True)
    want = oracle_eval(wl)[0]
    launched = []
    got, _ = run_on_gpu(device, wl, via="device", launched=launched)
    assert families(launched) == [family] and (epilogue is None or launched[0].endswith(epilogue)), launched
    assert_bit_exact(got[0], want, wl.name)
    check_own_kernels(device, wl, [want], "device")


@pytest.mark.parametrize("columns", list(range(497, 512)) + [1000, 1018])
@pytest.mark.parametrize("realistic", [True, False])
def test_linear(device, columns, realistic):
    check(device, w.fully_connected_workload(4101, 96, columns, realistic=realistic), "igemm_dense_i8", ",3,0>" if realistic else ",0,0>")  # the general tail: through LDS


@pytest.mark.parametrize("kw", [dict(N=20, H=33, W=33, C=64, O=130), dict(N=16, H=56, W=56, C=128, O=136, output_min=-128), dict(N=24, H=40, W=41, C=48, O=99, stride=(1, 2))],
                         ids=lambda kw: "x".join(str(v) for v in kw.values()))
def test_window(device, kw):
    check(device, w.conv2d_workload(realistic=True, **kw), "igemm_dense_conv_i8", ",3,0>")


@pytest.mark.parametrize("O", [1, 8, 15, 17, 31, 40, 63, 65, 90, 95])
def test_patch(device, O):
    check(device, w.conv2d_workload(N=17, H=56, W=54, C=32, O=O, realistic=True), "conv_patch_i8")
