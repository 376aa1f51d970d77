"""Channel counts that fill no 16-byte chunks: rows padded, then a dense kernel; against the oracle and record by record."""
import numpy as np
import pytest

from helpers import assert_bit_exact, oracle_eval, run_on_gpu
from torq_compiler_amd import workloads as w

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [
    lambda: w.fully_connected_workload(1, 17, 33, realistic=True), lambda: w.fully_connected_workload(16, 2230, 109, realistic=True),  # few rows
    lambda: w.fully_connected_workload(17, 1, 16), lambda: w.fully_connected_workload(300, 333, 520, realistic=True),
    lambda: w.fully_connected_workload(1300, 250, 131), lambda: w.matmul_workload(2, 40, 75, 40, constant_rhs=True, out_dtype=np.int32),
    lambda: w.matmul_workload(1, 70, 75, 48, constant_rhs=True), lambda: w.matmul_workload(1, 65, 31, 83, constant_rhs=True),
    lambda: w.conv2d_workload(N=2, H=9, W=11, C=63, O=52, KH=1, KW=1, pad=(0, 0, 0, 0), realistic=True),
    lambda: w.conv2d_workload(N=1, H=17, W=13, C=53, O=148, realistic=True), lambda: w.conv2d_workload(N=3, H=8, W=9, C=9, O=20, input_zp=101, output_min=-128, realistic=True),
    lambda: w.conv2d_workload(N=2, H=15, W=16, C=133, O=34, stride=(2, 2), pad=(1, 1, 0, 1), realistic=True, nhwc=False),
    lambda: w.conv2d_workload(N=2, H=12, W=12, C=40, O=24, KH=1, KW=1, stride=(2, 2), pad=(0, 0, 0, 0), realistic=True),
    lambda: w.conv2d_workload(N=1, H=20, W=20, C=200, O=300, KH=5, KW=5, pad=(2, 2, 2, 2)),
], ids=range(14))
def test_padded(device, make, tmp_path, monkeypatch):
    monkeypatch.setenv("THIP_PAD_ROWS", "1")
    wl = make()
    print("[gpu-case]", wl.name, flush=True)
    want = oracle_eval(wl)[0]
    for via in ("device", "host"):
        launched = []
        got, _ = run_on_gpu(device, wl, via=via, launched=launched)
        assert "pad_rows_i8" in launched, launched
        assert_bit_exact(got[0], want, wl.name)
    device.set_event_log(str(tmp_path / "log.csv"))  # a log has its records launched one by one
    try:
        got, _ = run_on_gpu(device, wl)
    finally:
        device.set_event_log(None)
    assert_bit_exact(got[0], want, wl.name + " record by record")


@pytest.mark.parametrize("make", [lambda: w.fully_connected_workload(300, 333, 520, realistic=True), lambda: w.conv2d_workload(N=1, H=17, W=13, C=53, O=148, realistic=True)], ids=["linear", "conv"])
def test_without_memory_for_the_padded_operands(device, make, monkeypatch):
    """The rows padded to whole chunks and the weights spread to match want memory that the op's own kernel does not: where there is too
    little the op runs by that."""
    wl = make()
    print("[gpu-case]", wl.name, flush=True)
    want = oracle_eval(wl)[0]
    monkeypatch.setenv("THIP_PAD_ROWS", "1")
    for room, padded in ((0, False), (16 * 1024, False), (64 << 20, True)):
        monkeypatch.setenv("THIP_STEP_BYTES", str(room))
        launched = []
        got, kernels = run_on_gpu(device, wl, via="device", launched=launched)
        assert ("pad_rows_i8" in launched) == padded and (padded or launched == kernels), launched
        assert_bit_exact(got[0], want, "%s, %d bytes" % (wl.name, room))


@pytest.mark.parametrize("make", [
    lambda: w.fully_connected_workload(20, 1, 16), lambda: w.fully_connected_workload(2, 11, 33, realistic=True), lambda: w.fully_connected_workload(1, 21, 33, realistic=True),
    lambda: w.fully_connected_workload(31, 2230, 109, realistic=True), lambda: w.fully_connected_workload(33, 161, 31, realistic=True), lambda: w.fully_connected_workload(300, 95, 520, realistic=True),
    lambda: w.matmul_workload(1, 40, 75, 42, constant_rhs=True, out_dtype=np.int32), lambda: w.matmul_workload(1, 70, 79, 47, constant_rhs=True),
    lambda: w.conv2d_workload(N=2, H=9, W=11, C=63, O=53, KH=1, KW=1, pad=(0, 0, 0, 0), realistic=True), lambda: w.conv2d_workload(N=1, H=17, W=13, C=53, O=148, realistic=True),
    lambda: w.conv2d_workload(N=3, H=8, W=9, C=9, O=20, input_zp=101, output_min=-128, realistic=True),
    lambda: w.conv2d_workload(N=2, H=15, W=16, C=133, O=34, stride=(2, 2), pad=(1, 1, 0, 1), realistic=True, nhwc=False),
    lambda: w.conv2d_workload(N=2, H=12, W=12, C=40, O=24, KH=1, KW=1, stride=(2, 2), pad=(0, 0, 0, 0), realistic=True),
    lambda: w.conv2d_workload(N=1, H=12, W=14, C=200, O=30, KH=5, KW=5, pad=(2, 2, 2, 2), realistic=True), lambda: w.conv2d_workload(N=6, H=70, W=70, C=31, O=9, realistic=True),
], ids=range(15))
def test_rows_as_they_are(device, make, monkeypatch):
    """Chunks that reach into the next row and, at the tensor's end, begin before their place."""
    monkeypatch.setenv("THIP_PAD_ROWS", "2")
    wl = make()
    print("[gpu-case]", wl.name, flush=True)
    want = oracle_eval(wl)[0]
    for via in ("device", "host"):
        launched = []
        got, _ = run_on_gpu(device, wl, via=via, launched=launched)
        assert {"igemm_direct_i8<%d,%d,%d>" % (window, waves, how) for window in (0, 1) for waves in (4, 8) for how in (1, 2)} & set(launched) and "pad_rows_i8" not in launched, launched
        assert_bit_exact(got[0], want, wl.name)
