"""Convolutions with weights and a patch of the image in LDS: strips, k-chunks that straddle taps, ragged frames and channels, every
requant tail; against the oracle and against the record's own kernel."""
import pytest

from helpers import assert_bit_exact, check_own_kernels, families, oracle_eval, run_on_gpu
from torq_compiler_amd import workloads as w

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [
    dict(N=16, H=56, W=56, C=96, O=96, realistic=True), dict(N=12, H=65, W=67, C=32, O=64), dict(N=60, H=31, W=29, C=16, O=16, KH=5, KW=5, pad=(2, 2, 2, 2), realistic=True),
    dict(N=5, H=120, W=112, C=48, O=80, KH=3, KW=4, pad=(1, 2, 0, 2), realistic=True), dict(N=20, H=60, W=50, C=112, O=32, KH=7, KW=2, pad=(0, 1, 3, 3), realistic=True),
    dict(N=1100, H=7, W=7, C=64, O=64, realistic=True), dict(N=8, H=90, W=83, C=32, O=32, nhwc=False, realistic=True),
    dict(N=6, H=100, W=100, C=80, O=48, pad=(0, 0, 0, 0), input_zp=-90, output_min=-128), dict(N=40, H=34, W=40, C=16, O=16, KH=5, KW=5, pad=(4, 4, 4, 4)),
    dict(N=20, H=51, W=50, C=24, O=48, realistic=True),  # channels padded to 32 on the way
], ids=lambda kw: "x".join(str(v) for v in kw.values()))
def test_conv_patch(device, kw, monkeypatch):
    monkeypatch.setenv("THIP_PAD_ROWS", "1")
    wl = w.conv2d_workload(**kw)
    print("[gpu-case]", wl.name, flush=True)
    want = oracle_eval(wl)[0]
    launched = []
    got, _ = run_on_gpu(device, wl, via="device", launched=launched)
    assert "conv_patch_i8" in families(launched), launched
    assert_bit_exact(got[0], want, wl.name)
    check_own_kernels(device, wl, [want], "device")


@pytest.mark.parametrize("shift", [31, 32, 33, 40, 41, 45, 46])
@pytest.mark.parametrize("bounds", [dict(output_min=-128), dict(output_min=17, output_zp=20), dict(output_min=-128, output_max=126)], ids=lambda b: "_".join(str(v) for v in b.values()))
def test_packed_requant(device, shift, bounds, monkeypatch):
    """Both packed tails at the ends of their shifts, and the ones beside them; bit for bit."""
    top = min(shift - 11, 30)  # a multiplier's highest bit: results over all of int8 where the shift allows it
    monkeypatch.setattr(w, "random_requant", lambda rng, n, realistic: (rng.integers(1 << top, (2 << top) - 1, size=n).astype("int32"), [shift] * n))
    wl = w.conv2d_workload(N=17, H=56, W=54, C=16, O=48, realistic=True, **bounds)
    print("[gpu-case]", wl.name, shift, bounds, flush=True)
    launched = []
    got, _ = run_on_gpu(device, wl, via="device", launched=launched)
    assert "conv_patch_i8" in families(launched), launched
    want = oracle_eval(wl)[0]
    assert len(set(want.reshape(-1).tolist())) > 8, wl.name
    assert_bit_exact(got[0], want, wl.name)
