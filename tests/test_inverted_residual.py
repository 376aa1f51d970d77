"""Pointwise + depthwise convolution as one launch: strips, shared workgroups, ragged frames and channels, every requant tail."""
import numpy as np
import pytest

from helpers import assert_bit_exact, families, oracle_network, run_on_gpu
from torq_compiler_amd import Program, workloads as w

pytestmark = pytest.mark.gpu


def block(N, H, W, C, E, stride, pad=(1, 1, 1, 1), shift=None, first=None, seed=1060, top=127):
    """widen (pointwise, or `first` = (window, stride, pad) over few channels) -> depthwise 3x3, the wide image an intermediate; `shift`: a literal requant range for both (results
    saturate, the general 32-bit tail) instead of one that spreads them."""
    rng = np.random.default_rng(seed)
    x = rng.integers(-128, 128, size=(N, H, W, C)).astype(np.int8)
    layers = []
    k, cs, cpad = first or (1, 1, (0, 0, 0, 0))
    for op, shape, fan, zp, zout in (("conv2d", (E, C, k, k), C * k * k, -3, -120), ("depthwise_conv2d", (E, 1, 3, 3), 9, -120, 7)):
        wt = rng.integers(-127, 128, size=shape).astype(np.int8)
        mult, sh = w.quantize_multiplier(60 / (np.sqrt(fan) * 5400) * rng.uniform(0.8, 1.2, E))
        if shift is not None:
            sh = np.full(E, shift, dtype=np.int8)
        sb, sf = w.derive_scale_bias(mult, sh, rng.integers(-4000, 4000, E), wt, zp)
        attrs = dict(input_zp=zp, output_zp=zout, output_min=-120 if op == "conv2d" else -128, output_max=top, shift_factor=sf)
        attrs.update(pad=cpad, stride=(cs, cs)) if op == "conv2d" else attrs.update(pad=pad, stride=(stride, stride))
        layers.append(w.Layer(op, [len(layers)], attrs, wt, sb))
    H, W = (H + cpad[2] + cpad[3] - k) // cs + 1, (W + cpad[0] + cpad[1] - k) // cs + 1
    oh, ow = (H + pad[2] + pad[3] - 3) // stride + 1, (W + pad[0] + pad[1] - 3) // stride + 1
    p = Program()
    h = p.conv2d(p.binding(0, x.shape), layers[0].weights, layers[0].scale_bias, nhwc_input=True, **layers[0].attrs)
    p.depthwise_conv2d(h, layers[1].weights, layers[1].scale_bias, nhwc_input=True, init=p.binding(1, (N, oh, ow, E)), **layers[1].attrs)
    return w.Workload("block_%dx%dx%dx%d_k%d_e%d_s%d" % (N, H, W, C, k, E, stride), p, [x], [((N, oh, ow, E), np.int8)], 0, 0, dict(layers=layers, nhwc=True))


def fused(device, wl):
    launched = []
    got, _ = run_on_gpu(device, wl, via="device", launched=launched)
    assert families(launched) == ["ir_expand_dw_i8"], launched
    return got


@pytest.mark.parametrize("kw", [
    dict(N=1, H=14, W=14, C=64, E=384, stride=1), dict(N=2, H=13, W=15, C=16, E=48, stride=1), dict(N=1, H=9, W=7, C=48, E=80, stride=2),
    dict(N=3, H=20, W=21, C=32, E=144, stride=2, pad=(0, 1, 0, 1)), dict(N=2, H=7, W=7, C=160, E=960, stride=1), dict(N=1, H=3, W=3, C=192, E=16, stride=1, pad=(0, 0, 0, 0)),
    dict(N=1, H=1, W=1, C=16, E=32, stride=1), dict(N=1, H=2, W=2, C=16, E=32, stride=2, pad=(0, 1, 0, 1)), dict(N=2, H=9, W=11, C=32, E=64, stride=1, pad=(2, 2, 2, 2)),
    dict(N=1, H=40, W=131, C=16, E=96, stride=1), dict(N=1, H=41, W=130, C=24 + 8, E=96, stride=2),   # several strips
    dict(N=130, H=5, W=9, C=48, E=272, stride=1), dict(N=131, H=9, W=5, C=48, E=272, stride=2), dict(N=200, H=7, W=7, C=32, E=192, stride=1),  # several images per workgroup
    dict(N=2, H=31, W=30, C=3, E=32, stride=1, first=(3, 2, (0, 1, 0, 1))), dict(N=1, H=224, W=224, C=3, E=32, stride=1, first=(3, 2, (0, 1, 0, 1))),
    dict(N=3, H=19, W=23, C=1, E=16, stride=2, first=(4, 1, (2, 1, 1, 2))), dict(N=2, H=16, W=17, C=5, E=64, stride=1, first=(3, 1, (1, 1, 1, 1))),
    dict(N=600, H=12, W=10, C=4, E=32, stride=1, first=(2, 2, (0, 0, 0, 0))),
    dict(N=1, H=12, W=12, C=32, E=48, stride=1, shift=8), dict(N=1, H=12, W=12, C=32, E=48, stride=2, shift=32),
], ids=lambda kw: "x".join(str(v) for v in kw.values()))
def test_expand_depthwise(device, kw, tmp_path):
    wl = block(**kw)
    print("[gpu-case]", wl.name, flush=True)
    want = oracle_network(wl)
    got = fused(device, wl)
    assert_bit_exact(got[0], want, wl.name)
    device.set_event_log(str(tmp_path / "log.csv"))  # a log has its records launched one by one
    try:
        got, _ = run_on_gpu(device, wl)
    finally:
        device.set_event_log(None)
    assert_bit_exact(got[0], want, wl.name + " record by record")


def test_expand_depthwise_ragged_channels(device):
    """A widened image that something else reads too, and one the depthwise kernel has its own layout for, stay two launches."""
    for kw in (dict(N=1, H=8, W=8, C=16, E=24, stride=1), dict(N=1, H=8, W=8, C=208, E=32, stride=1), dict(N=1, H=8, W=8, C=16, E=32, stride=1, shift=0)):
        wl = block(**kw)
        launched = []
        got, _ = run_on_gpu(device, wl, via="device", launched=launched)
        assert "ir_expand_dw_i8" not in families(launched), launched
        assert_bit_exact(got[0], oracle_network(wl), wl.name)


@pytest.mark.parametrize("kw", [
    dict(N=1100, H=1, W=1, C=16, E=256, stride=1), dict(N=300, H=8, W=16, C=16, E=256, stride=1), dict(N=300, H=4, W=3, C=64, E=512, stride=2),
    dict(N=300, H=4, W=3, C=80, E=512, stride=1), dict(N=2, H=5, W=64, C=32, E=64, stride=1), dict(N=1, H=3, W=128, C=16, E=32, stride=2), dict(N=1, H=6, W=129, C=16, E=32, stride=1),
    dict(N=700, H=5, W=7, C=3, E=96, stride=1, first=(3, 1, (1, 1, 1, 1))), dict(N=1, H=300, W=3, C=2, E=16, stride=1, first=(3, 1, (1, 1, 1, 1))),
], ids=lambda kw: "x".join(str(v) for v in kw.values()))
def test_expand_depthwise_walk(device, kw):
    """A tile's 128 pixels that are whole images, whole rows, a row and a bit, less than a row; images that share a workgroup."""
    wl = block(**kw)
    print("[gpu-case]", wl.name, flush=True)
    assert_bit_exact(fused(device, wl)[0], oracle_network(wl), wl.name)


@pytest.mark.parametrize("kw", [
    dict(N=300, H=8, W=8, C=16, E=256, stride=2, pad=(0, 0, 0, 0)), dict(N=256, H=14, W=14, C=96, E=576, stride=2, pad=(0, 0, 0, 0)), dict(N=300, H=7, W=7, C=16, E=256, stride=2, pad=(1, 1, 1, 0)),
    dict(N=300, H=8, W=8, C=3, E=256, stride=2, pad=(0, 0, 0, 0), first=(3, 1, (1, 1, 1, 1))), dict(N=256, H=14, W=14, C=3, E=576, stride=2, pad=(0, 0, 0, 0), first=(3, 1, (1, 1, 1, 1))),
    dict(N=300, H=7, W=7, C=3, E=256, stride=2, pad=(1, 1, 1, 0), first=(3, 1, (1, 1, 1, 1))),
], ids=lambda kw: "x".join(str(v) for v in kw.values()))
def test_rows_no_window_reaches(device, kw):
    """Several images per workgroup whose last row lies below every window."""
    wl = block(**kw)
    print("[gpu-case]", wl.name, flush=True)
    assert_bit_exact(fused(device, wl)[0], oracle_network(wl), wl.name)


@pytest.mark.parametrize("kw", [
    dict(N=1, H=9, W=10, C=32, E=48, stride=1), dict(N=1, H=11, W=3, C=16, E=32, stride=2), dict(N=1, H=5, W=65, C=16, E=32, stride=1),   # segments with fewer rows, or none
    dict(N=257, H=7, W=7, C=160, E=960, stride=1), dict(N=259, H=13, W=14, C=96, E=592, stride=1), dict(N=66, H=2, W=1, C=64, E=1040, stride=1),  # a last workgroup of fewer images
    dict(N=1, H=5, W=510, C=16, E=32, stride=1), dict(N=1, H=5, W=407, C=16, E=32, stride=2), dict(N=2, H=100, W=640, C=16, E=32, stride=2), dict(N=600, H=34, W=5, C=16, E=272, stride=1), dict(N=300, H=66, W=3, C=32, E=272, stride=2),   # the widest rows of two windows and of one, and the most LDS
    dict(N=2, H=12, W=12, C=32, E=48, stride=1, top=100), dict(N=2, H=12, W=12, C=32, E=48, stride=2, shift=41), dict(N=2, H=9, W=9, C=3, E=48, stride=1, first=(3, 1, (1, 1, 1, 1)), top=90),
], ids=lambda kw: "x".join(str(v) for v in kw.values()))
def test_expand_depthwise_lanes(device, kw):
    """Lanes that share a product but not its rows: short segments, workgroups with fewer images; results that are clamped below their type's maximum, and long shifts."""
    wl = block(**kw)
    print("[gpu-case]", wl.name, flush=True)
    assert_bit_exact(fused(device, wl)[0], oracle_network(wl), wl.name)


@pytest.mark.parametrize("kw", [
    dict(N=1, H=5, W=511, C=16, E=32, stride=1), dict(N=1, H=5, W=640, C=16, E=32, stride=1), dict(N=2, H=40, W=600, C=16, E=48, stride=1), dict(N=1, H=5, W=640, C=16, E=32, stride=2),
    dict(N=1, H=5, W=410, C=16, E=32, stride=2),
], ids=lambda kw: "x".join(str(v) for v in kw.values()))
def test_rows_too_wide_for_two_windows(device, kw):
    """Strips of one row widen most pixels again: two launches where these are ahead."""
    wl = block(**kw)
    print("[gpu-case]", wl.name, flush=True)
    launched = []
    got, _ = run_on_gpu(device, wl, via="device", launched=launched)
    assert "ir_expand_dw_i8" not in families(launched) and len(launched) == 2, launched
    assert_bit_exact(got[0], oracle_network(wl), wl.name)
