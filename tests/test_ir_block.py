"""A whole inverted-residual block as one launch: strips, blocks of columns, ragged frames and channels, the add, every first layer."""
import numpy as np
import pytest

from helpers import assert_bit_exact, families, oracle_network, run_on_gpu
from torq_compiler_amd import Program, workloads as w

pytestmark = pytest.mark.gpu


def block(N, H, W, C, E, O, stride, pad=(1, 1, 1, 1), add=None, first=None, zp=7, lowest=-128, seed=1070, steep=None):
    """widen (pointwise, or `first` = (window, stride, pad) over few channels) -> depthwise 3x3 -> narrow, and with `add` (0 or 1: the place
    of the block's input among the add's operands) the residual add; the intermediates leave no launch.  `steep`: the scale of a channel of the
    depthwise op, at 1/2 and above a shift below 32 for all of them."""
    rng = np.random.default_rng(seed)
    x = rng.integers(-128, 128, size=(N, H, W, C)).astype(np.int8)
    layers = []
    k, cs, cpad = first or (1, 1, (0, 0, 0, 0))
    for op, shape, fan, zin, zout, low in (("conv2d", (E, C, k, k), C * k * k, -3, -120, -120), ("depthwise_conv2d", (E, 1, 3, 3), 9, -120, -117, -117),
                                           ("conv2d", (O, E, 1, 1), E, -117, zp, lowest)):
        wt = rng.integers(-127, 128, size=shape).astype(np.int8)
        scales = 60 / (np.sqrt(fan) * 5400) * rng.uniform(0.8, 1.2, shape[0])
        if op == "depthwise_conv2d" and steep is not None:
            scales[shape[0] // 2] = steep
        mult, sh = w.quantize_multiplier(scales)
        sb, sf = w.derive_scale_bias(mult, sh, rng.integers(-4000, 4000, shape[0]), wt, zin)
        attrs = dict(input_zp=zin, output_zp=zout, output_min=low, output_max=127, shift_factor=sf)
        attrs.update(pad=(0, 0, 0, 0), stride=(1, 1))
        if len(layers) == 0:
            attrs.update(pad=cpad, stride=(cs, cs))
        elif len(layers) == 1:
            attrs.update(pad=pad, stride=(stride, stride))
        layers.append(w.Layer(op, [len(layers)], attrs, wt, sb))
    if add is not None:
        wts, sb, sf = w.add_params(0.7, 0.6, *((-3, zp) if add == 0 else (zp, -3)))
        layers.append(w.Layer("add", [0, 3] if add == 0 else [3, 0], dict(output_zp=4, output_min=-128, output_max=127, shift_factor=sf), wts, sb))
    H, W = (H + cpad[2] + cpad[3] - k) // cs + 1, (W + cpad[0] + cpad[1] - k) // cs + 1
    oh, ow = (H + pad[2] + pad[3] - 3) // stride + 1, (W + pad[0] + pad[1] - 3) // stride + 1
    p = Program()
    values = [p.binding(0, x.shape)]
    out = p.binding(1, (N, oh, ow, O))
    for i, L in enumerate(layers):
        src = [values[j] for j in L.inputs]
        init = dict(init=out) if i + 1 == len(layers) else {}
        if L.op == "add":
            values.append(p.add(src[0], src[1], L.weights, L.scale_bias, **L.attrs, **init))
        else:
            values.append(getattr(p, L.op)(src[0], L.weights, L.scale_bias, nhwc_input=True, **L.attrs, **init))
    return w.Workload("block_%dx%dx%dx%d_k%d_e%d_o%d_s%d" % (N, H, W, C, k, E, O, stride), p, [x], [((N, oh, ow, O), np.int8)], 0, 0, dict(layers=layers, nhwc=True))


CASES = [
    dict(N=1, H=28, W=28, C=32, E=192, O=32, stride=1, add=0), dict(N=2, H=56, W=56, C=32, E=144, O=32, stride=1, add=1), dict(N=1, H=14, W=14, C=96, E=576, O=96, stride=1, add=0),
    dict(N=2, H=14, W=14, C=64, E=384, O=96, stride=1), dict(N=1, H=112, W=112, C=16, E=96, O=32, stride=2, pad=(0, 1, 0, 1)), dict(N=3, H=28, W=28, C=32, E=192, O=64, stride=2, pad=(0, 1, 0, 1)),
    dict(N=1, H=13, W=15, C=16, E=48, O=48, stride=1), dict(N=1, H=9, W=7, C=48, E=80, O=80, stride=2), dict(N=2, H=1, W=1, C=16, E=32, O=16, stride=1), dict(N=1, H=2, W=2, C=16, E=16, O=16, stride=2, pad=(0, 1, 0, 1)),
    dict(N=1, H=9, W=11, C=32, E=64, O=48, stride=1, pad=(2, 2, 2, 2)), dict(N=1, H=3, W=5, C=64, E=64, O=64, stride=1, pad=(0, 0, 0, 0)),
    # the widest rows
    dict(N=1, H=6, W=64, C=16, E=48, O=16, stride=1, add=0), dict(N=1, H=23, W=128, C=16, E=96, O=32, stride=2), dict(N=2, H=9, W=127, C=32, E=32, O=32, stride=2), dict(N=1, H=12, W=63, C=80, E=48, O=80, stride=1),
    # first layers, in blocks of columns too (65, 112, 130 wide)
    dict(N=1, H=9, W=130, C=3, E=32, O=16, stride=1, first=(3, 2, (0, 1, 0, 1))), dict(N=1, H=11, W=130, C=3, E=16, O=32, stride=1, first=(3, 1, (1, 1, 1, 1))), dict(N=2, H=11, W=140, C=2, E=32, O=32, stride=2, first=(3, 1, (1, 1, 1, 1))),
    dict(N=2, H=31, W=30, C=3, E=32, O=16, stride=1, first=(3, 2, (0, 1, 0, 1))), dict(N=1, H=224, W=224, C=3, E=32, O=16, stride=1, first=(3, 2, (0, 1, 0, 1))),
    dict(N=3, H=19, W=23, C=1, E=16, O=32, stride=2, first=(4, 1, (2, 1, 1, 2))), dict(N=2, H=16, W=17, C=5, E=32, O=16, stride=1, first=(3, 1, (1, 1, 1, 1))), dict(N=5, H=12, W=10, C=4, E=32, O=16, stride=1, first=(2, 2, (0, 0, 0, 0))),
    # a clamp in the narrow convolution, a zero point at its end, one output row a strip
    dict(N=1, H=20, W=21, C=32, E=64, O=32, stride=1, zp=-128), dict(N=40, H=5, W=64, C=16, E=32, O=32, stride=1, lowest=-20), dict(N=700, H=7, W=9, C=16, E=96, O=16, stride=1, add=1),
]


@pytest.mark.parametrize("kw", CASES, ids=lambda kw: "x".join(str(v) for v in kw.values()))
def test_block(device, kw, monkeypatch):
    monkeypatch.setenv("THIP_IR_BLOCK", "1")
    wl = block(**kw)
    print("[gpu-case]", wl.name, flush=True)
    launched = []
    got, _ = run_on_gpu(device, wl, via="device", launched=launched)
    assert families(launched) == ["ir_block_i8"], launched
    assert_bit_exact(got[0], oracle_network(wl), wl.name)


@pytest.mark.parametrize("kw", CASES, ids=lambda kw: "x".join(str(v) for v in kw.values()))
@pytest.mark.parametrize("steep", [0.6, 100.0])
def test_block_with_a_steep_channel(device, kw, steep, monkeypatch):
    """The kernel's other depthwise requant, of a shift below 32 for all channels."""
    monkeypatch.setenv("THIP_IR_BLOCK", "1")
    wl = block(steep=steep, **kw)
    print("[gpu-case]", wl.name, steep, flush=True)
    launched = []
    got, _ = run_on_gpu(device, wl, via="device", launched=launched)
    assert len(launched) == 1 and launched[0].startswith("ir_block_i8<") and launched[0].endswith(",3>"), launched
    assert_bit_exact(got[0], oracle_network(wl), wl.name)


def test_large_batches_take_it(device):
    """By the rule, without the switch: a batch that fills the chip, and one image that does not."""
    for n, kernels in ((200, ["ir_block_i8"]), (1, ["ir_expand_dw_i8"])):
        wl = block(N=n, H=28, W=28, C=32, E=192, O=32, stride=1)
        launched = []
        got, _ = run_on_gpu(device, wl, via="device", launched=launched)
        assert families(launched)[:1] == kernels, launched
        assert_bit_exact(got[0], oracle_network(wl), wl.name)


def test_other_requants_stay_apart(device, monkeypatch):
    """Records without the packed tail (a maximum below 127, a shift above what it takes) keep the launches of their own."""
    monkeypatch.setenv("THIP_IR_BLOCK", "1")
    for op, attr, value in ((0, "output_max", 100), (1, "output_max", 90), (2, "output_max", 60), (1, "shift_factor", 41)):
        wl = block(N=1, H=8, W=8, C=16, E=32, O=16, stride=1)
        L = wl.attrs["layers"]
        L[op].attrs[attr] = value
        p = Program()
        h = p.conv2d(p.binding(0, (1, 8, 8, 16)), L[0].weights, L[0].scale_bias, nhwc_input=True, **L[0].attrs)
        h = p.depthwise_conv2d(h, L[1].weights, L[1].scale_bias, nhwc_input=True, **L[1].attrs)
        p.conv2d(h, L[2].weights, L[2].scale_bias, nhwc_input=True, init=p.binding(1, (1, 8, 8, 16)), **L[2].attrs)
        wl.program = p
        launched = []
        got, _ = run_on_gpu(device, wl, via="device", launched=launched)
        assert "ir_block_i8" not in families(launched), launched
        assert_bit_exact(got[0], oracle_network(wl), wl.name)


@pytest.mark.parametrize("N", [1, 3])
@pytest.mark.parametrize("H,W,C,first", [(13, 71, 4, (4, 1, (3, 3, 3, 3))), (13, 70, 3, (4, 1, (0, 3, 3, 0))), (9, 40, 1, (3, 1, (2, 2, 2, 2))), (8, 35, 5, (3, 2, (2, 1, 0, 2))), (40, 150, 3, (3, 2, (1, 1, 1, 1))),
                                         (5, 3, 4, (4, 1, (3, 3, 3, 3)))])
def test_padding_of_a_first_layer(device, N, H, W, C, first, monkeypatch):
    """Runs that begin or end in the padding at every byte of their dwords, in the first, the last and an inner image."""
    monkeypatch.setenv("THIP_IR_BLOCK", "1")
    wl = block(N, H, W, C, 32, 16, 1, first=first)
    print("[gpu-case]", wl.name, flush=True)
    launched = []
    got, _ = run_on_gpu(device, wl, via="device", launched=launched)
    assert families(launched) == ["ir_block_i8"], launched
    assert_bit_exact(got[0], oracle_network(wl), wl.name)
