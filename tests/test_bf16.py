"""bf16 rows of fully_connected / matmul: the oracle's pins, the emitter, and (on a GPU) the kernel, which is a
tolerance row: at most one bf16 ULP from the oracle per element."""
import os

import numpy as np
import pytest

import desc_interp
from helpers import assert_bf16_close, assert_bit_exact, bf16_ordered, families, oracle_eval, run_on_gpu
from oracle import oracle as orc
from torq_compiler_amd import Executable, Program, ThipError, runtime, workloads as w


# ---- oracle pins ---------------------------------------------------------------------------------
def test_bf16_conversion_matches_torch_and_is_nearest_even():
    import torch
    rng = np.random.default_rng(1)
    vals = np.concatenate([rng.standard_normal(5000).astype(np.float32) * 10.0 ** rng.integers(-30, 30, 5000),
                           np.array([0.0, -0.0, 1.0, 1.00390625, 1.01171875, 3.3e38, -3.4e38, 1e-40, np.inf, -np.inf], dtype=np.float32)])
    got = orc.to_bf16(vals)
    want = torch.tensor(vals).to(torch.bfloat16).view(torch.int16).numpy().astype(np.uint16)
    assert np.array_equal(got, want)
    # ties: 1 + 2^-8 is exactly between 1 and 1 + 2^-7 -> even mantissa (1.0); 1 + 3*2^-8 -> 1 + 2^-6
    assert orc.to_bf16(np.float32(1 + 2.0 ** -8)) == 0x3f80 and orc.to_bf16(np.float32(1 + 3 * 2.0 ** -8)) == 0x3f82
    assert np.array_equal(orc.from_bf16(got[:5000]).view(np.uint32) & 0xffff, np.zeros(5000, dtype=np.uint32))
    assert np.isnan(orc.from_bf16(orc.to_bf16(np.float32(np.nan))))


def test_bf16_fully_connected_closed_forms():
    # small integers: every product and sum is exact, so the result is the integer matmul plus the bias
    rng = np.random.default_rng(2)
    xi, wi = rng.integers(-8, 9, size=(5, 24)), rng.integers(-8, 9, size=(7, 24))
    bias = rng.integers(-4, 5, size=7).astype(np.float32)
    out = orc.fully_connected_bf16(orc.to_bf16(xi), orc.to_bf16(wi), bias)
    want = (xi @ wi.T + bias).astype(np.float32)
    assert np.array_equal(out, orc.to_bf16(want))
    # clamp to [0, 6] (a ReLU6) with float bit patterns; bias only, no scale
    out = orc.fully_connected_bf16(orc.to_bf16(xi), orc.to_bf16(wi), bias, output_min=w.float_bits(0.0), output_max=w.float_bits(6.0))
    assert np.array_equal(out, orc.to_bf16(np.clip(want, 0.0, 6.0)))
    # a transposed operand or a dropped bias would show
    assert not np.array_equal(orc.fully_connected_bf16(orc.to_bf16(xi), orc.to_bf16(wi), 0 * bias), orc.to_bf16(want))


def test_bf16_oracle_against_float64():
    rng = np.random.default_rng(3)
    for M, K, N in [(3, 64, 5), (9, 1152, 33), (2, 6912, 8)]:
        x, wt = orc.to_bf16(rng.standard_normal((M, K))), orc.to_bf16(rng.standard_normal((N, K)) / np.sqrt(K))
        bias = rng.standard_normal(N).astype(np.float32)
        got = orc.fully_connected_bf16(x, wt, bias)
        exact = orc.from_bf16(x).astype(np.float64) @ orc.from_bf16(wt).astype(np.float64).T + bias
        assert_bf16_close(got, orc.to_bf16(exact.astype(np.float32)), "fp32 accumulate vs float64")
        # matmul is the same arithmetic with input2 = weights^T and one bias
        mm = orc.matmul_bf16(x, np.ascontiguousarray(wt.T), np.array([0.25], dtype=np.float32))
        fc = orc.fully_connected_bf16(x, wt, np.full(N, 0.25, dtype=np.float32))
        assert np.array_equal(mm.reshape(M, N), fc)


def test_bf16_matmul_batches_broadcast():
    rng = np.random.default_rng(4)
    a, b = orc.to_bf16(rng.standard_normal((4, 3, 16))), orc.to_bf16(rng.standard_normal((1, 16, 10)))
    out = orc.matmul_bf16(a, b, np.zeros(1, dtype=np.float32))
    for i in range(4):
        assert np.array_equal(out[i], orc.matmul_bf16(a[i], b[0], np.zeros(1, dtype=np.float32))[0])


def test_bf16_conv_oracle_pins():
    """conv2d / depthwise_conv2d on bf16: exact on small integers (vs an integer convolution), within one bf16 ULP of
    torch's float64 convolution on random data, both layouts, asymmetric padding and strides."""
    import torch
    import torch.nn.functional as F
    rng = np.random.default_rng(7)
    for (N, C, H, W, O, KH, KW, pad, stride) in [(2, 5, 9, 8, 6, 3, 3, (1, 0, 2, 1), (2, 1)), (1, 8, 7, 7, 4, 1, 1, (0, 0, 0, 0), (1, 1)),
                                                 (1, 3, 12, 10, 7, 5, 2, (0, 1, 2, 2), (3, 2))]:
        xi = rng.integers(-6, 7, size=(N, C, H, W))
        wi = rng.integers(-6, 7, size=(O, C, KH, KW))
        bi = rng.integers(-9, 10, size=O).astype(np.float32)
        padded = F.pad(torch.tensor(xi, dtype=torch.float64), (pad[0], pad[1], pad[2], pad[3]))
        want = F.conv2d(padded, torch.tensor(wi, dtype=torch.float64), torch.tensor(bi, dtype=torch.float64), stride=stride).numpy()
        got = orc.conv2d_bf16(orc.to_bf16(xi), orc.to_bf16(wi), bi, pad=pad, stride=stride)
        assert np.array_equal(got, orc.to_bf16(want.astype(np.float32)))
        nhwc = orc.conv2d_bf16(orc.to_bf16(xi.transpose(0, 2, 3, 1)), orc.to_bf16(wi), bi, pad=pad, stride=stride, layout=orc.NHWC)
        assert np.array_equal(nhwc.transpose(0, 3, 1, 2), got)
        x = orc.to_bf16(rng.standard_normal((N, C, H, W)))
        wt = orc.to_bf16(rng.standard_normal((O, C, KH, KW)) / np.sqrt(C * KH * KW))
        b = rng.standard_normal(O).astype(np.float32)
        padded = F.pad(torch.tensor(orc.from_bf16(x), dtype=torch.float64), (pad[0], pad[1], pad[2], pad[3]))
        exact = F.conv2d(padded, torch.tensor(orc.from_bf16(wt), dtype=torch.float64), torch.tensor(b, dtype=torch.float64), stride=stride).numpy()
        got = orc.conv2d_bf16(x, wt, b, pad=pad, stride=stride, output_min=w.float_bits(-0.5), output_max=w.float_bits(1.0))
        assert_bf16_close(got, orc.to_bf16(np.clip(exact, -0.5, 1.0).astype(np.float32)), "conv2d bf16 vs float64")
        # depthwise = grouped convolution with one input channel per group
        wd = orc.to_bf16(rng.standard_normal((C, 1, KH, KW)) / np.sqrt(KH * KW))
        bd = rng.standard_normal(C).astype(np.float32)
        exact = F.conv2d(padded, torch.tensor(orc.from_bf16(wd), dtype=torch.float64), torch.tensor(bd, dtype=torch.float64), stride=stride, groups=C).numpy()
        got = orc.depthwise_conv2d_bf16(x, wd, bd, pad=pad, stride=stride)
        assert_bf16_close(got, orc.to_bf16(exact.astype(np.float32)), "depthwise bf16 vs float64")


def test_bf16_avg_pool_and_expand_weights_oracle_pins():
    """Global average pool: exact on small integers with a power-of-two weight, within one ULP of the float64 mean.
    expand_weights: exact when scale and bias are small integers (and equal to (w - zp) * scale, the dequantisation the
    op stands for), within one ULP of float64 otherwise, clamp, padded bias rows."""
    rng = np.random.default_rng(11)
    xi = rng.integers(-8, 9, size=(3, 4, 4, 10))
    got = orc.avg_pool2d_bf16(orc.to_bf16(xi), orc.to_bf16(np.array([1.0 / 16])), np.array([2.0], dtype=np.float32))
    assert np.array_equal(got.reshape(3, 10), orc.to_bf16((xi.sum(axis=(1, 2)) / 16.0 + 2.0).astype(np.float32)))
    x = orc.to_bf16(rng.standard_normal((2, 7, 7, 33)) + 0.5)
    wt = orc.to_bf16(np.array([1.0 / 49]))
    exact = orc.from_bf16(x).astype(np.float64).sum(axis=(1, 2)) * float(orc.from_bf16(wt)[0])
    got = orc.avg_pool2d_bf16(x, wt, np.zeros(1, dtype=np.float32), output_min=w.float_bits(0.0), output_max=w.float_bits(0.75))
    mag = np.abs(orc.from_bf16(x).astype(np.float64)).sum(axis=(1, 2)) * float(orc.from_bf16(wt)[0])
    assert_bf16_close(got.reshape(2, 33), orc.to_bf16(np.clip(exact, 0.0, 0.75).astype(np.float32)), "avgpool bf16 vs float64", magnitude=mag)

    K, N, block = 64, 10, 32
    wq = rng.integers(-128, 128, size=(K, N), dtype=np.int8)
    sci = rng.integers(1, 4, size=(2, N))
    zp = rng.integers(-5, 6, size=(2, N))
    qb = np.zeros((2, N + 2), dtype=np.float32)
    qb[:, :N] = -zp * sci
    got = orc.expand_weights(wq, orc.to_bf16(sci), qb, block_size=block)
    want = (wq.astype(np.int64) - np.repeat(zp, block, axis=0)) * np.repeat(sci, block, axis=0)
    assert np.array_equal(got, orc.to_bf16(want.astype(np.float32)))
    sc = orc.to_bf16(rng.uniform(0.001, 0.02, size=(2, N)))
    qb = rng.standard_normal((2, N)).astype(np.float32)
    exact = wq.astype(np.float64) * np.repeat(orc.from_bf16(sc).astype(np.float64), block, axis=0) + np.repeat(qb.astype(np.float64), block, axis=0)
    got = orc.expand_weights(wq, sc, qb, block_size=block, output_min=w.float_bits(-1.0), output_max=w.float_bits(1.5))
    assert_bf16_close(got, orc.to_bf16(np.clip(exact, -1.0, 1.5).astype(np.float32)), "expand_weights vs float64", magnitude=np.abs(exact) + 1)


def test_bf16_add_closed_forms():
    # weights 1 and -1 on equal inputs cancel exactly: the bias alone remains; small integers are exact
    rng = np.random.default_rng(6)
    x = orc.to_bf16(rng.standard_normal(1000))
    out = orc.add_bf16(x, x, orc.to_bf16(np.array([1.0, -1.0], dtype=np.float32)), np.array([0.375], dtype=np.float32))
    assert np.array_equal(out, np.full(1000, orc.to_bf16(np.float32(0.375)), dtype=np.uint16))
    ai, bi = rng.integers(-20, 21, size=500), rng.integers(-20, 21, size=500)
    out = orc.add_bf16(orc.to_bf16(ai), orc.to_bf16(bi), orc.to_bf16(np.array([2.0, 3.0], dtype=np.float32)), np.array([-1.0], dtype=np.float32),
                       output_min=w.float_bits(-10.0), output_max=w.float_bits(40.0))
    assert np.array_equal(out, orc.to_bf16(np.clip(2.0 * ai + 3.0 * bi - 1.0, -10.0, 40.0).astype(np.float32)))
    # against float64 on random data: one bf16 step at most (two fp32 roundings before the bf16 one)
    a, b = orc.to_bf16(rng.standard_normal(4000)), orc.to_bf16(rng.standard_normal(4000))
    wts = orc.to_bf16(np.array([0.7, 1.3], dtype=np.float32))
    got = orc.add_bf16(a, b, wts, np.array([0.1], dtype=np.float32))
    wf = orc.from_bf16(wts).astype(np.float64)
    exact = orc.from_bf16(a).astype(np.float64) * wf[0] + orc.from_bf16(b).astype(np.float64) * wf[1] + np.float64(np.float32(0.1))
    assert_bf16_close(got, orc.to_bf16(exact.astype(np.float32)), "bf16 add vs float64")


# ---- emitter ------------------------------------------------------------------------------------------
@pytest.mark.parametrize("make", [lambda: w.fully_connected_bf16_workload(5, 64, 40), lambda: w.fully_connected_bf16_workload(33, 1152, 7, clamp=(-0.5, 0.75)),
                                  lambda: w.matmul_bf16_workload(4, 1, 256, 96, batch2=False), lambda: w.matmul_bf16_workload(3, 2, 64, 24),
                                  lambda: w.matmul_bf16_workload(1, 6, 32, 20, batch1=False, batch2=False, constant_rhs=True, bias=0.5),
                                  lambda: w.matmul_bf16_workload(2, 5, 16, 12, batch1=False, constant_rhs=True),
                                  lambda: w.conv2d_bf16_workload(), lambda: w.conv2d_bf16_workload(N=2, H=9, W=11, C=5, O=7, KH=2, KW=3, stride=(2, 1), pad=(0, 2, 1, 0), nhwc=False),
                                  lambda: w.conv2d_bf16_workload(N=2, H=6, W=6, C=16, O=40, KH=1, KW=1, pad=(0, 0, 0, 0)),
                                  lambda: w.conv2d_bf16_workload(depthwise=True, C=12, stride=(2, 2), pad=(0, 1, 0, 1), clamp=(-0.5, 0.5)),
                                  lambda: w.conv2d_bf16_workload(depthwise=True, N=2, C=5, H=7, W=9, nhwc=False),
                                  lambda: w.avg_pool2d_bf16_workload(), lambda: w.avg_pool2d_bf16_workload(N=3, H=5, W=4, C=7, weight=1.0, clamp=(-1.0, 1.0)),
                                  lambda: w.expand_weights_workload(), lambda: w.expand_weights_workload(M=70, K=128, N=40, block=64, clamp=(-2.0, 2.0)),
                                  lambda: w.expand_weights_workload(M=3, K=96, N=20, block=48, bias_pad=2),
                                  lambda: w.expand_weights_workload(M=2, K=64, N=33, fold=False, expand_clamp=(-0.01, 0.02), bias_pad=1),
                                  lambda: w.add_bf16_workload(), lambda: w.add_bf16_workload((3, 5, 7), 0.5, -1.25, 0.125, clamp=(-1.0, 2.0))])
def test_bf16_descriptor(make):
    wl = make()
    outs = [np.zeros(s, dtype=dt) for s, dt in wl.outputs]
    d = desc_interp.run(wl.program.serialize(), list(wl.inputs) + outs)
    for got, want in zip(outs, oracle_eval(wl)):
        assert_bit_exact(got, want.reshape(got.shape), wl.name)
    kinds = [int(o["kind"]) for o in d.ops]
    assert {desc_interp.K_FC_BF16, desc_interp.K_ADD_BF16, desc_interp.K_DW_BF16, desc_interp.K_AVGPOOL_BF16} & set(kinds)


def test_expand_weights_folding():
    """An expansion that only feeds a bf16 matmul emits no kernel: few rows take the int8 weights (layout 2), many rows
    or a block size the kernel does not take get weights expanded at serialisation; an expansion that is also an
    output, or THIP_NO_EXPAND_FOLD, stays a kernel of its own followed by the transpose of a run-time input2."""
    def kinds_loader(wl):
        d = desc_interp.Descriptor(wl.program.serialize())
        return [int(o["kind"]) for o in d.ops], [int(o["loader"]) for o in d.ops if int(o["kind"]) == desc_interp.K_FC_BF16]

    assert kinds_loader(w.expand_weights_workload()) == ([desc_interp.K_FC_BF16], [2])
    assert kinds_loader(w.expand_weights_workload(M=70, K=128, N=40, block=64)) == ([desc_interp.K_FC_BF16], [1])
    assert kinds_loader(w.expand_weights_workload(M=3, K=96, N=20, block=48)) == ([desc_interp.K_FC_BF16], [1])
    kinds, loaders = kinds_loader(w.expand_weights_workload(fold=False))
    assert kinds == [desc_interp.K_EXPAND, desc_interp.K_TRANSPOSE, desc_interp.K_FC_BF16] and loaders == [0]
    os.environ["THIP_NO_EXPAND_FOLD"] = "1"
    try:
        kinds, _ = kinds_loader(w.expand_weights_workload())
    finally:
        del os.environ["THIP_NO_EXPAND_FOLD"]
    assert kinds == [desc_interp.K_EXPAND, desc_interp.K_TRANSPOSE, desc_interp.K_FC_BF16]


def test_bf16_rejections():
    def expect(code, build):
        p = Program()
        with pytest.raises(ThipError) as e:
            build(p)
            p.serialize()
        assert e.value.code == code, e.value

    wt = np.zeros((8, 16), dtype=np.uint16)
    bias = np.zeros(8, dtype=np.float32)
    ok = dict(output_zp=0, output_min=w.NO_CLAMP[0], output_max=w.NO_CLAMP[1], shift_factor=0, input_zp=0)
    expect(runtime.INVALID_ARGUMENT, lambda p: p.fully_connected(p.binding(0, (2, 16), np.uint16), wt, bias, init=p.binding(1, (2, 8), np.uint16), **dict(ok, shift_factor=3)))
    expect(runtime.INVALID_ARGUMENT, lambda p: p.fully_connected(p.binding(0, (2, 16), np.uint16), wt, bias, init=p.binding(1, (2, 8), np.uint16), **dict(ok, output_zp=1)))
    expect(runtime.INVALID_ARGUMENT, lambda p: p.fully_connected(p.binding(0, (2, 16), np.uint16), wt, bias[:4], init=p.binding(1, (2, 8), np.uint16), **ok))
    expect(runtime.UNIMPLEMENTED, lambda p: p.fully_connected(p.binding(0, (2, 12), np.uint16), wt[:, :12].copy(), bias, init=p.binding(1, (2, 8), np.uint16), **ok))
    # int8 weights under a bf16 input
    expect(runtime.INVALID_ARGUMENT, lambda p: p.fully_connected(p.binding(0, (2, 16), np.uint16), np.zeros((8, 16), dtype=np.int8), bias, init=p.binding(1, (2, 8), np.uint16), **ok))


# ---- GPU ------------------------------------------------------------------------------------------------
def _magnitude(wl):
    """Per output element: sum of |x * w| + |bias|, what the fp32 rounding errors scale with."""
    f = lambda bits: np.abs(orc.from_bf16(bits).astype(np.float64))
    if wl.name.startswith("fcbf16"):
        return f(wl.inputs[0]) @ f(wl.attrs["weights"]).T + np.abs(wl.attrs["bias"])
    return np.matmul(f(wl.inputs[0]), f(wl.attrs["input2"])) + abs(float(wl.attrs["bias"][0]))


def _check_gpu(device, wl, via="host"):
    print("[gpu-case]", wl.name, flush=True)
    got, kernels = run_on_gpu(device, wl, via=via)
    assert_bf16_close(got[0], oracle_eval(wl)[0], wl.name + " (gpu)", magnitude=_magnitude(wl))
    assert any("fc_bf16" in k for k in kernels), kernels
    return got[0]


@pytest.mark.gpu
def test_gpu_bf16_fully_connected(device):
    """Decoder linear shapes at 1 and 32 tokens, ragged M / N / K, a clamp; exact on small integers."""
    for M, K, N in [(1, 1152, 1024), (32, 1152, 256), (1, 1152, 6912), (32, 6912, 1152), (5, 64, 40), (33, 1152, 7), (70, 24, 130), (3, 8, 2)]:
        _check_gpu(device, w.fully_connected_bf16_workload(M, K, N))
    _check_gpu(device, w.fully_connected_bf16_workload(9, 200, 44, clamp=(-0.25, 0.5)), via="device")
    rng = np.random.default_rng(5)
    xi, wi = rng.integers(-8, 9, size=(6, 48)), rng.integers(-8, 9, size=(20, 48))
    bias = rng.integers(-4, 5, size=20).astype(np.float32)
    p = Program()
    p.fully_connected(p.binding(0, (6, 48), np.uint16), w.to_bf16(wi), bias, init=p.binding(1, (6, 20), np.uint16), output_zp=0,
                      output_min=w.NO_CLAMP[0], output_max=w.NO_CLAMP[1], shift_factor=0, input_zp=0)
    exe = Executable(device, p.serialize())
    out = np.zeros((6, 20), dtype=np.uint16)
    exe.run_host([w.to_bf16(xi), out])
    exe.close()
    assert_bit_exact(out, w.to_bf16((xi @ wi.T + bias).astype(np.float32)), "exact small integers")


@pytest.mark.gpu
def test_gpu_bf16_conv2d_and_depthwise(device):
    """conv2d as patch matrix + GEMM (tolerance row), pointwise conv2d straight on the image, depthwise (same order of
    fp32 operations as the oracle: bit-exact), N,C,H,W bindings through the 16-bit transpose."""
    for wl in [w.conv2d_bf16_workload(), w.conv2d_bf16_workload(N=2, H=9, W=11, C=5, O=7, KH=2, KW=3, stride=(2, 1), pad=(0, 2, 1, 0), nhwc=False),
               w.conv2d_bf16_workload(N=2, H=28, W=28, C=32, O=64, KH=1, KW=1, pad=(0, 0, 0, 0)),
               w.conv2d_bf16_workload(N=1, H=56, W=56, C=24, O=48, stride=(2, 2), pad=(0, 1, 0, 1), clamp=(0.0, 6.0))]:
        print("[gpu-case]", wl.name, flush=True)
        got, kernels = run_on_gpu(device, wl)
        f = lambda bits: np.abs(orc.from_bf16(bits).astype(np.float64))
        # sum of |products| per output: a convolution of magnitudes (through the oracle's own loop nest in float64 is
        # overkill; bound it by |x|max * sum|w| + |b|)
        wabs = f(wl.attrs["weights"]).reshape(wl.attrs["weights"].shape[0], -1).sum(axis=1) * f(wl.inputs[0]).max() + np.abs(wl.attrs["bias"])
        shape = [1, 1, 1, 1]
        shape[3 if wl.attrs["nhwc"] else 1] = -1
        assert_bf16_close(got[0], oracle_eval(wl)[0], wl.name + " (gpu)", magnitude=np.broadcast_to(wabs.reshape(shape), got[0].shape))
        assert "fc_bf16" in families(kernels)
    for wl in [w.conv2d_bf16_workload(depthwise=True, C=12, stride=(2, 2), pad=(0, 1, 0, 1), clamp=(-0.5, 0.5)),
               w.conv2d_bf16_workload(depthwise=True, N=2, C=5, H=7, W=9, nhwc=False),
               w.conv2d_bf16_workload(depthwise=True, N=4, C=144, H=56, W=56)]:
        print("[gpu-case]", wl.name, flush=True)
        got, kernels = run_on_gpu(device, wl, via="device")
        assert_bit_exact(got[0], oracle_eval(wl)[0], wl.name)
        assert "depthwise_bf16" in families(kernels)


@pytest.mark.gpu
def test_gpu_bf16_wide_n(device):
    """A vocabulary-sized N with a short K: every wave streams its own columns through two register buffers
    (bf16 weights, block-quantized weights with and without the expansion clamp, ragged N and K, two row tiles)."""
    for wl in [w.fully_connected_bf16_workload(3, 200, 32800), w.fully_connected_bf16_workload(40, 1152, 32768, clamp=(-0.5, 0.75))]:
        _check_gpu(device, wl, via="device")
    f = lambda bits: np.abs(orc.from_bf16(bits).astype(np.float64))
    for wl in [w.expand_weights_workload(M=5, K=192, N=32808, block=64), w.expand_weights_workload(M=33, K=1152, N=32768, block=128),
               w.expand_weights_workload(M=2, K=320, N=32768, block=32, expand_clamp=(-0.002, 0.003))]:
        print("[gpu-case]", wl.name, flush=True)
        got, kernels = run_on_gpu(device, wl, via="device")
        w16 = orc.expand_weights(wl.attrs["weights"], wl.attrs["scale"], wl.attrs["qbias"], block_size=wl.attrs["block"],
                                 output_min=wl.attrs["expand_min"], output_max=wl.attrs["expand_max"])
        assert_bf16_close(got[0], oracle_eval(wl)[0].reshape(got[0].shape), wl.name + " (gpu)", magnitude=f(wl.inputs[0]) @ f(w16))
        assert families(kernels) == ["fc_bf16_wide"], kernels  # >= 1024 column blocks, short K: every wave streams its own columns


@pytest.mark.gpu
@pytest.mark.parametrize("K,N,M", [(64, 32768 * 5 + 33, 1), (128, 32768 * 9 + 1, 3), (192, 32768 * 4 + 63, 33), (512, 32768 * 5, 40)])
@pytest.mark.parametrize("scaled", [False, True])
def test_gpu_bf16_wide_n_rounds(device, K, N, M, scaled):
    """More columns than the chip's blocks make at a time: waves with one set of columns more than others, an odd and an even number of
    loads per set, one of fewer steps than a load takes; rows of a last block that is not full."""
    wl = w.expand_weights_workload(M=M, K=K, N=N, block=64) if scaled else w.fully_connected_bf16_workload(M, K, N, clamp=(-0.5, 0.75) if M == 3 else None)
    print("[gpu-case]", wl.name, flush=True)
    got, kernels = run_on_gpu(device, wl, via="device")
    assert families(kernels) == ["fc_bf16_wide"], kernels
    f = lambda bits: np.abs(orc.from_bf16(bits).astype(np.float64))
    w16 = orc.expand_weights(wl.attrs["weights"], wl.attrs["scale"], wl.attrs["qbias"], block_size=64, output_min=wl.attrs["expand_min"], output_max=wl.attrs["expand_max"]) if scaled else wl.attrs["weights"]
    magnitude = f(wl.inputs[0]) @ (f(w16) if f(w16).shape[0] == K else f(w16).T)
    assert_bf16_close(got[0], oracle_eval(wl)[0].reshape(got[0].shape), wl.name + " (gpu)", magnitude=magnitude)


@pytest.mark.gpu
@pytest.mark.parametrize("waves", [4, 8, 16])
def test_gpu_bf16_wide_n_waves_per_block(device, waves, monkeypatch):
    """The waves of a block share its input rows in LDS: four, eight or sixteen of them, every one with columns of its
    own; the last block has waves without columns."""
    monkeypatch.setenv("THIP_FC_WIDE_WAVES", str(waves))
    for wl, label in [(w.fully_connected_bf16_workload(33, 200, 32800 + 96), "fc_bf16_wide<0,2,%d>" % waves),
                      (w.expand_weights_workload(M=7, K=320, N=32768 + 160, block=64), "fc_bf16_wide<1,4,%d>" % waves),
                      (w.expand_weights_workload(M=40, K=192, N=32768, block=32, expand_clamp=(-0.002, 0.003)), "fc_bf16_wide<2,4,%d>" % waves)]:
        print("[gpu-case]", wl.name, flush=True)
        got, kernels = run_on_gpu(device, wl, via="device")
        if "qbias" in wl.attrs:
            f = lambda bits: np.abs(orc.from_bf16(bits).astype(np.float64))
            w16 = orc.expand_weights(wl.attrs["weights"], wl.attrs["scale"], wl.attrs["qbias"], block_size=wl.attrs["block"],
                                     output_min=wl.attrs["expand_min"], output_max=wl.attrs["expand_max"])
            magnitude = f(wl.inputs[0]) @ f(w16)
        else:
            magnitude = _magnitude(wl)
        assert_bf16_close(got[0], oracle_eval(wl)[0].reshape(got[0].shape), wl.name + " (gpu)", magnitude=magnitude)
        assert label in kernels, (label, kernels)


@pytest.mark.gpu
def test_gpu_bf16_avg_pool(device):
    """The kernel walks the frame in the oracle's order: bit-exact."""
    for wl in [w.avg_pool2d_bf16_workload(), w.avg_pool2d_bf16_workload(N=64), w.avg_pool2d_bf16_workload(N=3, H=5, W=4, C=7, weight=1.0, clamp=(-1.0, 1.0)),
               w.avg_pool2d_bf16_workload(N=1, H=14, W=14, C=96, weight=0.0078125)]:
        print("[gpu-case]", wl.name, flush=True)
        got, kernels = run_on_gpu(device, wl, via="device")
        assert_bit_exact(got[0], oracle_eval(wl)[0], wl.name)
        assert families(kernels) == ["avgpool_bf16"]


@pytest.mark.gpu
def test_gpu_expand_weights(device):
    """Block-quantized weights: expanded in registers by the matmul (decoder shapes at 1 and 32 tokens, split K, ragged
    N, an expansion clamp), by the grouped decode kernel where its shape rules hold (blocks of a multiple of 128 rows, N a
    multiple of 16, at most 32 rows), expanded at serialisation (many rows), and as a kernel of its own, whose result is bit-exact."""
    f = lambda bits: np.abs(orc.from_bf16(bits).astype(np.float64))
    cases = [(w.expand_weights_workload(), "q8"), (w.expand_weights_workload(M=1, K=1152, N=1024, block=128), "grouped"),
             (w.expand_weights_workload(M=32, K=6912, N=1152, block=64), "q8"), (w.expand_weights_workload(M=9, K=6912, N=200, block=128), "q8"), (w.expand_weights_workload(M=5, K=192, N=45, block=96, bias_pad=1), "q8"),
             (w.expand_weights_workload(M=7, K=128, N=70, expand_clamp=(-0.004, 0.006), clamp=(-0.05, 0.05)), "q8"),
             (w.expand_weights_workload(M=70, K=128, N=40, block=64), "folded"), (w.expand_weights_workload(M=2, K=64, N=33, fold=False, bias_pad=1), "own")]
    for wl, how in cases:
        print("[gpu-case]", wl.name, how, flush=True)
        got, kernels = run_on_gpu(device, wl)
        want = oracle_eval(wl)
        w16 = orc.expand_weights(wl.attrs["weights"], wl.attrs["scale"], wl.attrs["qbias"], block_size=wl.attrs["block"],
                                 output_min=wl.attrs["expand_min"], output_max=wl.attrs["expand_max"])
        assert_bf16_close(got[0], want[0].reshape(got[0].shape), wl.name + " (gpu)", magnitude=f(wl.inputs[0]) @ f(w16))
        if how == "own":
            assert_bit_exact(got[1], want[1], wl.name + " expansion")
            assert families(kernels) == ["expand_weights_bf16", "transpose_i8", "fc_bf16"], kernels
        else:
            assert families(kernels) == ["dec_linear" if how == "grouped" else "fc_bf16"], kernels


@pytest.mark.gpu
def test_gpu_bf16_add(device):
    """Elementwise: the kernel does the oracle's three fp32 operations in the oracle's order, so it is bit-exact."""
    for wl in [w.add_bf16_workload(), w.add_bf16_workload((3, 5, 7), 0.5, -1.25, 0.125, clamp=(-1.0, 2.0)),
               w.add_bf16_workload((64, 56, 56, 24), 0.7, 1.3, -0.01)]:
        print("[gpu-case]", wl.name, flush=True)
        got, kernels = run_on_gpu(device, wl, via="device")
        assert_bit_exact(got[0], oracle_eval(wl)[0], wl.name)
        assert families(kernels) == ["add_bf16"]


@pytest.mark.gpu
def test_gpu_bf16_split_k_is_deterministic(device):
    """A long K over fewer output tiles than CUs: K is split over blocks whose partial sums a second kernel adds in
    slice order; repeated dispatches give the same bits."""
    wl = w.fully_connected_bf16_workload(32, 6912, 256)
    split = lambda M, K, N: int(desc_interp.Descriptor(w.fully_connected_bf16_workload(M, K, N).program.serialize()).ops[0]["w0"])
    assert split(32, 6912, 256) == 9      # about 12 k-steps of 64 per block
    assert split(32, 6912, 1152) == 7     # 36 tiles: at most one block per CU
    assert split(32, 1152, 6912) == 1     # a short K: the second launch costs more than it saves
    assert split(200, 6912, 1152) == 1    # enough tiles already
    first = _check_gpu(device, wl, via="device")
    exe = Executable(device, wl.program.serialize())
    for _ in range(5):
        out = np.zeros_like(first)
        exe.run_host([wl.inputs[0], out])
        assert np.array_equal(out, first)
    exe.close()
    _check_gpu(device, w.fully_connected_bf16_workload(3, 1152, 40))


@pytest.mark.gpu
def test_gpu_bf16_matmul(device):
    """Attention-shaped matmuls (4 query heads sharing one K / V, length 1024, head size 256) with a run-time input2,
    per-batch input2, and a constant input2."""
    _check_gpu(device, w.matmul_bf16_workload(4, 1, 256, 1024, batch2=False))
    _check_gpu(device, w.matmul_bf16_workload(4, 1, 1024, 256, batch2=False))
    _check_gpu(device, w.matmul_bf16_workload(3, 2, 64, 24))
    _check_gpu(device, w.matmul_bf16_workload(2, 5, 16, 12, batch1=False, constant_rhs=True))
    _check_gpu(device, w.matmul_bf16_workload(1, 6, 32, 20, batch1=False, batch2=False, constant_rhs=True, bias=0.5))


@pytest.mark.gpu
def test_gpu_bf16_tolerance_tally(device):
    """Which elements needed more than one bf16 step.  Every tolerance comparison of this process is tallied by
    assert_bf16_close; the elements that differ from the oracle by more than one step and pass only because their sum
    cancelled (|difference| <= 2^-17 of sum |x w| + |bias|) are counted, printed per case, and must stay a small
    minority: the one-step bound is the binding one wherever nothing cancels."""
    import helpers
    gpu_cases = [t for t in helpers.BF16_TALLY if t[0].endswith("(gpu)")]
    if not gpu_cases:
        pytest.skip("no bf16 GPU comparison ran in this process before this test")
    compared = sum(n for _, n, _ in gpu_cases)
    widened = sum(k for _, _, k in gpu_cases)
    for what, n, k in gpu_cases:
        if k:
            print("[bf16-tolerance] %s: %d of %d elements beyond one step, admitted by the cancellation bound" % (what, k, n), flush=True)
    print("[bf16-tolerance] total: %d of %d elements (%.4f %%) in %d comparisons" % (widened, compared, 100.0 * widened / compared, len(gpu_cases)), flush=True)
    assert widened <= compared * 1e-4
