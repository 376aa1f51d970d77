"""dec_linear with two workgroups per column tile: whole and broken pairs of k-blocks, every row count, adds, zero points, clamps."""
import numpy as np
import pytest

from oracle import programs as prog
from test_decoder_sweep import _run_gpu, device  # noqa: F401  (the fixture)
from torq_compiler_amd import workloads as w

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("kw", [
    dict(K=17 * 128, N=16), dict(K=18 * 128, N=80), dict(K=17 * 128, N=17 * 128, mode="residual"), dict(K=33 * 128, N=48, zero_points=True), dict(K=19 * 128, N=32, mode="pair"),
    dict(K=17 * 128, N=64, expand_clamp=(0.01, 0.5)), dict(K=21 * 128, N=48, clamp=(-0.5, 0.25)),
], ids=lambda kw: "_".join("%s%s" % kv for kv in kw.items()))
def test_split(device, monkeypatch, M, kw):
    wl = w.grouped_linear_workload(M=M, **kw)
    if kw["N"] > 2048:
        monkeypatch.setenv("THIP_DEC_SPLIT", "2")  # more tiles than the rule splits
    outs, kernels = _run_gpu(device, wl)
    assert kernels[0].startswith("dec_linear<1,1,1,") and kernels[0].endswith(",2>"), kernels
    prog.check_grouped_linear(wl, outs, prog.assert_bf16_close, prog.assert_bit_exact)
    # infinities and NaN reach the results that they reach with one workgroup per tile, and no others
    wl.inputs[0].reshape(-1)[-1] = 0x7f80
    split, _ = _run_gpu(device, wl)
    monkeypatch.setenv("THIP_DEC_SPLIT", "1")
    whole, kernels = _run_gpu(device, wl)
    assert kernels[0].endswith(",1>"), kernels
    for a, b in zip(split, whole):
        a, b = prog.orc.from_bf16(a), prog.orc.from_bf16(b)
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isinf(a), np.isinf(b)) and np.array_equal(a[np.isinf(a)], b[np.isinf(b)])
