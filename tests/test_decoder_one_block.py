"""dec_linear with a wave per k-block and more input rows than come through LDS: every number of waves at its ends, row groups, adds, zero points, clamps."""
import pytest

from oracle import programs as prog
from test_decoder_sweep import _run_gpu, device  # noqa: F401  (the fixture)
from torq_compiler_amd import workloads as w

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [5, 16, 17, 32])
@pytest.mark.parametrize("kw", [
    dict(K=128, N=16), dict(K=9 * 128, N=257 * 16), dict(K=16 * 128, N=257 * 16, mode="pair"), dict(K=13 * 128, N=13 * 128, mode="residual"), dict(K=16 * 128, N=272, zero_points=True),
    dict(K=12 * 128, N=257 * 16, expand_clamp=(0.01, 0.5)), dict(K=15 * 128, N=48, mode="concat", clamp=(-0.5, 0.25)),
], ids=lambda kw: "_".join("%s%s" % kv for kv in kw.items()))
def test_one_block(device, M, kw):
    wl = w.grouped_linear_workload(M=M, **kw)
    print("[gpu-case]", wl.name, flush=True)
    outs, kernels = _run_gpu(device, wl)
    assert kernels[0].startswith(("dec_linear<1,2,0,", "dec_linear<2,1,0,")) and kernels[0].endswith(",1,1>"), kernels
    prog.check_grouped_linear(wl, outs, prog.assert_bf16_close, prog.assert_bit_exact)
