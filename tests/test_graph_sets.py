"""Graph replays of a program dispatched on several sets of device bindings in turn: a graph per set, as long as they fit."""
import numpy as np
import pytest

from helpers import assert_bit_exact, oracle_eval
from torq_compiler_amd import runtime
from torq_compiler_amd import workloads as w
from torq_compiler_amd.runtime import Executable

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sets", [1, 3, 8, 11])
def test_rotating_sets_match_oracle(device, sets):
    """Three rounds over `sets` buffer pairs (eager, captured, replayed; beyond eight sets some stay eager), then one set alone for
    longer than an unused graph is kept, then all of them again: every dispatch on fresh inputs, every result the oracle's."""
    M, K, N = 33, 64, 40
    wl = w.branches_workload(M, K, N)
    print("[gpu-case]", wl.name, "%d sets" % sets, flush=True)
    exe = Executable(device, wl.program.serialize())
    x = wl.inputs[0]
    rng = np.random.default_rng(sets)
    bufs = [(device.upload(x), device.upload(np.zeros((M, N), dtype=np.int8))) for _ in range(sets)]

    def dispatch(k, what):
        pin, pout = bufs[k]
        x[...] = rng.integers(-128, 128, size=x.shape).astype(np.int8)
        runtime.check(runtime.lib().thip_device_h2d(device.handle, pin, x.ctypes.data, x.nbytes))
        device.synchronize()
        exe.run_device([pin, pout], [x.nbytes, M * N])
        assert_bit_exact(device.download(pout, (M, N), np.int8), oracle_eval(wl)[0], "set %d, %s" % (k, what))

    for it in range(4):
        for k in range(sets):
            dispatch(k, "round %d" % it)
    for it in range(70):
        dispatch(sets - 1, "alone %d" % it)
    for it in range(3):
        for k in range(sets):
            dispatch(k, "again %d" % it)
    exe.close()
    for pin, pout in bufs:
        device.free(pin)
        device.free(pout)
