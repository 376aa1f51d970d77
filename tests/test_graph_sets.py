"""Graph replays of a program dispatched on several sets of device bindings in turn: a graph per set, as long as they fit."""
import time

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


def test_a_new_set_does_not_wait_for_the_old_ones(device):
    """Sets that are new on every dispatch, and new ones in place of sets with a graph: no call waits for the work in front of it."""
    wl = w.mobilenet_v2_workload(batch=256)
    print("[gpu-case]", wl.name, "new sets", flush=True)
    exe = Executable(device, wl.program.serialize())
    x = wl.inputs[0]
    out_bytes = int(np.prod(wl.outputs[0][0]))
    pin, pout = device.alloc(x.nbytes + 16 * 200), device.alloc(out_bytes + 16 * 200)  # a set is an offset
    lens = [x.nbytes, out_bytes]
    try:
        def dispatch(k, times=1):
            longest = 0.0
            for _ in range(times):
                t0 = time.perf_counter()
                exe.enqueue_device([pin + 16 * k, pout + 16 * k], lens)
                longest = max(longest, time.perf_counter() - t0)
            return longest

        dispatch(0)
        exe.wait()
        for what, sets in (("new sets only", [(k, 1) for k in range(90)]),
                           ("graphs that make room", [(100 + k, 2) for k in range(8)] + [(107, 70)] + [(120 + k, 2) for k in range(6)])):
            t0 = time.perf_counter()
            longest = max(dispatch(k, times) for k, times in sets)
            exe.wait()
            total = time.perf_counter() - t0
            assert longest < 0.4 * total, "%s: one call of %.1f ms, %.1f ms in all" % (what, longest * 1e3, total * 1e3)
    finally:
        exe.close()
        device.free(pin)
        device.free(pout)


def test_replaced_graphs_in_flight(device):
    """Sets that take the place of others while these have replays on the stream: every set's result is its own."""
    M, K, N = 33, 64, 40
    wl = w.branches_workload(M, K, N)
    print("[gpu-case]", wl.name, "sets replaced in flight", flush=True)
    exe = Executable(device, wl.program.serialize())
    x, rng, sets, wants = wl.inputs[0], np.random.default_rng(3), [], []
    for _ in range(24):
        x[...] = rng.integers(-128, 128, size=x.shape).astype(np.int8)
        sets.append((device.upload(x), device.upload(np.zeros((M, N), dtype=np.int8))))
        wants.append(oracle_eval(wl)[0].copy())
    lens = [x.nbytes, M * N]
    try:
        for _ in range(2):
            for first in (0, 8, 16):
                for times, group in ((3, sets[first:first + 8]), (80, sets[first + 7:first + 8])):
                    for _ in range(times):
                        for pair in group:
                            exe.enqueue_device(list(pair), lens)
        exe.wait()
        for k, ((_, pout), want) in enumerate(zip(sets, wants)):
            assert_bit_exact(device.download(pout, (M, N), np.int8), want, "set %d" % k)
    finally:
        exe.close()
        for pin, pout in sets:
            device.free(pin)
            device.free(pout)
