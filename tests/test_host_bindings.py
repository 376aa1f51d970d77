"""Dispatches on host memory: the copies to pinned memory and back, at sizes around their pieces and limits, results whole numbers."""
import ctypes
import subprocess
import threading

import numpy as np
import pytest

import torq_compiler_amd as thip
from helpers import host_check

PIECE, HALF, RESULT = 256 << 10, 8 << 20, 1 << 20  # what a thread copies at a time, half of the pinned memory, the largest result out of it


def test_copies_shared_among_threads(tmp_path):
    exe = host_check("copy_crew", tmp_path, sanitize=["thip_host_copy.cpp"])
    done = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert done.returncode == 0 and done.stdout == "copied\n", done.stdout[-3000:]


def added(sizes):
    """Pairs of inputs of `sizes` bytes, xor of each pair."""
    p = thip.Program()
    for i, size in enumerate(sizes):
        a, b = p.binding(3 * i, (size,)), p.binding(3 * i + 1, (size,))
        p.elementwisebinary(2, a, b, init=p.binding(3 * i + 2, (size,)))
    return p


def arrays(sizes, seed):
    rng = np.random.default_rng(seed)
    ins = [rng.integers(-128, 128, size=(2, size), dtype=np.int8) for size in sizes]
    return [a for pair in ins for a in (pair[0], pair[1], np.full_like(pair[0], 85))], [pair[0] ^ pair[1] for pair in ins]


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [
    (1,), (PIECE - 1,), (PIECE,), (PIECE + 1,), (RESULT,), (RESULT + 1,), (5 * PIECE + 3,), (HALF // 2, 3), (HALF - 256, 512), (HALF,), (HALF + 1, 100, PIECE), (2 * HALF + 77, 1, 3 * HALF),
    (RESULT, RESULT, RESULT, RESULT, 7, 300),
], ids=str)
def test_gpu_sizes(device, sizes):
    exe = thip.Executable(device, added(sizes).serialize())
    for seed in range(3):
        got, want = arrays(sizes, seed)
        exe.run_host(got)
        assert all(np.array_equal(got[3 * i + 2], want[i]) for i in range(len(sizes)))
    exe.close()


@pytest.mark.gpu
def test_gpu_threads_share_the_helpers(device):
    sizes = (3 << 20, (20 << 20) + 5, 70000)
    exes = [thip.Executable(device, added((n,)).serialize()) for n in sizes]
    failed = []

    def dispatch(which):
        for seed in range(6):
            got, want = arrays((sizes[which],), 10 * which + seed)
            exes[which].run_host(got)
            if not np.array_equal(got[2], want[0]):
                failed.append((which, seed))

    threads = [threading.Thread(target=dispatch, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not any(t.is_alive() for t in threads) and not failed, failed
    for exe in exes:
        exe.close()


@pytest.mark.gpu
def test_gpu_memory_that_is_pinned_already(device):
    hip = ctypes.CDLL("libamdhip64.so")
    size = 3 * PIECE + 5
    exe = thip.Executable(device, added((size,)).serialize())
    held = [ctypes.c_void_p() for _ in range(3)]
    for p in held:
        assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(size), ctypes.c_uint(0)) == 0
    got = [np.ctypeslib.as_array((ctypes.c_int8 * size).from_address(p.value)) for p in held]
    fresh, want = arrays((size,), 1)
    for g, f in zip(got, fresh):
        g[...] = f
    exe.run_host(got)
    assert np.array_equal(got[2], want[0])
    exe.close()
    for p in held:
        assert hip.hipHostFree(p) == 0
