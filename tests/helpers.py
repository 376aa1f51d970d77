"""Shared helpers of the test-suite: run a workload through the C-ABI, evaluate it with the oracle."""
import numpy as np
import pytest

from oracle.programs import (BF16_TALLY, assert_bf16_close, assert_bit_exact, bf16_ordered,  # noqa: F401  (re-exported)
                             eval_network as oracle_network, eval_workload as oracle_eval)


def run_on_gpu(device, wl, via="host", launched=None):
    """Serialises the workload's program, loads it and runs one dispatch; returns the outputs and the kernels that its ops have of their
    own.  `launched` (a list): receives the kernels that the dispatch launches."""
    import torq_compiler_amd as thip

    blob = wl.program.serialize()
    exe = thip.Executable(device, blob)
    if launched is not None:
        launched += exe.launch_kernels()
    outs = [np.full(shape, 0x55, dtype=dt) for shape, dt in wl.outputs]
    try:
        if via == "host":
            exe.run_host(list(wl.inputs) + outs)
        else:
            ptrs = [device.upload(a) for a in wl.inputs] + [device.upload(o) for o in outs]
            lens = [a.nbytes for a in wl.inputs] + [o.nbytes for o in outs]
            exe.run_device(ptrs, lens)
            n_in = len(wl.inputs)
            outs = [device.download(ptrs[n_in + i], o.shape, o.dtype) for i, o in enumerate(outs)]
            for p in ptrs:
                device.free(p)
        return outs, exe.op_kernels()
    finally:
        exe.close()


def check_own_kernels(device, wl, want, via="host"):
    """Where a dispatch takes other kernels than its ops' own, a run of the ops by these, against `want` (the outputs)."""
    with pytest.MonkeyPatch.context() as m:
        launched = []
        m.setenv("THIP_PLAIN_RECORDS", "1")
        got, kernels = run_on_gpu(device, wl, via=via, launched=launched)
        assert launched == kernels, (launched, kernels)
        for g, e in zip(got, want):
            assert_bit_exact(g, e, wl.name + " by the ops' own kernels")


def families(kernels):
    """Kernel names without their template arguments: "maxpool_i8<16>" -> "maxpool_i8"."""
    return [k.split("<")[0] for k in kernels]


def host_check(name, directory, sanitize=()):
    """Builds tests/host/<name>.cpp against the package's library with the host compiler, with the library's `sanitize` sources (none of
    them calls HIP) under the sanitizers; returns the program's path."""
    import os
    import shutil
    import subprocess

    from torq_compiler_amd import runtime

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    gxx = shutil.which("g++")
    assert gxx, "g++ is needed for the host check"
    exe = os.path.join(str(directory), name)
    csrc = os.path.join(root, "torq-compiler_amd", "csrc")
    flags = ["-g", "-fsanitize=address,undefined", "-static-libasan", "-fno-sanitize-recover=undefined"] if sanitize else []
    built = subprocess.run([gxx, "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + csrc] + flags +
                           [os.path.join(root, "tests", "host", name + ".cpp")] + [os.path.join(csrc, s) for s in sanitize] + [runtime.LIB_PATH, "-Wl,-rpath," + os.path.dirname(runtime.LIB_PATH),
                            "-Wl,--allow-shlib-undefined", "-o", exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert built.returncode == 0, built.stdout[-3000:]
    return exe
