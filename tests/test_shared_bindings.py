"""A caller may pass one piece of memory as an input and as an output: the results are those of every op as a launch of its own, whatever launches
stand for several of them."""
import ctypes
import subprocess

import numpy as np
import pytest

from helpers import assert_bit_exact, host_check, oracle_eval, oracle_network
from test_inverted_residual import block as expand_depthwise
from test_ir_block import block
from torq_compiler_amd import Program, runtime, workloads as w
from torq_compiler_amd.runtime import Executable

WHOLE = dict(N=2, H=56, W=40, C=32, E=144, O=32, stride=1)  # several strips and chunks an image


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    where = tmp_path_factory.mktemp("plan")
    exe = host_check("plan", where)

    def steps(wl, at):
        path = where / "blob"
        path.write_bytes(bytes(wl.program.serialize()))
        done = subprocess.run([exe, str(path)] + [hex(a) for a in at], stdout=subprocess.PIPE, text=True, timeout=120)
        assert done.returncode == 0
        return done.stdout.splitlines()[:-1]

    return steps


A, B, C = 0x10000000, 0x20000000, 0x30000000


@pytest.mark.parametrize("add", [None, 0, 1])
def test_a_block_in_place_is_told_from_one_that_is_not(plan, add, monkeypatch):
    monkeypatch.setenv("THIP_IR_BLOCK", "1")
    wl = block(add=add, **WHOLE)
    size = wl.inputs[0].nbytes
    for out, shared in ((B, ""), (A, " shared"), (A + size - 16, " shared"), (A - size + 16, " shared"), (A + size, ""), (A - size, "")):
        assert [s.replace(" igemm_direct_i8", "") for s in plan(wl, (A, out))] == ["ir_block_i8 0 3" + shared], hex(out)


def test_other_runs_of_records_in_place(plan):
    pair, product = expand_depthwise(N=1, H=20, W=21, C=16, E=48, stride=1), w.matmul_workload(2, 64, 48, 96, out_dtype=np.int8)
    assert plan(pair, (A, B)) == ["ir_expand_dw_i8 0 2"] and plan(pair, (A, A)) == ["ir_expand_dw_i8 0 2 shared"]
    rt = plan(product, (A, B, C))
    assert len(rt) == 1 and rt[0].startswith("igemm_rt_i8")
    assert plan(product, (A, B, A)) == plan(product, (A, B, B)) == [rt[0] + " shared"]


# what a result in the place of its input runs by: a copy of the rows, or the op's own kernel, which takes 64 columns at a time
PLACES = [
    (lambda: w.fully_connected_workload(301, 301, 301, realistic=True), "padded 0 1 igemm_direct_i8 as it is"), (lambda: w.fully_connected_workload(77, 500, 500, realistic=True), "padded 0 1 igemm_direct_i8 as it is"),
    (lambda: w.conv2d_workload(N=3, H=9, W=8, C=61, O=61, realistic=True), "padded 0 1 igemm_direct_i8 as it is"),
    (lambda: w.fully_connected_workload(400, 63, 63, realistic=True), "record 0 1 igemm_direct_i8 as it is"), (lambda: w.fully_connected_workload(400, 64, 64, realistic=True), "record 0 1 igemm_direct_i8"),
]
PLACE_IDS = [c[0]().name for c in PLACES]


def in_one_binding(wl):
    """The same op from binding 0 to binding 0."""
    p = Program()
    x = p.binding(0, wl.inputs[0].shape)
    attrs = dict(wl.attrs)
    weights, scale_bias = attrs.pop("weights"), attrs.pop("scale_bias")
    if len(wl.inputs[0].shape) == 2:
        p.fully_connected(x, weights, scale_bias, init=x, **attrs)
    else:
        p.conv2d(x, weights, scale_bias, init=x, nhwc_input=attrs.pop("nhwc"), **attrs)
    return w.Workload(wl.name, p, wl.inputs, [], wl.ops, wl.bytes, wl.attrs)


@pytest.mark.parametrize("make,line", PLACES, ids=PLACE_IDS)
def test_rows_that_are_written_over(plan, make, line):
    wl = make()
    assert plan(wl, (A, B)) == [line] and plan(wl, (A, A)) == [line + " shared"] and plan(wl, (A, A + wl.inputs[0].nbytes - 16)) == [line + " shared"]
    (alone,) = plan(in_one_binding(wl), (A,))
    assert alone in ((line[:-len(" as it is")], "padded 0 1") if line.startswith("padded") else ("record 0 1",)), alone


def blocks(count, **kw):
    """`count` blocks beside one another in a program, block i from binding 2 i to binding 2 i + 1."""
    wls = [block(seed=1080 + i, **kw) for i in range(count)]
    p = Program()
    for i, wl in enumerate(wls):
        values = [p.binding(2 * i, wl.inputs[0].shape)]
        layers = wl.attrs["layers"]
        for j, L in enumerate(layers):
            src = [values[k] for k in L.inputs]
            init = dict(init=p.binding(2 * i + 1, wl.outputs[0][0])) if j + 1 == len(layers) else {}
            if L.op == "add":
                values.append(p.add(src[0], src[1], L.weights, L.scale_bias, **L.attrs, **init))
            else:
                values.append(getattr(p, L.op)(src[0], L.weights, L.scale_bias, nhwc_input=True, **L.attrs, **init))
    return p, wls


@pytest.mark.gpu
@pytest.mark.parametrize("add", [None, 0, 1])
@pytest.mark.parametrize("how", ["run_device", "enqueue_device_noalloc"])
def test_gpu_blocks_in_place(device, add, how, monkeypatch):
    """Four blocks, each of which writes over its input: eager, captured and replayed dispatches, and the one that allocates nothing."""
    monkeypatch.setenv("THIP_IR_BLOCK", "1")
    program, wls = blocks(4, add=add, **WHOLE)
    print("[gpu-case]", wls[0].name, "in place", add, how, flush=True)
    want = [oracle_network(wl) for wl in wls]
    exe = Executable(device, program.serialize())
    assert [k.split("<")[0] for k in exe.launch_kernels()] == ["ir_block_i8"] * 4
    ptrs = [device.upload(wl.inputs[0]) for wl in wls]
    other = [device.upload(wl.inputs[0]) for wl in wls]
    try:
        for it in range(4):
            for wl, ptr in zip(wls, ptrs):
                runtime.check(runtime.lib().thip_device_h2d(device.handle, ptr, wl.inputs[0].ctypes.data, wl.inputs[0].nbytes))
            device.synchronize()
            both = [p for ptr in ptrs for p in (ptr, ptr)]
            getattr(exe, how)(both, [wls[0].inputs[0].nbytes] * 8)
            exe.wait()
            for i, wl in enumerate(wls):
                assert_bit_exact(device.download(ptrs[i], wl.outputs[0][0], np.int8), want[i], "block %d in place, dispatch %d" % (i, it))
        # the same executable on memory that is not shared
        for wl, ptr in zip(wls, ptrs):
            runtime.check(runtime.lib().thip_device_h2d(device.handle, ptr, wl.inputs[0].ctypes.data, wl.inputs[0].nbytes))
        device.synchronize()
        getattr(exe, how)([p for pair in zip(ptrs, other) for p in pair], [wls[0].inputs[0].nbytes] * 8)
        exe.wait()
        for i, wl in enumerate(wls):
            assert_bit_exact(device.download(other[i], wl.outputs[0][0], np.int8), want[i], "block %d" % i)
    finally:
        device.synchronize()
        exe.close()
        for p in ptrs + other:
            device.free(p)


@pytest.mark.gpu
@pytest.mark.parametrize("make,line", PLACES, ids=PLACE_IDS)
@pytest.mark.parametrize("bindings", [2, 1])
def test_gpu_rows_that_are_written_over(device, make, line, bindings):
    wl = make()
    print("[gpu-case]", wl.name, "over its input", bindings, flush=True)
    x, want = wl.inputs[0], oracle_eval(wl)[0]
    exe = Executable(device, (wl if bindings == 2 else in_one_binding(wl)).program.serialize())
    ptr, other = device.upload(x), device.upload(x)
    try:
        for how in (exe.run_device, exe.enqueue_device_noalloc):
            runtime.check(runtime.lib().thip_device_h2d(device.handle, ptr, x.ctypes.data, x.nbytes))
            device.synchronize()
            how([ptr] * bindings, [x.nbytes] * bindings)
            exe.wait()
            assert_bit_exact(device.download(ptr, wl.outputs[0][0], np.int8), want.reshape(wl.outputs[0][0]), wl.name)
        if bindings == 2:
            runtime.check(runtime.lib().thip_device_h2d(device.handle, ptr, x.ctypes.data, x.nbytes))
            device.synchronize()
            exe.run_device([ptr, other], [x.nbytes] * 2)
            assert_bit_exact(device.download(other, wl.outputs[0][0], np.int8), want.reshape(wl.outputs[0][0]), wl.name)
    finally:
        exe.close()
        device.free(ptr)
        device.free(other)


@pytest.mark.gpu
def test_gpu_other_runs_of_records_in_place(device):
    # (the product's own kernels take 64 columns at a time: a workgroup has read its rows when it stores them)
    pair, product = expand_depthwise(N=2, H=40, W=41, C=16, E=96, stride=1), w.matmul_workload(2, 96, 64, 64, out_dtype=np.int8, shift=32, scale=1 << 20)
    for wl, want, inside in ((pair, oracle_network(pair), 0), (product, oracle_eval(product)[0], 0), (product, oracle_eval(product)[0], 1)):
        print("[gpu-case]", wl.name, "output over input", inside, flush=True)
        exe = Executable(device, wl.program.serialize())
        shape, dtype = wl.outputs[0]
        size = int(np.prod(shape)) * np.dtype(dtype).itemsize
        ptrs = [device.upload(np.resize(a.reshape(-1), max(a.size, size))) for a in wl.inputs]
        try:
            exe.run_device(ptrs + [ptrs[inside]], [a.nbytes for a in wl.inputs] + [size])
            assert_bit_exact(device.download(ptrs[inside], shape, dtype), want, wl.name)
        finally:
            exe.close()
            for p in ptrs:
                device.free(p)


@pytest.mark.gpu
@pytest.mark.parametrize("make,kernels", [
    (lambda: block(N=2, H=14, W=14, C=96, E=1152, O=96, stride=1), ["ir_block_i8"]), (lambda: w.fully_connected_workload(301, 301, 301, realistic=True), ["igemm_direct_i8"]),
    (lambda: w.fully_connected_workload(400, 64, 64, realistic=True), ["igemm_direct_i8"]),
], ids=["block", "ragged", "aligned"])
def test_gpu_the_first_dispatch_in_place_while_a_graph_is_captured(device, make, kernels, monkeypatch):
    """The kernels that only shared memory needs are known since creation: a capture of another stream, in the strictest mode, ends as it should."""
    monkeypatch.setenv("THIP_IR_BLOCK", "1")
    wl = make()
    print("[gpu-case]", wl.name, "in place during a capture", flush=True)
    hip, x = runtime.lib(), wl.inputs[0]
    want = oracle_network(wl) if "layers" in wl.attrs else oracle_eval(wl)[0].reshape(wl.outputs[0][0])
    exe = Executable(device, wl.program.serialize())
    assert [k.split("<")[0] for k in exe.launch_kernels()] == kernels
    ptr, other = device.upload(x), device.upload(x)
    stream, graph = ctypes.c_void_p(), ctypes.c_void_p()
    try:
        assert hip.hipStreamCreate(ctypes.byref(stream)) == 0 and hip.hipStreamBeginCapture(stream, ctypes.c_int(0)) == 0
        copied = hip.hipMemcpyAsync(ctypes.c_void_p(other), ctypes.c_void_p(other), ctypes.c_size_t(16), ctypes.c_int(3), stream)
        exe.enqueue_device_noalloc([ptr, ptr], [x.nbytes] * 2)
        assert (copied, hip.hipStreamEndCapture(stream, ctypes.byref(graph))) == (0, 0)
        exe.wait()
        assert_bit_exact(device.download(ptr, wl.outputs[0][0], np.int8), want, wl.name)
    finally:
        for handle, free in ((graph, hip.hipGraphDestroy), (stream, hip.hipStreamDestroy)):
            if handle:
                free(handle)
        exe.close()
        device.free(ptr)
        device.free(other)
