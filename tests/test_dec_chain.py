"""A decoder's step as one launch (dec_chain): which programs take it, each op against the oracle on the inputs the GPU gave it at the sizes where
the kernel can go wrong, what it may load, a launch whose workgroups give up waiting, executables in turn, and buffers that share memory."""
import subprocess
import threading

import numpy as np
import pytest

import torq_compiler_amd as thip
from helpers import host_check
from oracle import programs as prog
from torq_compiler_amd import workloads as w


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    exe = host_check("plan", tmp_path_factory.mktemp("plan"))

    def run(blob, env=None):
        path = tmp_path_factory.mktemp("blob") / "p.thip"
        path.write_bytes(blob)
        return subprocess.run([exe, str(path)], check=True, stdout=subprocess.PIPE, text=True, env=env).stdout.splitlines()

    return run


def linears(rows, widths, zero_points=False, seed=1060):
    """Linears on block-quantized weights one behind the other, widths[0] -> widths[1] -> ..., every result an output binding and nothing
    behind the last one: its weights and biases are the last constants of the program."""
    rng = np.random.default_rng(seed)
    p = thip.Program()
    x_in = w.to_bf16(rng.standard_normal((rows, widths[0])))
    x, ops, names, outputs = p.binding(0, x_in.shape, np.uint16), [], ["x_in"], []
    for i, (K, N) in enumerate(zip(widths, widths[1:])):
        wq, scale, qbias = w._block_quantized(rng, K, N, 128, 1.0)
        if zero_points:
            qbias = (-rng.integers(-8, 9, size=qbias.shape)).astype(np.float32) * w.from_bf16_np(scale)
        w16 = p.expand_weights(wq, scale, qbias, block_size=128, output_min=w.NO_CLAMP[0], output_max=w.NO_CLAMP[1])
        x = p.matmul(x, w16, np.zeros(1, np.float32), init=p.binding(i + 1, (rows, N), np.uint16), output_zp=0, output_min=w.NO_CLAMP[0],
                     output_max=w.NO_CLAMP[1], shift=0)
        ops.append(w.DecoderOp("linear", "y%d" % i, [names[-1]], (rows, N), weights=wq, scale=scale, qbias=qbias, block=128))
        names.append("y%d" % i)
        outputs.append(((rows, N), np.uint16))
    return w.Workload("linears_%dx%s%s" % (rows, "-".join(map(str, widths)), "_zp" if zero_points else ""), p, [x_in], outputs, 0, 0,
                      dict(ops=ops, names=names[1:]))


STEP = dict(layers=2, hidden=256, heads=2, head_dim=64, ffn=512, vocab=512, cache_len=64)


@pytest.mark.parametrize("case,chained", [
    (dict(), True), (dict(batch=4), True), (dict(expose=True), True), (dict(batch=5), False),
    # the input rows of one phase cost more than the launches saved (chainPays)
    (dict(batch=4, hidden=384, heads=8, head_dim=256, ffn=6272), False), (dict(heads=8, head_dim=256, cache_len=4096), False),
], ids=str)
def test_planned_where_it_pays(plan, case, chained):
    blob = w.decoder_step_workload(**dict(dict(batch=1), **dict(STEP, **case))).program.serialize()
    lines = plan(blob)
    assert (lines[0] == "dec_chain 0 13") == chained, lines
    assert all(l.startswith("record ") for l in plan(blob, env={"THIP_DEC_CHAIN": "0"})[:-1])


def test_weights_written_by_the_program_are_not_fetched_ahead(plan):
    """A matmul whose second operand an earlier one made ends the chain in front of it."""
    p = thip.Program()
    zero, none = np.zeros(1, np.float32), dict(output_zp=0, output_min=w.NO_CLAMP[0], output_max=w.NO_CLAMP[1], shift=0)
    x = p.binding(0, (1, 4, 64), np.uint16)
    caches = p.binding(1, (4, 64, 64), np.uint16)
    y = x
    for i in range(4):
        y = p.matmul(y, p.transpose(p.view(caches, (1, 64, 64), i * 4096), (0, 2, 1)), zero, **none)
    made = p.matmul(y, p.transpose(p.view(caches, (1, 64, 64), 0), (0, 2, 1)), zero, **none)  # [1, 4, 64]
    p.matmul(y, p.transpose(made, (0, 2, 1)), zero, init=p.binding(2, (1, 4, 4), np.uint16), **none)
    lines = plan(p.serialize(), env={"THIP_DEC_CHAIN": "1"})
    assert lines[:2] == ["dec_chain 0 5", "record 5 1"], lines


@pytest.fixture(scope="module")
def loads(tmp_path_factory):
    exe = host_check("chain_loads", tmp_path_factory.mktemp("loads"))

    def run(blob):
        """-> phases, linear ones, matmuls, linear ones with two jobs to a tile, and of these with an odd number of k-blocks"""
        path = tmp_path_factory.mktemp("blob") / "p.thip"
        path.write_bytes(blob)
        done = subprocess.run([exe, str(path)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120, env={"THIP_DEC_CHAIN": "1"})
        assert done.returncode == 0, done.stdout
        return [int(v) for v in done.stdout.split()]

    return run


# k-blocks: 11 and 13 in two halves to a tile, one half of the last unit not there; 12 and 10; 9 and 2, a job to a tile
@pytest.mark.parametrize("zero_points", [False, True])
@pytest.mark.parametrize("widths,shared,odd", [((256, 1408, 256, 1408, 256), 2, 2), ((1664, 1536, 1280, 48), 3, 1), ((1152, 256, 4096, 128), 1, 0),
                                               ((1408, 2048, 2176, 1408, 16), 3, 3)], ids=str)
def test_weights_loaded_of_linears(loads, widths, shared, odd, zero_points):
    assert loads(linears(2, widths, zero_points).program.serialize()) == [len(widths) - 1, len(widths) - 1, 0, shared, odd]


@pytest.mark.parametrize("case", [dict(), dict(cache_len=24, head_dim=72, heads=16), dict(cache_len=8, head_dim=8, heads=16), dict(hidden=1408, ffn=1664, vocab=2064, cache_len=1032, batch=3),
                                  dict(heads=16, head_dim=200, hidden=128, cache_len=40, batch=4)], ids=str)
def test_weights_loaded_of_steps(loads, case):
    phases, linear, matmul, shared, odd = loads(w.decoder_step_workload(**dict(dict(batch=1), **dict(STEP, **case))).program.serialize())
    assert phases >= 2 and linear + matmul == phases, (phases, linear, matmul)


@pytest.mark.parametrize("N", [1, 3, 17, 33])
@pytest.mark.parametrize("K", [8, 24, 40, 72, 104])
def test_weights_loaded_of_matmuls(loads, N, K):
    """Few columns and few of K: the last row of the operand ends inside the first half of a unit."""
    p = thip.Program()
    zero, none = np.zeros(1, np.float32), dict(output_zp=0, output_min=w.NO_CLAMP[0], output_max=w.NO_CLAMP[1], shift=0)
    for i in range(2):
        rhs = p.transpose(p.binding(3 * i + 1, (2, N, K), np.uint16), (0, 2, 1))
        p.matmul(p.binding(3 * i, (2, 4, K), np.uint16), rhs, zero, init=p.binding(3 * i + 2, (2, 4, N), np.uint16), **none)
    assert loads(p.serialize()) == [2, 0, 2, 0, 0]


def test_turns(tmp_path):
    exe = host_check("chain_turn", tmp_path, sanitize=["thip_chain_turn.cpp"])
    done = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert done.returncode == 0 and done.stdout == "in order\n", done.stdout[-3000:]


# ---- GPU ----------------------------------------------------------------------------------------------------------

SHAPES = [
    dict(batch=1, layers=2, vocab=4096),                                                          # the benchmark's widths
    dict(batch=2, layers=1, vocab=4096), dict(batch=3, layers=1, vocab=4096), dict(batch=4, layers=2, vocab=4096),
    # eleven k-blocks in two halves per tile, the last half empty; columns of a matmul that fill no tile, K that fills no unit
    dict(batch=1, layers=2, hidden=256, heads=2, head_dim=64, ffn=1408, vocab=48, cache_len=24),
    dict(batch=3, layers=2, hidden=128, heads=2, head_dim=64, ffn=1408, vocab=16, cache_len=8),
    dict(batch=2, layers=1, hidden=256, heads=16, head_dim=64, ffn=256, vocab=64, cache_len=200),   # sixteen rows of a matmul
    dict(batch=4, layers=1, hidden=256, heads=1, head_dim=128, ffn=8192, vocab=16384, cache_len=136),  # several passes and blocks a phase
    dict(batch=1, layers=1, hidden=1280, heads=8, head_dim=128, ffn=1536, vocab=1024, cache_len=2056),
]


def _id(c):
    return "-".join("%s%s" % (k, v) for k, v in c.items())


def _load(device, wl):
    exe = thip.Executable(device, wl.program.serialize())
    assert exe.launch_kernels()[0] == "dec_chain", exe.launch_kernels()
    return exe


def _buffers(device, wl):
    arrays = list(wl.inputs) + [np.full(s, 0x55, dtype=d) for s, d in wl.outputs]
    return [device.upload(a) for a in arrays], [a.nbytes for a in arrays]


def _outputs(device, wl, ptrs):
    return [device.download(ptrs[len(wl.inputs) + i], s, d) for i, (s, d) in enumerate(wl.outputs)]


@pytest.mark.gpu
@pytest.mark.parametrize("wait", [None, "0"], ids=["together", "given_up"])
@pytest.mark.parametrize("case", SHAPES, ids=_id)
def test_gpu_every_op(device, monkeypatch, case, wait):
    """wait 0: every workgroup gives up at its first wait, and the last one makes everything by itself."""
    monkeypatch.setenv("THIP_DEC_CHAIN", "1")
    if wait is not None:
        monkeypatch.setenv("THIP_DEC_CHAIN_WAIT", wait)
    wl = w.decoder_step_workload(expose=True, **case)
    print("[gpu-case]", wl.name, _id(case), wait, flush=True)
    exe = _load(device, wl)
    ptrs, lens = _buffers(device, wl)
    try:
        first = None
        for _ in range(3):
            exe.run_device(ptrs, lens)
            outs = _outputs(device, wl, ptrs)
            if first is None:
                prog.check_decoder_step(wl, outs, prog.assert_bf16_close, prog.assert_bit_exact)
                first = outs
            assert all(np.array_equal(a, b) for a, b in zip(outs, first))
    finally:
        exe.close()
        for q in ptrs:
            device.free(q)


@pytest.mark.gpu
@pytest.mark.parametrize("wait", [None, "0"], ids=["together", "given_up"])
@pytest.mark.parametrize("zero_points", [False, True])
@pytest.mark.parametrize("widths", [(256,) + (1408, 256) * 4, (1664, 1664, 48)], ids=str)
def test_gpu_nothing_behind_the_last_weights(device, monkeypatch, widths, zero_points, wait):
    """The last unit of the last matrix has a half that is not there, and nothing lies behind it."""
    monkeypatch.setenv("THIP_DEC_CHAIN", "1")
    if wait is not None:
        monkeypatch.setenv("THIP_DEC_CHAIN_WAIT", wait)
    wl = linears(1, widths, zero_points)
    print("[gpu-case]", wl.name, wait, flush=True)
    exe = _load(device, wl)
    ptrs, lens = _buffers(device, wl)
    try:
        for _ in range(3):
            exe.run_device(ptrs, lens)
            prog.check_grouped_linear(wl, _outputs(device, wl, ptrs), prog.assert_bf16_close, prog.assert_bit_exact)
    finally:
        exe.close()
        for q in ptrs:
            device.free(q)


@pytest.mark.gpu
def test_gpu_new_inputs_and_executables_in_turn(device, monkeypatch):
    """Two executables, two sets of buffers each, enqueued one behind the other without a wait: every dispatch leaves what one alone leaves."""
    monkeypatch.setenv("THIP_DEC_CHAIN", "1")
    wls = [w.decoder_step_workload(batch=1, seed=s, **STEP) for s in (3, 4)] + [w.decoder_step_workload(batch=2, seed=s, **STEP) for s in (5, 6)]
    print("[gpu-case]", [x.name for x in wls], flush=True)
    exes = [_load(device, wls[0]), _load(device, wls[2])]
    sets = [_buffers(device, x) for x in wls]
    try:
        def alone(k):
            exes[k // 2].run_device(*sets[k])
            return _outputs(device, wls[k], sets[k][0])

        want = [alone(k) for k in range(4)]
        for _ in range(10):
            for k in (0, 2, 1, 3, 0, 1, 2, 3):
                exes[k // 2].enqueue_device(*sets[k])
            for e in exes:
                e.wait()
            for k in range(4):
                assert all(np.array_equal(a, b) for a, b in zip(_outputs(device, wls[k], sets[k][0]), want[k])), k
    finally:
        for e in exes:
            e.close()
        for ptrs, _ in sets:
            for q in ptrs:
                device.free(q)


@pytest.mark.gpu
def test_gpu_a_launch_that_gave_up_is_not_tried_again_at_once(device, monkeypatch):
    """Workgroups that give up at their first wait: the step is still right, and the next ones run record by record."""
    wl = w.decoder_step_workload(batch=1, layers=2, vocab=512, expose=True, seed=12)  # fewer k-blocks leave the sums of both ways in one order
    print("[gpu-case]", wl.name, "gave up", flush=True)
    ptrs, lens = _buffers(device, wl)

    def dispatches(count, **env):
        for name in ("THIP_DEC_CHAIN", "THIP_DEC_CHAIN_WAIT"):
            monkeypatch.delenv(name, raising=False)
        for name, value in env.items():
            monkeypatch.setenv(name, value)
        exe = thip.Executable(device, wl.program.serialize())
        try:
            assert (exe.launch_kernels()[0] == "dec_chain") == (env.get("THIP_DEC_CHAIN") != "0")
            got = []
            for _ in range(count):
                exe.run_device(ptrs, lens)
                got.append(_outputs(device, wl, ptrs))
            return got
        finally:
            exe.close()

    same = lambda x, y: all(np.array_equal(a, b) for a, b in zip(x, y))
    try:
        launch, records = dispatches(1, THIP_DEC_CHAIN="1")[0], dispatches(1, THIP_DEC_CHAIN="0")[0]
        differ = not same(launch, records)  # (an assert would print them)
        assert differ, "the two ways are told apart by the order of their sums"
        got = dispatches(4, THIP_DEC_CHAIN_WAIT="0")
        prog.check_decoder_step(wl, got[0], prog.assert_bf16_close, prog.assert_bit_exact)
        assert [same(g, launch) for g in got] == [True, False, False, False] and all(same(g, records) for g in got[1:])
        assert all(same(g, launch) for g in dispatches(4))
    finally:
        for q in ptrs:
            device.free(q)


@pytest.mark.gpu
def test_gpu_beside_another_streams_kernels(device, monkeypatch):
    """Steps as one launch while GEMMs that fill the chip come and go on another stream."""
    monkeypatch.setenv("THIP_DEC_CHAIN", "1")
    wl, busy = w.decoder_step_workload(batch=1, expose=True, seed=13, **STEP), w.fully_connected_workload(4096, 1024, 4096, realistic=True)
    print("[gpu-case]", wl.name, busy.name, flush=True)
    exe, gemm = _load(device, wl), thip.Executable(device, busy.program.serialize())
    ptrs, lens = _buffers(device, wl)
    gemm_ptrs, gemm_lens = _buffers(device, busy)
    try:
        exe.run_device(ptrs, lens)
        want = _outputs(device, wl, ptrs)
        prog.check_decoder_step(wl, want, prog.assert_bf16_close, prog.assert_bit_exact)
        gemm.run_device(gemm_ptrs, gemm_lens)
        product = _outputs(device, busy, gemm_ptrs)[0]
        for k in range(30):
            for _ in range(20):
                gemm.enqueue_device(gemm_ptrs, gemm_lens)
            for _ in range(1 + k % 3):
                exe.enqueue_device(ptrs, lens)
            exe.wait()
            assert all(np.array_equal(a, b) for a, b in zip(_outputs(device, wl, ptrs), want)), k
            if k % 4 == 3:
                gemm.wait()
        gemm.wait()
        assert np.array_equal(_outputs(device, busy, gemm_ptrs)[0], product)
    finally:
        for e in (exe, gemm):
            e.close()
        for q in ptrs + gemm_ptrs:
            device.free(q)


@pytest.mark.gpu
def test_gpu_threads(device, monkeypatch):
    """A thread for each of two decoders, as it comes: one launch or beside the other, every op is right, and each way leaves one result."""
    wls = [w.decoder_step_workload(batch=b, expose=True, seed=9 + b, **STEP) for b in (1, 2)]
    print("[gpu-case]", [x.name for x in wls], "threads", flush=True)
    ways = []
    for chain in ("0", "1", None):
        if chain is None:
            monkeypatch.delenv("THIP_DEC_CHAIN")
        else:
            monkeypatch.setenv("THIP_DEC_CHAIN", chain)
        ways.append([thip.Executable(device, x.program.serialize()) for x in wls])
    exes = ways[2]
    assert all(e.launch_kernels()[0] == "dec_chain" for e in exes)
    sets = [_buffers(device, x) for x in wls]
    results, failed = [[], []], []

    def dispatches(i):
        try:
            for k in range(60):
                for _ in range(k % 3 + 1):
                    exes[i].enqueue_device(*sets[i])
                exes[i].wait()
                results[i].append(_outputs(device, wls[i], sets[i][0]))
        except Exception as e:  # reported by the test's own thread
            failed.append(e)

    try:
        threads = [threading.Thread(target=dispatches, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join(timeout=100)
        assert not failed and not any(t.is_alive() for t in threads), failed
        for i, wl in enumerate(wls):
            known = []
            for pair in ways[:2]:
                pair[i].run_device(*sets[i])
                known.append(_outputs(device, wl, sets[i][0]))
                prog.check_decoder_step(wl, known[-1], prog.assert_bf16_close, prog.assert_bit_exact)
            assert len(results[i]) == 60
            for got in results[i]:
                assert any(all(np.array_equal(a, b) for a, b in zip(got, want)) for want in known)
    finally:
        for pair in ways:
            for e in pair:
                e.close()
        for ptrs, _ in sets:
            for q in ptrs:
                device.free(q)


@pytest.mark.gpu
def test_gpu_an_abandoned_executable_holds_nobody_up(device, monkeypatch):
    """One executable's wait times out with some 200 ms of its launches on the way; another one's dispatch is done long before these."""
    monkeypatch.setenv("THIP_DEC_CHAIN", "1")
    wls = [w.decoder_step_workload(batch=1, expose=True, seed=s, **STEP) for s in (7, 8)]
    print("[gpu-case]", wls[0].name, "abandoned", flush=True)
    exes = [_load(device, x) for x in wls]
    sets = [_buffers(device, x) for x in wls]
    try:
        for _ in range(5000):
            exes[0].enqueue_device(*sets[0])
        exes[0].set_wait_timeout(1)
        exes[1].set_wait_timeout(50)
        with pytest.raises(thip.ThipError) as err:
            exes[0].wait()
        assert err.value.code == thip.runtime.INTERNAL
        exes[1].run_device(*sets[1])
        prog.check_decoder_step(wls[1], _outputs(device, wls[1], sets[1][0]), prog.assert_bf16_close, prog.assert_bit_exact)
    finally:
        device.synchronize()
        for e in exes:
            e.close()
        for ptrs, _ in sets:
            for q in ptrs:
                device.free(q)


@pytest.mark.gpu
def test_gpu_results_written_into_the_caches(device, monkeypatch):
    """A caller that has the new keys appended to its cache in place: the scores read them, as when every op is a launch of its own."""
    wl = w.decoder_step_workload(batch=1, **STEP)
    print("[gpu-case]", wl.name, "in place", flush=True)
    results = []
    for chain in ("1", "0"):
        monkeypatch.setenv("THIP_DEC_CHAIN", chain)
        exe = thip.Executable(device, wl.program.serialize())
        assert (exe.launch_kernels()[0] == "dec_chain") == (chain == "1")
        ptrs, lens = _buffers(device, wl)
        try:
            at = ptrs[1] + wl.inputs[1].nbytes // 2  # layer 1's cache; its scores come after every new key
            exe.run_device(ptrs[:4] + [at] + ptrs[5:], lens)
            keys = device.download(ptrs[1], wl.inputs[1].shape, np.uint16)
            outs = _outputs(device, wl, ptrs)
            results.append([outs[0], outs[2], keys])
        finally:
            exe.close()
            for q in ptrs:
                device.free(q)
    assert all(np.array_equal(a, b) for a, b in zip(*results))
    assert not np.array_equal(results[0][2], wl.inputs[1])
