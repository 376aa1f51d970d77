"""Intermediates of a decoder's step at more than four rows, in blocks of 32 columns: which ones are, and the same results as from rows one behind the
other (the sums are the same, so bit for bit; those are compared with the oracle elsewhere)."""
import subprocess

import numpy as np
import pytest

import torq_compiler_amd as thip
from helpers import host_check
from torq_compiler_amd import workloads as w

X, RES, ADD, OUT = 1, 2, 4, 8
SMALL = dict(layers=2, hidden=256, heads=2, head_dim=64, ffn=512, vocab=512, cache_len=64)
LAYER = [0, 0, OUT, X | ADD, X | ADD, X | RES | ADD]  # the first layer's input, and so its residual sum, is a binding; q and the scores are a matmul's


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    where = tmp_path_factory.mktemp("plan")
    exe = host_check("plan", where)

    def blocked(wl, **env):
        (where / "blob").write_bytes(wl.program.serialize())
        lines = subprocess.run([exe, str(where / "blob")], check=True, stdout=subprocess.PIPE, text=True, env=env).stdout.splitlines()[:-1]
        return [int(l.split("blocked ")[1]) if "blocked" in l else 0 for l in lines]

    return blocked


@pytest.mark.parametrize("case,want", [
    (dict(batch=32), LAYER + [X, 0, OUT, X | RES | ADD, X | ADD, X | RES | ADD, X]), (dict(batch=5, layers=1), LAYER + [X]), (dict(batch=4, layers=1, heads=8, cache_len=4096, head_dim=256), [0] * 7),
    (dict(batch=8, expose=True), [0] * 13),  # all of them are results of the program
    (dict(batch=8, layers=1, vocab=100), LAYER[:5] + [X | RES, 0]),  # a projection that another kernel makes reads the last one as it is
], ids=str)
def test_planned(plan, case, want):
    wl = w.decoder_step_workload(**dict(SMALL, **case))
    assert plan(wl) == want
    assert not any(plan(wl, THIP_PLAIN_RECORDS="1"))


def test_a_part_or_another_shape_of_it_is_left_as_it_lies(plan):
    """A result that is read as fewer, longer rows, and one of which only the lower half is read."""
    zero, none = np.zeros(1, np.float32), dict(output_zp=0, output_min=w.NO_CLAMP[0], output_max=w.NO_CLAMP[1])

    def linear(p, x, K, N, **init):
        w16 = p.expand_weights(np.ones((K, N), np.int8), np.full((K // 128, N), 0x3f80, np.uint16), np.zeros((K // 128, N), np.float32), block_size=128,
                               output_min=w.NO_CLAMP[0], output_max=w.NO_CLAMP[1])
        return p.matmul(x, w16, zero, shift=0, **dict(init, **none))

    for shape in ((8, 256), (8, 128)):
        p = thip.Program()
        y = linear(p, p.binding(0, (16, 128), np.uint16), 128, 128, init=p.tensor((16, 128), np.uint16))
        linear(p, p.view(y, shape), shape[1], 64, init=p.binding(1, (8, 64), np.uint16))
        assert plan(w.Workload("p", p, [], [], 0, 0)) == [0, 0]


@pytest.mark.gpu
@pytest.mark.parametrize("case", [
    dict(batch=5), dict(batch=16, hidden=384, heads=6), dict(batch=17, ffn=1408), dict(batch=31, heads=3, head_dim=128, ffn=4096), dict(batch=32, layers=3, hidden=1152, heads=4, head_dim=256, ffn=6912, cache_len=136),
    dict(batch=9, hidden=2048, heads=8, ffn=640, cache_len=200), dict(batch=32, hidden=128, heads=16, head_dim=64, ffn=8192, cache_len=24),
], ids=str)
def test_gpu(device, case, monkeypatch):
    wl = w.decoder_step_workload(**dict(SMALL, **case))
    blob, results = wl.program.serialize(), []
    for plain in (False, True):
        if plain:
            monkeypatch.setenv("THIP_PLAIN_RECORDS", "1")
        exe = thip.Executable(device, blob)
        for _ in range(2):  # what a dispatch leaves is not what the next one finds
            outs = [np.full(shape, 0x55, dtype=dt) for shape, dt in wl.outputs]
            exe.run_host(list(wl.inputs) + outs)
            results.append(outs)
        exe.close()
    for outs in results[:3]:
        assert all(np.array_equal(a, b) for a, b in zip(outs, results[3]))
