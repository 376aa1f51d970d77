"""Dispatches of the ring kernel in k-tiles of 128 bytes: which problems take them, and each tile against the oracle (whole numbers: exact) at ragged
rows and columns, with K that ends at every 16-byte chunk it may, at few tiles and more than the chip holds, and over windows."""
import subprocess

import pytest

from helpers import assert_bit_exact, host_check, oracle_eval, run_on_gpu
from torq_compiler_amd import workloads as w

WIDE = "record 0 1 igemm_dense_k128_i8"
FC, CONV = w.fully_connected_workload, w.conv2d_workload

# (make, the tile forced when the program is made, or None; taken)
CASES = [
    # 64 x 64: every ending of K in its last k-tile, N that ends inside a tile, more tiles than three per CU
    *[(lambda K=K: FC(1030, K, 976 + K // 16 % 4 * 4, realistic=True), 7, K > 1216) for K in (1216, 1232, 1248, 1264, 1280)],
    (lambda: FC(4097, 1152, 784), 7, True), (lambda: FC(1030, 1152, 1001), 7, True), (lambda: FC(1030, 1088, 1040), 7, False),
    # 64 x 128: up to one tile per CU and more
    (lambda: FC(1090, 1136, 1032, realistic=True), 13, True), (lambda: FC(3137, 1024, 1032), 13, True), (lambda: FC(1090, 896, 1032), 13, False),
    # 128 x 128: the same two sides
    (lambda: FC(1025, 1024, 1040, realistic=True), 5, True), (lambda: FC(4099, 1136, 1160, realistic=True), 5, True), (lambda: FC(4099, 1024, 1168), 5, True),
    # 128 x 64
    (lambda: FC(1025, 4096, 1032, realistic=True), 12, True), (lambda: FC(1153, 4208, 976), 12, True), (lambda: FC(1153, 2048, 1032), 12, False),
    # half of the last k-tile beyond the weights' rows, each tile
    *[(lambda K=K: FC(1030, K, 976, realistic=True), 7, True) for K in (2576, 2592, 2608, 2624)], (lambda: FC(1030, 2496, 976), 7, False),
    (lambda: FC(1090, 2096, 1032, realistic=True), 13, True), (lambda: FC(3137, 2112, 1000), 13, True), (lambda: FC(1090, 1984, 1032), 13, False),
    (lambda: FC(1025, 2112, 1040, realistic=True), 5, True), (lambda: FC(4099, 2224, 1160), 5, True), (lambda: FC(1025, 1984, 1040), 5, False), (lambda: FC(1025, 4160, 1032), 12, True),
    (lambda: CONV(N=8, H=14, W=14, C=304, O=304, realistic=True), None, True), (lambda: CONV(N=10, H=30, W=29, C=48, O=200, KH=5, KW=6, pad=(2, 3, 2, 2)), 7, True),
    (lambda: CONV(N=9, H=30, W=31, C=112, O=264, KH=5, KW=4, pad=(1, 2, 2, 2), realistic=True), 5, True), (lambda: CONV(N=10, H=30, W=29, C=144, O=200, KH=3, KW=3), 7, True),
    # windows: fewer channels than a k-tile (several wraps of the channel), taps outside the image, strides, K that ends inside a k-tile
    (lambda: CONV(N=8, H=14, W=14, C=256, O=256, realistic=True), None, True), (lambda: CONV(N=9, H=30, W=29, C=128, O=200, realistic=True), 7, True),
    (lambda: CONV(N=10, H=61, W=60, C=48, O=336, KH=6, KW=7, pad=(2, 3, 3, 2), stride=(2, 2), realistic=True), 7, True),
    (lambda: CONV(N=7, H=40, W=33, C=16, O=500, KH=7, KW=11, pad=(5, 5, 3, 3)), 7, True), (lambda: CONV(N=4, H=61, W=63, C=112, O=200, KH=5, KW=5, pad=(2, 2, 1, 2), realistic=True), 5, True),
    (lambda: CONV(N=20, H=33, W=32, C=128, O=264), 5, True), (lambda: CONV(N=20, H=33, W=32, C=96, O=264), 5, False),
]
IDS = ["%s-%s" % (c[0]().name, c[1]) for c in CASES]


class Made:
    """A serialised program."""

    def __init__(self, blob):
        self.blob = blob

    def serialize(self):
        return self.blob


def made(case):
    """The workload with its tile forced; the switches are gone when it is loaded."""
    with pytest.MonkeyPatch.context() as m:
        if case[1] is not None:
            m.setenv("THIP_IGEMM_DENSE_VARIANT", str(case[1]))
            m.setenv("THIP_WINDOW_VARIANT", str(case[1]))
        wl = case[0]()
        return wl, Made(wl.program.serialize())


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    where = tmp_path_factory.mktemp("plan")
    exe = host_check("plan", where)

    def run(blob, **env):
        (where / "blob").write_bytes(blob)
        return subprocess.run([exe, str(where / "blob")], check=True, stdout=subprocess.PIPE, text=True, env=env).stdout.splitlines()[:-1]

    return run


@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_taken(plan, case):
    blob = made(case)[1].blob
    assert plan(blob) == [WIDE if case[2] else "record 0 1"]
    assert plan(blob, THIP_NO_K128="1") == ["record 0 1"]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_gpu(device, case):
    wl, program = made(case)
    want = oracle_eval(wl)[0]
    wl.program = program
    assert_bit_exact(run_on_gpu(device, wl)[0][0], want, wl.name)
