"""Which kernel a dispatch takes for a GEMM-shaped op follows the alignment of its result too: results at every offset that the op's
own kernel stores at, planned on the host and run on the GPU against the oracle."""
import os
import subprocess

import numpy as np
import pytest

import desc_interp
from helpers import assert_bit_exact, families, host_check, oracle_eval, run_on_gpu
from torq_compiler_amd import Program, workloads as w


class Moved:
    """A serialised single-op program whose result lies `offset` bytes into its binding, 64 bytes of room behind it."""

    def __init__(self, wl, offset):
        blob = bytearray(wl.program.serialize())
        d = desc_interp.Descriptor(bytes(blob))
        assert len(d.ops) == 1 and int(d.ops[0]["out"]["index"]) == 1
        ops = np.frombuffer(blob, dtype=desc_interp.OP, count=1, offset=int(d.header["ops_offset"]))
        bindings = np.frombuffer(blob, dtype=desc_interp.BINDING, count=2, offset=int(d.header["bindings_offset"]))
        ops["out"]["offset"] = offset
        bindings["size"][1] += offset + 64
        self.blob = bytes(blob)

    def serialize(self):
        return self.blob


def at_offset(wl, offset):
    return w.Workload(wl.name, Moved(wl, offset), wl.inputs, [((int(np.prod(wl.outputs[0][0])) + offset + 64,), np.int8)], wl.ops, wl.bytes, wl.attrs)


def batched():
    """The second batch element's result lies at byte 2706."""
    return w.matmul_workload(2, 33, 64, 41, constant_rhs=True)


SMALL_LINEAR = lambda: w.fully_connected_workload(40, 64, 48, realistic=True)  # noqa: E731
SMALL_CONV = lambda: w.conv2d_workload(N=1, H=12, W=12, C=64, O=32, realistic=True)  # noqa: E731
PATCH_CONV = lambda: w.conv2d_workload(N=16, H=56, W=56, C=96, O=96, realistic=True)  # noqa: E731
PADDED = lambda: w.fully_connected_workload(100000, 25, 128, realistic=True)  # noqa: E731
DIRECT, PATCH, OWN = "record 0 1 igemm_direct_i8", "record 0 1 conv_patch_i8", "record 0 1"
CASES = [
    (SMALL_LINEAR, 4, DIRECT), (SMALL_LINEAR, 1, OWN), (SMALL_LINEAR, 2, OWN), (SMALL_LINEAR, 7, OWN), (SMALL_CONV, 8, DIRECT), (SMALL_CONV, 2, OWN),
    (PATCH_CONV, 32, PATCH), (PATCH_CONV, 8, OWN), (PATCH_CONV, 1, OWN), (PADDED, 16, "padded 0 1"), (PADDED, 8, OWN),
]
IDS = ["%s-%d" % (n, c[1]) for n, c in zip(["linear"] * 4 + ["conv"] * 2 + ["patch"] * 3 + ["padded"] * 2, CASES)]


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    where = tmp_path_factory.mktemp("plan")
    exe = host_check("plan", where)

    def steps(wl):
        path = where / "blob"
        path.write_bytes(bytes(wl.program.serialize()))
        done = subprocess.run([exe, str(path)], stdout=subprocess.PIPE, text=True, timeout=120)
        assert done.returncode == 0
        lines = done.stdout.splitlines()
        steps.replayed = lines.pop() == "replayed"
        return lines

    return steps


@pytest.mark.parametrize("make,offset,want", CASES, ids=IDS)
def test_route_by_offset(plan, make, offset, want):
    assert plan(at_offset(make(), offset)) == [want]


def test_route_of_a_batch(plan):
    assert plan(batched()) == ["record 0 1 igemm_direct_i8", "record 1 1"]


def test_mutated_descriptors_are_planned(tmp_path):
    """What the validation lets through is planned without a report of the sanitizers, every record in one launch."""
    from test_inverted_residual import block
    exe = host_check("plan_fuzz", tmp_path, sanitize=["thip_plan.cpp", "thip_validate.cpp", "thip_status.cpp"])
    programs = [w.conv2d_workload(N=1, H=9, W=9, C=3, O=8, realistic=True), w.conv2d_workload(N=1, H=8, W=8, C=24, O=16, realistic=True), w.conv2d_workload(N=1, H=8, W=8, C=32, O=16, realistic=True),
                w.fully_connected_workload(40, 72, 20, realistic=True), w.matmul_workload(2, 9, 61, 37), batched(), w.mobilenet_v2_workload(batch=1, resolution=32, classes=10, width=0.25),
                w.grouped_linear_workload(mode="residual", K=256, N=256), w.pointwise_add_workload(N=1, H=7, W=7, C=96, O=32), block(N=2, H=8, W=8, C=16, E=32, stride=2),
                block(N=2, H=8, W=8, C=3, E=32, stride=1, first=(3, 1, (1, 1, 1, 1)))]
    files = []
    for i, wl in enumerate(programs):
        files.append(tmp_path / ("blob%d" % i))
        files[-1].write_bytes(bytes(wl.program.serialize()))
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0:detect_leaks=0", UBSAN_OPTIONS="print_stacktrace=1")
    run = subprocess.run([exe, "600"] + [str(f) for f in files], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, env=env, timeout=300)
    assert run.returncode == 0 and run.stdout.startswith("planned "), run.stdout[-3000:]


def chain(blocks, channels):
    """3x3 convolutions one behind the other: 9 * channels^2 bytes of weights each."""
    p = Program()
    rng = np.random.default_rng(5)
    wt = rng.integers(-127, 128, size=(channels, channels, 3, 3)).astype(np.int8)
    mult, shift = w.quantize_multiplier(np.full(channels, 60 / (np.sqrt(channels * 9) * 5400)))
    sb, sf = w.derive_scale_bias(mult, shift, np.zeros(channels, dtype=np.int64), wt, 0)
    h = p.binding(0, (1, 14, 14, channels))
    for i in range(blocks):
        init = dict(init=p.binding(1, (1, 14, 14, channels))) if i == blocks - 1 else {}
        h = p.conv2d(h, wt, sb, nhwc_input=True, input_zp=0, output_zp=0, output_min=-128, output_max=127, shift_factor=sf, pad=(1, 1, 1, 1), stride=(1, 1), **init)
    return w.Workload("chain", p, [], [], 0, 0, {})


@pytest.mark.parametrize("blocks,channels,replayed", [(3, 256, False), (6, 256, False), (40, 256, False), (41, 256, True), (54, 256, True), (4, 64, True), (3, 64, False)])
def test_long_programs_and_short_ones_of_little_weight_are_replayed(plan, blocks, channels, replayed):
    assert len(plan(chain(blocks, channels))) == blocks and plan.replayed == replayed


RAGGED = [
    (lambda: w.fully_connected_workload(1500, 1333, 48), True), (lambda: w.fully_connected_workload(60, 776, 256), True), (lambda: w.fully_connected_workload(200000, 17, 16), True),
    (lambda: w.conv2d_workload(N=1, H=7, W=7, C=33, O=64), True), (lambda: w.conv2d_workload(N=16, H=56, W=56, C=13, O=24, KH=5, KW=5, pad=(2, 2, 2, 2)), True),
    (lambda: w.fully_connected_workload(60, 24, 64), False), (lambda: w.fully_connected_workload(30000, 72, 40), False), (lambda: w.conv2d_workload(N=1, H=112, W=112, C=8, O=32), False),
    (lambda: w.conv2d_workload(N=32, H=112, W=112, C=40, O=32, stride=(2, 2)), False), (lambda: w.conv2d_workload(N=4, H=56, W=56, C=264, O=96, KH=1, KW=1, stride=(2, 2), pad=(0, 0, 0, 0)), False),
]


@pytest.mark.parametrize("make,padded", RAGGED, ids=[c[0]().name for c in RAGGED])
def test_ragged_channels_are_padded_where_that_is_measured_ahead(plan, make, padded):
    assert [s.split()[0] for s in plan(make())] == ["padded" if padded else "record"]


AS_IT_IS = " igemm_direct_i8 as it is"
FC, CONV = w.fully_connected_workload, w.conv2d_workload
LINES = list(zip([c[0] for c in RAGGED], [["padded 0 1" + AS_IT_IS]] * 2 + [["padded 0 1"], ["padded 0 1" + AS_IT_IS], ["padded 0 1 conv_patch_i8"]] + [["record 0 1"]] * 4 + [["record 0 1" + AS_IT_IS]])) + [
    # few rows: to K = 2500; more: to 9000
    (lambda: FC(9, 2500, 100), ["padded 0 1" + AS_IT_IS]), (lambda: FC(9, 2501, 100), ["padded 0 1"]), (lambda: FC(100, 8999, 32), ["padded 0 1" + AS_IT_IS]), (lambda: FC(100, 9001, 32), ["padded 0 1 igemm_direct_i8"]),
    (lambda: CONV(N=1, H=19, W=19, C=387, O=134, KH=5, KW=5, pad=(2, 2, 2, 2)), ["padded 0 1 igemm_direct_i8"]), (lambda: CONV(N=1, H=19, W=19, C=359, O=134, KH=5, KW=5, pad=(2, 2, 2, 2)), ["padded 0 1" + AS_IT_IS]),
    # a window over ragged results: strips in one round of the CUs, in two that are high, wide or narrow enough, and in two that are not
    (lambda: CONV(N=19, H=53, W=53, C=64, O=89, pad=(1, 1, 1, 1)), [PATCH]), (lambda: CONV(N=45, H=56, W=56, C=96, O=15, KH=5, KW=5, pad=(2, 2, 2, 2)), [PATCH]), (lambda: CONV(N=20, H=64, W=64, C=112, O=8, KH=5, KW=5, pad=(2, 2, 2, 2)), [OWN]),
    (lambda: CONV(N=22, H=73, W=73, C=64, O=5, KH=7, KW=7, pad=(3, 3, 3, 3)), [OWN]), (lambda: CONV(N=27, H=46, W=46, C=80, O=33, KH=5, KW=5, pad=(2, 2, 2, 2)), [OWN]), (lambda: CONV(N=40, H=40, W=40, C=80, O=7, KH=7, KW=7, pad=(3, 3, 3, 3)), [OWN]),
    (lambda: CONV(N=7, H=105, W=105, C=64, O=53, KH=5, KW=5, pad=(2, 2, 2, 2)), [OWN]), (lambda: CONV(N=6, H=122, W=122, C=96, O=28, KH=5, KW=5, pad=(2, 2, 2, 2)), [OWN]), (lambda: CONV(N=6, H=122, W=122, C=96, O=32, KH=5, KW=5, pad=(2, 2, 2, 2)), [PATCH]),
    (lambda: CONV(N=5, H=104, W=104, C=16, O=45, pad=(1, 1, 1, 1)), [OWN]),
    # 256 tiles of 32 x 32, and one row more
    (lambda: FC(256, 77, 1024), ["padded 0 1" + AS_IT_IS]), (lambda: FC(257, 77, 1024), ["padded 0 1"]),
    # a gather of one k-tile: in single bytes, in pieces of eight
    (lambda: FC(40, 63, 63), ["record 0 1" + AS_IT_IS]), (lambda: FC(40, 56, 63), ["record 0 1"]), (lambda: FC(9, 100, 2303), ["record 0 1" + AS_IT_IS]),
]


@pytest.mark.parametrize("make,lines", LINES, ids=[c[0]().name for c in LINES])
def test_ragged_rows_by_each_way(plan, make, lines):
    assert plan(make()) == lines


@pytest.mark.parametrize("kw,taken", [
    (dict(N=1, H=224, W=224, C=3, E=32, O=16, stride=1, first=(3, 2, (0, 1, 0, 1))), True), (dict(N=1, H=112, W=112, C=16, E=96, O=32, stride=2, pad=(0, 1, 0, 1)), False),
    (dict(N=4, H=112, W=112, C=16, E=96, O=32, stride=2, pad=(0, 1, 0, 1)), True), (dict(N=8, H=28, W=28, C=32, E=192, O=32, stride=1), False), (dict(N=64, H=28, W=28, C=32, E=192, O=32, stride=1), True),
    (dict(N=200, H=14, W=14, C=64, E=384, O=64, stride=1), False),
    # many narrow channels, and few
    (dict(N=170, H=66, W=54, C=16, E=48, O=96, stride=1), False), (dict(N=101, H=64, W=55, C=16, E=96, O=64, stride=1), False), (dict(N=192, H=51, W=56, C=64, E=128, O=64, stride=1), False),
    (dict(N=101, H=64, W=55, C=16, E=96, O=16, stride=1), True),
    # two / one launch, us: 9.6 / 7.5, 8.0 / 6.4, 13.2 / 10.8; 33.7 / 37.7, 12.9 / 14.1
    (dict(N=132, H=8, W=20, C=16, E=48, O=80, stride=1), True), (dict(N=7, H=74, W=34, C=48, E=48, O=32, stride=1), True), (dict(N=104, H=33, W=10, C=64, E=160, O=48, stride=1), True),
    (dict(N=150, H=45, W=10, C=96, E=480, O=16, stride=1), False), (dict(N=33, H=49, W=49, C=32, E=192, O=32, stride=2), False),
], ids=lambda v: "x".join(str(x) for x in v.values()) if isinstance(v, dict) else str(v))
def test_blocks_are_one_launch_where_that_is_estimated_ahead(plan, kw, taken):
    from test_ir_block import block
    lines = plan(block(**kw))
    assert (lines == ["ir_block_i8 0 3"]) if taken else [s.split()[:3] for s in lines] == [["ir_expand_dw_i8", "0", "2"], ["record", "2", "1"]], lines


@pytest.mark.parametrize("kw,taken", [
    (dict(N=1, H=5, W=510, C=16, E=32, stride=1), True), (dict(N=1, H=5, W=511, C=16, E=32, stride=1), False), (dict(N=16, H=100, W=640, C=16, E=96, stride=1), False),
    (dict(N=1, H=5, W=407, C=16, E=32, stride=2), True), (dict(N=1, H=5, W=410, C=16, E=32, stride=2), False), (dict(N=1, H=98, W=640, C=16, E=32, stride=2), True),
    (dict(N=1, H=97, W=640, C=16, E=32, stride=2), False),
], ids=lambda v: "x".join(str(x) for x in v.values()) if isinstance(v, dict) else str(v))
def test_pairs_with_rows_too_wide_for_two_windows(plan, kw, taken):
    from test_inverted_residual import block
    assert [s.split()[0] for s in plan(block(**kw))] == (["ir_expand_dw_i8"] if taken else ["record"] * 2)


def test_wide_first_layers_are_one_launch_with_the_narrow_convolution(plan, monkeypatch):
    """Blocks of columns: the pair's strips of one row are no measure for them."""
    from test_ir_block import block
    monkeypatch.setenv("THIP_IR_BLOCK", "1")
    assert plan(block(N=1, H=30, W=640, C=3, E=32, O=16, stride=1, first=(3, 1, (1, 1, 1, 1)))) == ["ir_block_i8 0 3"]


def with_output_zp(wl, record, zp):
    """The serialised program, a record's zero point set by hand."""
    class Changed:
        @staticmethod
        def serialize():
            blob = bytearray(wl.program.serialize())
            d = desc_interp.Descriptor(bytes(blob))
            ops = np.frombuffer(blob, dtype=desc_interp.OP, count=len(d.ops), offset=int(d.header["ops_offset"]))
            ops["output_zp"][record] = zp
            return bytes(blob)

    return w.Workload(wl.name, Changed, wl.inputs, wl.outputs, wl.ops, wl.bytes, wl.attrs)


@pytest.mark.parametrize("steep", [None, 0.6])
@pytest.mark.parametrize("zp,taken", [(-32768, True), (32767, True), (-32769, False), (32768, False), (1 << 30, False), (-(1 << 31), False)])
def test_blocks_take_zero_points_that_fold_into_the_rounding(plan, steep, zp, taken, monkeypatch):
    """The builder writes no others; a descriptor from elsewhere may."""
    from test_ir_block import block
    monkeypatch.setenv("THIP_IR_BLOCK", "1")
    lines = plan(with_output_zp(block(N=1, H=12, W=12, C=16, E=48, O=32, stride=1, steep=steep), 1, zp))
    assert (lines[0].split()[:3] == ["ir_block_i8", "0", "3"]) == taken, lines


@pytest.mark.gpu
@pytest.mark.parametrize("make,offset,route", CASES, ids=IDS)
def test_gpu_result_at_offset(device, make, offset, route):
    wl = at_offset(make(), offset)
    print("[gpu-case]", wl.name, offset, flush=True)
    launched = []
    got, kernels = run_on_gpu(device, wl, via="device", launched=launched)
    assert {DIRECT: "igemm_direct_i8", PATCH: "conv_patch_i8", OWN: families(kernels)[0]}.get(route, "pad_rows_i8") == families(launched)[0], launched
    want = oracle_eval(make())[0].reshape(-1)
    assert_bit_exact(got[0][offset:offset + want.size], want, wl.name)
    assert np.all(got[0][:offset] == 0x55) and np.all(got[0][offset + want.size:] == 0x55), "bytes around the result"


@pytest.mark.gpu
def test_gpu_batch(device):
    wl = batched()
    print("[gpu-case]", wl.name, flush=True)
    got, _ = run_on_gpu(device, wl, via="device")
    assert_bit_exact(got[0], oracle_eval(wl)[0], wl.name)
