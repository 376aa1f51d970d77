"""The tile form of fc_bf16 (many input rows): every tile on ragged shapes, against the oracle."""
import numpy as np
import pytest

from helpers import assert_bf16_close, oracle_eval, run_on_gpu
from test_bf16 import _magnitude
from torq_compiler_amd import workloads as w

pytestmark = pytest.mark.gpu

# rows, K, columns: one row block and one column past a tile, K of one chunk, of a k-tile and a bit, of fewer k-tiles than
# the ring has stages, of an odd number of k-tiles for two groups, columns that no vector store covers
SHAPES = [(33, 8, 72), (65, 72, 131), (129, 200, 130), (257, 328, 264), (64, 640, 64), (300, 1160, 515)]


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5])
def test_every_tile(device, tile, monkeypatch):
    monkeypatch.setenv("THIP_FC_TILE", str(tile))
    cases = [w.fully_connected_bf16_workload(*s, clamp=(-0.5, 0.75) if i % 2 else None) for i, s in enumerate(SHAPES)]
    cases += [w.matmul_bf16_workload(2, 70, 136, 75), w.matmul_bf16_workload(1, 260, 320, 264)]  # run-time weights: rows
    for wl in cases:
        print("[gpu-case]", tile, wl.name, flush=True)
        got, kernels = run_on_gpu(device, wl, via="device")
        assert_bf16_close(got[0], oracle_eval(wl)[0], wl.name + " (gpu)", magnitude=_magnitude(wl))
        assert kernels[-1].startswith("fc_bf16<%d," % {1: 64, 2: 64, 3: 128, 4: 128, 5: 256}[tile]) and len(kernels[-1].split(",")) == 8, kernels


@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("columns", [57, 58, 59, 60, 61, 62, 63, 7, 1, 97, 258])
def test_ragged_columns(device, tile, columns, monkeypatch):
    """Every number of columns behind the last whole eight, rows that begin at any of their alignments; 0: the streaming form."""
    monkeypatch.setenv("THIP_FC_TILE", str(tile))
    wl = w.fully_connected_bf16_workload(70, 64, columns, clamp=(-0.5, 0.75) if columns % 2 else None)
    print("[gpu-case]", tile, wl.name, flush=True)
    got, _ = run_on_gpu(device, wl, via="device")
    assert_bf16_close(got[0], oracle_eval(wl)[0], wl.name + " (gpu)", magnitude=_magnitude(wl))


def test_nothing_beyond_k_reaches_a_result(device, monkeypatch):
    """K ends inside a k-tile: what follows a row in memory is the next row, infinite here, and must not be multiplied."""
    monkeypatch.setenv("THIP_FC_TILE", "1")
    wl = w.fully_connected_bf16_workload(66, 40, 64)
    wl.inputs[0][1::2] = 0x7f80
    got, _ = run_on_gpu(device, wl)
    want = oracle_eval(wl)[0]
    assert_bf16_close(got[0][0::2], want[0::2], wl.name, magnitude=_magnitude(wl)[0::2])


@pytest.mark.parametrize("rows,k,columns,tile", [(32, 256, 640, None), (64, 256, 640, 64), (400, 4096, 2048, 64), (512, 1152, 6912, 128), (2048, 1152, 6912, 256)])
def test_tile_by_shape(device, rows, k, columns, tile):
    _, kernels = run_on_gpu(device, w.fully_connected_bf16_workload(rows, k, columns), via="device")
    assert kernels[0].startswith("fc_bf16<%s," % (tile or 4)), kernels


@pytest.mark.parametrize("tile,columns,runs", [(1, 264, 0), (1, 262, 0), (3, 264, 0), (3, 262, 1), (4, 264, 0), (4, 263, 1), (5, 264, 1), (5, 261, 1)])
def test_how_results_are_stored(device, tile, columns, runs, monkeypatch):
    """Runs of rows through LDS (2 in the label's last number) for ragged columns of the wider tiles and for the widest."""
    monkeypatch.setenv("THIP_FC_TILE", str(tile))
    wl = w.fully_connected_bf16_workload(300, 136, columns)
    print("[gpu-case]", tile, wl.name, flush=True)
    got, kernels = run_on_gpu(device, wl, via="device")
    assert_bf16_close(got[0], oracle_eval(wl)[0], wl.name + " (gpu)", magnitude=_magnitude(wl))
    assert kernels[-1].endswith(",%d>" % (1 + 2 * runs)), kernels
