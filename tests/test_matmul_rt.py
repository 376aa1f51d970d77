"""int8 matmuls with a run-time input2 as one launch: every tile height, ragged ends of every kind, against the oracle."""
import numpy as np
import pytest

from helpers import assert_bit_exact, families, oracle_eval, run_on_gpu
from torq_compiler_amd import workloads as w

pytestmark = pytest.mark.gpu

I8 = dict(out_dtype=np.int8, scale=(1 << 30) + 12345, shift=41, output_zp=3)


@pytest.mark.parametrize("kw", [
    dict(B=1, M=1, K=16, N=4), dict(B=3, M=5, K=7, N=3, **I8),            # fewer bytes per batch than one load
    # fewer bytes of input2 than one load: four, fifteen as a column, as a row and of several columns, several batch elements
    dict(B=1, M=16, K=4, N=1), dict(B=1, M=40, K=15, N=1, **I8), dict(B=1, M=16, K=1, N=15), dict(B=1, M=9, K=3, N=5, out_dtype=np.int32), dict(B=2, M=17, K=2, N=3), dict(B=5, M=6, K=3, N=1, batch1=False, **I8),
    dict(B=7, M=5, K=7, N=2, batch2=False), dict(B=1, M=9000, K=5, N=2),
    dict(B=2, M=3, K=130, N=2, out_dtype=np.int32), dict(B=1, M=33, K=257, N=1), dict(B=2, M=40, K=129, N=3, **I8),
    dict(B=2, M=33, K=130, N=131, **I8), dict(B=2, M=31, K=100, N=129, bias=-77, out_dtype=np.int8, scale=3, shift=4, output_zp=-5, clamp=(-100, 90)),
    dict(B=3, M=70, K=200, N=90, batch1=False), dict(B=3, M=70, K=200, N=90, batch2=False, out_dtype=np.int32),
    dict(B=16, M=65, K=48, N=1030), dict(B=16, M=65, K=33, N=1030, **I8),  # 64 rows
    dict(B=16, M=300, K=40, N=1300), dict(B=16, M=300, K=45, N=1301, out_dtype=np.int32),  # 128 rows
], ids=lambda kw: "-".join(str(getattr(v, "__name__", v)) for v in kw.values()))
def test_runtime_input2(device, kw, tmp_path):
    wl = w.matmul_workload(**kw)
    print("[gpu-case]", wl.name, flush=True)
    want = oracle_eval(wl)[0]
    launched = []
    got, _ = run_on_gpu(device, wl, via="device", launched=launched)
    assert families(launched) == ["igemm_rt_i8"], launched
    assert_bit_exact(got[0], want, wl.name)
    device.set_event_log(str(tmp_path / "log.csv"))  # a log has its records launched one by one
    try:
        got, _ = run_on_gpu(device, wl, via="device")
    finally:
        device.set_event_log(None)
    assert_bit_exact(got[0], want, wl.name + " record by record")


# the smallest tile with one group of waves and with two, 64 rows, 128 rows: (B, M, N), template arguments up to the k-tile groups
TILES = [((2, 33, 17), (32, 1, 4)), ((16, 1, 144), (32, 1, 4)), ((9, 130, 250), (32, 1, 4)), ((16, 65, 1030), (64, 2, 2)), ((24, 400, 520), (128, 2, 2))]
TILE_IDS = ["32rows-ragged", "one-row", "32rows-batches", "64rows", "128rows"]
DTYPE_CODES = {np.int8: 1, np.int16: 2, np.int32: 3}


def on_tile(device, wl, rows, K, out):
    """Runs wl on the GPU, on tiles of `rows` and no others."""
    print("[gpu-case]", wl.name, K, flush=True)
    launched = []
    got, _ = run_on_gpu(device, wl, via="device", launched=launched)
    groups = 2 if rows[0] == 32 and K > 128 else 1
    assert launched == ["igemm_rt_i8<%d,%d,%d,%d,%d,0>" % (rows + (DTYPE_CODES[out], groups))], launched
    assert_bit_exact(got[0], oracle_eval(wl)[0], wl.name)


@pytest.mark.parametrize("K", [1, 16, 127, 128, 129, 143, 144, 256, 257, 300, 400, 513])
@pytest.mark.parametrize("sizes, rows", TILES, ids=TILE_IDS)
def test_k_tiles(device, sizes, rows, K):
    """The ends of k-tiles: one, two and an odd number of them, rows of B that end a byte before, at and behind a chunk."""
    B, M, N = sizes
    on_tile(device, w.matmul_workload(B=B, M=M, K=K, N=N, out_dtype=np.int32, seed=K), rows, K, np.int32)


@pytest.mark.parametrize("K", [129, 400])
@pytest.mark.parametrize("kw", [I8, dict(out_dtype=np.int16)], ids=["int8", "int16"])
@pytest.mark.parametrize("sizes, rows", TILES, ids=TILE_IDS)
def test_k_tiles_of_narrow_results(device, sizes, rows, kw, K):
    """Results narrower than the sums behind a loop of several k-tiles, with columns that fill no store."""
    B, M, N = sizes
    on_tile(device, w.matmul_workload(B=B, M=M, K=K, N=N - 1, seed=K, **kw), rows, K, kw["out_dtype"])
