"""The TILED GEMV of long rows (K = 1024, 1152) where its waves go from one tile to two and more:
8 waves per CU walk the 16-row tiles, every tile but a wave's last refilled group by group. A row's
arithmetic does not depend on the tile or wave that forms it, so the rows of a matrix are those of
its pieces bit for bit, and these are small enough for the oracle."""
import numpy as np
import pytest

from sapphire_amd import synth
from tests.conftest import close
from tests.test_gemv_gpu import _gemv

pytestmark = pytest.mark.gpu

TILED = 2
ROUND = 256 * 8 * 16          # rows of one tile per wave on 256 CUs


@pytest.mark.parametrize("dtype", [synth.Q4_0, synth.Q8_0], ids=["q4_0", "q8_0"])
@pytest.mark.parametrize("k", [1024, 1152])
@pytest.mark.parametrize("m", [ROUND - 16, ROUND, ROUND + 1, 2 * ROUND, 2 * ROUND + 17])
def test_rows_of_every_tile(hip, oracle, dtype, k, m):
    print(f"gemv tiles dtype={dtype} {m}x{k}", flush=True)
    unit = synth.quant_matrix(dtype, 1009, k, seed=13, tensor_id=k)       # repeats out of step with the tiles
    W = unit[np.arange(m) % 1009]
    x = synth.normal_f32(k, 13, 3)
    ok, err = close(ref := _gemv(hip, dtype, unit, x, TILED), oracle.gemv(dtype, unit, x, nthreads=4))
    assert ok, f"max abs err {err}"
    got = _gemv(hip, dtype, W, x, TILED)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)[np.arange(m) % 1009])
