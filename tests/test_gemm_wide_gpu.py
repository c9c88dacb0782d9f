"""More than 16 activation vectors through one quantized matrix (gemm_wide.hip) against the
float64 products of the dequantized weights, at the edges of its tiles: 32 tokens, 64 / 128 / 256
rows, K chunks of 32 blocks, K splits, passes of 512 tokens.

Tolerance: an output is a float32 sum of K products in chunks, each product with a relative error
of at most 2^-21 (two fp16 terms), so |error| <= (2^-21 + 2 sqrt(K) 2^-24) sum |w x| with room for
the order of the sums; a wrong or missing product is of the order of sum |w x| / K.
"""
import ctypes

import numpy as np
import pytest

import sapphire_amd
from sapphire_amd import synth
from tests.test_gemm_gpu import TILED, _gemm, _ref
from tests.test_nonfinite_gpu import _matrix, _patterns, _same_special

pytestmark = pytest.mark.gpu

CASES = [                 # m, k, batch
    (1, 128, 17),         # one row, one group, the first batch of the path
    (16, 1024, 32),       # one tile, one whole chunk
    (65, 1152, 33),       # a remainder of everything: chunk + one group, 32 + 1 tokens
    (640, 2048, 64),      # K split
    (1152, 6912, 100),    # K split, chunks cut by the split
    (129, 8192, 31),      # the longest K
    (130, 8320, 20),      # past it: passes of 16
    (4111, 640, 512),     # the 256-row tile (Q8_0: 128), one full pass
    (8192, 256, 300),
    (384, 384, 513),      # two passes, the second of one token
]


@pytest.mark.parametrize("dtype", [synth.Q4_0, synth.Q8_0], ids=["q4_0", "q8_0"])
@pytest.mark.parametrize("m,k,batch", CASES, ids=lambda v: str(v))
def test_gemm_wide(hip, dtype, m, k, batch):
    from sapphire_amd.device import QMatrix
    print(f"wide gemm dtype={dtype} {m}x{k} batch={batch}", flush=True)
    W = synth.quant_matrix(dtype, m, k, seed=51, tensor_id=m + k)
    X = synth.normal_f32((batch, k), 51, batch)
    X *= np.exp2(synth.rng(51, 9).integers(-20, 20, (batch, 1))).astype(np.float32)
    X[batch // 2] = 0.0
    X[0, k // 2] *= np.float32(4096.0)             # one chunk's range far from the others'
    got = _gemm(hip, QMatrix(dtype, W, layout=TILED), X)
    w = synth.unpack_ints(dtype, W).astype(np.float64) * np.repeat(W["scale"].astype(np.float64), 32, axis=1)
    ref, mag = X.astype(np.float64) @ w.T, np.abs(X.astype(np.float64)) @ np.abs(w).T
    bound = (2.0 ** -21 + 2.0 * np.sqrt(k) * 2.0 ** -24) * mag
    assert np.all(np.abs(got - ref) <= bound), f"worst {np.max(np.abs(got - ref) / np.maximum(bound, 1e-300)):.2f} of the bound"


def _plan(dtype, m, k, tokens):
    """(rows of the workgroup tile, K splits) that the library chooses on this device."""
    lib = ctypes.CDLL(sapphire_amd.LIB_PATH)         # C++ functions of the library, not of its API
    return tuple(getattr(lib, f"_ZN8sapphire{len(n)}{n}Eiiii")(dtype, m, k, tokens)
                 for n in ("gemm_wide_tile_rows", "gemm_wide_splits"))


def test_cases_reach_every_tile(hip):
    """The shapes above and below, on 256 CUs: each (dtype, tile) instance, its K splits, and beside
    the 64-row tile also K past the two-level sums' (2304)."""
    want = {
        (640, 2048, 64): [(64, True), (64, True)],
        (4111, 640, 512): [(256, False), (128, False)],
        (8192, 256, 300): [(256, False), (128, False)],
        (2305, 1152, 500): [(128, False), (128, False)],
        (4111, 2560, 300): [(128, False), (128, False)],
        (1152, 6912, 100): [(64, True), (64, True)],
    }
    for (m, k, t), tiles in want.items():
        for dtype, (rows, split) in zip((synth.Q4_0, synth.Q8_0), tiles):
            got = _plan(dtype, m, k, t)
            assert (got[0], got[1] > 1) == (rows, split), f"{m}x{k} {t} tokens dtype {dtype}: {got}"
    assert set(want) <= set(CASES) | set(TILE_CASES)


TILE_CASES = [            # the 128-row tile of both dtypes, ragged in rows and tokens
    (2305, 1152, 500),
    (4111, 2560, 300),    # K past the two-level sums of the 256-row tile
]


@pytest.mark.parametrize("dtype", [synth.Q4_0, synth.Q8_0], ids=["q4_0", "q8_0"])
@pytest.mark.parametrize("m,k,batch", TILE_CASES, ids=lambda v: str(v))
def test_gemm_wide_128_row_tile(hip, dtype, m, k, batch):
    test_gemm_wide(hip, dtype, m, k, batch)


@pytest.mark.parametrize("dtype", [synth.Q4_0, synth.Q8_0], ids=["q4_0", "q8_0"])
@pytest.mark.parametrize("m,k,batch", [(2305, 1152, 500), (4111, 640, 512)], ids=lambda v: str(v))
def test_gemm_wide_non_finite_in_larger_tiles(hip, oracle, dtype, m, k, batch):
    """Special values in the 128- and 256-row tiles: in their own vectors' rows, and nowhere else."""
    from sapphire_amd.device import QMatrix
    W = _matrix(dtype, m, k, 55)
    X = synth.normal_f32((batch, k), 55, 5)
    at = (0, 33, 64, batch - 1)
    for b, x in zip(at, _patterns(k, 56).values()):
        X[b] = x
    got = _gemm(hip, QMatrix(dtype, W, layout=TILED), X)
    ref = _ref(oracle, dtype, W, X[list(at)])
    for i, b in enumerate(at):
        _same_special(got[b], ref[i])
    assert np.isfinite(np.delete(got, at, axis=0)).all()


@pytest.mark.parametrize("dtype", [synth.Q4_0, synth.Q8_0], ids=["q4_0", "q8_0"])
@pytest.mark.parametrize("m,k", [(96, 1152), (80, 6912)])
def test_gemm_wide_non_finite(hip, oracle, dtype, m, k):
    """NaN and infinite activations (also with K split) give the oracle's special values, in
    their own rows only."""
    from sapphire_amd.device import QMatrix
    W = _matrix(dtype, m, k, 52)
    X = synth.normal_f32((40, k), 52, 5)
    for b, x in zip((1, 17, 32, 39), _patterns(k, 53).values()):
        X[b] = x
    got = _gemm(hip, QMatrix(dtype, W, layout=TILED), X)
    ref = _ref(oracle, dtype, W, X)
    for b in range(40):
        _same_special(got[b], ref[b])


@pytest.mark.parametrize("m,k,batch", [(300, 96, 17), (16, 136, 32), (2048, 640, 33), (40000, 264, 31), (150000, 128, 48)],
                         ids=lambda v: str(v))
def test_gemm_bf16_two_token_tiles(hip, m, k, batch):
    """17 to 32 vectors in one pass over BF16 weights (K remainders of a 128-element chunk, every
    number of tiles per wave, a last pass of one tile). Products are exact in three terms, so the
    bound is the fp32 sum's: 2 sqrt(3 K) 2^-24 of sum |w x|, and one vector's bits do not depend on
    how many share the pass."""
    from tests.test_gemv_f_gpu import run_gemm_bf16
    W = synth.bf16_normal((m, k), 54, m)
    X = synth.normal_f32((batch, k), 54, 2)
    got = run_gemm_bf16(W, X)
    w = (W.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    ref, mag = X.astype(np.float64) @ w.T, np.abs(X.astype(np.float64)) @ np.abs(w).T
    assert np.all(np.abs(got - ref) <= 2.0 * np.sqrt(3 * k) * 2.0 ** -24 * mag)
    assert np.array_equal(run_gemm_bf16(W, X[:5]), got[:5])
