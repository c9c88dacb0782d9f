"""Draws on the running-sum values around the 64-element groups of the sampler's walk, in rows
whose chains cross several binades inside one group (a steep rise) or one per many sub-chunks."""
import numpy as np
import pytest

from tests.test_sampling_gpu import PAD, L, _gpu_sample  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [63, 64, 65, 1023, 1024, 1025, 66000])
@pytest.mark.parametrize("shape", ["flat", "rise", "fall"])
def test_draws_at_group_edges(L, oracle, n, shape):
    i = np.arange(n, dtype=np.float32)
    noise = np.random.default_rng(n).standard_normal(n).astype(np.float32) * np.float32(0.3)
    row = {"flat": noise, "rise": noise + i * np.float32(60.0 / n), "fall": noise - i * np.float32(60.0 / n)}[shape]
    _, w = oracle.sample(row, 1.0, 0.5)
    s = np.add.accumulate(w, dtype=np.float32)[-1]
    cum = np.add.accumulate(w / s, dtype=np.float32)
    idx = sorted({k for e in (0, 64, 128, 960, 1024, 2048, n) for k in (e - 1, e, e + 1) if 0 <= k < n})
    draws = np.array([x for k in idx for x in (cum[k], np.nextafter(cum[k], np.float32(2)))] + [0.0, 1.0], np.float32)
    rows = np.tile(np.concatenate([row, np.zeros(PAD, np.float32)]), (draws.size, 1))
    toks, _ = _gpu_sample(L, rows, n, 1.0, draws)
    for j, r in enumerate(draws):
        hit = np.flatnonzero(cum >= r)
        assert toks[j] == (int(hit[0]) if hit.size else n - 1), (j, float(r))


@pytest.mark.parametrize("n", [4096, 4097])
def test_many_rows_of_each_walk(L, oracle, n):
    """The longest row of the walk that shares a CU and the shortest of the other, in more rows than
    there are CUs: every row its own draw."""
    g = np.random.default_rng(n)
    row = (g.standard_normal(n) * 3).astype(np.float32)
    _, w = oracle.sample(row, 1.0, 0.5)
    s = np.add.accumulate(w, dtype=np.float32)[-1]
    cum = np.add.accumulate(w / s, dtype=np.float32)
    draws = np.concatenate([g.random(298, np.float32), cum[[1023, 4095]]]).astype(np.float32)
    toks, _ = _gpu_sample(L, np.tile(np.concatenate([row, np.zeros(PAD, np.float32)]), (draws.size, 1)), n, 1.0, draws)
    want = [int(np.argmax(cum >= r)) if (cum >= r).any() else n - 1 for r in draws]
    assert toks.tolist() == want
