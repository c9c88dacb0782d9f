"""Prompts long enough for the many-token path (17 tokens and more) against the oracle run one
token at a time: K/V rows, then greedy decode on top of them. The shapes walk the attention's
forms (head_dim 64 / 128 / 256, 2 / 4 / 8 query heads per K/V head), prompts at the edges of its
tiles and passes, cached positions before the prompt, and windows shorter than the prompt.
"""
import dataclasses

import numpy as np
import pytest

from sapphire_amd import model as smodel
from sapphire_amd import synth
from tests.test_decode_gpu import _compare, _kv_close
from oracle.oracle import oracle_decode, oracle_prefill

pytestmark = pytest.mark.gpu

BASE = smodel.DecodeConfig(n_layers=3, hidden=128, n_heads=4, n_kv_heads=1, head_dim=64, ffn=256, vocab=4096,
                           max_ctx=400, sliding_window=40, global_layers=(1,))


def _cfg(**kw):
    return dataclasses.replace(BASE, **kw)


@pytest.mark.parametrize("cfg,kv0,n", [
    (_cfg(), 0, 17),                                                  # the shortest prompt of the path
    (_cfg(), 5, 333),                                                 # ragged, on a cache
    (_cfg(n_heads=8, hidden=256, wdtype=synth.Q8_0), 0, 64),          # 8 heads per K/V head
    (_cfg(n_heads=4, n_kv_heads=2, head_dim=128), 31, 65),            # 2 per K/V head
    (_cfg(n_heads=8, n_kv_heads=2, head_dim=64), 0, 127),
    (_cfg(head_dim=256, hidden=640, ffn=2048, n_layers=4, sliding_window=64), 3, 200),
    (_cfg(sliding_window=1000), 0, 130),                              # no position slides out
    (_cfg(hidden=1152, ffn=1152, head_dim=256, max_ctx=1200, sliding_window=512), 0, 1100),   # two passes
], ids=lambda v: f"{v.n_heads}x{v.head_dim}-{v.n_kv_heads}kv" if hasattr(v, "n_heads") else str(v))
def test_long_prompt(oracle, cfg, kv0, n):
    from sapphire_amd.engine import Decoder
    steps = 3
    print(f"prompt {cfg.n_layers}x{cfg.hidden} heads {cfg.n_heads}/{cfg.n_kv_heads}x{cfg.head_dim} kv0={kv0} n={n}", flush=True)
    m = smodel.synthetic_model(cfg, 61)
    k, v = m.kv_prefill(kv0)
    prompt = synth.rng(61, n).integers(0, cfg.vocab, n + 1).astype(np.int32)
    dec = Decoder(m)
    dec.set_kv(k, v)
    dec.prefill(prompt[:n], kv0)
    toks, logits, _ = dec.generate(int(prompt[n]), kv0 + n, steps, keep_logits=True)
    gk, gv = dec.get_kv()
    dec.close()
    rk, rv = k.copy(), v.copy()
    oracle_prefill(oracle, m, rk, rv, prompt[:n], kv0, nthreads=8)
    _kv_close(gk, rk, slice(kv0, kv0 + n), "K")
    _kv_close(gv, rv, slice(kv0, kv0 + n), "V")
    ref_toks, ref_logits = oracle_decode(oracle, m, rk, rv, int(prompt[n]), kv0 + n, steps, nthreads=8, keep_logits=True)
    assert _compare(ref_toks, ref_logits, toks, logits) == steps


@pytest.mark.parametrize("bad", [np.nan, np.inf], ids=["nan", "inf"])
def test_long_prompt_non_finite_token(oracle, bad):
    """A token with a non-finite embedding spoils its own rows and those of the later tokens that
    attend to it, and no earlier one: its weight there is 0, and 0 * inf must not be formed."""
    from sapphire_amd.engine import Decoder
    cfg, n, at = BASE, 90, 37
    m = smodel.synthetic_model(cfg, 62)
    prompt = synth.rng(62, 1).integers(0, cfg.vocab - 1, n).astype(np.int32)
    prompt[at] = cfg.vocab - 1
    m.embed_bf16[cfg.vocab - 1, 3] = (np.array([bad], np.float32).view(np.uint32) >> 16).astype(np.uint16)[0]
    k, v = m.kv_prefill(0)
    dec = Decoder(m)
    dec.set_kv(k, v)
    dec.prefill(prompt, 0)
    gk, gv = dec.get_kv()
    dec.close()
    rk, rv = k.copy(), v.copy()
    oracle_prefill(oracle, m, rk, rv, prompt, 0, nthreads=8)
    for got, ref, what in ((gk, rk, "K"), (gv, rv, "V")):
        got, ref = got[:, :, :n], ref[:, :, :n]
        fin = np.isfinite(ref)
        assert fin[:, :, :at].all() and not fin[:, :, at].all()
        assert np.array_equal(np.isfinite(got), fin), f"{what}: non-finite rows differ"
        assert np.abs(got[fin] - ref[fin]).max() <= 2e-3 * np.abs(ref[fin]).max()


def test_long_prompt_cached_keys_without_weight(oracle):
    """Cached keys whose scores are -inf (a run of them that fills a tile of 16 positions) have
    weight 0 and spoil nothing. One dim of the keys is infinite, with the sign against the two
    query heads': a dim that hardly turns with the position, found by trying them on the oracle."""
    from sapphire_amd.engine import Decoder
    cfg = _cfg(n_layers=2, n_heads=4, n_kv_heads=2, head_dim=64, sliding_window=1000, global_layers=(0, 1))
    kv0, n = 64, 20
    m = smodel.synthetic_model(cfg, 63)
    k0, v0 = m.kv_prefill(kv0)
    prompt = np.full(n, 7, np.int32)              # one token: its queries differ by their position only
    rows = slice(kv0, kv0 + n)

    def with_inf(signs):
        k = k0.copy()
        for h, (d, s) in enumerate(signs):
            if d is not None:
                k[0, h, 16:32, d] = s * np.inf
        return k

    def reference(signs):
        rk, rv = with_inf(signs), v0.copy()
        oracle_prefill(oracle, m, rk, rv, prompt, kv0, nthreads=4)
        return rk, rv, np.isfinite(rk[1, :, rows]).all() and np.isfinite(rv[1, :, rows]).all()

    tries = [(d, s) for d in range(63, 47, -1) for s in (1, -1)]
    none = (None, 0)
    signs = [next(t for t in tries if reference([t, none])[2]), next(t for t in tries if reference([none, t])[2])]
    rk, rv, finite = reference(signs)
    assert finite
    dec = Decoder(m)
    dec.set_kv(with_inf(signs), v0)
    dec.prefill(prompt, kv0)
    gk, gv = dec.get_kv()
    dec.close()
    _kv_close(gk, rk, rows, "K")
    _kv_close(gv, rv, rows, "V")
