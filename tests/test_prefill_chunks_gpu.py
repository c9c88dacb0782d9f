"""Prompts that run in chunks of 16 tokens against the oracle run one token at a time: those of up to
16 tokens, and longer ones of shapes that the passes of many tokens do not take (an ffn longer than
their GEMMs' rows). A chunk shorter than 16 is launched directly, a full one is captured once per
sequence and replayed."""
import dataclasses

import numpy as np
import pytest

from sapphire_amd import model as smodel
from sapphire_amd import synth
from tests.test_decode_gpu import _compare, _kv_close
from oracle.oracle import oracle_decode, oracle_prefill

pytestmark = pytest.mark.gpu

TINY = smodel.TINY                # local layers slide past 24 positions
WIDE_FFN = dataclasses.replace(TINY, ffn=8320)          # batched decoders only; K above 8192


@pytest.mark.parametrize("cfg,kv0,lengths", [
    (TINY, 0, [1]),
    (TINY, 7, [5, 15]),           # the second prompt behind the first, across the window
    (TINY, 0, [16, 16, 3]),       # the captured pass twice, then a short chunk
    (dataclasses.replace(TINY, n_heads=8, n_kv_heads=2, wdtype=synth.Q8_0), 30, [16, 1, 16]),
    (dataclasses.replace(TINY, head_dim=256, hidden=640, ffn=2048), 3, [16, 9]),
], ids=lambda v: str(v) if not hasattr(v, "ffn") else f"{v.n_heads}x{v.head_dim}")
def test_prompts_of_up_to_16_tokens(oracle, cfg, kv0, lengths):
    from sapphire_amd.engine import Decoder
    n, steps = sum(lengths), 4
    print(f"chunks {cfg.n_layers}x{cfg.hidden} kv0={kv0} lengths={lengths}", flush=True)
    m = smodel.synthetic_model(cfg, 71)
    k, v = m.kv_prefill(kv0)
    prompt = synth.rng(71, n).integers(0, cfg.vocab, n + 1).astype(np.int32)
    dec = Decoder(m)
    dec.set_kv(k, v)
    at = 0
    for c in lengths:
        dec.prefill(prompt[at:at + c], kv0 + at)
        at += c
    gk, gv = dec.get_kv()
    toks, logits, _ = dec.generate(int(prompt[n]), kv0 + n, steps, keep_logits=True)
    dec.close()
    rk, rv = k.copy(), v.copy()
    oracle_prefill(oracle, m, rk, rv, prompt[:n], kv0, nthreads=8)
    assert np.array_equal(gk[:, :, :kv0], k[:, :, :kv0]) and np.array_equal(gv[:, :, :kv0], v[:, :, :kv0])
    assert not gk[:, :, kv0 + n:].any()
    _kv_close(gk, rk, slice(kv0, kv0 + n), "K")
    _kv_close(gv, rv, slice(kv0, kv0 + n), "V")
    ref_toks, ref_logits = oracle_decode(oracle, m, rk, rv, int(prompt[n]), kv0 + n, steps, nthreads=8, keep_logits=True)
    assert _compare(ref_toks, ref_logits, toks, logits) == steps


@pytest.mark.parametrize("cfg,n", [(TINY, 16), (TINY, 11), (WIDE_FFN, 40), (WIDE_FFN, 32)],
                         ids=["one_full_chunk", "one_short_chunk", "16_16_8", "16_16"])
def test_chunks_of_a_batched_decoder(oracle, cfg, n):
    """Two sequences, each twice (the second time by replay), every other cache untouched."""
    from sapphire_amd.engine import Decoder
    print(f"chunks of a batched decoder ffn={cfg.ffn} n={n}", flush=True)
    m = smodel.synthetic_model(cfg, 72)
    kv0 = 9
    k, v = m.kv_prefill(kv0)
    prompts = {s: synth.rng(72, s).integers(0, cfg.vocab, n).astype(np.int32) for s in (0, 2)}
    dec = Decoder(m, batch=3)
    for b in range(3):
        dec.set_kv_seq(b, k, v)
    for _ in range(2):
        for s, p in prompts.items():
            dec.prefill(p, kv0, seq=s)
    got = [dec.get_kv_seq(b) for b in range(3)]
    dec.close()
    assert np.array_equal(got[1][0], k) and np.array_equal(got[1][1], v)
    for s, p in prompts.items():
        rk, rv = k.copy(), v.copy()
        oracle_prefill(oracle, m, rk, rv, p, kv0, nthreads=8)
        _kv_close(got[s][0], rk, slice(kv0, kv0 + n), "K")
        _kv_close(got[s][1], rv, slice(kv0, kv0 + n), "V")
        assert not got[s][0][:, :, kv0 + n:].any()
