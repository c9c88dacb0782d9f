"""What a decoder does when device memory runs out, and the sizes of its prompt buffers, on a HIP
runtime of host memory (fake_hip.c: launches do nothing, an allocation can be made to fail), so the
host code runs without a GPU: every launch's own checks of its shapes and buffers among it."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["gcc", "-O1", "-Wall", "-shared", "-fPIC", os.path.join(HERE, "fake_hip.c"), "-o", out], check=True)
    return out


PRELUDE = """
import ctypes as C, dataclasses, sys
fake = C.CDLL(sys.argv[1], C.RTLD_GLOBAL)      # before the library: its functions come first
for n in ("fake_live", "fake_allocations", "fake_graph_launches"):
    getattr(fake, n).restype = C.c_long
fake.fake_fail_at.argtypes = [C.c_long]
import numpy as np
from sapphire_amd import model as smodel
from sapphire_amd.engine import Decoder
CFG = dataclasses.replace(smodel.TINY, max_ctx=1100)
"""


def _child(fake, body):
    r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body), fake], cwd=ROOT, capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    return r.stdout.split()


@pytest.mark.parametrize("batch", [1, 4])
def test_every_allocation_failing_in_turn(fake, batch):
    """Creation fails and gives everything back, or, where only the long prompts' buffers are missing,
    succeeds: prompts then run in chunks of 16 (the captured pass of a full chunk is launched). The
    buffers are pieces of larger chunks of memory; of the cache sizes some let the prompt buffers
    begin a chunk."""
    out = _child(fake, f"""
    prompt = np.arange(40, dtype=np.int32)
    chunked = 0
    for ctx in (1100, 20000, 30000, 40000, 50000):
        cfg = dataclasses.replace(CFG, n_layers=1, n_heads=8, n_kv_heads=2, head_dim=256, max_ctx=ctx // {batch})
        m = smodel.synthetic_model(cfg, 5)
        before = fake.fake_allocations()
        Decoder(m, batch={batch}).close()
        total = fake.fake_allocations() - before
        assert fake.fake_live() == 0
        for k in range(1, total + 1):
            fake.fake_fail_at(k)
            try:
                dec = Decoder(m, batch={batch})
            except RuntimeError:
                assert fake.fake_live() == 0, k
                fake.hipGetLastError()         # the failed call's, which the next launch would report
                continue
            launches = fake.fake_graph_launches()
            dec.prefill(prompt, 0)
            assert fake.fake_graph_launches() == launches + 2, k
            dec.close()
            assert fake.fake_live() == 0, k
            chunked += 1
    print(chunked)
    """)
    assert int(out[-1]) >= 1


@pytest.mark.parametrize("heads,kv,hd", [(4, 1, 64), (4, 2, 64), (8, 1, 64), (8, 2, 128), (4, 1, 256)])
def test_prompt_of_every_length_fits_its_buffers(fake, heads, kv, hd):
    """Every launch of a prompt of 17 to 1100 tokens accepts its buffers (the attention's partials
    are checked against theirs), and none of them takes the chunks of 16."""
    _child(fake, f"""
    cfg = dataclasses.replace(CFG, n_layers=2, n_heads={heads}, n_kv_heads={kv}, head_dim={hd}, global_layers=(1,))
    dec = Decoder(smodel.synthetic_model(cfg, 6))
    prompt = np.zeros(1100, np.int32)
    for n in range(17, 1101):
        dec.prefill(prompt[:n], 0)
        if n < 400:
            dec.prefill(prompt[:n], 700)
    assert fake.fake_graph_launches() == 0
    dec.close()
    assert fake.fake_live() == 0
    """)
