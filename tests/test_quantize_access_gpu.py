"""The quantizer's unaligned row loads and its row ends (K around multiples of 8 and 32, sources
that start anywhere), its tie and non-finite paths inside waves of ordinary blocks, and the
rounding of halves, bit for bit against the oracle."""
import numpy as np
import pytest

from sapphire_amd import synth
from tests.test_quantize_gpu import BF16, F32, Q4, Q8, source

pytestmark = pytest.mark.gpu


def _run(dtype, src_dtype, src, lead):
    """quantize with the source `lead` elements into its allocation, and the blocks off 16 bytes."""
    from sapphire_amd.device import DeviceArray, check, lib
    m, k = src.shape
    flat = np.concatenate([np.zeros(lead, src.dtype), src.reshape(-1)])
    ds = DeviceArray.from_numpy(flat)
    nb = (k + 31) // 32
    at = 4 * (lead % 4)                                        # the blocks need 4-byte alignment only
    out = DeviceArray(m * nb * synth.BLOCK_BYTES[dtype] + 16)
    check(lib().sapphire_quantize_dev(dtype, src_dtype, ds.ptr + lead * src.itemsize, m, k, out.ptr + at, None))
    raw = out.numpy().tobytes()[at:at + m * nb * synth.BLOCK_BYTES[dtype]]
    return np.frombuffer(raw, synth.block_dtype(dtype)).reshape(m, nb)


@pytest.mark.parametrize("dtype", [Q4, Q8], ids=["q4_0", "q8_0"])
@pytest.mark.parametrize("src_dtype", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("k,lead", [(7, 0), (8, 1), (9, 0), (31, 1), (32, 1), (33, 3), (39, 0), (40, 0), (640, 1), (641, 0), (1147, 5)])
def test_quantize_rows_anywhere(hip, oracle, dtype, src_dtype, k, lead):
    src = source(src_dtype, 67, k, 5 + k)
    ref = oracle.quantize(dtype, src_dtype, src)
    got = _run(dtype, src_dtype, src, lead)
    assert got.tobytes() == np.ascontiguousarray(ref).tobytes()


@pytest.mark.parametrize("dtype", [Q4, Q8], ids=["q4_0", "q8_0"])
def test_quantize_mixed_wave(hip, oracle, dtype):
    """Ordinary blocks beside ties of both signs, halves, zeros and subnormal scales."""
    g = synth.rng(81, 1)
    f = g.standard_normal((64, 640)).astype(np.float32)
    for r in range(0, 64, 3):
        b = int(g.integers(0, 20)) * 32
        f[r, b:b + 32] = np.clip(f[r, b:b + 32], -1, 1)
        f[r, b + int(g.integers(0, 32))], f[r, b + int(g.integers(0, 32))] = 1.5, -1.5
    f[1, :32] = np.arange(-16, 16) * 0.5                       # halves of 1/127 steps' multiples
    f[2, 32:64] = (np.arange(32) - 15.5).astype(np.float32)
    f[2, 32] = 127.0
    f[4, 64:96] = 0.0
    f[5, :32] *= np.float32(1e-39)
    f[7, 96:128] = np.float32(1e-45)
    assert _run(dtype, F32, f, 0).tobytes() == np.ascontiguousarray(oracle.quantize(dtype, F32, f)).tobytes()
