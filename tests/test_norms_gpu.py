"""The device norms at the edges of their staging (a thread's loads ahead, the LDS row, rows past
it), bit for bit against the oracle: the sum of squares keeps the reference's order."""
import numpy as np
import pytest

from sapphire_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [1, 7, 8, 127, 128, 135, 256, 257, 2048, 2049, 2567, 8192, 8193])
def test_norms_bit_exact(hip, oracle, dim):
    from sapphire_amd.device import DeviceArray, check
    x = synth.normal_f32((2, dim), 71, dim) * 3
    w = (1 + 0.1 * synth.normal_f32(dim, 71, 1)).astype(np.float32)
    r = synth.normal_f32(dim, 71, 2)
    dx, dw, do = DeviceArray.from_numpy(x), DeviceArray.from_numpy(w), DeviceArray.empty(2 * dim)
    check(hip.sapphire_rmsnorm_delta_dev(do.ptr, dx.ptr, dw.ptr, 1e-6, dim, 2, None))
    ref = np.stack([oracle.rmsnorm_delta(x[b], w) for b in range(2)])
    assert np.array_equal(do.numpy().reshape(2, dim).view(np.uint32), ref.view(np.uint32))
    h, dr = DeviceArray.from_numpy(x[0]), DeviceArray.from_numpy(r)
    check(hip.sapphire_norm_residual_dev(h.ptr, dr.ptr, dw.ptr, 1e-6, dim, None))
    want = (r + ref[0]).astype(np.float32)
    assert np.array_equal(h.numpy().view(np.uint32), want.view(np.uint32))
    assert np.array_equal(dr.numpy().view(np.uint32), want.view(np.uint32))
