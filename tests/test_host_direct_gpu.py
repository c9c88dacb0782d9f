"""kernel_gemv around the length up to which the kernel stores its result straight into host
memory: repeated calls with other vectors, each result complete when the call returns."""
import ctypes as C

import numpy as np
import pytest

from sapphire_amd import synth
from tests.conftest import close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 4097, 16383, 16384, 16385])
@pytest.mark.parametrize("dtype", [synth.Q8_0, synth.BF16], ids=["q8_0", "bf16"])
def test_kernel_gemv_host_result(hip, oracle, m, dtype):
    k = 128
    W = synth.quant_matrix(dtype, m, k, 91) if dtype == synth.Q8_0 else synth.bf16_normal((m, k), 91, 1)
    ctx = hip.kernel_ctx_create(0, 0)
    assert hip.kernel_ctx_init(ctx) == 0
    t = hip.tensor_create_view(dtype, 2, (C.c_int * 2)(m, k), W.ctypes.data)
    try:
        y = np.empty(m, np.float32)
        for call in range(4):
            x = synth.normal_f32(k, 91, 10 + call)
            y.fill(np.nan)
            assert hip.kernel_gemv(ctx, y.ctypes.data, t, x.ctypes.data) == 0
            ok, err = close(y, oracle.gemv(dtype, W, x))
            assert ok, f"call {call}: {err}"
    finally:
        hip.tensor_release(t)
        hip.kernel_ctx_destroy(ctx)
