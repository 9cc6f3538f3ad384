"""QuantizeLinear / DequantizeLinear where the last vector is not whole and where the arrays start anywhere."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1024, 1026, (1 << 24) + 3])
@pytest.mark.parametrize("start", [0, 1, 3])
def test_remainders_and_starts(oracle, n, start):
    import gpu_util as g
    x = (np.random.default_rng(n).standard_normal(n + 3) * 2).astype(np.float32)
    for dt, zp in ((np.uint8, 120), (np.int8, 0)):
        q = g.ops.QuantizeLinear(g.dev(x)[start:start + n], 0.03, zp, g.dev(np.zeros(1, dt)).dtype)
        want = oracle.quantize_linear(x[start:start + n], 0.03, zp, dt)
        np.testing.assert_array_equal(g.host(q), want)
        codes = torch.zeros(n + 3, dtype=q.dtype, device="cuda")
        codes[start:start + n] = q
        np.testing.assert_array_equal(g.host(g.ops.DequantizeLinear(codes[start:start + n], 0.03, zp)), oracle.dequantize_linear(want, 0.03, zp))
        out = torch.full((n + 4,), 7, dtype=q.dtype, device="cuda")  # nothing around the result is written
        g.ops.QuantizeLinear(g.dev(x)[start:start + n], 0.03, zp, q.dtype, out=out[start:start + n])
        np.testing.assert_array_equal(g.host(out), np.concatenate([np.full(start, 7, dt), want, np.full(4 - start, 7, dt)]))
