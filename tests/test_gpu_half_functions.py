"""tanh and the sigmoid of float16 programs (csrc/elementwise_rtc.hip) at every float16 argument: the C library's float32
functions, each operation rounded to float16."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [65536, 63488])
def test_every_argument(oracle, count):
    import gpu_util as g
    x = np.arange(65536, dtype=np.uint16).view(np.float16)
    x = x if count == 65536 else x[~np.isnan(x)][:count]  # without the NaNs no wavefront evaluates anything twice
    prog = g.ops.fusion_program([("x", torch.float16)], [("t", "Tanh", "x"), ("s", "Sigmoid", "x")], [("t", torch.float16), ("s", torch.float16)])
    t, s = (g.host(v) for v in g.ops.ElementWiseNvrtc([g.dev(x)], 2, prog, 31))
    with np.errstate(over="ignore", invalid="ignore", divide="ignore"):
        half = lambda v: v.astype(np.float16)
        want_t = half(oracle.tanh(x.astype(np.float32)))
        d = half(1 + half(oracle.exp(-x.astype(np.float32))).astype(np.float32))
        want_s = half(np.float32(1) / d.astype(np.float32))
    for got, want in ((t, want_t), (s, want_s)):
        np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
        ok = ~np.isnan(want)
        np.testing.assert_array_equal(got[ok].view(np.uint16), want[ok].view(np.uint16))
