"""The short forms of the uint8 requantization (product_form, csrc/core.hip) in every kernel that takes them: codes over
their whole range at random scales, and at scales that are exact or nearly so, against the oracle."""
import numpy as np
import pytest
import torch

from test_gpu_conv_split import codes, forced, g  # noqa: F401 (g is a fixture)

pytestmark = pytest.mark.gpu

# kind: forced tile (None: the kernel follows from the shape), C, OC, filter, group
KINDS = {"staged": ((64, 64, 4), 16, 32, 1, 1), "point": ((64, 32, 4), 16, 32, 1, 1), "depthwise": (None, 32, 32, 3, 32), "stem": (None, 3, 32, 3, 1)}


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("zero_point,relu", [(0, False), (0, True), (3, True), (128, False), (255, False)])
def test_codes(g, oracle, kind, zero_point, relu):
    tile, C, OC, k, group = KINDS[kind]
    rng = np.random.default_rng(zero_point)
    x, w = codes(rng, (2, C, 64, 64), np.uint8), codes(rng, (OC, C // group, k, k), np.int8)
    ws = rng.uniform(0.002, 0.02, size=OC).astype(np.float32)
    wz = np.zeros(OC, np.int8)
    spread = 0.02 * 0.011 * 74 * 74 * np.sqrt(C // group * k * k)
    for y_scale in [spread / 40, spread / 91.3, float(np.float32(spread / 64)), 2.0 ** round(np.log2(spread / 60)), 3 * 2.0 ** round(np.log2(spread / 180))]:
        with forced(tile or (64, 64, 4)):
            plan = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(wz), None, pads=(k // 2, k // 2), group=group)
            xd = g.dev(x) if kind == "stem" else g.to_channels_last(g.dev(x))
            got = g.host(plan.run(xd, 0.02, 128, y_scale, zero_point, zero_point_dtype=torch.uint8, flags=g.capi.FUSE_RELU if relu else 0))
            plan.close()
        want = oracle.qlinear_conv_int(x, 0.02, 128, w, ws, wz, y_scale, zero_point, np.uint8, pads=(k // 2, k // 2), group=group)
        np.testing.assert_array_equal(got, np.maximum(want, zero_point) if relu else want)
        assert got.max() == 255 or zero_point == 0 and got.max() > 100
