"""ConvInteger from the weights as they are (csrc/conv_planar.hip) against exact integer arithmetic: layouts, strides,
uneven padding, groups, weight zero points, extents around the tiles, the K steps and the padded rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util
    return gpu_util


def codes(rng, shape, dt):
    lo, hi = (0, 256) if dt == np.uint8 else (-128, 128)
    return rng.integers(lo, hi, size=shape).astype(dt)


# N, C, H, W, OC, KH, KW, strides, pads (begin h, begin w, end h, end w), group
CASES = [
    (1, 16, 1, 1, 1, 1, 1, (1, 1), (0, 0, 0, 0), 1),
    (2, 3, 9, 8, 5, 3, 3, (1, 1), (1, 1, 1, 1), 1),
    (3, 17, 7, 7, 33, 3, 3, (1, 1), (1, 1, 1, 1), 1),
    (8, 64, 14, 14, 64, 3, 3, (1, 1), (1, 1, 1, 1), 1),
    (2, 24, 13, 11, 20, 3, 3, (2, 2), (1, 1, 1, 1), 1),
    (2, 8, 12, 15, 16, 5, 3, (2, 1), (2, 1, 2, 1), 1),
    (1, 40, 10, 9, 70, 1, 1, (2, 2), (0, 0, 0, 0), 1),
    (2, 12, 8, 9, 18, 3, 3, (1, 2), (0, 2, 1, 0), 1),
    (2, 12, 9, 8, 18, 3, 2, (2, 1), (0, 1, 1, 0), 3),
    (4, 130, 5, 70, 40, 3, 3, (1, 1), (1, 1, 1, 1), 1),
    (16, 256, 28, 28, 64, 1, 1, (1, 1), (0, 0, 0, 0), 1),
    (2, 32, 15, 14, 40, 1, 5, (2, 1), (1, 2, 1, 2), 4),  # more output rows than the shared padding leaves room for
    (2, 6, 20, 20, 8, 7, 7, (2, 2), (3, 3, 3, 3), 1),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("channels_last", [False, True])
def test_conv_integer(g, oracle, case, channels_last):
    N, C, H, W, OC, KH, KW, strides, pads, group = case
    rng = np.random.default_rng(C * 31 + OC)
    for xdt, wdt, xz, wz in [(np.uint8, np.int8, 128, np.zeros((), np.int8)), (np.uint8, np.uint8, 3, rng.integers(90, 140, size=OC).astype(np.uint8)),
                             (np.int8, np.int8, -7, rng.integers(-3, 4, size=OC).astype(np.int8)), (np.int8, np.uint8, 0, np.array([128], np.uint8))]:
        x, w = codes(rng, (N, C, H, W), xdt), codes(rng, (OC, C // group, KH, KW), wdt)
        xd = g.to_channels_last(g.dev(x)) if channels_last else g.dev(x)
        got = g.ops.ConvInteger(xd, g.dev(w), xz, g.dev(wz), strides=strides, pads=pads, group=group)
        want = oracle.conv_integer(np.pad(x, ((0, 0), (0, 0), (pads[0], pads[2]), (pads[1], pads[3])), constant_values=xz), w, xz, wz, strides=strides, pads=(0, 0),
                                   group=group)
        np.testing.assert_array_equal(g.host(got), want)
