"""ConvInteger in one launch (csrc/conv_strip.hip): strips that end inside the image, ragged columns, channels and filters,
strides, pads, each layout and signedness, zero points of x and of the weights."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util
    return gpu_util


# N, C, H, W, OC, k, stride, pad: one output row per strip up to the whole image in one; K ending inside a step (C = 20, 3x3)
CASES = [(1, 16, 8, 8, 5, 1, 1, 0), (2, 20, 9, 11, 33, 3, 1, 1), (1, 64, 56, 57, 64, 3, 1, 1), (3, 32, 13, 16, 100, 3, 2, 1), (2, 48, 14, 14, 70, 1, 2, 0),
         (1, 17, 10, 120, 32, 3, 1, 0), (1, 128, 7, 9, 40, 3, 1, 2), (1, 24, 5, 8, 65, 3, 2, 0),
         (16, 20, 12, 40, 33, 3, 1, 1), (40, 32, 15, 13, 70, 3, 2, 1), (33, 64, 7, 9, 130, 1, 1, 0),  # (enough strips for channels-last arrays)
         (8, 900, 3, 3, 512, 3, 1, 0), (8, 1024, 3, 3, 512, 3, 1, 0)]  # the most shared memory a launch takes, and beyond (conv_planar.hip)


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("channels_last", [False, True])
def test_against_the_oracle(g, oracle, case, channels_last):
    N, C, H, W, OC, k, st, pad = case
    rng = np.random.default_rng(OC)
    for xdt, wdt, xz, per_channel in [(np.uint8, np.int8, 128, None), (np.uint8, np.uint8, 3, False), (np.int8, np.int8, -7, True)]:
        lim = {np.uint8: (0, 256), np.int8: (-128, 128)}
        x, w = rng.integers(*lim[xdt], size=(N, C, H, W)).astype(xdt), rng.integers(*lim[wdt], size=(OC, C, k, k)).astype(wdt)
        wz = None if per_channel is None else rng.integers(*lim[wdt], size=OC if per_channel else ()).astype(wdt)
        xd = g.dev(x)
        if channels_last:
            xd = g.to_channels_last(xd)
        got = g.host(g.ops.ConvInteger(xd, g.dev(w), xz, None if wz is None else g.dev(wz), strides=(st, st), pads=(pad, pad)))
        if per_channel:
            want = np.concatenate([oracle.conv_integer(x, w[i:i + 1], xz, wz[i], strides=(st, st), pads=(pad, pad)) for i in range(OC)], axis=1)
        else:
            want = oracle.conv_integer(x, w, xz, wz, strides=(st, st), pads=(pad, pad))
        np.testing.assert_array_equal(got, want)
