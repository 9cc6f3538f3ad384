"""ConvInteger with 1x1 filters on the product kernels (csrc/contract_api.hip, run_conv_as_product): layouts, odd sizes and zero
points against exact sums in float64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util
    return gpu_util


def codes(rng, shape, dt):
    lo, hi = (0, 256) if dt == np.uint8 else (-128, 128)
    return rng.integers(lo, hi, size=shape).astype(dt)


def layouts(g, x):
    """Planar and channels-last arrays, dense and with gaps behind a pixel's channels or an image."""
    n, c, h, w = x.shape
    d = g.dev(x)
    gaps = torch.zeros((n, c + 3, h, w), dtype=d.dtype, device="cuda")
    gaps[:, :c] = d
    wide = torch.zeros((n, h, w, c + 5), dtype=d.dtype, device="cuda")
    wide[..., :c] = d.permute(0, 2, 3, 1)
    rows = torch.zeros((n, c, h, w + 2), dtype=d.dtype, device="cuda")  # (neither: for the other kernels)
    rows[..., :w] = d
    return [d, g.to_channels_last(d), gaps[:, :c], wide[..., :c].permute(0, 3, 1, 2), rows[..., :w]]


# K below, at and above what the product kernels take and a whole step; one pixel; images whose rows are no whole dwords; one filter
@pytest.mark.parametrize("N,C,H,W,OC", [(2, 15, 5, 5, 8), (3, 16, 7, 9, 5), (1, 64, 1, 1, 33), (5, 40, 13, 13, 17), (2, 33, 1, 6, 1), (1, 200, 31, 3, 130), (9, 264, 28, 28, 72)])
@pytest.mark.parametrize("dts", [(np.uint8, np.int8), (np.int8, np.uint8)])
def test_layouts(g, N, C, H, W, OC, dts):
    rng = np.random.default_rng(C + OC)
    x, w = codes(rng, (N, C, H, W), dts[0]), codes(rng, (OC, C, 1, 1), dts[1])
    x64, w64 = x.astype(np.float64), w[:, :, 0, 0].astype(np.float64)
    for xz, wz in [(0, None), (7, np.asarray(3)), (2, rng.integers(0, 90, size=OC))]:
        wz64 = np.zeros(OC) if wz is None else np.broadcast_to(wz, (OC,))
        want = np.einsum("oc,nchw->nohw", w64 - wz64[:, None], x64 - xz).astype(np.int64).astype(np.int32)  # (exact: below 2^53)
        for xd in layouts(g, x):
            got = g.ops.ConvInteger(xd, g.dev(w), xz, None if wz is None else g.dev(np.asarray(wz).astype(dts[1])))
            np.testing.assert_array_equal(g.host(got), want)


def test_other_geometries(g, oracle):
    rng = np.random.default_rng(1)
    w = codes(rng, (24, 32, 1, 1), np.int8)
    for N, H, W in [(2, 9, 8), (3, 8, 7), (1, 7, 5)]:
        x = codes(rng, (N, 32, H, W), np.uint8)
        for strides, pads in [((2, 2), (0, 0)), ((1, 2), (0, 0)), ((2, 1), (0, 0)), ((3, 3), (0, 0)), ((1, 1), (1, 1))]:
            want = oracle.conv_integer(x, w, 5, np.zeros(24, np.int8), strides=strides, pads=pads)
            for xd in layouts(g, x):
                np.testing.assert_array_equal(g.host(g.ops.ConvInteger(xd, g.dev(w), 5, None, strides=strides, pads=pads)), want)


# 15 G multiply-adds: the packed kernel; with zero points of the filters that are not 0, and at 13 G, the product
@pytest.mark.parametrize("OC", [1160, 1024])
@pytest.mark.parametrize("wz", [0, 3])
def test_large_layers(g, OC, wz):
    rng = np.random.default_rng(OC + wz)
    x, w = codes(rng, (64, 14, 14, 1024), np.uint8), codes(rng, (OC, 1024, 1, 1), np.int8)
    got = g.host(g.ops.ConvInteger(g.dev(x).permute(0, 3, 1, 2), g.dev(w), 5, g.dev(np.asarray(wz, np.int8)))).transpose(0, 2, 3, 1).reshape(-1, OC)
    pixels = sorted({0, 1, 127, 128, len(got) // 2, len(got) - 129, len(got) - 1} | set(range(77, len(got), 997)))
    want = (x.reshape(-1, 1024)[pixels].astype(np.float64) - 5) @ (w[:, :, 0, 0].astype(np.float64) - wz).T  # (exact: below 2^53)
    np.testing.assert_array_equal(got[pixels], want.astype(np.int32))


# where the product would be mostly padding or write parts of lines, and the calls beside those that stay products
@pytest.mark.parametrize("N,C,H,OC,stride", [(51, 216, 7, 1336, 1), (8, 1016, 7, 664, 1), (246, 32, 35, 200, 1), (55, 672, 10, 80, 2), (62, 544, 8, 1312, 2), (135, 552, 14, 304, 2)])
def test_short_and_parted_rows(g, N, C, H, OC, stride):
    rng = np.random.default_rng(N + C)
    x, w = codes(rng, (N, C, H, H), np.uint8), codes(rng, (OC, C, 1, 1), np.int8)
    xd = g.dev(x) if stride == 1 else g.to_channels_last(g.dev(x))
    got = g.host(g.ops.ConvInteger(xd, g.dev(w), 5, None, strides=(stride, stride)))
    for n in {0, 1, N // 2, N - 1}:
        want = np.tensordot(w[:, :, 0, 0].astype(np.float64), x[n, :, ::stride, ::stride].astype(np.float64) - 5, 1)  # (exact: below 2^53)
        np.testing.assert_array_equal(got[n], want.astype(np.int32))
