"""The 3x3 convolution kernel with its pixels in LDS and its weights in registers (csrc/conv_same.hip), each tile forced in turn,
against the oracle."""
import numpy as np
import pytest
import torch

from test_gpu_conv_split import codes, forced, g, pitched  # noqa: F401  (g: the fixture)

pytestmark = pytest.mark.gpu

TILES = [(64, 64, 4), (64, 128, 4), (128, 64, 4), (128, 128, 8)]  # output channels, pixels, wavefronts


class forced_same(forced):
    def __init__(self, tile, **more):
        super().__init__(tile, **more)
        self.env["CHX_HIP_TILE"] = "%d,%d,100,%d" % tile


# N, C, H, W, OC: one pixel, runs over the ends of rows and images, channels that are no whole 64 and K steps of two, four, six, eight and
# sixteen to a tap, output channels over the ends of tiles and of 16, more chunks than a work-group brings at a time
CASES = [(1, 64, 1, 1, 5), (3, 24, 5, 4, 70), (2, 128, 9, 2, 130), (1, 512, 7, 7, 64), (5, 160, 3, 3, 24), (2, 100, 14, 15, 128), (1, 48, 3, 75, 40), (2, 256, 8, 8, 200),
         (7, 64, 11, 13, 64)]


@pytest.mark.parametrize("tile", TILES)
def test_plain(g, oracle, tile):  # noqa: F811
    rng = np.random.default_rng(sum(tile))
    for i, (N, C, H, W, OC) in enumerate(CASES):
        # (zero point of the result, scale per tensor, bias): the product forms with and without a zero point, with a lower bound
        for xdt, xz, yz, relu, per_tensor, bias_mode, minus_128 in [(np.uint8, 0, 0, False, False, 2, False), (np.uint8, 77, 5, True, True, 2, True), (np.int8, -9, 131, False, False, 1, False),
                                                                   (np.int8, -128, 0, False, False, 0, True)]:
            x, w = codes(rng, (N, C, H, W), xdt), codes(rng, (OC, C, 3, 3), np.int8)
            ws, bias = rng.uniform(0.002, 0.02, size=1 if per_tensor else OC).astype(np.float32), rng.integers(-3000, 3000, size=OC).astype(np.int32) if bias_mode else None
            ys = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C * 9) / 40)
            flags = (0, g.capi.BIAS_REFERENCE_FLOAT, g.capi.BIAS_ONNX_INT32)[bias_mode] | (g.capi.FUSE_RELU if relu else 0) | (g.capi.STORE_MINUS_128 if minus_128 else 0)
            if bias_mode == 1:
                ys *= 100  # (the bias is added as it is)
            with forced_same(tile):
                plan = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(len(ws), np.int8)), g.dev(bias) if bias_mode else None, strides=(1, 1), pads=(1, 1))
                xd = g.to_channels_last(g.dev(x)) if C % 16 == 0 else pitched(x.shape, torch.uint8 if xdt == np.uint8 else torch.int8)
                xd.copy_(g.dev(x))
                if i % 2:  # pixels further apart than their channels
                    far = torch.zeros((N, H, W, (C + 15) // 16 * 16 + 48), dtype=xd.dtype, device="cuda")
                    far[..., :C] = xd.permute(0, 2, 3, 1)
                    xd = far[..., :C].permute(0, 3, 1, 2)
                out = pitched((N, OC, H, W), torch.int8 if minus_128 else torch.uint8)
                plan.run(xd, 0.02, xz, ys, yz, flags=flags, out=out)
            okw = dict(bias=bias, bias_mode=oracle.BIAS_ONNX_INT32 if bias_mode == 2 else oracle.BIAS_REFERENCE_FLOAT) if bias_mode else {}
            want = oracle.qlinear_conv_int(x, 0.02, xz, w, np.broadcast_to(ws, (OC,)).copy(), np.zeros(OC, np.int8), ys, yz, np.uint8, pads=(1, 1), **okw)
            if relu:
                want = np.maximum(want, yz)
            got = g.host(out)
            np.testing.assert_array_equal(got.view(np.uint8) ^ 0x80 if minus_128 else got, want, err_msg="case %d %s" % (i, (N, C, H, W, OC, xdt, xz)))
            plan.close()


# (the plan's measured configuration may be this kernel, which has no code for int8 results or rounding to nearest even)
@pytest.mark.parametrize("N,C,HW,OC", [(8, 512, 7, 512), (2, 64, 12, 96)])
def test_one_plan_with_other_quantizations(g, oracle, N, C, HW, OC):  # noqa: F811
    rng = np.random.default_rng(C)
    x, w, ws = codes(rng, (N, C, HW, HW), np.uint8), codes(rng, (OC, C, 3, 3), np.int8), rng.uniform(0.002, 0.02, size=OC).astype(np.float32)
    y_scale = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C * 9) / 40)
    plan, xd = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(OC, np.int8)), None, strides=(1, 1), pads=(1, 1)), g.to_channels_last(g.dev(x))
    for dtype, zero_point, rne in [(np.uint8, 128, False), (np.int8, -5, False), (np.uint8, 128, True), (np.uint8, 0, False), (np.int8, 0, True)]:
        got = plan.run(xd, 0.02, 77, y_scale, zero_point, torch.uint8 if dtype == np.uint8 else torch.int8, flags=g.capi.ROUND_ONNX_RNE if rne else 0)
        want = oracle.qlinear_conv_int(x, 0.02, 77, w, ws, np.zeros(OC, np.int8), y_scale, zero_point, dtype, pads=(1, 1),
                                       round_mode=oracle.ROUND_ONNX_RNE if rne else oracle.ROUND_REFERENCE)
        np.testing.assert_array_equal(g.host(got), want)
    plan.close()
