"""The small-tile convolution kernels whose pixels come from LDS (csrc/conv_split.hip, kPatch), each configuration forced
in turn: against the oracle for plain convolutions, against the staged tiles for residual sums, pairs and storage."""
import numpy as np
import pytest
import torch

from test_gpu_conv_split import TILES, codes, forced, g, pitched  # noqa: F401  (g: the fixture)

pytestmark = pytest.mark.gpu


class forced_patch(forced):
    def __init__(self, tile, **more):
        super().__init__(tile, **more)
        self.env["CHX_HIP_TILE"] = "%d,%d,1,%d" % tile


# N, C, H, W, OC, k, pad: windows over the ends of rows and images, one pixel, fewer columns than the filter, channels that
# are no whole 16 or 64, more chunks than a work-group loads at once, a form it refuses (the result's size differs)
CASES = [(1, 16, 1, 1, 5, 3, 1), (3, 24, 5, 4, 33, 3, 1), (2, 64, 9, 2, 70, 5, 2), (1, 512, 7, 7, 64, 3, 1), (5, 160, 3, 3, 24, 3, 1), (2, 128, 14, 15, 128, 3, 1),
         (1, 48, 3, 75, 40, 3, 1), (1, 96, 6, 6, 40, 3, 0)]


@pytest.mark.parametrize("tile", TILES)
def test_plain(g, oracle, tile):  # noqa: F811
    rng = np.random.default_rng(sum(tile))
    for i, (N, C, H, W, OC, k, pad) in enumerate(CASES):
        for xdt, ydt, xz, rne, relu in [(np.uint8, np.uint8, 0, False, False), (np.uint8, np.uint8, 77, False, True), (np.int8, np.int8, -9, True, False)]:
            x, w = codes(rng, (N, C, H, W), xdt), codes(rng, (OC, C, k, k), np.int8)
            ws, bias = rng.uniform(0.002, 0.02, size=OC).astype(np.float32), rng.integers(-3000, 3000, size=OC).astype(np.int32)
            ys = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C * k * k) / 40)
            flags = g.capi.BIAS_ONNX_INT32 | (g.capi.ROUND_ONNX_RNE if rne else 0) | (g.capi.FUSE_RELU if relu else 0)
            with forced_patch(tile):
                plan = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(OC, np.int8)), g.dev(bias), strides=(1, 1), pads=(pad, pad))
                xd = g.to_channels_last(g.dev(x))
                if i % 2:  # pixels further apart than their channels
                    far = torch.zeros((N, H, W, (C + 15) // 16 * 16 + 48), dtype=xd.dtype, device="cuda")
                    far[..., :C] = xd.permute(0, 2, 3, 1)
                    xd = far[..., :C].permute(0, 3, 1, 2)
                got = plan.run(xd, 0.02, xz, ys, 5, zero_point_dtype=torch.uint8 if ydt == np.uint8 else torch.int8, flags=flags)
            want = oracle.qlinear_conv_int(x, 0.02, xz, w, ws, np.zeros(OC, np.int8), ys, 5, ydt, strides=(1, 1), pads=(pad, pad), bias=bias,
                                           bias_mode=oracle.BIAS_ONNX_INT32, round_mode=oracle.ROUND_ONNX_RNE if rne else oracle.ROUND_REFERENCE)
            if relu:
                want = np.maximum(want, 5)  # the fused Relu: not below the zero point
            np.testing.assert_array_equal(g.host(got), want, err_msg="case %d %s" % (i, (N, C, H, W, OC, k, pad)))
            plan.close()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("minus_128", [False, True])
def test_residual_pair_and_storage(g, tile, minus_128):  # noqa: F811
    rng = np.random.default_rng(sum(tile) + 1)
    results = []
    N, C, H, W = 2, 48, 7, 6
    x, w = codes(rng, (N, C, H, W), np.uint8), codes(rng, (64 + 40, C, 3, 3), np.int8)
    ws, bias = rng.uniform(0.002, 0.02, size=104).astype(np.float32), rng.integers(-3000, 3000, size=104).astype(np.int32)
    ys = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C * 9) / 40)
    flags = g.capi.BIAS_ONNX_INT32 | (g.capi.STORE_MINUS_128 if minus_128 else 0)
    dt = torch.int8 if minus_128 else torch.uint8
    for force in (forced_patch(tile), forced((64, 64, 4))):
        with force:
            both = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(104, np.int8)), g.dev(bias), strides=(1, 1), pads=(1, 1))
            one = g.ops.QLinearConvPlan(g.dev(w[:40]), g.dev(ws[:40]), g.dev(np.zeros(40, np.int8)), g.dev(bias[:40]), strides=(1, 1), pads=(1, 1))
            xd = g.to_channels_last(g.dev(x))
            out = [pitched((N, 64, H, W), dt), pitched((N, 40, H, W), dt)]
            both.run_pair(xd, 0.02, 3, 64, ys, 120, ys * 1.5, 7, flags=(flags, flags), outs=out)
            r = pitched((N, 40, H, W), torch.uint8)
            r.copy_(g.dev(codes(np.random.default_rng(5), (N, 40, H, W), np.uint8)))
            s = pitched((N, 40, H, W), dt)
            one.run_add(xd, 0.02, 3, ys, 120, r, 0.03, 9, 0.05, 30, True, flags=flags, out=s)
            results.append([g.host(o) for o in out] + [g.host(s)])
            both.close()
            one.close()
    for a, b in zip(*results):
        np.testing.assert_array_equal(a, b)
        assert a.min() < a.max()
