"""The convolution kernel that streams pixels past weights in LDS (csrc/conv_point.hip), forced: against the oracle for
plain convolutions, against the staged tiles for residual sums, pairs and the minus-128 storage."""
import numpy as np
import pytest
import torch

from test_gpu_conv_split import codes, forced, g, pitched  # noqa: F401 (g is a fixture)

pytestmark = pytest.mark.gpu

POINT, STAGED = (64, 32, 4), (64, 64, 4)

# N, C, H, W, OC: 8192 pixels (the fewest it takes) and ragged numbers of them; one K step of 16 channels up to four;
# tiles of 16 channels that end short, one channel, several chunks of channels
CASES = [(8, 16, 32, 32, 96), (33, 24, 31, 33, 24), (32, 144, 33, 32, 5), (35, 64, 31, 31, 200), (32, 250, 32, 32, 300)]


@pytest.mark.parametrize("case", CASES)
def test_plain(g, oracle, case):
    N, C, H, W, OC = case
    rng = np.random.default_rng(OC)
    for xdt, ydt, xz, yz, bias_mode, rne, relu in [(np.uint8, np.uint8, 0, 0, 2, False, True), (np.uint8, np.uint8, 77, 5, 1, False, True),
                                                   (np.uint8, np.uint8, 3, 120, 2, False, False), (np.int8, np.int8, -9, 5, 0, True, False)]:
        x, w = codes(rng, (N, C, H, W), xdt), codes(rng, (OC, C, 1, 1), np.int8)
        ws, bias = rng.uniform(0.002, 0.02, size=OC).astype(np.float32), rng.integers(-3000, 3000, size=OC).astype(np.int32)
        ys = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C) / 40)
        flags = (g.capi.ROUND_ONNX_RNE if rne else 0) | (g.capi.FUSE_RELU if relu else 0) | (g.capi.BIAS_ONNX_INT32 if bias_mode == 2 else 0)
        got = []
        for tile in (POINT, STAGED):
            with forced(tile):
                plan = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(OC, np.int8)), g.dev(bias) if bias_mode else None)
                got.append(g.host(plan.run(g.to_channels_last(g.dev(x)), 0.02, xz, ys, yz, zero_point_dtype=torch.uint8 if ydt == np.uint8 else torch.int8, flags=flags)))
                plan.close()
        np.testing.assert_array_equal(got[0], got[1])
        okw = dict(bias=bias, bias_mode=oracle.BIAS_ONNX_INT32 if bias_mode == 2 else oracle.BIAS_REFERENCE_FLOAT) if bias_mode else {}
        last = x[-1:, :, -2:]  # the oracle on the last rows
        want = oracle.qlinear_conv_int(last, 0.02, xz, w, ws, np.zeros(OC, np.int8), ys, yz, ydt, round_mode=oracle.ROUND_ONNX_RNE if rne else oracle.ROUND_REFERENCE, **okw)
        np.testing.assert_array_equal(got[0][-1:, :, -2:], np.maximum(want, yz) if relu else want)


@pytest.mark.parametrize("dense_first", [True, False])
def test_one_plan_on_a_dense_image_and_on_crops(g, oracle, dense_first):
    """The configuration measured on a dense image is not the crop's (nothing forced)."""
    rng = np.random.default_rng(7)
    N, C, H, W, OC = 16, 64, 32, 32, 64
    big, w = codes(rng, (N, C, 36, 40), np.uint8), codes(rng, (OC, C, 1, 1), np.int8)
    ws = rng.uniform(0.002, 0.02, size=OC).astype(np.float32)
    ys = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C) / 40)
    plan = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(OC, np.int8)), None)
    bd = g.to_channels_last(g.dev(big))
    views = [(g.to_channels_last(g.dev(big[:, :, :H, :W])), big[:, :, :H, :W]), (bd[:, :, :H, :W], big[:, :, :H, :W]), (bd[:, :, 4:, 8:], big[:, :, 4:, 8:])]
    if not dense_first:
        views.reverse()
    for xd, x in views + views:
        got = g.host(plan.run(xd, 0.02, 128, ys, 128))
        want = oracle.qlinear_conv_int(x[-1:], 0.02, 128, w, ws, np.zeros(OC, np.int8), ys, 128, np.uint8)
        np.testing.assert_array_equal(got[-1:], want)
    plan.close()


@pytest.mark.parametrize("affine", ["1", "0"])
@pytest.mark.parametrize("minus_128", [False, True])
@pytest.mark.parametrize("C,OC", [(48, 40), (200, 72)])
def test_residual_pair_and_storage(g, affine, minus_128, C, OC):
    rng = np.random.default_rng(C)
    results = []
    N, H, W = 33, 31, 33
    x, w = codes(rng, (N, C, H, W), np.uint8), codes(rng, (64 + OC, C, 1, 1), np.int8)
    ws, bias = rng.uniform(0.002, 0.02, size=64 + OC).astype(np.float32), rng.integers(-3000, 3000, size=64 + OC).astype(np.int32)
    ys = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C) / 40)
    flags = g.capi.BIAS_ONNX_INT32 | (g.capi.STORE_MINUS_128 if minus_128 else 0)
    dt = torch.int8 if minus_128 else torch.uint8
    for t in (POINT, STAGED):
        with forced(t, CHX_HIP_AFFINE_RESIDUAL=affine):
            both = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(64 + OC, np.int8)), g.dev(bias))
            one = g.ops.QLinearConvPlan(g.dev(w[:OC]), g.dev(ws[:OC]), g.dev(np.zeros(OC, np.int8)), g.dev(bias[:OC]))
            xd = pitched((N, C, H, W), torch.uint8)
            xd.copy_(g.dev(x))
            out = [pitched((N, 64, H, W), dt), pitched((N, OC, H, W), dt)]
            both.run_pair(xd, 0.02, 3, 64, ys, 120, ys * 1.5, 7, flags=(flags, flags), outs=out)
            results.append([g.host(o) for o in out])
            for relu, rz, oz in [(True, 0, 0), (True, 9, 30), (False, 100, 128)]:
                r = pitched((N, OC, H, W), torch.uint8)
                r.copy_(g.dev(codes(np.random.default_rng(5), (N, OC, H, W), np.uint8)))
                s = pitched((N, OC, H, W), dt)
                one.run_add(xd, 0.02, 3, ys, 120, r, 0.03, rz, 0.05, oz, relu, flags=flags, out=s)
                results[-1].append(g.host(s))
            both.close()
            one.close()
    for a, b in zip(*results):
        np.testing.assert_array_equal(a, b)
        assert a.min() < a.max()
