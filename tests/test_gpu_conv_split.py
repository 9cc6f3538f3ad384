"""The small-tile convolution kernels (csrc/conv_split.hip), each configuration forced in turn: against the oracle for
plain convolutions, against the staged tiles for residual sums, pairs and the minus-128 storage."""
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TILES = [(16, 16, 8), (16, 16, 16), (16, 32, 4), (16, 32, 8), (16, 32, 16), (32, 32, 2), (32, 32, 4), (32, 32, 8), (32, 64, 4), (32, 64, 8)]


@pytest.fixture(scope="module")
def g():
    import gpu_util
    return gpu_util


class forced(object):
    """CHX_HIP_TILE (read when a plan is created) for the plans made inside."""

    def __init__(self, tile, **more):
        self.env = dict({"CHX_HIP_TILE": "%d,%d,0,%d" % tile}, **more)

    def __enter__(self):
        self.before = {k: os.environ.get(k) for k in self.env}
        os.environ.update(self.env)

    def __exit__(self, *a):
        for k, v in self.before.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v


def codes(rng, shape, dt):
    lo, hi = (0, 256) if dt == np.uint8 else (-128, 128)
    return rng.integers(lo, hi, size=shape).astype(dt)


# N, C, H, W, OC, k, stride, pad: one pixel, ragged channels and pixels, K from one step to many, padding wider than a row
CASES = [(1, 16, 1, 1, 5, 1, 1, 0), (1, 64, 7, 7, 70, 1, 1, 0), (2, 24, 9, 5, 33, 3, 1, 1), (1, 128, 7, 7, 128, 3, 1, 1), (3, 96, 8, 8, 100, 1, 2, 0),
         (1, 256, 5, 6, 64, 3, 2, 1), (1, 32, 6, 6, 40, 5, 1, 2), (5, 160, 4, 4, 24, 1, 1, 0), (1, 320, 5, 5, 48, 3, 1, 1)]


@pytest.mark.parametrize("tile", TILES)
def test_plain(g, oracle, tile):
    rng = np.random.default_rng(sum(tile))
    for i, (N, C, H, W, OC, k, st, pad) in enumerate(CASES):
        for xdt, ydt, xz, bias_mode, rne, relu in [(np.uint8, np.uint8, 0, 2, False, False), (np.uint8, np.uint8, 77, 1, False, True), (np.int8, np.int8, -9, 0, True, False)]:
            x, w = codes(rng, (N, C, H, W), xdt), codes(rng, (OC, C, k, k), np.int8)
            ws, bias = rng.uniform(0.002, 0.02, size=OC).astype(np.float32), rng.integers(-3000, 3000, size=OC).astype(np.int32)
            ys = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C * k * k) / 40)
            okw = dict(strides=(st, st), pads=(pad, pad))
            flags = (g.capi.ROUND_ONNX_RNE if rne else 0) | (g.capi.FUSE_RELU if relu else 0)
            if bias_mode:
                okw.update(bias=bias, bias_mode=oracle.BIAS_ONNX_INT32 if bias_mode == 2 else oracle.BIAS_REFERENCE_FLOAT)
                flags |= g.capi.BIAS_ONNX_INT32 if bias_mode == 2 else 0
            with forced(tile):
                plan = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(OC, np.int8)), g.dev(bias) if bias_mode else None, strides=(st, st), pads=(pad, pad))
                got = plan.run(g.to_channels_last(g.dev(x)), 0.02, xz, ys, 5, zero_point_dtype=torch.uint8 if ydt == np.uint8 else torch.int8, flags=flags)
            want = oracle.qlinear_conv_int(x, 0.02, xz, w, ws, np.zeros(OC, np.int8), ys, 5, ydt,
                                           round_mode=oracle.ROUND_ONNX_RNE if rne else oracle.ROUND_REFERENCE, **okw)
            if relu:
                want = np.maximum(want, 5)  # the fused Relu: not below the zero point
            np.testing.assert_array_equal(g.host(got), want, err_msg="case %d %s" % (i, (N, C, H, W, OC, k, st, pad)))
            plan.close()


def pitched(shape, dtype):
    """Channels-last memory with the pixel pitch rounded up to 16 bytes, as the runtime allocates it."""
    n, c, h, w = shape
    return torch.zeros((n, h, w, (c + 15) // 16 * 16), dtype=dtype, device="cuda")[..., :c].permute(0, 3, 1, 2)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("C,OC,k,st,scales", [(48, 64, 3, 1, 64), (80, 70, 3, 2, 70), (16, 4, 1, 1, 4), (144, 68, 1, 2, 1)])
def test_taps_without_padding(g, oracle, tile, C, OC, k, st, scales):
    """Filters of several taps that no pixel has outside the image, one tap; constants of four channels at once and one by one."""
    rng = np.random.default_rng(C + OC)
    x, w = codes(rng, (2, C, 7, 6), np.uint8), codes(rng, (OC, C, k, k), np.int8)
    ws, bias = rng.uniform(0.002, 0.02, size=scales).astype(np.float32), rng.integers(-3000, 3000, size=OC).astype(np.int32)
    ys = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C * k * k) / 40)
    for b in (bias, None):
        with forced(tile):
            plan = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(scales, np.int8)), None if b is None else g.dev(b), strides=(st, st), pads=(0, 0))
            got = plan.run(g.to_channels_last(g.dev(x)), 0.02, 77, ys, 5, zero_point_dtype=torch.uint8, flags=g.capi.BIAS_ONNX_INT32)
        okw = {} if b is None else dict(bias=b, bias_mode=oracle.BIAS_ONNX_INT32)
        want = oracle.qlinear_conv_int(x, 0.02, 77, w, np.broadcast_to(ws, (OC,)).copy(), np.zeros(OC, np.int8), ys, 5, np.uint8, strides=(st, st), pads=(0, 0), **okw)
        np.testing.assert_array_equal(g.host(got), want)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("affine", ["1", "0"])
@pytest.mark.parametrize("minus_128", [False, True])
def test_residual_pair_and_storage(g, tile, affine, minus_128):
    rng = np.random.default_rng(sum(tile) + 1)
    results = []
    N, C, H, W = 2, 48, 7, 6
    x, w = codes(rng, (N, C, H, W), np.uint8), codes(rng, (64 + 40, C, 3, 3), np.int8)
    ws, bias = rng.uniform(0.002, 0.02, size=104).astype(np.float32), rng.integers(-3000, 3000, size=104).astype(np.int32)
    ys = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C * 9) / 40)
    flags = g.capi.BIAS_ONNX_INT32 | (g.capi.STORE_MINUS_128 if minus_128 else 0)
    dt = torch.int8 if minus_128 else torch.uint8
    for t in (tile, (64, 64, 4)):
        with forced(t, CHX_HIP_AFFINE_RESIDUAL=affine):
            both = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(104, np.int8)), g.dev(bias), strides=(1, 1), pads=(1, 1))
            one = g.ops.QLinearConvPlan(g.dev(w[:40]), g.dev(ws[:40]), g.dev(np.zeros(40, np.int8)), g.dev(bias[:40]), strides=(1, 1), pads=(1, 1))
            xd = g.to_channels_last(g.dev(x))
            out = [pitched((N, 64, H, W), dt), pitched((N, 40, H, W), dt)]
            both.run_pair(xd, 0.02, 3, 64, ys, 120, ys * 1.5, 7, flags=(flags, flags), outs=out)
            results.append([g.host(o) for o in out])
            for relu, rz, oz in [(True, 0, 0), (True, 9, 30), (False, 100, 128)]:
                r = pitched((N, 40, H, W), torch.uint8)
                r.copy_(g.dev(codes(np.random.default_rng(5), (N, 40, H, W), np.uint8)))
                s = pitched((N, 40, H, W), dt)
                one.run_add(xd, 0.02, 3, ys, 120, r, 0.03, rz, 0.05, oz, relu, flags=flags, out=s)
                results[-1].append(g.host(s))
            both.close()
            one.close()
    for a, b in zip(*results):
        np.testing.assert_array_equal(a, b)
        assert a.min() < a.max()
