"""A convolution with 1x1 filters and the DequantizeLinear behind it as one launch (csrc/conv_split.hip), against the oracle."""
import ctypes
import importlib

import numpy as np
import pytest
import torch

from test_gpu_conv_split import codes, g, pitched  # noqa: F401  (g: the fixture)

pytestmark = pytest.mark.gpu

# N, C, H, W, OC, stride: one result, channels and pixels over the ends of tiles of 16 and 32, no whole four channels, K of two steps and of many
CASES = [(1, 64, 1, 1, 1, 1), (128, 1280, 1, 1, 1000, 1), (33, 512, 1, 1, 10, 1), (5, 48, 7, 3, 37, 1), (2, 100, 9, 8, 66, 2), (64, 2048, 1, 1, 1000, 1), (3, 16, 17, 1, 15, 1)]


@pytest.mark.parametrize("case", CASES)
def test_floats(g, oracle, case):  # noqa: F811
    N, C, H, W, OC, stride = case
    rng = np.random.default_rng(C + OC)
    for xdt, xz, ydt, yz, bias_mode, relu, rne, dqz in [(np.uint8, 77, np.uint8, 120, 2, False, False, 120), (np.int8, -9, np.uint8, 0, 1, True, False, 3), (np.uint8, 0, np.int8, -7, 0, False, True, -7)]:
        x, w, ws = codes(rng, (N, C, H, W), xdt), codes(rng, (OC, C, 1, 1), np.int8), rng.uniform(0.002, 0.02, size=OC).astype(np.float32)
        y_scale = np.float32(0.02 * 0.01 * 74 * 74 * np.sqrt(C) / 40)
        most = 3000 if bias_mode == 2 else 2 + int(20 * y_scale)
        bias = rng.integers(-most, most + 1, size=OC).astype(np.int32) if bias_mode else None
        okw = dict(bias=bias, bias_mode=oracle.BIAS_ONNX_INT32 if bias_mode == 2 else oracle.BIAS_REFERENCE_FLOAT) if bias_mode else {}
        want = oracle.qlinear_conv_int(x, 0.02, xz, w, ws, np.zeros(OC, np.int8), y_scale, yz, ydt, strides=(stride,) * 2, round_mode=oracle.ROUND_ONNX_RNE if rne else oracle.ROUND_REFERENCE, **okw)
        want = oracle.dequantize_linear(np.maximum(want, yz).astype(ydt) if relu else want, np.float32(0.37), dqz)
        plan = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(OC, np.int8)), g.dev(bias) if bias_mode else None, strides=(stride,) * 2)
        xd = pitched(x.shape, torch.uint8 if xdt == np.uint8 else torch.int8)
        xd.copy_(g.dev(x))
        handle = plan._plan_of(g.capi.ConvParams(stride, stride, 0, 0, 0, 0, 1))
        flags = (0, g.capi.BIAS_REFERENCE_FLOAT, g.capi.BIAS_ONNX_INT32)[bias_mode] | (g.capi.FUSE_RELU if relu else 0) | (g.capi.ROUND_ONNX_RNE if rne else 0)
        for room in (0, 5):  # (pixels further apart than their channels)
            out = torch.full((N,) + want.shape[2:] + (OC + room,), -1.0, device="cuda")[..., :OC].permute(0, 3, 1, 2)
            for _ in range(2):  # (measured, and from what was measured)
                g.capi.check(g.capi.lib().chx_hip_qconv_plan_run_dequantize(
                    handle, g.capi.ref(xd), ctypes.c_float(0.02), xz, ctypes.c_float(y_scale), yz, g.capi.INT8 if ydt == np.int8 else g.capi.UINT8, ctypes.c_uint32(flags), ctypes.c_float(0.37), dqz,
                    g.capi.ref(out), g.capi.stream_ptr()))
            np.testing.assert_array_equal(g.host(out), want)
        # the same plan still gives codes
        got = plan.run(xd, 0.02, xz, y_scale, yz, torch.uint8 if ydt == np.uint8 else torch.int8, flags=flags)
        np.testing.assert_array_equal(oracle.dequantize_linear(g.host(got), np.float32(0.37), dqz), want)
        plan.close()


@pytest.mark.parametrize("N,C,H,OC,kernel,fused", [(3, 64, 1, 100, 1, True), (2, 48, 5, 32, 1, True), (1, 32, 1, 17, 1, True), (2, 64, 6, 32, 3, False), (2, 3, 4, 32, 1, False), (60, 64, 20, 64, 1, False)])
def test_programs(g, oracle, N, C, H, OC, kernel, fused):  # noqa: F811
    """One launch where the kernel takes them, the two instructions otherwise, with the same arrays; eagerly, recorded, and with the codes as an
    output, which keeps the two apart."""
    vm = importlib.import_module(g.pkg.__name__ + ".chxvm")
    rng = np.random.default_rng(C)
    x, w, ws, bias = codes(rng, (N, C, H, H), np.uint8), codes(rng, (OC, C, kernel, kernel), np.int8), rng.uniform(0.002, 0.02, size=OC).astype(np.float32), rng.integers(-3000, 3000, size=OC).astype(np.int32)
    y_scale = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C * kernel * kernel) / 40)
    q = oracle.qlinear_conv_int(x, 0.02, 77, w, ws, np.zeros(OC, np.int8), y_scale, 120, np.uint8, pads=(kernel // 2,) * 2, bias=bias, bias_mode=oracle.BIAS_ONNX_INT32)
    want = oracle.dequantize_linear(q, np.float32(y_scale), 120)
    for keep_codes in (False, True):
        b = vm.ProgramBuilder()
        xs = b.input("x", "uint8", list(x.shape))
        ys, yz = b.scalar(y_scale, "float32"), b.scalar(120, "uint8")
        c = b.QLinearConv(xs, b.scalar(0.02, "float32"), b.scalar(77, "uint8"), b.constant(w), b.constant(ws), b.constant(np.zeros(OC, np.int8)), ys, yz, b.constant(bias),
                          [1, 1], [kernel // 2] * 2, 1, "")
        b.Free(xs)
        f = b.DequantizeLinear(c, ys, yz)
        if keep_codes:
            b.output("codes", c)
        b.Free(c)
        b.output("y", f)
        prog = vm.Program(b.serialize())
        prog.set_option("qlinearconv_bias", "onnx_int32")
        xd = g.to_channels_last(torch.from_numpy(x).cuda()) if C % 16 == 0 else torch.from_numpy(x).cuda()
        before = vm.counter("dequantized_convolutions")
        got = prog.run({"x": xd})
        assert vm.counter("dequantized_convolutions") - before == (1 if fused and not keep_codes else 0)
        np.testing.assert_array_equal(got["y"], want)
        if keep_codes:
            np.testing.assert_array_equal(got["codes"], q)
        replay = prog.capture({"x": xd})
        for i in range(3):
            xd.copy_(torch.from_numpy(np.roll(x, i, axis=0)))
            torch.cuda.synchronize()
            replay.launch()
            replay.synchronize()
            np.testing.assert_array_equal(replay.outputs()["y"], np.roll(want, i, axis=0))
        replay.close()
