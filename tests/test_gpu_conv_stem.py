"""First layers, few channels in planar rows (csrc/conv_stem.hip): bytes, and floats that are quantized on the way in, against the oracle."""
import ctypes
import importlib

import numpy as np
import pytest
import torch

from test_gpu_conv_split import codes, g, pitched  # noqa: F401  (g: the fixture)

pytestmark = pytest.mark.gpu

# N, C, H, W, OC, KH, KW, stride, pad: K blocks of each count that the kernel has code for, filter rows of 4 and of 8 bytes, one and two groups of
# output channels and more than a block of them, no whole 16, tiles over the image's ends, rows of no whole dword and of one, pads wider than
# the image, patches of up to 3 and of up to 8 dwords per thread (the last two)
CASES = [(2, 3, 31, 33, 64, 7, 7, 2, 3), (1, 1, 9, 4, 5, 3, 3, 1, 0), (3, 4, 17, 21, 70, 5, 5, 1, 2), (2, 2, 40, 6, 33, 3, 1, 3, 0), (1, 3, 7, 7, 64, 7, 7, 1, 6), (1, 10, 65, 18, 8, 3, 3, 1, 1),
         (40, 3, 33, 50, 32, 3, 3, 2, 1), (1, 4, 20, 37, 96, 8, 8, 1, 4), (2, 8, 23, 30, 16, 4, 4, 2, 1), (4, 5, 12, 51, 130, 6, 6, 2, 2)]
# zero point of the result, Relu, bias: each form of the requantization
FORMS = [(0, False, 2), (120, False, 1), (5, True, 2), (0, False, 1)]


def operands(oracle, x, case, form, quantization):
    N, C, H, W, OC, KH, KW, stride, pad = case
    rng = np.random.default_rng(OC + W)
    yz, relu, bias_mode = form
    x_scale, x_zp = quantization
    w, ws = codes(rng, (OC, C, KH, KW), np.int8), rng.uniform(0.002, 0.02, size=OC).astype(np.float32)
    y_scale = float(x_scale * 0.01 * 74 * 74 * np.sqrt(C * KH * KW) / 40)
    most = 3000 if bias_mode == 2 else 2 + int(20 * y_scale)  # (added as it is, or at the scale of the products)
    bias = rng.integers(-most, most + 1, size=OC).astype(np.int32)
    want = oracle.qlinear_conv_int(x, x_scale, x_zp, w, ws, np.zeros(OC, np.int8), y_scale, yz, np.uint8, strides=(stride,) * 2, pads=(pad,) * 2, bias=bias,
                                   bias_mode=oracle.BIAS_ONNX_INT32 if bias_mode == 2 else oracle.BIAS_REFERENCE_FLOAT)
    return w, ws, bias, y_scale, np.maximum(want, yz) if relu else want


def plan_of(g, w, ws, bias, case):  # noqa: F811
    return g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(len(ws), np.int8)), g.dev(bias), strides=(case[7],) * 2, pads=(case[8],) * 2)


def flags_of(g, form):  # noqa: F811
    return (0, g.capi.BIAS_REFERENCE_FLOAT, g.capi.BIAS_ONNX_INT32)[form[2]] | (g.capi.FUSE_RELU if form[1] else 0)


# rows of fewer than 4 bytes; tiles whose rows only fit without the columns in front of them (up to 10 dwords per thread)
NARROW = [(2, 3, 9, 3, 7, 3, 3, 1, 1), (3, 3, 5, 1, 40, 3, 3, 1, 1), (2, 1, 18, 2, 64, 7, 7, 2, 3), (1, 2, 3, 3, 33, 4, 4, 1, 3)]
LARGE = [(2, 4, 57, 61, 64, 3, 3, 4, 1), (1, 4, 30, 33, 20, 3, 3, 4, 3)]


@pytest.mark.parametrize("case", CASES + NARROW + LARGE)
def test_codes(g, oracle, case):  # noqa: F811
    for i, form in enumerate(FORMS):
        x = codes(np.random.default_rng(i), case[:4], np.int8 if i % 2 else np.uint8)
        zero_point = (77, -9, 255, -128)[i]
        w, ws, bias, y_scale, want = operands(oracle, x, case, form, (0.02, zero_point))
        plan, out = plan_of(g, w, ws, bias, case), pitched(want.shape, torch.uint8)
        xd = g.dev(x)
        if i == 1:  # a part of a larger image, each row at another byte of its dword
            far = torch.zeros((case[0], case[1] + 1, case[2] + 2, case[3] + 5), dtype=xd.dtype, device="cuda")
            far[:, 1:, 1:-1, 3:-2] = xd
            xd = far[:, 1:, 1:-1, 3:-2]
        plan.run(xd, 0.02, zero_point, y_scale, form[0], flags=flags_of(g, form), out=out)
        assert len(np.unique(want)) > min(20, want.size // 10)
        np.testing.assert_array_equal(g.host(out), want, err_msg=str(form))
        plan.close()


@pytest.mark.parametrize("case", CASES)
def test_floats(g, oracle, case):  # noqa: F811
    rng = np.random.default_rng(case[3])
    for i, form in enumerate(FORMS):
        # (the codes' scale and zero point need not be those that the convolution reads them with)
        scale, zero_point = np.float32((0.02, 1.0, 0.0078125, 12.5)[i]), (0, 128, 255, 3)[i]
        x = (rng.normal(size=case[:4]) * 60 * scale).astype(np.float32)
        flat = x.reshape(-1)
        borders = ((np.arange(flat.size) % 260 - 2.5 - zero_point) * scale).astype(np.float32).view(np.int32) + (np.arange(flat.size) % 5 - 2).astype(np.int32)
        flat[3::7] = borders.view(np.float32)[3::7]
        if i != 1:
            flat[:9] = [np.nan, np.inf, -np.inf, 3e38, -3e38, 1e-42, -0.0, -np.nan, np.float32(2.0 ** -126)]
            flat[-(flat.size // 3):] = rng.integers(0, 1 << 32, size=flat.size // 3, dtype=np.uint32).view(np.float32)
        q = oracle.quantize_linear(x, scale, zero_point, np.uint8)
        w, ws, bias, y_scale, want = operands(oracle, q, case, form, (0.02, 7))
        plan, out = plan_of(g, w, ws, bias, case), pitched(want.shape, torch.uint8)
        xd = g.dev(x)
        if i == 2:
            far = torch.zeros((case[0], case[1] + 1, case[2] + 2, case[3] + 5), device="cuda")
            far[:, 1:, 1:-1, 3:-2] = xd
            xd = far[:, 1:, 1:-1, 3:-2]
        handle = plan._plan_of(g.capi.ConvParams(*(case[7],) * 2, *(case[8],) * 4, 1))
        rc = g.capi.lib().chx_hip_qconv_plan_run_quantize(
            handle, g.capi.ref(xd), ctypes.c_float(scale), zero_point, ctypes.c_float(0.02), 7, ctypes.c_float(y_scale), form[0], ctypes.c_uint32(flags_of(g, form)),
            g.capi.ref(out), g.capi.stream_ptr())
        assert rc == (g.capi.EUNSUPPORTED if case in CASES[-2:] else 0)
        if rc == 0:
            np.testing.assert_array_equal(g.host(out), want, err_msg=str(form))
        plan.close()


# H, kernel, stride, bytes between rows: more than 2^32 from a tile's first row to its last, most of which the image does not have; just less
@pytest.mark.parametrize("H,kernel,stride,row", [(1, 7, 2, 1 << 28), (1, 3, 1, (1 << 30) - 4), (4, 7, 2, 215 << 20), (4, 7, 2, 195 << 20)])
def test_rows_far_apart(g, oracle, H, kernel, stride, row):  # noqa: F811
    case = (1, 3, H, 21, 32, kernel, kernel, stride, kernel // 2)
    for floats in (False, True):
        row = row // 4 if floats else row
        if floats:
            x = (np.random.default_rng(H).normal(size=case[:4]) * 1.2).astype(np.float32)
            q = oracle.quantize_linear(x, np.float32(0.02), 31, np.uint8)
        else:
            x = q = codes(np.random.default_rng(H), case[:4], np.uint8)
        # (the channels lie side by side in each row)
        xd = torch.empty(row * (H - 1) + 64, dtype=torch.float32 if floats else torch.uint8, device="cuda").as_strided(case[:4], (row, 21, row, 1))
        xd.copy_(torch.from_numpy(x))
        w, ws, bias, y_scale, want = operands(oracle, q, case, FORMS[0], (0.02, 31))
        plan, out = plan_of(g, w, ws, bias, case), pitched(want.shape, torch.uint8)
        if floats:
            rc = g.capi.lib().chx_hip_qconv_plan_run_quantize(
                plan._plan_of(g.capi.ConvParams(stride, stride, *(kernel // 2,) * 4, 1)), g.capi.ref(xd), ctypes.c_float(0.02), 31, ctypes.c_float(0.02), 31, ctypes.c_float(y_scale), 0,
                ctypes.c_uint32(flags_of(g, FORMS[0])), g.capi.ref(out), g.capi.stream_ptr())
            assert rc == (g.capi.EUNSUPPORTED if row * 4 == 215 << 20 else 0)
            if rc != 0:
                plan.close()
                continue
        else:
            plan.run(xd, 0.02, 31, y_scale, 0, flags=flags_of(g, FORMS[0]), out=out)
        np.testing.assert_array_equal(g.host(out), want)
        plan.close()


@pytest.mark.parametrize("channels,image,kernel,fused", [(3, 40, 7, True), (3, 33, 3, True), (3, 3, 3, False), (32, 12, 1, False)])
def test_programs(g, oracle, channels, image, kernel, fused):  # noqa: F811
    """QuantizeLinear and the convolution behind it in a program: one launch where the kernel takes them, the two instructions otherwise; eagerly,
    recorded, and with the codes as an output, which keeps the two apart."""
    vm = importlib.import_module(g.pkg.__name__ + ".chxvm")
    case = (2, channels, image, image, 24, kernel, kernel, 1 if image < 20 else 2, kernel // 2)
    rng = np.random.default_rng(channels + image)
    x = (rng.normal(size=case[:4]) * 1.2).astype(np.float32)
    x.reshape(-1)[:3] = [np.nan, np.inf, -np.inf]
    q = oracle.quantize_linear(x, np.float32(0.02), 31, np.uint8)
    w, ws, bias, y_scale, want = operands(oracle, q, case, FORMS[0], (0.02, 31))

    def program(keep_codes):
        b = vm.ProgramBuilder()
        xs = b.input("x", "float32", list(case[:4]))
        s, z = b.scalar(0.02, "float32"), b.scalar(31, "uint8")
        c = b.QuantizeLinear(xs, s, z, debug_info="codes")
        b.Free(xs)
        y = b.QLinearConv(c, b.scalar(0.02, "float32"), b.scalar(31, "uint8"), b.constant(w), b.constant(ws), b.constant(np.zeros(24, np.int8)), b.scalar(y_scale, "float32"),
                          b.scalar(0, "uint8"), b.constant(bias), [case[7]] * 2, [case[8]] * 2, 1, "", debug_info="y")
        if keep_codes:
            b.output("codes", c)
        b.Free(c)
        b.output("y", y)
        return vm.Program(b.serialize())

    for keep_codes in (False, True):
        prog = program(keep_codes)
        prog.set_option("qlinearconv_bias", "onnx_int32")
        before, xd = vm.counter("quantized_convolutions"), torch.from_numpy(x).cuda()
        got = prog.run({"x": xd})
        assert vm.counter("quantized_convolutions") - before == (1 if fused and not keep_codes else 0)
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
