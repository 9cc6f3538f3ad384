"""The tail of a bottleneck block and the next block's reduction as one launch (csrc/bottleneck.hip): whole networks against the
oracle, value by value, and single blocks at the edges of the kernel's tiles with quantizations that no network here has."""
import ctypes
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util
    gpu_util.capi.init(0)
    return gpu_util


@pytest.fixture(scope="module")
def vm(g):
    return importlib.import_module(g.pkg.__name__ + ".chxvm")


# batch, image, blocks per stage; the launches of them that are one.  Odd images, a stage whose last block has no reduction
# behind it, many images for the 256 channels of the third stage.
@pytest.mark.parametrize("batch,image,blocks,fused", [(2, 64, (3, 2), 5), (3, 50, (1, 2, 1), 3), (40, 224, (1, 1, 3), 5)])
def test_networks(g, vm, oracle, batch, image, blocks, fused):
    wl = g.pkg.workloads
    model = wl.build_resnet50(batch=batch, image=image, seed=batch, blocks=blocks, classes=10)
    # the sums, and the values that the next block's convolutions take (a value that is kept has another reader)
    keep = ["logits"] + [ins[1] for ins in model["program"] if ins[0] == "AddRelu" or ins[1].endswith("_a")]
    prog = vm.Program(wl.program_to_chxvm(model, vm, g.pkg.ops, keep=keep).serialize())
    plain = vm.Program(wl.program_to_chxvm(model, vm, g.pkg.ops).serialize())
    x = torch.from_numpy(model["input"]).cuda()
    picks = list(range(batch)) if batch < 8 else [0, batch // 2, batch - 1]
    oracle.set_threads(16)
    try:
        ref = wl.run_reference(model, oracle, model["input"][picks], keep=set(keep))
    finally:
        oracle.set_threads(1)
    for p in (prog, plain):
        p.set_option("qlinearconv_bias", "onnx_int32")
        before = vm.counter("bottlenecks")
        got = p.run({"x": x})
        assert vm.counter("bottlenecks") - before == fused
        for name in got:
            np.testing.assert_array_equal(got[name][picks], ref[name], err_msg=name)
    replay = plain.capture({"x": x})
    for i in range(3):
        x.copy_(torch.from_numpy(np.roll(model["input"], i, axis=0)))
        torch.cuda.synchronize()
        replay.launch()
        replay.synchronize()
        np.testing.assert_array_equal(replay.outputs()["logits"], plain.run({"x": x})["logits"])
    replay.close()


# channels (in between, behind the sum, of the reduction or 0), N, H, W, x's type and zero point, zero points of the convolutions and of
# the sum, scales per tensor, bias, Relu, results stored as code - 128.  Pixels at the edges of tiles of 32 and 64, rows and columns of
# one, an image wider than a tile, several tiles of channels of the reduction for a wavefront or for none.
BLOCKS = [
    ((64, 256, 64), 1, 1, 1, np.uint8, 77, (13, 200, 128), 40, False, True, True, False),
    ((64, 256, 64), 1, 7, 9, np.int8, -9, (0, 0, 5), 0, True, False, False, True),
    ((64, 256, 0), 2, 8, 8, np.uint8, 0, (0, 128, 0), 0, False, True, True, True),
    ((64, 256, 288), 5, 13, 1, np.int8, 100, (255, 9, 117), 150, False, True, True, False),
    ((64, 256, 32), 1, 3, 90, np.uint8, 255, (128, 128, 3), 77, True, False, False, True),
    ((64, 256, 128), 2, 1, 97, np.int8, 0, (0, 100, 0), 0, False, True, True, True),
    ((128, 512, 128), 1, 1, 31, np.uint8, 4, (60, 61, 62), 3, True, True, False, False),
    ((128, 512, 160), 3, 11, 3, np.int8, -128, (0, 131, 0), 0, False, True, True, True),
    ((128, 256, 0), 5, 5, 13, np.uint8, 131, (31, 7, 90), 90, False, False, True, False),
    ((128, 512, 256), 31, 29, 29, np.int8, -128, (0, 117, 0), 0, False, True, True, True),
    ((256, 1024, 256), 13, 14, 15, np.int8, -128, (0, 131, 0), 0, False, True, True, True),
    ((256, 1024, 64), 51, 14, 14, np.uint8, 33, (7, 99, 201), 13, False, True, False, False),
    ((256, 512, 0), 60, 7, 21, np.int8, 5, (0, 0, 0), 0, True, True, True, True),
    # more tiles than two groups of wavefronts are for (512), and as many; rows whose pixels fit for one group only
    ((64, 256, 64), 11, 55, 55, np.int8, -128, (0, 117, 0), 0, False, True, True, True),
    ((64, 256, 0), 32, 32, 32, np.uint8, 9, (5, 77, 0), 30, False, True, True, False),
    ((128, 512, 128), 20, 29, 29, np.uint8, 50, (0, 131, 0), 0, True, True, True, False),
    ((128, 512, 96), 16, 32, 32, np.int8, -128, (0, 131, 9), 11, False, False, False, True),
    ((64, 256, 64), 1, 2, 831, np.uint8, 3, (0, 128, 0), 0, False, True, True, True),
    ((128, 512, 128), 2, 1, 447, np.int8, -128, (1, 130, 2), 5, False, True, False, False),
]


@pytest.mark.parametrize("case", range(len(BLOCKS)))
def test_single_blocks(g, oracle, case):
    (mid, wide, nxt), N, H, W, x_type, x_zp, zero_points, out_zp, per_tensor, bias, relu, minus_128 = BLOCKS[case]
    from test_gpu_conv_split import codes, pitched
    rng = np.random.default_rng(case)
    lib, capi = g.capi.lib(), g.capi
    operands, kept, scales = [], [], []

    def convolution(h, scale, zp, shape, i):
        w, n = codes(rng, shape, np.int8), 1 if per_tensor else shape[0]
        ws, b = rng.uniform(0.002, 0.02, size=n).astype(np.float32), rng.integers(-3000, 3000, size=shape[0]).astype(np.int32) if bias else None
        y_scale = np.float32(scale * ws.mean() * 74 * 74 * np.sqrt(np.prod(shape[1:])) / 60)
        okw = dict(bias=b, bias_mode=oracle.BIAS_ONNX_INT32) if bias else {}
        y = oracle.qlinear_conv_int(h, scale, zp, w, np.broadcast_to(ws, shape[:1]).copy(), np.zeros(shape[0], np.int8), y_scale, zero_points[i], np.uint8,
                                    pads=(shape[2] // 2,) * 2, **okw)
        tensors = [g.dev(w), g.dev(ws), g.dev(np.zeros(n, np.int8))] + ([g.dev(b)] if bias else [])
        descs = [capi.desc(t) for t in tensors]
        kept.extend(tensors + descs)
        operands.extend([ctypes.addressof(d) for d in descs] + ([] if bias else [None]))
        scales.append(y_scale)
        return y

    x, r = codes(rng, (N, mid, H, W), x_type), codes(rng, (N, wide, H, W), np.uint8)
    oracle.set_threads(16)
    try:
        h = convolution(x, 0.02, x_zp, (mid, mid, 3, 3), 0)
        h = convolution(h, scales[0], zero_points[0], (wide, mid, 1, 1), 1)
        r_scale, out_scale, r_zp = np.float32(0.71 * scales[1]), np.float32(1.57 * scales[1]), 21
        total = oracle.binary(oracle.ADD, oracle.dequantize_linear(h, scales[1], zero_points[1]), oracle.dequantize_linear(r, r_scale, r_zp))
        total = oracle.quantize_linear(oracle.relu(total) if relu else total, out_scale, out_zp, np.uint8)
        want = [total] + ([convolution(total, out_scale, out_zp, (nxt, wide, 1, 1), 2)] if nxt else [])
    finally:
        oracle.set_threads(1)
    block, stages = ctypes.c_void_p(), 3 if nxt else 2
    capi.check(lib.chx_hip_bottleneck_create((ctypes.c_void_p * (4 * stages))(*operands), stages, capi.stream_ptr(), ctypes.byref(block)))
    xd, rd = pitched(x.shape, torch.uint8 if x_type == np.uint8 else torch.int8), pitched(r.shape, torch.uint8)
    xd.copy_(g.dev(x))
    rd.copy_(g.dev(r))
    results = [pitched(v.shape, torch.int8 if minus_128 else torch.uint8) for v in want]
    store = capi.STORE_MINUS_128 if minus_128 else 0
    capi.check(lib.chx_hip_bottleneck_run(
        block, capi.ref(xd), ctypes.c_float(0.02), x_zp, (ctypes.c_float * 3)(*scales), (ctypes.c_int32 * 3)(*zero_points), capi.UINT8, capi.BIAS_ONNX_INT32 if bias else 0,
        capi.ref(rd), ctypes.c_float(r_scale), r_zp, ctypes.c_float(out_scale), out_zp, int(relu), store, capi.ref(results[0]), store, capi.ref(results[1]) if nxt else None, capi.stream_ptr()))
    for got, ref in zip(results, want):
        got = g.host(got)
        assert len(np.unique(ref)) > 20
        np.testing.assert_array_equal(got.view(np.uint8) ^ 0x80 if minus_128 else got, ref)
    lib.chx_hip_bottleneck_destroy(block)


@pytest.mark.parametrize("mid,H,W,relu,r_zp", [(64, 5, 13, True, -17), (128, 3, 31, False, 90), (256, 57, 28, True, -128)])
@pytest.mark.parametrize("affine", [True, False])
def test_sums(g, oracle, monkeypatch, affine, mid, H, W, relu, r_zp):
    """Both ways of the sum, its short form and operation by operation, with a residual of int8."""
    from test_gpu_conv_split import codes, pitched
    if not affine:
        monkeypatch.setenv("CHX_HIP_AFFINE_RESIDUAL", "0")
    rng, lib, capi, wide = np.random.default_rng(mid + W), g.capi.lib(), g.capi, 4 * mid
    x, r = codes(rng, (2, mid, H, W), np.uint8), codes(rng, (2, wide, H, W), np.int8)
    operands, kept, h, scales = [], [], x, [np.float32(0.02)]
    oracle.set_threads(16)
    try:
        for shape, zp, y_zp in (((mid, mid, 3, 3), 33, 0), ((wide, mid, 1, 1), 0, 117)):
            w, ws = codes(rng, shape, np.int8), rng.uniform(0.002, 0.02, size=shape[0]).astype(np.float32)
            scales.append(np.float32(scales[-1] * ws.mean() * 74 * 74 * np.sqrt(np.prod(shape[1:])) / 60))
            h = oracle.qlinear_conv_int(h, scales[-2], zp, w, ws, np.zeros(shape[0], np.int8), scales[-1], y_zp, np.uint8, pads=(shape[2] // 2,) * 2)
            tensors = [g.dev(w), g.dev(ws), g.dev(np.zeros(shape[0], np.int8))]
            kept += [tensors, [capi.desc(t) for t in tensors]]
            operands += [ctypes.addressof(d) for d in kept[-1]] + [None]
        r_scale, out_scale = np.float32(0.71 * scales[2]), np.float32(1.57 * scales[2])
        want = oracle.binary(oracle.ADD, oracle.dequantize_linear(h, scales[2], 117), oracle.dequantize_linear(r, r_scale, r_zp))
        want = oracle.quantize_linear(oracle.relu(want) if relu else want, out_scale, 40, np.uint8)
    finally:
        oracle.set_threads(1)
    block = ctypes.c_void_p()
    capi.check(lib.chx_hip_bottleneck_create((ctypes.c_void_p * 8)(*operands), 2, capi.stream_ptr(), ctypes.byref(block)))
    xd, rd, out = pitched(x.shape, torch.uint8), pitched(r.shape, torch.int8), pitched(want.shape, torch.uint8)
    xd.copy_(g.dev(x))
    rd.copy_(g.dev(r))
    capi.check(lib.chx_hip_bottleneck_run(
        block, capi.ref(xd), ctypes.c_float(0.02), 33, (ctypes.c_float * 2)(*scales[1:]), (ctypes.c_int32 * 2)(0, 117), capi.UINT8, 0, capi.ref(rd), ctypes.c_float(r_scale), r_zp,
        ctypes.c_float(out_scale), 40, int(relu), 0, capi.ref(out), 0, None, capi.stream_ptr()))
    assert len(np.unique(want)) > 20
    np.testing.assert_array_equal(g.host(out), want)
    lib.chx_hip_bottleneck_destroy(block)
