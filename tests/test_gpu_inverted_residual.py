"""Inverted residual blocks as one launch (csrc/inverted_residual.hip): whole networks, every block's output bit for bit
against the oracle's convolutions and sums; and single blocks with quantizations that no network here has."""
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


def check(g, vm, oracle, model, keep, blocks):
    """Through Program.run and a recording of it, in which the input changes."""
    wl = g.pkg.workloads
    prog = vm.Program(wl.program_to_chxvm(model, vm, g.pkg.ops, keep=keep).serialize())
    prog.set_option("qlinearconv_bias", "onnx_int32")
    x = torch.from_numpy(model["input"]).cuda()
    before = vm.counter("inverted_residuals")
    got = prog.run({"x": x})
    assert vm.counter("inverted_residuals") - before == blocks
    oracle.set_threads(16)
    try:
        for i in range(2):
            ref = wl.run_reference(model, oracle, model["input"][::-1] if i else model["input"], keep=set(keep))
            if i:
                replay = prog.capture({"x": x})
                x.copy_(torch.from_numpy(model["input"][::-1].copy()))
                torch.cuda.synchronize()
                for _ in range(3):
                    replay.launch()
                    replay.synchronize()
                    again = prog.run({"x": x})
                got = replay.outputs()
                for name in keep:
                    np.testing.assert_array_equal(again[name], ref[name], err_msg=name)
            for name in keep:
                np.testing.assert_array_equal(got[name], ref[name], err_msg="%d %s" % (i, name))
    finally:
        oracle.set_threads(1)
    replay.close()
    prog.close()


def block_outputs(model):
    """The last value of every block: a sum, or the result of a projection that no sum follows."""
    program = model["program"]
    summed = {ins[2] for ins in program if ins[0] == "Add"}  # (the other operand is an earlier block's value)
    names = [ins[1] for ins in program if ins[0] == "Add" or (ins[0] == "QLinearConv" and ins[3].endswith("_project") and ins[1] not in summed)]
    assert len(names) == sum(ins[0] == "QLinearConv" and ins[3].endswith("_project") for ins in program)
    return names


# image: what the first block sees is half of it; (expansion, channels, repeats, stride)
@pytest.mark.parametrize("batch,image,blocks,stem", [
    (2, 64, ((1, 16, 1, 1), (6, 24, 2, 2), (6, 32, 1, 2)), 32),                  # 16 -> 96 channels, a pixel of one chunk
    (3, 30, ((1, 8, 1, 1), (6, 40, 2, 1), (3, 48, 2, 2)), 24),                   # 15x15 and 8x8: odd rows, odd chunks
    (130, 14, ((6, 64, 1, 1), (6, 96, 1, 1), (6, 160, 2, 2), (6, 320, 1, 1)), 32),  # 7x7 and 4x4, two tiles of channels for a wavefront
    (1, 14, ((6, 64, 1, 1), (6, 96, 2, 1), (6, 256, 1, 2)), 32),                 # eight tiles of channels and few rows
    (5, 2, ((6, 32, 2, 1),), 32),                                                # one pixel
    (2, 6, ((2, 17, 2, 1), (5, 33, 1, 2)), 20),                                  # 3x3, channels that are no multiple of anything
    (2, 226, ((6, 24, 2, 1),), 16),                                              # 113 columns
])
def test_networks(g, vm, oracle, batch, image, blocks, stem):
    model = g.pkg.workloads.build_mobilenetv2(batch=batch, image=image, seed=batch + image, blocks=blocks, stem=stem, head=64, classes=10)
    count = sum(n for t, _, n, _ in blocks if t != 1)
    check(g, vm, oracle, model, ["logits"] + block_outputs(model), count)


@pytest.mark.parametrize("batch", [1, 40, 80])
def test_full_size(g, vm, oracle, batch):
    """All blocks of the network at the sizes it is used at, on few and on many images."""
    model = g.pkg.workloads.build_mobilenetv2(batch=batch, seed=11)
    wl = g.pkg.workloads
    prog = vm.Program(wl.program_to_chxvm(model, vm, g.pkg.ops, keep=["logits"] + block_outputs(model)).serialize())
    prog.set_option("qlinearconv_bias", "onnx_int32")
    got = prog.run({"x": torch.from_numpy(model["input"]).cuda()})
    picks = [0] if batch == 1 else [0, batch // 2, batch - 1]
    oracle.set_threads(16)
    try:
        ref = wl.run_reference(model, oracle, model["input"][picks], keep=set(got))
    finally:
        oracle.set_threads(1)
    for name in got:
        np.testing.assert_array_equal(got[name][picks], ref[name], err_msg=name)
    prog.close()


# N, channels (in, expanded, out), H, W, stride, x's type and zero point, the three results' zero points, scales per tensor, bias, sum
# (0 none, 1, 2 with Relu), result stored as code - 128.  Odd images, padding with another zero point than 0, one pixel, several
# tiles of channels out for a wavefront.
BLOCKS = [
    (2, (16, 96, 24), 9, 7, 1, np.uint8, 77, (13, 200, 128), False, True, 0, False),
    (2, (16, 96, 24), 9, 7, 2, np.int8, -9, (13, 0, 5), True, False, 0, True),
    (3, (40, 130, 33), 8, 11, 2, np.uint8, 0, (0, 255, 0), True, True, 0, False),
    (1, (24, 72, 40), 5, 5, 1, np.int8, 100, (255, 9, 117), False, False, 1, False),
    (2, (17, 33, 17), 6, 13, 1, np.uint8, 255, (128, 128, 3), True, False, 2, True),
    (3, (64, 64, 64), 1, 1, 2, np.uint8, 4, (60, 61, 62), True, True, 1, False),
    (75, (160, 96, 320), 7, 7, 1, np.uint8, 131, (31, 7, 90), True, True, 2, False),
    (2, (96, 384, 256), 5, 9, 1, np.int8, 0, (0, 0, 128), False, True, 1, True),
]


@pytest.mark.parametrize("case", range(len(BLOCKS)))
def test_single_blocks(g, oracle, case):
    N, (cin, hid, cout), H, W, stride, x_type, x_zp, zero_points, per_tensor, bias, with_sum, minus_128 = BLOCKS[case]
    from test_gpu_conv_split import codes, pitched
    rng = np.random.default_rng(case)
    lib, capi = g.capi.lib(), g.capi
    x = codes(rng, (N, cin, H, W), x_type)
    h, scale, zp = x, 0.02, x_zp
    operands, kept, scales = [], [], []
    for i, (shape, group, step, pad) in enumerate((((hid, cin, 1, 1), 1, 1, 0), ((hid, 1, 3, 3), hid, stride, 1), ((cout, hid, 1, 1), 1, 1, 0))):
        w, n = codes(rng, shape, np.int8), 1 if per_tensor else shape[0]
        ws, b = rng.uniform(0.002, 0.02, size=n).astype(np.float32), rng.integers(-3000, 3000, size=shape[0]).astype(np.int32) if bias else None
        y_scale = np.float32(scale * ws.mean() * 74 * 74 * np.sqrt(np.prod(shape[1:])) / 60)
        okw = dict(bias=b, bias_mode=oracle.BIAS_ONNX_INT32) if bias else {}
        h = oracle.qlinear_conv_int(h, scale, zp, w, np.broadcast_to(ws, shape[:1]).copy(), np.zeros(shape[0], np.int8), y_scale, zero_points[i], np.uint8,
                                    strides=(step, step), pads=(pad, pad), group=group, **okw)
        assert len(np.unique(h)) > 20
        kept += [g.dev(w), g.dev(ws), g.dev(np.zeros(n, np.int8))] + ([g.dev(b)] if bias else [])
        descs = [capi.desc(t) for t in kept[-(4 if bias else 3):]]
        kept += descs
        operands += [ctypes.addressof(d) for d in descs] + ([] if bias else [None])
        scales.append(y_scale)
        scale, zp = y_scale, zero_points[i]
    block = ctypes.c_void_p()
    capi.check(lib.chx_hip_inverted_residual_create((ctypes.c_void_p * 12)(*operands), stride, capi.stream_ptr(), ctypes.byref(block)))
    xd = pitched(x.shape, torch.uint8 if x_type == np.uint8 else torch.int8)
    xd.copy_(g.dev(x))
    y, rd = pitched(h.shape, torch.int8 if minus_128 else torch.uint8), None
    r_scale, out_scale, out_zp, r_zp = np.float32(0.7 * scale), np.float32(1.6 * scale), 40, 21
    if with_sum:
        r = codes(rng, h.shape, np.uint8)
        rd = pitched(h.shape, torch.uint8)
        rd.copy_(g.dev(r))
        total = oracle.binary(oracle.ADD, oracle.dequantize_linear(h, scale, zp), oracle.dequantize_linear(r, r_scale, r_zp))
        h = oracle.quantize_linear(oracle.relu(total) if with_sum == 2 else total, out_scale, out_zp, np.uint8)
    flags = (capi.BIAS_ONNX_INT32 if bias else 0) | (capi.STORE_MINUS_128 if minus_128 else 0)
    capi.check(lib.chx_hip_inverted_residual_run(
        block, capi.ref(xd), ctypes.c_float(0.02), x_zp, (ctypes.c_float * 3)(*scales), (ctypes.c_int32 * 3)(*zero_points), capi.UINT8, flags,
        capi.ref(rd) if with_sum else None, ctypes.c_float(r_scale), r_zp, ctypes.c_float(out_scale), out_zp, int(with_sum == 2), capi.ref(y), capi.stream_ptr()))
    got = g.host(y)
    np.testing.assert_array_equal(got.view(np.uint8) ^ 0x80 if minus_128 else got, h)
    lib.chx_hip_inverted_residual_destroy(block)
