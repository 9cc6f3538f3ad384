"""Which programs quantize inside their first convolution and leave floats from their last (runtime/chxvm.cc), without a GPU."""
import ctypes
import re

import pytest

import host_hip


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["one_launch_each", "frees_between", "refused_forms", "larger_results", "far_apart", "another_device", "instruction_by_instruction"])
def test_case(host_so, case):
    host_hip.run_case(host_so, __file__, case)


# x float32 -> QuantizeLinear -> convolution -> convolution with 1x1 filters -> DequantizeLinear
def program(host, channels=(3, 32, 10), image=8, kernel=3, last_kernel=1, code_type="uint8", free=False, keep=(), batch=2, group=1):
    import numpy as np
    b = host.chxvm.ProgramBuilder()
    cin, mid, out = channels
    x = b.input("x", "float32", [batch, cin, image, image])
    zero = 0 if code_type == "int8" else 7
    s, z = b.scalar(0.1, "float32"), b.scalar(zero, code_type)
    values = [b.QuantizeLinear(x, s, z)]
    if free:
        b.Free(x)
    scale = (s, z)
    for shape, g in (((mid, cin // group, kernel, kernel), group), ((out, mid, last_kernel, last_kernel), 1)):
        w, ws, wz = b.constant(np.ones(shape, np.int8)), b.constant(np.full(shape[0], 0.01, np.float32)), b.constant(np.zeros(shape[0], np.int8))
        ys = b.scalar(0.2, "float32"), b.scalar(0, "uint8")
        values.append(b.QLinearConv(values[-1], *scale, w, ws, wz, *ys, b.constant(np.zeros(shape[0], np.int32)), [1, 1], [shape[2] // 2] * 2, g, ""))
        if free:
            for slot in (w, ws, wz, values[-2]):
                b.Free(slot)
        scale = ys
    y = b.DequantizeLinear(values[-1], *scale)
    for i in keep:
        b.output("kept%d" % i, values[i])
    b.output("y", y)
    return host.program(b)


def kernels(host, p, channels=(3, 32, 10), image=8, batch=2):
    rt = host.chxvm.runtime()
    assert rt.chxvm_set_option(b"qlinearconv_bias", b"onnx_int32") == 0
    x = host.tensor("float32", (batch, channels[0], image, image))
    host.clear()
    out = ctypes.c_void_p()
    assert rt.chxvm_program_run(p, *host.names_and({"x": x}), 0, ctypes.byref(out)) == 0, rt.chxvm_last_error()
    names = [re.match(r"(?:void )?(?:\w+::|\(anonymous namespace\)::)*(\w+)", line).group(1) for line in host.launches()]
    rt.chxvm_outputs_destroy(out)
    return names


def ends(host, p, **kw):
    """(quantized inside the convolution, floats from the convolution)"""
    kernels(host, p, **kw)  # (measures)
    names = kernels(host, p, **kw)
    return not any(n.startswith("quantize") for n in names), not any(n.startswith("dequantize") for n in names)


def one_launch_each(host):
    for kw in ({}, dict(channels=(1, 64, 1000)), dict(channels=(4, 16, 17), batch=1, image=5)):
        p = program(host, **kw)
        at = {k: v for k, v in kw.items() if k in ("channels", "image", "batch")}
        assert ends(host, p, **at) == (True, True), kw
        assert len(kernels(host, p, **at)) == 2, kw


def frees_between(host):
    p = program(host, free=True)
    assert ends(host, p) == (True, True) and ends(host, p) == (True, True)


def refused_forms(host):
    for kw, expected in ((dict(code_type="int8"), (False, True)), (dict(channels=(40, 32, 10)), (False, True)), (dict(last_kernel=3), (True, False)), (dict(image=3), (False, True)),
                         (dict(keep=(0,)), (False, True)), (dict(keep=(2,)), (True, False)), (dict(channels=(4, 32, 10), group=2), (False, True))):
        at = {k: v for k, v in kw.items() if k in ("channels", "image", "batch")}
        assert ends(host, program(host, **kw), **at) == expected, kw


def larger_results(host):
    for batch, one in ((8, True), (9, False)):  # (2^19 results and more)
        at = dict(channels=(3, 32, 64), image=32, batch=batch)
        assert ends(host, program(host, **at), **at) == (True, one), batch


def far_apart(host):
    """Rows and channels of floats whose distances do not fit the kernel's 32 bits, one short of it and at it."""
    w, ws, zp = host.tensor("int8", (32, 3, 3, 3)), host.tensor("float32", (32,)), host.tensor("int8", (32,))
    params, plan = host.capi.conv_params((1, 1), (1, 1), (1, 1), 1), ctypes.c_void_p()
    host.check(host.lib.chx_hip_qconv_plan_create(ctypes.byref(w), ctypes.byref(ws), ctypes.byref(zp), None, ctypes.byref(params), None, ctypes.byref(plan)))
    y = host.channels_last("uint8", (1, 32, 8, 8))
    for row, channel, taken in ((32, 256, True), ((1 << 27) - 4, 256, True), (1 << 27, 256, False), (32, (1 << 30) // 3 // 4 * 4, True), (32, (1 << 30) // 3 // 4 * 4 + 4, False),
                                (32, -((1 << 30) // 3 // 4 * 4 + 4), False), (1 << 28, 1 << 28, False)):
        x = host.tensor("float32", (1, 3, 8, 8))
        x.strides[1], x.strides[2] = channel, row
        host.clear()
        rc = host.lib.chx_hip_qconv_plan_run_quantize(plan, ctypes.byref(x), ctypes.c_float(0.1), 7, ctypes.c_float(0.1), 7, ctypes.c_float(0.2), 0, 0, ctypes.byref(y), None)
        assert (rc == 0, len(host.launches())) == ((True, 1) if taken else (False, 0)), (row, channel, rc)
        assert taken or rc == host.capi.EUNSUPPORTED


def another_device(host):
    """The plans are made on one device: on another one the instructions run."""
    p = program(host)
    host.check(host.lib.chx_hip_init(1))
    assert ends(host, p) == (False, False)
    host.check(host.lib.chx_hip_init(0))
    assert ends(host, p) == (True, True)


def instruction_by_instruction(host):
    rt, p = host.chxvm.runtime(), program(host)
    assert rt.chxvm_set_option(b"check_types", b"on") == 0
    assert ends(host, p) == (False, False)
    assert rt.chxvm_set_option(b"check_types", b"off") == 0
    assert ends(host, p) == (True, True)


if __name__ == "__main__":
    host_hip.main(globals())
