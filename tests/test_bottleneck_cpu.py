"""Which programs run the tail of a bottleneck block and the next block's reduction as one launch (runtime/chxvm.cc,
csrc/bottleneck.hip) and which instructions of theirs still run, without a GPU."""
import ctypes
import os
import re
import sys

import pytest

import host_hip

BLOCK, SEARCH = "bottleneck_kernel", "affine_residual_search_kernel"  # (the sum's short form is searched for once)


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.fixture(scope="module")
def sum_code():
    sys.path.insert(0, host_hip.ROOT)
    import __graft_entry__ as entry
    pkg = entry.load_package()
    return pkg.workloads.add_program(pkg.ops, (0.25, 128), (0.1, 7), (0.4, 120))


@pytest.mark.parametrize("case", ["whole_blocks", "without_reduction", "values_read_elsewhere", "frees_between", "refused_forms", "sizes", "nothing_launched", "errors", "another_device",
                                  "instruction_by_instruction", "long_rows", "channels_that_never_run", "asked_first", "sums"])
def test_case(host_so, sum_code, case):
    host_hip.run_case(host_so, __file__, case, SUM_CODE=sum_code)


def program(host, channels=(64, 256, 64), kernel=3, pads=(1, 0, 0), strides=(1, 1, 1), group=1, bias=True, y_type="uint8", chain_scale=0.4, free=False, keep=None, between=False, image=8,
            batch=2):
    """x, r uint8 -> 3x3 -> 1x1 -> sum with r -> 1x1"""
    import numpy as np
    b = host.chxvm.ProgramBuilder()
    mid, wide, nxt = channels
    x, r = b.input("x", "uint8", [batch, mid, image, image]), b.input("r", "uint8", [batch, wide, image, image])
    shapes = [(mid, mid // group, kernel, kernel), (wide, mid, 1, 1)] + ([(nxt, wide, 1, 1)] if nxt else [])
    h, scale, values = x, (0.1, 7), []
    for i, shape in enumerate(shapes):
        out = ((0.2, 0), (0.25, 128), (0.3, 0))[i]
        xs, xz = b.scalar(scale[0] if i != 2 else chain_scale, "float32"), b.scalar(scale[1], "uint8")
        w, ws, wz = b.constant(np.ones(shape, np.int8)), b.constant(np.full(shape[0], 0.01, np.float32)), b.constant(np.zeros(shape[0], np.int8))
        ys, yz = b.scalar(out[0], "float32"), b.scalar(out[1] if y_type == "uint8" else 0, y_type)
        bias_q = b.constant(np.zeros(shape[0], np.int32)) if bias else -1
        y = b.QLinearConv(h, xs, xz, w, ws, wz, ys, yz, bias_q, [strides[i]] * 2, [pads[i]] * 2, group if i == 0 else 1, "")
        if free:
            for s in (w, ws, wz, bias_q) + ((h,) if i else ()):
                b.Free(s)
        values.append(y)
        h, scale = y, out
        if i == 1:
            h, scale = b.ElementWiseNvrtc([y, r], 1, os.environ["SUM_CODE"], 0, num_list_outputs=1)[0], (0.4, 120)
            values.append(h)
            if free:
                b.Free(y)
            if between:
                b.output("copy", b.DequantizeLinear(h, b.scalar(0.4, "float32"), b.scalar(120, "uint8")))
    if keep is not None:
        b.output("kept", values[keep])
    b.output("y", h)
    return host.program(b)


def kernels(host, p, channels=(64, 256, 64), n=2, image=8, x=None):
    rt = host.chxvm.runtime()
    assert rt.chxvm_set_option(b"qlinearconv_bias", b"onnx_int32") == 0
    x = x or host.channels_last("uint8", (n, channels[0], image, image))
    host.clear()
    out = ctypes.c_void_p()
    assert rt.chxvm_program_run(p, *host.names_and({"x": x, "r": host.channels_last("uint8", (n, channels[1], image, image))}), 0, ctypes.byref(out)) == 0, rt.chxvm_last_error()
    names = [re.match(r"(?:void )?(?:\w+::|\(anonymous namespace\)::)*(\w+)", line).group(1) for line in host.launches()]
    rt.chxvm_outputs_destroy(out)
    return names


def whole_blocks(host):
    for channels in ((64, 256, 64), (128, 512, 128), (64, 256, 96), (128, 256, 32)):
        for bias in (True, False):
            p = program(host, channels, bias=bias)
            assert kernels(host, p, channels) == [SEARCH, BLOCK]
            assert kernels(host, p, channels) == [BLOCK]
    # one program, images of other sizes
    p = program(host)
    assert kernels(host, p, n=1, image=1) == [SEARCH, BLOCK] and kernels(host, p, n=3, image=31) == [BLOCK]


def without_reduction(host):
    assert kernels(host, program(host, (64, 256, 0)), (64, 256, 0)) == [SEARCH, BLOCK]
    # a third convolution that is not one, or that the kernel does not take, runs by itself
    for kw in (dict(strides=(1, 1, 2)), dict(pads=(1, 0, 1)), dict(channels=(64, 256, 40)), dict(between=True)):
        names = kernels(host, program(host, **kw), kw.get("channels", (64, 256, 64)))
        assert names[:2] == [SEARCH, BLOCK] and len(names) > 2, (kw, names)


def values_read_elsewhere(host):
    for keep in (0, 1):
        assert BLOCK not in kernels(host, program(host, keep=keep))
    assert kernels(host, program(host, keep=2)) == [SEARCH, BLOCK]  # the sum is written anyway


def frees_between(host):
    p = program(host, free=True)
    for i in range(2):
        assert kernels(host, p)[-1] == BLOCK
        # also where the instructions run one by one: pixels that are no whole chunks
        assert BLOCK not in kernels(host, p, x=host.channels_last("uint8", (2, 64, 8, 8), 65))


def refused_forms(host):
    for kw in (dict(pads=(0, 0, 0)), dict(pads=(2, 0, 0), kernel=5), dict(strides=(2, 1, 1)), dict(strides=(1, 2, 1)), dict(pads=(1, 1, 0)), dict(y_type="int8"), dict(group=2)):
        p = program(host, **kw)
        rt, out = host.chxvm.runtime(), ctypes.c_void_p()
        host.clear()
        assert rt.chxvm_set_option(b"qlinearconv_bias", b"onnx_int32") == 0
        rt.chxvm_program_run(p, *host.names_and({"x": host.channels_last("uint8", (2, 64, 8, 8)), "r": host.channels_last("uint8", (2, 256, 8, 8))}), 0, ctypes.byref(out))
        assert not any(BLOCK in line for line in host.launches()), kw
    for channels in ((32, 256, 64), (96, 256, 64), (64, 192, 64), (64, 768, 64), (512, 2048, 512)):
        assert BLOCK not in kernels(host, program(host, channels), channels), channels
    assert BLOCK not in kernels(host, program(host, chain_scale=0.41))  # another scale than the one it was written with
    assert BLOCK not in kernels(host, program(host), x=host.tensor("uint8", (2, 64, 8, 8)))  # an NCHW image
    assert BLOCK not in kernels(host, program(host, image=2000), n=1, image=2000) # a run of pixels that does not fit LDS


def sizes(host):
    """Blocks that are faster as single launches."""
    for channels, n, image, one in SIZES:
        p = program(host, channels, image=image, batch=n)
        assert (BLOCK in kernels(host, p, channels, n, image)) == one, (channels, n, image)


SIZES = [((64, 256, 64), 1, 56, True), ((64, 256, 64), 64, 56, True), ((128, 512, 128), 1, 28, True), ((128, 512, 128), 64, 28, True), ((256, 1024, 256), 64, 14, True),
         ((256, 1024, 256), 1, 14, False), ((256, 1024, 256), 8, 14, True), ((256, 1024, 512), 8, 14, False), ((64, 1024, 64), 8, 7, False)]


def nothing_launched(host):
    """What is refused has launched nothing: not the search for a sum's short form either."""
    lib, capi, ref = host.lib, host.capi, ctypes.byref
    keep, operands = [], []
    for shape in ((256, 256, 3, 3), (1024, 256, 1, 1)):
        tensors = host.tensor("int8", shape), host.tensor("float32", shape[:1]), host.tensor("int8", shape[:1])
        keep.append(tensors)
        operands += [ctypes.addressof(t) for t in tensors] + [None]
    block = ctypes.c_void_p()
    host.check(lib.chx_hip_bottleneck_create((ctypes.c_void_p * 8)(*operands), 2, None, ref(block)))
    scales, zeros = (ctypes.c_float * 2)(0.2, 0.25), (ctypes.c_int32 * 2)(0, 0)

    def run(n, r_channels=1024):
        x, r, y = host.channels_last("uint8", (n, 256, 14, 14)), host.channels_last("uint8", (n, r_channels, 14, 14)), host.channels_last("uint8", (n, 1024, 14, 14))
        host.clear()
        rc = lib.chx_hip_bottleneck_run(block, ref(x), ctypes.c_float(0.1), 7, scales, zeros, capi.UINT8, 0, ref(r), ctypes.c_float(0.15), 3, ctypes.c_float(0.4), 120, 0, 0, ref(y), 0, None,
                                        None)
        return rc, len(host.launches())

    assert run(1) == (2, 0)  # CHX_HIP_EUNSUPPORTED: few pixels for so many weights
    assert run(64, 512) == (2, 0)
    assert run(64) == (0, 2)  # the search and the block
    assert run(64) == (0, 1)


def long_rows(host):
    """Rows that do not fit LDS are refused, however long: 31 and 32 bits of bytes are reached at some 13 and 27 million pixels."""
    lib, capi, ref = host.lib, host.capi, ctypes.byref
    keep, operands = [], []
    for shape in ((64, 64, 3, 3), (256, 64, 1, 1)):
        tensors = host.tensor("int8", shape), host.tensor("float32", shape[:1]), host.tensor("int8", shape[:1])
        keep.append(tensors)
        operands += [ctypes.addressof(t) for t in tensors] + [None]
    block, small = ctypes.c_void_p(), host.channels_last("uint8", (1, 256, 1, 1))
    host.check(lib.chx_hip_bottleneck_create((ctypes.c_void_p * 8)(*operands), 2, None, ref(block)))

    def run(w):  # (nothing is read or written)
        x, r, y = (capi.make_desc(small.data + (i << 40), capi.UINT8, (1, c, 1, w), (w * c, 1, w * c, c)) for i, c in enumerate((64, 256, 256)))
        host.clear()
        rc = lib.chx_hip_bottleneck_run(block, ref(x), ctypes.c_float(0.1), 7, (ctypes.c_float * 2)(0.2, 0.25), (ctypes.c_int32 * 2)(0, 0), capi.UINT8, 0, ref(r), ctypes.c_float(0.15), 3,
                                        ctypes.c_float(0.4), 120, 0, 0, ref(y), 0, None, None)
        return rc, sum(BLOCK in line for line in host.launches())

    assert run(800) == (0, 1)
    for w in (1000, 8191, 8192, 13_000_000, 13_500_000, 14_000_000, 20_000_000, 26_843_400, 26_843_540, 40_265_000, 100_000_000, (1 << 30) - 1):
        assert run(w) == (capi.EUNSUPPORTED, 0), w


def channels_that_never_run(host):
    """Channels that the kernel takes for no number of pixels are refused when the block is created, before anything is laid out."""
    lib, ref = host.lib, ctypes.byref
    for mid, wide, nxt, taken in ((64, 256, 64, True), (64, 512, 64, False), (128, 512, 1024, True), (128, 1024, 0, False), (256, 1024, 256, True), (256, 2048, 256, False), (256, 512, 1056, False)):
        keep, operands = [], []
        for shape in ((mid, mid, 3, 3), (wide, mid, 1, 1)) + (((nxt, wide, 1, 1),) if nxt else ()):
            tensors = host.tensor("int8", shape), host.tensor("float32", shape[:1]), host.tensor("int8", shape[:1])
            keep.append(tensors)
            operands += [ctypes.addressof(t) for t in tensors] + [None]
        block = ctypes.c_void_p()
        host.clear()
        rc = lib.chx_hip_bottleneck_create((ctypes.c_void_p * len(operands))(*operands), len(keep), None, ref(block))
        assert (rc == 0) == taken and (taken or (rc == host.capi.EUNSUPPORTED and not host.log())), (mid, wide, nxt, host.log())


def asked_first(host):
    """chx_hip_bottleneck_takes says what chx_hip_bottleneck_run does."""
    lib, capi, ref = host.lib, host.capi, ctypes.byref
    for mid, wide, nxt in ((64, 256, 64), (128, 512, 0), (256, 1024, 256), (256, 512, 0)):
        keep, operands = [], []
        for shape in ((mid, mid, 3, 3), (wide, mid, 1, 1)) + (((nxt, wide, 1, 1),) if nxt else ()):
            tensors = host.tensor("int8", shape), host.tensor("float32", shape[:1]), host.tensor("int8", shape[:1])
            keep.append(tensors)
            operands += [ctypes.addressof(t) for t in tensors] + [None]
        block = ctypes.c_void_p()
        host.check(lib.chx_hip_bottleneck_create((ctypes.c_void_p * len(operands))(*operands), len(keep), None, ref(block)))
        takes = lambda *s: lib.chx_hip_bottleneck_takes(block, *[ctypes.c_int64(v) for v in s])
        seen = set()
        for n, h, w in ((1, 1, 1), (1, 14, 14), (8, 14, 14), (13, 14, 14), (400, 14, 14), (1, 3, 300), (1, 3, 1200), (70000, 14, 14), (1, 1, 14_000_000)):
            x, r, y, z = (capi.make_desc((i + 1) << 44, capi.UINT8, (n, c, h, w), (h * w * c, 1, w * c, c)) for i, c in enumerate((mid, wide, wide, nxt or 1)))
            rc = lib.chx_hip_bottleneck_run(block, ref(x), ctypes.c_float(0.1), 7, (ctypes.c_float * 3)(0.2, 0.25, 0.3), (ctypes.c_int32 * 3)(0, 0, 0), capi.UINT8, 0, ref(r),
                                            ctypes.c_float(0.15), 3, ctypes.c_float(0.4), 120, 0, 0, ref(y), 0, ref(z) if nxt else None, None)
            assert takes(n, h, w) == rc, (mid, wide, nxt, n, h, w)
            seen.add(rc)
        assert seen == {0, capi.EUNSUPPORTED}
        for s in ((0, 1, 1), (1, -1, -1), (1 << 40, 1 << 40, 1 << 40), (1 << 62, 4, 1)):
            assert takes(*s) == capi.EUNSUPPORTED


def sums(host):
    """The kernel's form for the sum's short form, and the one for all others."""
    def forms(p):
        kernels(host, p)
        return re.findall(r"bottleneck_kernel<.*(true|false)>", "\n".join(host.launches())), any(SEARCH in line for line in host.launches())

    p = program(host)
    os.environ["CHX_HIP_AFFINE_RESIDUAL"] = "0"
    without = program(host)
    assert forms(without) == (["false"], False)
    assert forms(p)[1]  # (the stand-in's search finds what it finds)


def errors(host):
    """An error names the convolution that it is of: the first."""
    x = host.channels_last("uint8", (2, 128, 8, 8))  # (twice the channels)
    said = host.run_fails(program(host), {"x": x, "r": host.channels_last("uint8", (2, 256, 8, 8))})
    assert "Exception in QLinearConv" in said, said


def another_device(host):
    """The operands are laid out in one device's memory: on another one the convolutions run."""
    p = program(host)
    host.check(host.lib.chx_hip_init(1))
    assert BLOCK not in kernels(host, p)
    host.check(host.lib.chx_hip_init(0))
    assert BLOCK in kernels(host, p)


def instruction_by_instruction(host):
    """A run that looks at the values between the instructions sees all of them."""
    rt = host.chxvm.runtime()
    p = program(host)
    assert rt.chxvm_set_option(b"check_types", b"on") == 0
    assert BLOCK not in kernels(host, p)
    assert rt.chxvm_set_option(b"check_types", b"off") == 0
    assert kernels(host, p)[-1] == BLOCK


if __name__ == "__main__":
    host_hip.main(globals())
