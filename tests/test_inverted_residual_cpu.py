"""Which programs run an inverted residual block as one launch (runtime/chxvm.cc, csrc/inverted_residual.hip) and which
instructions of theirs still run, without a GPU."""
import ctypes
import os
import re
import sys

import pytest

import host_hip

BLOCK, SEARCH = "inverted_residual_kernel", "affine_residual_search_kernel"  # (the sum's short form is searched for once)


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.fixture(scope="module")
def sum_code():
    sys.path.insert(0, host_hip.ROOT)
    import __graft_entry__ as entry
    pkg = entry.load_package()
    return pkg.workloads.add_program(pkg.ops, (0.3, 128), (0.1, 7), (0.4, 120))


@pytest.mark.parametrize("case", ["whole_blocks", "sums", "values_read_twice", "frees_between", "refused_forms", "few_rows", "slower_blocks", "nothing_launched", "errors", "another_device", "instruction_by_instruction"])
def test_case(host_so, sum_code, case):
    host_hip.run_case(host_so, __file__, case, SUM_CODE=sum_code)


def program(host, channels=(16, 96, 24), stride=1, pads=(0, 1, 0), groups=None, strides=None, dilated_filter=3, bias=True, y_type="uint8", chain_scale=0.2,
            sums=0, free=False, keep=None, image=8, batch=2):
    """x uint8 -> expansion -> depthwise -> projection (-> sum with x, or with x twice over)"""
    import numpy as np
    b = host.chxvm.ProgramBuilder()
    cin, hid, cout = channels
    x = b.input("x", "uint8", [batch, cin, image, image])
    shapes = [(hid, cin, 1, 1), (hid, 1, dilated_filter, dilated_filter), (cout, hid, 1, 1)]
    group = groups or (1, hid, 1)
    step = strides or (1, stride, 1)
    h = x
    scale, between = (0.1, 7), []
    for i, shape in enumerate(shapes):
        out = ((0.2, 0), (0.25, 0), (0.3, 128))[i]
        xs, xz = b.scalar(scale[0] if i != 1 else chain_scale, "float32"), b.scalar(scale[1], "uint8")
        w, ws, wz = b.constant(np.ones(shape, np.int8)), b.constant(np.full(shape[0], 0.01, np.float32)), b.constant(np.zeros(shape[0], np.int8))
        ys, yz = b.scalar(out[0], "float32"), b.scalar(out[1] if y_type == "uint8" else 0, y_type)
        bias_q = b.constant(np.zeros(shape[0], np.int32)) if bias else -1
        y = b.QLinearConv(h, xs, xz, w, ws, wz, ys, yz, bias_q, [step[i]] * 2, [pads[i]] * 2, group[i], "")
        if free:
            for s in (w, ws, wz, bias_q) + ((h,) if i else ()):
                b.Free(s)
        if keep == i:
            b.output("between", y)
        h, scale = y, out
    for k in range(sums):
        h = b.ElementWiseNvrtc([h, x], 1, os.environ["SUM_CODE"], k, num_list_outputs=1)[0]
    b.output("y", h)
    return host.program(b)


def kernels(host, p, shape, dtype="uint8", x=None):
    rt = host.chxvm.runtime()
    assert rt.chxvm_set_option(b"qlinearconv_bias", b"onnx_int32") == 0
    pitch = (shape[1] + 15) // 16 * 16
    x = x or host.channels_last(dtype, shape, pitch)
    host.clear()
    out = ctypes.c_void_p()
    assert rt.chxvm_program_run(p, *host.names_and({"x": x}), 0, ctypes.byref(out)) == 0, rt.chxvm_last_error()
    names = [re.match(r"(?:void )?(?:\w+::|\(anonymous namespace\)::)*(\w+)", line).group(1) for line in host.launches()]
    rt.chxvm_outputs_destroy(out)
    return names


def one(host, p, shape=(2, 16, 8, 8), **kw):
    return kernels(host, p, shape, **kw).count(BLOCK)


def whole_blocks(host):
    for stride in (1, 2):
        for bias in (True, False):
            p = program(host, stride=stride, bias=bias)
            for _ in range(2):
                assert kernels(host, p, (2, 16, 8, 8)) == [BLOCK]
    assert kernels(host, program(host, (160, 960, 320), batch=128, image=7), (128, 160, 7, 7)) == [BLOCK]
    assert kernels(host, program(host, (17, 33, 5)), (2, 17, 8, 8)) == [BLOCK]
    # one program, images of other sizes
    p = program(host)
    assert kernels(host, p, (1, 16, 1, 2)) == [BLOCK] and kernels(host, p, (3, 16, 30, 31)) == [BLOCK]


def sums(host):
    same = (16, 96, 16)
    for free in (False, True):
        p = program(host, same, sums=1, free=free)
        assert kernels(host, p, (2, 16, 8, 8)) == [SEARCH, BLOCK]
        assert kernels(host, p, (2, 16, 8, 8)) == [BLOCK]
    # the second sum is a launch of its own, and the block's result has another reader than the sum
    names = kernels(host, program(host, same, sums=2), (2, 16, 8, 8))
    assert names[:2] == [SEARCH, BLOCK] and len(names) == 3
    names = kernels(host, program(host, same, sums=1, keep=2), (2, 16, 8, 8))
    assert names[0] == BLOCK and len(names) == 2


def values_read_twice(host):
    for keep in (0, 1):
        assert one(host, program(host, keep=keep)) == 0
    assert one(host, program(host, keep=2)) == 1


def frees_between(host):
    p = program(host, free=True)
    for _ in range(2):
        assert kernels(host, p, (2, 16, 8, 8)) == [BLOCK]
        # also where the instructions run one by one: pixels that are no whole chunks
        assert one(host, p, x=host.channels_last("uint8", (2, 16, 8, 8), 17)) == 0


def refused_forms(host):
    assert one(host, program(host, pads=(1, 1, 0))) == 0
    assert one(host, program(host, pads=(0, 0, 0))) == 0
    assert one(host, program(host, pads=(0, 1, 1))) == 0
    assert one(host, program(host, strides=(2, 1, 1))) == 0
    assert one(host, program(host, strides=(1, 1, 2))) == 0
    assert one(host, program(host, strides=(1, 3, 1))) == 0
    assert one(host, program(host, dilated_filter=5, pads=(0, 2, 0))) == 0
    assert one(host, program(host, y_type="int8")) == 0
    assert one(host, program(host, chain_scale=0.21)) == 0  # another scale than the one it was written with
    assert one(host, program(host, (161, 96, 24)), (2, 161, 8, 8)) == 0
    assert one(host, program(host, (16, 96, 321)), (40, 16, 16, 16)) == 0
    assert one(host, program(host), x=host.tensor("uint8", (2, 16, 8, 8))) == 0  # an NCHW image
    assert one(host, program(host, image=4000), (1, 16, 2, 4000)) == 0  # a row that does not fit LDS


def few_rows(host):
    """More than 256 channels out and fewer than 512 rows."""
    for channels, n, blocks in (((160, 960, 320), 64, 0), ((160, 960, 320), 74, 1), ((160, 960, 256), 1, 1), ((160, 960, 257), 1, 0)):
        assert one(host, program(host, channels, image=7), (n, channels[0], 7, 7)) == blocks


def slower_blocks(host):
    """Blocks whose strips are a row or two of a wide image, or whose halo costs more than it saves, run as three launches."""
    for n, channels, image, stride, blocks in ((70, (24, 144, 104), 104, 1, 0), (54, (8, 48, 80), 86, 1, 0), (60, (128, 768, 208), 51, 1, 0), (126, (16, 48, 8), 99, 1, 0),
                                               (1, (152, 912, 208), 64, 2, 0), (10, (160, 960, 160), 56, 1, 0), (128, (16, 96, 24), 112, 2, 1), (128, (24, 144, 24), 56, 1, 1),
                                               (32, (24, 144, 32), 56, 2, 1), (128, (96, 576, 160), 14, 2, 1), (1, (160, 960, 160), 7, 1, 1)):
        assert one(host, program(host, channels, stride=stride, image=image, batch=n), (n, channels[0], image, image)) == blocks, (n, channels, image)


def nothing_launched(host):
    """What is refused has launched nothing: not the search for a sum's short form either."""
    lib, capi, ref = host.lib, host.capi, ctypes.byref
    keep, operands = [], []
    for shape in ((96, 16, 1, 1), (96, 1, 3, 3), (257, 96, 1, 1)):
        tensors = host.tensor("int8", shape), host.tensor("float32", shape[:1]), host.tensor("int8", shape[:1])
        keep.append(tensors)
        operands += [ctypes.addressof(t) for t in tensors] + [None]
    block = ctypes.c_void_p()
    host.check(lib.chx_hip_inverted_residual_create((ctypes.c_void_p * 12)(*operands), 1, None, ref(block)))
    scales, zeros = (ctypes.c_float * 3)(0.2, 0.25, 0.3), (ctypes.c_int32 * 3)(0, 0, 128)

    def run(n):
        x, r, y = host.channels_last("uint8", (n, 16, 8, 8)), host.channels_last("uint8", (n, 257, 8, 8), 272), host.channels_last("uint8", (n, 257, 8, 8), 272)
        host.clear()
        rc = lib.chx_hip_inverted_residual_run(block, ref(x), ctypes.c_float(0.1), 7, scales, zeros, capi.UINT8, 0, ref(r), ctypes.c_float(0.15), 3,
                                               ctypes.c_float(0.4), 120, 0, ref(y), None)
        return rc, len(host.launches())

    assert run(2) == (2, 0)  # CHX_HIP_EUNSUPPORTED: 16 rows for more than 256 channels
    assert run(64) == (0, 2)  # the search and the block
    assert run(64) == (0, 1)


def errors(host):
    """An error names the convolution that it is of: the expansion."""
    x = host.channels_last("uint8", (2, 32, 8, 8))  # (twice the channels)
    said = host.run_fails(program(host), {"x": x})
    assert "Exception in QLinearConv (pc 9)" in said, said


def another_device(host):
    """The operands are laid out in one device's memory: on another one the convolutions run."""
    p = program(host)
    host.check(host.lib.chx_hip_init(1))
    assert one(host, p) == 0
    host.check(host.lib.chx_hip_init(0))
    assert one(host, p) == 1


def instruction_by_instruction(host):
    """A run that looks at the values between the instructions sees all of them."""
    rt = host.chxvm.runtime()
    p = program(host, (16, 96, 16), sums=1)
    assert rt.chxvm_set_option(b"check_types", b"on") == 0
    names = kernels(host, p, (2, 16, 8, 8))
    assert BLOCK not in names and len(names) >= 3
    assert rt.chxvm_set_option(b"check_types", b"off") == 0
    assert kernels(host, p, (2, 16, 8, 8))[-1] == BLOCK


if __name__ == "__main__":
    host_hip.main(globals())
