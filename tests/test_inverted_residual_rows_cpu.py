"""Which inverted residual blocks take the kernel with one buffer of each kind (csrc/inverted_residual.hip), without a GPU: its codes are those
of the kernel with two, so that tests/test_gpu_inverted_residual_rows.py cannot tell which ran."""
import ctypes
import re

import pytest

import host_hip


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["one_buffer", "two_buffers"])
def test_case(host_so, case):
    from test_gpu_inverted_residual_rows import BLOCKS
    host_hip.run_case(host_so, __file__, case, BLOCKS=repr([(b[:5], k) for b, k in BLOCKS]))


def kernel(host, N, channels, H, W, stride):
    cin, hid, cout = channels
    operands, kept = [], []
    for shape in ((hid, cin, 1, 1), (hid, 1, 3, 3), (cout, hid, 1, 1)):
        d = [host.tensor("int8", shape), host.tensor("float32", shape[:1]), host.tensor("int8", shape[:1])]
        kept += d
        operands += [ctypes.addressof(t) for t in d] + [None]
    block, lib = ctypes.c_void_p(), host.lib
    host.check(lib.chx_hip_inverted_residual_create((ctypes.c_void_p * 12)(*operands), stride, None, ctypes.byref(block)))
    pitch = [(c + 15) // 16 * 16 for c in channels]
    x, y = host.channels_last("uint8", (N, cin, H, W), pitch[0]), host.channels_last("uint8", (N, cout, (H - 1) // stride + 1, (W - 1) // stride + 1), pitch[2])
    host.clear()
    host.check(lib.chx_hip_inverted_residual_run(
        block, ctypes.byref(x), ctypes.c_float(0.02), 77, (ctypes.c_float * 3)(0.03, 0.05, 0.07), (ctypes.c_int32 * 3)(0, 0, 128), host.capi.UINT8, 0, None,
        ctypes.c_float(0), 0, ctypes.c_float(0), 0, 0, ctypes.byref(y), None))
    line, = host.launches()
    lib.chx_hip_inverted_residual_destroy(block)
    for t in kept + [x, y]:
        host.check(lib.chx_hip_free(ctypes.c_void_p(t.data)))
    return tuple(int(v) for v in re.search(r"inverted_residual_kernel<(\d+), (\d+), (\d+), (\d+), (\d+)>", line).groups())


def one_buffer(host):
    import os
    for (N, channels, H, W, stride), (tiles, per_interval, steps) in eval(os.environ["BLOCKS"]):
        assert kernel(host, N, channels, H, W, stride) == (stride, tiles, per_interval, steps, 1), (N, channels, H, W, stride)


def two_buffers(host):
    """Where a strip is most of an image, or one round does not fill the chip, and for more input channels than the registers take."""
    for block in ((128, (64, 384, 64), 14, 14, 1), (128, (96, 576, 160), 14, 14, 2), (128, (160, 960, 160), 7, 7, 1), (1, (24, 144, 24), 56, 56, 1), (2, (16, 96, 24), 112, 112, 2),
                  (40, (100, 300, 24), 30, 30, 1)):
        assert kernel(host, *block)[4] == 2, block


if __name__ == "__main__":
    host_hip.main({f.__name__: f for f in (one_buffer, two_buffers)})
