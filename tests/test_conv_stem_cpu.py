"""Which first layers the planar-input kernel takes (csrc/conv_stem.hip), without a GPU: its codes are those of the other kernels, so that
tests/test_gpu_conv_stem.py cannot tell which ran."""
import ctypes

import pytest

import host_hip


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["rows_far_apart", "small_images_and_large_tiles"])
def test_case(host_so, case):
    host_hip.run_case(host_so, __file__, case)


def kernel(host, dtype, shape, kernel, stride, pad, OC=32, row=None, channel=None):
    """The kernel that takes the convolution, from memory that only its descriptor says is there; None: refused."""
    N, C, H, W = shape
    w, ws, zp = host.tensor("int8", (OC, C, kernel, kernel)), host.tensor("float32", (OC,)), host.tensor("int8", (OC,))
    params, plan = host.capi.conv_params((stride, stride), (pad, pad), (pad, pad), 1), ctypes.c_void_p()
    host.check(host.lib.chx_hip_qconv_plan_create(ctypes.byref(w), ctypes.byref(ws), ctypes.byref(zp), None, ctypes.byref(params), None, ctypes.byref(plan)))
    x = host.tensor(dtype, shape)
    x.strides[2], x.strides[1], x.data = row or x.strides[2], channel or x.strides[1], x.data + (1 << 44)  # (apart from y)
    y = host.channels_last("uint8", (N, OC) + tuple((n + 2 * pad - kernel) // stride + 1 for n in (H, W)), (OC + 15) // 16 * 16)
    host.clear()
    if dtype == "float32":
        rc = host.lib.chx_hip_qconv_plan_run_quantize(plan, ctypes.byref(x), ctypes.c_float(0.1), 7, ctypes.c_float(0.1), 7, ctypes.c_float(0.2), 0, 0, ctypes.byref(y), None)
    else:
        rc = host.plan_run(plan, x, y)
    assert rc == 0 or (dtype == "float32" and rc == host.capi.EUNSUPPORTED and not host.launches())
    names = [line.split("<")[0].split("::")[-1].split("(")[0] for line in host.launches()]
    host.lib.chx_hip_qconv_plan_destroy(plan)
    return names[0] if names else None


def rows_far_apart(host):
    """The kernel's offsets are 32 bits, for a tile's rows outside the image as well: 21 of them with 7x7 filters and a stride of 2, ten with 3x3."""
    for dtype, other in (("uint8", "conv_direct_kernel"), ("float32", None)):
        for k, stride, rows in ((7, 2, 21), (3, 1, 10)):
            most = ((1 << 32) - 1 - 3 * 256) // rows // 4 * 4
            for H in (2, 3):
                for row in (1 << 20, most, most + 4, ((1 << 30) - 1) // H // 4 * 4):
                    taken = row <= most
                    if row * H < 1 << 30:
                        assert kernel(host, dtype, (1, 3, H, 21), k, stride, k // 2, row=row, channel=256) == ("conv_stem_kernel" if taken else other), (dtype, k, H, row)
            # one row has no distance to another
            assert kernel(host, dtype, (1, 3, 1, 21), k, stride, k // 2, row=(1 << 30) - 4, channel=256) == "conv_stem_kernel"


def small_images_and_large_tiles(host):
    """Images of fewer than four columns, and tiles whose rows only fit without the columns in front of them, need no scratch memory; floats are for the others."""
    for shape, k, stride, pad in (((2, 3, 9, 1), 3, 1, 1), ((2, 3, 9, 3), 3, 1, 1), ((1, 3, 2, 2), 7, 2, 3), ((2, 4, 56, 56), 3, 4, 0), ((2, 4, 56, 56), 3, 4, 1), ((1, 4, 56, 57), 3, 4, 3)):
        assert kernel(host, "uint8", shape, k, stride, pad) == "conv_stem_kernel", (shape, pad)
        assert kernel(host, "float32", shape, k, stride, pad) is None, (shape, pad)


if __name__ == "__main__":
    host_hip.main(globals())
