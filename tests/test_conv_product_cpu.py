"""Which ConvInteger calls are products (csrc/contract_api.hip, run_conv_as_product), without a GPU."""
import ctypes

import pytest

import host_hip


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["products", "other_forms", "packed_weights", "short_and_parted_rows"])
def test_case(host_so, case):
    host_hip.run_case(host_so, __file__, case)


def is_product(host, n=3, c=40, h=9, w=7, oc=24, k=1, strides=(1, 1), pads=(0, 0), group=1, channels_last=False, pitch=None, y_channels_last=None, zero_points=0, w_strides=None):
    oh, ow = (h + 2 * pads[0] - k) // strides[0] + 1, (w + 2 * pads[1] - k) // strides[1] + 1
    x = host.channels_last("uint8", (n, c, h, w), pitch) if channels_last else host.tensor("uint8", (n, c, h, w), pitch and [c * h * pitch, h * pitch, pitch, 1])
    y = (host.channels_last if (channels_last if y_channels_last is None else y_channels_last) else host.tensor)("int32", (n, oc, oh, ow))
    f = host.tensor("int8", (oc, c // group, k, k), w_strides)
    zp = host.tensor("int8", (zero_points,)) if zero_points else None
    params = host.capi.conv_params(strides, pads, pads, group)
    host.clear()
    host.check(host.lib.chx_hip_conv_integer(ctypes.byref(x), ctypes.byref(f), 5, ctypes.byref(zp) if zp else None, ctypes.byref(params), ctypes.byref(y), None))
    assert not any("gemm_i8_stage" in name for name in host.launches())  # (more than 64 KB of LDS)
    return any("gemm_i8" in name for name in host.launches())


def products(host):
    for channels_last in (False, True):
        assert is_product(host, channels_last=channels_last)
        assert is_product(host, channels_last=channels_last, zero_points=1)
        assert is_product(host, channels_last=channels_last, h=1, w=1)
        assert is_product(host, channels_last=channels_last, n=1, w=1)
    assert is_product(host, channels_last=True, zero_points=24) and not is_product(host, zero_points=24)
    assert is_product(host, channels_last=True, pitch=57)
    # strides: rows of results equally far apart, or one image
    assert is_product(host, strides=(2, 2), channels_last=True, h=8) and is_product(host, strides=(2, 1), channels_last=True, h=8) and is_product(host, strides=(1, 3), channels_last=True)
    assert is_product(host, strides=(2, 2), channels_last=True, n=1) and not is_product(host, strides=(2, 2), channels_last=True, h=9) and not is_product(host, strides=(2, 2))
    assert is_product(host, n=64, c=200, h=56, w=56, oc=200) and is_product(host, n=64, c=200, h=56, w=56, oc=200, channels_last=True)


def other_forms(host):
    assert not is_product(host, k=3, pads=(1, 1)) and not is_product(host, pads=(1, 1)) and not is_product(host, pads=(1, 1), channels_last=True)
    assert not is_product(host, group=2) and not is_product(host, c=15)
    assert not is_product(host, pitch=9)  # rows apart
    assert not is_product(host, channels_last=True, y_channels_last=False) and not is_product(host, y_channels_last=True)
    assert not is_product(host, w_strides=[1, 24, 1, 1])  # filters across


def packed_weights(host):
    """Large channels-last layers multiply on the packed kernel, which reads the filters' zero points back and packs them on every
    call; where a product is faster, in a recording, and with zero points that are not 0 they are a product."""
    def kernels(n, c, hw, oc, zero_point=0, stride=1, stream=None):
        o = (hw - 1) // stride + 1
        x, y = host.channels_last("uint8", (n, c, hw, hw)), host.channels_last("int32", (n, oc, o, o))
        f, zp = host.tensor("int8", (oc, c, 1, 1)), host.tensor("int8", ())
        host.bytes(zp.data, bytes([zero_point]))
        params = host.capi.conv_params((stride, stride), (0, 0), (0, 0), 1)
        host.clear()
        host.check(host.lib.chx_hip_conv_integer(ctypes.byref(x), ctypes.byref(f), 5, ctypes.byref(zp), ctypes.byref(params), ctypes.byref(y), stream))
        for a in (x, y, f):
            host.check(host.lib.chx_hip_free(ctypes.c_void_p(a.data)))
        return ["packed" if "conv_mfma" in k else "product" if "gemm_i8" in k else "other" for k in host.launches() if "pack_weights" not in k]

    assert kernels(64, 1024, 28, 1024) == ["packed"] and kernels(64, 512, 56, 512) == ["packed"]
    assert kernels(64, 1024, 28, 1024, zero_point=3) == ["product"]
    assert kernels(32, 1024, 56, 1024, stride=2) == ["packed"] and kernels(64, 2000, 28, 400, stride=2) == ["packed"]
    assert kernels(64, 256, 56, 384) == ["product"] and kernels(64, 512, 28, 320) == ["product"]  # (few channels, 8 G multiply-adds)
    assert kernels(64, 1024, 14, 1024) == ["product"] and kernels(32, 256, 112, 512) == ["product"]
    assert kernels(64, 2048, 7, 3072) == ["product"]  # 3136 pixels, 6 MB of filters
    # few filters beside a tile of 128, and as many as fill it; rows of results with strides
    assert kernels(20, 512, 72, 280) == ["packed"] and kernels(48, 1696, 30, 152) == ["packed"] and kernels(48, 1696, 30, 120) == ["product"]
    assert kernels(59, 400, 37, 1872, stride=2) == ["packed"] and kernels(20, 400, 38, 1872, stride=2) == ["product"]
    s, graph = host.stream(), ctypes.c_void_p()
    host.check(host.lib.chx_hip_capture_begin(s))
    assert kernels(64, 1024, 28, 1024, stream=s) == ["product"]
    host.check(host.lib.chx_hip_capture_end(s, ctypes.byref(graph)))


def short_and_parted_rows(host):
    """Products that would be mostly padding, or write parts of lines, are for the other kernels, but in a recording."""
    assert not is_product(host, n=51, c=216, h=7, w=7, oc=1336) and is_product(host, n=8, c=1016, h=7, w=7, oc=664)  # 49 columns, many and few tiles
    assert is_product(host, n=125, c=160, h=11, w=11, oc=128)
    assert not is_product(host, n=73, c=1640, h=5, w=5, oc=960) and not is_product(host, n=247, c=120, h=5, w=5, oc=200)  # 25 columns
    assert not is_product(host, n=36, c=16, h=38, w=38, oc=1168) and not is_product(host, n=16, c=120, h=29, w=29, oc=1936)  # parts of lines
    assert not is_product(host, n=246, c=32, h=35, w=35, oc=200) and is_product(host, n=230, c=32, h=56, w=56, oc=104)
    assert not is_product(host, n=55, c=672, h=10, w=10, oc=80, strides=(2, 2), channels_last=True)  # strips
    assert is_product(host, n=10, c=136, h=48, w=48, oc=320, strides=(2, 2), channels_last=True)
    assert not is_product(host, n=62, c=544, h=8, w=8, oc=1312, strides=(2, 2), channels_last=True)  # planes
    assert is_product(host, n=135, c=552, h=14, w=14, oc=304, strides=(2, 2), channels_last=True)
    # what the others do not take: rows of results that are strided differently, a stride of 3
    assert is_product(host, n=62, c=544, h=8, w=8, oc=1312, strides=(2, 1), channels_last=True) and is_product(host, n=62, c=544, h=12, w=12, oc=1312, strides=(3, 3), channels_last=True)


if __name__ == "__main__":
    host_hip.main(globals())
