"""Which convolutions the 3x3 kernel with the pixels in LDS takes (csrc/conv_same.hip), without a GPU: its codes are those of the
other kernels, so that tests/test_gpu_conv_same.py cannot tell which ran."""
import ctypes
import os

import pytest

import host_hip


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["cases", "limits", "described"])
def test_case(host_so, case):
    from test_gpu_conv_same import CASES, TILES
    host_hip.run_case(host_so, __file__, case, CASES=repr(CASES), TILES=repr(TILES))


def taken(host, tile, N, C, H, W, OC, k=3, pad=1, stride=1, pixels=None, rows=None, y_type="uint8"):
    os.environ["CHX_HIP_TILE"] = "%d,%d,100,%d" % tile
    w, ws, zp = host.tensor("int8", (OC, C, k, k)), host.tensor("float32", (OC,)), host.tensor("int8", (OC,))
    params, plan = host.capi.conv_params((stride, stride), (pad, pad), (pad, pad), 1), ctypes.c_void_p()
    host.check(host.lib.chx_hip_qconv_plan_create(ctypes.byref(w), ctypes.byref(ws), ctypes.byref(zp), None, ctypes.byref(params), None, ctypes.byref(plan)))
    pixels = pixels or (C + 15) // 16 * 16
    rows = rows or W * pixels
    o = [(n + 2 * pad - k) // stride + 1 for n in (H, W)]
    x, y = host.tensor("uint8", (N, C, H, W), [H * rows, 1, rows, pixels]), host.channels_last(y_type, (N, OC, o[0], o[1]), (OC + 15) // 16 * 16)
    host.clear()
    host.check(host.plan_run(plan, x, y))
    names = host.launches()
    host.lib.chx_hip_qconv_plan_destroy(plan)
    for a in (x, y, w, ws, zp):
        host.check(host.lib.chx_hip_free(ctypes.c_void_p(a.data)))
    return "conv_same_kernel" in names[0]


def cases(host):
    for tile in eval(os.environ["TILES"]):
        for case in eval(os.environ["CASES"]):
            assert taken(host, tile, *case), (tile, case)


def limits(host):
    tile = (64, 64, 4)
    shape = (1, 64, 14, 14, 32)
    assert taken(host, tile, *shape) and taken(host, tile, *shape, pixels=128)
    for kw in (dict(k=1, pad=0), dict(k=5, pad=2), dict(pad=0), dict(stride=2), dict(rows=15 * 64), dict(y_type="int8")):
        assert not taken(host, tile, *shape, **kw), kw
    assert not taken(host, tile, 1, 320, 5, 5, 32)  # ten K steps to a tap
    # (64 + 2 W + 2) pixels of 272 bytes in 160 KB less the tables
    assert taken(host, tile, 1, 256, 3, 260, 16) and not taken(host, tile, 1, 256, 3, 270, 16)


def described(host):
    """A configuration that brings the pixels into LDS once names no number of work-groups."""
    os.environ.pop("CHX_HIP_TILE", None)
    for n, kernel, lds in ((8, "conv_same_kernel", True), (9, "conv_mfma_kernel", False)):  # (what was measured is shared between plans)
        x, y = host.channels_last("uint8", (n, 64, 28, 28)), host.channels_last("uint8", (n, 64, 28, 28))
        host.hh.hh_prefer(kernel.encode())
        plan, buf = host.plan(64, 64, 3, pads=(1, 1)), ctypes.create_string_buffer(1024)
        host.check(host.plan_run(plan, x, y))
        host.check(host.lib.chx_hip_qconv_plan_describe(plan, buf, ctypes.c_size_t(len(buf))))
        fields = dict(f.split("=") for f in buf.value.decode().split() if "=" in f)
        assert (fields.get("pixels") == "lds") == lds and int(fields["wgs_per_cu"]) <= 4, (kernel, buf.value)


if __name__ == "__main__":
    host_hip.main(globals())
