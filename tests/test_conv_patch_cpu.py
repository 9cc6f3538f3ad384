"""Which convolutions the small tiles run with their pixels in LDS (csrc/conv_split.hip, kPatch), without a GPU: the form gives the
codes of the others, so that tests/test_gpu_conv_patch.py cannot tell."""
import ctypes
import os

import pytest

import host_hip


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["cases", "limits"])
def test_case(host_so, case):
    from test_gpu_conv_patch import CASES, TILES
    host_hip.run_case(host_so, __file__, case, CASES=repr(CASES), TILES=repr(TILES))


def form(host, tile, N, C, H, W, OC, k, pad, stride=1, pixels=None, rows=None, patch=1):
    """kPoint, kTaps or kPatch of the launch with this tile."""
    os.environ["CHX_HIP_TILE"] = "%d,%d,%d,%d" % (tile[0], tile[1], patch, tile[2])
    w, ws, zp = host.tensor("int8", (OC, C, k, k)), host.tensor("float32", (OC,)), host.tensor("int8", (OC,))
    params, plan = host.capi.conv_params((stride, stride), (pad, pad), (pad, pad), 1), ctypes.c_void_p()
    host.check(host.lib.chx_hip_qconv_plan_create(ctypes.byref(w), ctypes.byref(ws), ctypes.byref(zp), None, ctypes.byref(params), None, ctypes.byref(plan)))
    pixels = pixels or (C + 15) // 16 * 16
    rows = rows or W * pixels
    o = [(n + 2 * pad - k) // stride + 1 for n in (H, W)]
    x, y = host.tensor("uint8", (N, C, H, W), [H * rows, 1, rows, pixels]), host.channels_last("uint8", (N, OC, o[0], o[1]), (OC + 15) // 16 * 16)
    host.clear()
    host.check(host.plan_run(plan, x, y))
    names = host.launches()
    host.lib.chx_hip_qconv_plan_destroy(plan)
    for a in (x, y, w, ws, zp):
        host.check(host.lib.chx_hip_free(ctypes.c_void_p(a.data)))
    assert len(names) == 1 and "conv_split_kernel<%d, %d, %d, " % (tile[0], tile[1] // tile[0], tile[2]) in names[0], (tile, names)
    return ("kPoint", "kTaps", "kPatch")[int(names[0].split("Form)")[1][0])]


def cases(host):
    for tile in eval(os.environ["TILES"]):
        for case in eval(os.environ["CASES"]):
            same_size = 2 * case[6] == case[5] - 1
            assert form(host, tile, *case) == ("kPatch" if same_size else "kTaps"), (tile, case)
            assert form(host, tile, *case, patch=0) == "kTaps"


def limits(host):
    tile = (16, 16, 8)
    shape = (1, 64, 14, 14, 32)
    assert form(host, tile, *shape, 3, 1) == "kPatch" and form(host, tile, *shape, 5, 2) == "kPatch" and form(host, tile, *shape, 1, 0) == "kPoint"
    assert form(host, tile, *shape, 3, 1, stride=2) == "kTaps" and form(host, tile, *shape, 3, 0) == "kTaps"
    assert form(host, tile, *shape, 3, 1, pixels=128) == "kPatch"
    assert form(host, tile, *shape, 3, 1, rows=15 * 64) == "kTaps"  # a crop: a tap is no distance in pixels
    # (16 + 2 W + 2) pixels of 1040 bytes in 160 KB less 8 KB of partial sums
    assert form(host, tile, 1, 1024, 4, 64, 32, 3, 1) == "kPatch" and form(host, tile, 1, 1024, 4, 66, 32, 3, 1) == "kTaps"


if __name__ == "__main__":
    host_hip.main(globals())
