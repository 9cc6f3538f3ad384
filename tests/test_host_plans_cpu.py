"""Which kernels the entry points launch, on what memory, and what they compile at run time, without a GPU."""
import ctypes
import random
import threading
import time

import pytest

import host_hip


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["one_plan_on_dense_images_and_crops", "packed_pixels", "requantization_forms", "shared_memory_of_conv_integer", "kernels_of_a_fused_group", "what_a_plan_costs", "fused_groups_of_many_elements"])
def test_case(host_so, case):
    host_hip.run_case(host_so, __file__, case)


def one_plan_on_dense_images_and_crops(host):
    """A measured configuration is for the strides it was measured on: the pixel-streaming kernel takes dense images only."""
    n, c, h, w = 8, 64, 32, 32
    dense, crop = host.channels_last("uint8", (n, c, h, w)), host.tensor("uint8", (n, c, h, w), [36 * 40 * c, 1, 40 * c, c])
    rows = host.tensor("uint8", (n, c, h, w), [36 * w * c, 1, w * c, c])
    y = host.channels_last("uint8", (n, 64, h, w))
    host.hh.hh_prefer(b"conv_point_kernel")
    for order in ([dense, crop, rows, dense], [crop, dense, rows], [rows, dense, crop]):
        plan = host.plan(64, c, 1)
        for x in order:
            host.check(host.plan_run(plan, x, y))  # measures
            host.clear()
            host.check(host.plan_run(plan, x, y))
            assert len(host.launches()) == 1 and ("conv_point_kernel" in host.launches()[0]) == (x is dense)
        host.lib.chx_hip_qconv_plan_destroy(plan)
    # one image whose rows alone lie apart, on a plan of its own: what other plans have measured is shared
    dense, apart = host.channels_last("uint8", (1, c, 96, 96)), host.tensor("uint8", (1, c, 96, 96), [96 * 96 * c, 1, 100 * c, c])
    y = host.channels_last("uint8", (1, 64, 96, 96))
    for x in (dense, apart, dense):
        plan = host.plan(64, c, 1)
        host.check(host.plan_run(plan, x, y))


def packed_pixels(host):
    """Channels-last arrays whose pixels are no multiple of 16 bytes: what ran without the plan's scratch memory before there
    was a copy for them (in a recording, on a pinned plan, on several streams at once) does so still."""
    n, c, h, w, oc = 2, 24, 14, 14, 40
    x, y, nchw = host.channels_last("uint8", (n, c, h, w)), host.channels_last("uint8", (n, oc, h, w)), host.tensor("uint8", (n, oc, h, w))
    larger = host.channels_last("uint8", (2 * n, c, h, w)), host.channels_last("uint8", (2 * n, oc, h, w))
    streams = [None, host.stream(), host.stream()]
    memory = lambda: [line for line in host.log() if "alloc" in line.lower() or "Synchronize" in line]
    # no warm-up: straight into a recording
    plan, graph = host.plan(oc, c, 1), ctypes.c_void_p()
    host.check(host.lib.chx_hip_capture_begin(streams[1]))
    host.clear()
    host.check(host.plan_run(plan, x, y, stream=streams[1]))
    assert ["conv_direct" in k for k in host.launches()] == [True] and not memory()
    host.check(host.lib.chx_hip_capture_end(streams[1], ctypes.byref(graph)))
    # pinned, and inputs that grow; results channels-last and NCHW
    host.check(host.lib.chx_hip_qconv_plan_pin(plan, 1))
    for xd, yd in [(x, y), larger, (x, nchw), larger]:
        for s in streams:
            host.check(host.plan_run(plan, xd, yd, stream=s))
            host.clear()
            host.check(host.plan_run(plan, xd, yd, stream=s))
            assert any("pixels" in k for k in host.launches()) and not any("conv_direct" in k for k in host.launches())
            # memory of the call on a stream of the caller's, the null stream's block otherwise
            assert [line.startswith("hipMallocAsync") and line.endswith("stream=0x%x" % s.value) for line in memory()] == [True] if s else memory() == []
    host.check(host.lib.chx_hip_qconv_plan_pin(plan, -1))
    # two convolutions as one launch: not for these arrays, and nothing is launched
    both, y2 = host.plan(128, c, 1), host.channels_last("uint8", (n, 64, h, w))
    y1 = host.channels_last("uint8", (n, 64, h, w))
    host.clear()
    rc = host.lib.chx_hip_qconv_plan_run_pair(both, ctypes.byref(x), ctypes.c_float(0.02), 128, 64, ctypes.c_float(0.05), 3, 0, ctypes.byref(y1), ctypes.c_float(0.05), 3, 0,
                                              ctypes.byref(y2), None)
    assert rc == host.capi.EUNSUPPORTED and not host.launches()


def what_a_plan_costs(host):
    """One launch and one allocation (two where one would pass 2 MB).  The weights are there twice, in the order of the staged and
    of the small tiles, but for filters that the small tiles do not take."""
    for oc, c, k, copies, apart in ((128, 64, 1, 2, False), (128, 256, 3, 2, False), (128, 64, 5, 2, False), (128, 64, 7, 1, False), (2048, 512, 1, 2, True), (512, 512, 3, 2, False)):
        host.clear()
        plan = host.plan(oc, c, k)
        weights, sums = oc * k * k * c, oc * 4 * (17 if 1 < k < 6 else 1)
        sizes = [weights + sums, weights] if apart else [weights * copies + sums]
        assert len(host.launches()) == 1
        # (behind those of the filters, scales, zero points that host.plan makes)
        assert [line for line in host.log() if "hipMalloc" in line][3:] == ["hipMalloc %d" % n for n in sizes]
        host.clear()
        host.lib.chx_hip_qconv_plan_destroy(plan)
        assert host.log().count("hipFree") == len(sizes)


def requantization_forms(host):
    """The search for a short form (csrc/core.hip, product_form) runs once per scale and zero point, however many there are
    and whichever thread asks: a network of hundreds of convolutions goes through all of them on every run."""
    plan, x, y = host.plan(64, 64, 1), host.channels_last("uint8", (1, 64, 7, 7)), host.channels_last("uint8", (1, 64, 7, 7))
    params = [(0.01 * 1.003 ** i, i % 5 and 100) for i in range(700)]

    def through_all():
        start = time.perf_counter()
        for scale, zero_point in params:
            host.check(host.plan_run(plan, x, y, scale, zero_point))
        return time.perf_counter() - start

    host.check(host.plan_run(plan, x, y))  # measures
    first, later = through_all(), []
    for target in (lambda: later.append(through_all()),) * 3:
        thread = threading.Thread(target=target)
        thread.start()
        thread.join()
    assert min(later) < first / 3, (first, later)


def shared_memory_of_conv_integer(host):
    """No launch of ConvInteger asks for more than 64 KB of dynamic shared memory, the most that any launch may have without
    being arranged with the device runtime."""
    rng, strips = random.Random(3), 0
    shapes = [(8, 1024, 3, 3, 512, 3, 1, True, 0), (8, 1024, 3, 3, 512, 3, 1, False, 1), (2, 600, 8, 8, 64, 1, 1, False, 0), (1, 48, 9, 8, 64, 3, 2, False, 1)]
    while len(shapes) < 600:
        shapes.append((rng.choice([1, 2, 8, 64]), int(2 ** rng.uniform(2, 11)), rng.choice([3, 8, 9, 14, 28, 57]), rng.choice([1, 3, 8, 14, 28, 57, 112]), rng.choice([16, 64, 512]),
                       rng.choice([1, 3]), rng.choice([1, 2]), rng.random() < 0.5, rng.choice([0, 1])))
    memory = host.malloc(1 << 28)
    for n, c, h, w, oc, k, stride, last, pad in shapes:
        c = c // 4 * 4
        oh, ow = (h + 2 * pad - k) // stride + 1, (w + 2 * pad - k) // stride + 1
        if min(h, w) + 2 * pad < k or max(n * c * h * w, n * oc * oh * ow * 4, oc * c * k * k) > 1 << 28:
            continue
        x = host.tensor("uint8", (n, c, h, w), [h * w * c, 1, w * c, c] if last else None, base=memory)
        wt, y = host.tensor("int8", (oc, c, k, k), base=memory), host.tensor("int32", (n, oc, oh, ow), base=memory)
        params = host.capi.conv_params((stride, stride), (pad, pad), (pad, pad), 1)
        host.clear()
        host.check(host.lib.chx_hip_conv_integer(ctypes.byref(x), ctypes.byref(wt), 128, None, ctypes.byref(params), ctypes.byref(y), None))
        for launch in host.launches():
            assert int(launch.split("lds=")[1].split()[0]) <= 64 * 1024, ((n, c, h, w, oc, k, stride, last, pad), launch)
            strips += "conv_strip_kernel" in launch
    assert strips > 20


def kernels_of_a_fused_group(host):
    """A call compiles the kernel it takes and no other, and calls that differ in ranks and extents share one: the general
    kernel is one per way in which the operands are addressed."""
    def call(program, dtype, shapes, strides=(None, None, None)):
        ins = [host.tensor(dtype, s, st) for s, st in zip(shapes, strides)]
        nd = max(len(s) for s in shapes)
        out = host.tensor(dtype, [max(s[k - nd] if k - nd >= -len(s) else 1 for s in shapes) for k in range(nd)])
        host.clear()
        host.check(host.lib.chx_hip_elementwise(program.encode(), 5, host.capi.tensor_array(ins), len(ins), host.capi.tensor_array([out]), 1, None))
        loads = sum(line == "hipModuleLoadData" for line in host.log())
        return loads, [k.split()[0] for k in host.launches()]

    text = "chxhip-fusion 1\nin a:%s b:%s c:%s\nm = Mul b c\ny = Add a m\nout y:%s\n"
    # dense, a row, one per row: one to three axes, one row, a short last vector
    ranks = [((9, 1001), (1001,), (9, 1)), ((2, 9, 77), (77,), (1, 9, 1)), ((5, 6, 333), (6, 333), (5, 6, 1)), ((3, 2, 19), (3, 1, 19), (2, 1))]
    short = [((9, 3), (3,), (9, 1)), ((2, 9, 3), (9, 3), (2, 1, 3)), ((7, 2, 3), (1, 2, 1), (3,))]
    for dtype in ("float16", "float32"):
        program = text % ((dtype,) * 4)
        for group in (ranks, short):
            results = [call(program, dtype, shapes) for shapes in group]
            assert results == [(1, ["fusion5_gen"])] + [(0, ["fusion5_gen"])] * (len(group) - 1), results
        strided = [call(program, dtype, [(n, 21)] * 3, [[42, 2]] * 3) for n in (1, 5, 300)]
        assert strided == [(1, ["fusion5_gen"]), (0, ["fusion5_gen"]), (0, ["fusion5_gen"])]
    # the vector kernel, and the general one when a call needs it
    assert call(program, "float32", [(64, 64)] * 3) == (1, ["fusion5_vec"]) and call(program, "float32", [(8, 128)] * 3) == (0, ["fusion5_vec"])
    assert call(program, "float32", [(3, 7)] * 3) == (1, ["fusion5_gen"]) and call(program, "float32", [(2, 3, 5)] * 3) == (0, ["fusion5_gen"])
    # which of them a general call needs does not make the vector kernel another
    assert call(program, "float32", [(64, 64)] * 3) == (0, ["fusion5_vec"]) and call(program, "float32", [(4, 8, 8, 4)] * 3) == (0, ["fusion5_vec"])


def fused_groups_of_many_elements(host):
    """A launch has fewer than 2^32 threads; a group of more elements than those of one launch take is several."""
    memory = host.malloc(64)
    for dtype, rows, row in [("float32", 1 << 31, 3), ("float32", 5 << 20, 1001), ("float16", 1 << 31, 5), ("float16", 1 << 34, 1)]:
        text = "chxhip-fusion 1\nin a:%s b:%s\ny = Add a b\nout y:%s\n" % ((dtype,) * 3)
        wide, one, out = host.tensor(dtype, (rows, row), base=memory), host.tensor(dtype, (rows, 1), base=memory), host.tensor(dtype, (rows, row), base=memory)
        host.clear()
        host.check(host.lib.chx_hip_elementwise(text.encode(), 6, host.capi.tensor_array([wide, one]), 2, host.capi.tensor_array([out]), 1, None))
        grids = [int(k.split("grid=")[1]) for k in host.launches()]
        assert max(grids) * 256 < 1 << 32 and len(grids) >= 1, grids
        per_thread = 1 if row in (3, 5) else 8 if dtype == "float16" else 4
        assert sum(grids) == -(-rows * row // (256 * per_thread)), grids


if __name__ == "__main__":
    host_hip.main(globals())
