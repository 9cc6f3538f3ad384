"""QLinearConv plans on NCHW arrays and on packed channels-last ones: the planar depthwise kernel
(csrc/depthwise_planar.hip) and the layout changes around the matrix-core kernel (csrc/layout.hip), at rows shorter than an access, ragged tiles and the last bytes of an array."""
import numpy as np
import pytest
import torch

from test_gpu_conv_split import codes, g  # noqa: F401 (g is a fixture)

pytestmark = pytest.mark.gpu

# N, C, H, W, OC, k, stride, pad, group
CASES = [(1, 16, 1, 1, 16, 3, 1, 1, 16), (2, 32, 7, 7, 32, 3, 1, 1, 32), (1, 16, 9, 8, 16, 3, 2, 1, 16), (3, 48, 13, 30, 48, 3, 1, 0, 48), (2, 16, 18, 37, 16, 3, 2, 1, 16),
         (1, 64, 8, 8, 64, 1, 1, 0, 1), (2, 70, 7, 7, 33, 3, 1, 1, 1), (1, 24, 5, 13, 130, 1, 1, 0, 1), (1, 17, 3, 43, 16, 3, 2, 1, 1)]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("channels_last", [False, True])
def test_against_the_oracle(g, oracle, case, channels_last):
    N, C, H, W, OC, k, st, pad, group = case
    rng = np.random.default_rng(C + W)
    for xdt, ydt, xz, yz, rne, relu, bias_mode in [(np.uint8, np.uint8, 0, 0, False, True, 2), (np.uint8, np.uint8, 77, 9, False, True, 1),
                                                   (np.uint8, np.uint8, 3, 120, False, False, 0), (np.int8, np.int8, -9, 5, True, False, 2)]:
        x, w = codes(rng, (N, C, H, W), xdt), codes(rng, (OC, C // group, k, k), np.int8)
        ws, bias = rng.uniform(0.002, 0.02, size=OC).astype(np.float32), rng.integers(-3000, 3000, size=OC).astype(np.int32)
        ys = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C // group * k * k) / 40)
        flags = (g.capi.ROUND_ONNX_RNE if rne else 0) | (g.capi.FUSE_RELU if relu else 0) | (g.capi.BIAS_ONNX_INT32 if bias_mode == 2 else 0)
        plan = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(OC, np.int8)), g.dev(bias) if bias_mode else None, strides=(st, st), pads=(pad, pad), group=group)
        got = plan.run(g.to_channels_last(g.dev(x)) if channels_last else g.dev(x), 0.02, xz, ys, yz, zero_point_dtype=torch.uint8 if ydt == np.uint8 else torch.int8, flags=flags)
        assert channels_last or got.is_contiguous()
        okw = dict(bias=bias, bias_mode=oracle.BIAS_ONNX_INT32 if bias_mode == 2 else oracle.BIAS_REFERENCE_FLOAT) if bias_mode else {}
        want = oracle.qlinear_conv_int(x, 0.02, xz, w, ws, np.zeros(OC, np.int8), ys, yz, ydt, strides=(st, st), pads=(pad, pad), group=group,
                                       round_mode=oracle.ROUND_ONNX_RNE if rne else oracle.ROUND_REFERENCE, **okw)
        np.testing.assert_array_equal(g.host(got), np.maximum(want, yz) if relu else want)
        plan.close()


@pytest.mark.parametrize("result", ["channels_last", "nchw"])
def test_packed_pixels_on_two_streams_and_in_a_recording(g, oracle, result):
    """One plan over packed channels-last arrays: on two streams at once, and recorded without a run before."""
    import ctypes
    rng, N, C, H, W, OC = np.random.default_rng(2), 8, 24, 28, 28, 40
    w, ws = codes(rng, (OC, C, 3, 3), np.int8), rng.uniform(0.002, 0.02, size=OC).astype(np.float32)
    ys = float(0.02 * 0.01 * 74 * 74 * np.sqrt(C * 9) / 40)
    xs = [codes(rng, (N, C, H, W), np.uint8) for _ in range(2)]
    wants = [oracle.qlinear_conv_int(x, 0.02, 3, w, ws, np.zeros(OC, np.int8), ys, 120, np.uint8, pads=(1, 1)) for x in xs]
    lib, like = g.capi.lib(), lambda: torch.empty((N, OC, H, W), dtype=torch.uint8, device="cuda").contiguous(
        memory_format=torch.channels_last if result == "channels_last" else torch.contiguous_format)
    x_dev, outs = [g.to_channels_last(g.dev(x)) for x in xs], [like() for _ in xs]
    plan = g.ops.QLinearConvPlan(g.dev(w), g.dev(ws), g.dev(np.zeros(OC, np.int8)), None, pads=(1, 1))
    run = lambda i, o: plan.run(x_dev[i], 0.02, 3, ys, 120, out=o)
    torch.cuda.synchronize()
    plan._plan_for(x_dev[0])
    stream, graph = torch.cuda.Stream(), ctypes.c_void_p()
    recorded = like()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        s = ctypes.c_void_p(stream.cuda_stream)
        g.capi.check(lib.chx_hip_capture_begin(s))
        try:
            run(0, recorded)
        finally:
            g.capi.check(lib.chx_hip_capture_end(s, ctypes.byref(graph)))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for _ in range(20):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                for o in outs[i:i + 1] * 3:
                    o.zero_()
                    run(i, o)
        recorded.zero_()
        torch.cuda.synchronize()
        g.capi.check(lib.chx_hip_graph_launch(graph, ctypes.c_void_p(stream.cuda_stream)))
        torch.cuda.synchronize()
        for got, want in zip(outs + [recorded], wants + wants[:1]):
            np.testing.assert_array_equal(g.host(got), want)
    lib.chx_hip_graph_destroy(graph)
    plan.close()
