"""The general fused kernel (emit_general in csrc/elementwise_rtc.hip): operands of every addressing form, result sizes
around the vector width, unaligned views, each element type."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util
    return gpu_util


# shapes of the operands of a + b * c: flat, rows repeated (C), inner axis repeated (Z), one element, rows shorter than a vector
CASES = [((7,), (7,), ()), ((1,), (1,), (1,)), ((3, 5), (5,), (3, 1)), ((4, 3, 2), (3, 1), (2,)), ((9, 1001), (1001,), (9, 1)),
         ((5, 1, 17), (6, 1), (1, 6, 17)), ((2, 3, 1, 9), (3, 4, 1), (4, 9)), ((33, 8), (8,), (33, 8)), ((2, 257, 3), (257, 1), (3,)),
         ((2, 1, 3, 1, 5), (1, 4, 1, 6, 1), (5,)), ((2, 3, 2, 2, 19), (3, 1, 2, 1), (2, 1, 2, 1, 19))]


@pytest.mark.parametrize("shapes", CASES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.float64])
def test_broadcast_forms(g, shapes, dtype):
    rng = np.random.default_rng(len(str(shapes)))
    prog = g.ops.fusion_program([(n, dtype) for n in "abc"], [("m", "Mul", "b", "c"), ("y", "Add", "a", "m")], [("m", dtype), ("y", dtype)])
    t = [g.dev(rng.standard_normal(s).astype(np.float32)).to(dtype).reshape(s) for s in shapes]
    for _ in range(2):  # the second call takes the kept plan
        m, y = g.ops.ElementWiseNvrtc(t, 2, prog, 21)
        want_m = (t[1] * t[2]).expand(y.shape)
        assert torch.equal(m, want_m) and torch.equal(y, t[0] + want_m)
    # a view that starts one element into its memory, and one with a stride on the innermost axis
    base = g.dev(rng.standard_normal((int(np.prod(shapes[0])) + 1,)).astype(np.float32)).to(dtype)
    a = base[1:].reshape(shapes[0])
    wide = g.dev(rng.standard_normal((int(np.prod(shapes[0])), 3)).astype(np.float32)).to(dtype)
    for a in (a, wide[:, 1].reshape(shapes[0]) if len(shapes[0]) == 1 else torch.stack([a, a], -1)[..., 0]):
        m, y = g.ops.ElementWiseNvrtc([a, t[1], t[2]], 2, prog, 21)
        assert torch.equal(y, a + want_m)


@pytest.mark.parametrize("n", [1, 3, 15, 16, 17, 1023])
def test_codes_of_every_count(g, oracle, n):
    rng = np.random.default_rng(n)
    qa, qb = rng.integers(0, 256, size=(2, n)).astype(np.uint8), rng.integers(-128, 128, size=(n,)).astype(np.int8)
    for mixed in (False, True):
        prog = g.ops.fusion_program(
            [("qa", torch.uint8), ("qb", torch.int8)],
            [("a", "DequantizeLinear", "qa", 0.05, 128), ("b", "DequantizeLinear", "qb", 0.02, -3), ("s", "Add", "a", "b"),
             ("q", "QuantizeLinear", "s", 0.06, 7, "int8")], [("q", torch.int8)] + ([("s", torch.float32)] if mixed else []))
        out = g.ops.ElementWiseNvrtc([g.dev(qa), g.dev(qb)], 2 if mixed else 1, prog, 22)
        s = oracle.binary(oracle.ADD, oracle.dequantize_linear(qa, 0.05, 128), oracle.dequantize_linear(np.broadcast_to(qb, (2, n)).copy(), 0.02, -3))
        np.testing.assert_array_equal(g.host(out[0]), oracle.quantize_linear(s, 0.06, 7, np.int8))
        if mixed:
            np.testing.assert_array_equal(g.host(out[1]), s)


def test_operands_that_reach_far_or_backwards(g):
    """64-bit offsets: rows 2^31 elements apart, and strides below zero."""
    import ctypes
    rng = np.random.default_rng(4)
    prog = g.ops.fusion_program([(n, torch.float16) for n in "ab"], [("y", "Sub", "a", "b")], [("y", torch.float16)])
    far = torch.empty((1 << 31) + 4096, dtype=torch.float16, device="cuda").as_strided((2, 1001), (1 << 31, 1))
    near = g.dev(rng.standard_normal((2, 1001)).astype(np.float16))
    far.copy_(g.dev(rng.standard_normal((2, 1001)).astype(np.float16)))
    row = near[0]
    for a, b in [(far, near), (row, far), (far, far)]:
        assert torch.equal(g.ops.ElementWiseNvrtc([a, b], 1, prog, 23)[0], a - b)
    # descriptors made by hand: torch has no strides below zero
    src = g.dev(rng.standard_normal((3, 40)).astype(np.float16))
    out = torch.empty((3, 40), dtype=torch.float16, device="cuda")
    backwards = g.capi.make_desc(src.data_ptr() + 2 * (3 * 40 - 1), g.capi.FLOAT16, (3, 40), (-80, -2))
    ins = g.capi.tensor_array([backwards, g.capi.desc(src)])
    outs = g.capi.tensor_array([g.capi.desc(out)])
    code = prog.encode() if isinstance(prog, str) else prog
    g.capi.check(g.capi.lib().chx_hip_elementwise(code, 24, ins, 2, outs, 1, g.capi.stream_ptr()))
    assert torch.equal(out, src.flip(0, 1) - src)


def test_more_elements_than_one_launch_takes(g):
    prog = g.ops.fusion_program([(n, torch.float16) for n in "ab"], [("y", "Add", "a", "b")], [("y", torch.float16)])
    rows = (1 << 30) + 5  # of three: an element per thread, two launches
    a = torch.arange(rows, device="cuda", dtype=torch.int32).remainder_(997).to(torch.float16).unsqueeze(1)
    b = torch.tensor([1.0, 2.0, 4.0], device="cuda", dtype=torch.float16)
    y = g.ops.ElementWiseNvrtc([a, b], 1, prog, 25)[0]
    for k in range(3):
        assert torch.equal(y[:, k], a[:, 0] + b[k])
