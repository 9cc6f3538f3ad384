"""Chains of quantized products as one launch (csrc/matmul_chain.hip), codes and floats bit for bit against the oracle."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util
    gpu_util.capi.init(0)
    return gpu_util


@pytest.fixture(scope="module")
def vm(g):
    return importlib.import_module(g.pkg.__name__ + ".chxvm")


def build(vm, rng, rows, dims, types, quantize=True, dequantize=True):
    """A program, its layers' operands, and what it is fed.  types: (a, b) of every layer, then of the result."""
    b = vm.ProgramBuilder()
    zps = [int(rng.integers(0, 256)) if t[0] == "uint8" else int(rng.integers(-128, 128)) for t in types]
    scales = [0.01] + [0.01 * 0.004 * 70 * 40 * np.sqrt(k) / 40 for k in dims[:-1]]
    layers = []
    x = b.input("x", "float32" if quantize else types[0][0], [rows, dims[0]])
    h = b.QuantizeLinear(x, b.scalar(scales[0], "float32"), b.scalar(zps[0], types[0][0])) if quantize else x
    for i in range(len(dims) - 1):
        lo, hi = (0, 256) if types[i][1] == "uint8" else (-128, 128)
        w = rng.integers(lo, hi, size=(dims[i], dims[i + 1])).astype(types[i][1])
        w_zp = int(rng.integers(lo, hi)) if i != 1 else 0
        fa = b.DequantizeLinear(h, b.scalar(scales[i], "float32"), b.scalar(zps[i], types[i][0]))
        fb = b.DequantizeLinear(b.constant(w), b.scalar(0.004, "float32"), b.scalar(w_zp, types[i][1]))
        h = b.QuantizeLinear(b.MatMul(fa, fb), b.scalar(scales[i + 1], "float32"), b.scalar(zps[i + 1], types[i + 1][0]))
        layers.append((w, w_zp))
    if dequantize:
        h = b.DequantizeLinear(h, b.scalar(scales[-1], "float32"), b.scalar(zps[-1], types[-1][0]))
    b.output("y", h)
    return vm.Program(b.serialize()), layers, scales, zps


def expected(oracle, x, layers, scales, zps, types, quantize=True, dequantize=True):
    h = oracle.quantize_linear(x, np.float32(scales[0]), zps[0], np.dtype(types[0][0]).type) if quantize else x
    for i, (w, w_zp) in enumerate(layers):
        h = oracle.qlinear_matmul_int(h, scales[i], zps[i], w, 0.004, w_zp, scales[i + 1], zps[i + 1], np.dtype(types[i + 1][0]).type)
    return oracle.dequantize_linear(h, np.float32(scales[-1]), zps[-1]) if dequantize else h


U, I = ("uint8", "int8"), ("int8", "uint8")


@pytest.mark.parametrize("rows,dims,types", [
    (1, (1, 1), (U, U)),                                      # the smallest
    (17, (64, 16, 2), (U, U, U)),                             # a row past a work-group, fewer columns than a dword holds
    (16, (63, 65, 3), (I, U, I)),                             # a K step that is not whole, a column past a tile
    (33, (784, 100, 100, 10), (U, U, U, U)),
    (5, (1024, 512, 512, 4), (U, I, U, U)),                   # the largest
    (48, (130, 321, 192, 449, 77), (I, I, U, I, U)),          # 6, 3 and 8 tiles of columns: K in 2, 5 and 2 parts
    (2, (20, 64, 128, 64, 33, 7, 5), (U, U, I, U, U, I, U)),  # as many layers as there can be
])
@pytest.mark.parametrize("ends", [(True, True), (True, False), (False, True)])
def test_chain(g, vm, oracle, rows, dims, types, ends):
    rng = np.random.default_rng(sum(dims) + rows)
    program, layers, scales, zps = build(vm, rng, rows, dims, types, *ends)
    if ends[0]:
        x = (rng.standard_normal((rows, dims[0])) * 0.5).astype(np.float32)
        x.ravel()[:3] = (np.inf, -np.inf, np.nan)[:x.size]
    else:
        x = rng.integers(0, 256, size=(rows, dims[0])).astype(np.uint8).view(types[0][0])
    before = vm.counter("matmul_chains")
    got = program.run({"x": g.dev(x)})["y"]
    assert vm.counter("matmul_chains") == before + 1
    want = expected(oracle, x, layers, scales, zps, types, *ends)
    assert got.dtype == want.dtype
    np.testing.assert_array_equal(got.view(np.uint8), want.view(np.uint8))
    # recorded, with other input in the same buffer, and with eager runs in between
    buf = g.dev(x)
    replay = program.capture({"x": buf})
    for i in range(3):
        other = np.roll(x, i, axis=0)
        buf.copy_(g.dev(other))
        torch.cuda.synchronize()
        replay.launch()
        replay.synchronize()
        want = expected(oracle, other, layers, scales, zps, types, *ends)
        np.testing.assert_array_equal(replay.outputs()["y"].view(np.uint8), want.view(np.uint8))
        np.testing.assert_array_equal(program.run({"x": buf})["y"].view(np.uint8), want.view(np.uint8))


def test_rows_of_a_larger_array(g, vm, oracle):
    """Strided rows are taken as they are; columns that are not next to each other run as the program wrote them."""
    rng = np.random.default_rng(4)
    types = (U, U, U)
    program, layers, scales, zps = build(vm, rng, 20, (96, 40, 12), types)
    whole = rng.standard_normal((20, 200)).astype(np.float32)
    for view, chains in ((lambda t: t[:, 3:99], 1), (lambda t: t[:, ::2][:, :96], 0)):
        before = vm.counter("matmul_chains")
        got = program.run({"x": view(g.dev(whole))})["y"]
        assert vm.counter("matmul_chains") == before + chains
        np.testing.assert_array_equal(got, expected(oracle, np.ascontiguousarray(view(whole)), layers, scales, zps, types))
