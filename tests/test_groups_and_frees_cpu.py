"""Programs whose groups of instructions, each of which would run as one launch (runtime/chxvm.cc), overlap around the Free of an operand that they
share, without a GPU: every such program runs, twice."""
import ctypes
import os
import re
import sys

import pytest

import host_hip


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.fixture(scope="module")
def sum_code():
    sys.path.insert(0, host_hip.ROOT)
    import __graft_entry__ as entry
    pkg = entry.load_package()
    return pkg.workloads.add_program(pkg.ops, (0.2, 0), (0.1, 7), (0.4, 120))


@pytest.mark.parametrize("case", ["first_layers", "last_layers", "scales", "inverted_residuals", "bottlenecks", "products", "a_pool_between", "one_group"])
def test_case(host_so, sum_code, case):
    host_hip.run_case(host_so, __file__, case, SUM_CODE=sum_code)


class Program:
    def __init__(self, host):
        self.host, self.b = host, host.chxvm.ProgramBuilder()
        self.b.scales = lambda s, z: (self.b.scalar(s, "float32"), self.b.scalar(z, "uint8"))

    def convolution(self, x, scale, shape, out, stride=1, group=1):
        import numpy as np
        b = self.b
        w, ws, wz = b.constant(np.ones(shape, np.int8)), b.constant(np.full(shape[0], 0.01, np.float32)), b.constant(np.zeros(shape[0], np.int8))
        return b.QLinearConv(x, *scale, w, ws, wz, *out, b.constant(np.zeros(shape[0], np.int32)), [stride] * 2, [shape[2] // 2] * 2, group, "")

    def kernels(self, inputs):
        """The kernels of the second of two runs."""
        rt, p = self.host.chxvm.runtime(), self.host.program(self.b)
        assert rt.chxvm_set_option(b"qlinearconv_bias", b"onnx_int32") == 0
        for _ in range(2):
            self.host.clear()
            out = ctypes.c_void_p()
            assert rt.chxvm_program_run(p, *self.host.names_and(inputs), 0, ctypes.byref(out)) == 0, rt.chxvm_last_error()
            rt.chxvm_outputs_destroy(out)
        return [re.match(r"(?:void )?(?:\w+::|\(anonymous namespace\)::)*(\w+)", line).group(1) for line in self.host.launches()]


def first_layers(host):
    """Two convolutions over one image, each with a quantization of its own."""
    p = Program(host)
    x = p.b.input("x", "float32", [2, 3, 8, 8])
    scales = [p.b.scales(0.1 * (i + 1), 7) for i in range(2)]
    q = [p.b.QuantizeLinear(x, *s) for s in scales]
    p.b.Free(x)
    for i in range(2):
        p.b.output("y%d" % i, p.convolution(q[i], scales[i], (32, 3, 3, 3), p.b.scales(0.2, 0)))
    names = p.kernels({"x": host.tensor("float32", (2, 3, 8, 8))})
    assert names.count("quantize_flat_kernel") == 1 and names.count("conv_stem_kernel") == 2, names


def last_layers(host):
    """Two heads on one feature map."""
    p = Program(host)
    x, scale = p.b.input("x", "uint8", [2, 64, 8, 8]), p.b.scales(0.1, 7)
    heads = []
    for i in range(2):
        own = p.b.scales(0.2, 3)
        heads.append((p.convolution(x, scale, (16, 64, 1, 1), own, stride=i + 1), own))
    p.b.Free(x)
    for i, (h, own) in enumerate(heads):
        p.b.output("y%d" % i, p.b.DequantizeLinear(h, *own))
    names = p.kernels({"x": host.channels_last("uint8", (2, 64, 8, 8))})
    assert len(names) == 3 and sum(n.startswith("dequantize") for n in names) == 1, names


def scales(host):
    """... and on two, with scales and zero points in common."""
    p = Program(host)
    x, own = [p.b.input("x%d" % i, "uint8", [2, 64, 8, 8]) for i in range(2)], p.b.scales(0.2, 3)
    scale = p.b.scales(0.1, 7)
    heads = [p.convolution(x[i], scale, (16, 64, 1, 1), own) for i in range(2)]
    for slot in scale:
        p.b.Free(slot)
    for i, h in enumerate(heads):
        p.b.output("y%d" % i, p.b.DequantizeLinear(h, *own))
    names = p.kernels({"x%d" % i: host.channels_last("uint8", (2, 64, 8, 8)) for i in range(2)})
    assert len(names) == 3, names


def inverted_residuals(host):
    p = Program(host)
    x, scale = [p.b.input("x%d" % i, "uint8", [2, 16, 8, 8]) for i in range(2)], p.b.scales(0.1, 7)
    mid = p.b.scales(0.2, 0)
    h = [p.convolution(v, scale, (96, 16, 1, 1), mid) for v in x]
    for slot in scale:
        p.b.Free(slot)
    h = [p.convolution(v, mid, (96, 1, 3, 3), mid, group=96) for v in h]
    for i, v in enumerate(h):
        p.b.output("y%d" % i, p.convolution(v, mid, (24, 96, 1, 1), p.b.scales(0.3, 128)))
    names = p.kernels({"x%d" % i: host.channels_last("uint8", (2, 16, 8, 8)) for i in range(2)})
    assert names.count("inverted_residual_kernel") == 1 and len(names) == 4, names


def bottlenecks(host):
    """A block's own operand is freed inside it, where a last layer reads it too."""
    p = Program(host)
    x, r, f = p.b.input("x", "uint8", [2, 64, 8, 8]), p.b.input("r", "uint8", [2, 256, 8, 8]), p.b.input("f", "uint8", [2, 64, 1, 1])
    shared, mid = p.b.scales(0.1, 7), p.b.scales(0.2, 0)
    head = p.convolution(f, shared, (16, 64, 1, 1), mid)
    h = p.convolution(x, shared, (64, 64, 3, 3), mid)
    for slot in shared:
        p.b.Free(slot)
    h = p.convolution(h, mid, (256, 64, 1, 1), mid)
    p.b.output("sum", p.b.ElementWiseNvrtc([h, r], 1, os.environ["SUM_CODE"], 0, num_list_outputs=1)[0])
    p.b.output("y", p.b.DequantizeLinear(head, *mid))
    names = p.kernels({"x": host.channels_last("uint8", (2, 64, 8, 8)), "r": host.channels_last("uint8", (2, 256, 8, 8)), "f": host.channels_last("uint8", (2, 64, 1, 1))})
    assert names.count("bottleneck_kernel") == 1 and len(names) == 3, names


def products(host):
    """Two chains over one matrix."""
    import numpy as np
    p = Program(host)
    x, scale, zero = p.b.input("x", "float32", [32, 64]), p.b.scales(0.1, 7), p.b.scalar(0, "int8")
    q = [p.b.QuantizeLinear(x, *scale) for _ in range(2)]
    p.b.Free(x)
    for i in range(2):
        own = p.b.scales(0.2, 3)
        w = p.b.DequantizeLinear(p.b.constant(np.ones((64, 32), np.int8)), p.b.scalar(0.01, "float32"), zero)
        y = p.b.QuantizeLinear(p.b.MatMul(p.b.DequantizeLinear(q[i], *scale), w), *own)
        p.b.output("y%d" % i, p.b.DequantizeLinear(y, *own))
    names = p.kernels({"x": host.tensor("float32", (32, 64))})
    assert names.count("matmul_chain_kernel") == 1, names


def a_pool_between(host):
    """The Free waits for a pool that runs on the codes, inside the range of a last layer with the same scale."""
    p = Program(host)
    x, f = p.b.input("x", "uint8", [2, 64, 8, 8]), p.b.input("f", "uint8", [2, 64, 1, 1])
    shared, own = p.b.scales(0.1, 7), p.b.scales(0.2, 3)
    head = p.convolution(f, shared, (16, 64, 1, 1), own)
    d, pooled = p.b.DequantizeLinear(x, *shared), p.b.new_slot()
    p.b.add_raw("AveragePool", [("ARRAY", d), ("INTS", [2, 2]), ("INTS", [2, 2]), ("INTS", [0, 0]), ("INT", 0)], [pooled, -1])
    for slot in shared:
        p.b.Free(slot)
    p.b.output("pooled", p.b.QuantizeLinear(pooled, *p.b.scales(0.3, 0)))
    p.b.output("y", p.b.DequantizeLinear(head, *own))
    names = p.kernels({"x": host.channels_last("uint8", (2, 64, 8, 8)), "f": host.channels_last("uint8", (2, 64, 1, 1))})
    assert len(names) == 3, names


def one_group(host):
    """A Free that one group has for itself is no hindrance, nor is one between two groups."""
    p = Program(host)
    x, scale, mid = p.b.input("x", "float32", [2, 3, 8, 8]), p.b.scales(0.1, 7), p.b.scales(0.2, 0)
    q = p.b.QuantizeLinear(x, *scale)
    p.b.Free(x)
    h = p.convolution(q, scale, (32, 3, 3, 3), mid)
    for slot in (q,) + scale:
        p.b.Free(slot)
    head = p.convolution(h, mid, (16, 32, 1, 1), mid)
    p.b.Free(h)
    p.b.output("y", p.b.DequantizeLinear(head, *mid))
    names = p.kernels({"x": host.tensor("float32", (2, 3, 8, 8))})
    assert len(names) == 2, names


if __name__ == "__main__":
    host_hip.main(globals())
