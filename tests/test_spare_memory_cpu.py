"""Programs whose operands there is no memory for in a second order (runtime/chxvm.cc), without a GPU: they load and run as they are written."""
import ctypes
import os
import re

import pytest

import host_hip
from test_groups_and_frees_cpu import Program, sum_code  # noqa: F401  (sum_code: the fixture)


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["bottleneck", "inverted_residual", "chain", "plans_of_the_ends"])
def test_case(host_so, sum_code, case):  # noqa: F811
    host_hip.run_case(host_so, __file__, case, SUM_CODE=sum_code)


def without_memory(host, build, inputs, kernel, layout):
    """build(): a program; kernel: of its one launch; layout: of the kernel that lays its operands out."""
    host.hh.hh_no_memory.argtypes = [ctypes.c_size_t]
    rt = host.chxvm.runtime()
    assert rt.chxvm_set_option(b"qlinearconv_bias", b"onnx_int32") == 0
    host.clear()
    p = host.program(build())
    log = host.log()
    at = next(i for i, line in enumerate(log) if line.startswith("launch ") and layout in line)
    size = int(next(line for line in reversed(log[:at]) if line.startswith("hipMalloc ")).split()[1])

    def fused(p):
        out = ctypes.c_void_p()
        host.clear()
        assert rt.chxvm_program_run(p, *host.names_and(inputs), 0, ctypes.byref(out)) == 0, rt.chxvm_last_error()
        rt.chxvm_outputs_destroy(out)
        names = [re.match(r"(?:void )?(?:\w+::|\(anonymous namespace\)::)*(\w+)", line).group(1) for line in host.launches()]
        return kernel in names

    assert fused(p)
    host.hh.hh_no_memory(size)
    without = host.program(build())
    host.hh.hh_no_memory(0)
    assert not fused(without) and not fused(without) and fused(host.program(build()))


def bottleneck(host):
    def build():
        p = Program(host)
        x, r, mid = p.b.input("x", "uint8", [2, 64, 8, 8]), p.b.input("r", "uint8", [2, 256, 8, 8]), p.b.scales(0.2, 0)
        h = p.convolution(p.convolution(x, p.b.scales(0.1, 7), (64, 64, 3, 3), mid), mid, (256, 64, 1, 1), mid)
        p.b.output("y", p.b.ElementWiseNvrtc([h, r], 1, os.environ["SUM_CODE"], 0, num_list_outputs=1)[0])
        return p.b

    without_memory(host, build, {"x": host.channels_last("uint8", (2, 64, 8, 8)), "r": host.channels_last("uint8", (2, 256, 8, 8))}, "bottleneck_kernel", "pack_bottleneck")


def inverted_residual(host):
    def build():
        p = Program(host)
        mid = p.b.scales(0.2, 0)
        h = p.convolution(p.b.input("x", "uint8", [2, 16, 8, 8]), p.b.scales(0.1, 7), (96, 16, 1, 1), mid)
        p.b.output("y", p.convolution(p.convolution(h, mid, (96, 1, 3, 3), mid, group=96), mid, (24, 96, 1, 1), p.b.scales(0.3, 128)))
        return p.b

    without_memory(host, build, {"x": host.channels_last("uint8", (2, 16, 8, 8))}, "inverted_residual_kernel", "pack_inverted")


def chain(host):
    import numpy as np

    def build():
        p = Program(host)
        scale, own = p.b.scales(0.1, 7), p.b.scales(0.2, 3)
        w = p.b.DequantizeLinear(p.b.constant(np.ones((64, 32), np.int8)), p.b.scalar(0.01, "float32"), p.b.scalar(0, "int8"))
        x = p.b.DequantizeLinear(p.b.QuantizeLinear(p.b.input("x", "float32", [32, 64]), *scale), *scale)
        p.b.output("y", p.b.DequantizeLinear(p.b.QuantizeLinear(p.b.MatMul(x, w), *own), *own))
        return p.b

    without_memory(host, build, {"x": host.tensor("float32", (32, 64))}, "matmul_chain_kernel", "chain_weights_kernel")


def plans_of_the_ends(host):
    """A convolution has one plan, of the launch with its quantization in front or behind and of its instruction where that launch does not take it; one
    that there is no memory for is missed by the instruction first."""
    host.hh.hh_no_memory.argtypes = [ctypes.c_size_t]
    rt = host.chxvm.runtime()
    assert rt.chxvm_set_option(b"qlinearconv_bias", b"onnx_int32") == 0

    def build():
        p = Program(host)
        scale, mid = p.b.scales(0.1, 7), p.b.scales(0.2, 0)
        h = p.convolution(p.convolution(p.b.QuantizeLinear(p.b.input("x", "float32", [8, 3, 32, 32]), *scale), scale, (32, 3, 3, 3), mid), mid, (64, 32, 1, 1), mid)
        p.b.output("y", p.b.DequantizeLinear(h, *mid))
        return p.b

    def run(program, batch):
        out = ctypes.c_void_p()
        rc = rt.chxvm_program_run(program, *host.names_and({"x": host.tensor("float32", (batch, 3, 32, 32))}), 0, ctypes.byref(out))
        rt.chxvm_outputs_destroy(out)
        return rc

    for batches in ((8, 9, 8), (9, 8, 9)):  # (the last layer's results: 2^19 and more)
        host.clear()
        program = host.program(build())
        for n in batches:
            at = len(host.launches())
            assert run(program, n) == 0, rt.chxvm_last_error()
            assert any("dequantize" in k for k in host.launches()[at:]) == (n == 9)
        names = " ".join(host.launches())
        # (the first layer's weights are laid out in two orders by a launch each)
        assert (names.count("pack_weights_stem_kernel"), names.count("pack_weights_dense_kernel"), names.count("pack_weights_kernel")) == (1, 1, 1), names
        graph = ctypes.c_void_p()  # the plan of a recording outlives the program
        assert rt.chxvm_program_capture(program, *host.names_and({"x": host.tensor("float32", (batches[0], 3, 32, 32))}), ctypes.byref(graph)) == 0, rt.chxvm_last_error()
        rt.chxvm_program_destroy(program)
        assert rt.chxvm_replay_launch(graph, None) == 0
        rt.chxvm_replay_destroy(graph)
    log = host.log()
    at = next(i for i, line in enumerate(log) if "pack_weights_kernel" in line)
    host.hh.hh_no_memory(int(next(line for line in reversed(log[:at]) if line.startswith("hipMalloc ")).split()[1]))
    program = host.program(build())
    assert run(program, 8) != 0 and b"hipMalloc" in rt.chxvm_last_error()
    host.hh.hh_no_memory(0)
    assert run(program, 8) == 0, rt.chxvm_last_error()


if __name__ == "__main__":
    host_hip.main(globals())
