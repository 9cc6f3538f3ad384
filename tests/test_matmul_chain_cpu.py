"""Which programs run products as a chain (runtime/chxvm.cc) and which instructions of theirs still run, without a GPU."""
import ctypes
import re

import pytest

import host_hip

CHAIN, QUANTIZE, PRODUCT, DEQUANTIZE = "matmul_chain_kernel", "quantize_flat_kernel", "gemm_i8_split_kernel", "dequantize_flat_kernel"


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["whole_networks", "values_read_twice", "frees_between", "frees_in_front", "refused_forms", "many_rows", "errors", "another_device", "instruction_by_instruction"])
def test_case(host_so, case):
    host_hip.run_case(host_so, __file__, case)


def program(host, dims=(96, 64, 32), rows=8, quantize=True, dequantize=True, free=False, extra=None, x_shape=None, quantized_again=False):
    import numpy as np
    b = host.chxvm.ProgramBuilder()
    h = b.input("x", "float32" if quantize else "uint8", x_shape or [rows, dims[0]])
    scale, zp = b.scalar(0.1, "float32"), b.scalar(128, "uint8")

    def free_of(*slots):
        if free:
            for s in slots:
                b.Free(s)

    if quantize:
        q = b.QuantizeLinear(h, scale, zp)
        free_of(h)
        h = q
    for i in range(len(dims) - 1):
        w, ws, wz = b.constant(np.ones((dims[i], dims[i + 1]), np.int8)), b.scalar(0.01, "float32"), b.scalar(0, "int8")
        fa = b.DequantizeLinear(h, scale, zp)
        free_of(h, scale, zp)
        fb = b.DequantizeLinear(w, ws, wz)
        free_of(w, ws, wz)
        product = b.MatMul(fa, fb)
        free_of(fa, fb)
        scale, zp = b.scalar(0.3 + i, "float32"), b.scalar(128, "uint8")
        h = b.QuantizeLinear(product, scale, zp)
        free_of(product)
        if extra == i:
            b.output("between", h)
    if dequantize:
        d = b.DequantizeLinear(h, scale, zp)
        free_of(h, scale, zp)
        h = d
    if quantized_again:
        h = b.QuantizeLinear(d, b.scalar(0.7, "float32"), b.scalar(1, "uint8"))
        free_of(d)
    b.output("y", h)
    return host.program(b)


def kernels(host, p, x_shape, dtype="float32", strides=None):
    x = host.tensor(dtype, x_shape, strides)
    host.clear()
    rt, out = host.chxvm.runtime(), ctypes.c_void_p()
    assert rt.chxvm_program_run(p, *host.names_and({"x": x}), 0, ctypes.byref(out)) == 0, rt.chxvm_last_error()
    names = [re.match(r"(?:void )?(?:\w+::|\(anonymous namespace\)::)*(\w+)", line).group(1) for line in host.launches()]
    rt.chxvm_outputs_destroy(out)
    return names


def whole_networks(host):
    for free in (False, True):
        for _ in range(2):
            assert kernels(host, program(host, free=free), (8, 96)) == [CHAIN]
    assert kernels(host, program(host, dequantize=False), (8, 96)) == [CHAIN]
    assert kernels(host, program(host, quantize=False), (8, 96), "uint8") == [CHAIN]
    assert kernels(host, program(host, (96, 64), quantize=False, dequantize=False), (8, 96), "uint8") == [PRODUCT]
    assert kernels(host, program(host, (96,) + (64,) * 8), (8, 96)) == [CHAIN, CHAIN]  # eight layers


def values_read_twice(host):
    # what the program gives out between two layers ends one chain and starts another
    assert kernels(host, program(host, (96, 64, 32, 16), extra=1), (8, 96)) == [CHAIN, CHAIN]


def frees_between(host):
    p = program(host, (96, 64, 32, 16), free=True)
    for _ in range(3):
        assert kernels(host, p, (8, 96)) == [CHAIN]
        # also where the instructions run one by one: every other column of an array
        assert kernels(host, p, (8, 96), strides=[192, 2]) == ["quantize_strided_kernel", PRODUCT, PRODUCT, PRODUCT, DEQUANTIZE]


def frees_in_front(host):
    """A chain without a QuantizeLinear in front gives back its input: the Free of it stands in front of the chain's first instruction."""
    # six layers, two layers, and a QuantizeLinear whose result (512 KB) takes the place of what lies between the two chains
    p = program(host, (64,) * 9, rows=8192, free=True, quantized_again=True)
    assert kernels(host, p, (8192, 64)) == [CHAIN, CHAIN, QUANTIZE]
    assert host.log().count("hipMalloc %d" % (8192 * 64)) == 1


def refused_forms(host):
    # a layer that is too large, and the chain of the others
    assert kernels(host, program(host, (1025, 64, 32)), (8, 1025)) == [QUANTIZE, PRODUCT, CHAIN]
    assert kernels(host, program(host, (96, 513, 32)), (8, 96)) == [QUANTIZE, PRODUCT, CHAIN]
    assert kernels(host, program(host, (96, 64, 513)), (8, 96)) == [CHAIN, PRODUCT, DEQUANTIZE]


def many_rows(host):
    """Above 8192 rows narrow layers are launches of their own."""
    for dims, rows, chain in (((1005, 32, 107), 15797, False), ((1005, 32, 107), 8192, True), ((784, 100, 100, 10), 16384, True), ((1024, 512, 512, 100), 16384, True),
                              ((512,) * 7, 16384, True), ((64, 512, 16), 16385, False)):
        codes = dims[0] == 1005
        p = program(host, dims, rows=rows, quantize=not codes, dequantize=not codes)
        assert (CHAIN in kernels(host, p, (rows, dims[0]), "uint8" if codes else "float32")) == chain, (dims, rows)


def errors(host):
    """An error names the instruction that it is of, not the one that the chain stands in the place of."""
    # x has a column too many for the first product, the 12th instruction
    assert "Exception in QuantizeLinear (pc 12)" in host.run_fails(program(host), {"x": host.tensor("float32", (8, 97))})


def another_device(host):
    """The weights are laid out in one device's memory: on another one the instructions run."""
    p = program(host)
    host.check(host.lib.chx_hip_init(1))
    assert kernels(host, p, (8, 96)) == [QUANTIZE, PRODUCT, PRODUCT, DEQUANTIZE]
    host.check(host.lib.chx_hip_init(0))
    assert kernels(host, p, (8, 96)) == [CHAIN]


def instruction_by_instruction(host):
    """A run that looks at the values between the instructions sees all of them."""
    rt = host.chxvm.runtime()
    p = program(host)
    assert rt.chxvm_set_option(b"check_types", b"on") == 0
    assert kernels(host, p, (8, 96)) == [QUANTIZE, PRODUCT, PRODUCT, DEQUANTIZE]
    assert rt.chxvm_set_option(b"check_types", b"off") == 0
    assert kernels(host, p, (8, 96)) == [CHAIN]


if __name__ == "__main__":
    host_hip.main(globals())
