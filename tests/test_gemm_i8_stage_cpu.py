"""Which kernel an integer product runs on (csrc/gemm_i8.hip), without a GPU: the tiles that tests/test_gpu_gemm_i8_stage.py
means to reach, and the forms that the staged kernel does not take."""
import ctypes

import pytest

import host_hip


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["tiles", "other_forms", "short_k", "batches", "large", "few_columns"])
def test_case(host_so, case):
    from test_gpu_gemm_i8_stage import SHAPES
    host_hip.run_case(host_so, __file__, case, SHAPES=repr(SHAPES))


def kernel(host, a, b, y):
    host.clear()
    host.check(host.lib.chx_hip_matmul_integer(ctypes.byref(a), ctypes.byref(b), None, None, ctypes.byref(y), None))
    names = host.launches()
    assert len(names) == 1
    return names[0]


def product(host, M, K, N, transposed=False, a_strides=None, b_strides=None):
    a, y = host.tensor("uint8", (M, K), a_strides), host.tensor("int32", (M, N))
    b = host.tensor("int8", (K, N), [1, K] if transposed else b_strides)
    return kernel(host, a, b, y)


def tiles(host):
    import os
    for M, K, N, tile, tile_transposed in eval(os.environ["SHAPES"]):
        for transposed, want in ((False, tile), (True, tile_transposed)):
            name = product(host, M, K, N, transposed)
            if want is None:
                assert "gemm_i8_split_kernel" in name, (M, K, N, name)
            else:
                assert "gemm_i8_stage_kernel<%s, %s>" % ("true" if transposed else "false", want) in name, (M, K, N, transposed, name)


def other_forms(host):
    assert "stage" in product(host, 1024, 1024, 4096)
    assert "stage" in product(host, 1024, 1024, 4096, a_strides=[1100, 1])
    assert "stage" not in product(host, 1024, 1024, 4096, a_strides=[1 << 24, 1])  # offsets in a tile beyond 32 bits
    assert "stage" not in product(host, 4096, 4096, 15)  # a row shorter than a read
    assert "stage" not in product(host, 4096, 176, 4096)  # one stage and a part
    assert "stage" not in product(host, 32, 512, 512)


def short_k(host):
    """Two or three whole stages of K: the split kernel, but for b transposed, rows of y that are no whole lines, and int32 from K 256 on."""
    def codes(M, K, N):
        a, b, y = host.tensor("uint8", (M, K)), host.tensor("int8", (K, N)), host.tensor("uint8", (M, N))
        host.clear()
        scale = ctypes.c_float
        host.check(host.lib.chx_hip_qlinear_matmul(ctypes.byref(a), scale(0.02), 128, ctypes.byref(b), scale(0.005), 0, scale(0.04), 128, None, 0, ctypes.byref(y), None))
        return host.launches()[0]

    assert "split" in codes(8192, 192, 4096) and "split" in codes(32768, 256, 4096) and "split" in codes(8192, 320, 1024)
    assert "stage" in codes(8192, 384, 1024) and "stage" in codes(26288, 252, 2944) and "stage" in codes(8192, 256, 2712)
    assert "split" in product(host, 100352, 192, 256) and "split" in product(host, 8192, 192, 8192)
    assert "stage" in product(host, 8192, 384, 1024) and "stage" in product(host, 33449, 192, 1044)
    assert "stage" in product(host, 8192, 256, 1024) and "stage" in product(host, 8192, 192, 8192, transposed=True)


def batches(host):
    """Two or three stages of K in batches whose tiles are mostly padding: the split kernel."""
    def kernel_of(batch, M, K, N):
        a, b, y = host.tensor("uint8", (batch, M, K)), host.tensor("int8", (batch, K, N)), host.tensor("int32", (batch, M, N))
        return kernel(host, a, b, y)

    assert "split" in kernel_of(17, 638, 295, 146) and "split" in kernel_of(454, 68, 259, 21)
    assert "stage" in kernel_of(7, 704, 213, 634) and "stage" in kernel_of(331, 304, 302, 79) and "stage" in kernel_of(17, 638, 400, 146)


def large(host):
    """Operands that leave the caches, for which the times behind the choice would name the split kernel."""
    def codes(M, K, N):
        a, b, y = host.tensor("uint8", (M, K)), host.tensor("int8", (K, N)), host.tensor("uint8", (M, N))
        host.clear()
        scale = ctypes.c_float
        host.check(host.lib.chx_hip_qlinear_matmul(ctypes.byref(a), scale(0.02), 128, ctypes.byref(b), scale(0.005), 0, scale(0.04), 128, None, 0, ctypes.byref(y), None))
        return host.launches()[0]

    for shape in ((27015, 4416, 3968), (13507, 5184, 6528), (12686, 3152, 6208), (65536, 768, 128)):
        assert "gemm_i8_stage_kernel" in codes(*shape) and "gemm_i8_stage_kernel" in product(host, *shape), shape


def few_columns(host):
    assert "stage_short" in product(host, 65281, 768, 15) and "stage_short" in product(host, 65281, 768, 4) and "stage_short" in product(host, 65281, 1000, 8, b_strides=[20, 1])
    assert "split" in product(host, 65280, 768, 15) and "split" in product(host, 65281, 767, 15) and "split" in product(host, 65281, 768, 3)
    assert "gemm_i8_stage_kernel<true, 2, 1, 4>" in product(host, 65281, 768, 8, transposed=True) and "split" in product(host, 65281, 768, 8, b_strides=[7, 1])  # (rows that overlap)


if __name__ == "__main__":
    host_hip.main(globals())
