"""The matrix-core integer products (csrc/gemm_i8.hip) against exact integer arithmetic, where their tiles, K steps and
rows have remainders."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util
    return gpu_util


def codes(rng, shape, dt):
    lo, hi = (0, 256) if dt == np.uint8 else (-128, 128)
    return rng.integers(lo, hi, size=shape).astype(dt)


def exact(a, b, az, bz):
    return np.matmul(a.astype(np.int64) - az, b.astype(np.int64) - bz).astype(np.int32)


# M, N, K around the tiles of 32, 64 and 128, the K steps of 32 and 128, rows shorter than a dword; one shape per kernel
SHAPES = [(1, 1, 16), (1, 2, 17), (5, 3, 31), (32, 4, 32), (33, 5, 33), (31, 127, 47), (64, 128, 64), (65, 129, 100), (197, 1001, 770), (2, 10, 4096),
          (1024, 130, 48), (2100, 1030, 144), (1700, 1800, 131)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("dts", [(np.uint8, np.int8), (np.int8, np.uint8)])
def test_matmul_integer_shapes(g, M, N, K, dts):
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    a, b = codes(rng, (M, K), dts[0]), codes(rng, (K, N), dts[1])
    for az, bz in [(None, None), (128 if dts[0] == np.uint8 else -3, 0), (7, rng.integers(0, 100, size=N))]:
        bzt = None if bz is None else g.dev(np.asarray(bz).astype(dts[1]))
        azt = None if az is None else g.dev(np.asarray(az).astype(dts[0]))
        want = exact(a, b, 0 if az is None else az, 0 if bz is None else np.asarray(bz))
        got = g.ops.MatMulInteger(g.dev(a), g.dev(b), azt, bzt)
        np.testing.assert_array_equal(g.host(got), want)
        # b as the transposed view of an [N, K] array
        bt = g.dev(np.ascontiguousarray(b.T)).t()
        np.testing.assert_array_equal(g.host(g.ops.MatMulInteger(g.dev(a), bt, azt, bzt)), want)


@pytest.mark.parametrize("batch,M,N,K", [(3, 16, 40, 64), (12, 200, 190, 64), (40, 512, 384, 33)])
def test_matmul_integer_batches(g, batch, M, N, K):
    rng = np.random.default_rng(batch)
    a, b = codes(rng, (batch, M, K), np.uint8), codes(rng, (batch, K, N), np.int8)
    got = g.ops.MatMulInteger(g.dev(a), g.dev(b), g.dev(np.array(9, np.uint8)), g.dev(np.array(-5, np.int8)))
    np.testing.assert_array_equal(g.host(got), exact(a, b, 9, -5))


@pytest.mark.parametrize("M,N,K", [(5, 3, 31), (32, 100, 784), (65, 129, 100), (2100, 1030, 144)])
@pytest.mark.parametrize("flags", ["reference", "rne_relu"])
def test_qlinear_matmul_shapes(g, oracle, M, N, K, flags):
    rng = np.random.default_rng(M + N + K)
    a, b, bias = codes(rng, (M, K), np.uint8), codes(rng, (K, N), np.int8), rng.integers(-3000, 3000, size=N).astype(np.int32)
    s_y = float(0.02 * 0.005 * 74 * 74 * np.sqrt(K) / 32)
    rne = flags == "rne_relu"
    fl = (g.capi.ROUND_ONNX_RNE | g.capi.FUSE_RELU) if rne else 0
    for bz in (0, 4):
        got = g.ops.QLinearMatMul(g.dev(a), 0.02, 117, g.dev(b), 0.005, bz, s_y, 128, g.dev(bias), flags=fl)
        want = oracle.qlinear_matmul_int(a, 0.02, 117, b, 0.005, bz, s_y, 128, bias=bias, relu=rne,
                                         round_mode=oracle.ROUND_ONNX_RNE if rne else oracle.ROUND_REFERENCE)
        np.testing.assert_array_equal(g.host(got), want)


def test_views_into_larger_arrays(g):
    """Rows of every alignment: operands and result are blocks of larger arrays."""
    rng = np.random.default_rng(0)
    A, B = codes(rng, (80, 411), np.uint8), codes(rng, (300, 517), np.int8)
    at, bt = g.dev(A), g.dev(B)
    y = torch.zeros((80, 600), dtype=torch.int32, device="cuda")
    for off in (1, 2, 3, 7):
        a, b = at[3:70, off:off + 201], bt[5:206, off:off + 333]
        out = y[2:69, off:off + 333]
        y.zero_()
        g.ops.MatMulInteger(a, b, None, None, out=out)
        np.testing.assert_array_equal(g.host(out), exact(A[3:70, off:off + 201], B[5:206, off:off + 333], 0, 0))
        y[2:69, off:off + 333] = 0
        assert not y.any()


# tiles of 64 x 128 of gemm_i8_stage_kernel, many and with remainders of each
LARGE = (4099, 2070, 1037)
ROWS = sorted({0, 1, 30, 31, 32, 63, 64, 127, 128, 255, 256, 257, 1023, 2047, 4095, 4096, 4097, 4098})


@pytest.mark.parametrize("transposed", [False, True])
def test_large_products(g, oracle, transposed):
    M, N, K = LARGE
    rng = np.random.default_rng(1)
    a, b = codes(rng, (M, K), np.uint8), codes(rng, (K, N), np.int8)
    bd = g.dev(np.ascontiguousarray(b.T)).t() if transposed else g.dev(b)
    bz = rng.integers(-9, 9, size=N).astype(np.int8)
    for az, z in [(128, np.zeros((), np.int8)), (3, bz)]:
        got = g.ops.MatMulInteger(g.dev(a), bd, g.dev(np.array(az, np.uint8)), g.dev(z))
        want = np.matmul(a.astype(np.float64) - az, b.astype(np.float64) - z).astype(np.int32)  # (exact: below 2^53)
        np.testing.assert_array_equal(g.host(got), want)
    s_y = float(0.02 * 0.005 * 74 * 74 * np.sqrt(K) / 40)
    for zp, fl, dt in [(0, 0, torch.uint8), (128, g.capi.FUSE_RELU, torch.uint8), (-5, g.capi.ROUND_ONNX_RNE, torch.int8)]:
        got = g.host(g.ops.QLinearMatMul(g.dev(a), 0.02, 117, bd, 0.005, 4, s_y, zp, None, flags=fl, zero_point_dtype=dt))
        want = oracle.qlinear_matmul_int(a[ROWS], 0.02, 117, b, 0.005, 4, s_y, zp, y_dtype=np.uint8 if dt == torch.uint8 else np.int8, relu=fl == g.capi.FUSE_RELU,
                                         round_mode=oracle.ROUND_ONNX_RNE if fl == g.capi.ROUND_ONNX_RNE else oracle.ROUND_REFERENCE)
        np.testing.assert_array_equal(got[ROWS], want)


# shapes by the wavefronts that share a tile's rows out, and ragged columns
@pytest.mark.parametrize("M,N,K", [(16, 64, 16), (40, 70, 64), (33, 130, 400), (300, 258, 2000), (1030, 515, 40), (2100, 1031, 144)])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -3, 1e-25, 1e25])
def test_every_form_of_the_requantization(g, oracle, M, N, K, scale):
    """The short forms, the folded ones and, at scales whose values might leave float32's range on the way, the divisions."""
    rng = np.random.default_rng(M + K)
    a, b, bias = codes(rng, (M, K), np.uint8), codes(rng, (K, N), np.int8), rng.integers(-3000, 3000, size=N).astype(np.int32)
    rows = [r for r in ROWS if r < M - 1] + [M - 1]
    s_a = 0.02 * scale
    s_y = float(np.float32(s_a * 0.005 * 74 * 74 * np.sqrt(K) / 45))
    for zp, relu, rne, dt in [(0, False, False, torch.uint8), (0, True, False, torch.uint8), (128, False, False, torch.uint8), (9, True, False, torch.uint8),
                              (3, False, False, torch.int8), (-7, True, False, torch.int8), (120, False, True, torch.uint8), (5, True, True, torch.int8)]:
        fl = (g.capi.ROUND_ONNX_RNE if rne else 0) | (g.capi.FUSE_RELU if relu else 0)
        for bd, bq in [(g.dev(bias), bias), (None, None)]:
            got = g.host(g.ops.QLinearMatMul(g.dev(a), s_a, 117, g.dev(b), 0.005, 0, s_y, zp, bd, flags=fl, zero_point_dtype=dt))
            want = oracle.qlinear_matmul_int(a[rows], s_a, 117, b, 0.005, 0, s_y, zp, bias=bq, y_dtype=np.uint8 if dt == torch.uint8 else np.int8, relu=relu,
                                             round_mode=oracle.ROUND_ONNX_RNE if rne else oracle.ROUND_REFERENCE)
            np.testing.assert_array_equal(got[rows], want)
